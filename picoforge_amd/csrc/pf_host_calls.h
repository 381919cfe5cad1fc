/* What the C11 host side calls beside the public shim (include/pf_moe_hip.h): plain C. */
#pragma once
#include "../../include/pf_moe_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* pf_hip_moe_forward_host that also looks for input values that are not finite, in the pass that brings the rows into
 * page-locked memory; where it finds one, *nonfinite_input is set, nothing of the caller's has been written and no kernel
 * has been launched. */
int pf_host_forward_checked(const PfHipMoe *moe, PfHipWork *work, const float *x, size_t x_pitch_bytes, float *y, size_t y_pitch_bytes,
                            uint32_t *ids, size_t ids_pitch_bytes, float *weights, size_t weights_pitch_bytes, size_t tokens,
                            uint32_t *error_word, int *nonfinite_input);
/* Whether all of rows x cols floats are finite. */
int pf_host_finite(const float *x, size_t pitch_bytes, size_t rows, size_t cols);

#ifdef __cplusplus
}
#endif
