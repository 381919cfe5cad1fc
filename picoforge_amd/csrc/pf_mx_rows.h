// Digit rows: the activation rows of the MXFP4 down projection as operands of v_mfma_scale_f32_32x32x64_f8f6f4 (pf_moe_mx.hip).
//
// A row whose largest magnitude m is outside [2^-61, 2^60) is divided by the power of two that brings it there, other rows are taken
// as they are: a product with a block scale of 2^125 or 2^-127 is then no larger or smaller on its way than the result.  (Rows
// divided down to [0.5, 1) overflowed on scales that small rows made up for.)  Per group of 32 values with largest
// magnitude below 2^E, plane p is what planes 0 .. p - 1 leave, rounded to a six-bit float (two exponent, three mantissa bits)
// times 2^(E - 2 - 5 p): a remainder is below 4 of its plane's steps, the rounding leaves an eighth of a step at most, so five planes
// leave 2^-25 of the binade of the group's largest magnitude (the two-part halfs of the other grouped products: 2^-23 of the
// value, and not under 2^-25 of the row's).  E is -100 at least, 39 binades under the smallest m.
//
// 128 bytes a group: 16 bytes of each plane's 24 (chunks 0..4), the planes' other 8 bytes, then the five scale bytes, the
// row's exponent and padding.  A slot order within the group that follows MXFP4's nibbles: slot 2 i is column i, slot 2 i + 1 column 16 + i.
#pragma once
#include "pf_grouped.h"

#define PF_MX_PLANES 5
#define PF_MX_TAIL_AT(plane) (80 + 8 * (plane))
#define PF_MX_SCALE_AT(plane) (120 + (plane))
#define PF_MX_EXPONENT_AT 125
#define PF_MX_LINE 128   // bytes of a group; a row of K values takes 4 K bytes

typedef int int8v __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float32v __attribute__((ext_vector_type(32)));
typedef uint32_t uint6v __attribute__((ext_vector_type(6)));

// 32 values as six-bit floats times `scale`, slot 2 i from a[i], slot 2 i + 1 from b[i], and back.  (In assembly: the destination must
// not overlap the sources, which the compiler's own form of the instruction allows.)
__device__ __forceinline__ uint6v pf_to_e2m3(const float16v &a, const float16v &b, float scale) {
    uint6v q;
    asm("v_cvt_scalef32_2xpk16_fp6_f32 %0, %1, %2, %3" : "=&v"(q) : "v"(a), "v"(b), "v"(scale));
    return q;
}
__device__ __forceinline__ float32v pf_from_e2m3(const uint6v &q, float scale) {
    float32v v;
    asm("v_cvt_scalef32_pk32_f32_fp6 %0, %1, %2" : "=&v"(v) : "v"(q), "v"(scale));
    return v;
}

// A lane per group; a wave takes as many whole rows as its lanes hold groups (cols at most 1024, a multiple of 32).
__host__ __device__ constexpr int pf_mx_rows_a_wave(int cols) { return 64 / (cols / 32); }
__device__ __forceinline__ void pf_rows_to_digits(size_t block, const float *src, int cols, size_t rows, uint32_t *dst, float *scale_out, uint32_t *error_word) {   // dst may be src: a lane writes the bytes that it has read
    const int lane = pf_lane(), groups = cols / 32, at = lane / groups, group = lane - at * groups, together = pf_mx_rows_a_wave(cols);
    const size_t row = (block * 4 + (threadIdx.x >> 6)) * together + at;
    const bool mine = at < together && row < rows;
    float16v a, b;   // columns 0..15 and 16..31 of the group
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r = q;
        if (mine) { const float4 *s = reinterpret_cast<const float4 *>(src + row * cols + 32 * group); q = s[i]; r = s[4 + i]; }
        a[4 * i] = q.x; a[4 * i + 1] = q.y; a[4 * i + 2] = q.z; a[4 * i + 3] = q.w;
        b[4 * i] = r.x; b[4 * i + 1] = r.y; b[4 * i + 2] = r.z; b[4 * i + 3] = r.w;
    }
    float most = 0.0f;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 16; i++) { bad |= !(pf_finite(a[i]) && pf_finite(b[i])); most = fmaxf(most, fmaxf(fabsf(a[i]), fabsf(b[i]))); }
    if (__any(bad) && lane == 0) atomicOr(error_word, PF_HIP_ERR_NONFINITE);
    float m = most;   // of the row: each step doubles the groups, in a ring, that a lane has seen
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) m = fmaxf(m, __shfl(m, at * groups + (group + d) % groups));
    const int binade = ((__float_as_int(m) >> 23) & 255) - 126;   // m in [2^(binade-1), 2^binade); a nonfinite row: 129
    const int shift = max(binade - 60, min(binade + 60, 0));
    const float inv = __int_as_float((127 - shift) << 23);
    const int E = max(((__float_as_int(most * inv) >> 23) & 255) - 126, -100);
#pragma unroll
    for (int i = 0; i < 16; i++) { a[i] *= inv; b[i] *= inv; }
    uint6v plane[PF_MX_PLANES];
#pragma unroll
    for (int p = 0; p < PF_MX_PLANES; p++) {
        const float scale = __int_as_float((127 + E - 2 - 5 * p) << 23);
        plane[p] = pf_to_e2m3(a, b, scale);
        if (p + 1 == PF_MX_PLANES) break;
        const float32v back = pf_from_e2m3(plane[p], scale);
#pragma unroll
        for (int i = 0; i < 16; i++) { a[i] -= back[2 * i]; b[i] -= back[2 * i + 1]; }
    }
    if (!mine) return;
    if (group == 0 && scale_out) scale_out[row] = __int_as_float((127 + shift) << 23);
    uint4v *line = reinterpret_cast<uint4v *>(dst + row * cols + 32 * group);
#pragma unroll
    for (int p = 0; p < PF_MX_PLANES; p++) line[p] = uint4v{plane[p][0], plane[p][1], plane[p][2], plane[p][3]};
    line[5] = uint4v{plane[0][4], plane[0][5], plane[1][4], plane[1][5]};
    line[6] = uint4v{plane[2][4], plane[2][5], plane[3][4], plane[3][5]};
    const uint32_t s0 = (uint32_t)(127 + E - 2);   // plane p: 5 p less
    line[7] = uint4v{plane[4][4], plane[4][5], s0 * 0x01010101u - 0x0F0A0500u, (s0 - 20u) | (uint32_t)(127 + shift) << 8};
}
