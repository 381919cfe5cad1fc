// Digit images of the decode kernels' activation rows (pf_moe_decode.hip), and the lane moves and scalar pieces of the block
// formats that they share with the other kernels with integer products (pf_moe_batch.hip, whose images are finer).
#pragma once
#include "pf_moe_internal.h"

__device__ __forceinline__ int dpp_quad_xor1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true); }
__device__ __forceinline__ int dpp_quad_xor2(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true); }

// ---- digit images in global memory (kernels whose lanes are weight rows) ------------------------
// Where every lane of a wave is a weight row, the activation digits are the same for the whole wave and
// travel through scalar registers: the image lives in global memory (pf_image2_words), written by the
// kernel before.  PF_IMG_PLANES balanced base-256 digits (signed bytes): the values as integers relative
// to a step per 32-group that puts the group's largest magnitude at 127 * 256^(planes - 1); the rounding
// error is at most 2^-24 of that magnitude with three planes.
#define PF_IMG_TOP (PF_IMG_PLANES == 3 ? 8323072.0f : 32512.0f)   // the integer the group's largest magnitude becomes: 127 * 256^(planes - 1)
__device__ __forceinline__ void group_step2(float m, float &step, float &inv) {
    const bool none = !(m > 1e-30f);   // an all-zero (or vanishing) group
    inv = none ? 0.0f : PF_IMG_TOP / m;
    step = none ? 0.0f : m * (1.0f / PF_IMG_TOP);
}
// balanced base-256 digits of q, lowest first (each in -128..127)
template <int PLANES> __device__ __forceinline__ void image_digits(int q, int (&d)[PLANES]) {
#pragma unroll
    for (int p = 0; p + 1 < PLANES; p++) {
        d[p] = ((q + 128) & 255) - 128;
        q = (q - d[p]) >> 8;
    }
    d[PLANES - 1] = q;
}
// the integer dot product from its per-plane parts (float: three planes leave 32 bits)
__device__ __forceinline__ float image_value(const int (&part)[PF_IMG_PLANES]) {
    float v = (float)part[PF_IMG_PLANES - 1];
#pragma unroll
    for (int p = PF_IMG_PLANES - 2; p >= 0; p--) v = fmaf(256.0f, v, (float)part[p]);
    return v;
}

// Thread j of a group of four neighbouring lanes: the eight values 8j..8j+7 of a K-vector into its image.
__device__ __forceinline__ bool image2_chunk(uint32_t *img, const float4 a, const float4 b, int j, int K) {
    bool bad = false;
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; c++) { m = fmaxf(m, fabsf(v[c])); bad |= !pf_finite(v[c]); }
    m = fmaxf(m, __int_as_float(dpp_quad_xor1(__float_as_int(m))));
    m = fmaxf(m, __int_as_float(dpp_quad_xor2(__float_as_int(m))));
    float step, inv;
    group_step2(m, step, inv);
    uint32_t w[PF_IMG_PLANES][2] = {};
    int sum = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int q = __float2int_rn(v[c] * inv);
        sum += q;
        int d[PF_IMG_PLANES];
        image_digits(q, d);
#pragma unroll
        for (int p = 0; p < PF_IMG_PLANES; p++) w[p][c >> 2] |= (uint32_t)(d[p] & 255) << (8 * (c & 3));
    }
    sum += dpp_quad_xor1(sum);
    sum += dpp_quad_xor2(sum);
    const int g = j >> 2, at = PF_IMG_GROUP * g + 2 * (j & 3);
#pragma unroll
    for (int p = 0; p < PF_IMG_PLANES; p++) { img[at + 8 * p] = w[p][0]; img[at + 8 * p + 1] = w[p][1]; }
    if ((j & 3) == 0) {
        img[PF_IMG_GROUP * (K / 32) + g] = __float_as_uint(step);
        img[(PF_IMG_GROUP + 1) * (K / 32) + g] = (uint32_t)sum;
    }
    return bad;
}

// Lanes 0..31 of a wave, one value each: group g of a K-vector's image.
__device__ __forceinline__ int dpp_row_step(int v, const int which) {
    switch (which) {
    case 0: return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);    // quad_perm [1,0,3,2]
    case 1: return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);    // quad_perm [2,3,0,1]
    case 2: return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);   // row_half_mirror
    default: return __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true);  // row_mirror
    }
}

__device__ __forceinline__ void image2_group(uint32_t *img, float v, int g, int K, int lane) {   // lanes 32..63 idle along
    float m = fabsf(v);
#pragma unroll
    for (int k = 0; k < 4; k++) m = fmaxf(m, __int_as_float(dpp_row_step(__float_as_int(m), k)));
    m = fmaxf(m, __shfl_xor(m, 16));
    float step, inv;
    group_step2(m, step, inv);
    const int q = __float2int_rn(v * inv);
    int sum = q;
#pragma unroll
    for (int k = 0; k < 4; k++) sum += dpp_row_step(sum, k);
    sum += __shfl_xor(sum, 16);
    int d[PF_IMG_PLANES];
    image_digits(q, d);
    uint8_t *bytes = reinterpret_cast<uint8_t *>(img + PF_IMG_GROUP * g);
    if (lane < 32) {
#pragma unroll
        for (int p = 0; p < PF_IMG_PLANES; p++) bytes[32 * p + lane] = (uint8_t)d[p];
    }
    if (lane == 0) {
        img[PF_IMG_GROUP * (K / 32) + g] = __float_as_uint(step);
        img[(PF_IMG_GROUP + 1) * (K / 32) + g] = (uint32_t)sum;
    }
}

__device__ __forceinline__ float half_bits(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)h);
}

// MXFP4: four E2M1 codes of a dword as signed bytes holding twice their value (0, 1, 2, 3, 4, 6, 8, 12):
// one byte permute per sign, merged under the sign bits' byte mask
__device__ __forceinline__ int e2m1_twice4(uint32_t nibbles) {
    const uint32_t sel = nibbles & 0x07070707u;
    const uint32_t pos = __builtin_amdgcn_perm(0x0C080604u, 0x03020100u, sel);
    const uint32_t neg = __builtin_amdgcn_perm(0xF4F8FAFCu, 0xFDFEFF00u, sel);
    const uint32_t mask = ((nibbles >> 3) & 0x01010101u) * 0xFFu;
    return (int)((neg & mask) | (pos & ~mask));
}
