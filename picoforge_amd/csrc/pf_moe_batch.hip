// Batches between decode and prefill: the expert products of a few rows per expert.
//
// A batch of some tens of tokens meets most of a layer's experts with one to a few rows each.  The grouped product of
// pf_moe_prefill.hip pays for 32 rows whatever a tile holds, and the decode kernels read and unpack an expert's weights once
// per (token, expert) pair.  Here a work item is an expert's row tile (up to 32 rows) against one slab of weight rows: the
// weights come from memory once, and once in registers serve eight rows at a time.
//
//   pf_k_batch_gate_up   gate and up products of 32 units, SwiGLU, the activation rows' digit images (expert order)
//   pf_k_batch_down      down products of 128 output rows, FP32, in expert order (pf_k_pf_combine adds them up); of larger batches
//                        of the q4 profile the shared expert's only, the routed ones by pf_k_mx_down
//
// Arithmetic: the decode kernels'.  Activations are digit images (integers per 32-group as balanced base-256 digits), weight
// codes signed bytes, the group's dot product exact in integers, the group's scale and minimum applied in FP32.  PLANES digits:
//
//   3   resident layers: the decode kernels' 24 bits relative to the group's largest magnitude
//   4   streamed layers, whose batches would otherwise run on FP32 rows (the general kernels): 30 bits and a power of two as the
//       step, 2^-29 of the binade of the group's largest magnitude, so that a value within 2^6 of it is exact, a smaller one
//       off by at most 2^-30 of it, and no group vanishes
//
// Distance to the result in 64 bits, 60 tokens of an IQ2_XXS layer (2-norm; normal rows, and rows with a few channels 300 times
// larger): three digits 2.8e-7 and 3.8e-7, four 1.9e-7 and 1.9e-7; the grouped product of prefill 4.1e-7 and 11e-7, the general
// kernels 2.4e-7 and 2.6e-7.  The fourth digit costs 1 to 3 % of a kernel's time (another addition per sum, a third more
// image to read).  The integer products run on v_mfma_i32_32x32x32_i8, one instruction per 32-group:
//
//   A (rows)     lane (m = lane % 32, h = lane / 32): digit plane m % 4 of the chunk's token m / 4, bytes 16 h .. 16 h + 15
//                of the group (with three planes, plane 3 repeats plane 2; its results are not looked at)
//   B (columns)  lane (n = lane % 32, h): weight row n's codes 16 h .. 16 h + 15 of the group
//   D            lane (n, h), register 4 q + p: weight row n, token 2 q + h, plane p
//
// so the planes of a (row, token) sum meet in one lane, the lane's weight row is the one whose scales it holds, and a
// chunk of up to 2 q tokens only recombines q of the four register quads.  Per 32 x 32 weights: 6 (Q4_K) to 28 (MXFP4)
// vector instructions for the codes, about 5 for the scales, 7 or 8 per quad -- against 36 per token for the dot-product
// instructions of the decode kernels and about 75, whatever the rows, for the FP16 product of the prefill kernels.
#include "pf_grouped.h"
#include "pf_image.h"
#include "pf_route_device.h"

typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int16v __attribute__((ext_vector_type(16)));
typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));

#define BATCH_ROWS 8           // rows of a chunk

// ---- the weights of one 32-row tile and one piece of K ----------------------------------------------
// GROUPS 32-groups in registers: lane (row = lane % 32, h = lane / 32).  operand(g): the row's codes 16 h .. 16 h + 15 of
// group g as signed bytes; scale(g), minimum(g): the factors of the products' and of the activations' sums.
// ROWS: stored row by row; else in the tile order where the format has one.
template <int FMT, bool ROWS> struct BatchRows;

template <bool ROWS> struct BatchRows<PF_Q4_K, ROWS> {   // in tile order a 64-weight run of the tile is one 1 KB load; else GGUF rows
    static constexpr int GROUPS = 8;
    static constexpr bool MINIMA = true, MIN_OPERAND = false;
    uint4 hdr, q[4];
    uint32_t sc[2], mn[2];
    float d, dmin;
    __device__ __forceinline__ void load(const PfKernelArgs &a, int t, size_t e, int tile, int piece, int, int lane, const uint32_t *) {
        if constexpr (!ROWS) {
            const uint8_t *chunk = a.wt[t] + pf_q4t_chunk_at(a.expert_bytes[t], e, tile, a.blocks_per_row[t], piece);
            hdr = *reinterpret_cast<const uint4 *>(chunk + pf_q4t_header_at(lane & 31));
#pragma unroll
            for (int run = 0; run < 4; run++) q[run] = *reinterpret_cast<const uint4 *>(chunk + pf_q4t_piece_at(run, 0, 0) + 16 * lane);
        } else {
            const uint8_t *block = a.w[t] + (e * (size_t)a.n_out[t] + (size_t)(32 * tile)) * a.row_bytes[t] + 144 * (size_t)piece;   // uniform
            const uint32_t at = (uint32_t)(lane & 31) * (uint32_t)a.row_bytes[t], code_at = at + 16 * (uint32_t)(lane >> 5);
            hdr = *reinterpret_cast<const uint4 *>(block + at);
#pragma unroll
            for (int run = 0; run < 4; run++) q[run] = *reinterpret_cast<const uint4 *>((block + 16 + 32 * run) + code_at);
        }
    }
    __device__ __forceinline__ void open() {   // src/qwen4_packed.c:89-90
        d = half_bits(hdr.x & 0xffffu); dmin = half_bits(hdr.x >> 16);
        sc[0] = hdr.y & 0x3f3f3f3fu; mn[0] = hdr.z & 0x3f3f3f3fu;
        sc[1] = (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u);
        mn[1] = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
    }
    __device__ __forceinline__ int4v operand(int g, const uint32_t *) const {
        const uint4 v = q[g >> 1];
        const int s = 4 * (g & 1);
        return int4v{(int)((v.x >> s) & 0x0f0f0f0fu), (int)((v.y >> s) & 0x0f0f0f0fu), (int)((v.z >> s) & 0x0f0f0f0fu), (int)((v.w >> s) & 0x0f0f0f0fu)};
    }
    __device__ __forceinline__ int4v min_operand(int) const { return int4v{0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int g) const { return d * (float)((sc[g >> 2] >> (8 * (g & 3))) & 255u); }
    __device__ __forceinline__ float minimum(int g) const { return dmin * (float)((mn[g >> 2] >> (8 * (g & 3))) & 255u); }
};

// four unsigned magnitudes of at least one and their signs' byte mask: negated where the mask is set (no carry leaves a byte)
__device__ __forceinline__ int signed_bytes(uint32_t magnitudes, uint32_t mask) { return (int)((magnitudes ^ mask) + (mask & 0x01010101u)); }

template <bool ROWS> struct BatchRows<PF_IQ2_XXS, ROWS> {   // in tile order, else payloads row by row; LDS: 256 x 8 magnitudes, then 128 masks of eight sign bytes
    static constexpr int GROUPS = 8;
    static constexpr bool MINIMA = false, MIN_OPERAND = false;
    uint4 q[4];
    uint32_t dbits;
    float d;
    __device__ __forceinline__ void load(const PfKernelArgs &a, int t, size_t e, int tile, int piece, int, int lane, const uint32_t *) {
        const int kblocks = a.blocks_per_row[t];
        if constexpr (!ROWS) {
            const uint8_t *chunk = a.wi[t] + pf_i2t_chunk_at(pf_i2t_expert_bytes(a.n_out[t], kblocks), e, tile, kblocks, piece);
#pragma unroll
            for (int run = 0; run < 4; run++) q[run] = *reinterpret_cast<const uint4 *>(chunk + pf_i2t_piece_at(run, lane & 31));
            dbits = *reinterpret_cast<const uint16_t *>(chunk + pf_i2t_scale_at(lane & 31));
        } else {
            const size_t row0 = e * (size_t)a.n_out[t] + (size_t)(32 * tile);   // uniform
            const uint8_t *block = a.w[t] + row0 * a.row_bytes[t] + 64 * (size_t)piece;
            const uint8_t *scales = a.w[t] + a.scale_offset[t] + 2 * (row0 * (size_t)kblocks + (size_t)piece);
            const uint32_t at = (uint32_t)(lane & 31) * (uint32_t)a.row_bytes[t];
#pragma unroll
            for (int run = 0; run < 4; run++) q[run] = *reinterpret_cast<const uint4 *>((block + 16 * run) + at);
            dbits = *reinterpret_cast<const uint16_t *>(scales + 2 * (uint32_t)(lane & 31) * (uint32_t)kblocks);
        }
    }
    __device__ __forceinline__ void open() { d = 0.125f * half_bits(dbits); }
    __device__ __forceinline__ int4v operand(int g, const uint32_t *tables) const {
        const uint4 v = q[g >> 1];
        const bool high = pf_lane() >= 32;   // the lane's half: slots 0 and 1, or 2 and 3
        const uint32_t idx = ((g & 1) ? v.z : v.x) >> (high ? 16 : 0), signs = ((g & 1) ? v.w : v.y) >> (high ? 14 : 0);
        const uint2 *grid = reinterpret_cast<const uint2 *>(tables), *masks = grid + 256;
        const uint2 m0 = grid[idx & 255u], m1 = grid[(idx >> 8) & 255u], s0 = masks[signs & 127u], s1 = masks[(signs >> 7) & 127u];
        return int4v{signed_bytes(m0.x, s0.x), signed_bytes(m0.y, s0.y), signed_bytes(m1.x, s1.x), signed_bytes(m1.y, s1.y)};
    }
    __device__ __forceinline__ int4v min_operand(int) const { return int4v{0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int g) const { return d * (float)(2u * (((g & 1) ? q[g >> 1].w : q[g >> 1].y) >> 28) + 1u); }
    __device__ __forceinline__ float minimum(int) const { return 0.0f; }
};

template <bool ROWS> struct BatchRows<PF_Q8_0, ROWS> {   // the checkpoint profiles' shared expert: gate and up in tile order, down row by row
    static constexpr int GROUPS = 4;
    static constexpr bool MINIMA = false, MIN_OPERAND = false;
    uint4 q[4];
    uint32_t d2[2];
    __device__ __forceinline__ void load(const PfKernelArgs &a, int t, size_t e, int tile, int piece, int groups, int lane, const uint32_t *) {
        if constexpr (!ROWS) {
            const int runs = a.blocks_per_row[t] / 2, h = lane >> 5;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const uint8_t *chunk = a.wq[t] + pf_q8t_chunk_at(0, 0, tile, runs, 2 * piece + r);
                q[2 * r] = *reinterpret_cast<const uint4 *>(chunk + pf_q8t_piece_at(h, lane & 31));
                q[2 * r + 1] = *reinterpret_cast<const uint4 *>(chunk + pf_q8t_piece_at(2 + h, lane & 31));
                d2[r] = *reinterpret_cast<const uint32_t *>(chunk + pf_q8t_scales_at(lane & 31));
            }
        } else {
            const size_t row0 = e * (size_t)a.n_out[t] + (size_t)(32 * tile);   // uniform; the lane's row by a 32-bit offset
            const uint8_t *codes = a.w[t] + row0 * a.row_bytes[t], *scales = a.w[t] + a.scale_offset[t] + 2 * row0 * (size_t)a.blocks_per_row[t];
            const uint32_t code_at = (uint32_t)(lane & 31) * (uint32_t)a.row_bytes[t] + 16 * (uint32_t)(lane >> 5);
            const uint32_t scale_at = 2 * (uint32_t)(lane & 31) * (uint32_t)a.blocks_per_row[t];
#pragma unroll
            for (int r = 0; r < 2; r++) {   // groups come in pairs (widths are whole 64-value segments)
                const int g = min(GROUPS * piece + 2 * r, groups - 2);
                q[2 * r] = *reinterpret_cast<const uint4 *>((codes + 32 * g) + code_at);
                q[2 * r + 1] = *reinterpret_cast<const uint4 *>((codes + 32 * (g + 1)) + code_at);
                d2[r] = *reinterpret_cast<const uint32_t *>((scales + 2 * g) + scale_at);
            }
        }
    }
    __device__ __forceinline__ void open() {}
    __device__ __forceinline__ int4v operand(int g, const uint32_t *) const { return int4v{(int)q[g].x, (int)q[g].y, (int)q[g].z, (int)q[g].w}; }
    __device__ __forceinline__ int4v min_operand(int) const { return int4v{0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int g) const { return half_bits((g & 1) ? d2[g >> 1] >> 16 : d2[g >> 1] & 0xffffu); }
    __device__ __forceinline__ float minimum(int) const { return 0.0f; }
};

template <bool ROWS> struct BatchRows<PF_MXFP4, ROWS> {   // in tile order or row by row: a lane reads its row's whole block and keeps the low or the high nibbles
    static constexpr int GROUPS = 8;
    static constexpr bool MINIMA = false, MIN_OPERAND = false;
    uint4 q[8];
    uint32_t e2[4];
    __device__ __forceinline__ void load(const PfKernelArgs &a, int t, size_t e, int tile, int piece, int groups, int lane, const uint32_t *) {
        const size_t row0 = e * (size_t)a.n_out[t] + (size_t)(32 * tile);
        const int units = groups / 4;
        const uint8_t *codes = ROWS ? a.w[t] + row0 * a.row_bytes[t] : a.wm + row0 / 32 * units * PF_I2T_CHUNK;
        const uint8_t *scales = a.w[t] + a.scale_offset[t] + row0 * (size_t)a.blocks_per_row[t];   // (ROWS)
        const uint32_t code_at = (uint32_t)(lane & 31) * (ROWS ? (uint32_t)a.row_bytes[t] : 16u);
        const uint32_t scale_at = (uint32_t)(lane & 31) * (ROWS ? (uint32_t)a.blocks_per_row[t] : 4u);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int g = min(GROUPS * piece + 2 * r, groups - 2);
            const uint8_t *unit = codes + (g >> 2) * PF_I2T_CHUNK;
#pragma unroll
            for (int i = 0; i < 2; i++)
                q[2 * r + i] = *reinterpret_cast<const uint4 *>((ROWS ? codes + 16 * (g + i) : unit + pf_mxt_piece_at((g & 3) + i, 0)) + code_at);
            e2[r] = *reinterpret_cast<const uint16_t *>((ROWS ? scales + g : unit + pf_mxt_scales_at(0) + (g & 3)) + scale_at);
        }
    }
    __device__ __forceinline__ void open() {}
    __device__ __forceinline__ int4v operand(int g, const uint32_t *) const {
        const int s = pf_lane() >= 32 ? 4 : 0;
        return int4v{e2m1_twice4(q[g].x >> s), e2m1_twice4(q[g].y >> s), e2m1_twice4(q[g].z >> s), e2m1_twice4(q[g].w >> s)};
    }
    __device__ __forceinline__ int4v min_operand(int) const { return int4v{0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int g) const { return 0.5f * pf_e8m0_scale((e2[g >> 1] >> (8 * (g & 1))) & 255u); }   // the integers are twice the values
    __device__ __forceinline__ float minimum(int) const { return 0.0f; }
};

// Q2_K: a lane's half of a group is one sub-group of 16, so its 4-bit scale goes into the codes (at most 45) and its 4-bit
// minimum is an operand of its own (the sum of the activations of a sub-group is a product with it).  ROWS: from memory, a
// dword of 32 rows at a time; else from the wave's copy of the whole tile in LDS (batch_stage_rows).
template <bool ROWS> struct BatchRows<PF_Q2_K, ROWS> {
    static constexpr int GROUPS = 8;
    static constexpr bool MINIMA = true, MIN_OPERAND = true;
    uint32_t q[8], sm[4], dd;
    float d, dmin;
    __device__ __forceinline__ void load(const PfKernelArgs &a, int t, size_t e, int tile, int piece, int, int lane, const uint32_t *stage) {
        const size_t row0 = e * (size_t)a.n_out[t] + (size_t)(32 * tile);
        const uint32_t at = (uint32_t)(lane & 31) * (uint32_t)(a.row_bytes[t] / 4), code_at = at + 4 + 4 * (uint32_t)(lane >> 5);
        auto take = [&](const uint32_t *blocks) {
#pragma unroll
            for (int i = 0; i < 4; i++) sm[i] = blocks[at + i];
#pragma unroll
            for (int i = 0; i < 8; i++) q[i] = blocks[code_at + 8 * (i >> 2) + (i & 3)];
            dd = blocks[at + 20];
        };
        if constexpr (!ROWS) take(stage + 21 * piece);
        else take(reinterpret_cast<const uint32_t *>(a.w[t] + row0 * a.row_bytes[t] + 84 * (size_t)piece));
    }
    __device__ __forceinline__ void open() { d = half_bits(dd & 0xffffu); dmin = half_bits(dd >> 16); }
    __device__ __forceinline__ uint32_t scale_min(int g) const {   // byte 2 g + h
        return (sm[g >> 1] >> (16 * (g & 1) + (pf_lane() >= 32 ? 8 : 0))) & 255u;
    }
    __device__ __forceinline__ int4v operand(int g, const uint32_t *) const {
        const unsigned short s = (unsigned short)(scale_min(g) & 15u);
        int4v out;
#pragma unroll
        for (int i = 0; i < 4; i++) {   // two codes of at most 3 per 16 bits: no carry between them
            const uint32_t codes = (q[4 * (g >> 2) + i] >> (2 * (g & 3))) & 0x03030303u;
            out[i] = __builtin_bit_cast(int, __builtin_bit_cast(ushort2v, codes) * ushort2v{s, s});
        }
        return out;
    }
    __device__ __forceinline__ int4v min_operand(int g) const {
        const uint32_t m = scale_min(g) >> 4;
        const int all = (int)__builtin_amdgcn_perm(m, m, 0u);
        return int4v{all, all, all, all};
    }
    __device__ __forceinline__ float scale(int) const { return d; }
    __device__ __forceinline__ float minimum(int) const { return dmin; }
};

// ---- a chunk's rows against a piece ------------------------------------------------------------------
struct BatchFactor { float step, sum; };   // a (token, group)'s step, and the sum of the group's integers

// A sum from its planes, in two parts of at most 28 bits: its value is 65536 upper + lower.
template <int PLANES> __device__ __forceinline__ float batch_upper(const int16v &d, int q) {
    return (float)(PLANES == 4 ? d[4 * q + 2] + (d[4 * q + 3] << 8) : d[4 * q + 2]);
}
__device__ __forceinline__ float batch_lower(const int16v &d, int q) { return (float)(d[4 * q] + (d[4 * q + 1] << 8)); }
template <int PLANES> __device__ __forceinline__ float batch_value(const int16v &d, int q) {
    return fmaf(65536.0f, batch_upper<PLANES>(d, q), batch_lower(d, q));
}

// acc[s][q] += the products of set s's piece with tokens 2 q + h of the chunk.  OWN: the piece is added up by itself first, as a chain's
// rounding grows with its length; in layers of one format (24 tokens 2.90 -> 2.72e-7 from 64 bits for IQ2_XXS, 3.16 -> 3.10 for Q4_K: no
// further than the decode kernels).  The profiles' kernels have no registers for it (101 tokens of the q2 profile 3 % slower).
template <int FMT, bool ROWS, int PLANES, int SETS, int QUADS, bool OWN>
__device__ __forceinline__ void batch_piece(const BatchRows<FMT, ROWS> (&w)[SETS], const int4v (&x)[BatchRows<FMT, ROWS>::GROUPS], const BatchFactor *factors,
                                            int here, const uint32_t *tables, float (&acc)[SETS][4]) {
    typedef BatchRows<FMT, ROWS> Rows;
    const int16v zero = {0};
    float own[SETS][4] = {};
    auto &part = *(OWN ? &own : &acc);
#pragma unroll
    for (int g = 0; g < Rows::GROUPS; g++) {
        if (g >= here) break;   // the ragged end of a row
        int16v d[SETS], m[SETS];
#pragma unroll
        for (int s = 0; s < SETS; s++) {
            d[s] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[g], w[s].operand(g, tables), zero, 0, 0, 0);
            if (Rows::MIN_OPERAND) m[s] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[g], w[s].min_operand(g), zero, 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < SETS; s++) {
            const float scale = w[s].scale(g), minimum = Rows::MINIMA ? w[s].minimum(g) : 0.0f;
#pragma unroll
            for (int q = 0; q < QUADS; q++) {
                const BatchFactor f = factors[16 * q + g];
                if (Rows::MIN_OPERAND && PLANES == 4) {   // the two products nearly cancel: their difference part by part, the upper one's with what its product lost
                    const float mu = batch_upper<PLANES>(m[s], q), product = minimum * mu;
                    const float upper = fmaf(scale, batch_upper<PLANES>(d[s], q), -product) - fmaf(minimum, mu, -product);
                    const float lower = fmaf(scale, batch_lower(d[s], q), -minimum * batch_lower(m[s], q));
                    part[s][q] = fmaf(f.step, fmaf(65536.0f, upper, lower), part[s][q]);
                } else if (Rows::MIN_OPERAND) {
                    part[s][q] = fmaf(f.step, fmaf(scale, batch_value<PLANES>(d[s], q), -minimum * batch_value<PLANES>(m[s], q)), part[s][q]);
                } else if (Rows::MINIMA) {
                    part[s][q] = fmaf(f.step, fmaf(scale, batch_value<PLANES>(d[s], q), -minimum * f.sum), part[s][q]);
                } else {
                    part[s][q] = fmaf(f.step * batch_value<PLANES>(d[s], q), scale, part[s][q]);
                }
            }
        }
    }
    if (!OWN) return;
#pragma unroll
    for (int s = 0; s < SETS; s++)
#pragma unroll
        for (int q = 0; q < QUADS; q++) acc[s][q] += own[s][q];
}

// The chunk's activation operands of a piece and the piece's factors into the wave's LDS (factors[8 * token + group]).
// at, factor_at: the dword offsets in `images` of the images of the lane's token (lane % 32) / 4, and lane / 8.  Groups
// beyond the row's last repeat it with a factor of zero.
template <int PLANES, int GROUPS>
__device__ __forceinline__ void batch_operands(int4v (&x)[GROUPS], BatchFactor *factors, const uint32_t *images, uint32_t at, uint32_t factor_at,
                                               int piece, int groups, int lane) {
    const uint32_t mine = at + 8 * (uint32_t)min(lane & 3, PLANES - 1) + 4 * (uint32_t)(lane >> 5);
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const uint32_t *group = images + 8 * PLANES * min(GROUPS * piece + g, groups - 1);   // uniform
        x[g] = *reinterpret_cast<const int4v *>(group + mine);
    }
    const int fg = GROUPS * piece + (lane & 7), last = min(fg, groups - 1);
    const float step = fg < groups ? __uint_as_float((images + 8 * PLANES * groups)[factor_at + (uint32_t)last]) : 0.0f;
    const float sum = fg < groups ? __uint_as_float((images + (8 * PLANES + 1) * groups)[factor_at + (uint32_t)last]) : 0.0f;
    pf_wave_lds_fence();   // the piece before has been read
    factors[lane] = BatchFactor{step, sum};
    pf_wave_lds_fence();
}

// The lane's index, not known to be the same from one chunk to the next: the addresses that depend on it are formed where
// they are used, as a uniform base and a 32-bit offset, instead of being kept as 64-bit pointers across the chunks (two
// registers a pointer, which spilled).
__device__ __forceinline__ int batch_lane() {
    int lane = pf_lane();
    asm volatile("" : "+v"(lane));
    return lane;
}

// image_at(r): dword offset in `images` of the image of the chunk's row r
template <int FMT, bool ROWS, int PLANES, bool OWN, int SETS, typename ImageAt>
__device__ __forceinline__ void batch_chunk(const PfKernelArgs &a, const int (&tensor)[SETS], size_t e, int tile, int first_piece, int piece_step,
                                            int groups, const uint32_t *images, ImageAt image_at, BatchFactor *factors, int rows,
                                            const uint32_t *tables, float (&acc)[SETS][4], const uint32_t *stage = nullptr) {
    typedef BatchRows<FMT, ROWS> Rows;
    const int pieces = (groups + Rows::GROUPS - 1) / Rows::GROUPS;
    if (first_piece >= pieces) return;
    Rows w[SETS];
    uint32_t at, factor_at;
    {
        const int lane = batch_lane();
#pragma unroll
        for (int s = 0; s < SETS; s++) w[s].load(a, tensor[s], e, tile, first_piece, groups, lane, stage);   // on their way while the rows are looked up
        at = image_at(min((lane & 31) >> 2, rows - 1));
        factor_at = image_at(min(lane >> 3, rows - 1));
    }
    for (int piece = first_piece; piece < pieces; piece += piece_step) {
        const int lane = batch_lane();
        int4v x[Rows::GROUPS];
        batch_operands<PLANES, Rows::GROUPS>(x, factors, images, at, factor_at, piece, groups, lane);
#pragma unroll
        for (int s = 0; s < SETS; s++) w[s].open();
        const BatchFactor *mine = factors + 8 * (lane >> 5);
        const int here = groups - Rows::GROUPS * piece;
        if (rows <= 2) batch_piece<FMT, ROWS, PLANES, SETS, 1, OWN>(w, x, mine, here, tables, acc);
        else if (rows <= 4) batch_piece<FMT, ROWS, PLANES, SETS, 2, OWN>(w, x, mine, here, tables, acc);
        else batch_piece<FMT, ROWS, PLANES, SETS, 4, OWN>(w, x, mine, here, tables, acc);
        if (piece + piece_step < pieces) {
            const int lane = batch_lane();
#pragma unroll
            for (int s = 0; s < SETS; s++) w[s].load(a, tensor[s], e, tile, piece + piece_step, groups, lane, stage);
        }
    }
}

// ---- work items ------------------------------------------------------------------------------------
struct BatchItem {
    bool shared;
    int first, rows;      // the item's rows (expert order; the shared expert's rows follow the pairs)
    int token0;           // shared expert: the first row's token
    size_t e;             // where the expert's weights are: its id, or its pool slot
};
// Number q of a launch.  The shared expert's rows, the list's last items, are a chunk of eight a number: `shared` numbers.  They come
// first, unless `last` is set: then the routed tiles do, the longest at the head of the list (batch_shared_last).  (As row tiles, four chunks
// one after the other, at the list's end they were a launch's end: 101 tokens of the q2 profile 283 us a forward, first 248; for a layer
// of few experts they were as long as all else.)  False: no such item.
__device__ __forceinline__ bool batch_item(const PfKernelArgs &a, uint32_t q, uint32_t shared, bool last, BatchItem &it) {
    const uint32_t count = a.tiles[0], routed = count - (shared + 3) / 4;
    if (q >= shared + routed) return false;
    const uint32_t own = last ? q - routed : q;   // its number among the shared expert's, if it is one
    it.shared = last ? q >= routed : q < shared;
    const uint4 entry = reinterpret_cast<const uint4 *>(a.items)[it.shared ? routed + own / 4 : last ? q : q - shared];   // {expert, first row, rows, first row within the expert}
    const int chunk = it.shared ? BATCH_ROWS * (int)(own % 4) : 0;
    const int expert = (int)entry.x;
    it.first = (int)entry.y + chunk;
    it.rows = it.shared ? min(BATCH_ROWS, (int)entry.z - chunk) : (int)entry.z;
    it.token0 = (int)entry.w + chunk;
    it.e = it.shared ? 0 : (size_t)expert;
    if (a.slots && !it.shared) {   // expert streaming: the rows of an expert share its pool slot
        uint32_t slot = a.slots[a.row_to_pair[it.first]];
        if (slot >= a.pool_slots) {
            if (threadIdx.x == 0) atomicOr(a.error_word, PF_HIP_ERR_BOUNDS);
            slot = 0;
        }
        it.e = slot;
    }
    return true;
}

template <int FMT> __host__ __device__ constexpr bool batch_tables() { return FMT == PF_IQ2_XXS; }
#define BATCH_TABLE_BYTES 3072
__device__ __forceinline__ void batch_stage_tables(uint32_t *tables, const PfKernelArgs &a) {
    for (int i = (int)threadIdx.x; i < 256; i += (int)blockDim.x) reinterpret_cast<uint64_t *>(tables)[i] = a.iq2_grid[i];
    for (int i = (int)threadIdx.x; i < 128; i += (int)blockDim.x) {
        const uint32_t bits = (uint32_t)i | (pf_parity7((uint32_t)i) << 7);   // the eighth sign: the others' parity
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo |= ((bits >> j) & 1u ? 255u : 0u) << (8 * j);
            hi |= ((bits >> (4 + j)) & 1u ? 255u : 0u) << (8 * j);
        }
        reinterpret_cast<uint2 *>(tables)[256 + i] = make_uint2(lo, hi);
    }
    __syncthreads();
}

// A group's step and its inverse.  Four planes: the power of two that puts the largest magnitude m between 2^29 and 2^30, or the
// smallest normal one.
template <int PLANES> __device__ __forceinline__ void batch_step(float m, float &step, float &inv) {
    if constexpr (PLANES == 3) {
        group_step2(m, step, inv);
    } else {
        const int exponent = max((int)(__float_as_uint(m) >> 23) - 29, 1);
        step = __uint_as_float((uint32_t)exponent << 23);
        inv = __uint_as_float((uint32_t)(254 - exponent) << 23);
    }
}
// What a vector's group ends with: the step, and the sum of its integers (at most 36 bits, from the sums of their upper and
// lower 16 bits); WHOLE: as the decode kernels keep it, three planes' 29 bits as an integer.
template <int PLANES, bool WHOLE = false> __device__ __forceinline__ void batch_image_end(uint32_t *img, int g, int K, float step, int upper, int lower) {
    img[8 * PLANES * (K / 32) + g] = __float_as_uint(step);
    img[(8 * PLANES + 1) * (K / 32) + g] = WHOLE ? (uint32_t)(65536 * upper + lower) : __float_as_uint(fmaf(65536.0f, (float)upper, (float)lower));
}

// Thread j of a group of four neighbouring lanes: the eight values 8j..8j+7 of a K-vector into its image.
template <int PLANES, bool WHOLE> __device__ __forceinline__ void batch_image_chunk(uint32_t *img, const float (&v)[8], int j, int K) {
    float m = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; c++) m = fmaxf(m, fabsf(v[c]));
    m = fmaxf(m, __int_as_float(dpp_quad_xor1(__float_as_int(m))));
    m = fmaxf(m, __int_as_float(dpp_quad_xor2(__float_as_int(m))));
    float step, inv;
    batch_step<PLANES>(m, step, inv);
    uint32_t w[PLANES][2] = {};
    int upper = 0, lower = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int q = __float2int_rn(v[c] * inv);
        upper += q >> 16;
        lower += q & 0xffff;
        int d[PLANES];
        image_digits(q, d);
#pragma unroll
        for (int p = 0; p < PLANES; p++) w[p][c >> 2] |= (uint32_t)(d[p] & 255) << (8 * (c & 3));
    }
    upper += dpp_quad_xor1(upper); upper += dpp_quad_xor2(upper);
    lower += dpp_quad_xor1(lower); lower += dpp_quad_xor2(lower);
    const int g = j >> 2, at = 8 * PLANES * g + 2 * (j & 3);
#pragma unroll
    for (int p = 0; p < PLANES; p++) { img[at + 8 * p] = w[p][0]; img[at + 8 * p + 1] = w[p][1]; }
    if ((j & 3) == 0) batch_image_end<PLANES, WHOLE>(img, g, K, step, upper, lower);
}

// Lanes 0..31 and 32..63, one value each: group g of two K-vectors' images (store: whether the lane's vector exists).
template <int PLANES> __device__ __forceinline__ void batch_image_group(uint32_t *img, float v, int g, int K, int lane, bool store) {
    float m = fabsf(v);
#pragma unroll
    for (int k = 0; k < 4; k++) m = fmaxf(m, __int_as_float(dpp_row_step(__float_as_int(m), k)));
    m = fmaxf(m, __shfl_xor(m, 16));
    float step, inv;
    batch_step<PLANES>(m, step, inv);
    const int q = __float2int_rn(v * inv);
    int upper = q >> 16, lower = q & 0xffff;
#pragma unroll
    for (int k = 0; k < 4; k++) { upper += dpp_row_step(upper, k); lower += dpp_row_step(lower, k); }
    upper += __shfl_xor(upper, 16);
    lower += __shfl_xor(lower, 16);
    int d[PLANES];
    image_digits(q, d);
    if (!store) return;
    uint8_t *bytes = reinterpret_cast<uint8_t *>(img + 8 * PLANES * g);
#pragma unroll
    for (int p = 0; p < PLANES; p++) bytes[32 * p + (lane & 31)] = (uint8_t)d[p];
    if ((lane & 31) == 0) batch_image_end<PLANES>(img, g, K, step, upper, lower);
}

// blockIdx.x: 32 units; blockIdx.y: row tile.  The workgroup's waves share K (a 256-block each, in turn); their partial
// sums meet in LDS and are added in wave order, a wave per pair of rows.
// Bound by the chain a workgroup lives through (item, weights, products, the same for a second 256-block, sums): three
// workgroups a compute unit keep 120 KB on their way, 3.9 TB/s of weights at 32 tokens (72 us for 283 MB).  IQ2_XXS, whose
// table look-ups lengthen the chain and whose weights are half the bytes, is held to the registers of four workgroups a compute
// unit: 101 tokens of the q2 profile 178 -> 163 us, 24 tokens 82 -> 74; Q4_K spills at that (175 -> 199 us).  With the weights
// read from a cache the two take 138 and 124 us of these: the products' chain, not the memory, is the longer part.  Measured and left out: eight waves with a block each,
// five waves for rows of ten blocks (1.4 times slower: every workgroup's fifth wave meets the same SIMD), two
// waves with four (slower), the next block's weights asked for before the products (no gain, the rows' operands wait behind
// them), the operands past the registers through LDS (slower: LDS becomes the bottleneck for
// IQ2_XXS), one matrix a wave at twice the occupancy (85 us).
#define BATCH_WAVES 4
// float_rows: the routed experts' activation rows leave the kernel as FP32 (they become digit rows for pf_k_mx_down), else as images.
template <int FMT, int FMTS, bool ROWS, int PLANES>
__global__ void __launch_bounds__(64 * BATCH_WAVES) __attribute__((amdgpu_waves_per_eu(FMT == PF_IQ2_XXS ? 4 : 3))) pf_k_batch_gate_up(PfKernelArgs a, uint32_t shared_items, int shared_last, int float_rows) {
    __shared__ float partial[BATCH_WAVES][2][4][64];
    __shared__ BatchFactor factors[BATCH_WAVES][64];
    __shared__ __align__(16) uint32_t tables[batch_tables<FMT>() ? BATCH_TABLE_BYTES / 4 : 4];
    BatchItem it;
    if (!batch_item(a, blockIdx.y, shared_items, shared_last != 0, it)) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int tile = blockIdx.x, I = it.shared ? a.shared_inter : a.inter;
    if (32 * tile >= I) return;
    if (batch_tables<FMT>()) batch_stage_tables(tables, a);
    const int groups = a.hidden / 32, K = a.top_k;
    const uint32_t words = (uint32_t)pf_batch_image_words(PLANES, a.hidden);
    const size_t act_words = pf_batch_image_words(PLANES, a.inter > a.shared_inter ? a.inter : a.shared_inter);
    const bool rows_only = float_rows && !it.shared;
    for (int c0 = 0; c0 < it.rows; c0 += BATCH_ROWS) {
        const int rows = min(BATCH_ROWS, it.rows - c0);
        float acc[2][4] = {};
        const int tensor[2] = {it.shared ? 4 : 1, it.shared ? 5 : 2};
        auto image_at = [&](int r) {
            const uint32_t row = (uint32_t)(c0 + r);
            return (it.shared ? (uint32_t)it.token0 + row : a.row_to_pair[(uint32_t)it.first + row] / (uint32_t)K) * words;
        };
        if (FMT != FMTS && it.shared) batch_chunk<FMTS, ROWS, PLANES, false>(a, tensor, 0, tile, wave, BATCH_WAVES, groups, a.ximg, image_at, factors[wave], rows, tables, acc);
        else batch_chunk<FMT, ROWS, PLANES, FMT == FMTS>(a, tensor, it.e, tile, wave, BATCH_WAVES, groups, a.ximg, image_at, factors[wave], rows, tables, acc);
        const int lane = batch_lane();
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (2 * q < rows) {
                partial[wave][0][q][lane] = acc[0][q];
                partial[wave][1][q][lane] = acc[1][q];
            }
        __syncthreads();
        for (int q = wave; 2 * q < rows; q += BATCH_WAVES) {
            const int lane = batch_lane();
            float gate = 0.0f, up = 0.0f;
            for (int w = 0; w < BATCH_WAVES; w++) {
                gate += partial[w][0][q][lane];
                up += partial[w][1][q][lane];
            }
            const float act = pf_silu(gate) * up;
            const int r = 2 * q + (lane >> 5);
            if (r < rows && !pf_finite(act)) atomicOr(a.error_word, PF_HIP_ERR_NONFINITE);
            const size_t row = (size_t)(it.first + c0 + min(r, rows - 1));
            if (rows_only) {
                if (r < rows) a.act[row * I + 32 * tile + (lane & 31)] = act;
            } else {
                batch_image_group<PLANES>(a.aimg + row * act_words, act, tile, I, lane, r < rows);
            }
        }
        if (c0 + BATCH_ROWS < it.rows) __syncthreads();   // the sums have been read
    }
}

// A tile of Q2_K rows of at most BATCH_STAGE_BYTES into the wave's LDS, as it lies in memory.  A row's blocks are 84 bytes, so
// lanes that read the same dword of 32 rows touch a line each, 64 accesses for 128 bytes: at 101 tokens of the checkpoints'
// width the kernel stood at 1.9 TB/s (138 us).  The tile is one run of bytes, asked for at once, and in LDS rows of an odd
// number of dwords meet no bank twice: 104 us (24 tokens 67 -> 53).  Rows of more than three blocks stay on the loads by row.
#define BATCH_STAGE_BYTES (32 * 3 * 84)
__device__ __forceinline__ void batch_stage_rows(uint32_t *stage, const PfKernelArgs &a, int t, size_t e, int tile) {
    const uint32_t bytes = 32 * (uint32_t)a.row_bytes[t];
    const PfBuffer rows = pf_buffer(a.w[t] + (e * (size_t)a.n_out[t] + (size_t)(32 * tile)) * a.row_bytes[t], bytes);
#pragma unroll
    for (int i = 0; i < (BATCH_STAGE_BYTES + 1023) / 1024; i++)   // beyond the tile: zeros, without an access
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_byte *)stage + 1024 * i, 16, 1024 * i + 16 * pf_lane(), 0, 0, 0);
}

// blockIdx.x: 128 output rows, a 32-row tile a wave; blockIdx.y: row tile of the expert.  Bound by the products' chain of a wave
// (with the weights in a cache 90 us of 104 for Q2_K, 101 tokens).
template <int FMT, int FMTS, bool ROWS, int PLANES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) pf_k_batch_down(PfKernelArgs a, uint32_t shared_items, int shared_last) {
    constexpr bool STAGED = FMT == PF_Q2_K && !ROWS;
    __shared__ BatchFactor factors[4][64];
    __shared__ __align__(16) uint32_t tables[batch_tables<FMT>() ? BATCH_TABLE_BYTES / 4 : 4];
    __shared__ __align__(16) uint32_t staged[STAGED ? 4 : 1][STAGED ? 2048 : 4];
    BatchItem it;
    if (!batch_item(a, blockIdx.y, shared_items, shared_last != 0, it)) return;
    if (batch_tables<FMT>()) batch_stage_tables(tables, a);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), H = a.hidden;
    const int tile = 4 * blockIdx.x + wave;
    if (32 * tile >= H) return;
    const int groups = (it.shared ? a.shared_inter : a.inter) / 32;
    const uint32_t words = (uint32_t)pf_batch_image_words(PLANES, a.inter > a.shared_inter ? a.inter : a.shared_inter);
    uint32_t *stage = staged[STAGED ? wave : 0];
    if (STAGED && !it.shared) {
        batch_stage_rows(stage, a, 3, it.e, tile);
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the wave's own copy is there
        pf_wave_lds_fence();
    }
    for (int c0 = 0; c0 < it.rows; c0 += BATCH_ROWS) {
        const int rows = min(BATCH_ROWS, it.rows - c0);
        auto image_at = [&](int r) { return (uint32_t)(it.first + c0 + r) * words; };
        float acc[1][4] = {};
        const int tensor[1] = {it.shared ? 6 : 3};
        if (FMT != FMTS && it.shared) batch_chunk<FMTS, ROWS || FMTS == PF_Q8_0, PLANES, false>(a, tensor, 0, tile, 0, 1, groups, a.aimg, image_at, factors[wave], rows, tables, acc);
        else batch_chunk<FMT, ROWS, PLANES, FMT == FMTS>(a, tensor, it.e, tile, 0, 1, groups, a.aimg, image_at, factors[wave], rows, tables, acc, stage);
        const int lane = batch_lane();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = 2 * q + (lane >> 5);
            if (r < rows) a.down[(size_t)(it.first + c0 + r) * H + 32 * tile + (lane & 31)] = acc[0][q];
        }
    }
}

// ---- router ----------------------------------------------------------------------------------------
// Logits and sums of squared products of 16 tokens against 16 experts a workgroup, on v_mfma_f32_16x16x4_f32; sixteen waves
// share the columns.  The whole of a wave's part (at most ROUTER_LINES 128-byte lines of 16 + 16 rows) is requested at once:
// a workgroup waits for memory once, and small tiles spread a few tokens over the chip (a 32 x 32 tile keeps a compute
// unit's matrix cores busy for 7 us, this one for 2 + 2).  A line goes through the wave's own LDS because a product step
// wants element k of row i from lane (i, k).  The sums of squares (the routing's tolerance) are products of the squares.
// A logit is summed in four chains a wave and in pairs over the waves: the routes' share of the block's error is then what
// the other routers' is (8e-8 of the result, 14e-8 with one chain).
// The last row of workgroups takes a token a wave: its digit image, and the shared router's logit and sigmoid.
// Measured at a width of 2560: 101 tokens 37 -> 12.7 us, against the decode kernels' router in groups of four tokens (32
// tokens of width 2048: 14.0 -> 9.6).
typedef float float4v __attribute__((ext_vector_type(4)));
#define ROUTER_LINES 5      // 32-column lines a wave holds: hidden <= 2560
#define ROUTER_PITCH 36     // floats between rows of a staged line: neighbouring lanes' 16-byte reads cover all banks
template <int PLANES, bool WHOLE>   // WHOLE: the decode kernels' images
__global__ void __launch_bounds__(1024) pf_k_batch_router(PfKernelArgs a, int tokens) {
    __shared__ __align__(16) float staged[16][2][16 * ROUTER_PITCH];
    const int H = a.hidden, E = a.experts, lane = pf_lane(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (blockIdx.y == gridDim.y - 1) {
        const int t = 16 * blockIdx.x + wave;
        if (t >= tokens) return;
        const float4v *row = reinterpret_cast<const float4v *>(a.x + (size_t)t * a.x_pitch), *gate = reinterpret_cast<const float4v *>(a.w[7]);
        float4v zp = {0}, zq = {0};   // eight chains, as above
        for (int j = lane; j < H / 8; j += 64) {
            const float4v p = row[2 * j], q = row[2 * j + 1], u = gate[2 * j], v = gate[2 * j + 1];
            const float both[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
            batch_image_chunk<PLANES, WHOLE>(a.ximg + (size_t)t * pf_batch_image_words(PLANES, H), both, j, H);
#pragma unroll
            for (int c = 0; c < 4; c++) { zp[c] = fmaf(p[c], u[c], zp[c]); zq[c] = fmaf(q[c], v[c], zq[c]); }
        }
        zp += zq;
        const float z = pf_wave_sum((zp.x + zp.y) + (zp.z + zp.w));
        if (lane == 0) {
            a.shared_scale[t] = pf_sigmoid(z);
            if (!pf_finite(z)) atomicOr(a.error_word, PF_HIP_ERR_NONFINITE);
        }
        return;
    }
    const int t0 = 16 * blockIdx.x, e0 = 16 * blockIdx.y, lines = H / 32, l0 = lines * wave / 16, l1 = lines * (wave + 1) / 16;
    const int lr = lane >> 3, piece = lane & 7, i = lane & 15, kk = lane >> 4;
    float4v xg[ROUTER_LINES][2], wg[ROUTER_LINES][2];
#pragma unroll
    for (int l = 0; l < ROUTER_LINES; l++) {
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const int t = min(t0 + 8 * g + lr, tokens - 1), e = min(e0 + 8 * g + lr, E - 1);
            if (l0 + l < l1) {
                xg[l][g] = reinterpret_cast<const float4v *>(a.x + (size_t)t * a.x_pitch)[8 * (l0 + l) + piece];
                wg[l][g] = reinterpret_cast<const float4v *>(a.w[0] + (size_t)e * H * 4)[8 * (l0 + l) + piece];
            }
        }
    }
    float *xs = staged[wave][0], *ws = staged[wave][1];
    float4v part[4] = {}, sq = {0};   // four chains of the logits' sums: a chain's rounding grows with its length
#pragma unroll
    for (int l = 0; l < ROUTER_LINES; l++) {
        if (l0 + l >= l1) break;
        pf_wave_lds_fence();
#pragma unroll
        for (int g = 0; g < 2; g++) {
            *reinterpret_cast<float4v *>(xs + (8 * g + lr) * ROUTER_PITCH + 4 * piece) = xg[l][g];
            *reinterpret_cast<float4v *>(ws + (8 * g + lr) * ROUTER_PITCH + 4 * piece) = wg[l][g];
        }
        pf_wave_lds_fence();
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float4v x = *reinterpret_cast<const float4v *>(xs + i * ROUTER_PITCH + 16 * c + 4 * kk);
            const float4v w = *reinterpret_cast<const float4v *>(ws + i * ROUTER_PITCH + 16 * c + 4 * kk);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                part[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[k], w[k], part[k], 0, 0, 0);
                sq = __builtin_amdgcn_mfma_f32_16x16x4f32(x[k] * x[k], w[k] * w[k], sq, 0, 0, 0);
            }
        }
    }
    const float4v acc = (part[0] + part[1]) + (part[2] + part[3]);
    pf_wave_lds_fence();
#pragma unroll
    for (int r = 0; r < 4; r++) { xs[64 * r + lane] = acc[r]; xs[64 * (4 + r) + lane] = sq[r]; }   // the wave's own part of LDS: 512 floats
    __syncthreads();
    if (wave >= 8) return;
    float sums[16];   // register `wave` of every wave, added in pairs
#pragma unroll
    for (int w = 0; w < 16; w++) sums[w] = staged[w][0][64 * wave + lane];
#pragma unroll
    for (int n = 8; n; n /= 2)
#pragma unroll
        for (int w = 0; w < n; w++) sums[w] = sums[2 * w] + sums[2 * w + 1];
    const float sum = sums[0];
    const int t = t0 + 4 * kk + (wave & 3), e = e0 + i;
    if (t < tokens && e < E) {
        if (wave < 4) {
            a.logits[(size_t)t * E + e] = sum;
            // a nonfinite activation makes every product with it nonfinite, and a sum with such a term stays so
            if (!pf_finite(sum)) atomicOr(a.error_word, PF_HIP_ERR_NONFINITE);
        } else {
            // the squares of finite values beyond 1.8e19 are infinite (times a zero: NaN) where the logit is finite: a
            // tolerance without bound, so that the token is routed in serial order
            a.logit_ssq[(size_t)t * E + e] = pf_finite(sum) ? sum : INFINITY;
        }
    }
}

bool pf_batch_router_takes(int hidden) { return hidden % 32 == 0 && hidden <= 16 * 32 * ROUTER_LINES; }
void pf_launch_batch_router(const PfKernelArgs &a, int tokens, int planes, bool whole, hipStream_t stream) {
    const dim3 grid((tokens + 15) / 16, (a.experts + 15) / 16 + 1);
    auto *const kernel = whole ? pf_k_batch_router<3, true> : planes == 4 ? pf_k_batch_router<4, false> : pf_k_batch_router<3, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(1024), 0, stream, a, tokens);
}

// ---- dispatch --------------------------------------------------------------------------------------
// Where the shared expert's chunks come in the launches.  A routed tile is up to four chunks one after the other: with more than about three
// chunks an expert on average the routed tiles are the long items and start first, else the shared expert's, whose rows are all there
// are and, in a profile, the wider format.  Forwards, shared first : last, us: 350 tokens of 8 experts, two slots, 2048 x 512, Q4_K 93.8 : 80.3, the
// q2 profile 113.3 : 90.2, 250 tokens of 16 experts, four slots, 94.4 : 85.5, of 32 96.2 : 88.9; 64 tokens of 64 experts, eight slots 63.5 : 65.5, 40
// of 8, 1024 x 256, 34.3 : 37.8, 130 of 128, eight, 46.5 : 48.7.  Of 504 batches of 8 to 512 experts none is more than 2.5 % slower than in the
// other order from this line on, and 6 % before it (32 experts beside a shared expert twice as wide).
static bool batch_shared_last(int tokens, int experts, int top_k) { return (size_t)tokens * top_k >= (size_t)24 * experts; }
template <int FG, int FD, int FS, bool ROWS, int PLANES>
static void launch_batch_format(const PfKernelArgs &a, int tokens, unsigned routed_cap, hipStream_t stream, int last) {
    const int widest = a.inter > a.shared_inter ? a.inter : a.shared_inter;
    // The q4 profile's routed down projection on the block-scaled product, as a chunk's, where the work is taken to be worth its launches
    // (pf_batch_down_scaled, with both sides measured): 101 tokens of the checkpoints' widths 307 us a forward on the integers, 283 there.
    const bool scaled = FD == PF_MXFP4 && PLANES == 3 && a.wm && pf_batch_down_scaled(tokens, a.experts, a.top_k, a.hidden, a.inter, a.shared_inter);
    const unsigned shared = (unsigned)(tokens + BATCH_ROWS - 1) / BATCH_ROWS;
    const int last_shared = batch_shared_last(tokens, a.experts, a.top_k) ? 1 : 0;
    hipLaunchKernelGGL((pf_k_batch_gate_up<FG, FS, ROWS, PLANES>), dim3(widest / 32, shared + routed_cap), dim3(64 * BATCH_WAVES), 0, stream, a, shared, last_shared, scaled ? 1 : 0);
    if (last < 4) return;
    const dim3 grid((a.hidden + 127) / 128, shared + routed_cap);
    if (scaled) {
        pf_launch_rows_to_digits(a.act, a.inter, (size_t)tokens * a.top_k, reinterpret_cast<uint32_t *>(a.act16), a.act_scale, a.error_word, stream);
        pf_launch_mx_down(a, tokens, routed_cap, stream);
        hipLaunchKernelGGL((pf_k_batch_down<FD, FS, FD != FG || ROWS, PLANES>), dim3(grid.x, shared), dim3(256), 0, stream, a, shared, 0);   // the shared expert's numbers alone
        return;
    }
    // down rows: as gate and up where the layer has one format; Q2_K by whole tiles where they fit a wave's LDS, MXFP4 in tile order
    // where the layer keeps that
    constexpr bool either = FD == PF_Q2_K || (FD == PF_MXFP4 && PLANES == 3);
    const bool lines = FD == PF_Q2_K ? 32 * a.row_bytes[3] <= BATCH_STAGE_BYTES : a.wm != nullptr;
    if (either && lines) hipLaunchKernelGGL((pf_k_batch_down<FD, FS, either ? false : FD != FG || ROWS, PLANES>), grid, dim3(256), 0, stream, a, shared, last_shared);
    else hipLaunchKernelGGL((pf_k_batch_down<FD, FS, FD != FG || ROWS, PLANES>), grid, dim3(256), 0, stream, a, shared, last_shared);
}

template <int FG, int FD, int FS>
static void launch_batch_experts(const PfKernelArgs &a, int tokens, unsigned routed_cap, hipStream_t stream, int last) {
    // a layer keeps the tile-ordered copies of its gate and up tensors (and a one-format layer those of its down tensors,
    // the profiles those of the shared gate and up) or none of them; a streamed layer's pool keeps its slots that way
    const bool tiled = (FG == PF_Q4_K ? a.wt[1] && a.wt[2] : a.wi[1] && a.wi[2]) && (FS != PF_Q8_0 || (a.wq[4] && a.wq[5]));
    if (a.slots) launch_batch_format<FG, FD, FS, false, 4>(a, tokens, routed_cap, stream, last);
    else if (tiled) launch_batch_format<FG, FD, FS, false, 3>(a, tokens, routed_cap, stream, last);
    else launch_batch_format<FG, FD, FS, true, 3>(a, tokens, routed_cap, stream, last);
}

void pf_launch_batch_experts(const PfKernelArgs &a, int tokens, hipStream_t stream, int last) {
    // row tiles there can be: an expert with rows has at least one
    const unsigned pairs = (unsigned)(tokens * a.top_k), most = (unsigned)(pf_prefill_max_tiles(tokens, a.experts, a.top_k) - (tokens + 31) / 32), cap = min(pairs, most);
    switch (a.type[1] == PF_Q4_K ? (a.type[3] == PF_Q4_K ? 1 : 4) : (a.type[3] == PF_IQ2_XXS ? 2 : 3)) {
    case 1: launch_batch_experts<PF_Q4_K, PF_Q4_K, PF_Q4_K>(a, tokens, cap, stream, last); break;
    case 2: launch_batch_experts<PF_IQ2_XXS, PF_IQ2_XXS, PF_IQ2_XXS>(a, tokens, cap, stream, last); break;
    case 3: launch_batch_experts<PF_IQ2_XXS, PF_Q2_K, PF_Q8_0>(a, tokens, cap, stream, last); break;
    default: launch_batch_experts<PF_Q4_K, PF_MXFP4, PF_Q8_0>(a, tokens, cap, stream, last); break;
    }
}

void pf_launch_batch(const PfKernelArgs &a, int tokens, hipStream_t stream, int stage_limit) {
    const int last = stage_limit ? stage_limit : 4;
    pf_launch_batch_router(a, tokens, 3, false, stream);
    if (last < 2) return;
    pf_launch_dec_route(a, tokens, stream);
    pf_launch_group(a, a.ids, tokens, stream);
    if (last < 3) return;
    pf_launch_batch_experts(a, tokens, stream, last);
    if (last < 4) return;
    pf_launch_combine(a, tokens, stream);
}
