// The MXFP4 down projection of a chunk on the block-scaled matrix instruction.
//
// v_mfma_scale_f32_32x32x64_f8f6f4 takes four-bit floats with an exponent byte per 32 values: MXFP4 as the file stores it.  The
// weights need no vector instruction at all; the activations are five planes of six-bit floats (pf_mx_rows.h), whose products
// with a weight are exact, and the hardware's sums are FP32 (within 2^-23 of the sum of the magnitudes, measured against 64 bits).  Five
// products of 32 cycles for 64 columns, where the two-part halfs take eight and the codes' conversion about as long again.
//
// Workgroup = one 32-row tile of an expert against `per` slabs of 256 output rows.  The tile's digit rows stay in LDS (4 K bytes a
// row: two workgroups a compute unit up to K = 640), so the waves need no barrier after the first: each goes over 64 output rows
// at a time, the next 64 rows' bytes on their way into the registers that the products have just left.
//
//   LDS   [group of 32 columns][eight rows][16-byte chunk of the group's line][row][16 bytes]; odd eights have their chunks in
//         pairs the other way round, so that neighbouring eights' reads fall on different banks
//
// Bound by memory: 2048 tokens of a layer of the checkpoints' widths (512 experts, 20480 rows of 640 against 2560 output rows) read
// 446 MB of weights and 58 MB of digit rows and write 210 MB in 155 us; the products keep the matrix cores busy for 52.  From
// the weights as the file orders their rows (16 bytes a lane, every lane another row) it took 204, bound by the address unit; the
// plain grouped product 300.  The rows' conversion takes 33 us instead of 21 for halfs.
#include "pf_grouped.h"
#include "pf_mx_rows.h"
#include "pf_upload_addr.h"

template <int UNITS>   // of 128 columns
__global__ void __launch_bounds__(256, 2) pf_k_mx_down(PfKernelArgs a, int slabs, int per, int shift, uint32_t shared_tiles) {
    extern __shared__ __align__(16) unsigned char mx_lds[];
    lds_byte *lds = (lds_byte *)mx_lds;
    GemmItem g;
    int slab;
    if (!gemm_item(a, slabs, shift, blockIdx.x, a.tiles[0] - shared_tiles, 0, 0, g, slab)) return;   // the routed tiles, ahead of the shared expert's
    constexpr int K = 128 * UNITS;
    const int lane = pf_lane(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, h = lane >> 5;
    const int slab1 = min((slab + 1) * per, a.hidden / 256);
    // weights in tile order: lane (n, h) takes block 2 s + h of row n of a tile in step s of a unit
    const uint32_t bytes = (uint32_t)pf_mxt_expert_bytes(a.n_out[3], UNITS);
    const uint8_t *tensor = a.wm + (size_t)g.expert * bytes;
    PfBuffer weights = pf_buffer(tensor, bytes);
    uint4v w[2][UNITS][2];
    uint32_t scale[2][UNITS];
    auto request = [&](int k, int pair) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t chunk = (uint32_t)((2 * pair + t) * UNITS + k) * PF_I2T_CHUNK;
            scale[t][k] = __builtin_amdgcn_raw_buffer_load_b32(weights, 4 * n, (int)(chunk + 2048), 0);
#pragma unroll
            for (int s = 0; s < 2; s++) w[t][k][s] = __builtin_amdgcn_raw_buffer_load_b128(weights, 16 * lane, (int)(chunk + 1024 * s), 0);
        }
    };
    int pair = 4 * slab * per + wave;
#pragma unroll
    for (int k = 0; k < UNITS; k++) request(k, pair);
    // the tile's digit rows: instruction i copies one group of eight rows; rows beyond the tile's last are zeros
    const PfBuffer source = pf_buffer(reinterpret_cast<const uint8_t *>(a.act16) + (size_t)g.first * 4 * K, (uint32_t)g.rows_here * 4 * K);
#pragma unroll
    for (int i = 0; i < UNITS; i++)
#pragma unroll
        for (int eight = 0; eight < 4; eight++) {
            const int group = 4 * i + wave;
            const uint32_t at = (uint32_t)(8 * eight + (lane & 7)) * 4 * K + 16u * (uint32_t)((lane >> 3) ^ (eight & 1));
            __builtin_amdgcn_raw_ptr_buffer_load_lds(source, lds + (4 * group + eight) * 1024, 16, (int)at, PF_MX_LINE * group, 0, 0);
        }
    const float scale_mine = a.act_scale[g.first + min(n, g.rows_here - 1)];
    lds_barrier<0>();
    const int odd = (n >> 3) & 1;
    const lds_byte *even = lds + (n >> 3) * 1024 + h * 4096 + (n & 7) * 16 + 128 * odd, *uneven = even - 256 * odd;   // of even and odd chunks
    auto chunk = [&](int c, int step) -> const lds_byte * { return ((c & 1) ? uneven : even) + 8192 * step + 128 * c; };
    struct Operand { int8v plane[PF_MX_PLANES]; uint32_t scale[2]; };
    auto take = [&](int step) -> Operand {
        Operand o;
#pragma unroll
        for (int p = 0; p < PF_MX_PLANES; p++) {
            const uint4v first = *reinterpret_cast<const __attribute__((address_space(3))) uint4v *>(chunk(p, step));
            const uint2v rest = *reinterpret_cast<const __attribute__((address_space(3))) uint2v *>(chunk(PF_MX_PLANES + p / 2, step) + 8 * (p & 1));
            o.plane[p] = int8v{(int)first.x, (int)first.y, (int)first.z, (int)first.w, (int)rest.x, (int)rest.y, 0, 0};
        }
        const uint2v s = *reinterpret_cast<const __attribute__((address_space(3))) uint2v *>(chunk(7, step) + 8);
        o.scale[0] = s.x; o.scale[1] = s.y;
        return o;
    };
    for (int s0 = slab * per; s0 < slab1; s0++, pair += 4) {
        const int next = s0 + 1 < slab1 ? pair + 4 : pair;
        if (s0 + 1 == slab1) weights = pf_buffer(tensor, 0);   // nothing is left to request
        float16v acc[2] = {{0}, {0}};
#pragma unroll
        for (int k = 0; k < UNITS; k++) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const Operand x = take(2 * k + s);
#pragma unroll
                for (int p = 0; p < PF_MX_PLANES; p++) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const uint4v c = w[t][k][s];
                        const int8v b = {(int)c.x, (int)c.y, (int)c.z, (int)c.w, 0, 0, 0, 0};
                        const int sb = (int)(scale[t][k] >> (16 * s + 8 * h));   // byte 0: of the lane's block
                        switch (p) {   // (which byte of the scales is part of the instruction)
                        case 0: acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x.plane[p], b, acc[t], 2, 4, 0, (int)x.scale[0], 0, sb); break;
                        case 1: acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x.plane[p], b, acc[t], 2, 4, 1, (int)x.scale[0], 0, sb); break;
                        case 2: acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x.plane[p], b, acc[t], 2, 4, 2, (int)x.scale[0], 0, sb); break;
                        case 3: acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x.plane[p], b, acc[t], 2, 4, 3, (int)x.scale[0], 0, sb); break;
                        default: acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x.plane[p], b, acc[t], 2, 4, 0, (int)x.scale[1], 0, sb); break;
                        }
                    }
                }
            }
            request(k, next);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the lane holds output row n of its tiles; register r is row 8 (r / 4) + 4 h + r % 4
        float *out = a.down + (size_t)g.first * a.hidden + 64 * pair + n;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = 8 * (r >> 2) + 4 * h + (r & 3);
            const float rs = __shfl(scale_mine, m);
            if (m < g.rows_here) {
                out[(size_t)m * a.hidden] = acc[0][r] * rs;
                out[(size_t)m * a.hidden + 32] = acc[1][r] * rs;
            }
        }
    }
}

// Rows of up to 640 values: five units' digit rows are 80 KB.
bool pf_mx_down_takes(const PfHipMoeDesc &d) { return d.type[3] == PF_MXFP4 && d.inter % 128 == 0 && d.inter <= 640 && d.hidden % 256 == 0; }

// Upload: 32-row tiles of units of four blocks (pf_mxt_*), a thread per 16-byte block or row's scales.
__global__ void pf_k_mx_tile(const uint8_t *payload, const uint8_t *scales, uint8_t *dst, size_t rows, int blocks_per_row) {
    const PfMove m = pf_mx_tile_move((size_t)blockIdx.x * blockDim.x + threadIdx.x, rows, blocks_per_row);
    if (!m.active) return;
    if (m.from == 0) *reinterpret_cast<uint4 *>(dst + m.dst) = *reinterpret_cast<const uint4 *>(payload + m.src);
    else *reinterpret_cast<uint32_t *>(dst + m.dst) = *reinterpret_cast<const uint32_t *>(scales + m.src);
}
void pf_launch_mx_tile(const uint8_t *d_payload, const uint8_t *d_scales, uint8_t *d_dst, size_t rows, int blocks_per_row, hipStream_t stream) {
    const size_t threads = pf_mx_tile_threads(rows, blocks_per_row);
    hipLaunchKernelGGL(pf_k_mx_tile, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, d_payload, d_scales, d_dst, rows, blocks_per_row);
}

template <int UNITS> static void launch(const PfKernelArgs &a, int tokens, unsigned routed_cap, hipStream_t stream) {
    const int lds = 32 * 4 * 128 * UNITS, all = a.hidden / 256, per = pf_slabs_each(all, 5, routed_cap), slabs = (all + per - 1) / per, shift = pf_group_shift(routed_cap);
    static const bool configured = hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_mx_down<UNITS>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    (void)configured;   // more than the default 64 KB
    hipLaunchKernelGGL(pf_k_mx_down<UNITS>, dim3(pf_item_numbers(slabs, shift, routed_cap, 0)), dim3(256), lds, stream, a, slabs, per, shift, (uint32_t)(tokens + 31) / 32);
}
// the routed experts' down products, from the digit rows in act16; routed_cap: their row tiles, at most
void pf_launch_mx_down(const PfKernelArgs &a, int tokens, unsigned routed_cap, hipStream_t stream) {
    switch (a.inter / 128) {
    case 1: launch<1>(a, tokens, routed_cap, stream); break;
    case 2: launch<2>(a, tokens, routed_cap, stream); break;
    case 3: launch<3>(a, tokens, routed_cap, stream); break;
    case 4: launch<4>(a, tokens, routed_cap, stream); break;
    default: launch<5>(a, tokens, routed_cap, stream); break;
    }
}

// Activation rows as digit rows, for batches (a chunk's come with the shared expert's halfs).  dst may be src; scales may be null.
__global__ void __launch_bounds__(256) pf_k_rows_to_digits(const float *src, int cols, size_t rows, uint32_t *dst, float *scales, uint32_t *error_word) {
    pf_rows_to_digits(blockIdx.x, src, cols, rows, dst, scales, error_word);
}
void pf_launch_rows_to_digits(const float *d_src, int cols, size_t rows, uint32_t *d_dst, float *d_scales, uint32_t *d_error, hipStream_t stream) {
    const size_t block = 4 * (size_t)pf_mx_rows_a_wave(cols);
    if (rows) hipLaunchKernelGGL(pf_k_rows_to_digits, dim3((unsigned)((rows + block - 1) / block)), dim3(256), 0, stream, d_src, cols, rows, d_dst, d_scales, d_error);
}
