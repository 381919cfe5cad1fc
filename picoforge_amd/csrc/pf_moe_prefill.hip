// Prefill path: a chunk of tokens through one MoE layer as grouped matrix products on the
// matrix cores.
//
//   pf_k_pf_router      router logits [T, E], both factors as three bf16 parts
//   routing             the kernels of pf_moe_route.hip (serial-order re-route of close tokens)
//   pf_k_pf_group_rows  grouping of the pairs (pf_group_device.h); beside it f32 rows -> power-of-two scaled fp16
//                       pairs (high + low part) and the per-32-group sums, the scale, finite check
//   pf_k_pf_gemm        grouped product over the rows of each expert (the shared expert is
//                       expert E with every token) on v_mfma_f32_32x32x16_f16; gate/up with
//                       the SwiGLU epilogue, or down (routed MXFP4 down rows: pf_moe_mx.hip)
//   pf_k_pf_combine     slot-ordered weighted sum of the down rows, then the shared branch
//
// Numerics.  A Q4_K weight is d * (scale * code) - dmin * min (src/qwen4_packed.c:86-93) with
// 6-bit scale and min and a 4-bit code, so scale * code <= 945 and min <= 63 are integers that
// fp16 holds exactly.  The matrix cores therefore multiply exact integer weight operands:
// P = sum_k (scale * code)_k x_k over a 256-block and Q = sum_g min_g * (sum of x over group g),
// and the block's d and dmin are applied in FP32: acc += d * P - dmin * Q.  Activations are
// scaled per row by a power of two so that the largest magnitude lies in [0.5, 1) and split
// into two fp16 parts x = hi + lo (22 significant bits); every product is exact in the FP32
// accumulators, so the result differs from the reference's serial FP32 sum by accumulation
// order and the 2^-22 activation rounding only.
#include "pf_moe_internal.h"
#include "pf_upload_addr.h"
#include "pf_plain_walk.h"
#include "pf_grouped.h"
#include "pf_router_addr.h"
#include "pf_mx_rows.h"
#include "pf_group_device.h"

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));

// halfs per row of the fp16 form: high parts, low parts, per (started) 256 columns the 16 group-sum halfs
// [even groups: 4 high, 4 low][odd groups: 4 high, 4 low]
__host__ __device__ constexpr size_t pf_half_row(int cols) { return 2 * (size_t)cols + 16 * (((size_t)cols + 255) / 256); }
// the same with the sums of 16 columns, as Q2_K's minima want them: per started 256 columns 16 high, 16 low halfs
__host__ __device__ constexpr size_t pf_half_row16(int cols) { return 2 * (size_t)cols + 32 * (((size_t)cols + 255) / 256); }

// ---- Q4_K tensors in tile order (once, at upload) ---------------------------------------------
// A wave of the grouped product takes a 32-row tile's share of a 256-block at a time.
// In GGUF row order that is 32 pieces a row pitch apart; here the same bytes are regrouped so that
// it is 4608 consecutive bytes: [32 headers of 16 bytes][run 0..3: 16-byte halves 0 of the 32 rows,
// then halves 1].  One thread per 16-byte piece; rows is a multiple of 32.
__global__ void pf_k_q4k_tile(const uint8_t *src, uint8_t *dst, size_t rows, int blocks_per_row) {
    const PfMove m = pf_q4k_tile_move((size_t)blockIdx.x * blockDim.x + threadIdx.x, rows, blocks_per_row);
    if (!m.active) return;
    *reinterpret_cast<uint4 *>(dst + m.dst) = *reinterpret_cast<const uint4 *>(src + m.src);
}

void pf_launch_q4k_tile(const uint8_t *d_src, uint8_t *d_dst, size_t rows, int blocks_per_row, hipStream_t stream) {
    const size_t pieces = pf_q4k_tile_threads(rows, blocks_per_row);
    hipLaunchKernelGGL(pf_k_q4k_tile, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, d_src, d_dst, rows, blocks_per_row);
}

// ---- rows to scaled fp16 pairs ------------------------------------------------------------------
// One workgroup per row (cols a multiple of 32).  scale = 2^e with max|row| / scale in
// [0.5, 1) (1 for a zero row).  Thread j converts the eight values 8j..8j+7; four neighbouring
// threads form one 32-group.
// gate (may be null): a row of `cols` weights; gate_out[row] = sigmoid(row . gate), the shared router's scale (four
// partial sums a lane, lanes and waves added in a fixed order).
// tid: 0..255 of the row's threads; part, dots: four floats of LDS of theirs; store: whether the row is one to write (every
// thread of the workgroup comes along: barriers)
__device__ __forceinline__ void row_to_half(size_t row, bool store, int tid, float *part, float *dots, const float *src, size_t src_pitch, int cols, half_t *dst,
                                            float *scale_out, uint32_t *error_word, const float *gate, float *gate_out) {
    float dot = 0.0f;
    const float *s = src + row * src_pitch;
    float m = 0.0f;
    bool bad = false;
    constexpr int HELD = 2;   // pieces of eight values that a thread keeps between the maximum and the conversion; rows of more are read twice
    float kept[HELD][8];
    auto take = [&](int j, float (&v)[8]) {
        const float4 a = reinterpret_cast<const float4 *>(s)[2 * j], b = reinterpret_cast<const float4 *>(s)[2 * j + 1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    };
    auto look = [&](int j, const float (&v)[8]) {   // the maximum, and the shared router's sum
#pragma unroll
        for (int c = 0; c < 8; c++) { bad |= !pf_finite(v[c]); m = fmaxf(m, fabsf(v[c])); }
        if (gate) {
            const float4 ga = reinterpret_cast<const float4 *>(gate)[2 * j], gb = reinterpret_cast<const float4 *>(gate)[2 * j + 1];
            dot += ((v[0] * ga.x + v[1] * ga.y) + (v[2] * ga.z + v[3] * ga.w)) + ((v[4] * gb.x + v[5] * gb.y) + (v[6] * gb.z + v[7] * gb.w));
        }
    };
#pragma unroll
    for (int p = 0; p < HELD; p++)
        if (tid + 256 * p < cols / 8) take(tid + 256 * p, kept[p]);
#pragma unroll
    for (int p = 0; p < HELD; p++)
        if (tid + 256 * p < cols / 8) look(tid + 256 * p, kept[p]);
    for (int j = tid + 256 * HELD; j < cols / 8; j += 256) {
        float v[8];
        take(j, v);
        look(j, v);
    }
    m = pf_wave_max(m);
    if (pf_lane() == 0) part[tid >> 6] = m;
    if (__any(bad) && pf_lane() == 0) atomicOr(error_word, PF_HIP_ERR_NONFINITE);
    __syncthreads();
    m = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    int e = (__float_as_int(m) >> 23) & 255;                  // m in [2^(e-127), 2^(e-126))
    e = (e == 0 || e == 255) ? 126 : min(e, 252);             // zero, subnormal or nonfinite row: scale 1
    const float scale = __int_as_float((e + 1) << 23);        // 2^(e-126)
    const float inv = __int_as_float((253 - e) << 23);        // 2^(126-e)
    half_t *out = dst + row * pf_half_row(cols);
    auto convert = [&](int j, const float (&v)[8]) {
        half8v hi, lo;
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float x = v[c] * inv;
            const half_t h = (half_t)x, l = (half_t)(x - (float)h);
            hi[c] = h;
            lo[c] = l;
            sum += (float)h + (float)l;
        }
        if (store) {
            *reinterpret_cast<half8v *>(out + 8 * j) = hi;
            *reinterpret_cast<half8v *>(out + cols + 8 * j) = lo;
        }
        sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xB1, 0xF, 0xF, true));   // quad xor 1
        sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x4E, 0xF, 0xF, true));   // quad xor 2
        if ((j & 3) == 0 && store) {
            const int g = j >> 2;
            const half_t sh = (half_t)sum, sl = (half_t)(sum - (float)sh);
            half_t *sums = out + 2 * cols + 16 * (g >> 3) + 8 * (g & 1) + ((g & 7) >> 1);
            sums[0] = sh;
            sums[4] = sl;
        }
    };
#pragma unroll
    for (int p = 0; p < HELD; p++)
        if (tid + 256 * p < cols / 8) convert(tid + 256 * p, kept[p]);
    for (int j = tid + 256 * HELD; j < cols / 8; j += 256) {
        float v[8];
        take(j, v);
        convert(j, v);
    }
    if (gate) {   // uniform
        dot = pf_wave_sum(dot);
        if (pf_lane() == 0) dots[tid >> 6] = dot;
        __syncthreads();
        if (tid == 0 && store) {
            const float z = (dots[0] + dots[1]) + (dots[2] + dots[3]);
            gate_out[row] = pf_sigmoid(z);
            if (!pf_finite(z)) atomicOr(error_word, PF_HIP_ERR_NONFINITE);
        }
    }
    if (tid == 0 && store) scale_out[row] = scale;
}
__global__ void __launch_bounds__(256) pf_k_rows_to_half(const float *src, size_t src_pitch, int cols, half_t *dst, float *scale_out,
                                                         uint32_t *error_word, const float *gate, float *gate_out) {
    __shared__ float part[4], dots[4];
    row_to_half(blockIdx.x, true, threadIdx.x, part, dots, src, src_pitch, cols, dst, scale_out, error_word, gate, gate_out);
}

// The first workgroups group the pairs, 1024 each: every one counts all pairs for itself, those before its own apart (pf_group_pairs),
// and the first writes the lists.  The others convert the chunk's rows, four each.  1024 tokens of width 2048 12.5 us, 2048 of width 2560
// 16.5; with one workgroup for all pairs, and rows read twice, 15.3 and 24.8.
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) pf_k_pf_group_rows(PfKernelArgs a, int tokens, int place_blocks) {
    extern __shared__ __align__(16) uint32_t group_lds[];
    if ((int)blockIdx.x < place_blocks) {
        pf_group_pairs(group_lds, a.ids, tokens * a.top_k, a.experts, tokens, (int)blockIdx.x, a.offsets, a.tiles, reinterpret_cast<uint4 *>(const_cast<uint32_t *>(a.items)),
                       a.pair_to_row, a.row_to_pair);
        return;
    }
    __shared__ float part[4][4], dots[4][4];
    const int team = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8)), row = 4 * ((int)blockIdx.x - place_blocks) + team;
    row_to_half(min(row, tokens - 1), row < tokens, threadIdx.x & 255, part[team], dots[team], a.x, a.x_pitch, a.hidden, (half_t *)a.x16, a.x_scale,
                a.error_word, reinterpret_cast<const float *>(a.w[7]), a.shared_scale);
}

// The same for rows of at most 512 PARTS values (the activation rows): one wave per row, four rows per workgroup, the row
// read once -- a lane keeps its 8 PARTS values between the maximum and the conversion.  With a workgroup per row three
// of its four waves only took part in the maximum: 22528 rows of 640 values took 36.2 us (routed) + 8.8 (shared), 21.6 so.
template <int PARTS, bool SUMS16>
__device__ __forceinline__ void rows_to_half_short(size_t block, const float *src, size_t src_pitch, int cols, size_t rows, half_t *dst,
                                                   float *scale_out, uint32_t *error_word) {
    const size_t row = block * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = pf_lane();
    const float *s = src + row * src_pitch;
    float v[PARTS][8];
    float m = 0.0f;
    bool bad = false;
#pragma unroll
    for (int p = 0; p < PARTS; p++) {
        const int j = 64 * p + lane;
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
        if (j < cols / 8) { a = reinterpret_cast<const float4 *>(s)[2 * j]; b = reinterpret_cast<const float4 *>(s)[2 * j + 1]; }
        const float eight[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int c = 0; c < 8; c++) v[p][c] = eight[c];
    }
#pragma unroll
    for (int p = 0; p < PARTS; p++)
#pragma unroll
        for (int c = 0; c < 8; c++) { bad |= !pf_finite(v[p][c]); m = fmaxf(m, fabsf(v[p][c])); }
    m = pf_wave_max(m);
    if (__any(bad) && lane == 0) atomicOr(error_word, PF_HIP_ERR_NONFINITE);
    int e = (__float_as_int(m) >> 23) & 255;                  // m in [2^(e-127), 2^(e-126))
    e = (e == 0 || e == 255) ? 126 : min(e, 252);             // zero, subnormal or nonfinite row: scale 1
    const float scale = __int_as_float((e + 1) << 23);        // 2^(e-126)
    const float inv = __int_as_float((253 - e) << 23);        // 2^(126-e)
    half_t *out = dst + row * (SUMS16 ? pf_half_row16(cols) : pf_half_row(cols));
#pragma unroll
    for (int p = 0; p < PARTS; p++) {
        const int j = 64 * p + lane;
        const bool mine = j < cols / 8;
        half8v hi, lo;
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float x = v[p][c] * inv;
            const half_t h = (half_t)x, l = (half_t)(x - (float)h);
            hi[c] = h;
            lo[c] = l;
            sum += (float)h + (float)l;
        }
        if (mine) {
            *reinterpret_cast<half8v *>(out + 8 * j) = hi;
            *reinterpret_cast<half8v *>(out + cols + 8 * j) = lo;
        }
        sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xB1, 0xF, 0xF, true));   // quad xor 1
        if (SUMS16) {
            if (mine && (j & 1) == 0) {
                const half_t sh = (half_t)sum, sl = (half_t)(sum - (float)sh);
                half_t *sums = out + 2 * cols + 32 * (j >> 5) + ((j & 31) >> 1);
                sums[0] = sh;
                sums[16] = sl;
            }
            continue;
        }
        sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x4E, 0xF, 0xF, true));   // quad xor 2
        if (mine && (j & 3) == 0) {
            const int g = j >> 2;
            const half_t sh = (half_t)sum, sl = (half_t)(sum - (float)sh);
            half_t *sums = out + 2 * cols + 16 * (g >> 3) + 8 * (g & 1) + ((g & 7) >> 1);
            sums[0] = sh;
            sums[4] = sl;
        }
    }
    if (lane == 0) scale_out[row] = scale;
}

// Two matrices of such rows in one launch (the routed and the shared activation rows): workgroups [0, blocks_a) take
// the first, the others the second.  The first as KIND says: with the sums of 32 or of 16 columns, or as the digit rows of pf_moe_mx.hip
// (of at most 1024 values).
enum RowKind { ROWS_SUMS32, ROWS_SUMS16, ROWS_DIGITS };
template <int PARTS, RowKind KIND>
__global__ void __launch_bounds__(256) pf_k_rows_to_half_short2(const float *src_a, int cols_a, size_t rows_a, half_t *dst_a, float *scale_a,
                                                                unsigned blocks_a, const float *src_b, int cols_b, size_t rows_b,
                                                                half_t *dst_b, float *scale_b, uint32_t *error_word) {
    if (blockIdx.x < blocks_a) {
        if (KIND == ROWS_DIGITS) pf_rows_to_digits(blockIdx.x, src_a, cols_a, rows_a, reinterpret_cast<uint32_t *>(dst_a), scale_a, error_word);
        else rows_to_half_short<PARTS, KIND == ROWS_SUMS16>(blockIdx.x, src_a, (size_t)cols_a, cols_a, rows_a, dst_a, scale_a, error_word);
    }
    else rows_to_half_short<PARTS, false>(blockIdx.x - blocks_a, src_b, (size_t)cols_b, cols_b, rows_b, dst_b, scale_b, error_word);
}

static void launch_rows_to_half(const float *src, size_t src_pitch, int cols, size_t rows, half_t *dst, float *scale_out,
                                uint32_t *error_word, hipStream_t stream) {
    if (rows == 0) return;
    hipLaunchKernelGGL(pf_k_rows_to_half, dim3((unsigned)rows), dim3(256), 0, stream, src, src_pitch, cols, dst, scale_out,
                       error_word, (const float *)nullptr, (float *)nullptr);
}

// squared norm of every router row (once, at upload)
__global__ void __launch_bounds__(64) pf_k_row_norm2(const float *w, int cols, float *out) {
    const float *r = w + (size_t)blockIdx.x * cols;
    float s = 0.0f;
    for (int c = threadIdx.x; c < cols; c += 64) s = fmaf(r[c], r[c], s);
    s = pf_wave_sum(s);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

void pf_launch_row_norm2(const float *d_w, int rows, int cols, float *d_out, hipStream_t stream) {
    hipLaunchKernelGGL(pf_k_row_norm2, dim3(rows), dim3(64), 0, stream, d_w, cols, d_out);
}

// ---- router logits by three bf16 parts of every factor -----------------------------------------
// Workgroup = a tile of 32 TR tokens x 32 TC experts, its eight waves an eighth of the columns each (the
// partial tiles are added in wave order).  Also writes the routing tolerance's bound on the sum of
// squared products, max(x)^2 * |w_e|^2.  (The shared router's logit comes with the rows' conversion.)
//
// A value is h + m + l exactly: h its upper eight significant bits, rounded (but never to infinity: the largest floats keep theirs),
// m the rest rounded to eight, l what that leaves, |m| <= 2^-8 and |l| <= 2^-17 of the value.  Of the nine products of two values six are
// formed, exact in the FP32 sums; the three left out are below 2^-24 (1 + 2^-10) of the product together, what rounding it to FP32
// takes, as the reference does before it adds: the routing tolerance (pf_route_finish_wave) needs no more than that.
//
// The experts' parts are made once, at upload, in the order in which a wave takes them as operands (pf_k_router_parts): 1 KB an
// instruction, no conversion.  A row of x is fetched in 32-column pieces, whole 128-byte lines (lane = 8 * row + 16-byte piece),
// passes through LDS of the wave's own (row pitch 144 bytes; no barrier) because a product step wants columns 8 h .. 8 h + 7 of row i
// from lane (i, h), and is split there, a step ahead of its products.
//
// Bound by what the L2 hands out: 2048 tokens of width 2560 against 512 experts are 420 MB of operands in 42 us traced.  On the FP32
// instruction, whose products alone take 34, it was 75; with both factors split in the kernel 53, bound by the vector instructions.
// 1024 tokens of width 2048: 25.4 us (FP32 38); tiles of 64 x 32 instead of 32 x 64 27.1, two pieces ahead no faster.  Error
// against 64 bits, 2-norm (2047 tokens of width 2560, 1025, 600 of 2048) and largest of the magnitudes' sum: 2.8, 2.5, 2.5e-7 and 5.5, 5.1,
// 5.1e-8, on FP32 3.3, 2.9, 2.9e-7 and 6.4, 5.9, 5.9e-8.  With h cut off (|m| to 2^-7, 2^-22 of a product left out) the largest were 6.9, 7.7,
// 7.7e-8 at the same time; m l and l m as well bring nothing (the same errors to four digits) for 6 us of 2048 tokens' 43.
typedef float float4v __attribute__((ext_vector_type(4)));
typedef short short2v __attribute__((ext_vector_type(2)));
typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
struct RouterParts { uint4v part[3]; };
__device__ __forceinline__ uint32_t router_round2(float a, float b) {   // (whole vectors are converted a value at a time)
    typedef float float2v __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{a, b}, bf16x2));
}
__device__ __forceinline__ RouterParts router_parts(float4v a, float4v b) {
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    RouterParts r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // no infinity: as signed halves the positive values end at the largest, as unsigned ones the negative values
        const short2v most = {0x7f7f, 0x7f7f};
        const ushort2v least = {0xff7f, 0xff7f};
        uint32_t upper = router_round2(x[2 * i], x[2 * i + 1]);
        upper = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(short2v, upper), most));
        upper = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2v, upper), least));
        const float u1 = x[2 * i] - __uint_as_float(upper << 16), v1 = x[2 * i + 1] - __uint_as_float(upper & 0xffff0000u);
        const uint32_t middle = router_round2(u1, v1);
        r.part[0][i] = upper;
        r.part[1][i] = middle;
        r.part[2][i] = router_round2(u1 - __uint_as_float(middle << 16), v1 - __uint_as_float(middle & 0xffff0000u));
    }
    return r;
}

// Router rows [experts][cols] -> [tile of 32][16 columns][part][lane (i, h): row i, columns 8 h .. 8 h + 7][8 bf16]; rows beyond the
// last are zeros.  A thread per lane of a step.
__global__ void __launch_bounds__(256) pf_k_router_parts(const float *w, int experts, int cols, uint4v *out, size_t threads) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= threads) return;
    const size_t step = id >> 6, tile = step / (size_t)(cols / 16);
    const int lane = (int)(id & 63), row = (int)(32 * tile) + (lane & 31), c = 16 * (int)(step % (size_t)(cols / 16)) + 8 * (lane >> 5);
    float4v a = {0}, b = {0};
    if (row < experts) {
        const float4v *src = reinterpret_cast<const float4v *>(w + (size_t)row * cols + c);
        a = src[0]; b = src[1];
    }
    const RouterParts r = router_parts(a, b);
#pragma unroll
    for (int p = 0; p < 3; p++) out[(3 * step + p) * 64 + lane] = r.part[p];
}
void pf_launch_router_parts(const float *d_w, int experts, int cols, void *d_out, hipStream_t stream) {
    const size_t threads = (size_t)pf_router_tiles(experts) * (size_t)(cols / 16) * 64;
    hipLaunchKernelGGL(pf_k_router_parts, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, d_w, experts, cols, reinterpret_cast<uint4v *>(d_out), threads);
}

#define PF_ROUTER_PITCH 36   // floats between rows of a staged piece: eight neighbouring lanes' 16-byte reads cover all banks
#define PF_ROUTER_WAVES 8
// the staged pieces, later the partial tiles
constexpr int router_lds_bytes(int tr, int tc) { return PF_ROUTER_WAVES * 128 * tr * (32 * tc > PF_ROUTER_PITCH ? 32 * tc : PF_ROUTER_PITCH); }
template <int TR, int TC>
__global__ void __launch_bounds__(64 * PF_ROUTER_WAVES) __attribute__((amdgpu_waves_per_eu(2))) pf_k_pf_router(PfKernelArgs a, int tokens) {
    extern __shared__ __align__(16) float router_lds[];   // [wave][x row][column]; later the waves' partial tiles
    __shared__ uint32_t largest[32 * TR];                 // the rows' largest magnitudes, as bits
    const int H = a.hidden, E = a.experts, lane = pf_lane(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.x * 32 * TR, e0 = blockIdx.y * 32 * TC;
    if (threadIdx.x < 32 * TR) largest[threadIdx.x] = 0;
    const int i = lane & 31, kk = lane >> 5;
    // the waves split the rows' 128-byte lines (hidden is a multiple of 32)
    const int lines = H / 32, l0 = lines * wave / PF_ROUTER_WAVES, l1 = lines * (wave + 1) / PF_ROUTER_WAVES;
    const int lr = lane >> 3, piece = lane & 7;   // fetch: row within a group of eight, 16-byte piece of the line
    constexpr int GROUPS = 4 * TR;                // of eight rows
    // the x rows by their addresses, in place of those beyond the last token the last one again; the experts' parts in a buffer that no
    // load leaves (its bound is not compared with the scalar part of an offset)
    const float4v *x_row[GROUPS];
#pragma unroll
    for (int g = 0; g < GROUPS; g++) x_row[g] = reinterpret_cast<const float4v *>(a.x + (size_t)min(t0 + 8 * g + lr, tokens - 1) * a.x_pitch) + piece;
    const PfBuffer experts = pf_buffer(a.router_parts + pf_router_tile_at(e0 / 32, H), (uint32_t)min(TC, pf_router_tiles(E) - e0 / 32) * (uint32_t)pf_router_tile_at(1, H));
    float *mine = router_lds + (size_t)wave * TR * 32 * PF_ROUTER_PITCH;
    float16v acc[TR][TC];
#pragma unroll
    for (int r = 0; r < TR; r++)
#pragma unroll
        for (int c = 0; c < TC; c++) acc[r][c] = float16v{0};
    float most[GROUPS] = {};
    float4v fetched[GROUPS], raw[TR][2];
    RouterParts x[2][TR], w[2][TC];   // of the two steps of 16 columns that a piece is
    auto fetch = [&](int l) {
#pragma unroll
        for (int g = 0; g < GROUPS; g++) fetched[g] = x_row[g][8 * min(l, l1 - 1)];
    };
    auto request = [&](int step, int l) {
#pragma unroll
        for (int c = 0; c < TC; c++) {
            const int tile = pf_router_tile_read(E, e0 / 32, c);
#pragma unroll
            for (int p = 0; p < 3; p++)
                w[step][c].part[p] = __builtin_amdgcn_raw_buffer_load_b128(experts, (int)pf_router_part_at(0, 0, 0, 0, lane), (int)pf_router_part_at(tile, H, 2 * min(l, l1 - 1) + step, p, 0), 0);
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            const float4v v = fetched[g];
            *reinterpret_cast<float4v *>(mine + (8 * g + lr) * PF_ROUTER_PITCH + 4 * piece) = v;
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most[g]) : "v"(v.x), "v"(v.y));   // (fmaxf spends an instruction on quieting every operand)
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most[g]) : "v"(v.z), "v"(v.w));
        }
    };
    auto take = [&](int step) {
#pragma unroll
        for (int q = 0; q < TR; q++) {
            const float *at = mine + (32 * q + i) * PF_ROUTER_PITCH + 16 * step + 8 * kk;
            raw[q][0] = *reinterpret_cast<const float4v *>(at);
            raw[q][1] = *reinterpret_cast<const float4v *>(at + 4);
        }
    };
    // step's products, the other step's rows split meanwhile: a few vector instructions behind every product
    auto products = [&](int step) {
#pragma unroll
        for (int q = 0; q < TR; q++) x[step ^ 1][q] = router_parts(raw[q][0], raw[q][1]);
#pragma unroll
        for (int p = 0; p < 6; p++) {   // l h, h l, m m, m h, h m, h h
            constexpr int px[6] = {2, 0, 1, 1, 0, 0}, pw[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int r = 0; r < TR; r++)
#pragma unroll
                for (int c = 0; c < TC; c++)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x[step][r].part[px[p]]), __builtin_bit_cast(bf16x8, w[step][c].part[pw[p]]), acc[r][c], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < 6 * TR * TC; m++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                               // a product
            __builtin_amdgcn_sched_group_barrier(0x002, (54 * TR + 6 * TR * TC - 1) / (6 * TR * TC), 0);   // vector instructions
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (l0 < l1) {
        fetch(l0);
        request(0, l0);
        request(1, l0);
        stage();
        fetch(l0 + 1);
        take(0);
#pragma unroll
        for (int q = 0; q < TR; q++) x[0][q] = router_parts(raw[q][0], raw[q][1]);
        take(1);
        for (int l = l0; l < l1; l++) {
            products(0);
            request(0, l + 1);
            stage();   // the next piece
            fetch(l + 2);
            take(0);
            __builtin_amdgcn_sched_barrier(0);
            products(1);
            request(1, l + 1);
            take(1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();   // the staged pieces have been read
#pragma unroll
    for (int g = 0; g < GROUPS; g++) atomicMax(&largest[8 * g + lr], __float_as_uint(most[g]));
    constexpr int REGS = 16 * TR * TC;
#pragma unroll
    for (int r = 0; r < REGS; r++) router_lds[(wave * REGS + r) * 64 + lane] = acc[r / 16 / TC][r / 16 % TC][r % 16];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < REGS / PF_ROUTER_WAVES; q++) {   // added in wave order
        const int r = wave + PF_ROUTER_WAVES * q;
        float logit = router_lds[r * 64 + lane];
#pragma unroll
        for (int v = 1; v < PF_ROUTER_WAVES; v++) logit += router_lds[(v * REGS + r) * 64 + lane];
        const int row = t0 + 32 * (r / 16 / TC) + 8 * ((r & 15) >> 2) + 4 * kk + (r & 3), col = e0 + 32 * (r / 16 % TC) + i;
        if (row >= tokens || col >= E) continue;
        a.logits[(size_t)row * E + col] = logit;
        const float m = __uint_as_float(largest[row - t0]);
        a.logit_ssq[(size_t)row * E + col] = m * m * a.w_norm2[col];
    }
}
template <int TR, int TC>
static void launch_router(const PfKernelArgs &a, int tokens, hipStream_t stream) {
    static const bool configured = hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_pf_router<TR, TC>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       router_lds_bytes(TR, TC)) == hipSuccess;   // more than the default 64 KB
    (void)configured;
    const dim3 grid((tokens + 32 * TR - 1) / (32 * TR), (a.experts + 32 * TC - 1) / (32 * TC));
    hipLaunchKernelGGL((pf_k_pf_router<TR, TC>), grid, dim3(64 * PF_ROUTER_WAVES), router_lds_bytes(TR, TC), stream, a, tokens);
}

// ---- grouped product ------------------------------------------------------------------------------
enum { PF_GEMM_GATE_UP = 0, PF_GEMM_DOWN = 1 };

// Workgroup = one 32-row tile of an expert against 32 GW weight rows: eight waves, each with one 32-row weight tile (the gate and
// the up tiles of 128 units, or 256 down rows); a down workgroup goes over several such slabs.
//
// A wave takes its weights straight from memory into registers, 16 bytes a lane and whole cache lines an instruction, and
// requests the bytes of the next 256-block into the registers that the products have just left: 4 to 5 KB a wave on their way
// at any time, and no wave waits for another one's.  The activation rows are what the waves share: a block's 256 columns in LDS,
// two copies in turn, the next block's requested straight into the other copy.  One barrier a 256-block.  A wave with one tile
// keeps to 128 registers, so two workgroups, four waves a SIMD, share a compute unit: while one unpacks a block's headers, adds
// its block up or waits, the others feed the matrix core.
//
// Bound by power and by the bytes together: at 1024 tokens of the benchmark's Q4_K layer (640 row tiles, 604 MB of gate and up
// weights) the card draws 1.28 kW and its clock falls to 1.8 GHz; repeated by itself the launch takes 177 us, without the memory reads
// 137, without the products 157.  Before, loader waves moved every operand through a ring in LDS with a barrier every 64 columns.
// Traced within forwards, in turn, gate and up / down, us, before and now (units in slabs of 128, not 256): 1024 tokens 222 / 122 ->
// 207 / 117, 2048 tokens 317 / 168 -> 304 / 173, IQ2_XXS, 777 tokens 229 / 116 -> 184 / 106.
//
//   copy   [part: high, low][64 columns][eight rows][16-byte chunk of the 64 columns][row][16 bytes]
//
// Tiles of experts with at most 16 rows put the low parts of their rows into the tile's other 16 rows (PARTS = 1): one product
// instead of two, half of the operand reads and of the copy.
//
// Matrix-core operands.  Lane (n = lane % 32, h = lane / 32) holds column n (a weight row) and supplies K slots 8h..8h+7.  Which
// columns of the block those are is free as long as the activations' lanes take the same ones.  Q4_K: a lane loads half h of a
// run's 32 nibble bytes, steps 0 and 1 are the low nibbles (group 2j, columns 16h..16h+15 of it), steps 2 and 3 the high
// nibbles (group 2j + 1).  IQ2_XXS: a lane loads the 8 bytes of group 2j + h, a step is one of its four grid entries.
#define GW 8                                   // waves per workgroup
#define GEMM_IMAGE 1152                        // between eight-row images of 64 columns: 1 KB + 128, neighbours start on opposite bank halves
#define GEMM_PART_BYTES (16 * GEMM_IMAGE)      // one part of 32 rows x 256 columns
#define GEMM_COPY_BYTES (2 * GEMM_PART_BYTES)
#define GEMM_LDS (2 * GEMM_COPY_BYTES)
#define IQ2_GRID_OFF GEMM_LDS                  // IQ2_XXS: 256 grid entries of 8 magnitudes, then 128 entries of 8 sign bytes
#define IQ2_SIGN_OFF (IQ2_GRID_OFF + 2048)
#define GEMM_LDS_IQ2 (IQ2_SIGN_OFF + 1024)

__device__ __forceinline__ void to_lds(const void *global, unsigned char *lds) {
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t *>(global), reinterpret_cast<uint32_t *>(lds), 16, 0, 0);
}

// One expert's tensor as a wave reads it: the buffers and what the lanes add to an offset in them.  Tile order keeps a 32-row
// tile's 256-block together, row order a row's blocks.
struct GemmRows {
    const uint8_t *base, *head;         // codes, and block headers (the same bytes except for IQ2_XXS in row order: half scales)
    uint32_t bytes, head_bytes;
    uint32_t lane_at, head_at;          // per lane: of its codes, of its row's block header
    uint32_t tile_step, block_step, run_step, head_tile_step, head_step;
    uint32_t group_step, head_run_step; // Q8_0: between the two groups of a run, between the runs' scale pairs
};
template <int FMT> __device__ __forceinline__ GemmRows gemm_rows(const PfKernelArgs &a, int t, size_t expert) {
    const uint32_t n = pf_lane() & 31, h = pf_lane() >> 5, row_bytes = (uint32_t)a.row_bytes[t], blocks = (uint32_t)a.blocks_per_row[t];
    const bool tiled = FMT == PF_IQ2_XXS ? a.wi[t] != nullptr : FMT == PF_Q8_0 ? a.wq[t] != nullptr : a.wt[t] != nullptr;
    GemmRows r;
    if (FMT == PF_Q8_0 && tiled) {   // (a tensor of one expert)
        r.bytes = (uint32_t)pf_q8t_expert_bytes(a.n_out[t], (int)blocks / 2);
        r.base = a.wq[t];
        r.lane_at = 512 * h + 16 * n; r.head_at = 2048 + 4 * n;
        r.group_step = 1024; r.run_step = r.head_run_step = PF_I2T_CHUNK; r.block_step = r.head_step = 4 * PF_I2T_CHUNK;
        r.tile_step = r.head_tile_step = blocks / 2 * PF_I2T_CHUNK;
    } else if (FMT == PF_Q8_0) {     // payloads of all experts, then their scales
        r.bytes = (uint32_t)a.expert_bytes[t]; r.head_bytes = 2 * (uint32_t)a.n_out[t] * blocks;
        r.base = a.w[t] + expert * r.bytes;
        r.head = a.w[t] + a.scale_offset[t] + expert * r.head_bytes;
        r.lane_at = n * row_bytes + 16 * h; r.head_at = 2 * n * blocks;
        r.group_step = 32; r.run_step = 64; r.head_run_step = 4; r.block_step = 256; r.head_step = 16;
        r.tile_step = 32 * row_bytes; r.head_tile_step = 64 * blocks;
        return r;
    } else
    if (FMT == PF_IQ2_XXS && tiled) {
        r.bytes = (uint32_t)pf_i2t_expert_bytes(a.n_out[t], (int)blocks);
        r.base = a.wi[t] + expert * r.bytes;
        r.lane_at = 16 * n + 8 * h; r.head_at = 2048 + 2 * n;
        r.block_step = r.head_step = PF_I2T_CHUNK; r.run_step = 512;
        r.tile_step = r.head_tile_step = blocks * PF_I2T_CHUNK;
    } else if (FMT == PF_IQ2_XXS) {   // payloads of all experts, then their scales
        r.bytes = (uint32_t)a.expert_bytes[t]; r.head_bytes = 2 * (uint32_t)a.n_out[t] * blocks;
        r.base = a.w[t] + expert * r.bytes;
        r.head = a.w[t] + a.scale_offset[t] + expert * r.head_bytes;
        r.lane_at = n * row_bytes + 8 * h; r.head_at = 2 * n * blocks;
        r.block_step = 64; r.head_step = 2; r.run_step = 16;
        r.tile_step = 32 * row_bytes; r.head_tile_step = 64 * blocks;
        return r;
    } else if (FMT == PF_Q2_K) {   // GGUF rows
        r.bytes = (uint32_t)a.expert_bytes[t];
        r.base = a.w[t] + expert * a.expert_bytes[t];
        r.lane_at = n * row_bytes + 16 + 16 * h; r.head_at = n * row_bytes + 68 * h;
        r.block_step = r.head_step = 84; r.run_step = 32;
        r.tile_step = r.head_tile_step = 32 * row_bytes;
    } else {
        r.bytes = (uint32_t)a.expert_bytes[t];
        r.base = (tiled ? a.wt[t] : a.w[t]) + expert * a.expert_bytes[t];
        r.tile_step = r.head_tile_step = 32 * row_bytes;
        r.lane_at = tiled ? 512 + 512 * h + 16 * n : 16 + n * row_bytes + 16 * h;
        r.head_at = tiled ? 16 * n : n * row_bytes;
        r.block_step = r.head_step = tiled ? 4608 : 144; r.run_step = tiled ? 1024 : 32;
    }
    r.head = r.base; r.head_bytes = r.bytes;
    return r;
}

// Four nibbles (those under mask in a dword) times the group's scale as fp16 operands, exact: a nibble alone in a half is the
// subnormal q 2^-24 (16 q 2^-24 where a high nibble stays in place), s2 the scale times 2^10 (2^6) in both halves, the product
// q s 2^-14, a normal number.  The fold takes the 2^-14 away again.
__device__ __forceinline__ half4v q4_scaled_codes(uint32_t w, uint32_t mask, half2v s2) {
    const uint32_t q = w & mask;
    const half2v v0 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0u, q, 0x0C010C00u)) * s2;
    const half2v v1 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0u, q, 0x0C030C02u)) * s2;
    return half4v{v0.x, v0.y, v1.x, v1.y};
}

__device__ __forceinline__ half8v join(half4v a, half4v b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// A wave's weight tile over one 256-block: the bytes as they were loaded (code[run], head), and what the block's headers say (open).
// The block is sixteen steps of one matrix-core operand: step i is step i % 4 of run i / 4, against the 16-byte column chunk
// chunk(i) + chunk_h h of the run's 64 columns.
template <int FMT> struct GemmBlock;
template <> struct GemmBlock<PF_Q4_K> {
    uint4v code[4], head;
    half2v scale[4];         // groups 2j and 2j + 1: times 2^10 and 2^6
    float d, low;            // factors of the products (2^14 d) and of the minima's sums
    static __device__ __forceinline__ constexpr int chunk(int i) { return 4 * ((i & 3) >> 1) + (i & 1); }
    static constexpr int chunk_h = 2;
    static constexpr int requests = 6;   // of a block: its headers, the rows' sums, four runs
    __device__ __forceinline__ void request_run(int j, const PfBuffer &b, const GemmRows &r, uint32_t at) {
        code[j] = __builtin_amdgcn_raw_buffer_load_b128(b, (int)r.lane_at, (int)(at + (uint32_t)j * r.run_step), 0);
    }
    __device__ __forceinline__ void request_head(const PfBuffer &b, const GemmRows &r, uint32_t at) {
        head = __builtin_amdgcn_raw_buffer_load_b128(b, (int)r.head_at, (int)at, 0);
    }
    // Scales and minima of all eight groups (src/qwen4_packed.c:88-91), four bytes at a time; returns the minima as the operand
    // of the product with the rows' group sums: K slots 8h..8h+3 hold the high parts of groups h, 2 + h, 4 + h, 6 + h, slots
    // 8h+4..8h+7 their low parts, so the four minima appear once against each.
    __device__ __forceinline__ half8v open() {
        const uint4v w = head;
        const half2v dm = __builtin_bit_cast(half2v, w.x);
        d = (float)dm.x * 16384.0f; low = (float)dm.y;
        const uint32_t s03 = w.y & 0x3F3F3F3Fu, s47 = (w.w & 0x0F0F0F0Fu) | ((w.y >> 2) & 0x30303030u);
        const uint32_t m03 = w.z & 0x3F3F3F3Fu, m47 = ((w.w >> 4) & 0x0F0F0F0Fu) | ((w.z >> 2) & 0x30303030u);
        const uint32_t bias = 0x64646464u;   // a byte under the exponent byte 0x64 is 1024 + byte
        const half2v k = {(half_t)1024.0f, (half_t)1024.0f}, up = {(half_t)1024.0f, (half_t)64.0f};
        scale[0] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, s03, 0x04010400u)) - k) * up;
        scale[1] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, s03, 0x04030402u)) - k) * up;
        scale[2] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, s47, 0x04010400u)) - k) * up;
        scale[3] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, s47, 0x04030402u)) - k) * up;
        const uint32_t mine = __builtin_amdgcn_perm(m47, m03, pf_lane() >> 5 ? 0x07050301u : 0x06040200u);
        const half2v a = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, mine, 0x04010400u)) - k;
        const half2v b = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, mine, 0x04030402u)) - k;
        return half8v{a.x, a.y, b.x, b.y, a.x, a.y, b.x, b.y};
    }
    __device__ __forceinline__ half8v operand(int i, const lds_byte *) const {
        const int j = i >> 2, t = i & 3;
        const half_t f = t < 2 ? scale[j].x : scale[j].y;
        const uint32_t mask = t < 2 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
        return join(q4_scaled_codes(code[j][2 * (t & 1)], mask, half2v{f, f}), q4_scaled_codes(code[j][2 * (t & 1) + 1], mask, half2v{f, f}));
    }
};
// IQ2_XXS (src/qwen4_packed.c:95-121): a weight is d / 8 * (2 s + 1) * magnitude * sign with a 4-bit s per 32-group, magnitudes 8,
// 25 or 43 from the grid and d per 256-block, so (2 s + 1) * magnitude <= 1333 is an exact fp16 operand: a magnitude byte below its
// sign's byte (0 or 0x80) is the subnormal +-m 2^-24, times (2 s + 1) 2^10 the normal number +-m (2 s + 1) 2^-14.  A 256-block's
// result is (d / 8) * P, with the 2^-14 taken away again; there are no minima.
// Bound by the vector instructions and the tables' reads as much as by the products: sign bytes instead of masks of eight halves
// (half the bytes of that read) and one multiplication instead of a fused step and a bit flip, 8 instructions an operand
// for 12: gate and up / down of 1024 tokens, measured layer, 203 / 116 -> 186 / 103 us traced, of the q2 profile 289 -> 261.
template <> struct GemmBlock<PF_IQ2_XXS> {
    uint2v code[4];
    uint16_t head;
    float d, low;
    static __device__ __forceinline__ constexpr int chunk(int i) { return i & 3; }
    static constexpr int chunk_h = 4;
    static constexpr int requests = 5;
    __device__ __forceinline__ void request_run(int j, const PfBuffer &b, const GemmRows &r, uint32_t at) {
        code[j] = __builtin_amdgcn_raw_buffer_load_b64(b, (int)r.lane_at, (int)(at + (uint32_t)j * r.run_step), 0);
    }
    __device__ __forceinline__ void request_head(const PfBuffer &b, const GemmRows &r, uint32_t at) {
        head = __builtin_amdgcn_raw_buffer_load_b16(b, (int)r.head_at, (int)at, 0);
    }
    __device__ __forceinline__ void open() { d = (float)__builtin_bit_cast(half_t, head) * 2048.0f; }
    __device__ __forceinline__ half8v operand(int i, const lds_byte *tables) const {
        const uint2v g = code[i >> 2];
        const half_t f = (half_t)(int)((2u * (g.y >> 28) + 1u) << 10);
        const half2v s2 = {f, f};
        const uint2v m = *reinterpret_cast<const __attribute__((address_space(3))) uint2v *>(tables + 8u * ((g.x >> (8 * (i & 3))) & 255u));
        const uint2v sign = *reinterpret_cast<const __attribute__((address_space(3))) uint2v *>(tables + 2048 + 8u * ((g.y >> (7 * (i & 3))) & 127u));
        const half2v v0 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sign.x, m.x, 0x05010400u)) * s2;
        const half2v v1 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sign.x, m.x, 0x07030602u)) * s2;
        const half2v v2 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sign.y, m.y, 0x05010400u)) * s2;
        const half2v v3 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sign.y, m.y, 0x07030602u)) * s2;
        return half8v{v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
    }
};

// eight bytes as eight halfs, exact: a byte under the exponent byte 0x64 reads as 1024 + byte
__device__ __forceinline__ half8v half8_of_bytes(uint32_t b0, uint32_t b1, half_t offset) {
    const uint32_t bias = 0x64646464u;
    const half2v c = {offset, offset};
    const half2v v0 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, b0, 0x04010400u)) - c;
    const half2v v1 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, b0, 0x04030402u)) - c;
    const half2v v2 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, b1, 0x04010400u)) - c;
    const half2v v3 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, b1, 0x04030402u)) - c;
    return half8v{v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
}

// Q2_K (src/qwen4_packed.c:106-121): a weight is d * scale * code - dmin * min with a 4-bit scale and minimum for 16 columns and a
// 2-bit code, so scale * code <= 45 is an exact fp16 operand, made as Q4_K's are (the code stays where it is in its byte, the scale brings
// the power of four), and the minima are the operand of a product with the rows' sums of 16 columns.  Lane (n, h) loads bytes
// 16h..16h+15 of both halves of a block's codes; step i is the eight bytes i % 2 of them at bits 2 (i / 2 % 4), its columns those of Q4_K.
// Rows are read where they lie, 84 bytes a block: an instruction touches 32 lines or more for 512 to 1024 bytes, and the L2's lines
// bound the kernel.  So a block's three loads follow each other while its lines are there (apart 276 us for 1500 tokens of the
// checkpoints' widths, together 257), and the scales and the two factors are one load, the lower lanes' and the upper ones' (254).
// On the plain kernel it took 339, 239 -> 162 for 500 tokens, 164 -> 119 for 1000 of 2048 x 512; the distance to 64 bits is the same
// (4.9e-7 at 2560 x 640).  A block's loads asked for half a block earlier, in registers of their own: 24 of them spilled, 320.
template <> struct GemmBlock<PF_Q2_K> {
    uint4v code[2], head;    // head: the scales in lanes 0..31, the block's last 16 bytes in lanes 32..63
    half2v scale[4];         // of a 64-column run: the scales of its two groups' halves h, times 2^10 and 2^8, or 2^6 and 2^4
    float d, low;
    static __device__ __forceinline__ constexpr int chunk(int i) { return 4 * ((i & 3) >> 1) + (i & 1); }
    static constexpr int chunk_h = 2;
    static constexpr int requests = 5;   // of a block: the rows' sums (two), its header, two halves of codes
    __device__ __forceinline__ void request_half(int j, const PfBuffer &b, const GemmRows &r, uint32_t at) {
        code[j] = __builtin_amdgcn_raw_buffer_load_b128(b, (int)r.lane_at, (int)(at + (uint32_t)j * r.run_step), 0);
    }
    __device__ __forceinline__ void request_head(const PfBuffer &b, const GemmRows &r, uint32_t at) {
        head = __builtin_amdgcn_raw_buffer_load_b128(b, (int)r.head_at, (int)at, 0);
    }
    // Returns the minima of sub-groups 8h..8h+7 as an operand.
    __device__ __forceinline__ half8v open() {
        uint32_t sc[4], dm = 0;   // the lower lanes' words and the upper lanes' last one, in all lanes
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const auto halves = __builtin_amdgcn_permlane32_swap(head[c], head[c], false, false);
            sc[c] = halves[0];
            if (c == 3) dm = halves[1];
        }
        const half2v both = __builtin_bit_cast(half2v, dm);
        d = (float)both.x * 16384.0f; low = (float)both.y;
        const bool second = pf_lane() >> 5;
        const uint32_t bias = 0x64646464u;   // a byte under the exponent byte 0x64 is 1024 + byte
        const half2v k = {(half_t)1024.0f, (half_t)1024.0f}, up0 = {(half_t)1024.0f, (half_t)256.0f}, up1 = {(half_t)64.0f, (half_t)16.0f};
#pragma unroll
        for (int half = 0; half < 2; half++) {   // sub-groups h, 2 + h, 4 + h, 6 + h of the half
            const uint32_t mine = __builtin_amdgcn_perm(sc[2 * half + 1], sc[2 * half], second ? 0x07050301u : 0x06040200u) & 0x0F0F0F0Fu;
            scale[2 * half] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, mine, 0x04010400u)) - k) * up0;
            scale[2 * half + 1] = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(bias, mine, 0x04030402u)) - k) * up1;
        }
        return half8_of_bytes(((second ? sc[2] : sc[0]) >> 4) & 0x0F0F0F0Fu, ((second ? sc[3] : sc[1]) >> 4) & 0x0F0F0F0Fu, (half_t)1024.0f);
    }
    __device__ __forceinline__ half8v operand(int i) const {
        const half_t f = (i & 2) ? scale[i >> 2].y : scale[i >> 2].x;
        const uint32_t mask = 0x03030303u << (2 * ((i >> 1) & 3));
        return join(q4_scaled_codes(code[i >> 3][2 * (i & 1)], mask, half2v{f, f}), q4_scaled_codes(code[i >> 3][2 * (i & 1) + 1], mask, half2v{f, f}));
    }
};

// signed bytes: flip the sign bit, read as unsigned, take 128 more away
__device__ __forceinline__ half8v half8_of_signed_bytes(uint32_t b0, uint32_t b1) {
    return half8_of_bytes(b0 ^ 0x80808080u, b1 ^ 0x80808080u, (half_t)1152.0f);
}

// Q8_0: signed code bytes, a half scale per 32-group: a group's partial sums times its scale.  Lane (n, h) loads bytes 16h..16h+15 of a
// group; step i is half i % 2 of its bytes in group i / 2 of the block.  Half scales are no integers, so they stay out of the
// operand.  The shared expert of the checkpoint profiles: its gate and up tiles ride with the routed ones' launch (2048 tokens of 2560 x
// 640, the q4 profile: 433 us traced, before 490 and 90 for a launch of the plain kernel), its down tiles are a launch of 39 us.
template <> struct GemmBlock<PF_Q8_0> {
    uint4v code[8];
    uint32_t head[4];   // of a run: its two groups' scales
    static __device__ __forceinline__ constexpr int chunk(int i) { return 4 * ((i & 3) >> 1) + (i & 1); }
    static constexpr int chunk_h = 2;
    static constexpr int requests = 12;
    __device__ __forceinline__ void request_run(int j, const PfBuffer &b, const PfBuffer &heads, const GemmRows &r, uint32_t at, uint32_t head_at) {
#pragma unroll
        for (int e = 0; e < 2; e++)
            code[2 * j + e] = __builtin_amdgcn_raw_buffer_load_b128(b, (int)r.lane_at, (int)(at + (uint32_t)j * r.run_step + (uint32_t)e * r.group_step), 0);
        head[j] = __builtin_amdgcn_raw_buffer_load_b32(heads, (int)r.head_at, (int)(head_at + (uint32_t)j * r.head_run_step), 0);
    }
    __device__ __forceinline__ float scale(int g) const {
        return (float)__builtin_bit_cast(half_t, (unsigned short)((g & 1) ? head[g >> 1] >> 16 : head[g >> 1] & 0xffffu));
    }
    __device__ __forceinline__ half8v operand(int i) const {
        const uint4v c = code[i >> 1];
        return half8_of_signed_bytes(c[2 * (i & 1)], c[2 * (i & 1) + 1]);
    }
};

// What a wave's requests read of its item.
struct GemmSource {
    PfBuffer weights, heads, x[2];
    GemmRows rows;
    uint32_t a_at[2], sum_at;   // per lane: of the rows it copies, of the group sums of its operand row
    // Copies columns 64 (wave / 2) .. + 63 of the operand rows 16 (wave % 2) .. + 15.
    __device__ __forceinline__ void request_rows(int wave, int kb, lds_byte *to) const {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(x[p], to + p * GEMM_PART_BYTES + (2 * wave + i) * GEMM_IMAGE, 16, (int)a_at[i], 512 * kb, 0, 0);
        asm volatile("" ::: "memory");   // what is requested from here on is younger
        __builtin_amdgcn_sched_barrier(0);
    }
    // The operand row's sums of 16 columns of a block, high and low parts; of columns that do not exist: zeros.
    __device__ __forceinline__ void request_sums16(half8v (&sums)[2], int kb, bool whole) const {
        const uint32_t mine = whole || pf_lane() < 32 ? sum_at : PF_NOWHERE;
#pragma unroll
        for (int p = 0; p < 2; p++) sums[p] = __builtin_bit_cast(half8v, __builtin_amdgcn_raw_buffer_load_b128(x[0], (int)mine, 64 * kb + 32 * p, 0));
    }
};

// One 256-block of a wave's tile.  from, to: the copies of this block's rows (at the lane's) and of the next one's.  at, head_at: the
// wave's tile in its expert's tensor, at the next block.
template <int FMT, int PARTS>
__device__ __forceinline__ void gemm_block(GemmBlock<FMT> &w, half8v &sums, const GemmSource &src, uint32_t at, uint32_t head_at, int next_kb, int wave,
                                           const lds_byte *__restrict from, lds_byte *__restrict to, const lds_byte *__restrict tables, float16v &acc) {
    const float16v zero = {0};
    src.request_rows(wave, next_kb, to);
    if constexpr (FMT == PF_Q4_K) {
        const float16v q = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, w.open(), zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = fmaf(-w.low, q[r], acc[r]);
    } else {
        w.open();
    }
    const float d = w.d;
    w.request_head(src.heads, src.rows, head_at);
    if (FMT == PF_Q4_K) sums = __builtin_bit_cast(half8v, __builtin_amdgcn_raw_buffer_load_b128(src.x[0], (int)src.sum_at, 32 * next_kb, 0));
    float16v part = zero;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        half8v x[PARTS];
#pragma unroll
        for (int p = 0; p < PARTS; p++)
            x[p] = *reinterpret_cast<const __attribute__((address_space(3))) half8v *>(from + p * GEMM_PART_BYTES + (i >> 2) * 4 * GEMM_IMAGE + GemmBlock<FMT>::chunk(i) * 128);
        const half8v b = w.operand(i, tables);
#pragma unroll
        for (int p = 0; p < PARTS; p++) part = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[p], b, part, 0, 0, 0);
        if ((i & 3) == 3) { w.request_run(i >> 2, src.weights, src.rows, at); __builtin_amdgcn_sched_barrier(0); }
    }
    lds_barrier<GemmBlock<FMT>::requests>();   // the next block's rows are there; its weights, requested after them, may not be
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = fmaf(d, part[r], acc[r]);
}

// The same for Q2_K.  whole: the block's 256 columns exist, else its first 128 (next_whole: the next block's).
template <int PARTS>
__device__ __forceinline__ void gemm_block_q2(GemmBlock<PF_Q2_K> &w, half8v (&sums)[2], const GemmSource &src, uint32_t at, uint32_t head_at, int next_kb,
                                              bool whole, bool next_whole, int wave, const lds_byte *__restrict from, lds_byte *__restrict to, float16v &acc) {
    const float16v zero = {0};
    src.request_rows(wave, next_kb, to);
    const half8v minima = w.open();
    float16v q = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[0], minima, zero, 0, 0, 0);
    q = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums[1], minima, q, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = fmaf(-w.low, q[r], acc[r]);
    const float d = w.d;
    src.request_sums16(sums, next_kb, next_whole);
    float16v part = zero;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if (half == 0 || whole) {   // (uniform)
#pragma unroll
            for (int i = 8 * half; i < 8 * half + 8; i++) {
                const half8v b = w.operand(i);
#pragma unroll
                for (int p = 0; p < PARTS; p++) {
                    const half8v x = *reinterpret_cast<const __attribute__((address_space(3))) half8v *>(from + p * GEMM_PART_BYTES + (i >> 2) * 4 * GEMM_IMAGE +
                                                                                                         GemmBlock<PF_Q2_K>::chunk(i) * 128);
                    part = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, b, part, 0, 0, 0);
                }
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    w.request_head(src.heads, src.rows, head_at);
    w.request_half(0, src.weights, src.rows, at);
    w.request_half(1, src.weights, src.rows, at);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier<GemmBlock<PF_Q2_K>::requests>();
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = fmaf(d, part[r], acc[r]);
}

// The same for Q8_0, whose groups are added up one by one, the even and the odd ones apart (a row of sums half as long); groups: 8,
// or 4 in the last block of a row of an odd number of 128 columns.
template <int PARTS>
__device__ __forceinline__ void gemm_block_q8(GemmBlock<PF_Q8_0> &w, const GemmSource &src, uint32_t at, uint32_t head_at, int next_kb, int groups, int wave,
                                              const lds_byte *__restrict from, lds_byte *__restrict to, float16v (&acc)[2]) {
    const float16v zero = {0};
    src.request_rows(wave, next_kb, to);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (2 * j < groups) {   // (uniform)
#pragma unroll
            for (int g = 2 * j; g < 2 * j + 2; g++) {
                float16v part = zero;
#pragma unroll
                for (int i = 2 * g; i < 2 * g + 2; i++) {
                    const half8v b = w.operand(i);
#pragma unroll
                    for (int p = 0; p < PARTS; p++) {
                        const half8v x = *reinterpret_cast<const __attribute__((address_space(3))) half8v *>(from + p * GEMM_PART_BYTES + j * 4 * GEMM_IMAGE +
                                                                                                             GemmBlock<PF_Q8_0>::chunk(i) * 128);
                        part = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, b, part, 0, 0, 0);
                    }
                }
                const float d = w.scale(g);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[g & 1][r] = fmaf(d, part[r], acc[g & 1][r]);
            }
        }
        w.request_run(j, src.weights, src.heads, src.rows, at, head_at);
        __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier<GemmBlock<PF_Q8_0>::requests>();
}

// The slabs [slab0, slab1) of a row tile.  PARTS = 2: high and low parts of up to 32 rows; 1: both parts of up to 16 rows as one
// 32-row operand (row 16 + m: the low part of row m).
template <int MODE, int FMT, int PARTS>
__device__ __forceinline__ void gemm_tile(const PfKernelArgs &a, const GemmItem &g, int slab0, int slab1, lds_byte *lds) {
    const int lane = pf_lane(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, h = lane >> 5;
    const int K = a.top_k, a_cols = MODE == PF_GEMM_GATE_UP ? a.hidden : g.inter, kblocks = (a_cols + 255) / 256;
    // weights: gate tiles of the first four waves, up tiles of the others; a wave beyond the matrix's last rows repeats them
    const int t = MODE == PF_GEMM_GATE_UP ? (g.shared ? 4 : 1) + (wave >> 2) : g.shared ? 6 : 3;
    const int last_tile = (MODE == PF_GEMM_GATE_UP ? g.inter : a.hidden) / 32 - 1;
    auto tile_of = [&](int slab) -> int { return MODE == PF_GEMM_GATE_UP ? 4 * slab + (wave & 3) : GW * slab + wave; };
    GemmSource src;
    src.rows = gemm_rows<FMT>(a, t, g.shared ? 0 : (size_t)g.expert);
    src.weights = pf_buffer(src.rows.base, src.rows.bytes);
    src.heads = pf_buffer(src.rows.head, src.rows.head_bytes);
    GemmBlock<FMT> w;
    {   // the first block's are on their way while the rows are looked up
        const uint32_t tile = (uint32_t)min(tile_of(slab0), last_tile);
        if constexpr (FMT == PF_Q8_0) {
#pragma unroll
            for (int j = 0; j < 4; j++) w.request_run(j, src.weights, src.heads, src.rows, tile * src.rows.tile_step, tile * src.rows.head_tile_step);
        } else {
            w.request_head(src.heads, src.rows, tile * src.rows.head_tile_step);
            if constexpr (FMT == PF_Q2_K) {
                w.request_half(0, src.weights, src.rows, tile * src.rows.tile_step);
                w.request_half(1, src.weights, src.rows, tile * src.rows.tile_step);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) w.request_run(j, src.weights, src.rows, tile * src.rows.tile_step);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // activation rows: the tile's own rows (down, and the shared expert's tokens) or gathered by token
    const bool gathered = MODE == PF_GEMM_GATE_UP && !g.shared;
    const uint32_t a_pitch = 2u * (uint32_t)(FMT == PF_Q2_K ? pf_half_row16(a_cols) : pf_half_row(a_cols));   // bytes
    const int row0 = gathered ? 0 : g.shared ? g.m0 : g.first;
    const uint8_t *base = reinterpret_cast<const uint8_t *>(MODE == PF_GEMM_GATE_UP ? a.x16 : g.shared ? a.sact16 : a.act16) + (size_t)row0 * a_pitch;
    const uint32_t bytes = gathered ? (uint32_t)min((size_t)a.token_cap * a_pitch, (size_t)PF_NOWHERE) : (uint32_t)g.rows_here * a_pitch;
    src.x[0] = pf_buffer(base, bytes);
    src.x[1] = pf_buffer(base + 2 * (size_t)a_cols, PARTS == 2 ? bytes - 2 * (uint32_t)a_cols : 0);
    const uint32_t mine = gathered ? a.row_to_pair[g.first + min(n, g.rows_here - 1)] / (uint32_t)K : (uint32_t)min(n, g.rows_here - 1);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int v = 16 * (wave & 1) + 8 * i + (lane & 7), m = PARTS == 1 ? v & 15 : v;
        const uint32_t row = __shfl(mine, m), low = PARTS == 1 && v >= 16 ? 2u * (uint32_t)a_cols : 0u;
        src.a_at[i] = m < g.rows_here ? row * a_pitch + low + 128u * (uint32_t)(wave >> 1) + 16u * (uint32_t)(lane >> 3) : PF_NOWHERE;
    }
    src.sum_at = n < g.rows_here ? mine * a_pitch + 4u * (uint32_t)a_cols + 16u * (uint32_t)h : PF_NOWHERE;
    const float scale_mine = (MODE == PF_GEMM_GATE_UP ? a.x_scale : g.shared ? a.sact_scale : a.act_scale)[row0 + (int)mine];
    src.request_rows(wave, 0, lds);
    half8v sums, sums16[2];
    auto whole = [&](int kb) { return 256 * kb + 256 <= a_cols; };   // (widths are whole halves of a block)
    if (FMT == PF_Q4_K) sums = __builtin_bit_cast(half8v, __builtin_amdgcn_raw_buffer_load_b128(src.x[0], (int)src.sum_at, 0, 0));
    if (FMT == PF_Q2_K) src.request_sums16(sums16, 0, whole(0));
    lds_barrier<0>();
    const lds_byte *take = lds + (n >> 3) * GEMM_IMAGE + GemmBlock<FMT>::chunk_h * h * 128 + (n & 7) * 16;
    float16v acc = {0}, apart[2] = {{0}, {0}};
    int copy = 0, kb = 0, slab = slab0;
    for (int left = (slab1 - slab0) * kblocks; left; left--) {
        const bool wraps = kb + 1 == kblocks;
        const int next_kb = wraps ? 0 : kb + 1;
        const uint32_t tile = (uint32_t)min(tile_of(wraps ? slab + 1 : slab), last_tile);
        if (left == 1) { src.weights = pf_buffer(src.rows.base, 0); src.heads = pf_buffer(src.rows.head, 0); }   // no block is left to request
        const uint32_t at = tile * src.rows.tile_step + (uint32_t)next_kb * src.rows.block_step;
        const uint32_t head_at = tile * src.rows.head_tile_step + (uint32_t)next_kb * src.rows.head_step;
        const lds_byte *from = take + copy * GEMM_COPY_BYTES;
        lds_byte *to = lds + (copy ^ 1) * GEMM_COPY_BYTES;
        if constexpr (FMT == PF_Q8_0) gemm_block_q8<PARTS>(w, src, at, head_at, next_kb, min(8, (a_cols - 256 * kb) / 32), wave, from, to, apart);
        else if constexpr (FMT == PF_Q2_K) gemm_block_q2<PARTS>(w, sums16, src, at, head_at, next_kb, whole(kb), whole(next_kb), wave, from, to, acc);
        else gemm_block<FMT, PARTS>(w, sums, src, at, head_at, next_kb, wave, from, to, lds + IQ2_GRID_OFF, acc);
        copy ^= 1;
        kb = next_kb;
        if (!wraps) continue;
        // epilogue: the lane holds column n of its tile; register r is row 8 (r / 4) + 4 h + r % 4
        constexpr int REGS = 8 * PARTS;
        if (FMT == PF_Q8_0) {
#pragma unroll
            for (int r = 0; r < 16; r++) { acc[r] = apart[0][r] + apart[1][r]; apart[0][r] = apart[1][r] = 0.0f; }
        }
        const bool exist = tile_of(slab) <= last_tile;
        int row_in_4 = 4 * h, col = n;
        asm volatile("" : "+v"(row_in_4), "+v"(col));   // what follows from them is formed here, not kept in registers through the products
        float v[REGS];
#pragma unroll
        for (int r = 0; r < REGS; r++) v[r] = (PARTS == 1 ? acc[r] + acc[r + 8] : acc[r]) * __shfl(scale_mine, 8 * (r >> 2) + row_in_4 + (r & 3));
        if (MODE == PF_GEMM_GATE_UP) {   // (one slab) the gate waves hand their rows to the up waves through LDS
            __attribute__((address_space(3))) float *meet = reinterpret_cast<__attribute__((address_space(3))) float *>(lds) + (wave & 3) * 1024 + lane;
            if (wave < 4) {
#pragma unroll
                for (int r = 0; r < REGS; r++) meet[64 * r] = pf_silu(v[r]);
            }
            lds_barrier<0>();
            if (wave < 4 || !exist) return;
            float *out = (g.shared ? a.shared_act + (size_t)g.m0 * g.inter : a.act + (size_t)g.first * g.inter) + 32 * tile_of(slab) + col;
#pragma unroll
            for (int r = 0; r < REGS; r++) {
                const int m = 8 * (r >> 2) + row_in_4 + (r & 3);
                if (m < g.rows_here) out[(size_t)m * g.inter] = meet[64 * r] * v[r];
            }
            return;
        }
        float *out = a.down + (size_t)g.first * a.hidden + 32 * tile_of(slab) + col;
#pragma unroll
        for (int r = 0; r < REGS; r++) {
            const int m = 8 * (r >> 2) + row_in_4 + (r & 3);
            if (m < g.rows_here && exist) out[(size_t)m * a.hidden] = v[r];
        }
        acc = float16v{0};
        slab++;
    }
}

// FMT, SHARED: the routed tensors' format and the shared expert's.  slabs: workgroups that share a row tile; per: slabs that each of
// them takes (gate and up: one); shift: of the groups of tiles; shared_tiles: the shared expert's; only_shared: of them alone.
template <int MODE, int FMT, int SHARED>
__global__ void __launch_bounds__(64 * GW, 4) pf_k_pf_gemm(PfKernelArgs a, int slabs, int per, int shift, uint32_t shared_tiles, int only_shared) {
    extern __shared__ __align__(16) unsigned char gemm_lds[];
    GemmItem g;
    int slab;
    const uint32_t routed = a.tiles[0] - shared_tiles;
    if (!gemm_item(a, slabs, shift, blockIdx.x, only_shared ? 0 : routed, shared_tiles, only_shared ? routed : 0, g, slab)) return;
    if (a.type[MODE == PF_GEMM_GATE_UP ? (g.shared ? 4 : 1) : (g.shared ? 6 : 3)] != (uint32_t)(g.shared ? SHARED : FMT)) return;   // the plain kernel's
    const int width = MODE == PF_GEMM_GATE_UP ? 16 * GW : 32 * GW, all = ((MODE == PF_GEMM_GATE_UP ? g.inter : a.hidden) + width - 1) / width;
    const int slab0 = slab * per, slab1 = min(slab0 + per, all);
    if (slab0 >= slab1) return;
    if (FMT == PF_IQ2_XXS && (SHARED == FMT || !g.shared)) {
        // grid magnitudes, and for every 7-bit sign field the sign bytes of its eight weights (the eighth sign makes the number of
        // negative weights even)
        if (threadIdx.x < 256) reinterpret_cast<uint64_t *>(gemm_lds + IQ2_GRID_OFF)[threadIdx.x] = a.iq2_grid[threadIdx.x];
        else if (threadIdx.x < 384) {
            const uint32_t s7 = threadIdx.x - 256, s8 = s7 | ((__popc(s7) & 1u) << 7);
            // bit b of s8 -> bit 7 of byte b: four bits spread to the bytes of a word
            auto spread = [](uint32_t four) { return ((four * 0x00204081u) & 0x01010101u) << 7; };
            reinterpret_cast<uint2 *>(gemm_lds + IQ2_SIGN_OFF)[s7] = make_uint2(spread(s8 & 15u), spread(s8 >> 4));
        }
    }
    // by the expert's rows, not the tile's: which of them a tile holds differs from run to run, and the two add up in another order
    lds_byte *lds = (lds_byte *)gemm_lds;
    const bool narrow = g.m0 == 0 && g.rows_here <= 16;
    if (SHARED != FMT && g.shared) {
        if (narrow) gemm_tile<MODE, SHARED, 1>(a, g, slab0, slab1, lds);
        else gemm_tile<MODE, SHARED, 2>(a, g, slab0, slab1, lds);
        return;
    }
    if (narrow) gemm_tile<MODE, FMT, 1>(a, g, slab0, slab1, lds);
    else gemm_tile<MODE, FMT, 2>(a, g, slab0, slab1, lds);
}

// Histogram of the routed pairs.  counts[] is zero on entry: the workspace starts zeroed and
// pf_k_pf_scan_tiles clears it again once it has been read.
__global__ void pf_k_pf_count(const uint32_t *ids, int pairs, int E, uint32_t *counts) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < pairs && ids[p] < (uint32_t)E) atomicAdd(&counts[ids[p]], 1u);
}

// One workgroup: exclusive scan of counts[E] into offsets[E + 1], and the row tiles: every
// expert's rows (the shared expert = expert E with all tokens) cut into tiles of 32; tiles[0] =
// count, tiles[1 + i] = expert | (tile index within the expert) << 16, items[i] = {expert, first row, rows, first row
// within the expert}.  Leaves counts[] zero.
__global__ void __launch_bounds__(256) pf_k_pf_scan_tiles(uint32_t *counts, int E, int tokens, uint32_t *offsets,
                                                          uint32_t *tiles, uint4 *items) {
    __shared__ uint32_t rows_before[256], tiles_before[256];
    const int tid = threadIdx.x, per = (E + 1 + 255) / 256, lo = tid * per, hi = min(E + 1, lo + per);
    uint32_t rows = 0, ntiles = 0;
    for (int e = lo; e < hi; e++) {
        const uint32_t c = e < E ? counts[e] : (uint32_t)tokens;
        if (e < E) rows += c;
        ntiles += (c + 31u) / 32u;
    }
    rows_before[tid] = rows;
    tiles_before[tid] = ntiles;
    __syncthreads();
    // inclusive scan of the 256 partial sums in eight doubling steps, then made exclusive
    uint32_t run_rows = rows, run_tiles = ntiles;
    for (int d = 1; d < 256; d <<= 1) {
        const uint32_t add_rows = tid >= d ? rows_before[tid - d] : 0u, add_tiles = tid >= d ? tiles_before[tid - d] : 0u;
        __syncthreads();
        run_rows += add_rows;
        run_tiles += add_tiles;
        rows_before[tid] = run_rows;
        tiles_before[tid] = run_tiles;
        __syncthreads();
    }
    if (tid == 255) {
        offsets[E] = run_rows;
        tiles[0] = run_tiles;
    }
    __syncthreads();
    rows_before[tid] = run_rows - rows;
    tiles_before[tid] = run_tiles - ntiles;
    uint32_t row = rows_before[tid], at = tiles_before[tid];
    for (int e = lo; e < hi; e++) {
        const uint32_t c = e < E ? counts[e] : (uint32_t)tokens, n = (c + 31u) / 32u;
        for (uint32_t i = 0; i < n; i++) {
            tiles[1 + at + i] = (uint32_t)e | (i << 16);
            items[at + i] = make_uint4((uint32_t)e, row + 32u * i, min(32u, c - 32u * i), 32u * i);
        }
        if (e < E) {
            offsets[e] = row;
            row += c;
            counts[e] = 0;
        }
        at += n;
    }
}

// ---- the grouped product for the other formats of real checkpoints --------------------------------
// Q2_K, and MXFP4 and Q8_0 where the kernels made for them do not apply, have no operand path in the kernel
// above.  This kernel computes the same items with the same operands' arithmetic (exact
// integer weight operands in fp16, two-part fp16 activations, FP32 accumulation, scales applied to
// the partial sums in FP32): a workgroup is one row tile against one slab
// of 4 x 32 (gate/up) or 4 x 64 (down) weight rows, a wave takes its operands straight from global
// memory (the activation fragments are shared through the caches by the four waves and the slabs).
// Group scales that are not integers (Q8_0: a half per 32 weights; MXFP4: a power of two per 32)
// multiply the group's partial sums; Q2_K folds its 4-bit scale into the operand (scale * code
// <= 45) and obtains sum(min * x) from a second product with the minimum as the operand, as
// d * P - dmin * Q per 256-block.

// Eight E2M1 codes (one per byte of two dwords, in the low nibble) as halfs holding twice their value:
// 0, 1, 2, 3, 4, 6, 8, 12 are 0x0000, 0x3C00, 0x4000, 0x4200, 0x4400, 0x4600, 0x4800, 0x4A00, so a byte
// permute looks up the halfs' high bytes, bit 3 of the code becomes the sign bit, and two more permutes
// spread the four bytes over two pairs of halfs (selector 0x0C writes a zero byte).
__device__ __forceinline__ half8v half8_of_e2m1(uint32_t n0, uint32_t n1) {
    auto pairs = [](uint32_t n, uint32_t &lo, uint32_t &hi) {
        uint32_t top = __builtin_amdgcn_perm(0x4A484644u, 0x42403C00u, n & 0x07070707u);
        top |= (n << 4) & 0x80808080u;
        lo = __builtin_amdgcn_perm(0u, top, 0x010C000Cu);
        hi = __builtin_amdgcn_perm(0u, top, 0x030C020Cu);
    };
    uint4 bits;
    pairs(n0, bits.x, bits.y);
    pairs(n1, bits.z, bits.w);
    return __builtin_bit_cast(half8v, bits);
}

struct PlainRow {            // one weight row as the kernel reads it
    const uint8_t *payload;  // first byte of the row (device layout of its format)
    const uint8_t *scales;   // first scale of the row, for the formats stored split
};

__device__ __forceinline__ PlainRow plain_row(const PfKernelArgs &a, int t, size_t e, size_t row) {
    const size_t index = e * a.n_out[t] + row;
    PlainRow r;
    r.payload = a.w[t] + index * a.row_bytes[t];
    r.scales = a.w[t] + a.scale_offset[t] + index * a.blocks_per_row[t] * (a.type[t] == PF_MXFP4 ? 1 : 2);
    return r;
}

// One batch of a wave's two weight rows: the bytes of 128 columns (Q2_K: of a 256-block), as they were loaded.  The kernel
// requests a batch while it multiplies the one before, across the passes too: without that a wave waited for memory once a
// batch, about twice as long as the products of a batch take, with two waves a SIMD to cover for one another (MXFP4 down launch of a
// 2048-token chunk at the checkpoints' widths 497 -> 412 us, Q2_K, 1024 tokens, 315 -> 293 us).
template <int FMT, int S> struct PlainBatch;
template <int S> struct PlainBatch<PF_Q8_0, S> {
    static constexpr int COLS = 128;
    uint2 q[S][4][2], scales[S];   // [row][group][half of its columns]; four half scales
    __device__ __forceinline__ void load(const PlainRow (&r)[S], int batch, int h) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            scales[s] = *reinterpret_cast<const uint2 *>(r[s].scales + 8 * (size_t)batch);
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int t = 0; t < 2; t++) q[s][g][t] = *reinterpret_cast<const uint2 *>(r[s].payload + 32 * (size_t)(4 * batch + g) + 16 * t + 8 * h);
        }
    }
    __device__ __forceinline__ float scale(int s, int g) const {
        const uint32_t two = g < 2 ? scales[s].x : scales[s].y;
        return (float)__builtin_bit_cast(half_t, (unsigned short)((g & 1) ? two >> 16 : two & 0xffffu));
    }
    __device__ __forceinline__ half8v operand(int s, int g, int t) const { return half8_of_signed_bytes(q[s][g][t].x, q[s][g][t].y); }
};
template <int S> struct PlainBatch<PF_MXFP4, S> {   // bytes 8h..8h+7 of a block: low nibbles values 8h.., high nibbles values 16 + 8h..
    static constexpr int COLS = 128;
    uint2 q[S][4];
    uint32_t scales[S];
    __device__ __forceinline__ void load(const PlainRow (&r)[S], int batch, int h) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            scales[s] = *reinterpret_cast<const uint32_t *>(r[s].scales + 4 * (size_t)batch);
#pragma unroll
            for (int g = 0; g < 4; g++) q[s][g] = *reinterpret_cast<const uint2 *>(r[s].payload + 16 * (size_t)(4 * batch + g) + 8 * h);
        }
    }
    __device__ __forceinline__ float scale(int s, int g) const { return 0.5f * pf_e8m0_scale((scales[s] >> (8 * g)) & 255u); }   // the operands are twice the values
    __device__ __forceinline__ half8v operand(int s, int g, int t) const {
        return half8_of_e2m1((q[s][g].x >> (4 * t)) & 0x0F0F0F0Fu, (q[s][g].y >> (4 * t)) & 0x0F0F0F0Fu);
    }
};
template <int S> struct PlainBatch<PF_Q2_K, S> {
    static constexpr int COLS = 256;
    uint32_t codes[S][2][2][2], scales[S][4], dd[S];   // [row][half of the block][sub-group of 16][dword]
    __device__ __forceinline__ void load(const PlainRow (&r)[S], int batch, int h) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            const uint32_t *block = reinterpret_cast<const uint32_t *>(r[s].payload + 84 * (size_t)batch);   // 4-byte aligned
            dd[s] = block[20];
#pragma unroll
            for (int k = 0; k < 4; k++) scales[s][k] = block[k];
#pragma unroll
            for (int half = 0; half < 2; half++)
#pragma unroll
                for (int k = 0; k < 4; k++) codes[s][half][k >> 1][k & 1] = block[4 + 8 * half + 2 * h + 4 * (k >> 1) + (k & 1)];
        }
    }
};

// acc[row] += the staged activation columns of the batch (local columns k0..) x the batch.  ahi / alo: this lane's activation
// row in LDS (high and low parts); sums: the row's sums over every 16 staged columns (high parts, low parts sums_low further
// on; Q2_K only); cols: staged columns.
template <int FMT, int S>
__device__ __forceinline__ void plain_product(const PlainBatch<FMT, S> &w, const half_t *ahi, const half_t *alo, const half_t *, int, int k0, int, int h,
                                              float16v (&acc)[S]) {
    const float16v zero = {0};
#pragma unroll
    for (int g = 0; g < 4; g++) {
        float16v part[S];
#pragma unroll
        for (int s = 0; s < S; s++) part[s] = zero;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int k = k0 + 32 * g + 16 * t + 8 * h;
            const half8v xh = *reinterpret_cast<const half8v *>(ahi + k), xl = *reinterpret_cast<const half8v *>(alo + k);
#pragma unroll
            for (int s = 0; s < S; s++) {
                const half8v v = w.operand(s, g, t);
                part[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, v, part[s], 0, 0, 0);
                part[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, v, part[s], 0, 0, 0);
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
            const float scale = w.scale(s, g);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[s][r] = fmaf(scale, part[s][r], acc[s][r]);
        }
    }
}
template <int S>
__device__ __forceinline__ void plain_product(const PlainBatch<PF_Q2_K, S> &w, const half_t *ahi, const half_t *alo, const half_t *sums, int sums_low,
                                                       int k0, int cols, int h, float16v (&acc)[S]) {
    // a row's last block may be half used (logical width 640 of 768 stored): its second half is skipped, and the sums of the
    // groups beyond the width are zero
    const float16v zero = {0};
    float16v part[S], low[S];
#pragma unroll
    for (int s = 0; s < S; s++) part[s] = zero;
    // Q: the 16 groups' minima (scale bytes 8h..8h+7, high nibbles) against the rows' sums over the same groups
    const half8v sh = *reinterpret_cast<const half8v *>(sums + k0 / 16 + 8 * h), sl = *reinterpret_cast<const half8v *>(sums + sums_low + k0 / 16 + 8 * h);
#pragma unroll
    for (int s = 0; s < S; s++) {
        const uint32_t m0 = h ? w.scales[s][2] : w.scales[s][0], m1 = h ? w.scales[s][3] : w.scales[s][1];
        const half8v mv = half8_of_bytes((m0 >> 4) & 0x0F0F0F0Fu, (m1 >> 4) & 0x0F0F0F0Fu, (half_t)1024.0f);
        low[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sh, mv, zero, 0, 0, 0);
        low[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sl, mv, low[s], 0, 0, 0);
    }
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if (k0 + 128 * half >= cols) break;
#pragma unroll
        for (int j = 0; j < 8; j++) {   // groups of 16 weights
            const int gi = 8 * half + j, k = k0 + 16 * gi + 8 * h;
            const half8v xh = *reinterpret_cast<const half8v *>(ahi + k), xl = *reinterpret_cast<const half8v *>(alo + k);
#pragma unroll
            for (int s = 0; s < S; s++) {
                // byte-wise scale * code: at most 15 * 3, no carry between bytes
                const uint32_t f = (w.scales[s][gi >> 2] >> (8 * (gi & 3))) & 15u, *c = w.codes[s][half][j & 1];
                const half8v v = half8_of_bytes(((c[0] >> (2 * (j >> 1))) & 0x03030303u) * f, ((c[1] >> (2 * (j >> 1))) & 0x03030303u) * f, (half_t)1024.0f);
                part[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, v, part[s], 0, 0, 0);
                part[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, v, part[s], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < S; s++) {
        const half2v dm = __builtin_bit_cast(half2v, w.dd[s]);
        const float d = (float)dm.x, n = (float)dm.y;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[s][r] = fmaf(d, part[s][r], fmaf(-n, low[s][r], acc[s][r]));
    }
}

#define PLAIN_CHUNK PF_PLAIN_CHUNK          // activation columns staged per pass (256, three workgroups a compute unit: slower)
#define PLAIN_PITCH (PLAIN_CHUNK + 8)       // halfs between staged rows: 16 bytes of padding spread the rows over the banks
#define PLAIN_SUMS (PLAIN_CHUNK / 16 + 8)   // halfs between the rows' sums over 16 columns
#define PLAIN_TILE_BYTES (2 * 32 * PLAIN_PITCH * 2)
#define PLAIN_LDS (PLAIN_TILE_BYTES + 2 * 32 * PLAIN_SUMS * 2)

// Stages PLAIN_CHUNK columns of the tile's 32 activation rows (high and low parts), one 1 KB row part per load instruction, and
// multiplies them, pass after pass (pf_plain_walk.h).  A wave takes every `parts`-th batch of the row starting with batch
// `part`: with parts > 1 the waves of a workgroup share one pair of rows and their partial sums are added afterwards.
struct PlainTile { half_t *tile, *sums; const half_t *a16; const uint32_t *src_row; int a_cols; };
template <int FMT, int S>
__device__ __forceinline__ void plain_passes(const PlainTile &a, const PlainRow (&rows)[S], bool active, int part, int parts, float16v (&acc)[S]) {
    typedef PlainBatch<FMT, S> Batch;
    const int lane = pf_lane(), wave = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    const half_t *ahi = a.tile + (size_t)n * PLAIN_PITCH, *alo = ahi + 32 * PLAIN_PITCH;
    Batch w, next;
    auto stage = [&](int c0, int cols) {
        if (c0) __syncthreads();   // the previous pass has been consumed
        // 64 row parts (32 rows, high and low) over the four waves; a lane moves 16 bytes of each
#pragma unroll 4
        for (int i = 0; i < 16; i++) {
            const int row_part = 16 * wave + i, row = row_part & 31, low = row_part >> 5;
            if (16 * lane < 2 * cols)
                to_lds(a.a16 + (size_t)a.src_row[row] * pf_half_row(a.a_cols) + (size_t)low * a.a_cols + c0 + 8 * lane,
                       reinterpret_cast<unsigned char *>(a.tile + ((size_t)low * 32 + row) * PLAIN_PITCH));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (FMT == PF_Q2_K) {
            // sums of the staged rows over every 16 columns, as two-part halfs like the values themselves:
            // thread = (row, four neighbouring groups)
            const int row = threadIdx.x >> 3, g0 = 4 * (threadIdx.x & 7);
#pragma unroll
            for (int g = g0; g < g0 + 4; g++) {
                float total = 0.0f;
                if (16 * g < cols) {
                    const half_t *hi = a.tile + (size_t)row * PLAIN_PITCH + 16 * g, *lo = hi + 32 * PLAIN_PITCH;
                    const half8v a0 = *reinterpret_cast<const half8v *>(hi), a1 = *reinterpret_cast<const half8v *>(hi + 8);
                    const half8v b0 = *reinterpret_cast<const half8v *>(lo), b1 = *reinterpret_cast<const half8v *>(lo + 8);
#pragma unroll
                    for (int i = 0; i < 8; i++) total += ((float)a0[i] + (float)b0[i]) + ((float)a1[i] + (float)b1[i]);
                }
                const half_t top = (half_t)total;
                a.sums[(size_t)row * PLAIN_SUMS + g] = top;
                a.sums[(size_t)(32 + row) * PLAIN_SUMS + g] = (half_t)(total - (float)top);
            }
            __syncthreads();
        }
    };
    pf_plain_walk(a.a_cols, Batch::COLS, part, parts, active, stage, [&](int batch) { next.load(rows, batch, h); }, [&] { w = next; },
                  [&](int k0, int cols) { plain_product(w, ahi, alo, a.sums + (size_t)n * PLAIN_SUMS, 32 * PLAIN_SUMS, k0, cols, h, acc); });
}

// which: all items of the list, or the shared expert's (the grid: its tiles alone).
enum { PLAIN_ALL, PLAIN_SHARED };

// grid: (row tiles the list can hold) x slabs; 4 waves.  Items whose tensors are in a format of pf_k_pf_gemm
// are skipped here, as that kernel skips these.
// split != 0 (gate/up only): the four waves share 32 units and take a quarter of the columns each; their
// partial sums meet in LDS and wave 0 adds them in wave order.  For matrices with few row tiles (the
// shared expert) that gives four times as many workgroups.
template <int MODE>
__global__ void __launch_bounds__(256) pf_k_pf_gemm_plain(PfKernelArgs a, int tokens, int slabs, int split, int which) {
    extern __shared__ __align__(16) unsigned char plain_lds[];
    __shared__ uint32_t src_row[32];
    __shared__ float src_scale[32];
    half_t *tile = reinterpret_cast<half_t *>(plain_lds), *sums = reinterpret_cast<half_t *>(plain_lds + PLAIN_TILE_BYTES);
    const int lane = pf_lane(), wave = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    const int E = a.experts, K = a.top_k, P = tokens * K;
    const uint32_t all = a.tiles[0], slab = blockIdx.x % slabs;
    const uint32_t item_tile = blockIdx.x / slabs + (which == PLAIN_SHARED ? all - (uint32_t)((tokens + 31) / 32) : 0u);   // the shared expert's tiles are the list's last
    if (item_tile >= all) return;
    const uint32_t entry = a.tiles[1 + item_tile];
    const int expert = entry & 0xffffu, m0 = 32 * (int)(entry >> 16);
    const bool shared = expert == E;
    const int first = shared ? P : (int)a.offsets[expert];
    const int count = shared ? tokens : (int)a.offsets[expert + 1] - first;
    if (count <= m0) return;
    const int rows_here = min(32, count - m0), inter = shared ? a.shared_inter : a.inter;
    const size_t ex = shared ? 0 : (size_t)expert;
    const int t0 = MODE == PF_GEMM_GATE_UP ? (shared ? 4 : 1) : (shared ? 6 : 3);
    const uint32_t fmt = a.type[t0];
    if (fmt != PF_Q8_0 && fmt != PF_Q2_K && fmt != PF_MXFP4) return;
    constexpr int S = 2;   // 32-row tiles of a wave: a gate tile and the up tile of the same units, or two down tiles (four: one wave a SIMD, slower)
    const int slab_rows = MODE != PF_GEMM_GATE_UP ? 128 * S : split ? 32 : 128, limit = MODE == PF_GEMM_GATE_UP ? inter : a.hidden;
    const int row0 = MODE == PF_GEMM_GATE_UP ? slab_rows * (int)slab + (split ? 0 : 32 * wave) + n : slab_rows * (int)slab + 32 * S * wave + n;
    if (slab_rows * (int)slab >= limit) return;   // the slab starts beyond the matrix: the whole workgroup
    const bool active = row0 - n < limit;        // this wave has rows (the others stay for the barriers)
    const int part = split ? wave : 0, parts = split ? 4 : 1;
    // the tile's activation rows (the all-zero row beyond the tile's last) and their scales
    const int a_cols = MODE == PF_GEMM_GATE_UP ? a.hidden : inter;
    const half_t *a16 = reinterpret_cast<const half_t *>(MODE == PF_GEMM_GATE_UP ? a.x16 : shared ? a.sact16 : a.act16);
    const float *a_scale = MODE == PF_GEMM_GATE_UP ? a.x_scale : shared ? a.sact_scale : a.act_scale;
    if (threadIdx.x < 32) {
        const int m = threadIdx.x;
        uint32_t src;
        if (m >= rows_here) src = MODE == PF_GEMM_GATE_UP || shared ? a.token_cap : a.token_cap * (uint32_t)K;
        else if (shared) src = (uint32_t)(m0 + m);
        else src = MODE == PF_GEMM_GATE_UP ? a.row_to_pair[first + m0 + m] / (uint32_t)K : (uint32_t)(first + m0 + m);
        src_row[m] = src;
        src_scale[m] = m < rows_here ? a_scale[src] : 0.0f;
    }
    __syncthreads();
    PlainRow rows[S];
#pragma unroll
    for (int q = 0; q < S; q++)
        rows[q] = MODE == PF_GEMM_GATE_UP ? plain_row(a, t0 + q, ex, min(row0, limit - 1)) : plain_row(a, t0, ex, min(row0 + 32 * q, limit - 1));
    const PlainTile staged = {tile, sums, a16, src_row, a_cols};
    float16v acc[S];
#pragma unroll
    for (int q = 0; q < S; q++) acc[q] = float16v{0};
    if (fmt == PF_Q8_0) plain_passes<PF_Q8_0, S>(staged, rows, active, part, parts, acc);
    else if (fmt == PF_MXFP4) plain_passes<PF_MXFP4, S>(staged, rows, active, part, parts, acc);
    else plain_passes<PF_Q2_K, S>(staged, rows, active, part, parts, acc);
    if (split) {   // every wave is active here: the partial sums of waves 1..3 go through LDS (over the staged columns)
        __syncthreads();
        float *partial = reinterpret_cast<float *>(plain_lds);
        if (wave) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                partial[((wave - 1) * 32 + r) * 64 + lane] = acc[0][r];
                partial[((wave - 1) * 32 + 16 + r) * 64 + lane] = acc[1][r];
            }
        }
        __syncthreads();
        if (wave) return;
#pragma unroll
        for (int w = 0; w < 3; w++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[0][r] += partial[(w * 32 + r) * 64 + lane];
                acc[1][r] += partial[(w * 32 + 16 + r) * 64 + lane];
            }
        }
    }
    if (!active) return;
    // epilogue: the lane holds column n of its tiles; register r is row 8 (r / 4) + 4 h + r % 4
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int m = 8 * (r >> 2) + 4 * h + (r & 3);
        if (m >= rows_here) continue;
        const float rs = src_scale[m];
        if (MODE == PF_GEMM_GATE_UP) {
            if (row0 >= limit) continue;
            const float v = pf_silu(acc[0][r] * rs) * (acc[1][r] * rs);
            if (shared) a.shared_act[(size_t)(m0 + m) * inter + row0] = v;
            else a.act[(size_t)(first + m0 + m) * inter + row0] = v;
        } else {
            float *out = a.down + (size_t)(first + m0 + m) * a.hidden;
#pragma unroll
            for (int q = 0; q < S; q++) if (row0 + 32 * q < limit) out[row0 + 32 * q] = acc[q][r] * rs;
        }
    }
}

// ---- combine ---------------------------------------------------------------------------------------
// y[t] = sum over slots in order of weight * down row, then + sigmoid * shared down row.  Bound by HBM; with the streams'
// update 400 MB at 2048 tokens of 2560 x 10 slots, 80 us (4-byte accesses to the streams: 97).
// (src/qwen4_moe.c:362-372)
__global__ void __launch_bounds__(PF_ROW_THREADS) pf_k_pf_combine(PfKernelArgs a, int tokens) {
    const int t = blockIdx.x, H = a.hidden, K = a.top_k, P = tokens * K;
    __shared__ uint32_t rows[64];
    __shared__ float weights[64];
    if ((int)threadIdx.x < K) {
        rows[threadIdx.x] = a.pair_to_row[(size_t)t * K + threadIdx.x];
        weights[threadIdx.x] = a.route_weights[(size_t)t * K + threadIdx.x];
    }
    __syncthreads();
    const float ss = a.shared_scale[t];
    const bool quads = pf_output_quads(a);
    bool bad = false;
    // four columns a thread; the rows of sixteen slots at a time are all requested before the first of their sums
    for (int c = 4 * threadIdx.x; c < H; c += 4 * blockDim.x) {
        PfOutputQuad before;
        pf_output_quad_prefetch(a, t, c, quads, before);
        const float4 sh = *reinterpret_cast<const float4 *>(a.down + (size_t)(P + t) * H + c);
        float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int s0 = 0; s0 < K; s0 += 16) {
            float4 v[16];
#pragma unroll
            for (int s = 0; s < 16; s++)
                if (s0 + s < K) v[s] = *reinterpret_cast<const float4 *>(a.down + (size_t)rows[s0 + s] * H + c);
#pragma unroll
            for (int s = 0; s < 16; s++) {
                if (s0 + s < K) {
                    const float w = weights[s0 + s];
                    sum[0] += w * v[s].x; sum[1] += w * v[s].y; sum[2] += w * v[s].z; sum[3] += w * v[s].w;
                }
            }
        }
        const float4 y = make_float4(sum[0] + ss * sh.x, sum[1] + ss * sh.y, sum[2] + ss * sh.z, sum[3] + ss * sh.w);
        bad |= !pf_output_quad_commit(a, t, c, quads, y, before);
    }
    if (__any(bad) && pf_lane() == 0) atomicOr(a.error_word, PF_HIP_ERR_NONFINITE);
}

// ---- dispatch --------------------------------------------------------------------------------------
// Routed gate and up in Q4_K or IQ2_XXS (pf_k_pf_gemm's operand paths); the routed down tensor and the
// shared expert's three tensors in that same format or in Q2_K, MXFP4, Q8_0.
bool pf_prefill_supported(const PfHipMoeDesc &d) {
    const uint32_t g = d.type[1];
    auto covered = [&](uint32_t t) { return t == g || t == PF_Q8_0 || t == PF_Q2_K || t == PF_MXFP4; };
    if ((g != PF_Q4_K && g != PF_IQ2_XXS) || d.type[2] != g || !covered(d.type[3])) return false;
    if (d.type[5] != d.type[4] || !covered(d.type[4]) || !covered(d.type[6])) return false;
    // widths: whole 256-blocks where pf_k_pf_gemm reads the gate's format; where the plain kernel takes a down projection, whole
    // 128-column halves (the checkpoints' 640), and only Q2_K may be stored wider than its logical width
    auto width_ok = [&](uint32_t type, uint32_t k) { return k % (type == g ? 256u : 128u) == 0; };
    if (d.hidden % 256 || d.inter % 32 || d.shared_inter % 32 || !width_ok(d.type[3], d.inter) || !width_ok(d.type[6], d.shared_inter))
        return false;
    if (d.down_physical < d.inter || (d.down_physical != d.inter && d.type[3] != PF_Q2_K) ||
        (d.type[3] == PF_Q2_K && d.down_physical % 256))
        return false;
    if (d.top_k > 64 || d.top_k >= d.experts || d.experts >= 65535) return false;
    if ((size_t)d.hidden * (d.inter > d.shared_inter ? d.inter : d.shared_inter) > PF_NOWHERE || pf_prefill_most_tokens((int)d.hidden) == 0)
        return false;   // one expert's tensor, one token's row by 32-bit offsets
    return true;
}

// A Q2_K down projection beside a Q8_0 shared expert's on pf_k_pf_gemm: activation rows that the conversion holds in registers (at most
// 1024 values).  The others are the plain kernel's, 1.3 to 1.5 times slower.
static bool pf_q2_down(const uint32_t *type, int inter, int shared_inter) {
    return type[3] == PF_Q2_K && type[6] == PF_Q8_0 && inter <= 1024 && shared_inter <= 1024;
}
size_t pf_prefill_half_row(int cols) { return pf_half_row(cols); }
size_t pf_prefill_act_row(const PfHipMoeDesc &d) {
    return pf_q2_down(d.type, (int)d.inter, (int)d.shared_inter) ? pf_half_row16((int)d.inter) : pf_half_row((int)d.inter);
}
size_t pf_prefill_most_tokens(int hidden) { return PF_NOWHERE / (2 * pf_half_row(hidden)) / 32 * 32; }
// sum over experts of ceil(rows / 32) <= pairs / 32 + experts, plus the shared expert's tiles
int pf_prefill_max_tiles(int tokens, int experts, int top_k) {
    return (int)(((size_t)tokens * top_k) / 32 + experts + (tokens + 31) / 32 + 1);
}

// The tile list's length is only known on the device: a workgroup beyond it ends at once.  routed_cap: routed row tiles, at most (0: the
// shared expert's only, one slab a workgroup, they are few).
template <int MODE, int FMT, int SHARED>
static void launch_gemm(const PfKernelArgs &a, int tokens, unsigned routed_cap, int width, int cols, hipStream_t stream) {
    const size_t lds = FMT == PF_IQ2_XXS ? GEMM_LDS_IQ2 : GEMM_LDS;
    static const bool configured = hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_pf_gemm<MODE, FMT, SHARED>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)lds) == hipSuccess;   // more than the default 64 KB
    (void)configured;
    const int rows = MODE == PF_GEMM_GATE_UP ? 16 * GW : 32 * GW, all = (width + rows - 1) / rows;
    const unsigned shared = (unsigned)(tokens + 31) / 32;
    const int per = MODE == PF_GEMM_GATE_UP || !routed_cap ? 1 : pf_slabs_each(all, max(1, 8 / max(1, cols / 256)), routed_cap + shared);
    const int slabs = (all + per - 1) / per;
    const int shift = pf_group_shift(routed_cap);
    hipLaunchKernelGGL((pf_k_pf_gemm<MODE, FMT, SHARED>), dim3(pf_item_numbers(slabs, shift, routed_cap, shared)), dim3(64 * GW), lds, stream, a, slabs, per,
                       shift, shared, routed_cap ? 0 : 1);
}

template <int MODE>
static void launch_gemm_plain(const PfKernelArgs &a, int tokens, unsigned tile_cap, int slabs, int split, int which, hipStream_t stream) {
    static bool configured = false;   // once per instantiation: more than the default 64 KB of dynamic LDS
    if (!configured) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_pf_gemm_plain<MODE>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, PLAIN_LDS);
        configured = true;
    }
    hipLaunchKernelGGL(pf_k_pf_gemm_plain<MODE>, dim3(tile_cap * slabs), dim3(256), PLAIN_LDS, stream, a, tokens, slabs, split, which);
}

// the pairs by expert: offsets, row tiles, pair <-> row
void pf_launch_group(const PfKernelArgs &a, const uint32_t *ids, int tokens, hipStream_t stream) {
    const int E = a.experts, P = tokens * a.top_k;
    if (pf_launch_group_fused(ids, P, E, tokens, a.offsets, a.tiles, const_cast<uint32_t *>(a.items), a.pair_to_row, a.row_to_pair, stream)) return;
    hipLaunchKernelGGL(pf_k_pf_count, dim3((P + 255) / 256), dim3(256), 0, stream, ids, P, E, a.counts);
    hipLaunchKernelGGL(pf_k_pf_scan_tiles, dim3(1), dim3(256), 0, stream, a.counts, E, tokens, a.offsets, a.tiles,
                       reinterpret_cast<uint4 *>(const_cast<uint32_t *>(a.items)));
    pf_launch_group_place(ids, P, E, a.offsets, a.pair_to_row, a.row_to_pair, stream);
}
void pf_launch_combine(const PfKernelArgs &a, int tokens, hipStream_t stream) {
    hipLaunchKernelGGL(pf_k_pf_combine, dim3(tokens), dim3(pf_row_threads((unsigned)a.hidden / 4)), 0, stream, a, tokens);
}

void pf_launch_prefill(const PfKernelArgs &a, int tokens, hipStream_t stream, int stage_limit) {
    const int H = a.hidden, E = a.experts, K = a.top_k, I = a.inter, Is = a.shared_inter, P = tokens * K;
    const int last = stage_limit ? stage_limit : 4;
    // stage 1: router logits
    // the tile whose rounds over the chip are the least matrix work, the larger of two equal ones (it reads less per product)
    auto work = [&](int tr, int tc) {
        const long tiles = (long)((tokens + 32 * tr - 1) / (32 * tr)) * ((E + 32 * tc - 1) / (32 * tc));
        return (tiles + 255) / 256 * tr * tc;
    };
    if (work(2, 2) <= work(1, 2) && work(2, 2) <= work(1, 1)) launch_router<2, 2>(a, tokens, stream);
    else if (work(1, 2) <= work(1, 1)) launch_router<1, 2>(a, tokens, stream);
    else launch_router<1, 1>(a, tokens, stream);
    if (last < 2) return;
    // stage 2: routes, grouping, fp16 parts of x
    // (the shared router's column rides with the conversion: as a column of the router product it cost a 17th column
    // tile of full depth, and 544 workgroups do not spread evenly over 256 compute units, 512 do)
    pf_launch_route(a, tokens, stream);
    if (pf_group_fits(a.ids, P, E)) {
        static const bool configured = hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_pf_group_rows), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                           GROUP_PAIRS_LDS) == hipSuccess;
        (void)configured;
        const unsigned place_blocks = (unsigned)(P + 1023) / 1024;
        hipLaunchKernelGGL(pf_k_pf_group_rows, dim3(place_blocks + (unsigned)(tokens + 3) / 4), dim3(1024), 2 * GROUP_COPIES * pf_group_pitch(E) * sizeof(uint32_t), stream, a, tokens,
                           (int)place_blocks);
    } else {
        hipLaunchKernelGGL(pf_k_rows_to_half, dim3(tokens), dim3(256), 0, stream, a.x, a.x_pitch, H, (half_t *)a.x16, a.x_scale, a.error_word,
                           reinterpret_cast<const float *>(a.w[7]), a.shared_scale);
        pf_launch_group(a, a.ids, tokens, stream);
    }
    if (last < 3) return;
    // stage 3: gate/up + SwiGLU, then fp16 parts of the activation rows
    // pf_k_pf_gemm takes the items whose tensors are in the routed gate's format and the Q8_0 shared expert, the plain kernel the rest
    const int gi = I > Is ? I : Is;
    const bool iq2 = a.type[1] == PF_IQ2_XXS;
    const uint32_t gate_fmt = a.type[1];
    const unsigned shared_tiles = (unsigned)(tokens + 31) / 32, routed_cap = (unsigned)pf_prefill_max_tiles(tokens, E, K) - shared_tiles;
    const bool q8 = a.type[4] == PF_Q8_0;   // the shared expert of the checkpoint profiles
    if (iq2 && q8) launch_gemm<PF_GEMM_GATE_UP, PF_IQ2_XXS, PF_Q8_0>(a, tokens, routed_cap, gi, H, stream);
    else if (iq2) launch_gemm<PF_GEMM_GATE_UP, PF_IQ2_XXS, PF_IQ2_XXS>(a, tokens, routed_cap, gi, H, stream);
    else if (q8) launch_gemm<PF_GEMM_GATE_UP, PF_Q4_K, PF_Q8_0>(a, tokens, routed_cap, gi, H, stream);
    else launch_gemm<PF_GEMM_GATE_UP, PF_Q4_K, PF_Q4_K>(a, tokens, routed_cap, gi, H, stream);
    // only the shared expert's tiles (tokens / 32 of them) are left for this launch: columns split over the waves
    if (a.type[4] != gate_fmt && !q8) launch_gemm_plain<PF_GEMM_GATE_UP>(a, tokens, shared_tiles, (Is + 31) / 32, 1, PLAIN_SHARED, stream);
    const int widest = I > Is ? I : Is;
    const bool digits = a.wm != nullptr;   // the routed rows as digits (they are of at most 640 values)
    const bool q2_down = pf_q2_down(a.type, I, Is);
    if (widest <= 1024 && P > 0 && tokens > 0) {
        const unsigned rows_a = digits ? 4u * pf_mx_rows_a_wave(I) : 4u, blocks_a = ((unsigned)P + rows_a - 1) / rows_a, blocks_b = (unsigned)((tokens + 3) / 4);
        hipLaunchKernelGGL(digits ? (widest <= 512 ? pf_k_rows_to_half_short2<1, ROWS_DIGITS> : pf_k_rows_to_half_short2<2, ROWS_DIGITS>)
                           : q2_down ? (widest <= 512 ? pf_k_rows_to_half_short2<1, ROWS_SUMS16> : pf_k_rows_to_half_short2<2, ROWS_SUMS16>)
                                     : (widest <= 512 ? pf_k_rows_to_half_short2<1, ROWS_SUMS32> : pf_k_rows_to_half_short2<2, ROWS_SUMS32>),
                           dim3(blocks_a + blocks_b), dim3(256), 0, stream, a.act, I, (size_t)P, (half_t *)a.act16, a.act_scale, blocks_a, a.shared_act, Is, (size_t)tokens,
                           (half_t *)a.sact16, a.sact_scale, a.error_word);
    } else {
        if (digits) pf_launch_rows_to_digits(a.act, I, (size_t)P, reinterpret_cast<uint32_t *>(a.act16), a.act_scale, a.error_word, stream);
        else launch_rows_to_half(a.act, (size_t)I, I, (size_t)P, (half_t *)a.act16, a.act_scale, a.error_word, stream);
        launch_rows_to_half(a.shared_act, (size_t)Is, Is, (size_t)tokens, (half_t *)a.sact16, a.sact_scale, a.error_word, stream);
    }
    if (last < 4) return;
    // stage 4: down and combine
    if (a.type[3] == gate_fmt || a.type[6] == gate_fmt) {
        if (iq2) launch_gemm<PF_GEMM_DOWN, PF_IQ2_XXS, PF_IQ2_XXS>(a, tokens, routed_cap, H, gi, stream);
        else launch_gemm<PF_GEMM_DOWN, PF_Q4_K, PF_Q4_K>(a, tokens, routed_cap, H, gi, stream);
    }
    if (digits) pf_launch_mx_down(a, tokens, routed_cap, stream);
    if (q2_down) {
        launch_gemm<PF_GEMM_DOWN, PF_Q2_K, PF_Q8_0>(a, tokens, routed_cap, H, gi, stream);
        pf_launch_combine(a, tokens, stream);
        return;
    }
    // (beside routed items of the plain kernel a Q8_0 shared expert's cost nothing: in a launch of its own it made the down stage of
    // the q2 profile's 1024-token chunk 169 us instead of 157, at the checkpoints' widths 291 instead of 271)
    const bool plain_routed = a.type[3] != gate_fmt && !digits, q8_shared = a.type[6] == PF_Q8_0 && !plain_routed;
    const bool plain_shared = a.type[6] != gate_fmt && !q8_shared;
    if (plain_routed || plain_shared)
        launch_gemm_plain<PF_GEMM_DOWN>(a, tokens, plain_routed ? routed_cap + shared_tiles : shared_tiles, (H + 255) / 256, 0,
                                        plain_routed ? PLAIN_ALL : PLAIN_SHARED, stream);
    if (q8_shared) launch_gemm<PF_GEMM_DOWN, PF_Q8_0, PF_Q8_0>(a, tokens, 0, H, Is, stream);
    pf_launch_combine(a, tokens, stream);
}
