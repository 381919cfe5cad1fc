// Re-routing of several flagged tokens by the waves of one workgroup: the steps of pf_route_fix.h (candidates, serial sums, order, the
// long way) one by one, so that the candidates of several tokens can share the chain's wave, a lane each, and their rows are asked for a
// chunk before their products are put down.  pf_route_fix_block has the same steps in a form of its own: built from these
// it moved the one-token kernels' code, 0.5 to 1.5 % of a token's four layers (65.8 us against 66.8).
#pragma once
#include "pf_route_fix.h"

#define PF_FIX_THREADS 1024   // of the workgroup: the chain's wave and fifteen that feed it
#define PF_FIX_HELPERS (PF_FIX_THREADS - PF_WAVE)
#define PF_FIX_PLACES ((2048 + PF_FIX_HELPERS - 1) / PF_FIX_HELPERS)   // 16-byte pieces of a chunk a thread brings

// Four values of a token's row, wherever it starts.
__device__ __forceinline__ float4 pf_fix_values(const float *x, int k) {
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) return *reinterpret_cast<const float4 *>(x + k);
    return make_float4(x[k], x[k + 1], x[k + 2], x[k + 3]);
}

// The candidates of a token, by one wave: v, s2 its fast logits and their noise terms (expert lane NPL + j in register j), kth
// and best_z the smallest and the largest of its k best fast logits (kth as extracted: a lower value only adds candidates).
// Returns their number, their ids in cand (LDS, 64 words); 0: the token goes the long way.
template <int NPL>
__device__ __forceinline__ int pf_fix_candidates(const float (&v)[NPL], const float (&s2)[NPL], float kth, float best_z, int E, int picks,
                                                 int H, bool by_pieces, uint32_t *cand, int lane) {
    float worst_s2 = 0.0f;   // the largest noise term of the token
#pragma unroll
    for (int j = 0; j < NPL; j++) worst_s2 = fmaxf(worst_s2, s2[j]);
    worst_s2 = pf_wave_max(worst_s2);
    const float u = 5.9604645e-8f, hk = (float)H / 6.0f;
    const float tol = 16.0f * u * sqrtf(hk * worst_s2) + 4e-6f * fmaxf(1.0f, best_z - kth + 1.0f);
    const float floor_z = kth - tol;
    // rows the chunk loads cannot take in 16-byte pieces go the long way, as do logits beyond exp's range
    if (!(best_z - floor_z < 80.0f) || !pf_finite(best_z) || !pf_finite(kth) || !by_pieces) return 0;
    // position in the list = candidates of lower registers, then of lower lanes in this register
    int count = 0;
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int j = 0; j < NPL; j++) {
        const bool in = lane * NPL + j < E && v[j] >= floor_z;
        const unsigned long long m = __ballot(in);
        const int to = count + __popcll(m & below);
        if (in && to < PF_WAVE) cand[to] = (uint32_t)(lane * NPL + j);
        count += __popcll(m);
    }
    return count > PF_WAVE || count < picks ? 0 : count;
}
__device__ __forceinline__ bool pf_fix_by_pieces(const float *router, int H) { return H % 4 == 0 && (reinterpret_cast<uintptr_t>(router) & 15) == 0; }

// Serial sums of n <= 64 router rows, lane r of wave 0 the r-th: row_at(r) is the row, on a 16-byte boundary, values_at(r, k) the
// token's values k .. k + 3.  Every wave calls it (workgroup barriers inside).  stage: 2 PF_FIX_CHUNK_FLOATS floats of LDS.
template <typename RowAt, typename ValuesAt>
__device__ __forceinline__ float pf_fix_sums(int n, int H, float *stage, RowAt row_at, ValuesAt values_at, int wave, int lane) {
#pragma clang fp contract(off)
    const int me = (int)threadIdx.x - PF_WAVE;   // place among the waves after the first
    float sum = 0.0f;
    const int shift = n <= 16 ? 7 : n <= 32 ? 6 : 5;   // 16-byte pieces of a row in a chunk: 2048 for 16, 32 or 64 rows
    const int per_chunk = 1 << shift, pitch = 4 * per_chunk + 4, pieces = H / 4, chunks = (pieces + per_chunk - 1) >> shift;
    // A thread brings the same places of every chunk, and asks for them a chunk before it puts their products down.
    auto ask = [&](int c, float4 (&w)[PF_FIX_PLACES], float4 (&x)[PF_FIX_PLACES]) {
        if (c >= chunks) return;
#pragma unroll
        for (int j = 0; j < PF_FIX_PLACES; j++) {   // beyond the rows or the columns: the last ones again, not put down
            const int i = me + j * PF_FIX_HELPERS, row = min(i >> shift, n - 1), piece = min((c << shift) + (i & (per_chunk - 1)), pieces - 1);
            w[j] = reinterpret_cast<const float4 *>(row_at(row))[piece];
            x[j] = values_at(row, 4 * piece);
        }
    };
    auto put = [&](int c, const float4 (&w)[PF_FIX_PLACES], const float4 (&x)[PF_FIX_PLACES]) {   // the products, each rounded once, as the reference forms them before it adds
        float *buf = stage + (c & 1) * PF_FIX_CHUNK_FLOATS;
#pragma unroll
        for (int j = 0; j < PF_FIX_PLACES; j++) {
            const int i = me + j * PF_FIX_HELPERS, row = i >> shift, at = i & (per_chunk - 1);
            if (row < n && (c << shift) + at < pieces)
                reinterpret_cast<float4 *>(buf + row * pitch)[at] = float4{w[j].x * x[j].x, w[j].y * x[j].y, w[j].z * x[j].z, w[j].w * x[j].w};
        }
    };
    // The two sides apart, so that neither's registers weigh on the other's; both meet chunks + 1 barriers.
    if (wave == 0) {
        __syncthreads();
        for (int c = 0; c < chunks; c++) {   // lanes beyond the rows sum the last row again, unused
            sum = pf_serial_chunk(sum, stage + (c & 1) * PF_FIX_CHUNK_FLOATS + min(lane, n - 1) * pitch, min(per_chunk, pieces - (c << shift)));
            __syncthreads();
        }
        return sum;
    }
    float4 rows[PF_FIX_PLACES], values[PF_FIX_PLACES];
    ask(0, rows, values);
    put(0, rows, values);
    ask(1, rows, values);
    __syncthreads();
    for (int c = 0; c < chunks; c++) {   // chunk c is summed, c + 1 put down, c + 2 asked for
        if (c + 1 < chunks) put(c + 1, rows, values);
        ask(c + 2, rows, values);
        __syncthreads();
    }
    return sum;
}

// A token's routes from its candidates' serial sums, by one wave: lane c < count holds candidate c's id and logit, v the token's
// fast logits.  False, and nothing written: the sum over all experts is needed, the token goes the long way.
template <int NPL>
__device__ __forceinline__ bool pf_fix_finish(int count, uint32_t candidate, float logit, const float (&v)[NPL], int E, int picks, bool norm,
                                              uint32_t *ids_out, float *w_out, int lane) {
#pragma clang fp contract(off)
    const bool active = lane < count;
    const uint32_t id = active ? candidate : 0xffffffffu;
    const float mine = active ? logit : -INFINITY;
    const float zmax = pf_wave_max(mine);
    float shifted = mine - zmax;
    const float pc = active ? pf_expf_libm(shifted) : -1.0f;
    // rank by (p descending, id ascending)
    int rank = 0;
    for (int c = 0; c < count; c++) {
        const float po = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pc), c));
        const uint32_t io = (uint32_t)__builtin_amdgcn_readlane((int)id, c);
        rank += (po > pc || (po == pc && io < id)) ? 1 : 0;
    }
    const int to = active ? rank : lane;   // a permutation of the lanes
    const uint32_t sid = (uint32_t)__builtin_amdgcn_ds_permute(to * 4, (int)id);
    const float sp = __int_as_float(__builtin_amdgcn_ds_permute(to * 4, __float_as_int(pc)));
    if (pf_fix_doubtful(sp, sid, picks, count, lane)) return false;
    const float chosen = pf_wave_sum(lane < picks ? sp : 0.0f);
    float weight;
    if (norm) {
        weight = sp / chosen;
    } else {   // the softmax denominator from the fast logits (weights are compared within a tolerance)
        float total = 0.0f;
#pragma unroll
        for (int j = 0; j < NPL; j++) total += lane * NPL + j < E ? expf(v[j] - zmax) : 0.0f;
        total = pf_wave_sum(total);
        weight = sp / total;
    }
    if (lane < picks) { ids_out[lane] = sid; w_out[lane] = weight; }
    return true;
}

// The long way, every wave of the workgroup: all logits of the token x in serial order, 64 experts a pass, then the reference's
// routing step by step.  z: 3 E floats of LDS.
__device__ __forceinline__ void pf_fix_long_way(const float *router, const float *x, int E, int K, bool norm, int H, float *stage, float *z,
                                                uint32_t *ids_out, float *w_out, int wave, int lane) {
    if (pf_fix_by_pieces(router, H)) {
        for (int e0 = 0; e0 < E; e0 += PF_WAVE) {
            const int rows = min(PF_WAVE, E - e0);
            const float ze = pf_fix_sums(rows, H, stage, [&](int r) { return router + (size_t)(e0 + r) * H; }, [&](int, int k) { return pf_fix_values(x, k); }, wave, lane);
            if (wave == 0 && lane < rows) z[e0 + lane] = ze;
        }
    } else {   // rows that cannot be fetched in 16-byte pieces: a thread per expert
        for (int e = threadIdx.x; e < E; e += blockDim.x) z[e] = pf_serial_logit(router + (size_t)e * H, x, H);
    }
    __syncthreads();
    if (wave == 0) pf_route_exact_wave(z, z + E, z + 2 * E, E, K, norm, ids_out, w_out, lane);
}

// One token, called by every wave of a workgroup of PF_FIX_THREADS threads, whose routing knows the smallest and the largest of the k
// best logits (wave 0).  lds: pf_fix_token_lds_floats; the rest as pf_route_fix_block.
__host__ __device__ constexpr size_t pf_fix_token_lds_floats(int E) { return 68 + 2 * PF_FIX_CHUNK_FLOATS + 3 * (size_t)E; }
template <int NPL>
__device__ __forceinline__ int pf_fix_token(const float *router, const float *x, const float *z_row, const float *ssq_row, float kth, float best_z, int E,
                                            int K, bool norm, int H, float *lds, uint32_t *ids_out, float *w_out, int wave, int lane) {
    uint32_t *cand = reinterpret_cast<uint32_t *>(lds), *hand = cand + 64;   // hand[0]: candidates (0: the long way), hand[1]: outcome
    float *stage = lds + 68;
    const int picks = K < E ? K : E;
    float v[NPL];
    int count = 0;
    if (wave == 0) {
        float s2[NPL];
        pf_load_row<NPL>(z_row, E, lane, -INFINITY, v);
        pf_load_row<NPL>(ssq_row, E, lane, 0.0f, s2);
        count = pf_fix_candidates<NPL>(v, s2, kth, best_z, E, picks, H, pf_fix_by_pieces(router, H), cand, lane);
        if (lane == 0) hand[0] = (uint32_t)count;
    }
    __syncthreads();
    const int n = (int)hand[0];
    float logit = 0.0f;
    if (n > 0) logit = pf_fix_sums(n, H, stage, [&](int r) { return router + (size_t)cand[r] * H; }, [&](int, int k) { return pf_fix_values(x, k); }, wave, lane);
    if (wave == 0) {
        const bool settled = n > 0 && pf_fix_finish<NPL>(count, lane < count ? cand[lane] : 0u, logit, v, E, picks, norm, ids_out, w_out, lane);
        if (lane == 0) hand[1] = settled ? 1u : 2u;
    }
    __syncthreads();
    const int how = (int)hand[1];
    if (how == 2) pf_fix_long_way(router, x, E, K, norm, H, stage, stage + 2 * PF_FIX_CHUNK_FLOATS, ids_out, w_out, wave, lane);
    __syncthreads();
    return how;
}
