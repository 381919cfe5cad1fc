// Routing (softmax, top-k, renormalisation) and expert grouping kernels.
//
// Two routing paths exist.  The fast one keeps a token's logits in the registers
// of one wave and selects in logit space.  It also measures how close the k+1
// best logits are; when two of them are closer than the rounding noise a
// differently ordered logit sum could have, the token is routed again by the
// exact path, which recomputes its logits in the reference's serial order
// (src/qwen4_packed.c:164-179) and follows src/qwen4_moe.c:219-247 step by step.
#include "pf_moe_internal.h"
#include "pf_route_device.h"
#include "pf_route_fast.h"
#include "pf_route_fix_many.h"
#include "pf_group_device.h"

#define ROUTE_MAX_FAST_EXPERTS 1024

// ---- routing inside a forward: chunks and the general path --------------------------------------
// A workgroup routes up to sixteen tokens, a wave each, and then those of them whose best logits are too close, together
// (pf_route_fix_many.h): the candidates of all of them, as many as there are lanes, share the chain's wave, which costs the same for
// one token as for five.  exact_rows[0] counts the tokens routed again, exact_rows[1] those of them that went the long way.
// Bound by that chain, a dependent addition a column.  1024 tokens of width 2048 25 us traced, 2048 of width 2560 28, where a launch
// that routed and one that routed again, a workgroup a flagged token, took 8.2 + 22.6 and 9.1 + 23.9.  (Handing every pair its rank among its
// expert's here, by additions to a counter an expert in memory, took 10 us: a popular one's queue.)
#define ROUTE_TOKENS 16
#define ROUTE_UNFLAGGED 0xffffffffu
template <int NPL>
__global__ void __launch_bounds__(1024) pf_k_route_tokens(PfKernelArgs a, int tokens) {
    extern __shared__ __align__(16) float route_lds[];   // the two chunk buffers, then the long way's 3 E floats
    __shared__ uint32_t cand[ROUTE_TOKENS][PF_WAVE], list[PF_WAVE], found[ROUTE_TOKENS], ids[ROUTE_TOKENS * PF_WAVE];
    __shared__ float weights[ROUTE_TOKENS * PF_WAVE], sums[PF_WAVE];
    __shared__ uint32_t again[ROUTE_TOKENS];   // 0: settled at once, 1: by the candidates, 2: the long way
    const int E = a.experts, K = a.top_k, H = a.hidden, picks = K < E ? K : E, lane = pf_lane();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), grid = (int)gridDim.x;
    const int here = (tokens - (int)blockIdx.x + grid - 1) / grid;   // tokens blockIdx.x, + grid, ...: flagged neighbours go to several workgroups
    const bool norm = a.norm_topk != 0;
    const float *router = reinterpret_cast<const float *>(a.w[0]);
    auto token = [&](int w) { return (size_t)((int)blockIdx.x + w * grid); };
    const size_t at = token(min(wave, here - 1)) * E;   // this wave's token's logits
    if (wave < here) {
        const PfRouteResult r = pf_route_fast_wave<NPL>(a.logits + at, a.logit_ssq + at, E, K, norm, H, lane);
        if (r.bad && lane == 0) atomicOr(a.error_word, PF_HIP_ERR_NONFINITE);
        if (lane < K) { ids[wave * K + lane] = r.id; weights[wave * K + lane] = r.weight; }
        uint32_t count = ROUTE_UNFLAGGED;
        if (r.close) {
            float v[NPL], s2[NPL];
            pf_load_row<NPL>(a.logits + at, E, lane, -INFINITY, v);
            pf_load_row<NPL>(a.logit_ssq + at, E, lane, 0.0f, s2);
            count = (uint32_t)pf_fix_candidates<NPL>(v, s2, r.kth, r.best, E, picks, H, pf_fix_by_pieces(router, H), cand[wave], lane);
        }
        if (lane == 0) { found[wave] = count; again[wave] = count == ROUTE_UNFLAGGED ? 0u : 2u; }
    }
    __syncthreads();
    // the flagged tokens in turn, as many at a time as their candidates fit the chain's lanes
    for (int w = 0; w < here;) {
        int n = 0, mine = -1, count = 0;
        for (; w < here; w++) {
            const uint32_t c = found[w];
            if (c == ROUTE_UNFLAGGED || c == 0u) continue;
            if (n + (int)c > PF_WAVE) break;
            if (w == wave) { mine = n; count = (int)c; }
            n += (int)c;
        }
        if (n == 0) break;
        if (mine >= 0 && lane < count) list[mine + lane] = (uint32_t)wave << 16 | cand[wave][lane];
        __syncthreads();
        const float logit = pf_fix_sums(n, H, route_lds, [&](int r) { return router + (size_t)(list[r] & 0xffffu) * H; },
                                        [&](int r, int k) { return pf_fix_values(a.x + token((int)(list[r] >> 16)) * a.x_pitch, k); }, wave, lane);
        if (wave == 0) sums[lane] = logit;
        __syncthreads();
        if (mine >= 0) {
            float v[NPL];
            pf_load_row<NPL>(a.logits + at, E, lane, -INFINITY, v);
            const bool active = lane < count;
            const bool settled = pf_fix_finish<NPL>(count, active ? cand[wave][lane] : 0u, active ? sums[mine + lane] : 0.0f, v, E, picks, norm,
                                                    ids + wave * K, weights + wave * K, lane);
            if (lane == 0 && settled) again[wave] = 1u;
        }
    }
    __syncthreads();
    for (int w = 0; w < here; w++) {
        if (again[w] != 2u) continue;   // the same for every thread
        pf_fix_long_way(router, a.x + token(w) * a.x_pitch, E, K, norm, H, route_lds, route_lds + 2 * PF_FIX_CHUNK_FLOATS, ids + w * K,
                        weights + w * K, wave, lane);
        __syncthreads();
    }
    if ((int)threadIdx.x < here && again[threadIdx.x]) {
        atomicAdd(a.exact_rows, 1u);
        if (again[threadIdx.x] == 2u) atomicAdd(a.exact_rows + 1, 1u);
    }
    const int p = threadIdx.x;
    if (p < here * K) {   // at most 16 * 62
        const size_t to = token(p / K) * K + p % K;
        a.ids[to] = ids[p];
        a.route_weights[to] = weights[p];
    }
}

// Serial-order recomputation for flagged tokens, in two kernels so that a token's logits
// spread over many compute units: one workgroup per (token, slab of 64 experts), lane e of its
// first wave owns expert e and the sum runs over k in order, as the reference's.  The router copy
// is laid out for this, [slab][hidden / 4][64 experts][4 consecutive k]: four steps of the wave
// are one 1 KB piece.  The sum is one dependent chain of 2 x hidden operations; what it must never
// do is wait for memory, so two more waves stream the slab's pieces into an eight-batch LDS ring
// (16 pieces = 64 steps per batch, six batches ahead: about 100 KB on their way) and the token's
// row sits in LDS too, read as broadcasts.  One workgroup barrier per batch hands a batch over and
// frees the one before it.
#define FIX_RING 8
#define FIX_AHEAD 6    // batches on their way or waiting in the ring beyond the one being handed over
#define FIX_BATCH 16   // 1 KB pieces per batch
__global__ void __launch_bounds__(192) pf_k_route_fix_logits(PfKernelArgs a) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char fix_lds[];   // the ring, then the token's row
    const int E = a.experts, H = a.hidden, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = blockIdx.y * PF_WAVE + lane;
    float4 *ring = reinterpret_cast<float4 *>(fix_lds);
    float *xs = reinterpret_cast<float *>(fix_lds + FIX_RING * FIX_BATCH * 1024);
    const float4 *__restrict__ w = reinterpret_cast<const float4 *>(a.router_t) + (size_t)blockIdx.y * ((H + 3) / 4) * PF_WAVE;
    const int batches = H / 64;
    const uint32_t listed = a.route_flags[0];
    for (uint32_t item = blockIdx.x; item < listed; item += gridDim.x) {   // the workgroup's share of the listed tokens
    const int t = (int)a.route_flags[1 + item];
    const float *__restrict__ row = a.x + (size_t)t * a.x_pitch;
    __syncthreads();   // the previous token's row has been used up
    for (int k = threadIdx.x; k < H; k += blockDim.x) xs[k] = row[k];
    __syncthreads();
    if (wave >= 1) {   // two loaders: wave 1 the even batches, wave 2 the odd ones, three batches each on their way
        const int mine = wave - 1;
        auto issue = [&](int b) {   // batch b into slot b % FIX_RING: piece j lands at [slot][j][lane]
            const float4 *src = w + (size_t)(FIX_BATCH * b) * PF_WAVE + lane;
            unsigned char *dst = fix_lds + (size_t)(b % FIX_RING) * FIX_BATCH * 1024;
#pragma unroll
            for (int j = 0; j < FIX_BATCH; j++)
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t *>(src + j * PF_WAVE),
                                                 reinterpret_cast<uint32_t *>(dst + j * 1024), 16, 0, 0);
        };
        for (int b = mine; b < FIX_AHEAD && b < batches; b += 2) issue(b);
        for (int s = 0; s < batches; s++) {
            if ((s & 1) == mine) {
                // batch s has landed when only this wave's younger batches (s + 2, s + 4) are outstanding
                if (s + 4 < batches) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * FIX_BATCH) : "memory");
                else if (s + 2 < batches) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIX_BATCH) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            __builtin_amdgcn_s_barrier();   // hands batch s over; batch s - 1 has been consumed
            if ((s & 1) == mine && s + FIX_AHEAD < batches) issue(s + FIX_AHEAD);
        }
        continue;
    }
    float sum = 0.0f;
    for (int s = 0; s < batches; s++) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const float4 *slot = ring + (size_t)(s % FIX_RING) * FIX_BATCH * PF_WAVE + lane;
        const float4 *x4 = reinterpret_cast<const float4 *>(xs + 64 * s);
        float4 wv[FIX_BATCH], xv[FIX_BATCH];
#pragma unroll
        for (int j = 0; j < FIX_BATCH; j++) { wv[j] = slot[j * PF_WAVE]; xv[j] = x4[j]; }
#pragma unroll
        for (int j = 0; j < FIX_BATCH; j++) {
            const float p0 = wv[j].x * xv[j].x;
            sum = sum + p0;
            const float p1 = wv[j].y * xv[j].y;
            sum = sum + p1;
            const float p2 = wv[j].z * xv[j].z;
            sum = sum + p2;
            const float p3 = wv[j].w * xv[j].w;
            sum = sum + p3;
        }
    }
    const float *tail = reinterpret_cast<const float *>(w + lane);
    for (int k = 64 * batches; k < H; k++) {   // the lane's k-quad at 256 (k / 4) floats
        const float p = tail[(size_t)(k / 4) * 4 * PF_WAVE + (k & 3)] * xs[k];
        sum = sum + p;
    }
    if (e < E) a.logits[(size_t)t * E + e] = sum;
    }
}

// router [experts][hidden] -> [slab][ceil(hidden / 4)][64][4] (expert 64 * slab + lane, four
// consecutive columns together; zeros beyond the last expert and the last column), once at upload
size_t pf_router_slab_floats(int experts, int hidden) {
    return (size_t)((experts + PF_WAVE - 1) / PF_WAVE) * ((hidden + 3) / 4) * 4 * PF_WAVE;
}

__global__ void pf_k_router_slabs(const float *src, int experts, int hidden, float *dst, size_t total) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const size_t quads = (size_t)(hidden + 3) / 4;
    const int c = (int)(i & 3), lane = (int)((i >> 2) % PF_WAVE);
    const size_t quad = (i / (4 * PF_WAVE)) % quads, slab = i / (4 * PF_WAVE * quads);
    const size_t e = slab * PF_WAVE + lane, k = 4 * quad + c;
    dst[i] = (e < (size_t)experts && k < (size_t)hidden) ? src[e * hidden + k] : 0.0f;
}

void pf_launch_router_slabs(const float *d_src, int experts, int hidden, float *d_dst, hipStream_t stream) {
    const size_t total = pf_router_slab_floats(experts, hidden);
    hipLaunchKernelGGL(pf_k_router_slabs, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, d_src, experts, hidden,
                       d_dst, total);
}

__global__ void __launch_bounds__(64) pf_k_route_fix_select(PfKernelArgs a) {
    extern __shared__ float lds[];
    const int E = a.experts;
    float *z = lds, *p = z + E, *q = p + E;
    const uint32_t listed = a.route_flags[0];
    for (uint32_t item = blockIdx.x; item < listed; item += gridDim.x) {
        const int t = (int)a.route_flags[1 + item];
        for (int e = threadIdx.x; e < E; e += PF_WAVE) z[e] = a.logits[(size_t)t * E + e];
        pf_wave_lds_fence();
        pf_route_exact_wave(z, p, q, E, a.top_k, a.norm_topk != 0, a.ids + (size_t)t * a.top_k,
                            a.route_weights + (size_t)t * a.top_k, threadIdx.x);
        if (threadIdx.x == 0) atomicAdd(a.exact_rows, 1u);
    }
}

// Every token through the exact path (expert counts the fast kernel cannot hold): the full list.
__global__ void pf_k_flag_all(uint32_t *list, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) list[0] = (uint32_t)n;
    if (i < n) list[1 + i] = (uint32_t)i;
}

template <int NPL>
static void launch_route_tokens(const PfKernelArgs &a, int tokens, hipStream_t stream) {
    static bool configured = false;   // once per instantiation: more than the default 64 KB of dynamic LDS
    if (!configured) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_route_tokens<NPL>), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
        configured = true;
    }
    // a workgroup a compute unit (its LDS and threads leave room for no second one) while sixteen tokens each suffice
    const int per = min(ROUTE_TOKENS, (tokens + 255) / 256);
    const size_t lds = (2 * PF_FIX_CHUNK_FLOATS + 3 * (size_t)a.experts) * sizeof(float);
    hipLaunchKernelGGL(pf_k_route_tokens<NPL>, dim3((tokens + per - 1) / per), dim3(1024), lds, stream, a, tokens);
}

bool pf_route_needs_slabs(int experts, int top_k) { return experts > ROUTE_MAX_FAST_EXPERTS || top_k >= PF_WAVE - 1; }

void pf_launch_route(const PfKernelArgs &a, int tokens, hipStream_t stream) {
    const int npl = (a.experts + PF_WAVE - 1) / PF_WAVE;
    if (!pf_route_needs_slabs(a.experts, a.top_k)) {   // the fast routing keeps top_k + 2 keys, one per lane
        if (npl <= 1) launch_route_tokens<1>(a, tokens, stream);
        else if (npl <= 2) launch_route_tokens<2>(a, tokens, stream);
        else if (npl <= 4) launch_route_tokens<4>(a, tokens, stream);
        else if (npl <= 8) launch_route_tokens<8>(a, tokens, stream);
        else launch_route_tokens<16>(a, tokens, stream);
        return;
    }
    hipLaunchKernelGGL(pf_k_flag_all, dim3((tokens + 255) / 256), dim3(256), 0, stream, a.route_flags, tokens);
    const int workers = tokens < 256 ? tokens : 256;
    // more experts than a wave's registers hold: every token is listed and all its logits are summed serially
    const size_t fix_lds = (size_t)FIX_RING * FIX_BATCH * 1024 + (size_t)a.hidden * sizeof(float);
    static bool configured = false;   // more than the default 64 KB of dynamic LDS
    if (!configured) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_route_fix_logits),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        configured = true;
    }
    hipLaunchKernelGGL(pf_k_route_fix_logits, dim3(workers, (a.experts + PF_WAVE - 1) / PF_WAVE), dim3(3 * PF_WAVE), fix_lds, stream, a);
    hipLaunchKernelGGL(pf_k_route_fix_select, dim3(workers), dim3(PF_WAVE), 3 * (size_t)a.experts * sizeof(float), stream,
                       a);
}

// ---- qwen4_moe_route on caller-provided logits ----------------------------------
__global__ void pf_k_logits_finite(const float *z, size_t n, int experts, uint32_t *error, unsigned long long *bad_row) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !pf_finite(z[i])) {
        atomicOr(error, PF_HIP_ERR_NONFINITE);
        atomicMin(bad_row, (unsigned long long)(i / experts));
    }
}

__global__ void __launch_bounds__(64) pf_k_route_exact(const float *logits, int E, int K, int norm, float *probs,
                                                       uint32_t *ids, float *weights) {
    extern __shared__ float lds[];
    const int t = blockIdx.x, lane = threadIdx.x;
    float *z = lds, *p = z + E, *q = p + E;
    for (int e = lane; e < E; e += PF_WAVE) z[e] = logits[(size_t)t * E + e];
    pf_wave_lds_fence();
    pf_route_exact_wave(z, p, q, E, K, norm != 0, ids + (size_t)t * K, weights + (size_t)t * K, lane);
    for (int e = lane; e < E; e += PF_WAVE) probs[(size_t)t * E + e] = p[e];
}

int pf_route_exact_device(const float *d_logits, int tokens, int experts, int top_k, int norm, float *d_probs,
                          uint32_t *d_ids, float *d_weights, uint32_t *d_error, unsigned long long *d_bad_row,
                          hipStream_t stream) {
    const size_t n = (size_t)tokens * experts;
    if (n == 0) return PF_HIP_OK;
    hipLaunchKernelGGL(pf_k_logits_finite, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, d_logits, n,
                       experts, d_error, d_bad_row);
    uint32_t err = 0;
    if (hipMemcpyAsync(&err, d_error, 4, hipMemcpyDeviceToHost, stream) != hipSuccess ||
        hipStreamSynchronize(stream) != hipSuccess)
        return PF_HIP_E_RUNTIME;
    if (err) return PF_HIP_OK;   // caller reads the error word; nothing was written
    const size_t lds = 3 * (size_t)experts * sizeof(float);
    if (lds > 64 * 1024) return PF_HIP_E_UNSUPPORTED;
    hipLaunchKernelGGL(pf_k_route_exact, dim3(tokens), dim3(64), lds, stream, d_logits, experts, top_k, norm,
                       d_probs, d_ids, d_weights);
    return hipGetLastError() == hipSuccess ? PF_HIP_OK : PF_HIP_E_RUNTIME;
}

__global__ void pf_k_fill_u32(uint32_t *p, int n, uint32_t value) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// ---- grouping: stable counting sort of (token, slot) pairs by expert ------------
// first_bad = min over offending (token, slot) of 2 * pair + kind, kind 0 = id out
// of range, 1 = id repeated within the token: the error a scan in pair order
// meets first (src/qwen4_moe.c:277-284)
__global__ void pf_k_group_check(const uint32_t *ids, int tokens, int E, int K, uint32_t *first_bad) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= tokens) return;
    const uint32_t *row = ids + (size_t)t * K;
    for (int s = 0; s < K; s++) {
        const uint32_t pair = (uint32_t)(t * K + s);
        if (row[s] >= (uint32_t)E) { atomicMin(first_bad, 2u * pair); return; }
        for (int j = 0; j < s; j++)
            if (row[j] == row[s]) { atomicMin(first_bad, 2u * pair + 1u); return; }
    }
}

__global__ void pf_k_group_count(const uint32_t *ids, int pairs, int E, uint32_t *counts) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < pairs && ids[p] < (uint32_t)E) atomicAdd(&counts[ids[p]], 1u);
}

// one block: exclusive scan of counts[E] into offsets[E+1]
__global__ void __launch_bounds__(256) pf_k_group_scan(const uint32_t *counts, int E, uint32_t *offsets) {
    __shared__ uint32_t part[256];
    const int tid = threadIdx.x, per = (E + 255) / 256, lo = tid * per, hi = min(E, lo + per);
    uint32_t s = 0;
    for (int e = lo; e < hi; e++) s += counts[e];
    part[tid] = s;
    __syncthreads();
    if (tid == 0) {
        uint32_t run = 0;
        for (int i = 0; i < 256; i++) { uint32_t v = part[i]; part[i] = run; run += v; }
        offsets[E] = run;
    }
    __syncthreads();
    uint32_t run = part[tid];
    for (int e = lo; e < hi; e++) { offsets[e] = run; run += counts[e]; }
}

// one wave per expert walks the pairs in order: rank = earlier pairs of the
// same expert, so placement is stable without ordered atomics.  The ids pass through LDS in
// pieces; a lane looks at four consecutive pairs per step (one 16-byte LDS read), two steps'
// reads are requested together.
#define PLACE_PIECE 8192
__global__ void __launch_bounds__(256) pf_k_group_place(const uint32_t *ids, int pairs, int E, const uint32_t *offsets,
                                                        uint32_t *pair_to_row, uint32_t *row_to_pair) {
    __shared__ __align__(16) uint32_t staged[PLACE_PIECE];
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6), lane = pf_lane();
    const bool active = e < E && offsets[min(e, E - 1) + 1] != offsets[min(e, E - 1)];
    uint32_t base = e < E ? offsets[e] : 0u;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int piece = 0; piece < pairs; piece += PLACE_PIECE) {
        const int len = min(PLACE_PIECE, pairs - piece), padded = (len + 511) & ~511;
        __syncthreads();
        // all of a thread's loads are requested before the first is stored (the piece starts on a
        // 16-byte boundary of ids; its ragged end is read id by id)
        uint4 held[PLACE_PIECE / 4 / 256];
#pragma unroll
        for (int j = 0; j < PLACE_PIECE / 4 / 256; j++) {
            const int i = 4 * ((int)threadIdx.x + 256 * j);
            uint4 v = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
            if (i + 4 <= len) {
                v = *reinterpret_cast<const uint4 *>(ids + piece + i);
            } else if (i < len) {
                v.x = ids[piece + i];
                if (i + 1 < len) v.y = ids[piece + i + 1];
                if (i + 2 < len) v.z = ids[piece + i + 2];
            }
            held[j] = v;
        }
#pragma unroll
        for (int j = 0; j < PLACE_PIECE / 4 / 256; j++) {
            const int i = 4 * ((int)threadIdx.x + 256 * j);
            if (i < padded) *reinterpret_cast<uint4 *>(staged + i) = held[j];
        }
        __syncthreads();
        if (!active) continue;
        // step: 256 pairs, lane l holds pairs 4l .. 4l + 3 of it
        auto place = [&](const uint4 &v, int p0) {
            const bool h0 = v.x == (uint32_t)e, h1 = v.y == (uint32_t)e, h2 = v.z == (uint32_t)e, h3 = v.w == (uint32_t)e;
            const int mine = (int)h0 + (int)h1 + (int)h2 + (int)h3;
            const unsigned long long any = __ballot(mine != 0);
            if (!any) return;
            // pairs of lower lanes come first, then this lane's own earlier ones
            const unsigned long long m0 = __ballot(h0), m1 = __ballot(h1), m2 = __ballot(h2), m3 = __ballot(h3);
            uint32_t row = base + __popcll(m0 & below) + __popcll(m1 & below) + __popcll(m2 & below) + __popcll(m3 & below);
            const int p = piece + p0 + 4 * lane;
            if (h0) { pair_to_row[p] = row; row_to_pair[row] = (uint32_t)p; row++; }
            if (h1) { pair_to_row[p + 1] = row; row_to_pair[row] = (uint32_t)(p + 1); row++; }
            if (h2) { pair_to_row[p + 2] = row; row_to_pair[row] = (uint32_t)(p + 2); row++; }
            if (h3) { pair_to_row[p + 3] = row; row_to_pair[row] = (uint32_t)(p + 3); }
            base += __popcll(m0) + __popcll(m1) + __popcll(m2) + __popcll(m3);
        };
        const uint4 *quads = reinterpret_cast<const uint4 *>(staged);
        for (int p0 = 0; p0 < padded; p0 += 512) {
            const uint4 va = quads[p0 / 4 + lane], vb = quads[p0 / 4 + 64 + lane];
            place(va, p0);
            place(vb, p0 + 256);
        }
    }
}

void pf_launch_group_place(const uint32_t *d_ids, int pairs, int experts, const uint32_t *d_offsets,
                           uint32_t *d_pair_to_row, uint32_t *d_row_to_pair, hipStream_t stream) {
    hipLaunchKernelGGL(pf_k_group_place, dim3((experts + 3) / 4), dim3(256), 0, stream, d_ids, pairs, experts, d_offsets,
                       d_pair_to_row, d_row_to_pair);
}

// ---- grouping in one launch (pf_group_device.h) ---------------------------------------------------------
__global__ void __launch_bounds__(1024) pf_k_group_fused(const uint32_t *ids, int pairs, int E, int tokens, uint32_t *offsets,
                                                         uint32_t *tiles, uint4 *items, uint32_t *pair_to_row, uint32_t *row_to_pair) {
    extern __shared__ __align__(16) uint32_t fused_lds[];
    pf_group_block(fused_lds, ids, pairs, E, tokens, offsets, tiles, items, pair_to_row, row_to_pair);
}

bool pf_group_fits(const uint32_t *d_ids, int pairs, int experts) {
    return pairs > 0 && pairs <= GROUP_FUSED_MAX_PAIRS && experts <= GROUP_FUSED_MAX_EXPERTS && (reinterpret_cast<uintptr_t>(d_ids) & 15) == 0;
}

bool pf_launch_group_fused(const uint32_t *d_ids, int pairs, int experts, int tokens, uint32_t *d_offsets, uint32_t *d_tiles,
                           uint32_t *d_items, uint32_t *d_pair_to_row, uint32_t *d_row_to_pair, hipStream_t stream) {
    if (!pf_group_fits(d_ids, pairs, experts)) return false;
    const size_t lds = pf_group_lds_words(pairs, experts) * sizeof(uint32_t);
    static const bool configured = hipFuncSetAttribute(reinterpret_cast<const void *>(pf_k_group_fused), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       GROUP_FUSED_LDS) == hipSuccess;   // more than the default 64 KB
    (void)configured;
    hipLaunchKernelGGL(pf_k_group_fused, dim3(1), dim3(1024), lds, stream, d_ids, pairs, experts, tokens, d_offsets, d_tiles,
                       reinterpret_cast<uint4 *>(d_items), d_pair_to_row, d_row_to_pair);
    return true;
}

int pf_group_pairs_device(const uint32_t *d_ids, int tokens, int experts, int top_k, uint32_t *d_counts,
                          uint32_t *d_offsets, uint32_t *d_pair_to_row, uint32_t *d_row_to_pair, uint32_t *d_first_bad,
                          hipStream_t stream) {
    const int pairs = tokens * top_k;
    hipLaunchKernelGGL(pf_k_fill_u32, dim3(1), dim3(64), 0, stream, d_first_bad, 1, 0xffffffffu);
    hipLaunchKernelGGL(pf_k_fill_u32, dim3((experts + 255) / 256), dim3(256), 0, stream, d_counts, experts, 0u);
    if (tokens > 0) {
        hipLaunchKernelGGL(pf_k_group_check, dim3((tokens + 255) / 256), dim3(256), 0, stream, d_ids, tokens, experts,
                           top_k, d_first_bad);
        hipLaunchKernelGGL(pf_k_group_count, dim3((pairs + 255) / 256), dim3(256), 0, stream, d_ids, pairs, experts,
                           d_counts);
    }
    hipLaunchKernelGGL(pf_k_group_scan, dim3(1), dim3(256), 0, stream, d_counts, experts, d_offsets);
    if (tokens > 0)
        hipLaunchKernelGGL(pf_k_group_place, dim3((experts + 3) / 4), dim3(256), 0, stream, d_ids, pairs, experts,
                           d_offsets, d_pair_to_row, d_row_to_pair);
    return hipGetLastError() == hipSuccess ? PF_HIP_OK : PF_HIP_E_RUNTIME;
}
