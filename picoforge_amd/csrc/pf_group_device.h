// Grouping of a batch's pairs by expert: in one workgroup (pf_moe_route.hip, alone in a launch), or in several (pf_moe_prefill.hip, beside
// the activation rows' conversion).
#pragma once
#include "pf_device.h"

// One workgroup of 1024 threads: counts the pairs per expert in LDS, scans the counts (offsets, and the row tiles:
// tiles[0] = count, tiles[1 + i] = expert | tile index << 16, items[i] = {expert, first row, rows, first row within the expert}; the
// shared expert = expert E with every token, the list's last), and hands every pair the next free row of its expert through an LDS cursor.  The rows
// of an expert are therefore in no particular order (pf_k_group_place keeps them in pair order): every row of the
// grouped products is computed on its own and found again through pair_to_row, so the order changes no result, and a
// walk over all pairs per expert, which the order costs, took three times as long as everything else here.
#define GROUP_FUSED_MAX_PAIRS 32768
#define GROUP_FUSED_MAX_EXPERTS 2047
//
// The list's order.  The few-row kernels take a tile in chunks of eight rows, one after the other: the tiles of experts with more than 24
// rows come first, then more than 16, more than 8, the others (101 tokens of the q2 profile, gate and up 156 -> 146 us traced, down 99 ->
// 94).  CHUNK: the grouped product's tiles stay in the experts' order, where those that wait for memory and those that wait
// for the matrix cores are mixed, but for the experts of no more than half of the average rows, the shortest items, which come last: in any
// order a launch ended with whatever the list ended with (1024 tokens of the Q4_K layer 361 -> 357 us a forward, 2048 of the q4 profile
// 836 -> 830; by classes as above 367 and 828, experts of several tiles first 366 and 867).
// Bound by one compute unit's chain of loads, LDS atomics and stores.  An expert has GROUP_COPIES counters, a lane's by its number,
// so that a popular one's pairs do not queue for one word, and the rows' pairs are collected in LDS and written in order: scattered
// stores are a cache line each.
#define GROUP_COPIES 8
#define GROUP_FUSED_LDS ((GROUP_COPIES * GROUP_FUSED_MAX_EXPERTS + GROUP_FUSED_MAX_PAIRS / 2) * 4)   // 128 KB, at most
// words of fused_lds: the counters, then the pair of every row in 16 bits
__host__ __device__ constexpr size_t pf_group_lds_words(int pairs, int E) { return (size_t)GROUP_COPIES * E + (pairs + 7) / 8 * 4; }
// The scan, by 1024 threads: rows_of(e) pairs an expert, start(e, row) is told its first row; the lists are written where `lists` is
// set.  Returns the pairs of experts there are.
template <bool CHUNK, typename RowsOf, typename Start>
__device__ __forceinline__ uint32_t pf_group_scan(int pairs, int E, int tokens, RowsOf rows_of, Start start, bool lists, uint32_t *offsets, uint32_t *tiles, uint4 *items) {
    __shared__ uint32_t wave_rows[16];
    __shared__ uint64_t wave_tiles[16];
    const int tid = threadIdx.x;
    // exclusive scan of the counts (rows) and of the row-tile counts, thread t owning `per` consecutive experts
    const int per = (E + 1 + 1023) / 1024, lo = tid * per, hi = min(E + 1, lo + per);
    // the routed tiles of each class, 16 bits each
    const uint32_t few = (uint32_t)pairs / (2 * (uint32_t)E);
    auto class_at = [&](uint32_t c) { return CHUNK ? (c > few ? 0 : 16) : c > 24u ? 0 : c > 16u ? 16 : c > 8u ? 32 : 48; };
    uint32_t rows = 0;
    uint64_t ntiles = 0;
    for (int e = lo; e < min(hi, E); e++) {
        const uint32_t c = rows_of(e);
        rows += c;
        ntiles += (uint64_t)((c + 31u) / 32u) << class_at(c);
    }
    // inclusive scan over the 1024 threads: within a wave by shuffles, then the sixteen waves' totals through LDS
    const int lane = pf_lane(), wave = tid >> 6;
    uint32_t run_rows = rows;
    uint64_t run_tiles = ntiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t up_rows = __shfl_up(run_rows, d);
        const uint64_t up_tiles = (uint64_t)__shfl_up((uint32_t)(run_tiles >> 32), d) << 32 | __shfl_up((uint32_t)run_tiles, d);
        if (lane >= d) { run_rows += up_rows; run_tiles += up_tiles; }
    }
    if (lane == 63) { wave_rows[wave] = run_rows; wave_tiles[wave] = run_tiles; }
    __syncthreads();
    uint32_t placed = 0;   // pairs of experts there are
    uint64_t listed = 0;
    for (int w = 0; w < 16; w++) {
        if (w < wave) { run_rows += wave_rows[w]; run_tiles += wave_tiles[w]; }
        placed += wave_rows[w];
        listed += wave_tiles[w];
    }
    const uint64_t until = listed + (listed << 16) + (listed << 32) + (listed << 48);   // the tiles of the classes up to each
    const uint32_t routed = (uint32_t)(until >> 48);
    if (lists && tid == 1023) {
        offsets[E] = run_rows;
        tiles[0] = routed + ((uint32_t)tokens + 31u) / 32u;
    }
    uint32_t row = run_rows - rows;
    uint64_t before = run_tiles - ntiles + (until - listed);
    for (int e = lo; e < hi; e++) {
        const uint32_t c = e < E ? rows_of(e) : (uint32_t)tokens, n = (c + 31u) / 32u, at = e < E ? (uint32_t)(before >> class_at(c)) & 0xffffu : routed;
        for (uint32_t i = 0; lists && i < n; i++) {
            tiles[1 + at + i] = (uint32_t)e | (i << 16);
            items[at + i] = make_uint4((uint32_t)e, (e < E ? row : (uint32_t)pairs) + 32u * i, min(32u, c - 32u * i), 32u * i);
        }
        if (e == E) break;
        before += (uint64_t)n << class_at(c);
        if (lists) offsets[e] = row;
        start(e, row);
        row += c;
    }
    return placed;
}
__device__ __forceinline__ void pf_group_block(uint32_t *fused_lds, const uint32_t *ids, int pairs, int E, int tokens, uint32_t *offsets,
                                               uint32_t *tiles, uint4 *items, uint32_t *pair_to_row, uint32_t *row_to_pair) {
    const int tid = threadIdx.x, quads = pairs / 4;
    uint32_t *counts = fused_lds;   // [expert][copy]; later the next free row
    uint16_t *pair_of = reinterpret_cast<uint16_t *>(fused_lds + (size_t)GROUP_COPIES * E);
    for (int i = tid; i < GROUP_COPIES * E; i += 1024) counts[i] = 0;
    // four pairs a thread and step (ids on a 16-byte boundary), all of a thread's asked for at once and kept for the second walk; the
    // ragged end pair by pair
    constexpr int STEPS = GROUP_FUSED_MAX_PAIRS / 4 / 1024;
    uint4 four[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; k++)
        if (1024 * k < quads) four[k] = reinterpret_cast<const uint4 *>(ids)[min(tid + 1024 * k, quads - 1)];
    const int tail = 4 * quads + tid;   // at most three pairs
    const uint32_t last = tail < pairs ? ids[tail] : 0xffffffffu;
    uint32_t *mine = counts + tid % GROUP_COPIES;
    __syncthreads();
    auto count = [&](uint32_t id) { if (id < (uint32_t)E) atomicAdd(&mine[GROUP_COPIES * id], 1u); };
#pragma unroll
    for (int k = 0; k < STEPS; k++) {
        if (tid + 1024 * k >= quads) break;
        count(four[k].x); count(four[k].y); count(four[k].z); count(four[k].w);
    }
    count(last);
    __syncthreads();
    const uint32_t placed = pf_group_scan<false>(pairs, E, tokens, [&](int e) {
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GROUP_COPIES; r++) c += counts[GROUP_COPIES * e + r];
        return c;
    }, [&](int e, uint32_t row) {
#pragma unroll
        for (int r = 0; r < GROUP_COPIES; r++) {
            const uint32_t here = counts[GROUP_COPIES * e + r];
            counts[GROUP_COPIES * e + r] = row;
            row += here;
        }
    }, true, offsets, tiles, items);
    __syncthreads();
    auto place = [&](uint32_t id, int p) -> uint32_t {
        if (id >= (uint32_t)E) return 0u;   // only with nonfinite logits
        const uint32_t r = atomicAdd(&mine[GROUP_COPIES * id], 1u);
        pair_of[r] = (uint16_t)p;
        return r;
    };
#pragma unroll
    for (int k = 0; k < STEPS; k++) {
        const int q = tid + 1024 * k;
        if (q >= quads) break;
        const uint4 v = four[k];
        uint4 r;
        r.x = place(v.x, 4 * q); r.y = place(v.y, 4 * q + 1); r.z = place(v.z, 4 * q + 2); r.w = place(v.w, 4 * q + 3);
        reinterpret_cast<uint4 *>(pair_to_row)[q] = r;
    }
    if (tail < pairs) pair_to_row[tail] = place(last, tail);
    __syncthreads();
    for (uint32_t q = tid; 4 * q + 3 < placed; q += 1024) {
        const uint2 v = reinterpret_cast<const uint2 *>(pair_of)[q];
        reinterpret_cast<uint4 *>(row_to_pair)[q] = make_uint4(v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16);
    }
    const uint32_t rest = (placed & ~3u) + tid;
    if (tid < 4 && rest < placed) row_to_pair[rest] = pair_of[rest];
}

// The same by several workgroups of 1024 threads, number `block` of them placing pairs 1024 block and on: none waits for another, as
// each counts all pairs, those before its own in counters of their own, and scans the counts.
#define GROUP_PAIRS_LDS (2 * GROUP_COPIES * GROUP_FUSED_MAX_EXPERTS * 4)   // at most
// words of a copy's counters: an odd number, so that an expert's copies lie in different banks, as neighbouring experts' counters do
__host__ __device__ constexpr int pf_group_pitch(int E) { return E | 1; }
__device__ __forceinline__ void pf_group_pairs(uint32_t *counts, const uint32_t *ids, int pairs, int E, int tokens, int block, uint32_t *offsets, uint32_t *tiles,
                                               uint4 *items, uint32_t *pair_to_row, uint32_t *row_to_pair) {
    const int tid = threadIdx.x, quads = pairs / 4, own = 1024 * block, pitch = pf_group_pitch(E);
    for (int i = tid; i < 2 * GROUP_COPIES * pitch; i += 1024) counts[i] = 0;   // [before its own, from there on][copy][expert]; later [0][0]: the next free row
    const uint32_t mine = ids[min(own + tid, pairs - 1)];
    const int tail = 4 * quads + tid;   // at most three pairs
    const uint32_t last = tail < pairs ? ids[tail] : 0xffffffffu;
    __syncthreads();
    auto count = [&](uint32_t id, int p) {
        if (id < (uint32_t)E) atomicAdd(&counts[((p < own ? 0 : GROUP_COPIES) + tid % GROUP_COPIES) * pitch + (int)id], 1u);
    };
    for (int q0 = 0; q0 < quads; q0 += 4 * 1024) {   // four loads of four ids on their way
        uint4 four[4];
#pragma unroll
        for (int k = 0; k < 4; k++) four[k] = reinterpret_cast<const uint4 *>(ids)[min(q0 + 1024 * k + tid, quads - 1)];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int q = q0 + 1024 * k + tid;
            if (q >= quads) break;
            count(four[k].x, 4 * q); count(four[k].y, 4 * q); count(four[k].z, 4 * q); count(four[k].w, 4 * q);   // (own is a multiple of four)
        }
    }
    count(last, tail);
    __syncthreads();
    auto copies = [&](int e, int from) {
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < GROUP_COPIES; r++) c += counts[(from + r) * pitch + e];
        return c;
    };
    pf_group_scan<true>(pairs, E, tokens, [&](int e) { return copies(e, 0) + copies(e, GROUP_COPIES); },
                        [&](int e, uint32_t row) { counts[e] = row + copies(e, 0); }, block == 0, offsets, tiles, items);
    __syncthreads();
    if (own + tid >= pairs) return;
    const bool placed = mine < (uint32_t)E;   // (not with nonfinite logits)
    const uint32_t row = placed ? atomicAdd(&counts[mine], 1u) : 0u;
    pair_to_row[own + tid] = row;
    if (placed) row_to_pair[row] = (uint32_t)(own + tid);
}
