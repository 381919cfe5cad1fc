// Device pieces that the grouped products (pf_moe_prefill.hip, pf_moe_mx.hip) share: buffers with bounds, the barrier between
// uses of an LDS copy, work items.
#pragma once
#include "pf_moe_internal.h"
#include "pf_item_order.h"

typedef _Float16 half_t;
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

// Barrier between the uses of an LDS copy: the wave's own LDS accesses are over, of its loads from memory the youngest LATER may
// still be on their way.
template <int LATER> __device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((LATER & 15) | (LATER >> 4) << 14 | 0x70);   // vmcnt(LATER) lgkmcnt(0), in a form that the compiler counts with
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A buffer whose reads beyond `bytes` give zero and cost no memory access.
typedef __amdgpu_buffer_rsrc_t PfBuffer;
typedef __attribute__((address_space(3))) unsigned char lds_byte;
__device__ __forceinline__ PfBuffer pf_buffer(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
#define PF_NOWHERE 0xC0000000u   // an offset beyond every buffer: none is larger

struct GemmItem {   // a 32-row tile of an expert
    bool shared;
    int expert, first, m0, rows_here;   // first row of the tile in expert order and within the expert, rows in it
    int inter;
};

// The item that number q of the launch is (pf_item_order.h); shared: the shared expert's row tiles, the list's last; skip: tiles at
// the list's start that the launch leaves out.  False: nothing to do for q.
__device__ __forceinline__ bool gemm_item(const PfKernelArgs &a, int slabs, int shift, uint32_t q, uint32_t routed, uint32_t shared, uint32_t skip, GemmItem &g, int &slab) {
    const PfItemPlace p = pf_item_place(q, slabs, shift, routed, shared);
    if (!p.any) return false;
    const uint4 item = reinterpret_cast<const uint4 *>(a.items)[skip + p.tile];
    slab = p.slab;
    g.expert = (int)item.x; g.first = (int)item.y; g.rows_here = (int)item.z; g.m0 = (int)item.w;
    g.shared = g.expert == a.experts;
    g.inter = g.shared ? a.shared_inter : a.inter;
    return true;
}
