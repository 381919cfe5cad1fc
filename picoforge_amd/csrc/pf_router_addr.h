// What a chunk's router (pf_k_pf_router) reads of the experts' parts, as functions that compile for the host as well: the kernels call
// them for their addresses, pf_hip_moe_create for the allocation's size, and a host-side test walks every load of every workgroup.
#pragma once
#include "pf_decode_addr.h"

// [tile of 32 experts][step of 16 columns][part][lane][16 bytes]; experts beyond the last of the last tile are zeros.
PF_HD int pf_router_tiles(int experts) { return (experts + 31) / 32; }
PF_HD size_t pf_router_parts_bytes(int experts, int cols) { return (size_t)pf_router_tiles(experts) * 192 * (size_t)cols; }
PF_HD size_t pf_router_tile_at(int tile, int cols) { return (size_t)tile * 192 * (size_t)cols; }
// Tile c of a workgroup whose first tile is `first`; a workgroup takes a fixed number of tiles, and in place of those beyond the
// last one it reads the last again (their columns are not stored).
PF_HD int pf_router_tile_read(int experts, int first, int c) {
    const int last = pf_router_tiles(experts) - 1 - first;
    return c < last ? c : last;
}
// Byte offset of a step's part within the workgroup's tiles, tile as pf_router_tile_read gives it.
PF_HD uint32_t pf_router_part_at(int tile, int cols, int step, int part, int lane) {
    return (uint32_t)tile * 192u * (uint32_t)cols + 3072u * (uint32_t)step + 1024u * (uint32_t)part + 16u * (uint32_t)lane;
}
