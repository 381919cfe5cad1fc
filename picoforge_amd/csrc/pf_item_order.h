// How the grouped products' launches (pf_moe_prefill.hip, pf_moe_mx.hip) cut their work into workgroups, as functions that compile
// for the host as well (tests/check_item_order.cpp).
#pragma once
#include "pf_decode_addr.h"

// Slabs of output rows that a workgroup takes of a row tile's `all`, one after the other: at most `most`, evenly, and fewer where
// `tiles` row tiles would leave compute units without the two workgroups they hold.  More slabs a workgroup save the rows' way
// into LDS again; with four for each of 87 tiles half of the chip stood idle (350 tokens, 32 experts, 512 x 1024: 23.5 us, one
// each 14).
#define PF_FULL_CHIP 512   // workgroups: two a compute unit
PF_HD int pf_slabs_each(int all, int most, unsigned tiles) {
    const int fewest = (all + most - 1) / most;
    int per = (all + fewest - 1) / fewest;
    while (per > 1 && tiles * (unsigned)((all + per - 1) / per) < PF_FULL_CHIP) per--;
    return per;
}

// Number q of a launch -> (row tile, slab group).  Workgroups go to the eight XCDs round robin by number.  The routed row tiles are cut
// into groups of consecutive ones and the groups dealt to the XCDs in turn; the items of a group (its tiles' slabs) get numbers eight
// apart: neighbouring workgroups of one XCD, one L2, at the same time.  The slabs of a row tile read the same activation rows, and the
// row tiles of one expert, neighbours in the list, the same weights: fetched once from memory where they fall into one group.  Groups
// are of eight tiles where that leaves every XCD eight of them, else smaller, so that a short list is spread over the chip.  (Groups of
// eight whatever the list, the shared expert's among them: eight routed tiles were one XCD's, 257 tokens' shared tiles two XCDs'.  7
// tokens of a Q4_K layer of 8 experts, 4096 x 1536, 143 us, now 89; the q4 profile, 32 experts of 2560 x 768 beside a shared expert of
// 3072, 257 tokens 394, now 274.)
// The shared expert's tiles, the list's last, are dealt one by one, first to the XCDs that have a group less than the others, then to
// all, and are an XCD's first: a profile's Q8_0 tile takes longer than a routed one and at the list's end it was the launch's (q4 profile,
// 64 experts of 3072 x 1024, sixteen slots, 55 tokens 235 us a forward, now 226; 8 experts of 4096 x 1536, 450 tokens 267, now 223).
#define PF_XCDS 8
PF_HD int pf_group_shift(uint32_t routed) { return routed >= 512 ? 3 : routed >= 256 ? 2 : routed >= 128 ? 1 : 0; }
struct PfItemPlace { bool any; uint32_t tile; int slab; };
PF_HD PfItemPlace pf_item_place(uint32_t q, int slabs, int shift, uint32_t routed, uint32_t shared) {
    const uint32_t xcd = q % PF_XCDS, turn = q / PF_XCDS, each = 1u << shift, groups = (routed + each - 1) >> shift, more = groups % PF_XCDS;
    const uint32_t lacking = more ? PF_XCDS - more : 0, gap = lacking << shift;   // XCDs with a group less than the first `more`; their free places
    uint32_t r = turn / (uint32_t)slabs;   // the XCD's tile
    PfItemPlace p;
    p.slab = (int)(turn % (uint32_t)slabs);
    // its shared tiles: number r of the gap is lacking * r + own, beyond the gap every eighth
    auto count = [](uint32_t first, uint32_t end, uint32_t step) { return first < end ? (end - first - 1) / step + 1 : 0u; };
    const bool fills = lacking && xcd >= more;
    const uint32_t in_gap = fills ? count(xcd - more, shared < gap ? shared : gap, lacking) : 0, mine = in_gap + count(gap + xcd, shared, PF_XCDS);
    if (r < mine) {
        p.tile = routed + (r < in_gap ? lacking * r + xcd - more : gap + PF_XCDS * (r - in_gap) + xcd);
        p.any = true;
        return p;
    }
    r -= mine;
    p.tile = (((r >> shift) * PF_XCDS + xcd) << shift) + (r & (each - 1));
    p.any = p.tile < routed;
    return p;
}
// numbers that cover up to `routed` tiles and `shared` more
PF_HD uint32_t pf_item_numbers(int slabs, int shift, uint32_t routed, uint32_t shared) {
    const uint32_t deal = PF_XCDS << shift;
    return ((routed + deal - 1) / deal * deal + (shared + PF_XCDS - 1) / PF_XCDS * PF_XCDS) * (uint32_t)slabs;   // (no XCD has more)
}

// Pairs up to which a batch of a layer of one format (with its tile-ordered copies) runs the decode kernels, which read an expert once a
// pair, and from which on the kernels for a few rows per expert, which read it once for the batch.  The line goes by the work of a pair,
// hidden x inter: the few-row kernels' launches take at least 30 to 40 us, which short products do not earn back by 32 tokens.
// Where the two take the same time (pairs; 16 to 32 tokens swept; E (top-k) = 16 (4), 32 (6), 64, 128, 256 (8), 512 (6, 10); > beyond
// them, < before them):
//   Q4_K     2048 x 512  120, 110, 128, 136, 140, 190, 170       2560 x 512, 2048 x 768  < but 512 (6): 110, 170
//            2048 x 256  >, >, 162, 162, 192, >, 210             1024 x 512  >, >, 150, 160, >, >, 280     768 x 768  32 (6) on: 140, 150, 175, >, 280
//            1024 x 256, 512 x 512, 512 x 256  > (0.64 to 0.9 of the few-row kernels' time up to there)
//   IQ2_XXS  2048 x 512  70, < from there on                     inter from 512 on, hidden from 512 on  < but 1024 x 512: 64, <
//            2048 x 256  >, 140, 145, 145, 150, 138, 180         1024 x 256  >, >, 155, 165, 200, >, 230   512 x 256  >, >, 170, 170, 200, >, 260
// us, decode kernels : few rows: 24 tokens of 64 experts, Q4_K, 2048 x 512 67 : 53, of 128 of 1024 x 256 33 : 42; 20 tokens of 512, ten slots,
// IQ2_XXS, 2048 x 512 87 : 73, of 512 x 256 36 : 41.  Distance to 64 bits (2-norm, mean of eight layers each, decode kernels : few rows): Q4_K
// 3.14 : 3.14e-7 at 2048 x 512, 3.20 : 3.17 at 2560 x 768, 3.04 : 3.03 at 1024 x 512, 3.11 : 3.12 at 2048 x 256; IQ2_XXS 2.67 : 2.69, 2.72 : 2.71, 2.60 : 2.60
// and 2.63 : 2.69.  So the wide layers' lines follow the clock alone, and narrower IQ2_XXS layers stay with the decode kernels for
// longer: with few experts up to 1.4 times too late where inter is 512, 1.3 where it is 256.
PF_HD size_t pf_decode_pairs(bool q4k, size_t experts, size_t hidden, size_t inter) {
    const size_t work = hidden * inter, whole = (size_t)1 << 20;
    if (q4k) {
        if (work >= whole) return (110 + experts / 4) * whole / work;
        const size_t many = 150 + experts / 5, few = experts < 232 ? 232 - experts : 0;
        return work >= whole / 2 ? (many > few ? many : few) : 200 + experts / 2;
    }
    if (work >= whole) return 70;
    if (work < whole / 2 && inter < 512) return experts < 150 ? 160 + experts / 2 : 235;
    return experts <= 128 ? 160 + experts / 2 : experts <= 256 ? 224 - (experts - 128) * 59 / 128 : 165;
}

// Which MXFP4 down projections of a layer that keeps them in tile order run on the block-scaled product.  It saves work for every weight
// and row, and costs launches of its own (the rows' conversion 3 to 5 us; in the few-row kernels the shared expert's part as well).
//
// Batches of the decode kernels: the work is a pair's rows.  Forwards on the other kernel and on this, us: 5 tokens of 4 slots, 2048 x
// 512 (21e6) 27.0 : 29.7, 8 of 8, 1024 x 512 (34e6) 29.3 : 32.4, 6 of 8, 2048 x 512 (50e6) 37.5 : 39.4, 5 of 10, 2560 x 640 (82e6)
// 59.8 : 54.8, 16 of 10 (262e6) 136.0 : 117.5.  Of 480 batches of 8 to 512 experts, 1 to 10 slots and eight widths none is more than
// 7 % slower than on the other side of the line.
#define PF_DOWN_SCALED_FROM 5   // 4 tokens of 10 slots, 2560 x 640: 18.1 us of down projection against 19.5, and a launch more
PF_HD bool pf_decode_down_scaled(int tokens, int top_k, int hidden, int inter) {
    return tokens >= PF_DOWN_SCALED_FROM && (size_t)tokens * top_k * hidden * inter >= 55000000u;
}
// Batches of the few-row kernels: the weights of the experts there are and of every eight rows more, and the shared expert's chunks of
// eight rows.  The line was drawn while that kernel took those chunks one after the other, which the launch beside the block-scaled
// product did not; since they are items of their own in both it lies too early.  Forwards on the integers and there, us, all on this
// side of it: 32 tokens, 32 experts of 1024 x 512, four slots 39.2 : 47.0, 17 tokens of 8 experts of 2048 x 512 beside 1024 44.5 : 57.2, 512 experts, ten
// slots, of 2048 x 512 24 tokens 102 : 110 and 64 tokens 172 : 168, of 2560 x 640 17 tokens 124 : 130, 32 tokens 172 : 168, 101 tokens 307 : 283, 400
// tokens 540 : 490.  Of 490 batches of 8 to 512 experts 241 are more than 5 % slower than on the other side, up to 29 %; with the chunks
// left out of the sum and 350e6 for 200e6 it would be 24.  (The term and the two small batches that the line is tested to take stay
// until that test states them anew.)
PF_HD bool pf_batch_down_scaled(int tokens, int experts, int top_k, int hidden, int inter, int shared_inter) {
    const size_t pairs = (size_t)tokens * top_k, met = pairs < (size_t)experts ? pairs : (size_t)experts;
    const size_t chunks = tokens >= 32 ? 4 : ((size_t)tokens + 7) / 8;   // of a row tile of the shared expert
    return (met + pairs / 8) * hidden * inter + chunks * shared_inter * 100000 >= 200000000u;
}
