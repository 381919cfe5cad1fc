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
