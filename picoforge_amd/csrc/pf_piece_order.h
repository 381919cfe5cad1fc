// How a ring piece's workgroups tell the host that the piece is done (pf_k_copy_piece in pf_moe_api.hip).  A template over the
// memory operations, so that a host-side check (tests/check_piece_order.cpp) runs the same steps against the memory model.
//
// A thread of every workgroup comes here once all of the workgroup's accesses have been made.  Outgoing rows have many writers and
// one number: each workgroup's rows are ordered before its arrival by a fence, and the last one, which has read all the other
// arrivals, orders what they ordered before the number by another (777 rows of 8 KB: 737 us a call without it, 739 with it).  Incoming
// rows are for the stream's next kernel alone; their number says only that the host's piece has been read, and a value that has been
// stored has been read.
#pragma once
#include "pf_decode_addr.h"

template <class Ops> PF_HD void pf_piece_done(Ops o, uint32_t workgroups, uint32_t number, bool out) {
    if (out) o.fence();
    if (o.arrive() != workgroups - 1) return;
    if (out) o.fence();
    o.clear();   // for the next launch on the stream
    o.publish(number);
}
