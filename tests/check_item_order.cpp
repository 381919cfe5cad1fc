// Host-side check of how the grouped products' launches cut their work (picoforge_amd/csrc/pf_item_order.h).  Compiled with g++ by
// tests/test_item_order.py.  Exit status 1 on a violation.
#include <stdio.h>
#include <vector>
#include "../picoforge_amd/csrc/pf_item_order.h"

static int bad = 0;
static void expect(bool ok, const char *what, int a, int b, int c) {
    if (!ok && bad++ < 10) printf("%s: %d %d %d\n", what, a, b, c);
}

// no workgroup has more slabs than it may, or none; compute units stay idle only where every slab has a workgroup of its own, and beyond
// that there are no more workgroups than needed
static void slabs() {
    for (int all = 1; all <= 40; all++)
        for (int most = 1; most <= 8; most++)
            for (unsigned tiles = 1; tiles <= 2000; tiles += tiles < 40 ? 1 : 37) {
                const int per = pf_slabs_each(all, most, tiles), groups = per > 0 ? (all + per - 1) / per : 0;
                expect(per >= 1 && per <= most, "slabs of a workgroup", all, most, (int)tiles);
                if (per < 1) continue;
                expect(per == 1 || tiles * (unsigned)groups >= PF_FULL_CHIP, "idle compute units", all, most, (int)tiles);
                if (tiles >= PF_FULL_CHIP) expect(groups == (all + most - 1) / most, "more workgroups than needed", all, most, (int)tiles);
                expect(all - (groups - 1) * per >= 1, "a workgroup without a slab", all, most, (int)tiles);
            }
}

// every item once, and no XCD with more than its share of the routed groups or the shared expert's tiles
static void places() {
    const uint32_t routed_of[] = {0, 1, 7, 8, 9, 63, 64, 65, 75, 640, 1001}, shared_of[] = {0, 1, 5, 8, 9, 11, 24, 64};
    for (uint32_t routed : routed_of)
        for (uint32_t shared : shared_of)
            for (int slabs = 1; slabs <= 12; slabs++)
                for (uint32_t more : {0u, 40u, 300u}) {   // the numbers are for an upper bound of the routed tiles
                    const int shift = pf_group_shift(routed + more);
                    const uint32_t tiles = routed + shared, numbers = pf_item_numbers(slabs, shift, routed + more, shared);
                    std::vector<int> times((size_t)tiles * slabs);
                    uint32_t routed_on[PF_XCDS] = {}, shared_on[PF_XCDS] = {}, routed_seen[PF_XCDS] = {};
                    for (uint32_t q = 0; q < numbers; q++) {
                        const PfItemPlace p = pf_item_place(q, slabs, shift, routed, shared);
                        if (!p.any) continue;
                        if (p.tile < routed) routed_seen[q % PF_XCDS] = 1;
                        else expect(!routed_seen[q % PF_XCDS], "a shared tile behind a routed one", (int)routed, (int)shared, (int)q);
                        expect(p.tile < tiles && p.slab >= 0 && p.slab < slabs, "an item that is not there", (int)routed, (int)shared, (int)q);
                        if (p.tile >= tiles || p.slab < 0 || p.slab >= slabs) continue;
                        times[(size_t)p.tile * slabs + p.slab]++;
                        (p.tile < routed ? routed_on : shared_on)[q % PF_XCDS]++;
                    }
                    for (int t : times) expect(t == 1, "an item left out or taken twice", (int)routed, (int)shared, slabs);
                    for (int x = 0; x < PF_XCDS; x++) {   // an XCD's part: no more than a group above the least, and of them all
                        expect(shared_on[x] <= ((shared + PF_XCDS - 1) / PF_XCDS + (1u << shift)) * slabs, "the shared expert on few XCDs", (int)routed, (int)shared, (int)shared_on[x]);
                        expect(routed_on[x] <= (routed / PF_XCDS + (1u << shift)) * slabs, "routed tiles on few XCDs", (int)routed, (int)shared, (int)routed_on[x]);
                        expect(routed_on[x] + shared_on[x] <= (tiles / PF_XCDS + (1u << shift) + 1) * slabs, "tiles on few XCDs", (int)routed, (int)shared, x);
                    }
                    if (routed >= 8 && more == 0) expect(1u << shift <= (routed + 63) / 64, "groups larger than an eighth of an XCD's part", (int)routed, shift, 0);
                }
}

// batches that are clearly faster on one of the two down projections
static void decode_down() {
    expect(!pf_decode_down_scaled(5, 2, 768, 256) && !pf_decode_down_scaled(8, 2, 2048, 512) && !pf_decode_down_scaled(5, 4, 2048, 512), "small batches", 0, 0, 0);
    expect(pf_decode_down_scaled(5, 10, 2560, 640) && pf_decode_down_scaled(13, 10, 2560, 640) && pf_decode_down_scaled(8, 8, 2048, 512), "large batches", 0, 0, 0);
    expect(!pf_decode_down_scaled(4, 10, 2560, 640), "four tokens", 0, 0, 0);
}

static void batch_down() {
    expect(!pf_batch_down_scaled(17, 8, 2, 2048, 512, 512) && !pf_batch_down_scaled(400, 32, 2, 768, 256, 256) && !pf_batch_down_scaled(24, 128, 8, 512, 256, 256),
           "small batches", 0, 0, 0);
    expect(pf_batch_down_scaled(17, 512, 10, 2560, 640, 640) && pf_batch_down_scaled(101, 512, 10, 2560, 640, 640) && pf_batch_down_scaled(32, 32, 4, 1024, 512, 512),
           "large batches", 0, 0, 0);
}

int main() {
    batch_down();
    decode_down();
    slabs();
    places();
    return bad != 0;
}
