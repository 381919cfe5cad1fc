// Host-side check of how the grouped products' launches cut their work (picoforge_amd/csrc/pf_item_order.h).  Compiled with g++ by
// tests/test_item_order.py.  Exit status 1 on a violation.
#include <stdio.h>
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

int main() {
    slabs();
    return bad != 0;
}
