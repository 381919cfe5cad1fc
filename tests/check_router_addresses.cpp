// Host-side walk over every load that a chunk's router (pf_k_pf_router) makes of the experts' parts.  Compiled with g++ by
// tests/test_router_addresses.py; includes the header the kernel takes its addresses from (picoforge_amd/csrc/pf_router_addr.h).  For
// every workgroup column of a grid of 32- and of 64-expert tiles it checks that each load ends inside the allocation, and that the loads
// reach every byte of it.  Prints the number of loads checked; exit status 1 on a violation.
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "../picoforge_amd/csrc/pf_router_addr.h"

int main(int argc, char **argv) {
    if (argc != 3) {
        fprintf(stderr, "usage: %s experts hidden\n", argv[0]);
        return 2;
    }
    const int E = atoi(argv[1]), H = atoi(argv[2]);
    const size_t bytes = pf_router_parts_bytes(E, H);
    long long checked = 0, bad = 0;
    for (int tc = 1; tc <= 2; tc++) {
        std::vector<unsigned char> reached(bytes / 16);
        for (int first = 0; 32 * first < E; first += tc)   // a workgroup column's first tile
            for (int c = 0; c < tc; c++) {
                const int tile = pf_router_tile_read(E, first, c);
                for (int step = 0; step < H / 16; step++)
                    for (int part = 0; part < 3; part++)
                        for (int lane = 0; lane < 64; lane++, checked++) {
                            const size_t at = pf_router_tile_at(first, H) + pf_router_part_at(tile, H, step, part, lane);
                            if (tile < 0 || at + 16 > bytes || at % 16) {
                                if (bad++ < 10)
                                    fprintf(stderr, "%d experts, %d tiles a workgroup, tiles from %d: tile %d step %d part %d lane %d reads [%zu, +16) of %zu bytes\n", E, tc, first, c,
                                            step, part, lane, at, bytes);
                            } else {
                                reached[at / 16] = 1;
                            }
                        }
            }
        for (size_t i = 0; i < reached.size(); i++)
            if (!reached[i] && bad++ < 10) fprintf(stderr, "%d experts, %d tiles a workgroup: bytes %zu are not read\n", E, tc, 16 * i);
    }
    printf("%lld loads\n", checked);
    return bad != 0;
}
