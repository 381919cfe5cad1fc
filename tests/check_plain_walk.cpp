// Host-side walk of the plain grouped product's weight batches.  Compiled with g++ by tests/test_plain_walk.py; includes the
// header the kernel takes its order from (picoforge_amd/csrc/pf_plain_walk.h).  For a row of `width` columns in batches of
// `batch_cols` shared by `parts` waves, every wave is walked and each multiplication checked: the batch in hand is the one the
// columns belong to, requests stay inside the row, and the waves together multiply every batch once.
// usage: check_plain_walk width batch_cols parts; prints the multiplications, exit status 1 on a violation.
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "../picoforge_amd/csrc/pf_plain_walk.h"

int main(int argc, char **argv) {
    if (argc != 4) return 2;
    const int width = atoi(argv[1]), batch_cols = atoi(argv[2]), parts = atoi(argv[3]), batches = (width + batch_cols - 1) / batch_cols;
    std::vector<int> times(batches);
    int bad = 0, total = 0;
    auto expect = [&](bool ok, const char *what, int part, int c0, int k0) {
        if (!ok && bad++ < 10) fprintf(stderr, "wave %d, columns %d + %d: %s\n", part, c0, k0, what);
    };
    for (int part = 0; part < parts; part++) {
        int staged = -1, staged_cols = 0, next = -1, held = -1, rounds = 0;
        pf_plain_walk(width, batch_cols, part, parts, true,
            [&](int c0, int cols) {
                expect(c0 == rounds * PF_PLAIN_CHUNK && cols > 0 && c0 + cols <= width, "another round staged", part, c0, 0);
                staged = c0; staged_cols = cols; rounds++;
            },
            [&](int batch) { expect(batch >= 0 && batch < batches, "a request beyond the row", part, staged, batch); next = batch; },
            [&] { held = next; },
            [&](int k0, int cols) {
                expect(cols == staged_cols && k0 >= 0 && k0 < cols && k0 % batch_cols == 0, "columns that are not staged", part, staged, k0);
                expect(held == (staged + k0) / batch_cols, "another batch's weights", part, staged, k0);
                if (held >= 0 && held < batches) times[held]++;
                total++;
            });
        expect(rounds == (width + PF_PLAIN_CHUNK - 1) / PF_PLAIN_CHUNK, "a round left out", part, 0, 0);   // its barriers
        // a wave without rows stages (and meets the barriers) and multiplies nothing
        int idle = 0;
        pf_plain_walk(width, batch_cols, part, parts, false, [&](int, int) { idle++; }, [&](int) { expect(false, "an idle wave requests", part, 0, 0); },
                      [] {}, [&](int, int) { expect(false, "an idle wave multiplies", part, 0, 0); });
        expect(idle == rounds, "an idle wave leaves out a round", part, 0, 0);
    }
    for (int b = 0; b < batches; b++) expect(times[b] == 1, "a batch not multiplied once", -1, 0, b * batch_cols);
    printf("%d\n", total);
    return bad != 0;
}
