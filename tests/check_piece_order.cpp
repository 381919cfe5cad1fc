// Happens-before check of pf_piece_done (picoforge_amd/csrc/pf_piece_order.h): its operations run on vector clocks, workgroup after
// workgroup in a random order of steps, with the C++ rules for fences, relaxed read-modify-writes (a release sequence goes on through
// them) and stores.  The host's acquire of the number has to come after every workgroup's rows.
//
//   check_piece_order WORKGROUPS OUT   prints "0 unordered workgroups"
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "../picoforge_amd/csrc/pf_piece_order.h"

typedef std::vector<unsigned> Clock;
static void join(Clock &a, const Clock &b) { for (size_t i = 0; i < a.size(); i++) if (b[i] > a[i]) a[i] = b[i]; }

struct Location { uint32_t value = 0; Clock released; };
struct Thread { Clock now, seen, fenced; };   // seen: what its relaxed reads would synchronise with; fenced: its last fence

struct Model {
    Thread *t;
    Location *counter, *word;
    void fence() { join(t->now, t->seen); t->fenced = t->now; }
    uint32_t arrive() {   // relaxed
        join(t->seen, counter->released);
        join(counter->released, t->fenced);
        return counter->value++;
    }
    void clear() { counter->value = 0; counter->released = t->fenced; }
    void publish(uint32_t number) { word->value = number; word->released = t->fenced; }   // relaxed
};

int main(int argc, char **argv) {
    if (argc != 3) return 2;
    const unsigned n = (unsigned)atoi(argv[1]);
    const bool out = atoi(argv[2]) != 0;
    const Clock zero(n, 0u);
    Location counter, word;
    counter.released = word.released = zero;
    unsigned unordered = 0;
    srand(n);
    for (uint32_t launch = 1; launch <= 3; launch++) {
        std::vector<Thread> group(n, Thread{zero, zero, zero});
        std::vector<unsigned> order(n);
        for (unsigned i = 0; i < n; i++) order[i] = i;
        for (unsigned i = n; i > 1; i--) { const unsigned j = (unsigned)rand() % i; const unsigned k = order[i - 1]; order[i - 1] = order[j]; order[j] = k; }
        counter.released = zero;   // a launch starts after the one before it
        for (unsigned i : order) {
            group[i].now[i] = launch;   // its rows
            pf_piece_done(Model{&group[i], &counter, &word}, n, launch, out);
        }
        if (word.value != launch || counter.value != 0) { printf("launch %u: no number\n", launch); return 1; }
        for (unsigned i = 0; i < n && out; i++) unordered += word.released[i] < launch;
    }
    printf("%u unordered workgroups\n", unordered);
    return unordered != 0;
}
