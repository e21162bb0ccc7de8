// Checks of the library's host-callable index and protocol functions (opencfd-ec_amd/csrc), built and
// run on the CPU by test_csrc_functions.py: argv[1] names the check, the exit status is its result.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <vector>

#include "ocfd_dev.h"

using namespace ocfd;

#define CHECK(c, ...)                                                            \
    do {                                                                         \
        if (!(c)) { std::printf("%s: ", #c); std::printf(__VA_ARGS__); std::printf("\n"); return 1; } \
    } while (0)

// Four waves in lockstep by barriers, in every order between two of them: when one or two of them give
// up, all leave at the barrier that ends the round of the first (or at the tile's end).
static int give_up() {
    for (int nsteps : {1, 3, 4, 5, 8, 13})
        for (int q1 = 0; q1 < nsteps; q1++)
            for (int q2 = q1; q2 < nsteps; q2++)
                for (int w1 = 0; w1 < 4; w1++)
                    for (int w2 = 0; w2 < 4; w2++) {
                        int order[4] = {0, 1, 2, 3};
                        do {
                            GaveUp g;
                            g.start(0);
                            int left[4] = {nsteps, nsteps, nsteps, nsteps};
                            // between two barriers a wave asks about the step that ended, if it ended
                            // a round, and then works on the next step, in which it may give up
                            for (int q = 0; q <= nsteps; q++)
                                for (int w : order) {
                                    if (left[w] < q) continue;
                                    if (q > 0 && q % LU_RING == 0 && g.raised(q - 1)) { left[w] = q - 1; continue; }
                                    if (q < nsteps && ((w == w1 && q == q1) || (w == w2 && q == q2))) g.raise(q);
                                }
                            const int end = q1 / LU_RING * LU_RING + LU_RING - 1, expect = end < nsteps ? end : nsteps;
                            for (int w = 0; w < 4; w++)
                                CHECK(left[w] == expect, "nsteps %d, waves %d and %d at steps %d and %d: wave %d leaves at %d, not %d", nsteps,
                                      w1, w2, q1, q2, w, left[w], expect);
                        } while (std::next_permutation(order, order + 4));
                    }
    return 0;
}

int main(int argc, char** argv) {
    if (argc > 1 && !std::strcmp(argv[1], "give_up")) return give_up();
    std::printf("unknown check\n");
    return 2;
}
