// Checks of the library's host-callable index and protocol functions (opencfd-ec_amd/csrc), built and
// run on the CPU by test_csrc_functions.py: argv[1] names the check, the exit status is its result.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <vector>

#include "ocfd_launch.h"
#include "ocfd_pack.h"

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

// The element order of a vector group and the places of a run's groups.
template <int NV>
static int vec() {
    using F = Pk<NV>;
    std::vector<int> seen(NV * LU_COLS, 0);
    for (int w = 0; w < NV * LU_COLS; w++) {
        int v, c;
        F::vec_at(w, v, c);
        CHECK(v >= 0 && v < NV && c >= 0 && c < LU_COLS, "NV %d element %d: component %d column %d", NV, w, v, c);
        CHECK(F::vec_off(v, c) == w, "NV %d element %d", NV, w);
        seen[v * LU_COLS + c]++;
    }
    for (int n : seen) CHECK(n == 1, "NV %d", NV);
    CHECK(F::DUB == F::DUF + NV * LU_COLS && F::RUN == F::DUB + NV * LU_COLS, "NV %d", NV);
    CHECK(F::DUF % 2 == 0 && F::RUN % 2 == 0 && F::NBR % 2 == 0, "NV %d: 16-byte pieces", NV);
    CHECK(lusgs_run(NV) == F::RUN, "NV %d", NV);
    return 0;
}

static int faces() {
    for (int scale : {1, 7, 61, 515})
        for (int m = 0; m < 125; m++) {
            const int n[3] = {m % 5 * scale + (m > 60), m / 5 % 5 * scale, m / 25 * scale - (m / 25 > 1)};
            std::vector<int> seen[3];
            for (int d = 0; d < 3; d++) seen[d].assign(n[d], 0);
            for (int w = 0; w < face_grid(n); w++) {
                int d, t;
                if (face_tile(w, n, d, t)) { CHECK(d >= 0 && d < 3 && t >= 0 && t < n[d], "workgroup %d", w); seen[d][t]++; }
            }
            for (int d = 0; d < 3; d++)
                for (int t = 0; t < n[d]; t++) CHECK(seen[d][t] == 1, "%d %d %d tiles: direction %d tile %d taken %d times", n[0], n[1], n[2], d, t, seen[d][t]);
        }
    return 0;
}

static const std::vector<std::vector<std::vector<int>>> LISTS = {
    {{3, 3, 3}},  {{2, 2, 2}}, {{17, 17, 9}}, {{33, 20, 13}, {9, 5, 18}}, {{34, 25, 9}}, {{12, 40, 7}, {20, 3, 3}, {2, 6, 31}},
    {{9, 65, 17}}, {{97, 4, 34}}, {{65, 34, 2}, {33, 2, 34}, {32, 9, 9}}};

// the steps a tile marches
static int nsteps(const Blk& b, const LuTask& t) { return b.nx - 1 + t.tj + t.tk - 2; }

static std::vector<Blk> blocks(const std::vector<std::vector<int>>& dims) {
    std::vector<Blk> out;
    for (const auto& d : dims) {
        Blk b{};
        b.nx = d[0]; b.ny = d[1]; b.nz = d[2];
        out.push_back(b);
    }
    return out;
}

// Tables of the sweeps: every cell in one tile and window, tiles apart in the storage, an upstream tile
// numbered lower, loads of steps before and behind a tile inside the buffer, and the DU elements of every
// step reset by exactly one window, those a neighbour tile waits for among them.
template <int NV>
static int tables() {
    const int run = Pk<NV>::RUN, far = LU_RING - 1;
    for (const auto& dims : LISTS)
        for (int tj : {4, 8, 16}) {
            const std::vector<Blk> blks = blocks(dims);
            const int tk = LU_COLS / tj;
            long long total = 0;
            std::vector<LuTask> f = lusgs_tasks(blks, true, run, tj, tk, &total), b = lusgs_tasks(blks, false, run, tj, tk, nullptr);
            lusgs_start_order(f);
            lusgs_start_order(b);
            CHECK(total % run == 0 && f.size() == b.size(), "tj %d", tj);
            // who holds a run of the storage, how often its DU elements are reset
            std::vector<int> owner(total / run, -1), reset(total / run, 0);
            std::vector<std::vector<int>> cells;
            for (const Blk& q : blks) cells.push_back(std::vector<int>((q.nx - 1) * (q.ny - 1) * (q.nz - 1), 0));
            for (size_t q = 0; q < f.size(); q++) {
                const LuTask& t = f[q];
                CHECK(t.pofs % run == 0 && t.tj >= 1 && t.tj <= tj && t.tk >= 1 && t.tk <= tk, "tile %zu", q);
                for (int s = 0; s < nsteps(blks[t.blk], t); s++) {
                    const long long r = t.pofs / run + s;
                    CHECK(r >= LU_PAD_STEPS && r < total / run - LU_PAD_STEPS && owner[r] < 0, "tile %zu step %d", q, s);
                    owner[r] = (int)q;
                }
            }
            for (const int2& w : lusgs_window_list(blks, f)) {
                const LuTask& t = f[w.x];
                const Blk& q = blks[t.blk];
                const int W = std::min(PK_W, q.nx - w.y), n = sentinel_steps(q.nx, t.tj, t.tk, w.y, W);
                for (int s = 0; s < n; s++) {
                    const long long r = t.pofs / run + w.y - 1 + s;
                    CHECK(owner[r] == w.x, "a window resets a run that is not its tile's (tile %d, i %d, step %d)", w.x, w.y, s);
                    reset[r]++;
                }
                for (int k = t.k0; k < t.k0 + t.tk; k++)
                    for (int j = t.j0; j < t.j0 + t.tj; j++)
                        for (int i = w.y; i < w.y + W; i++) cells[t.blk][i - 1 + (q.nx - 1) * (j - 1 + (q.ny - 1) * (k - 1))]++;
            }
            for (size_t r = 0; r < reset.size(); r++) CHECK(reset[r] == (owner[r] >= 0), "run %zu reset %d times (NV %d, tj %d)", r, reset[r], NV, tj);
            for (const auto& c : cells)
                for (int n : c) CHECK(n == 1, "a cell in %d windows", n);
            for (bool fwd : {true, false}) {
                const std::vector<LuTask>& l = fwd ? f : b;
                for (int q = 0; q < (int)l.size(); q++) {
                    const LuTask& t = l[q];
                    const Blk& k = blks[t.blk];
                    const int ns = nsteps(k, t), d = fwd ? 1 : -1;
                    // the run of the tile's step s, and of the cells its edge lanes need at that step
                    const long long own = t.pofs / run + (fwd ? 0 : ns - 1);
                    CHECK(own - d >= 0 && own + d * (ns + far) >= 0 && own + d * (ns + far) < total / run && own - d < total / run, "tile %d", q);
                    for (int e = 0; e < 2; e++) {
                        const int dep = e ? t.dep_k : t.dep_j;
                        if (dep < 0) continue;
                        CHECK(dep < q && l[dep].blk == t.blk, "tile %d waits for tile %d", q, dep);
                        const LuTask& u = l[dep];
                        CHECK(u.pofs == (e ? t.pofs_k : t.pofs_j) && (e ? u.tk == t.tk_up && u.tj == t.tj : u.tj == t.tj_up && u.tk == t.tk), "tile %d", q);
                        CHECK(e ? u.j0 == t.j0 && (fwd ? u.k0 + u.tk == t.k0 : t.k0 + t.tk == u.k0) : u.k0 == t.k0 && (fwd ? u.j0 + u.tj == t.j0 : t.j0 + t.tj == u.j0), "tile %d", q);
                        const long long up = u.pofs / run + (fwd ? (e ? u.tk : u.tj) - 1 : k.nx - 1 + (e ? t.tj : t.tk) - 2);
                        CHECK(up >= 0 && up < total / run && up + d * (ns + far) >= 0 && up + d * (ns + far) < total / run, "tile %d", q);
                        // the upstream column across the edge at each cell of the lane beside it
                        for (int x = 0; x < (e ? t.tj : t.tk); x++)
                            for (int i = 1; i < k.nx; i++) {
                                const int jl = e ? x : fwd ? u.tj - 1 : 0, kl = e ? (fwd ? u.tk - 1 : 0) : x;
                                const long long r = u.pofs / run + i - 1 + jl + kl;
                                const int lag = fwd ? x : (e ? t.tj : t.tk) - 1 - x, s = fwd ? i - 1 + lag : k.nx - 1 - i + lag;
                                CHECK(r == up + d * s && owner[r] >= 0 && reset[r] == 1 && f[owner[r]].pofs == u.pofs,
                                      "tile %d waits for a run that its upstream tile does not reset (NV %d, tj %d, i %d)", q, NV, tj, i);
                            }
                    }
                }
            }
        }
    return 0;
}

int main(int argc, char** argv) {
    if (argc > 1 && !std::strcmp(argv[1], "give_up")) return give_up();
    if (argc > 1 && !std::strcmp(argv[1], "vector_groups")) return vec<5>() | vec<6>() | vec<7>();
    if (argc > 1 && !std::strcmp(argv[1], "face_tiles")) return faces();
    if (argc > 1 && !std::strcmp(argv[1], "sweep_tables")) return tables<5>() | tables<6>() | tables<7>();
    std::printf("unknown check\n");
    return 2;
}
