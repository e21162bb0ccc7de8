// The way of a tile's cells from the block arrays into the sweep-ordered storage of the pipelined
// LU-SGS sweeps (Pk in ocfd_dev.h).
#pragma once
#include "ocfd_dev.h"

namespace ocfd {

constexpr int PK_T = LU_COLS * PK_W;      // a thread per cell

// The steps [i0 - 1, i0 - 1 + n) of a tile whose DU elements the window of W cells from i0 on resets:
// as many as it has cells, the last window's to the tile's end, so a tile's windows take every step
// once.
__device__ __host__ __forceinline__ int sentinel_steps(int nx, int tj, int tk, int i0, int W) {
    return i0 + W == nx ? nx - 1 + tj + tk - 2 - (i0 - 1) : W;
}

// One tile and i-window of PK_W cells on its way from the block arrays to the sweep order, through
// LDS so both sides move in contiguous runs: get() reads, a thread per cell (i fastest) with all its
// fields in flight at once, put() writes, a wave per step with the lanes along the step's elements.
// What a lane writes of every step (field, column, place in the run) is worked out once per field
// group, not per element, and the pitch of PK_W + 2 keeps its skewed LDS reads on different banks.
template <int NV, int TJ>
struct PackTile {
    using F = Pk<NV>;
    static constexpr int TK = LU_COLS / TJ, ROWS = PK_W + TJ + TK - 2;      // steps a window's cells span
    double (*buf)[LU_COLS][PK_W + 2];
    const LuTask& T;
    const Blk& b;
    double* run;             // the run of the window's first step
    int i0, W;

    // the cells' N fields, f(s, v[N]) of box index s
    template <int N, typename Get>
    __device__ __forceinline__ void get(Get&& f) const {
        const int x = (int)threadIdx.x % PK_W, c = (int)threadIdx.x / PK_W, jl = c % TJ, kl = c / TJ;
        if (jl < T.tj && kl < T.tk && x < W) {
            double v[N];
            f(IX(b, i0 + x, T.j0 + jl, T.k0 + kl), v);
#pragma unroll
            for (int m = 0; m < N; m++) buf[m][c][x] = v[m];
        }
    }
    // element w (of N LU_COLS) of a step is field v of column c after at(w, v, c) and goes to the
    // run's element pos(w, v, c)
    template <int N, typename At, typename Pos>
    __device__ __forceinline__ void put(At&& at, Pos&& pos) const {
#pragma unroll
        for (int w = (int)threadIdx.x % 64; w < N * LU_COLS; w += 64) {
            int v, c;
            at(w, v, c);
            const int jl = c % TJ, kl = c / TJ, d = jl + kl;
            if (jl >= T.tj || kl >= T.tk) continue;
            const double* src = buf[v][c] - d;
            double* dst = run + pos(w, v, c);
#pragma unroll 4
            for (int q = (int)threadIdx.x / 64; q < ROWS; q += PK_T / 64)
                if (q >= d && q < d + W) dst[(size_t)q * F::RUN] = src[q];
        }
    }
    // the sentinel into both DU arrays, which end a run, of the window's own steps
    __device__ __forceinline__ void sentinel() const {
        const int steps = sentinel_steps(b.nx, T.tj, T.tk, i0, W);
        constexpr int PAIRS = (F::RUN - F::DUF) / 2;
        double2 s;
        s.x = s.y = sentinel_value();
        for (int e = (int)threadIdx.x; e < steps * PAIRS; e += PK_T)
            reinterpret_cast<double2*>(run + (size_t)(e / PAIRS) * F::RUN + F::DUF)[e % PAIRS] = s;
    }
};

}  // namespace ocfd
