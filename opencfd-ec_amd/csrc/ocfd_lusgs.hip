// LU-SGS sweeps (du_LU_SGS, sub_LU_SGS.f90:4-129) as one persistent, pipelined launch per sweep.
//
// The forward sweep of a cell needs the final DU of its i-1, j-1 and k-1 neighbours (the
// backward sweep: i+1, j+1, k+1), and nothing else that changes during the sweep.  Any order that
// honours those three dependencies gives the reference's hyperplane result bit for bit, because
// every cell evaluates the same expression in the same order once its neighbours are final.
//
// Fenced schedule: the (j,k) cross-section of a block is cut into 8x8 tiles; one 64-lane wave owns a
// tile and marches along i, lane (jl,kl) handling cell i = q - jl - kl + 1 at local step q (a
// hyperplane inside the tile).  Within the tile the j/k neighbours come through LDS (the lane
// that computed them one step earlier) and the i neighbour stays in registers.  Across tiles the
// upstream tile publishes its last completed step in a progress counter (agent-scope release)
// and the downstream tile waits (agent-scope acquire) for the step that produced the cells it
// reads.  Tiles are numbered so that every upstream tile has a lower workgroup index; workgroups
// are dispatched in index order, so every wait is on a workgroup already running or finished,
// and every wait is also bounded by a poll limit that raises an error flag instead of hanging.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "ocfd_dev.h"
#include "ocfd_launch.h"
#include "ocfd_pack.h"
#include "ocfd_phys.h"

namespace ocfd {

constexpr int LU_TJ = 8, LU_TK = 8;
static_assert(LU_TJ * LU_TK == LU_NT, "the fenced sweep's tiles are 8 x 8");
constexpr long LU_POLL_LIMIT = 1L << 26;
constexpr int LU_HOP = 5;             // steps a tile trails its upstream tile by beyond that tile's width

// err[0]: the error flag a wait sets when it gives up.  err[2]: nonzero makes every wait that
// finds its producer behind give up at its first poll (the host's failure-path test).  The poll
// limit itself stays a compile-time constant: a limit read at run time changes the register
// allocation of the team sweep and costs it a sixth of its speed.
__device__ __forceinline__ bool lu_fail_waits(const int* err) {
    return __hip_atomic_load(err + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// Per-lane record shared through LDS with the downstream lanes of the tile.
template <int NV>
struct LuSlot {
    double U[NV], DU[NV];
    double Lc[2], Lv[2], S[2];   // j and k direction values of the cell (S: backward sweep only)
};

template <int NV, bool FWD>
__global__ void __launch_bounds__(LU_NT) k_lusgs_sweep(const Blk* __restrict__ blks, const LuTask* __restrict__ tasks,
                                                       int* __restrict__ prog, int* __restrict__ prog_other,
                                                       int n_other, int* __restrict__ err, Par p) {
    __shared__ LuSlot<NV> slot[2][LU_NT];
    __shared__ int gave_up;
    const int w = blockIdx.x, lane = threadIdx.x;
    // this launch re-arms the counters of the other sweep (same tile count) for its next launch
    if (lane == 0 && w < n_other) prog_other[w] = -1;
    // a sweep of this iteration (or an earlier one of the same launch sequence) gave up: nothing to do
    if (lane == 0) gave_up = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (gave_up != 0) return;

    const LuTask T = tasks[w];
    const Blk& b = blks[T.blk];
    const int jl = lane % LU_TJ, kl = lane / LU_TJ;
    const bool live = jl < T.tj && kl < T.tk;
    // tile-local offsets along the sweep direction
    const int jo = FWD ? jl : T.tj - 1 - jl, ko = FWD ? kl : T.tk - 1 - kl;
    const int j = T.j0 + jl, k = T.k0 + kl;
    const int nxm = b.nx - 1;
    const size_t sj = (size_t)b.NI, sk = (size_t)b.NI * b.NJ;
    const double wlu = p.w_LU, gamma = p.gamma;
    const bool visc = p.visc == 1;
    const int nsteps = nxm + T.tj + T.tk - 2;
    int known_j = -1, known_k = -1;

    // i-direction neighbour (the previous cell of this lane)
    double pU[NV], pDU[NV], pLc = 0.0, pLv = 0.0, pS = 0.0;
#pragma unroll
    for (int m = 0; m < NV; m++) { pU[m] = 0.0; pDU[m] = 0.0; }

    for (int q = 0; q < nsteps; q++) {
        const int buf = q & 1;
        // ---- wait for the upstream tiles (lane 0 polls, the barrier releases the wave) ----
        if (lane == 0) {
            int need_j = T.dep_j >= 0 ? min(q + T.off_j, T.last_j) : -1;
            int need_k = T.dep_k >= 0 ? min(q + T.off_k, T.last_k) : -1;
            bool fresh = false;
            long polls = 0;
            while (known_j < need_j || known_k < need_k) {
                if (known_j < need_j) known_j = __hip_atomic_load(prog + T.dep_j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (known_k < need_k) known_k = __hip_atomic_load(prog + T.dep_k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                fresh = true;
                if (known_j >= need_j && known_k >= need_k) break;
                if (++polls > LU_POLL_LIMIT || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
                    lu_fail_waits(err)) {
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    known_j = known_k = -2;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (fresh) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) return;

        const int i = FWD ? q - jo - ko + 1 : nxm - (q - jo - ko);
        const bool act = live && i >= 1 && i <= nxm;
        double oU[NV], oDU[NV], oLc1 = 0.0, oLc2 = 0.0, oLv1 = 0.0, oLv2 = 0.0, oS1 = 0.0, oS2 = 0.0;
        if (act) {
            const size_t s = IX(b, i, j, k);
            double Lc0 = b.Lc[0][s], Lc1 = b.Lc[1][s], Lc2 = b.Lc[2][s];
            double Lv0 = b.Lv[0][s], Lv1 = b.Lv[1][s], Lv2 = b.Lv[2][s];
            double vol = b.vol[s];
            double sumLc = (Lc0 + Lc1) + Lc2;
            double sumLv = (Lv0 + Lv1) + Lv2;
            double alfa0 = vol / b.dt[s] + wlu * sumLc;
            double alfa[NV];
#pragma unroll
            for (int m = 0; m < NV; m++) alfa[m] = alfa0;
            if (visc) {
#pragma unroll
                for (int m = 0; m < NV; m++) alfa[m] = alfa[m] + 2.0 * sumLv;
                if (NV == 6) {
                    if (FWD) alfa[5] = alfa[5] + sumLv;
                    else alfa[5] = ((alfa[5] + Lv0) + Lv1) + Lv2;
                }
            }
#pragma unroll
            for (int m = 0; m < NV; m++) alfa[m] = alfa[m] + 0.0 * vol;
            double acc[NV];
#pragma unroll
            for (int m = 0; m < NV; m++) acc[m] = FWD ? b.Res[m][s] : 0.0;
#pragma unroll
            for (int dir = 0; dir < 3; dir++) {
                const int pos = dir == 0 ? i : (dir == 1 ? j : k);
                const int lim = dir == 0 ? nxm : (dir == 1 ? b.ny - 1 : b.nz - 1);
                const bool has = FWD ? pos != 1 : pos != lim;
                double du[NV];
                if (has) {
                    double Un[NV], DUn[NV], Lcn, Lvn, Sn;
                    const int src = dir == 0 ? 0 : (dir == 1 ? (jo > 0 ? 1 : 2) : (ko > 0 ? 1 : 2));
                    if (src == 0) {            // previous cell of this lane
#pragma unroll
                        for (int m = 0; m < NV; m++) { Un[m] = pU[m]; DUn[m] = pDU[m]; }
                        Lcn = pLc; Lvn = pLv; Sn = pS;
                    } else if (src == 1) {     // lane of the same tile, one step earlier
                        const int nl = dir == 1 ? (FWD ? lane - 1 : lane + 1) : (FWD ? lane - LU_TJ : lane + LU_TJ);
                        const LuSlot<NV>& o = slot[buf ^ 1][nl];
                        const int d = dir - 1;
#pragma unroll
                        for (int m = 0; m < NV; m++) { Un[m] = o.U[m]; DUn[m] = o.DU[m]; }
                        Lcn = o.Lc[d]; Lvn = o.Lv[d]; Sn = o.S[d];
                    } else {                   // upstream tile, through global memory
                        const size_t t = FWD ? s - (dir == 1 ? sj : sk) : s + (dir == 1 ? sj : sk);
#pragma unroll
                        for (int m = 0; m < NV; m++) { Un[m] = b.U[m][t]; DUn[m] = b.DU[m][t]; }
                        Lcn = b.Lc[dir][t]; Lvn = b.Lv[dir][t]; Sn = FWD ? 0.0 : b.S[dir][t];
                    }
#pragma unroll
                    for (int m = 5; m < NV; m++) if (Un[m] < 0.0) Un[m] = 0.0;     // limit_vt
                    double DF[NV];
                    comput_dfn<NV>(DF, Un, DUn, b.nv[3 * dir][s], b.nv[3 * dir + 1][s], b.nv[3 * dir + 2][s], gamma);
                    const double wLc = wlu * Lcn;
                    if (FWD) {
                        const double Sd = b.S[dir][s];
#pragma unroll
                        for (int m = 0; m < NV; m++) du[m] = 0.5 * (DF[m] * Sd + wLc * DUn[m]);
                    } else {
#pragma unroll
                        for (int m = 0; m < NV; m++) du[m] = -0.5 * (DF[m] * Sn - wLc * DUn[m]);
                    }
                    if (visc) {
#pragma unroll
                        for (int m = 0; m < NV; m++) du[m] = du[m] + Lvn * DUn[m];
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < NV; m++) du[m] = 0.0;
                }
#pragma unroll
                for (int m = 0; m < NV; m++) acc[m] = acc[m] + du[m];
            }
#pragma unroll
            for (int m = 0; m < NV; m++) {
                oU[m] = b.U[m][s];
                oDU[m] = FWD ? acc[m] / alfa[m] : b.DU[m][s] + acc[m] / alfa[m];
                b.DU[m][s] = oDU[m];
            }
            oLc1 = Lc1; oLc2 = Lc2; oLv1 = Lv1; oLv2 = Lv2;
            if (!FWD) { oS1 = b.S[1][s]; oS2 = b.S[2][s]; }
            // this cell is the i neighbour of the lane's next cell
#pragma unroll
            for (int m = 0; m < NV; m++) { pU[m] = oU[m]; pDU[m] = oDU[m]; }
            pLc = Lc0; pLv = Lv0; pS = FWD ? 0.0 : b.S[0][s];
        }
        LuSlot<NV>& me = slot[buf][lane];
        if (act) {
#pragma unroll
            for (int m = 0; m < NV; m++) { me.U[m] = oU[m]; me.DU[m] = oDU[m]; }
            me.Lc[0] = oLc1; me.Lc[1] = oLc2; me.Lv[0] = oLv1; me.Lv[1] = oLv2; me.S[0] = oS1; me.S[1] = oS2;
        }
        __syncthreads();
        if (lane == 0) __hip_atomic_store(prog + w, q, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------------------------
// Team sweep: the same in-tile hyperplanes on tiles of 16 (j,k) columns, four lanes (a DPP quad) per
// column, three direction waves and a loader wave per tile.  Wave d (d = 0, 1, 2 for i, j, k) owns
// the contribution of the upstream neighbour in direction d.  At step q each wave first completes
// the DU of the cell it reads, the one its lane's neighbour computed at step q - 1 (its own previous
// cell for d = 0, the column across the j or k step for d = 1, 2): DU = (((Res + du_i) + du_j) + du_k) / alfa in the reference's order (backward sweep:
// DU + ((du_i + du_j) + du_k) / alfa) from the three waves' terms of step q - 1 in LDS.  It then
// evaluates the neighbour term of its direction for its own cell and writes it to LDS.  One
// workgroup barrier per step separates the terms of a step from their use in the next; the LDS
// terms are double-buffered by step parity.  Wave 0 stores each completed DU of its own cell.
//
// What bounds it: a lone tile's step is one wave's instruction stream (every instruction of a wave
// alone on its SIMD takes 4 to 5 clocks, dependent or not) plus the exchange (two LDS writes, the
// barrier and six LDS reads, about 210 clocks).  Hence the split: a quad holds a column's components
// (momentum and energy in the first slot, density and the turbulence variables in the second), so a
// wave issues about 70 FP64 and 24 DPP instructions per step where a lane with all components issued
// 170 FP64; the loader brings a step's inputs to the LDS by 16-byte loads (45 8-byte loads by the
// direction waves cost more than the arithmetic: 0.69 us per step with them, 0.36 without); and the
// pressure and the reciprocals that do not depend on DU are formed once per cell by the pack.  A
// step takes 0.42 us against 1.05 to 1.35 us with 64 columns per wave and all components per lane:
// forward sweep of the 257x97x33 C-grid (SA) 528 -> 238 us, of the 97x33x9 channel 137 -> 78, of the
// 24-block wing with 6.3 M cells 1085 -> 732.  A tile trails its upstream tile by about 2 us beyond
// its own width, so long chains of narrow tiles lose (16x1 tiles), and a launch starts its tiles in
// the order in which they can run (lusgs_start_order): block after block, the wing's sweep took
// 1560 us instead of 1120 with the same kernel, most resident tiles waiting.
//
// Cross-tile values travel through the sweep-ordered DU arrays themselves.  Before a sweep every
// element of the array it writes holds a sentinel NaN (a payload no arithmetic produces); the
// producer overwrites an element read by a neighbour tile with a device-coherent 64-bit store and
// the consumer reloads it, device-coherent, until the sentinel is gone.  No progress counter and
// no wait for store completion sit on the producer's path.  The forward sweep writes DUF and the
// backward sweep DUB; the pack of the next sweeps' inputs puts the sentinel back into both.
// Tiles are numbered upstream first and workgroups start in index order, so every wait is on a
// tile that is running or done; every wait is also bounded by a poll limit that raises the error
// flag.

__device__ __forceinline__ void st_coherent(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_coherent(const double* p) {
    return __longlong_as_double((long long)__hip_atomic_load(reinterpret_cast<unsigned long long*>(const_cast<double*>(p)),
                                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}


// the geometry the sweeps read (S, n), into sweep order once per plan
template <int NV, int TJ>
__global__ void __launch_bounds__(PK_T) k_lu_pack_geometry(ctab<Blk> blks, ctab<LuTask> tiles,
                                                           double* __restrict__ pk, ctab<int2> wins) {
    using F = Pk<NV>;
    __shared__ double buf[3][LU_COLS][PK_W + 2];
    const int2 wn = wins[xcd_tile((int)blockIdx.x, (int)gridDim.x)];
    const LuTask T = tiles[wn.x];
    const Blk& b = blks[T.blk];
    const PackTile<NV, TJ> P{buf, T, b, pk + T.pofs + (long long)(wn.y - 1) * F::RUN, wn.y, min(PK_W, b.nx - wn.y)};
    auto third = [](int w, int& v, int& c) { c = w / 3; v = w % 3; };
    P.template get<3>([&](size_t s, double* u) {
#pragma unroll
        for (int d = 0; d < 3; d++) u[d] = b.S[d][s];
    });
    __syncthreads();
    P.template put<3>(third, [](int, int v, int c) { return F::SG + 4 * c + v; });
#pragma unroll
    for (int d = 0; d < 3; d++) {
        __syncthreads();
        P.template get<3>([&](size_t s, double* u) {
#pragma unroll
            for (int r = 0; r < 3; r++) u[r] = b.nv[3 * d + r][s];
        });
        __syncthreads();
        P.template put<3>(third, [=](int, int v, int c) { return F::N + 9 * c + 3 * d + v; });
    }
}

// sweep order -> block arrays for the backward sweep's DU, for a host that reads DU: the storage
// holds it from the end of the backward sweep until the next pack
template <int NV, int TJ>
__global__ void __launch_bounds__(PK_T) k_lu_du_to_box(ctab<Blk> blks, ctab<LuTask> tiles,
                                                       const double* __restrict__ pk, ctab<int2> wins) {
    using F = Pk<NV>;
    constexpr int M = NV * LU_COLS;
    __shared__ double buf[NV][LU_COLS][PK_W + 2];
    const int2 wn = wins[xcd_tile((int)blockIdx.x, (int)gridDim.x)];
    const LuTask T = tiles[wn.x];
    const Blk& b = blks[T.blk];
    const int i0 = wn.y, W = min(PK_W, b.nx - 1 - i0 + 1), t = (int)threadIdx.x;
    for (int e = t; e < (W + TJ + LU_COLS / TJ - 2) * M; e += PK_T) {
        const int q = i0 - 1 + e / M, w = e % M;
        int v, c;
        F::vec_at(w, v, c);
        const int jl = c % TJ, kl = c / TJ, x = q - jl - kl + 1 - i0;
        if (jl < T.tj && kl < T.tk && x >= 0 && x < W) buf[v][c][x] = pk[(size_t)T.pofs + (size_t)q * F::RUN + F::DUB + w];
    }
    __syncthreads();
    for (int e = t; e < M * PK_W; e += PK_T) {
        const int x = e % PK_W, c = (e / PK_W) % LU_COLS, v = e / (PK_W * LU_COLS), jl = c % TJ, kl = c / TJ;
        if (jl < T.tj && kl < T.tk && x < W) b.DU[v][IX(b, i0 + x, T.j0 + jl, T.k0 + kl)] = buf[v][c][x];
    }
}

// the sentinel into every DUF and DUB element (and the padding)
template <int NV>
__global__ void k_fill_sentinel(double* p, long long n) {
    using F = Pk<NV>;
    const long long pad = (long long)LU_PAD_STEPS * F::RUN;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        if (e < pad || e >= n - pad || (int)((e - pad) % F::RUN) >= F::DUF) p[e] = sentinel_value();
    }
}


// value x of part M of the lane's quad
template <int M>
__device__ __forceinline__ double quad_get(double x) {
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)v, M * 0x55, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), M * 0x55, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double quad_sum3(double x) { return (quad_get<0>(x) + quad_get<1>(x)) + quad_get<2>(x); }

// the convective flux F(U) n of comput_DFn (sub_LU_SGS.f90:135-158) in the quad's components, from
// the density d, its reciprocal and the pressure; the normal velocity is formed by all four lanes
__device__ __forceinline__ void quad_flux(double Ua, double Ub, double d, double rd, double p, double n, bool energy, double& fa, double& fb) {
    const double un = div_nr(quad_sum3(Ua * n), d, rd);
    const double fm = Ua * un + p * n, fe = (Ua + p) * un;
    fa = energy ? fe : fm;
    fb = Ub * un;
}

// du of one upstream neighbour component (sub_LU_SGS.f90:42-60 forward, :94-119 backward); without
// viscosity Lv is zero
template <bool FWD>
__device__ __forceinline__ double team_term(double DF, double DU, double wLc, double Lv, double S) {
    const double t = FWD ? 0.5 * (DF * S + wLc * DU) : -0.5 * (DF * S - wLc * DU);
    return t + Lv * DU;
}

// a for the lanes whose bit of mk is set, else b: one v_cndmask per half, so the choice cannot
// become a masked overwrite of a register that a load may still be filling
__device__ __forceinline__ double pick(unsigned long long mk, double a, double b) {
    const unsigned long long ua = (unsigned long long)__double_as_longlong(a), ub = (unsigned long long)__double_as_longlong(b);
    unsigned lo, hi;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(lo) : "v"((unsigned)ub), "v"((unsigned)ua), "s"(mk));
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(hi) : "v"((unsigned)(ub >> 32)), "v"((unsigned)(ua >> 32)), "s"(mk));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// the high half of the sentinel is enough to know it by: no arithmetic produces a signalling NaN
__device__ __forceinline__ bool maybe_sentinel(double v) {
    return (unsigned)(__double_as_longlong(v) >> 32) == (unsigned)(LU_SENTINEL >> 32);
}

// reload an upstream DU (elements ea, eb) on the waiting lanes until the producer has replaced the
// sentinel; true when the wait gives up
__device__ __forceinline__ bool team_wait_remote(const double* ea, const double* eb, bool waiting, double& a, double& b, int* __restrict__ err) {
    long polls = 0;
    while (true) {
        const bool pend = waiting && (is_sentinel(a) || is_sentinel(b));
        if (__builtin_amdgcn_ballot_w64(pend) == 0) return false;
        if (++polls > LU_POLL_LIMIT ||
            ((polls & 255) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) ||
            (polls == 1 && lu_fail_waits(err))) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return true;
        }
        if (pend) { a = ld_coherent(ea); b = ld_coherent(eb); }
    }
}

__device__ __forceinline__ void team_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// LDS of a tile team.  ring: LU_RING slots of step inputs, filled by the loader wave; slot q holds
// step q's piece of the tile's run (R to N forward, NBR to DUF backward) and, for the lanes at the
// tile's upstream edges, the NBR (and backward SG) chunks that step q + 1 reads of the upstream
// tiles.  du: the three direction waves' neighbour terms, double-buffered by step parity.
constexpr int LU_FAR = LU_RING - 1;      // how many steps ahead the loader writes
template <int NV, bool FWD, int TJ> struct TeamLds {
    using F = Pk<NV>;
    static constexpr int BASE = FWD ? F::R : F::NBR;                 // first double of a run's piece
    static constexpr int EDGE = TJ + LU_COLS / TJ;                   // upstream columns: along j, then along k
    static constexpr int PIECE = F::SWEEP * 8, NBRS = PIECE, SGS = NBRS + EDGE * F::CS * 8,
                         SLOT = (SGS + (FWD ? 0 : EDGE * 32) + 15) / 16 * 16;      // byte offsets in a slot
    static constexpr int CHUNKS = EDGE * F::CS / 2;                  // 16-byte pieces of the upstream NBR chunks
    static constexpr int LOADS = (PIECE + 1023) / 1024 + (CHUNKS + 63) / 64 + (FWD ? 0 : 1);     // per step
    static_assert(PIECE % 16 == 0 && EDGE * 2 <= LU_NT && LOADS * (LU_FAR - 2) < 64, "loads of a step");
    alignas(16) char ring[LU_RING * SLOT];
    double du[2][3][2][LU_NT];        // [step parity][direction][component a, b][lane]
    GaveUp bail;
};

// inputs of one step of wave D for this lane's components (a: momentum or energy, b: density or a
// turbulence variable): its own cell's face normal and (forward) area in direction D; the
// neighbour's U, pressure, 1/density, Lc, Lv and (backward) S; and the Res (forward) or forward DU
// (backward), the diagonal and its reciprocal of the cell whose DU the wave completes at this step
struct TeamIn {
    double n, S;
    double Ua, Ub, P, RD, Lc, Lv;
    double Ra, Rb, ala, rala, alb, ralb;
};

// 16 bytes per lane from global memory to the LDS: lane l's go to dst + 16 l
__device__ __forceinline__ void to_lds(const char* src, char* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
// wait until at most n of this wave's loads are outstanding (the other counters are left alone)
template <int n>
__device__ __forceinline__ void wait_loads() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
}

// The loader wave of a tile: at step q it starts the loads of step q + LU_FAR into the ring and
// waits for those of step q + 2, which the direction waves read from the next barrier on.  The
// direction waves finished reading slot q - 1, the one written now, before the last barrier.  A
// step's piece of the run is contiguous, so its 5 KB take five loads of 16 bytes per lane; the
// direction waves would need 45 loads of 8 bytes for them, at 16 clocks of the CU's address path
// each, twice what the step's arithmetic takes.
template <int NV, bool FWD, int TJ>
__device__ void team_load(TeamLds<NV, FWD, TJ>& sh, const Blk& b, const LuTask& T, const double* __restrict__ pk, int lane) {
    using F = Pk<NV>;
    using L = TeamLds<NV, FWD, TJ>;
    constexpr int TK = LU_COLS / TJ, PPC = F::CS / 2;         // pieces per NBR chunk
    const int nxm = b.nx - 1, nsteps = nxm + T.tj + T.tk - 2;
    const long dstep = (FWD ? (long)F::RUN : -(long)F::RUN) * 8;
    const double* first = pk + T.pofs + (FWD ? 0L : (long)(nsteps - 1) * F::RUN);       // the tile's run at step 0
    const char* run0 = (const char*)(first + L::BASE) + 16 * lane;
    // the upstream column `e` of the edge list and its run at this tile's step 0; a tile without
    // that upstream tile takes its own, which nobody reads
    auto edge = [&](int e) -> const double* {
        const bool along_j = e < TK;
        const int jlu = FWD ? T.tj_up - 1 : 0, klu = FWD ? T.tk_up - 1 : 0;
        if ((along_j ? T.dep_j : T.dep_k) < 0) return first;
        const int c = along_j ? jlu + TJ * e : (e - TK) + TJ * klu;
        const int s0 = FWD ? (along_j ? jlu : klu) : nxm + (along_j ? T.tk : T.tj) - 2;
        return pk + (along_j ? T.pofs_j : T.pofs_k) + (long)s0 * F::RUN + (long)c * F::CS;
    };
    // element offsets within a run: the chunk's column is folded into edge(); the areas' chunks
    // lie 4 doubles apart instead of CS
    constexpr int NE = (L::CHUNKS + 63) / 64;
    const char* ep[NE];
#pragma unroll
    for (int u = 0; u < NE; u++) {
        const int r = min(u * 64 + lane, L::CHUNKS - 1);
        ep[u] = (const char*)(edge(r / PPC) + F::NBR) + 16 * (r % PPC);
    }
    const char* sp = nullptr;
    if constexpr (!FWD) {
        const int r = min(lane, 2 * L::EDGE - 1), e = r / 2;
        const bool along_j = e < TK;
        const int c = (along_j ? T.dep_j : T.dep_k) < 0 ? 0 : along_j ? TJ * e : e - TK;
        sp = (const char*)(edge(e) - (long)c * F::CS + F::SG + 4 * c) + 16 * (r % 2);
    }
    auto issue = [&](int q, int slot) {
        char* d = sh.ring + slot * L::SLOT;
        const char* s = run0 + (long)q * dstep;
#pragma unroll
        for (int o = 0; o + 1024 <= L::PIECE; o += 1024) to_lds(s + o, d + o);
        constexpr int REST = L::PIECE % 1024;
        if constexpr (REST > 0) {
            if (lane < REST / 16) to_lds(s + (L::PIECE - REST), d + (L::PIECE - REST));
        }
        // the upstream columns of the next step
#pragma unroll
        for (int u = 0; u < NE; u++)
            if (u * 64 + lane < L::CHUNKS) to_lds(ep[u] + (long)(q + 1) * dstep, d + L::NBRS + u * 1024);
        if constexpr (!FWD) {
            if (lane < 2 * L::EDGE) to_lds(sp + (long)(q + 1) * dstep, d + L::SGS);
        }
    };
    int slot = 0;
    issue(-1, LU_RING - 1);
#pragma unroll 1
    for (int q = 0; q < LU_FAR; q++) issue(q, q);
    slot = LU_FAR;
    wait_loads<L::LOADS * (LU_FAR - 2)>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_barrier();      // the direction waves have read slot -1, which step 0 overwrites
    asm volatile("" ::: "memory");     // and no load of step 0 moves ahead of that
#pragma unroll 1
    for (int q = 0; q < nsteps; q++) {
        issue(q + LU_FAR, slot);
        slot = slot + 1 == LU_RING ? 0 : slot + 1;
        wait_loads<L::LOADS * (LU_FAR - 2)>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (q % LU_RING == LU_RING - 1 && sh.bail.raised(q)) break;
    }
    wait_loads<0>();      // no load may reach the LDS after the workgroup has given it back
}

// One direction wave's part of a tile's sweep.  No arithmetic is masked: what a lane without a cell
// computes is read by no lane that has one, and it is stored to elements nobody reads, inside the
// tile's storage.
template <int NV, bool FWD, int D, int TJ>
__device__ void team_sweep(TeamLds<NV, FWD, TJ>& sh, const Blk& b, const LuTask& T, double* __restrict__ pk,
                           int* __restrict__ err, const Par& p, int lane) {
    using F = Pk<NV>;
    using L = TeamLds<NV, FWD, TJ>;
    constexpr int C = LU_COLS, NB = F::NB, TK = C / TJ;
    const int part = lane % LU_PARTS, col = lane / LU_PARTS;
    const int pb_ = part < NB ? part : NB - 1;              // this lane's slot of the (density, turbulence) group
    const int jl = col % TJ, kl = col / TJ;
    const bool live = jl < T.tj && kl < T.tk;
    const int jo = FWD ? jl : T.tj - 1 - jl, ko = FWD ? kl : T.tk - 1 - kl;
    const int j = T.j0 + jl, k = T.k0 + kl;
    const int nxm = b.nx - 1;
    const double wlu = p.w_LU, gamma = p.gamma;
    const int nsteps = nxm + T.tj + T.tk - 2;
    // the neighbour of direction D: another column of the tile, or the upstream tile
    const bool has_d = D == 0 ? true : D == 1 ? (FWD ? j != 1 : j != b.ny - 1) : (FWD ? k != 1 : k != b.nz - 1);
    const bool inside = D == 0 ? true : D == 1 ? jo > 0 : ko > 0;
    const bool remote = D > 0 && live && has_d && !inside;
    const unsigned long long rmask = __builtin_amdgcn_ballot_w64(remote);
    // the column whose cell of the previous step this lane reads (columns without one read their own)
    const int scol = D == 0 || !inside ? col : D == 1 ? (FWD ? col - 1 : col + 1) : (FWD ? col - TJ : col + TJ);
    const int src = scol * LU_PARTS + part;
    const bool energy = part == 3;

    // cell i of this lane at step q is i0 + dir q
    const int i0 = FWD ? 1 - jo - ko : nxm + jo + ko;
    const int dir = FWD ? 1 : -1;
    // the lane's elements of a ring slot: its own cell's, of column scol one step back, and of the
    // neighbour, which is column scol or a column of the upstream edge
    const int edge = D == 1 ? kl : TK + jl;
    const char* ring = sh.ring;
    const char* on = ring + 8 * (F::N - L::BASE + 9 * col + 3 * D + (part < 3 ? part : 2));
    const char* os = ring + 8 * (F::SG - L::BASE + 4 * col + D);
    const char* ra = ring + 8 * ((FWD ? F::R : F::DUF) - L::BASE + 4 * scol + part);
    const char* rb = ring + 8 * ((FWD ? F::R : F::DUF) - L::BASE + 4 * C + NB * scol + pb_);
    const char* al = ring + 8 * (F::AL - L::BASE + F::CA * scol);
    const char* alb = al + (NV == 6 && pb_ == 1 ? (FWD ? 16 : 32) : 0);
    const char* nb = ring + (remote ? L::NBRS + 8 * F::CS * edge : 8 * (F::NBR - L::BASE + F::CS * scol));
    const char* ns = ring + (remote ? L::SGS + 32 * edge : 8 * (F::SG - L::BASE + 4 * scol)) + 8 * D;
    const char *na = nb + 8 * part, *nbb = nb + 8 * (4 + pb_);
    auto ld = [](const char* a) { return *(const double*)a; };
    // step q's inputs: the own cell from slot q, the rest from slot q - 1
    auto read = [&](int own, int prev, TeamIn& t) {
        const int o = own * L::SLOT, s = prev * L::SLOT;
        t.Ua = ld(na + s);
        t.Ub = ld(nbb + s);
        t.P = ld(nb + s + 8 * F::P);
        t.RD = ld(nb + s + 8 * F::RD);
        t.n = ld(on + o);
        t.Ra = ld(ra + s);
        t.Rb = ld(rb + s);
        t.ala = ld(al + s);
        t.rala = ld(al + s + 8);
        if constexpr (NV == 6) { t.alb = ld(alb + s); t.ralb = ld(alb + s + 8); }
        t.Lc = ld(nb + s + 8 * (F::LC + D));
        t.Lv = ld(nb + s + 8 * (F::LV + D));
        t.S = FWD ? ld(os + o) : ld(ns + s);
    };

    // The upstream tile's DU (may still be the sentinel).  An ordinary load, which the L2 of this
    // XCD may serve: within a sweep an element only ever holds the sentinel or its final value, and
    // every kernel starts with the L2 invalidated, so a cached copy is either current or a
    // sentinel, and a sentinel sends the lane to the device-coherent reloads of team_wait_remote.
    // The columns of a row (D = 1) or line (D = 2) of the tile read the same upstream column.
    const long dstep = (FWD ? (long)F::RUN : -(long)F::RUN) * 8;
    char* run0 = (char*)(pk + T.pofs + (FWD ? 0L : (long)(nsteps - 1) * F::RUN));
    constexpr int DU = (FWD ? F::DUF : F::DUB) * 8;
    const int oa = 8 * (4 * col + part), ob = 8 * (4 * C + NB * col + pb_);
    const char *ea = run0 + DU + oa, *eb = run0 + DU + ob;
    if (D > 0 && (D == 1 ? T.dep_j : T.dep_k) >= 0) {
        const int jlu = FWD ? T.tj_up - 1 : 0, klu = FWD ? T.tk_up - 1 : 0;
        const int c = D == 1 ? jlu + TJ * kl : jl + TJ * klu;
        const int s0 = FWD ? (D == 1 ? jlu : klu) : nxm + (D == 1 ? T.tk : T.tj) - 2;
        const char* e = (const char*)(pk + (D == 1 ? T.pofs_j : T.pofs_k) + (long)s0 * F::RUN) + DU;
        ea = e + 8 * (4 * c + part);
        eb = e + 8 * (4 * C + NB * c + pb_);
    }
    auto load_du = [&](int q, double& a, double& c) { a = ld(ea + (long)q * dstep); c = ld(eb + (long)q * dstep); };

    // DU of the cell of column scol at the step before, from the terms of that step
    auto complete = [&](int par, const TeamIn& in, double& a, double& c) {
        const auto& d = sh.du[par ^ 1];
        const double ta = d[0][0][src], tb = d[0][1][src], ua = d[1][0][src], ub = d[1][1][src], va = d[2][0][src], vb = d[2][1][src];
        const double ab = NV == 6 ? in.alb : in.ala, rab = NV == 6 ? in.ralb : in.rala;
        if (FWD) {
            a = div_nr(((in.Ra + ta) + ua) + va, in.ala, in.rala);
            c = div_nr(((in.Rb + tb) + ub) + vb, ab, rab);
        } else {
            a = in.Ra + div_nr((ta + ua) + va, in.ala, in.rala);
            c = in.Rb + div_nr((tb + ub) + vb, ab, rab);
        }
    };
    // wave 0 stores the DU of its own cell of step q - 1 (device-coherent: the elements a
    // neighbour tile reads need it, and one kind of store for all lanes)
    auto store = [&](int q, double a, double c) {
        if (D == 0 && q >= 1) {
            char* e = run0 + (long)(q - 1) * dstep + DU;
            st_coherent((double*)(e + (unsigned)oa), a);
            st_coherent((double*)(e + (unsigned)ob), c);
        }
    };

    // one step (of parity par): the flux of the neighbour's undisturbed state, the DU of the read
    // cell, the flux of the disturbed state, this direction's term of the own cell
    auto step = [&](int q, int par, const TeamIn& in, double Da, double Db) {
        double DUa, DUb, f1a, f1b;
        const double d1 = NB == 1 ? in.Ub : quad_get<0>(in.Ub);
        quad_flux(in.Ua, in.Ub, d1, in.RD, in.P, in.n, energy, f1a, f1b);
        complete(par, in, DUa, DUb);
        store(q, DUa, DUb);
        const int i = i0 + dir * q;
        if constexpr (D > 0) {
            if ((__builtin_amdgcn_ballot_w64(maybe_sentinel(Da) || maybe_sentinel(Db)) & rmask) != 0) {
                const bool waiting = remote && i >= 1 && i <= nxm;
                if (team_wait_remote((const double*)(ea + (long)q * dstep), (const double*)(eb + (long)q * dstep), waiting, Da, Db, err)) sh.bail.raise(q);
            }
            DUa = pick(rmask, Da, DUa);
            DUb = pick(rmask, Db, DUb);
        }
        const double Ua = in.Ua + DUa, Ub = in.Ub + DUb;
        const double d2 = NB == 1 ? Ub : quad_get<0>(Ub), r2 = recip_nr(d2);
        const double ke = div_nr(0.5 * quad_sum3(Ua * Ua), d2, r2);
        double f2a, f2b;
        quad_flux(Ua, Ub, d2, r2, (gamma - 1.0) * (quad_get<3>(Ua) - ke), in.n, energy, f2a, f2b);
        const double wLc = wlu * in.Lc;
        const double da = team_term<FWD>(f2a - f1a, DUa, wLc, in.Lv, in.S), db = team_term<FWD>(f2b - f1b, DUb, wLc, in.Lv, in.S);
        // a lane's terms before its first cell and those of a direction without a neighbour stay zero
        if (D == 0 ? (FWD ? i > 1 : i < nxm) : has_d) {
            sh.du[par][D][0][lane] = da;
            sh.du[par][D][1][lane] = db;
        }
    };

    // The loop is unrolled over the ring's slots.  The inputs of step q + 1 are read during step q,
    // an upstream tile's DU is loaded LU_AHEAD steps before its use: every step more adds a step to
    // the lag of each tile hop (257x97x33 C-grid, forward: 232, 263 and 292 us for 1, 2 and 3).  The last step of a round
    // checks whether a wave gave up in it (an LDS read after the barrier that the others skip): that
    // wave has set the error flag, so the waits of the steps in between give up within 256 polls and
    // their values are discarded, and all waves leave at the same barrier (GaveUp).
    constexpr int LU_AHEAD = 1;
    static_assert(LU_RING % 2 == 0, "the step parity is fixed per unrolled step");
    TeamIn in[2];
    double Da[LU_RING], Db[LU_RING];
    if constexpr (D > 0) {
#pragma unroll
        for (int u = 0; u < LU_AHEAD; u++) load_du(u, Da[u], Db[u]);
    }
    team_barrier();
    read(0, LU_RING - 1, in[0]);
    team_barrier();
    for (int q0 = 0; q0 < nsteps; q0 += LU_RING) {
#pragma unroll
        for (int u = 0; u < LU_RING; u++) {
            const int q = q0 + u;
            if (q >= nsteps) break;
            constexpr int W = LU_RING;
            if constexpr (D > 0) load_du(q + LU_AHEAD, Da[(u + LU_AHEAD) % W], Db[(u + LU_AHEAD) % W]);
            read((u + 1) % W, u, in[(u + 1) & 1]);
            step(q, u & 1, in[u & 1], Da[u], Db[u]);
            team_barrier();
            if (u == W - 1 && sh.bail.raised(q)) return;
        }
    }
    // the DU of the last step
    if constexpr (D == 0) {
        double a, c;
        if (nsteps & 1) complete(1, in[1], a, c);
        else complete(0, in[0], a, c);
        store(nsteps, a, c);
    }
}

constexpr int LT_NT = 4 * LU_NT;      // the three direction waves and the loader
template <int NV, bool FWD, int TJ>
__global__ void __launch_bounds__(LT_NT) k_lusgs_team(const Blk* __restrict__ blks, const LuTask* __restrict__ tasks,
                                                      double* __restrict__ pk, int* __restrict__ err, Par p) {
    __shared__ TeamLds<NV, FWD, TJ> sh;
    const int wave = threadIdx.x / LU_NT, lane = threadIdx.x % LU_NT;
    // a sweep earlier in the launch sequence gave up waiting: this one does nothing either (its
    // DU stays unused, the update kernels leave U as it is)
    if (threadIdx.x == 0) sh.bail.start(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    // the terms of the steps before a lane's first cell, and of a direction without a neighbour
    for (int e = (int)threadIdx.x; e < 2 * 3 * 2 * LU_NT; e += LT_NT) (&sh.du[0][0][0][0])[e] = 0.0;
    __syncthreads();
    if (sh.bail.raised(0)) return;
    const LuTask T = tasks[blockIdx.x];
    const Blk& b = blks[T.blk];
    if (wave == 0) team_sweep<NV, FWD, 0, TJ>(sh, b, T, pk, err, p, lane);
    else if (wave == 1) team_sweep<NV, FWD, 1, TJ>(sh, b, T, pk, err, p, lane);
    else if (wave == 2) team_sweep<NV, FWD, 2, TJ>(sh, b, T, pk, err, p, lane);
    else team_load<NV, FWD, TJ>(sh, b, T, pk, lane);
}

// ---------------------------------------------------------------------------------------------
// host side

// The tiles of a launch in the order in which they can start: the first tiles of all blocks, then
// the next ones.  An upstream tile starts earlier, so it keeps a lower number.
void lusgs_start_order(std::vector<LuTask>& tasks) {
    std::vector<int> at(tasks.size()), num(tasks.size());
    for (size_t q = 0; q < at.size(); q++) at[q] = (int)q;
    std::stable_sort(at.begin(), at.end(), [&](int a, int b) { return tasks[a].start < tasks[b].start; });
    std::vector<LuTask> out;
    for (size_t q = 0; q < at.size(); q++) { num[at[q]] = (int)q; out.push_back(tasks[at[q]]); }
    for (LuTask& t : out) {
        if (t.dep_j >= 0) t.dep_j = num[t.dep_j];
        if (t.dep_k >= 0) t.dep_k = num[t.dep_k];
    }
    tasks.swap(out);
}

// Tiles of every block for one sweep direction, numbered so that upstream tiles come first.
// The sweep-ordered storage of a tile does not depend on the direction: tiles are laid out block
// after block in forward order, each taking nsteps runs of `run` doubles.
std::vector<LuTask> lusgs_tasks(const std::vector<Blk>& blks, bool forward, int run, int TJ, int TK, long long* total) {
    std::vector<LuTask> out;
    const long long pad = (long long)LU_PAD_STEPS * run;
    long long pbase = pad;
    for (size_t bi = 0; bi < blks.size(); bi++) {
        const Blk& b = blks[bi];
        int nj = b.ny - 1, nk = b.nz - 1;
        int NJt = (nj + TJ - 1) / TJ, NKt = (nk + TK - 1) / TK;
        int base = (int)out.size();
        auto size_j = [&](int J) { return std::min(TJ, nj - J * TJ); };
        auto size_k = [&](int K) { return std::min(TK, nk - K * TK); };
        // storage offsets in forward tile order
        std::vector<long long> pofs((size_t)NJt * NKt);
        for (int K = 0; K < NKt; K++) for (int J = 0; J < NJt; J++) {
            pofs[J + NJt * K] = pbase;
            pbase += (long long)((b.nx - 1) + size_j(J) + size_k(K) - 2) * run;
        }
        auto P = [&](int J, int K) { return pofs[J + NJt * K]; };
        // position of tile (J,K) in this block's list
        auto idx = [&](int J, int K) { return forward ? J + NJt * K : (NJt - 1 - J) + NJt * (NKt - 1 - K); };
        std::vector<LuTask> blk_tasks((size_t)NJt * NKt);
        for (int K = 0; K < NKt; K++) for (int J = 0; J < NJt; J++) {
            LuTask t{};
            t.blk = (int)bi; t.j0 = 1 + J * TJ; t.k0 = 1 + K * TK; t.tj = size_j(J); t.tk = size_k(K);
            t.pofs = P(J, K);
            int Ju = forward ? J - 1 : J + 1, Ku = forward ? K - 1 : K + 1;
            t.dep_j = t.dep_k = -1;
            t.start = (forward ? J : NJt - 1 - J) * (TJ + LU_HOP) + (forward ? K : NKt - 1 - K) * (TK + LU_HOP);
            if (Ju >= 0 && Ju < NJt) {
                t.dep_j = base + idx(Ju, K);
                t.off_j = size_j(Ju) - 1;
                t.last_j = (b.nx - 1) + size_j(Ju) + t.tk - 3;
                t.pofs_j = P(Ju, K);
                t.tj_up = size_j(Ju);
            }
            if (Ku >= 0 && Ku < NKt) {
                t.dep_k = base + idx(J, Ku);
                t.off_k = size_k(Ku) - 1;
                t.last_k = (b.nx - 1) + t.tj + size_k(Ku) - 3;
                t.pofs_k = P(J, Ku);
                t.tk_up = size_k(Ku);
            }
            blk_tasks[idx(J, K)] = t;
        }
        out.insert(out.end(), blk_tasks.begin(), blk_tasks.end());
    }
    if (total) *total = pbase + pad;
    return out;
}

template <int NV, int TJ>
static void sweep_nv(const LuPlan& L, const Par& p, bool forward, bool fenced, hipStream_t st) {
    if (!fenced) {
        if (forward) {
            hipLaunchKernelGGL((k_lusgs_team<NV, true, TJ>), dim3((unsigned)L.n_fwd), dim3(LT_NT), 0, st,
                               L.blks, L.fwd, L.pk, L.err, p);
        } else {
            // the update takes DU from the sweep-ordered storage
            hipLaunchKernelGGL((k_lusgs_team<NV, false, TJ>), dim3((unsigned)L.n_bwd), dim3(LT_NT), 0, st,
                               L.blks, L.bwd, L.pk, L.err, p);
        }
        return;
    }
    // the fenced sweep's plans always use 8x8 tiles
    if (forward)
        hipLaunchKernelGGL((k_lusgs_sweep<NV, true>), dim3((unsigned)L.n_fwd), dim3(LU_NT), 0, st,
                           L.blks, L.fwd, L.prog_fwd, L.prog_bwd, L.n_bwd, L.err, p);
    else
        hipLaunchKernelGGL((k_lusgs_sweep<NV, false>), dim3((unsigned)L.n_bwd), dim3(LU_NT), 0, st,
                           L.blks, L.bwd, L.prog_bwd, L.prog_fwd, L.n_fwd, L.err, p);
}

// NVAR and the plan's tile width as template arguments
template <template <int, int> class K, typename... A>
static void by_shape(int NV, int tj, A&&... a) {
    switch (NV * 100 + tj) {
    case 504: K<5, 4>::run(a...); break;
    case 508: K<5, 8>::run(a...); break;
    case 516: K<5, 16>::run(a...); break;
    case 604: K<6, 4>::run(a...); break;
    case 608: K<6, 8>::run(a...); break;
    case 616: K<6, 16>::run(a...); break;
    case 704: K<7, 4>::run(a...); break;
    case 708: K<7, 8>::run(a...); break;
    default: K<7, 16>::run(a...); break;
    }
}
template <int NV, int TJ> struct SweepK { static void run(const LuPlan& L, const Par& p, bool f, bool fe, hipStream_t st) { sweep_nv<NV, TJ>(L, p, f, fe, st); } };
template <int NV, int TJ> struct GeoK {
    static void run(const LuPlan& L, hipStream_t st) {
        hipLaunchKernelGGL((k_lu_pack_geometry<NV, TJ>), dim3((unsigned)L.nwins), dim3(PK_T), 0, st, L.blks, L.fwd, L.pk, L.win);
    }
};
template <int NV, int TJ> struct DuBoxK {
    static void run(const LuPlan& L, hipStream_t st) {
        hipLaunchKernelGGL((k_lu_du_to_box<NV, TJ>), dim3((unsigned)L.nwins), dim3(PK_T), 0, st, L.blks, L.fwd, L.pk, L.win);
    }
};

void launch_lusgs_pipelined(const LuPlan& L, const Par& p, bool forward, bool fenced, hipStream_t st) {
    by_shape<SweepK>(p.NV, fenced ? 8 : L.tj, L, p, forward, fenced, st);
}

bool lusgs_tile_ok(int tj) { return tj == 4 || tj == 8 || tj == 16; }

int lusgs_run(int NV) { return NV == 5 ? Pk<5>::RUN : NV == 6 ? Pk<6>::RUN : Pk<7>::RUN; }
std::vector<int2> lusgs_window_list(const std::vector<Blk>& blks, const std::vector<LuTask>& fwd) {
    std::vector<int2> out;
    std::vector<int> at(fwd.size());
    for (size_t q = 0; q < at.size(); q++) at[q] = (int)q;
    std::sort(at.begin(), at.end(), [&](int a, int b) { return fwd[a].pofs < fwd[b].pofs; });
    for (int t : at) {
        const int nxm = blks[fwd[t].blk].nx - 1;
        for (int i0 = 1; i0 <= nxm; i0 += PK_W) out.push_back(make_int2(t, i0));
    }
    return out;
}

// the sentinel into DUF and DUB (also after a sweep gave up waiting)
template <int NV>
static void reset_nv(const LuPlan& L, hipStream_t st) {
    using F = Pk<NV>;
    hipLaunchKernelGGL(k_fill_sentinel<NV>, dim3(1024), dim3(256), 0, st, L.pk, L.P);
}

void launch_lusgs_pack_geometry(const LuPlan& L, const Par& p, hipStream_t st) {
    if (L.nwins > 0) by_shape<GeoK>(p.NV, L.tj, L, st);
}
void launch_lusgs_du_to_box(const LuPlan& L, int NV, hipStream_t st) {
    if (L.nwins > 0) by_shape<DuBoxK>(NV, L.tj, L, st);
}

void launch_lusgs_reset(const LuPlan& L, int NV, hipStream_t st) {
    if (NV == 5) reset_nv<5>(L, st);
    else if (NV == 6) reset_nv<6>(L, st);
    else reset_nv<7>(L, st);
}

}  // namespace ocfd
