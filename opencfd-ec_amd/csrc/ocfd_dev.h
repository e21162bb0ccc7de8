// Device-side data model of one block: every per-block array (cell, face or node) lives in one
// padded box i in [-3, nx+3], j in [-3, ny+3], k in [-3, nz+3] (the reference's LAP=4 ghost
// range), i fastest, one array per variable (SoA).  Threads map to i so every access along a
// face or cell row is a coalesced 64-wide load.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace ocfd {

constexpr int LAP = 4;
constexpr int MAXV = 7;

// A pointer to device memory in a table that kernels read.  A plain pointer loaded from memory could
// point anywhere, so the compiler uses flat accesses: a 64-bit address in vector registers for each,
// and waits that cover LDS too.  In device code this one says that it points to global memory.
template <typename T>
struct gptr {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(1))) T* ptr;
#else
    typedef T* ptr;
#endif
    ptr p;
    __host__ __device__ __forceinline__ operator T*() const { return (T*)p; }
    __host__ __device__ __forceinline__ gptr& operator=(T* q) { p = (ptr)q; return *this; }
    // element s of a box: the base stays in scalar registers and a lane's address is one 32-bit byte
    // offset, shared by the arrays of a block.  A box array stays below 4 GiB: a block has 95 of them
    // or more, and a device 288 GB.
    __host__ __device__ __forceinline__ T& operator[](size_t s) const {
#if defined(__HIP_DEVICE_COMPILE__)
        return *(T*)(ptr)((__attribute__((address_space(1))) const char*)p + (uint32_t)((uint32_t)s * (uint32_t)sizeof(T)));
#else
        return p[s];
#endif
    }
    __host__ __device__ __forceinline__ T& operator[](uint32_t s) const { return (*this)[(size_t)s]; }
    __host__ __device__ __forceinline__ T& operator[](long s) const { return ((T*)p)[s]; }
    __host__ __device__ __forceinline__ T& operator[](int s) const { return ((T*)p)[s]; }
    // element s + o of an array that the kernel does not write (o the same in all lanes): the load may
    // move ahead of the kernel's stores, which a plain load does not, since the compiler cannot tell
    // the arrays of the table apart
    __device__ __forceinline__ T ro(size_t s, long o = 0) const {
#if defined(__HIP_DEVICE_COMPILE__)
        typedef __attribute__((address_space(4))) const char* cptr;
        return *(__attribute__((address_space(4))) const T*)((cptr)(p + o) + (uint32_t)((uint32_t)s * (uint32_t)sizeof(T)));
#else
        return p[s + o];
#endif
    }
    // the array shifted by an offset that is the same in all lanes (a stencil's neighbour): at(o)[s]
    // is element s + o
    __host__ __device__ __forceinline__ gptr at(long o) const { return gptr{p + o}; }
};

// s, worked out anew in the basic block that calls it (ID: no two calls are the same): the compiler
// keeps an array's base in scalar registers only if it sees in the same block that s has 32 bits
template <int ID>
__device__ __forceinline__ size_t in_block(size_t s) {
    uint32_t v = (uint32_t)s;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(v) : "i"(ID));
#endif
    return v;
}

// A table that no kernel writes (blocks, their parameters, tile maps), in the constant address space
// in device code.  Through a plain pointer the compiler has to assume that a kernel's stores may
// change the table: it then reads each array pointer with a vector load of its own, just before the
// array's element and after the stores ahead of it.  From here the pointers come in scalar loads.
template <typename T>
struct ctab {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(4))) const T* ptr;
#else
    typedef const T* ptr;
#endif
    ptr p;
    ctab() = default;
    __host__ __device__ __forceinline__ ctab(const T* q) : p((ptr)q) {}
    __host__ __device__ __forceinline__ const T& operator[](long i) const { return *(const T*)(p + i); }
};

struct Par {                 // control parameters after set_const_para (sub_read_parameter.f90:371-429)
    double Ma, Re, gamma, Cv, Cp, PrL, PrT, T_inf, Twall, AoA, A_alfa, A_beta, P_outlet;
    double CFL, dtmax, dtmin, dt_global, w_LU, MUT_MAX, Kt_inf, Wt_inf;
    double Ldmin, Ldmax, Lpmin, Lpmax, Lumax, LSAmax;
    int NV, visc, turb, scheme, flux, recon, bscheme, local_dt, dtime_mesh, positivity, limit_flow;
    int mixed;                   // 1: reconstruction, face fluxes and the SA terms in FP32
};

struct Blk {
    int nx, ny, nz, NI, NJ, NK;
    gptr<double> U[MAXV], Res[MAXV], DU[MAXV];
    gptr<double> dt, mu, muf, mut;        // mu: Sutherland; muf: mu after the turbulence-model (x*Re)/Re round trip
    gptr<double> prim[7]; // rho u v w p T c (per iteration; limiter snapshot afterwards)
    gptr<double> Lc[3], Lv[3];
    gptr<double> vol, S[3], nv[9], met[4][9], dw, dtm, x, y, z, xc, yc, zc;
    gptr<double> F[3][5]; // inviscid face flux, m = 1..5
    gptr<double> Fv[3][4]; // viscous face flux, m = 2..5
    gptr<double> Fsa[3][2]; // SA face terms: convection+diffusion flux, grad(vt).n S; SST: k and omega fluxes
    // mixed precision: FP32 primitives (rho u v w p T) and FP32 face terms; the face arrays share
    // the memory of their FP64 counterparts
    gptr<float> primf[6], Ff[3][5], Fvf[3][4], Fsaf[3][2];
    // mixed precision: FP32 copies of the geometry the FP32 kernels read (face normals, areas,
    // metrics, and per direction the node difference t1 of the inviscid flux's face frame), made
    // once per block from the FP64 arrays
    gptr<float> nvf[9], Sf[3], metf[4][9], t1f[3][3];
    gptr<double> aux; // turbulence scratch (SST f1)
    gptr<double> kt, wt; // SST: k and omega per unit mass, max(U, 0) / rho, on the box
    gptr<uint8_t> bcf[3]; // face-row flags (BcFlag; the upper face's bit is the lower's << 1)
    gptr<double> surf[6][3]; // Surf1..6 (wall viscous force of the i-/j-/k-/i+/j+/k+ faces)
    gptr<int> flags; // [0] IF_OverLimit latch, [1] limited cells this iteration, [2] SA cells above LSAmax
    gptr<unsigned long long> samask;          // SA cells above LSAmax, one bit per cell in (i,j,k) order (SA only)
};

// per face row of a direction: the lower face is physical, lies on a wall, takes the explicit flux
// of a physical k face; the upper face likewise in the next bit
enum BcFlag : int { BCF_PHYS = 1, BCF_WALL = 4, BCF_KBC = 16 };

__device__ __host__ __forceinline__ size_t IX(const Blk& b, int i, int j, int k) {
    return (uint32_t)(i + 3) + (uint32_t)b.NI * ((uint32_t)(j + 3) + (uint32_t)b.NJ * (uint32_t)(k + 3));
}
__device__ __host__ __forceinline__ size_t JK(const Blk& b, int j, int k) { return (uint32_t)(j + 3) + (uint32_t)b.NJ * (uint32_t)(k + 3); }
__device__ __host__ __forceinline__ size_t IK(const Blk& b, int i, int k) { return (uint32_t)(i + 3) + (uint32_t)b.NI * (uint32_t)(k + 3); }
__device__ __host__ __forceinline__ size_t IJ(const Blk& b, int i, int j) { return (uint32_t)(i + 3) + (uint32_t)b.NI * (uint32_t)(j + 3); }
// the distance between a cell and its neighbour (di, dj, dk) away
__device__ __host__ __forceinline__ long OFF(const Blk& b, int di, int dj, int dk) { return di + (long)b.NI * (dj + (long)b.NJ * dk); }

// what the residual norms read of a block
struct NormBlk {
    gptr<const double> res[MAXV];
    int nx, ny, nz, NI, NJ;
};

// one subface of the .inc table (sub_modules.f90:63-68)
struct Sub {
    int ib, ie, jb, je, kb, ke, bc, face, f_no;
    int ib1, ie1, jb1, je1, kb1, ke1, nb1, face1, f_no1;
    int L1, L2, L3;
};

// ---------------------------------------------------------------------------------------------
// Block sets: every block of a context (of every case it holds) goes through the same launch.
// A launch over an iteration space covers the tiles of all blocks; tile t belongs to block
// tile_blk[t] and is that block's (t - tile0[block])-th tile of 64 points (i fastest).

enum Space { SP_BOX = 0, SP_CELL, SP_FI, SP_FJ, SP_FK, SP_N0, SP_COUNT };

// extent and origin of an iteration space of one block
__device__ __host__ __forceinline__ void space_dims(int sp, const Blk& b, int& n0, int& n1, int& n2, int& o0, int& o1, int& o2) {
    switch (sp) {
    case SP_BOX: n0 = b.NI; n1 = b.NJ; n2 = b.NK; o0 = o1 = o2 = -3; break;
    case SP_CELL: n0 = b.nx - 1; n1 = b.ny - 1; n2 = b.nz - 1; o0 = o1 = o2 = 1; break;
    case SP_FI: n0 = b.nx; n1 = b.ny - 1; n2 = b.nz - 1; o0 = o1 = o2 = 1; break;
    case SP_FJ: n0 = b.nx - 1; n1 = b.ny; n2 = b.nz - 1; o0 = o1 = o2 = 1; break;
    case SP_FK: n0 = b.nx - 1; n1 = b.ny - 1; n2 = b.nz; o0 = o1 = o2 = 1; break;
    default: n0 = b.nx + 1; n1 = b.ny + 1; n2 = b.nz + 1; o0 = o1 = o2 = 0; break;
    }
}

struct BSet {
    ctab<Blk> blk;
    ctab<Par> par;
    ctab<int> tile_blk;      // for the launch's space
    ctab<int> tile0;
    const int* halt;         // nonzero *halt: an LU-SGS sweep of this iteration gave up; the update
                             // kernels then leave U as it is (may be null)
    int* limited;            // set by the update when a cell of any block needs the limiter
};

__device__ __forceinline__ bool halted(const BSet& S) { return S.halt && *(volatile const int*)S.halt != 0; }

// Workgroups of a one-dimensional grid are handed to the 8 XCDs in turn (workgroup t to XCD
// t mod 8).  Renumbering so that XCD x runs the x-th eighth of the tiles in order keeps the
// j/k neighbour rows of a stencil, which are also tiles of the same launch, in that XCD's L2;
// the last n mod 8 tiles keep their numbers (a bijection on [0, n)).
__device__ __forceinline__ int xcd_tile(int t, int n) {
    const int full = n & ~7;
    return t < full ? (t & 7) * (full >> 3) + (t >> 3) : t;
}

constexpr int ROW_CHUNK = 16;

// point `lane` of tile t of iteration space sp
__device__ __forceinline__ bool locate_point(int sp, const ctab<Blk>& blk, const ctab<int>& tile_blk, const ctab<int>& tile0, int t, int& bi, int& i, int& j,
                                             int& k, int lane) {
    bi = tile_blk[t];
    int n0, n1, n2, o0, o1, o2;
    space_dims(sp, blk[bi], n0, n1, n2, o0, o1, o2);
    // the block's points in i-fastest order, 64 per tile: a tile runs on into the next row when
    // a row is shorter or not a multiple of 64 (cut blocks of 16-cell rows keep every lane busy)
    const int a = (t - tile0[bi]) * 64 + lane;
    if (a >= n0 * n1 * n2) return false;
    const int r = a / n0;
    i = o0 + (a - r * n0);
    // rows (j, k) in chunks of ROW_CHUNK planes along k, k fastest inside a chunk: the rows a
    // stencil reads at j +- 1 are ROW_CHUNK rows away and those at k +- 1 (k +- 4 for the
    // reconstruction of the k faces) the neighbouring rows, so both stay in the L2 of the XCD that
    // runs the tile (the renumbering above keeps a launch's neighbouring tiles on one XCD)
    const int full = n2 / ROW_CHUNK * ROW_CHUNK;
    if (r < n1 * full) {
        const int c = r / (n1 * ROW_CHUNK), rr = r - c * (n1 * ROW_CHUNK);
        j = o1 + rr / ROW_CHUNK;
        k = o2 + c * ROW_CHUNK + rr % ROW_CHUNK;
    } else {
        const int rem = n2 - full, rr = r - n1 * full;
        j = o1 + rr / rem;
        k = o2 + full + rr % rem;
    }
    return true;
}

template <int SP>
__device__ __forceinline__ bool locate_tile(const BSet& S, int t, int& bi, int& i, int& j, int& k, int lane) {
    return locate_point(SP, S.blk, S.tile_blk, S.tile0, t, bi, i, j, k, lane);
}

template <int SP>
__device__ __forceinline__ bool locate(const BSet& S, int& bi, int& i, int& j, int& k) {
    return locate_tile<SP>(S, xcd_tile((int)blockIdx.x, (int)gridDim.x), bi, i, j, k, (int)threadIdx.x);
}

// The faces of the three directions in one launch: n[d] tiles of direction d (space SP_FI + d).
struct FaceSet {
    ctab<Blk> blk;
    ctab<Par> par;
    ctab<int> tile_blk[3];
    ctab<int> tile0[3];
    int n[3];
};

// Each XCD walks its eighth of every direction's tiles, FACE_GROUP tiles of i faces, then the j and
// the k faces of about the same cells, so that the cells' primitives are still in its L2 when the
// next direction reads them (4 to 256 tiles: the same within 1 %).
constexpr int FACE_GROUP = 16;
__device__ __host__ __forceinline__ int face_groups(const int n[3]) {
    const int m = n[0] > n[1] ? n[0] : n[1], most = m > n[2] ? m : n[2];
    return ((most + 7) / 8 + FACE_GROUP - 1) / FACE_GROUP;
}
// workgroups of the launch; some hold no tile
__device__ __host__ __forceinline__ int face_grid(const int n[3]) { return 8 * 3 * FACE_GROUP * face_groups(n); }
// direction d and tile of workgroup w, false if it has none (every tile of every direction belongs
// to exactly one workgroup of the grid)
__device__ __host__ __forceinline__ bool face_tile(int w, const int n[3], int& d, int& t) {
    const int xcd = w % 8, e = w / 8;
    d = e / FACE_GROUP % 3;
    const int u = e / (3 * FACE_GROUP) * FACE_GROUP + e % FACE_GROUP, per = (n[d] + 7) / 8;
    t = xcd * per + u;
    return u < per && t < n[d];
}

// direction of the workgroup's faces (-1: none) and the point of its thread
__device__ __forceinline__ int locate_face(const FaceSet& S, int& bi, int& i, int& j, int& k) {
    int d, t;
    if (!face_tile((int)blockIdx.x, S.n, d, t)) return -1;
    return locate_point(SP_FI + d, S.blk, S.tile_blk[d], S.tile0[d], t, bi, i, j, k, (int)threadIdx.x) ? d : -1;
}

#define OCFD_LOCATE(SP)                                  \
    int bi_, i, j, k;                                    \
    if (!locate<(SP)>(S, bi_, i, j, k)) return;          \
    const Blk& b = S.blk[bi_];                           \
    const Par& p = S.par[bi_];

// one subface of one block in a subface launch: n0 x n1 points, tiles of 64 along n0
enum SubKind { SUB_WALL = 0, SUB_FAR, SUB_SYM, SUB_EXT, SUB_AMUT, SUB_KBC };
struct SubTask {
    int blk, kind, arg, n0, n1, tile0;
    Sub B;
};
struct SubSet {
    ctab<Blk> blk;
    ctab<Par> par;
    ctab<SubTask> t;
    ctab<int> tile_task;
};

#define OCFD_SUB_LOCATE                                                      \
    const SubTask& T_ = S.t[S.tile_task[blockIdx.x]];                        \
    const Blk& b = S.blk[T_.blk];                                            \
    const Par& p = S.par[T_.blk];                                            \
    const Sub& B = T_.B;                                                     \
    const int lt_ = (int)blockIdx.x - T_.tile0, T0_ = (T_.n0 + 63) / 64;    \
    const int a = (lt_ % T0_) * 64 + (int)threadIdx.x, c = lt_ / T0_;

// block-to-block ghost copy of one inner subface (Umessage_send_mpi's index map)
struct HaloMap { int kb[3], kb1[3], ke1[3], L[3], P[3], ks[3]; };
struct HaloTask {
    int src, dst, n, tile0;      // n points, tiles of 256
    HaloMap h;
};
struct HaloSet {
    ctab<Blk> blk;
    ctab<HaloTask> t;
    ctab<int> tile_task;
};

// one tile of the pipelined LU-SGS sweep: cells j0..j0+tj-1, k0..k0+tk-1 of block `blk`, all i
struct LuTask {
    int blk, j0, k0, tj, tk;
    int dep_j, off_j, last_j;    // upstream tile along j: task index (-1: none), step offset, its last step
    int dep_k, off_k, last_k;    // upstream tile along k
    long long pofs;              // sweep-ordered storage of this tile: the run of step q at pofs + q RUN
    long long pofs_j;            // the j-upstream tile's storage offset
    long long pofs_k;            // the k-upstream tile's storage offset
    int tj_up, tk_up;            // the upstream tiles' j and k extents
    int start;                   // steps (and tile hops) between the sweep's start and the tile's
};

// device tables of the pipelined sweeps of one context
struct LuPlan {
    const Blk* blks = nullptr;
    const LuTask* fwd = nullptr;
    const LuTask* bwd = nullptr;
    int n_fwd = 0, n_bwd = 0;
    int* prog_fwd = nullptr;     // last completed step per tile, -1 before the sweep
    int* prog_bwd = nullptr;
    int* err = nullptr;          // set when a wait exceeds its poll limit
    // sweep-ordered copies of the sweep's inputs and of DU (layout below), P elements
    double* pk = nullptr;
    long long P = 0;
    const int2* win = nullptr;   // (forward tile, first i) of every i-window of PK_W cells of the tiles
    int nwins = 0;
    int tj = 8;                  // tile width in j (tiles are tj x 16/tj (j,k) columns)
};

// A wave of the pipelined LU-SGS sweep holds LU_COLS (j,k) columns of a tile, LU_PARTS lanes (a DPP
// quad) each: lane 4 c + m works on components m + 1 (momentum for m = 0, 1, 2, energy for m = 3)
// and on one of (density, the turbulence variables) of column c.
constexpr int LU_NT = 64, LU_PARTS = 4, LU_COLS = LU_NT / LU_PARTS;

// The sweep-ordered storage.  For a tile, step q (the cells its columns visit at forward step q; the
// backward sweep visits them at step nsteps-1-q) is one contiguous run of RUN doubles at
// pofs + q RUN, made of groups:
//   R, DUF, DUB   Res and the two DU arrays, NV components: components 2..5 of a column side by side
//                 (4 c + m), so a wave's 64 lanes take 512 consecutive bytes, then density and the
//                 turbulence variables (64 + NB c + m)
//   NBR           what a neighbour needs of a cell, CS doubles per column: U (components 2..5, then
//                 density and the turbulence variables with limit_vt's clamp applied), the pressure
//                 of U and the reciprocal of its density (recip_nr), Lc and Lv of the three directions
//   SG            the three face areas, four doubles per column
//   AL            the LU-SGS diagonal and its reciprocal, pairs, CA doubles per column: alfa of
//                 components 1..5 (and of 6, 7 for SST) and, for SA only, the SA component's alfa of
//                 the forward and of the backward sweep, which sum the viscous radii in different orders
//   N             the face normals, three directions of three components per column
// The forward sweep reads one contiguous piece of a run, R to N, the backward sweep NBR to DUF.  A
// column's NBR chunk is a multiple of 16 bytes, and CS and CA spread the columns over the LDS banks.
// The buffer has LU_PAD_STEPS steps of padding at both ends, so loads a few steps past either end
// of a tile (prefetches of steps that do not exist) stay inside it.
template <int NV> struct Pk {
    static constexpr int NB = NV - 4, NAL = NV == 6 ? 3 : 1;
    static constexpr int CS = NV == 7 ? 18 : 14, CA = 2 * NAL;
    static constexpr int P = 4 + NB, RD = P + 1, LC = RD + 1, LV = LC + 3;        // in an NBR chunk
    static constexpr int R = 0, NBR = NV * LU_COLS, SG = NBR + CS * LU_COLS, AL = SG + 4 * LU_COLS, N = AL + CA * LU_COLS,
                         DUF = N + 9 * LU_COLS, DUB = DUF + NV * LU_COLS, RUN = DUB + NV * LU_COLS;
    static constexpr int SWEEP = DUF - R;                                          // doubles of a run a sweep reads
    static_assert(LV + 3 <= CS && CS % 2 == 0, "an NBR chunk holds its fields in 16-byte pieces");
    // component (0..NV-1) and column of element w of a vector group, and the inverse
    static __device__ __host__ __forceinline__ void vec_at(int w, int& v, int& c) {
        if (w < 4 * LU_COLS) { c = w >> 2; v = (w & 3) + 1; }
        else { const int r = w - 4 * LU_COLS, m = r % NB; c = r / NB; v = m == 0 ? 0 : m + 4; }
    }
    static __device__ __host__ __forceinline__ int vec_off(int v, int c) {
        return v >= 1 && v <= 4 ? 4 * c + v - 1 : 4 * LU_COLS + NB * c + (v == 0 ? 0 : v - 4);
    }
};
constexpr int LU_PAD_STEPS = 24;

// The LDS ring of a tile's team holds the inputs of LU_RING steps; its waves run their steps in rounds
// of as many.
constexpr int LU_RING = 4;

// Whether a wave of a team gave up waiting.  The waves ask after the barrier that ends a round, and
// have to get the same answer to leave together, so each round has a word of its own: a wave that is
// ahead may raise the next round's word while another has still to ask about this one, but the round
// after that, which shares the word, begins behind a barrier that comes after the question.
struct GaveUp {
    int word[2];
    __host__ __device__ __forceinline__ void start(int v) { word[0] = word[1] = v; }
    __host__ __device__ __forceinline__ void raise(int q) { word[q / LU_RING & 1] = 1; }      // at step q
    // after the barrier that ends step q, the last of its round, and a fence (no volatile read: it would
    // be a flat one, which waits for the wave's global loads as well)
    __host__ __device__ __forceinline__ bool raised(int q) const { return word[q / LU_RING & 1] != 0; }
};
constexpr int PK_W = 32;      // i-window of one workgroup of the sweep-order transposes and cell pass

// Before a sweep every DU element it writes holds this NaN (a payload no arithmetic produces); a
// consumer in a downstream tile reloads an element until it is something else.
constexpr unsigned long long LU_SENTINEL = 0x7FF4C0DEDEADBEEFull;
__device__ __forceinline__ bool is_sentinel(double v) { return (unsigned long long)__double_as_longlong(v) == LU_SENTINEL; }
__device__ __forceinline__ double sentinel_value() { return __longlong_as_double((long long)LU_SENTINEL); }

}  // namespace ocfd
