"""CPU model of the storage addressing of the pipelined LU-SGS sweep (ocfd_lusgs.hip, Pk in
ocfd_dev.h): tiles of 16 (j,k) columns, four lanes per column, one contiguous run per step.

The model restates the task layout and the kernels' index arithmetic and checks, on ragged
multi-block shapes and every tile shape:
  - the element order of a vector group is a bijection and four lanes of a column cover it;
  - the element a lane reads across a tile edge is the one the upstream tile stores the DU of the
    cell it needs in, and it gets the sentinel from the pack;
  - pack and update windows visit every cell's element exactly once;
  - every load of the loader wave and of the upstream DU, prefetches beyond a tile's ends and the
    loads of tiles without an upstream tile included, stays inside the padded buffer, and the
    upstream chunks the loader brings for a step are the ones its lanes need."""
import random

import pytest

COLS, PARTS, PK_W, PAD, RING, AHEAD = 16, 4, 32, 24, 4, 1
FAR = RING - 1
TILES = (4, 8, 16)
SHAPES = [[(17, 17, 9)], [(33, 20, 13), (9, 5, 18)], [(65, 25, 9)], [(12, 40, 7), (20, 3, 3)], [(9, 65, 17)], [(3, 3, 3)]]
random.seed(11)
SHAPES += [[(random.randint(3, 40), random.randint(3, 30), random.randint(3, 30)) for _ in range(random.randint(1, 3))] for _ in range(3)]


def vec_off(NV, v, c):
    NB = NV - 4
    return 4 * c + v - 1 if 1 <= v <= 4 else 4 * COLS + NB * c + (0 if v == 0 else v - 4)


def vec_at(NV, w):
    NB = NV - 4
    if w < 4 * COLS:
        return (w & 3) + 1, w >> 2
    r = w - 4 * COLS
    return (0 if r % NB == 0 else r % NB + 4), r // NB


@pytest.mark.parametrize("NV", (5, 6, 7))
def test_vector_group_order(NV):
    NB = NV - 4
    seen = {}
    for w in range(NV * COLS):
        v, c = vec_at(NV, w)
        assert vec_off(NV, v, c) == w
        seen[(v, c)] = w
    assert sorted(seen) == [(v, c) for v in range(NV) for c in range(COLS)]
    # the lanes of a column: components 1..4 and, in the second slot, density and the rest
    for c in range(COLS):
        a = {seen[(p + 1, c)] for p in range(PARTS)}
        b = {4 * COLS + NB * c + min(p, NB - 1) for p in range(PARTS)}
        assert a == {4 * c + p for p in range(PARTS)}
        assert a | b == {vec_off(NV, v, c) for v in range(NV)}


def tasks(blocks, TJ, forward):
    TK = COLS // TJ
    out, pbase = [], PAD
    for bi, (nx, ny, nz) in enumerate(blocks):
        nj, nk = ny - 1, nz - 1
        NJt, NKt = -(-nj // TJ), -(-nk // TK)
        sj, sk = (lambda J: min(TJ, nj - J * TJ)), (lambda K: min(TK, nk - K * TK))
        pofs = {}
        for K in range(NKt):
            for J in range(NJt):
                pofs[J, K] = pbase
                pbase += nx - 1 + sj(J) + sk(K) - 2
        for K in range(NKt):
            for J in range(NJt):
                t = dict(blk=bi, j0=1 + J * TJ, k0=1 + K * TK, tj=sj(J), tk=sk(K), pofs=pofs[J, K], nsteps=nx - 1 + sj(J) + sk(K) - 2)
                Ju, Ku = (J - 1, K - 1) if forward else (J + 1, K + 1)
                if 0 <= Ju < NJt:
                    t.update(pofs_j=pofs[Ju, K], tj_up=sj(Ju))
                if 0 <= Ku < NKt:
                    t.update(pofs_k=pofs[J, Ku], tk_up=sk(Ku))
                out.append(t)
    return out, pbase + PAD


def cell_elements(blocks, TJ):
    """(run, column) of every cell, runs counted from the buffer's start."""
    el = {}
    for T in tasks(blocks, TJ, True)[0]:
        nxm = blocks[T["blk"]][0] - 1
        for jl in range(T["tj"]):
            for kl in range(T["tk"]):
                for i in range(1, nxm + 1):
                    el[T["blk"], i, T["j0"] + jl, T["k0"] + kl] = (T["pofs"] + i - 1 + jl + kl, jl + TJ * kl)
    return el


@pytest.mark.parametrize("TJ", TILES)
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_lanes_read_their_neighbours(TJ, shape):
    blocks = SHAPES[shape]
    el = cell_elements(blocks, TJ)
    assert len(set(el.values())) == len(el)
    for forward in (True, False):
        d = 1 if forward else -1
        tl, total = tasks(blocks, TJ, forward)
        for T in tl:
            nx, ny, nz = blocks[T["blk"]]
            nxm, ns = nx - 1, T["nsteps"]
            run0 = T["pofs"] + (0 if forward else ns - 1)
            for col in range(COLS):
                jl, kl = col % TJ, col // TJ
                live = jl < T["tj"] and kl < T["tk"]
                jo, ko = (jl, kl) if forward else (T["tj"] - 1 - jl, T["tk"] - 1 - kl)
                j, k = T["j0"] + jl, T["k0"] + kl
                i0 = 1 - jo - ko if forward else nxm + jo + ko
                for D in range(3):
                    has = [True, (j != 1 if forward else j != ny - 1), (k != 1 if forward else k != nz - 1)][D]
                    inside = [True, jo > 0, ko > 0][D]
                    remote = D > 0 and live and has and not inside
                    scol = col if D == 0 or not inside else col - d if D == 1 else col - d * TJ
                    assert not inside or not live or 0 <= scol < COLS
                    nbrun, nc = run0 - d, scol
                    if remote:
                        jlu, klu = (T["tj_up"] - 1 if D == 1 else 0, T["tk_up"] - 1 if D == 2 else 0) if forward else (0, 0)
                        nc = jlu + TJ * kl if D == 1 else jl + TJ * klu
                        s0 = (jlu if D == 1 else klu) if forward else nxm + (T["tk"] if D == 1 else T["tj"]) - 2
                        nbrun = T["pofs_j" if D == 1 else "pofs_k"] + s0
                    for q in range(ns):
                        i = i0 + d * q
                        if not (live and 1 <= i <= nxm):
                            continue
                        cell = (T["blk"], i, j, k)
                        assert el[cell] == (run0 + d * q, col)
                        up = [(i - d, j, k), (i, j - d, k), (i, j, k - d)][D]
                        if (T["blk"], *up) in el:
                            assert el[(T["blk"], *up)] == (nbrun + d * q, nc), (forward, D, cell)
                        else:
                            assert not has or D == 0


@pytest.mark.parametrize("TJ", TILES)
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_windows_visit_every_cell_once(TJ, shape):
    """pack and update: (step, element) pairs of every i-window; the sentinel's windows as well."""
    blocks, NV, TK = SHAPES[shape], 6, COLS // TJ
    el = cell_elements(blocks, TJ)
    seen, sent = set(), set()
    for T in tasks(blocks, TJ, True)[0]:
        nxm = blocks[T["blk"]][0] - 1
        for i0 in range(1, nxm + 1, PK_W):
            W = min(PK_W, nxm - i0 + 1)
            for q in range(i0 - 1, i0 - 1 + W + TJ + TK - 2):
                for w in range(NV * COLS):
                    v, c = vec_at(NV, w)
                    jl, kl = c % TJ, c // TJ
                    x = q - jl - kl + 1 - i0
                    if 0 <= x < W and q < T["nsteps"]:
                        sent.add((T["pofs"] + q, c, v))
                    if jl < T["tj"] and kl < T["tk"] and 0 <= x < W:
                        assert q < T["nsteps"]
                        key = (T["blk"], i0 + x, T["j0"] + jl, T["k0"] + kl, v)
                        assert key not in seen
                        seen.add(key)
                        assert el[key[:4]] == (T["pofs"] + q, c)
    assert len(seen) == NV * len(el)
    assert {(r, c, v) for r, c in el.values() for v in range(NV)} <= sent


def layout(NV):
    """Pk<NV>: doubles of a run's groups."""
    NB, NAL = NV - 4, 3 if NV == 6 else 1
    CS, CA = (18 if NV == 7 else 14), 2 * NAL
    NBR = NV * COLS
    SG = NBR + CS * COLS
    AL = SG + 4 * COLS
    N = AL + CA * COLS
    DUF = N + 9 * COLS
    DUB = DUF + NV * COLS
    return dict(NB=NB, CS=CS, CA=CA, R=0, NBR=NBR, SG=SG, AL=AL, N=N, DUF=DUF, DUB=DUB, RUN=DUB + NV * COLS)


@pytest.mark.parametrize("NV", (5, 6, 7))
@pytest.mark.parametrize("TJ", TILES)
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_loads_stay_inside_the_buffer(NV, TJ, shape):
    """team_load and load_du: byte ranges of the first and last loads of every lane, and the column
    and step of the upstream chunks."""
    blocks, L, TK = SHAPES[shape], layout(NV), COLS // TJ
    RUN, CS, PPC, EDGE = L["RUN"], L["CS"], L["CS"] // 2, TJ + COLS // TJ
    el = cell_elements(blocks, TJ)
    at = {e: cell for cell, e in el.items()}
    assert RUN % 2 == 0 and (L["DUF"] * 8) % 16 == 0 and (L["NBR"] * 8) % 16 == 0
    for forward in (True, False):
        d = 1 if forward else -1
        base = L["R"] if forward else L["NBR"]
        tl, total = tasks(blocks, TJ, forward)
        size = total * RUN * 8
        for T in tl:
            nx, ny, nz = blocks[T["blk"]]
            nxm, ns = nx - 1, T["nsteps"]
            first = (T["pofs"] + (0 if forward else ns - 1)) * RUN
            ends = []

            def span(start_bytes, step_first, step_last, width):
                for q in (step_first, step_last):
                    a = start_bytes + q * d * RUN * 8
                    assert a % 8 == 0
                    ends.append((a, a + width))

            # the tile's own piece: steps -1 .. nsteps - 1 + FAR
            span((first + base) * 8, -1, ns - 1 + FAR, (L["DUF"] - L["R"]) * 8)
            for e in range(EDGE):
                along_j = e < TK
                up = ("pofs_j" if along_j else "pofs_k") in T
                if up:
                    jlu, klu = ((T.get("tj_up", 1) - 1, T.get("tk_up", 1) - 1) if forward else (0, 0))
                    c = jlu + TJ * e if along_j else (e - TK) + TJ * klu
                    s0 = (jlu if along_j else klu) if forward else nxm + (T["tk"] if along_j else T["tj"]) - 2
                    start = (T["pofs_j" if along_j else "pofs_k"] + s0) * RUN
                else:
                    c, start = 0, first
                # NBR chunks are loaded for steps q + 1, q = -1 .. nsteps - 1 + FAR, backward areas too
                for piece in (0, PPC - 1):
                    span((start + c * CS + L["NBR"]) * 8 + 16 * piece, 0, ns + FAR, 16)
                if not forward:
                    for piece in (0, 1):
                        span((start + c * CS - c * CS + L["SG"] + 4 * c) * 8 + 16 * piece, 0, ns + FAR, 16)
                if up:
                    # the lane of this edge column and the cell it needs at each of its steps
                    jl, kl = ((0 if forward else T["tj"] - 1), e) if along_j else (e - TK, (0 if forward else T["tk"] - 1))
                    if jl < T["tj"] and kl < T["tk"]:
                        jo, ko = (jl, kl) if forward else (T["tj"] - 1 - jl, T["tk"] - 1 - kl)
                        i0 = 1 - jo - ko if forward else nxm + jo + ko
                        for q in range(ns):
                            i = i0 + d * q
                            if 1 <= i <= nxm:
                                j, k = T["j0"] + jl, T["k0"] + kl
                                assert at[start // RUN + d * q, c] == ((T["blk"], i, j - d, k) if along_j else (T["blk"], i, j, k - d))
            # the upstream DU of every column, or the tile's own where there is none
            for D in (1, 2):
                up = ("pofs_j" if D == 1 else "pofs_k") in T
                for col in range(COLS):
                    jl, kl = col % TJ, col // TJ
                    c, start = col, first
                    if up:
                        jlu, klu = ((T.get("tj_up", 1) - 1, T.get("tk_up", 1) - 1) if forward else (0, 0))
                        c = jlu + TJ * kl if D == 1 else jl + TJ * klu
                        s0 = (jlu if D == 1 else klu) if forward else nxm + (T["tk"] if D == 1 else T["tj"]) - 2
                        start = (T["pofs_j" if D == 1 else "pofs_k"] + s0) * RUN
                    g = L["DUF"] if forward else L["DUB"]
                    for o in (4 * c, 4 * c + 3, 4 * COLS + L["NB"] * c, 4 * COLS + L["NB"] * c + L["NB"] - 1):
                        span((start + g + o) * 8, 0, ns - 1 + AHEAD, 8)
            assert min(a for a, _ in ends) >= 0 and max(b for _, b in ends) <= size


@pytest.mark.parametrize("ns", (1, 2, 5, 6, 7, 13, 40))
def test_ring_slots_are_written_and_read_apart(ns):
    """The loader's writes and the direction waves' reads of the LDS ring, one list per interval
    between two barriers: a read finds its step's data, whose loads ended before the interval, and
    no slot is written in an interval in which it is read."""
    content, pending = {}, []          # slot -> step of finished loads; steps in flight, oldest first

    def settle(keep):
        while len(pending) > keep:
            step = pending.pop(0)
            content[step % RING] = step

    pending += [-1] + list(range(FAR))
    settle(FAR - 2)                                            # before the first barrier
    intervals = [([], [(0, 0), (RING - 1, -1)])]               # (steps written, (slot, step) read)
    for q in range(ns):
        intervals.append(([q + FAR], [((q + 1) % RING, q + 1), (q % RING, q)]))
    for writes, reads in intervals:
        done = dict(content)
        busy = {s % RING for s in pending + writes}
        for slot, step in reads:
            assert done.get(slot) == step and slot not in busy, (step, slot)
        pending += writes
        settle(FAR - 2)
