"""SA limiter's pass sorted by wavefront where its lists have their edges: more cells of one wavefront
than the workgroup has threads, a few cells in one or two clusters, the first and the last wavefront of
a block; the oracle's serial loop.  That the cells are left to the ordered pass, and how many of a
wavefront, is read from the field that the limiter gets (U6 + DU6 of the oracle's residual)."""
import re
from pathlib import Path

import numpy as np
import pytest

import oracle
import ocfd_amd as A
from helpers import oracle_U, oracle_geometry, rel_err
from ocfd_amd import cases as C

SRC = (Path(__file__).resolve().parents[1] / "opencfd-ec_amd" / "csrc" / "ocfd_kernels.hip").read_text()
THREADS, WMAX = (int(v) for v in re.search(r"constexpr int SA_ORD_T = (\d+), SA_WMAX = (\d+);", SRC).groups())


def _high(cells):
    def f(U6):
        for c in cells:
            U6[c] = 150.0
    return f


# name -> dims, LSAmax, change of the initial U6, least and most cells of the longest wavefront
CASES = {
    "over_a_workgroup": ((129, 41, 33), 4.9, lambda U6: None, THREADS + 1, 10**9),
    "one_pair": ((65, 25, 9), 100.0, _high([(20, 12, 4), (21, 12, 4)]), 1, 1),
    "first_and_last": ((33, 13, 5), 100.0, _high([(0, 0, 0), (1, 0, 0), (-1, -1, -1), (-2, -1, -1)]), 1, 1),
    "cube_and_pair": ((65, 25, 9), 100.0, _high([(30 + a, 10 + b, 3 + c) for a in range(3) for b in range(3) for c in range(3)]
                                                + [(5, 20, 6), (5, 21, 6)]), 2, 8),
}


def _wavefronts(o, case, lsamax):
    """Cells above LSAmax that have a neighbour above it, by w = i + 2j + 4k."""
    nx, ny, nz = case.blocks[0].dims
    o.residual()
    U6 = (o.get(1, "U6") + o.get(1, "DU6")).transpose(2, 1, 0)[4:nx + 3, 4:ny + 3, 4:nz + 3]
    flag = np.pad(U6 > lsamax, 1)
    near = sum(np.roll(flag, (a, b, c), (0, 1, 2)).astype(int) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1))
    i, j, k = np.nonzero((flag & (near > 1))[1:-1, 1:-1, 1:-1])
    return np.bincount(i + 2 * j + 4 * k)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_states_match_the_serial_loop(name):
    dims, lsamax, change, least, most = CASES[name]
    case = C.naca_cgrid(*dims, wall_spacing=0.02, Iflag_Flux=4, LSAmax=lsamax)
    nx, ny, nz = dims
    assert nx - 1 + 2 * (ny - 1) + 4 * (nz - 1) - 6 <= WMAX
    U0 = C.perturbed_state(case, seed=3, amp=1e-3)
    change(U0[0][5])
    o = oracle.Oracle(case)
    o.init_flow(); o.set_interior(U0); o.bc_halo()
    count = _wavefronts(o, case, lsamax)
    assert least <= count.max() <= most, (count.max(), count.sum())
    s = A.Solver(case.params)
    for no, (b, t) in enumerate(zip(case.blocks, A.inc_tables(case)), start=1):
        s.add_block_geom(no, b.dims, t, oracle_geometry(o, no, b.dims, True))
    s.init_flow(); s.set_interior(U0); s.bc(); s.halo()
    for _ in range(2):
        o.step(1); s.step(1)
        got = s.download_U(1)[:, 2:nx + 5, 2:ny + 5, 2:nz + 5]
        ref = oracle_U(o, 1, s.nv)[:, 2:nx + 5, 2:ny + 5, 2:nz + 5]
        finite = bool(np.isfinite(got).all())
        assert finite
        # the per-cell FP64 bar of the drop-in path
        assert rel_err(got, ref) <= 1e-11
    s.close()
