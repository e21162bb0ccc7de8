"""SST's fluxes formed with the viscous ones, and by themselves as for a wall subface inside a block,
give the same state bit for bit.

A wall subface off its block's face takes the second way.  The one added here holds no cell (its j
range is a single node line of the lower wall), so the flow does not change.
"""
import numpy as np
import pytest

import ocfd_amd as A
from ocfd_amd import cases as C


def _solver(case, extra, precision, states):
    s = A.Solver(case.params, precision)
    for no, (b, t) in enumerate(zip(case.blocks, A.inc_tables(case)), start=1):
        t = np.asarray(t, dtype=np.int32)
        if extra:
            row = np.zeros(21, dtype=np.int32)
            nk = b.dims[2]
            row[:9] = [1, 2, 1, 1, 1, nk, C.BC_WALL, 1, len(t) + 1]
            t = np.concatenate([t.reshape(-1, 21), row[None]])
        s.add_block_nodes(no, b.x, b.y, b.z, t)
    s.setup_geometry()
    s.init_flow()
    s.set_interior(states)
    s.bc()
    s.halo()
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims,turb", [((33, 17, 5), 3), ((18, 12, 9), 3), ((33, 17, 5), 2)])
def test_alone_equals_with_the_viscous_fluxes(dims, turb, precision):
    case = C.channel_bump(*dims, If_viscous=1, Iflag_turbulence_model=turb, Re=1.0e5, Iflag_Flux=6, CFL=0.5)
    U0 = C.perturbed_state(case, seed=3, amp=1e-4)
    a, b = _solver(case, False, precision, U0), _solver(case, True, precision, U0)
    for _ in range(3):
        a.step(1)
        b.step(1)
        assert np.all(np.isfinite(a.download_U(1)))
        assert np.array_equal(a.download_U(1), b.download_U(1))
        assert np.array_equal(a.field(1, A.F_MUT), b.field(1, A.F_MUT))
        assert np.array_equal(a.field(1, A.F_RES), b.field(1, A.F_RES))
    a.close()
    b.close()
