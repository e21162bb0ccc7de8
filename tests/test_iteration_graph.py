"""Stepping with one graph per iteration, timed stepping with a graph per stage, and eager launches
mixed in one solve give the eager solve's state bit for bit."""
import numpy as np
import pytest

import ocfd_amd as A
from ocfd_amd import cases as C


@pytest.mark.gpu
@pytest.mark.parametrize("cuts", [None, [[[17, 40], [12], [5]]]])
def test_step_and_timed_step_share_a_solve(cuts):
    case = C.naca_cgrid(65, 25, 9, wall_spacing=0.02, Iflag_Flux=4)
    if cuts:
        case = C.cut_blocks(case, cuts)
    U0 = C.perturbed_state(case, seed=5, amp=1e-4)
    a = A.solver_from_case(case, states=U0)
    b = A.solver_from_case(case, states=U0)
    b.set_graph(True)
    for n, how in [(1, "step"), (2, "timed"), (3, "step"), (1, "retile"), (2, "step"), (1, "timed"), (2, "eager"), (1, "step")]:
        a.step(n)
        if how == "retile":
            b.set_lu_tile(4)
        if how == "eager":
            b.set_graph(False)
        b.step_timed(n) if how == "timed" else b.step(n)
        b.set_graph(True)
        for no in range(1, len(case.blocks) + 1):
            assert np.array_equal(a.download_U(no), b.download_U(no)), (n, how, no)
            assert np.array_equal(a.field(no, A.F_DU), b.field(no, A.F_DU)), (n, how, no)
    a.close()
    b.close()
