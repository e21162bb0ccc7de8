"""NVAR larger than the turbulence model needs: the additional components have no residual of their own
(or, for SA with NVAR = 7, only the first has), and every LU-SGS schedule gives the same state."""
import numpy as np
import pytest

import ocfd_amd as A
from ocfd_amd import cases as C

CASES = {
    "inviscid_6": (6, lambda: C.channel_bump(33, 13, 9)),
    "inviscid_7": (7, lambda: C.channel_bump(33, 13, 9)),
    "laminar_6": (6, lambda: C.naca_cgrid(49, 17, 7, Iflag_turbulence_model=0, Re=1e4, Iflag_Flux=5, wall_spacing=0.02)),
    "sa_7": (7, lambda: C.naca_cgrid(49, 17, 7, Iflag_Flux=4, wall_spacing=0.02)),
}


def _solver(monkeypatch, case, nvar, states):
    const_params = A.const_params

    def widened(control, precision=0):
        P = const_params(control, precision)
        P.NVAR = nvar
        return P

    with monkeypatch.context() as m:
        m.setattr(A, "const_params", widened)
        return A.solver_from_case(case, states=states)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_pipelined_equals_hyperplane(monkeypatch, name):
    nvar, make = CASES[name]
    case = make()
    nx, ny, nz = case.blocks[0].dims
    own = C.perturbed_state(case, seed=4, amp=1e-4)
    more = np.random.default_rng(9).uniform(1.0, 3.0, (nvar - len(own[0]), nx - 1, ny - 1, nz - 1))
    states = [np.concatenate([own[0], more])]
    # the same solves once more after others have used the GPU: nothing left by them may show
    for _ in range(2):
        got, ref = _solver(monkeypatch, case, nvar, states), _solver(monkeypatch, case, nvar, states)
        ref.set_lu_schedule(A.LU_HYPERPLANE)
        plain = A.solver_from_case(case, states=own)
        for _ in range(3):
            for s in (got, ref, plain):
                s.step(1)
            finite = bool(np.isfinite(got.download_U(1)).all())
            assert finite
            assert np.array_equal(got.field(1, A.F_DU), ref.field(1, A.F_DU))
            assert np.array_equal(got.download_U(1), ref.download_U(1))
            # without a model the flow does not see the additional components
            assert name == "sa_7" or np.array_equal(got.download_U(1)[:5], plain.download_U(1)[:5])
        for s in (got, ref, plain):
            s.close()
