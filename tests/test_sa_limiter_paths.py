"""SA limiter with few and with nearly all cells above LSAmax, sorted by wavefront, and on a block with
more wavefronts than are sorted (each looked up in the cells' box): the oracle's serial loop."""
import numpy as np
import pytest

import oracle
import ocfd_amd as A
from helpers import oracle_U, oracle_geometry, rel_err
from ocfd_amd import cases as C


@pytest.mark.gpu
@pytest.mark.parametrize("dims,lsamax", [((65, 25, 9), 5.004), ((65, 25, 9), 4.99), ((33, 13, 5), 5.001), ((97, 25, 9), 4.999),
                                          ((33, 9, 1031), 5.002)])
def test_states_match_the_serial_loop(dims, lsamax):
    case = C.naca_cgrid(*dims, wall_spacing=0.02, Iflag_Flux=4, Ldmax=1.001, LSAmax=lsamax)
    U0 = C.perturbed_state(case, seed=3, amp=1e-3)
    o = oracle.Oracle(case)
    o.init_flow(); o.set_interior(U0); o.bc_halo()
    s = A.Solver(case.params)
    for no, (b, t) in enumerate(zip(case.blocks, A.inc_tables(case)), start=1):
        s.add_block_geom(no, b.dims, t, oracle_geometry(o, no, b.dims, True))
    s.init_flow(); s.set_interior(U0); s.bc(); s.halo()
    for _ in range(3):
        o.step(1); s.step(1)
        nx, ny, nz = case.blocks[0].dims
        got = s.download_U(1)[:, 2:nx + 5, 2:ny + 5, 2:nz + 5]
        ref = oracle_U(o, 1, s.nv)[:, 2:nx + 5, 2:ny + 5, 2:nz + 5]
        assert np.all(np.isfinite(got))
        # the per-cell FP64 bar of the drop-in path
        assert rel_err(got, ref) <= 1e-11
    s.close()
