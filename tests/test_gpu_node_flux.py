"""Conservative path at orders 0 and 1, one wave per tile: a node's flux is
computed with its admissibility check and handed to the face.  At the edges of
strips and tiles, on admissible states and with a cell of negative pressure (the
fallback there and the report of the first face), the right-hand side, the
fallback mask, the time step and the report are the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R, P = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE, orc.BC_PERIODIC


@pytest.mark.parametrize("system,energy", [(0, 3), (2, 7)])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("nx,ny,bc", [
    (3, 3, (T, T, R, R)), (61, 5, (P, P, P, P)), (62, 7, (T, R, R, T)), (63, 4, (R, R, P, P)), (125, 19, (T, T, R, R)),
])
def test_node_flux_matches_oracle(hip, system, energy, order, bad, nx, ny, bc):
    eos = states.EOS[system]
    U = states.rough_state(system, nx, ny, seed=51 + nx).copy()
    if bad:
        U[ny // 2, nx // 2, energy] *= -1.0
        U[ny - 1, nx - 1, energy] *= -1.0  # a corner, whose ghosts repeat it
    dom = (0.0, 1.0, 0.0, ny / nx)
    p = hip.make_problem(system, nx, ny, order=order, prim=False, domain=dom, bc=bc, **eos)
    p.options |= hip.OPT_ONE_WAVE_TILES
    op = orc.problem(system, nx, ny, N=order, prim=False, domain=dom, bc=bc, g1=eos["gamma1"], g2=eos["gamma2"],
                     p1=eos["pi1"], p2=eos["pi2"])
    ref = orc.rhs(op, U, want_fallback=True)
    with hip.Context(p) as ctx:
        for rows in (0, 1, 2, ny):
            if rows:
                ctx.set_tiling(min(rows, ny), 0)
            Rd, dt, mask, rc = ctx.rhs(U, fallback=True, allow_inadmissible=True)
            assert rc == ref["rc"], rows
            assert np.array_equal(Rd, ref["rhs"], equal_nan=True), rows
            assert np.array_equal(mask, ref["fallback"]), rows
            if bad:
                assert rc == hip.E_INADMISSIBLE and ctx.last_error()[1:] == (ref["err"].x, ref["err"].y), rows
            else:
                assert dt == ref["dt"], rows
