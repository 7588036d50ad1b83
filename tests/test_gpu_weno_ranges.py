"""The shared-reciprocal divisions of the WENO weights near the end of their range:
pressure jumps whose smoothness indicators straddle it (a jump J gives an indicator
of order J^2 and a divisor of its fourth power, compared with 2^388), at orders 2
and 3, in the layouts the system has.  Both division paths, mixed within a wave,
are bitwise the oracle's plain divisions."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T = orc.BC_TRANSMISSIVE


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("prim", [True, False])
@pytest.mark.parametrize("layout", ["", "ONE_WAVE", "SPLIT"])
def test_jumps_around_the_range(hip, order, prim, layout):
    nx, ny = 130, 12
    g = states.EOS[0]["gamma1"]
    X = ((np.arange(nx) + 0.5) / nx)[None, :] * np.ones((ny, 1))
    # a jump every ten cells, 2^40 .. 2^52 in turn
    big = 2.0 ** (40 + (np.arange(nx) // 10) % 13)
    pr = np.where((np.arange(nx) // 5) % 2 == 0, big, 1.0)[None, :] * (1.0 + 0.1 * np.cos(3 * X))
    U = states.euler_cons(1.0 + 0.1 * np.sin(7 * X), 0.0 * X, 0.01 * np.cos(5 * X), pr, g)
    dom = (0.0, 1.0, 0.0, ny / nx)
    p = hip.make_problem(hip.EULER, nx, ny, order=order, prim=prim, domain=dom, cfl=0.5, bc=(T,) * 4, gamma1=g)
    if layout:
        p.options |= getattr(hip, f"OPT_{layout}_TILES")
    op = orc.problem(orc.EULER, nx, ny, N=order, prim=prim, domain=dom, cfl=0.5, bc=(T,) * 4, g1=g)
    ref = orc.rhs(op, U)
    with hip.Context(p) as ctx:
        R, dt, rc = ctx.rhs(U, allow_inadmissible=True)
    assert rc == ref["rc"] and dt == ref["dt"]
    assert np.array_equal(R, ref["rhs"], equal_nan=True)
