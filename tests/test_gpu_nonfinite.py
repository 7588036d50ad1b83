"""Non-finite face states spread as the reference's products with the zero normal
component make them.  A transverse velocity that jumps by more than 1e38 overflows
the fourth power of every smoothness indicator, so its reconstruction is NaN while
every other component's is finite: the jump term of the volume fraction is NaN at a
face with such a state on either side."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T = orc.BC_TRANSMISSIVE


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("layout", ["", "SPLIT"])
def test_nan_transverse_velocity(hip, axis, order, layout):
    n, m = 70, 12  # along and across the direction of the jumps
    eos = states.EOS[1]
    one = np.ones((m, n))
    v = 1e40 * one
    v[:, (20, 41, 43)] = -1e40  # the energy is even in v: the pressure stays uniform
    U = states.kapila_cons(one, one, 0.0 * one, v, 1e82 * one, 0.5 * one, eos["gamma1"], eos["gamma2"], 0.0, 0.0)
    if axis == 1:
        U = np.ascontiguousarray(np.swapaxes(U, 0, 1))
        U[..., [2, 3]] = U[..., [3, 2]]
    ny, nx = U.shape[:2]
    dom = (0.0, 1.0, 0.0, ny / nx)
    p = hip.make_problem(1, nx, ny, order=order, prim=True, domain=dom, cfl=0.4, bc=(T,) * 4, **eos)
    if layout:
        p.options |= getattr(hip, f"OPT_{layout}_TILES")
    op = orc.problem(1, nx, ny, N=order, prim=True, domain=dom, cfl=0.4, bc=(T,) * 4, g1=eos["gamma1"],
                     g2=eos["gamma2"], p1=eos["pi1"], p2=eos["pi2"])
    ref = orc.rhs(op, U)
    nan = np.isnan(ref["rhs"][..., 5])
    assert nan.any() and not nan.all()
    with hip.Context(p) as ctx:
        got, _, rc = ctx.rhs(U, allow_inadmissible=True)
    assert rc == ref["rc"]
    assert np.array_equal(got, ref["rhs"], equal_nan=True)
