"""Right-hand sides of states whose velocities fall to subnormal numbers, as they do
ahead of a wave: mass and energy fluxes, and the jump terms that are a product with
a velocity, are subnormal there too, and halving such a number rounds.  In every
layout the returned right-hand side, and the state after some steps, are bitwise
the oracle's."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE
NX, NY = 126, 24


def tail_state(system, kind):
    """Uniform densities and pressures, smooth velocities of both signs.
    "velocity": the velocities fall from 1e-280 to zero along x.
    "jump": they do, in a volume fraction with exact differences, so that its
    dissipation vanishes or cancels beside the jump and volume terms.
    (The device's division rounds a subnormal quotient exactly halfway between two
    numbers down as often as to the even one; with these densities none is.)"""
    X, Y = np.meshgrid((np.arange(NX) + 0.5) / NX, (np.arange(NY) + 0.5) / NY)
    scale = 10.0 ** -np.linspace(280.0, 330.0, NX)
    u, v = np.cos(9 * X + 4 * Y) * scale, np.sin(7 * X - 5 * Y) * scale
    one = np.ones_like(X)
    a = 0.375 * one
    if kind == "jump":
        a = 0.25 + (np.arange(NX)[None, :] + 2.0 * np.arange(NY)[:, None]) / 512.0
    if system == 0:
        return states.euler_cons(1.1 * one, u, v, 0.7 * one, 1.4)
    e = states.EOS[system]
    k = (e["gamma1"], e["gamma2"], e["pi1"], e["pi2"])
    if system == 1:
        return states.kapila_cons(one, one, u, v, 1e5 * one, a, *k)
    return states.bn_cons(997.0 * one, u, v, 1e5 * one, one, 0.7 * v, 1.3 * u, 1e5 * one, a, *k)


CASES = [(s, lay, kind) for s, lays in ((0, ("", "ONE_WAVE", "SPLIT")), (1, ("", "SPLIT")), (2, ("", "ONE_WAVE")))
         for lay in lays for kind in (("velocity",) if s == 0 else ("velocity", "jump"))]


@pytest.mark.parametrize("system,layout,kind", CASES)
@pytest.mark.parametrize("prim", [True, False])
@pytest.mark.parametrize("order", [0, 1, 2, 3])
def test_subnormal_rhs_matches_oracle(hip, system, layout, kind, prim, order):
    U = tail_state(system, kind)
    eos = states.EOS[system]
    dom, bc = (0.0, 1.0, 0.0, NY / NX), (T, T, R, R)
    p = hip.make_problem(system, NX, NY, order=order, prim=prim, domain=dom, cfl=0.4, bc=bc, **eos)
    if layout:
        p.options |= getattr(hip, f"OPT_{layout}_TILES")
    op = orc.problem(system, NX, NY, N=order, prim=prim, domain=dom, cfl=0.4, bc=bc, g1=eos["gamma1"],
                     g2=eos["gamma2"], p1=eos["pi1"], p2=eos["pi2"])
    ref = orc.rhs(op, U)
    size = np.abs(ref["rhs"])
    assert ((size > 0) & (size < 2.2e-308)).any()
    with hip.Context(p) as ctx:
        got, dt, rc = ctx.rhs(U, allow_inadmissible=True)
        assert rc == ref["rc"] and dt == ref["dt"]
        assert np.array_equal(got, ref["rhs"]), [int(n) for n in np.sum(got != ref["rhs"], axis=(0, 1))]
        if order > 0:
            after, st = ctx.solve(U, 2)
            sref = orc.solve(op, U, 2)
            assert st.steps == sref["steps"] == 2
            assert np.array_equal(after, sref["U"]), [int(n) for n in np.sum(after != sref["U"], axis=(0, 1))]
