"""A first phase that vanishes: its volume fraction, and its mass, momentum and
energy per volume, fall below the smallest normal number, where every halving
rounds; smoothly along x, through the value at which the reconstruction changes
its form, or from an ordinary value to a subnormal one within a cell.  In every
layout the right-hand side, and the state after some steps, are bitwise the
oracle's."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE
NX, NY = 126, 24


def vanishing(system, kind):
    X, Y = np.meshgrid((np.arange(NX) + 0.5) / NX, (np.arange(NY) + 0.5) / NY)
    if kind == "deep":
        a = 10.0 ** -np.linspace(290.0, 314.0, NX) * (1.0 + 0.3 * np.sin(9 * Y))
    elif kind == "through":
        a = 10.0 ** -np.linspace(200.0, 314.0, NX) * (1.0 + 0.3 * np.sin(9 * Y))
    else:  # patches of 1 to 7 cells a side
        i, j = np.arange(NX)[None, :], np.arange(NY)[:, None]
        a = np.where((i * i // 7 + j * j // 5) % 3 == 0, 0.3 + 0.1 * np.sin(3 * X), 1e-311 * (1.3 + np.sin(9 * X + 5 * Y)))
    u, v, one = np.cos(9 * X + 4 * Y), np.sin(7 * X - 5 * Y), np.ones_like(X)
    e = states.EOS[system]
    k = (e["gamma1"], e["gamma2"], e["pi1"], e["pi2"])
    if system == 1:
        return states.kapila_cons(one, one, u, v, 1e5 * one, a, *k)
    return states.bn_cons(997.0 * one, u, v, 1e5 * one, one, 0.7 * v, 1.3 * u, 1e5 * one, a, *k)


@pytest.mark.parametrize("system,layout", [(1, ""), (1, "SPLIT"), (2, ""), (2, "ONE_WAVE")])
@pytest.mark.parametrize("kind", ["deep", "through", "patches"])
@pytest.mark.parametrize("prim", [True, False])
@pytest.mark.parametrize("order", [0, 1, 2, 3])
def test_vanishing_phase_matches_oracle(hip, system, layout, kind, prim, order):
    U = vanishing(system, kind)
    eos = states.EOS[system]
    dom, bc = (0.0, 1.0, 0.0, NY / NX), (T, T, R, R)
    p = hip.make_problem(system, NX, NY, order=order, prim=prim, domain=dom, cfl=0.4, bc=bc, **eos)
    if layout:
        p.options |= getattr(hip, f"OPT_{layout}_TILES")
    op = orc.problem(system, NX, NY, N=order, prim=prim, domain=dom, cfl=0.4, bc=bc, g1=eos["gamma1"],
                     g2=eos["gamma2"], p1=eos["pi1"], p2=eos["pi2"])
    assert ((U[..., -1] > 0) & (U[..., -1] < 2.2e-308)).any()
    ref = orc.rhs(op, U)
    with hip.Context(p) as ctx:
        got, dt, rc = ctx.rhs(U, allow_inadmissible=True)
        assert rc == ref["rc"] and dt == ref["dt"]
        assert np.array_equal(got, ref["rhs"], equal_nan=True), [int(n) for n in np.sum(got != ref["rhs"], axis=(0, 1))]
        if order > 0:
            after, st = ctx.solve(U, 2)
            sref = orc.solve(op, U, 2)
            assert st.steps == sref["steps"] == 2
            assert np.array_equal(after, sref["U"]), [int(n) for n in np.sum(after != sref["U"], axis=(0, 1))]
