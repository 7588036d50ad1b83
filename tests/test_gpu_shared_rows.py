"""The stage kernel whose two waves share every row of a tile (the layout small
grids get by default at order 2 and 3), at the edges of its tiles: one, two and
all rows, a width just below, at and above the 62 columns of a strip, the smallest
grid and a persistent queue.  The right-hand side
and a few steps are bitwise the oracle's, and those of the layouts that can be
forced: the arithmetic does not depend on how a tile is divided."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R, P = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE, orc.BC_PERIODIC


def setting(hip, system, prim, order, nx, ny, bc, options=0):
    eos = states.EOS[system]
    dom = (0.0, 1.0, 0.0, ny / nx)
    p = hip.make_problem(system, nx, ny, order=order, prim=prim, domain=dom, cfl=0.4, bc=bc, **eos)
    p.options |= options
    op = orc.problem(system, nx, ny, N=order, prim=prim, domain=dom, cfl=0.4, bc=bc, g1=eos["gamma1"],
                     g2=eos["gamma2"], p1=eos["pi1"], p2=eos["pi2"])
    return p, op


@pytest.mark.parametrize("system", [0, 1, 2])
@pytest.mark.parametrize("prim,order", [(True, 2), (False, 2), (True, 3), (False, 3)])
@pytest.mark.parametrize("nx,ny,bc", [
    (3, 3, (T, T, R, R)), (61, 5, (P, P, P, P)), (62, 7, (T, R, R, T)), (63, 4, (R, R, P, P)), (125, 19, (T, T, R, R)),
])
def test_shared_rows_match_oracle(hip, system, prim, order, nx, ny, bc):
    p, op = setting(hip, system, prim, order, nx, ny, bc)
    U0 = states.state(system, nx, ny, seed=31 + nx)
    ref, sref = orc.rhs(op, U0), orc.solve(op, U0, 3)
    with hip.Context(p) as ctx:
        for rows, grid in [(0, 0), (1, 0), (2, 0), (3, 3), (ny, 0)]:
            if rows:
                ctx.set_tiling(min(rows, ny), grid)
            Rd, dt, _ = ctx.rhs(U0, allow_inadmissible=True)
            assert np.array_equal(Rd, ref["rhs"], equal_nan=True) and dt == ref["dt"], (rows, grid)
            ctx.set_state(U0)
            ctx.begin(0.0, float("inf"), 3, hip.TS_CLIP)
            ctx.advance(3)
            st = ctx.sync(allow_inadmissible=True)
            assert st.steps == sref["steps"], (rows, grid)
            assert np.array_equal(ctx.get_state(), sref["U"], equal_nan=True), (rows, grid)


@pytest.mark.parametrize("system,prim,option", [(0, True, "ONE_WAVE"), (0, False, "SPLIT"), (1, True, "SPLIT"),
                                                (1, False, "SPLIT"), (2, True, "ONE_WAVE"), (2, False, "ONE_WAVE")])
def test_layouts_agree_on_rough_states(hip, system, prim, option):
    """Fallbacks and inadmissible faces: the same mask, result and report."""
    nx, ny = 70, 33
    U0 = states.rough_state(system, nx, ny, seed=41)
    seen = []
    for options in (0, getattr(hip, f"OPT_{option}_TILES")):
        p, _ = setting(hip, system, prim, 2, nx, ny, (T, T, R, R), options)
        with hip.Context(p) as ctx:
            Rd, dt, mask, rc = ctx.rhs(U0, fallback=True, allow_inadmissible=True)
            seen.append((Rd, dt, mask, rc, ctx.last_error()))
    a, b = seen
    assert np.array_equal(a[0], b[0], equal_nan=True) and np.array_equal(a[2], b[2])
    assert (a[1], a[3], a[4]) == (b[1], b[3], b[4])
    assert a[2].any()


def test_subnormal_tails(hip):
    """Velocities that fall to subnormal numbers ahead of a wave: halving them
    rounds, which the kernels' fused forms must not skip."""
    nx, ny = 96, 40
    U0 = states.state(1, nx, ny, seed=5)
    scale = np.ones((ny, nx))
    scale[:, 40:] = 10.0 ** -np.linspace(280.0, 325.0, nx - 40)
    eos = states.EOS[1]
    rho = U0[..., 0] + U0[..., 1]
    kin = 0.5 * (U0[..., 2] ** 2 + U0[..., 3] ** 2) / rho
    U0[..., 4] -= kin
    U0[..., 2] *= scale
    U0[..., 3] *= scale
    U0[..., 4] += 0.5 * (U0[..., 2] ** 2 + U0[..., 3] ** 2) / rho
    U0[:, 40:, (0, 1, 4, 5)] = U0[0, 95, (0, 1, 4, 5)]  # no force on the tail but its own motion
    dom = (0.0, 1.0, 0.0, ny / nx)
    kw = dict(order=2, prim=True, domain=dom, cfl=0.4, bc=(T, T, R, R))
    op = orc.problem(1, nx, ny, N=2, prim=True, domain=dom, cfl=0.4, bc=(T, T, R, R), g1=eos["gamma1"], g2=eos["gamma2"],
                     p1=eos["pi1"], p2=eos["pi2"])
    ref = orc.solve(op, U0, 3)
    tail = np.abs(ref["U"][:, 50:, 2:4])
    assert ((tail > 0) & (tail < 2.2e-308)).any()
    for options in (0, hip.OPT_SPLIT_TILES):
        p = hip.make_problem(1, nx, ny, **kw, **eos)
        p.options |= options
        with hip.Context(p) as ctx:
            U, st = ctx.solve(U0, 3)
        assert np.array_equal(U, ref["U"]), options
