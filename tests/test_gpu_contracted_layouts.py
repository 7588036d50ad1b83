"""HYPE_OPT_FMA: an instance's result does not depend on whether it runs alone or
in a batch, nor on the tile layout.  A small Euler grid alone runs split tiles, in
a batch one wave per tile; both kernels must contract the same operations."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R, P = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE, orc.BC_PERIODIC


def setting(hip, system, prim, order, nx, ny, bc):
    return hip.make_problem(system, nx, ny, order=order, prim=prim, domain=(0.0, 1.0, 0.0, ny / nx), cfl=0.4, bc=bc,
                            fma=True, **states.EOS[system])


@pytest.mark.parametrize("system", [0, 1, 2])
@pytest.mark.parametrize("prim", [True, False])
@pytest.mark.parametrize("order", [1, 2, 3])
def test_contracted_solo_equals_batched(hip, system, prim, order):
    sizes = [(64, 40, (T, T, R, R)), (125, 19, (P, P, P, P)), (63, 57, (T, R, R, T))]
    probs = [setting(hip, system, prim, order, *s) for s in sizes]
    U0s = [states.state(system, nx, ny, seed=61 + k) for k, (nx, ny, _) in enumerate(sizes)]
    steps = np.array([6, 5, 4], dtype=np.int32)
    with hip.Batch(probs) as b:
        for i, U in enumerate(U0s):
            b.set_state(i, U)
        b.begin(max_steps=steps)
        b.advance(7)
        st = b.sync(allow_inadmissible=True)
        got = [b.get_state(i) for i in range(len(probs))]
    for i, p in enumerate(probs):
        for options in (0, hip.OPT_ONE_WAVE_TILES, hip.OPT_SPLIT_TILES) if system == 0 else (0,):
            p.options = hip.OPT_FMA | options
            with hip.Context(p) as ctx:
                U, s = ctx.solve(U0s[i], int(steps[i]))
            assert (st[i].steps, st[i].t, st[i].err) == (s.steps, s.t, s.err), options
            assert np.array_equal(got[i], U), (options, np.max(np.abs(got[i] - U)))
