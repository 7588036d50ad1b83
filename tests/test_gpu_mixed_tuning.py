"""Measured tuning of a batch of different systems: the automatic plan gives each
system's tiles a height by the time its rows take, and tuning does not lose that.
At the height of the automatic plan, the tuner must end with a plan about as fast
(a common height for all systems takes 1.6 times as long here), and every
instance's result is bitwise its solo run."""
import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE


def problem(hip, system, prim, n, m):
    return hip.make_problem(system, n, m, order=2, prim=prim, domain=(0.0, 1.0, 0.0, m / n), cfl=0.4, bc=(T, T, R, R),
                            **states.EOS[system])


def timed(b, U0s):
    """Least time of 6 steps over 3 runs."""
    best = 1e300
    for _ in range(3):
        for i, U in enumerate(U0s):
            b.set_state(i, U)
        b.begin()
        b.advance(1)
        best = min(best, b.advance_timed(6))
    return best


def test_tuning_keeps_heights_by_system(hip):
    sizes = [(0, True, 500, 440), (0, True, 330, 410), (2, False, 300, 420), (1, True, 260, 300), (0, True, 512, 130),
             (2, False, 190, 350), (1, True, 120, 500), (0, True, 90, 70)]
    probs = [problem(hip, *s) for s in sizes]
    U0s = [states.state(s, n, m, seed=71 + k, sharp=False) for k, (s, _, n, m) in enumerate(sizes)]
    with hip.Batch(probs) as b:
        rows = b.tiling()[0]
        before = timed(b, U0s)
        best, ms = b.autotune([rows], steps=4)
        after = timed(b, U0s)
        print(f"rows {rows}: automatic {before:.3f} ms, tuned {after:.3f} ms, tiles {b.tiling()[1]}", flush=True)
        assert best == rows == b.tiling()[0] and ms > 0
        assert after <= 1.25 * before
        for i, U in enumerate(U0s):
            b.set_state(i, U)
        b.begin(max_steps=np.full(len(probs), 3, dtype=np.int32))
        b.advance(4)
        b.sync()
        got = [b.get_state(i) for i in range(len(probs))]
        b.set_rows(rows)  # the same height for every system
        print(f"common height: {timed(b, U0s):.3f} ms, tiles {b.tiling()[1]}", flush=True)
    for i, p in enumerate(probs):
        with hip.Context(p) as ctx:
            U, _ = ctx.solve(U0s[i], 3)
        assert np.array_equal(got[i], U), i
