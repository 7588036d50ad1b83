"""Contexts share pinned pages of 32 slots into which the device reports a
right-hand side's wave speed and error word.  More contexts than a page holds, made,
used and destroyed by several threads in an order that empties pages in the middle
of the list: every report is the context's own."""
import threading

import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE


def test_contexts_of_several_threads(hip):
    nx, ny, nthreads, each = 40, 24, 6, 14  # 84 contexts at a time: three pages
    dom = (0.0, 1.0, 0.0, ny / nx)
    kw = dict(domain=dom, cfl=0.4, bc=(T, T, R, R))
    want = []
    for k in range(nthreads):
        U = states.euler_state(nx, ny, seed=80 + k)
        if k % 2:  # the odd threads' states are reported inadmissible
            U[ny // 2, nx // 2 + k, 3] *= -1.0
        want.append((U, orc.rhs(orc.problem(0, nx, ny, N=2, prim=True, g1=1.4, **kw), U)))
    start = threading.Barrier(nthreads)
    failures = []

    def work(k):
        try:
            U, ref = want[k]
            p = hip.make_problem(hip.EULER, nx, ny, order=2, prim=True, gamma1=1.4, **kw)
            start.wait(30)
            ctxs = [hip.Context(p) for _ in range(each)]
            for rnd in range(3):
                for c in ctxs:
                    Rd, dt, rc = c.rhs(U, allow_inadmissible=True)
                    assert rc == ref["rc"] and dt == ref["dt"] and np.array_equal(Rd, ref["rhs"], equal_nan=True)
                for j in range(rnd, each, 3):  # leave holes, then fill them
                    ctxs[j].close()
                    ctxs[j] = hip.Context(p)
            for c in ctxs:
                c.close()
        except BaseException as e:  # noqa: BLE001  (reported by the main thread)
            failures.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(nthreads)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failures and not any(t.is_alive() for t in threads)
