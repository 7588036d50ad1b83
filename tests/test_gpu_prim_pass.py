"""The primitive pass at the edges of its blocks of 256 cells: fewer cells than a
block, one block, one cell more; and in place on a device buffer; against the
oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

H2D, D2H = 1, 2  # hipMemcpyHostToDevice, hipMemcpyDeviceToHost


@pytest.mark.parametrize("system", [0, 1, 2])
@pytest.mark.parametrize("nx,ny", [(3, 3), (5, 51), (16, 16), (257, 3), (64, 36)])
def test_blocks(hip, system, nx, ny):
    eos = states.EOS[system]
    p = hip.make_problem(system, nx, ny, order=2, domain=(0.0, 1.0, 0.0, ny / nx), **eos)
    op = orc.problem(system, nx, ny, domain=(0.0, 1.0, 0.0, ny / nx), g1=eos["gamma1"], g2=eos["gamma2"],
                     p1=eos["pi1"], p2=eos["pi2"])
    U = states.state(system, nx, ny, seed=nx + ny)
    want = orc.rhs(op, U, want_prim=True)["W"]
    rt = C.CDLL("libamdhip64.so")
    rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    rt.hipFree.argtypes = [C.c_void_p]
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    with hip.Context(p) as ctx:
        assert np.array_equal(ctx.cons2prim(U), want)
        d, out = C.c_void_p(), np.empty_like(U)
        assert rt.hipMalloc(C.byref(d), U.nbytes) == 0
        try:
            assert rt.hipMemcpy(d, U.ctypes.data, U.nbytes, H2D) == 0
            ptr = C.cast(d, C.POINTER(C.c_double))
            assert ctx.L.hype_cons2prim(ctx.h, ptr, ptr, hip.MEM_DEVICE) == hip.OK
            assert rt.hipMemcpy(out.ctypes.data, d, U.nbytes, D2H) == 0
        finally:
            rt.hipFree(d)
    assert np.array_equal(out, want)
