"""The layout the host picks for the grids that the shared-row and node-flux tests
run on: those tests are about particular kernels, so a change of the tile-shape
model must not move their grids to others unnoticed.  hype_pick_layout is an
internal function of csrc/host/common.c, reached through the library's exports."""
import ctypes as C

import pytest

import oracle_py as orc
import states

pytestmark = pytest.mark.gpu

T, R = orc.BC_TRANSMISSIVE, orc.BC_REFLECTIVE
ONE, SPLIT, SHARED = 0, 1, 2


def picked(hip, system, prim, order, nx, ny, options=0):
    p = hip.make_problem(system, nx, ny, order=order, prim=prim, domain=(0.0, 1.0, 0.0, ny / nx), bc=(T, T, R, R),
                         **states.EOS[system])
    p.options = options
    lay, nsy = C.c_int(), C.c_int()
    f = hip.lib().hype_pick_layout
    f.argtypes = [C.POINTER(hip.Problem), C.POINTER(C.c_int), C.POINTER(C.c_int), C.c_void_p]
    assert f(C.byref(p), C.byref(lay), C.byref(nsy), None) == 0
    assert 1 <= nsy.value <= ny
    return lay.value


@pytest.mark.parametrize("system", [0, 1, 2])
@pytest.mark.parametrize("prim,order", [(True, 2), (False, 2), (True, 3), (False, 3)])
@pytest.mark.parametrize("nx,ny", [(3, 3), (61, 5), (62, 7), (63, 4), (125, 19), (70, 33), (126, 24), (70, 12)])
def test_small_grids_share_rows(hip, system, prim, order, nx, ny):
    """Baer-Nunziato at order 3 is not built for it."""
    want = ONE if (system, order) == (2, 3) else SHARED
    assert picked(hip, system, prim, order, nx, ny) == want


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("prim", [True, False])
def test_low_orders_do_not(hip, prim, order):
    for system, want in ((0, SPLIT), (1, SPLIT), (2, ONE)):
        assert picked(hip, system, prim, order, 125, 19) == want


@pytest.mark.parametrize("system", [0, 1, 2])
def test_forced_and_contracted(hip, system):
    for option, lay in ((hip.OPT_ONE_WAVE_TILES, ONE), (hip.OPT_SPLIT_TILES, SPLIT)):
        if (system, lay) not in ((1, ONE), (2, SPLIT)):
            assert picked(hip, system, True, 2, 70, 33, option) == lay
    assert picked(hip, system, True, 2, 70, 33, hip.OPT_FMA) != SHARED
