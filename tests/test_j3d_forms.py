"""Which kernel form the 3D planner takes, on the host only: the two-step
windowed kernel or the plane-by-plane one (17- and 27-point shapes)."""
import pytest

import perks_amd as P
from perks_amd import _lib as L


def caps():
    c = L.DeviceCaps()
    c.cu_count, c.lds_per_cu, c.lds_per_block = 256, 160 * 1024, 160 * 1024
    c.vgprs_per_simd, c.simds_per_cu, c.warp_size, c.cooperative = 512, 4, 64, 1
    return c


def plan(n, occupancy, **kw):
    dims = (n, n, n) if isinstance(n, int) else n
    rc, info = P.plan(*dims, caps=caps(), occupancy=occupancy, method=kw.pop("method", "persistent"), **kw)
    assert rc == 0
    return info


WINDOWED, SWEEP = (2, 8), (1, 6)  # steps per pass, rows of a tile with its ghost rows


@pytest.mark.parametrize("shape", ["3d17pt", "3d27pt"])
@pytest.mark.parametrize("n,occupancy,tune,blkpsm,form", [
    (64, 4, None, 0, SWEEP), (64, 1, None, 0, WINDOWED), (64, 4, None, 1, WINDOWED),  # one workgroup per CU
    (80, 1, None, 0, SWEEP), (80, 4, None, 1, SWEEP), (80, 4, [0, 0, 0, 1], 0, SWEEP),
    (64, 4, [0, 0, 0, 0, 2], 0, WINDOWED),       # register streaming on 64 x 8 tiles, asked for
    (64, 4, [0, 0, 1, 0, 2], 0, SWEEP),          # one step per pass of it
    (64, 4, [0, 0, 2], 0, WINDOWED), (64, 4, [0, 0, 1], 0, SWEEP),
])
def test_streaming_form(shape, n, occupancy, tune, blkpsm, form):
    info = plan(n, occupancy, shape=shape, tune=tune, blkpsm=blkpsm)
    assert (info.reserved[0], info.tile_y) == form and info.tile_x == 64


# the last size of the plane-by-plane form and the first of the windowed one
@pytest.mark.parametrize("shape,dtype,method,last", [("3d17pt", "f64", "persistent", 275), ("3d17pt", "f64", "plain", 369),
                                                     ("3d17pt", "f32", "plain", 465), ("3d27pt", "f64", "persistent", 465)])
def test_limits(shape, dtype, method, last):
    assert plan(last, 4, shape=shape, dtype=dtype, method=method).tile_y == 6
    assert plan(last + 1, 4, shape=shape, dtype=dtype, method=method).tile_y == 8
