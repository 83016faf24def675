"""Levels and tile of the 7-point persistent kernel where the caller leaves them
open, as planned, on the host only."""
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


@pytest.mark.parametrize("dims,dtype,boundary,levels,tile_y", [
    ((512, 512, 512), "f64", "zero", 4, 36),    # the default
    ((64, 64, 64), "f64", "zero", 3, 36),       # fewer levels
    ((128, 128, 128), "f32", "clamp", 4, 32),   # the short tile
    ((512, 512, 512), "f16", "clamp", 3, 64),
    ((50, 512, 512), "f64", "clamp", 4, 36),    # flat: what a pass moves counts
    ((30, 512, 512), "f64", "clamp", 4, 36),
])
def test_seven_point_choice(dims, dtype, boundary, levels, tile_y):
    info = plan(dims, 1, dtype=dtype, boundary=boundary)
    assert (info.reserved[0], info.tile_y) == (levels, tile_y)
