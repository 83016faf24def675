"""What the planner says of a 3D run and what the run reports agree, and the two
forms of the 17- and 27-point shapes give the same bits on either side of the
size where the default changes from one to the other."""
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["3d17pt", "3d27pt"])
@pytest.mark.parametrize("n", [64, 80])
@pytest.mark.parametrize("blkpsm", [0, 1])
@pytest.mark.parametrize("boundary", ["zero", "clamp"])
def test_plan_is_what_runs(gpu, shape, n, blkpsm, boundary):
    print(f"[j3d-plan] {shape} {n}^3 blkpsm={blkpsm} {boundary}", flush=True)
    field = O.uniform(n ** 3, 3, -1.0, 1.0).reshape(n, n, n)
    got, rep = P.j3d_run(field, 5, shape=shape, method="persistent", boundary=boundary, blkpsm=blkpsm)
    rc, info = P.plan(n, n, n, caps=P.query_device(), occupancy=rep.occupancy, method="persistent", shape=shape,
                      boundary=boundary, blkpsm=blkpsm)
    assert rc == 0
    windowed = blkpsm == 1 and n == 64
    assert info.reserved[0] == rep.reserved[0] == (2 if windowed else 1)
    assert info.grid[0] == rep.grid[0] and info.block == rep.block and info.occupancy == rep.occupancy
    assert (info.tile_y, rep.reg_planes) == ((8, 9) if windowed else (6, 2))
    assert got.tobytes() == O.iterate(field, O.stencil_from_shape(P.shape_info(shape), boundary), 5).tobytes()


@pytest.mark.parametrize("shape,dtype,method,last", [("3d17pt", "f64", "persistent", 275), ("3d17pt", "f64", "plain", 369),
                                                     ("3d17pt", "f32", "plain", 465), ("3d27pt", "f64", "persistent", 465)])
def test_forms_agree_at_the_limits(gpu, shape, dtype, method, last):
    torch = gpu
    for n in (last, last + 1):
        print(f"[j3d-plan] {shape} {dtype} {method} {n}^3", flush=True)
        init = torch.empty(n ** 3, dtype=torch.float64 if dtype == "f64" else torch.float32, device="cuda")
        P.fill_uniform(init, n ** 3, 5, 0.0, 1.0, dtype=dtype)
        out = []
        for tune in (None, [0, 0, 0, 0, 2], [0, 0, 0, 0, 3]):  # the default, windowed, LDS planes
            a, b = init.clone(), torch.empty_like(init)
            rep = P.j3d_device(a, b, n, n, n, 3, dtype=dtype, shape=shape, method=method, boundary="zero", tune=tune)
            out.append((b if rep.result_in_b else a, rep.reg_planes))
            del a, b
        assert (out[0][1] == 2) == (n == last) and out[1][1] > 2
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][0], out[2][0])
        del out, init
        torch.cuda.empty_cache()
