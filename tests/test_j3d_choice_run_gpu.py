"""The 7-point persistent kernel's open plan: the run reports the levels and the
tile variant that were planned, with the per-step kernel's bits."""
import numpy as np
import pytest

import perks_amd as P

pytestmark = pytest.mark.gpu


# many steps: the plan's own count; levels that divide 24 steps evenly change nothing
@pytest.mark.parametrize("dims,dtype,boundary,levels,variant", [((64, 64, 64), "f64", "zero", 3, 0),
                                                                ((128, 128, 128), "f32", "clamp", 4, 3),
                                                                ((50, 512, 512), "f64", "clamp", 4, 0),
                                                                ((128, 128, 128), "f16", "clamp", 4, 3)])
def test_seven_point_choice_runs(gpu, dims, dtype, boundary, levels, variant):
    torch = gpu
    print(f"[j3d-plan] 3d7pt {dtype} {boundary} {dims}", flush=True)
    n, steps = int(np.prod(dims)), 24
    coefs = [0.1, 0.12, 0.14, 0.16, 0.11, 0.09, 0.27]
    tdt = {"f64": torch.float64, "f32": torch.float32, "f16": torch.int16}[dtype]
    init = torch.empty(n, dtype=tdt, device="cuda")
    P.fill_uniform(init, n, 7, 0.0, 1.0, dtype=dtype)
    res = []
    for method in ("persistent", "plain"):
        a, b = init.clone(), torch.empty_like(init)
        rep = P.j3d_device(a, b, *dims, steps, dtype=dtype, method=method, boundary=boundary, coefs=coefs)
        res.append((b if rep.result_in_b else a, rep))
    assert torch.equal(res[0][0], res[1][0])
    rep = res[0][1]
    assert (rep.reserved[0], rep.reserved[1], rep.reserved[2]) == (levels, steps // levels, variant)
    rc, info = P.plan(*dims, dtype=dtype, caps=P.query_device(), occupancy=rep.occupancy, method="persistent",
                      boundary=boundary, coefs=coefs)
    assert rc == 0 and info.reserved[0] == levels and info.block == rep.block
