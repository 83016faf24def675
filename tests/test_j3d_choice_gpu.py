"""The 7-point persistent kernel with variant, levels and slabs left open: the
pass the planner picks for the domain and the step count, bit for bit against
the oracle, at sizes on either side of its choices."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

COEFS = [0.1, 0.12, 0.14, 0.16, 0.11, 0.09, 0.27]
# small cubes (few planes a workgroup), a row count just under and over one tile's, flat and tall domains
DIMS = [(1, 1, 1), (5, 33, 64), (32, 32, 32), (70, 30, 61), (24, 61, 130), (24, 65, 130), (3, 130, 200), (150, 9, 20)]


@pytest.mark.parametrize("fmt", ["f64", "f32", "bf16", "bf16sr"])
@pytest.mark.parametrize("boundary", ["zero", "clamp"])
@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("steps", [1, 5, 12])
def test_open_plan_matches_oracle(gpu, fmt, boundary, dims, steps):
    torch = gpu
    print(f"[j3d-choice] {fmt} {boundary} dims={dims} steps={steps}", flush=True)
    n = int(np.prod(dims))
    st = O.stencil_from_shape(P.shape_info("3d7pt"), boundary, coefs=COEFS)
    if fmt in ("f64", "f32"):
        field = O.uniform(n, 3, -1.0, 1.0, np.float64 if fmt == "f64" else np.float32).reshape(dims)
        got, rep = P.j3d_run(field, steps, method="persistent", boundary=boundary, coefs=COEFS)
        want = O.iterate(field, st, steps)
    else:
        a = torch.empty(n, dtype=torch.int16, device="cuda")
        b = torch.empty_like(a)
        P.fill_uniform(a, n, 3, 0.0, 1.0, dtype="bf16")
        field = a.cpu().numpy().view(np.uint16).reshape(dims).copy()
        sr = dict(rounding="stochastic", round_seed=9) if fmt == "bf16sr" else {}
        rep = P.j3d_device(a, b, *dims, steps, dtype="bf16", method="persistent", boundary=boundary, coefs=COEFS, **sr)
        got = (b if rep.result_in_b else a).cpu().numpy().view(np.uint16).reshape(dims)
        want = O.iterate16_sr(field, st, steps, "bf16", 9) if sr else O.iterate16(field, st, steps, "bf16")
    assert 2 <= rep.reserved[0] <= 4 and rep.reserved[1] == -(-steps // rep.reserved[0])
    assert got.tobytes() == want.tobytes()
