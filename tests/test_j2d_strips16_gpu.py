"""The row-streaming 2D kernel with 16-bit storage where its strips, segments
and loop trips have edges: one and two columns per lane, both boundaries, both
roundings, and fields that start on any element, bit for bit against the
oracle."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

# odd widths: one column per lane; even: two.  From one row and one strip to segments of one and of
# several trips; three strips and more, so that some touch no side face
DIMS = [(1, 56), (2, 57), (6, 112), (8, 120), (9, 121), (16, 128), (33, 129), (61, 301), (61, 384), (1031, 40)]


@pytest.mark.parametrize("shape", ["2d5pt", "2ds9pt", "2d13pt", "2d9pt", "2d25pt"])
@pytest.mark.parametrize("fmt", ["f16", "bf16"])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
@pytest.mark.parametrize("method", ["plain", "persistent"])
@pytest.mark.parametrize("boundary", ["zero", "clamp"])
@pytest.mark.parametrize("dims", DIMS)
def test_strip_edges_match_oracle(gpu, shape, fmt, rounding, method, boundary, dims):
    torch = gpu
    steps = 5
    print(f"[j2d-strips16] {shape} {fmt} {rounding} {method} {boundary} dims={dims}", flush=True)
    n = dims[0] * dims[1]
    si = P.shape_info(shape)
    coefs = None if boundary == "clamp" else list(np.linspace(0.5, 1.5, len(si.coef)) / len(si.coef))
    start = 1 if dims[0] % 2 else 0  # elements: a field need not start on a 32-bit word
    a = torch.zeros(n + 1, dtype=torch.int16, device="cuda")[start:start + n]
    b = torch.zeros(n + 1, dtype=torch.int16, device="cuda")[start:start + n]
    P.fill_uniform(a, n, 6, 0.0, 1.0, dtype=fmt)
    field = a.cpu().numpy().view(np.uint16).reshape(dims).copy()
    rep = P.jacobi2d_device(a, b, *dims, steps, dtype=fmt, shape=shape, method=method, boundary=boundary,
                            coefs=coefs, rounding=rounding, round_seed=17)
    got = (b if rep.result_in_b else a).cpu().numpy().view(np.uint16).reshape(dims)
    st = O.stencil_from_shape(si, boundary, coefs=coefs)
    want = O.iterate16_sr(field, st, steps, fmt, 17) if rounding == "stochastic" else O.iterate16(field, st, steps, fmt)
    assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("shape", ["2d5pt", "2d9pt"])
@pytest.mark.parametrize("method", ["plain", "persistent"])
@pytest.mark.parametrize("start", [0, 1])
def test_fp32_pairs_on_any_element(gpu, shape, method, start):
    torch = gpu
    dims, steps = (61, 384), 5
    print(f"[j2d-strips16] f32 {shape} {method} start={start}", flush=True)
    n = dims[0] * dims[1]
    field = O.uniform(n, 8, -1.0, 1.0, np.float32)
    a = torch.zeros(n + 1, dtype=torch.float32, device="cuda")[start:start + n]
    b = torch.zeros_like(a)
    a.copy_(torch.from_numpy(field))
    rep = P.jacobi2d_device(a, b, *dims, steps, dtype="f32", shape=shape, method=method, boundary="zero")
    got = (b if rep.result_in_b else a).cpu().numpy().reshape(dims)
    want = O.iterate(field.reshape(dims), O.stencil_from_shape(P.shape_info(shape), "zero"), steps)
    assert got.tobytes() == want.tobytes()
