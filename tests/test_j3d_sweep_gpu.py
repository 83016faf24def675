"""The plane-by-plane kernel of the 17- and 27-point shapes (tiles of 62 x 4
cells over z-slabs) at the sizes where its tiles, slabs and loads have edges,
bit for bit against the oracle, in every storage format."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

# x: one lane, a tile less one, full, plus one, two tiles; y: remainders of a tile of 4 rows; z: from a
# single plane (every neighbour plane outside) to slabs of several stages with odd and even remainders
DIMS = [(1, 1, 1), (1, 4, 62), (2, 3, 63), (3, 5, 61), (4, 8, 124), (5, 9, 125), (19, 7, 64), (70, 6, 130)]


@pytest.mark.parametrize("shape", ["3d17pt", "3d27pt"])
@pytest.mark.parametrize("fmt", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("method", ["plain", "persistent"])
@pytest.mark.parametrize("boundary", ["clamp", "zero"])
@pytest.mark.parametrize("dims", DIMS)
def test_plane_by_plane_tiles_match_oracle(gpu, shape, fmt, method, boundary, dims):
    torch = gpu
    steps = 4
    print(f"[j3d-sweep] {shape} {fmt} {method} {boundary} dims={dims}", flush=True)
    si = P.shape_info(shape)
    # the table's own weights (with its divisor) under clamp, plain weights under zero
    coefs = None if boundary == "clamp" else list(np.linspace(0.5, 1.5, len(si.coef)) / len(si.coef))
    st = O.stencil_from_shape(si, boundary, coefs=coefs)
    n = int(np.prod(dims))
    if fmt in ("f64", "f32"):
        dt = np.float64 if fmt == "f64" else np.float32
        field = O.uniform(n, 3, -1.0, 1.0, dt).reshape(dims)
        got, rep = P.j3d_run(field, steps, shape=shape, method=method, boundary=boundary, coefs=coefs)
        want = O.iterate(field, st, steps)
    else:
        a = torch.empty(n, dtype=torch.int16, device="cuda")
        b = torch.empty_like(a)
        P.fill_uniform(a, n, 3, 0.0, 1.0, dtype=fmt)
        field = a.cpu().numpy().view(np.uint16).reshape(dims).copy()
        rep = P.j3d_device(a, b, *dims, steps, dtype=fmt, shape=shape, method=method, boundary=boundary, coefs=coefs)
        got = (b if rep.result_in_b else a).cpu().numpy().view(np.uint16).reshape(dims)
        want = O.iterate16(field, st, steps, fmt)
    assert rep.reserved[0] == 1, "one step per pass"
    assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("fmt", ["f16", "bf16"])
@pytest.mark.parametrize("dims", [(5, 9, 125), (3, 4, 62)])
def test_plane_by_plane_stochastic_rounding_matches_oracle(gpu, fmt, dims):
    torch = gpu
    n = int(np.prod(dims))
    a = torch.empty(n, dtype=torch.int16, device="cuda")
    b = torch.empty_like(a)
    P.fill_uniform(a, n, 4, 0.0, 1.0, dtype=fmt)
    field = a.cpu().numpy().view(np.uint16).reshape(dims).copy()
    rep = P.j3d_device(a, b, *dims, 5, dtype=fmt, shape="3d27pt", method="persistent", boundary="clamp",
                       rounding="stochastic", round_seed=11)
    got = (b if rep.result_in_b else a).cpu().numpy().view(np.uint16).reshape(dims)
    st = O.stencil_from_shape(P.shape_info("3d27pt"), "clamp")
    assert got.tobytes() == O.iterate16_sr(field, st, 5, fmt, 11).tobytes()
