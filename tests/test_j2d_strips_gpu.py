"""The row-streaming 2D kernel where its strips, segments and loop trips have
edges: widths around one and two strips of every depth, heights from one row to
many segments of a narrow grid, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

# strips store 64 - 2RL columns (pairs 128 - 2RL, rounded to even); a trip runs 2R + 1 or more rows at once
DIMS = [(1, 56), (2, 57), (3, 64), (4, 65), (6, 112), (7, 113), (8, 120), (9, 121), (16, 128), (33, 129), (4099, 40)]


@pytest.mark.parametrize("shape", ["2d5pt", "2ds9pt", "2d9pt", "2d25pt"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("method", ["plain", "persistent"])
@pytest.mark.parametrize("boundary", ["zero", "clamp"])
@pytest.mark.parametrize("dims", DIMS)
def test_strip_edges_match_oracle(gpu, shape, dtype, method, boundary, dims):
    steps = 5
    print(f"[j2d-strips] {shape} {np.dtype(dtype).name} {method} {boundary} dims={dims}", flush=True)
    si = P.shape_info(shape)
    coefs = None if boundary == "clamp" else list(np.linspace(0.5, 1.5, len(si.coef)) / len(si.coef))
    field = O.uniform(dims[0] * dims[1], 6, -1.0, 1.0, dtype).reshape(dims)
    got, _ = P.jacobi2d_run(field, steps, shape=shape, method=method, boundary=boundary, coefs=coefs)
    want = O.iterate(field, O.stencil_from_shape(si, boundary, coefs=coefs), steps)
    assert got.tobytes() == want.tobytes()
