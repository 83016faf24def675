"""CSR systems on either side of the sizes and row lengths where the CG kernel
changes the groups of 256 lanes that share a segment: a few iterations against
the oracle, bit for bit."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

SEGMENT = 4096


def banded(n, entries):
    """A symmetric, diagonally dominant band of `entries` to a row; the rows at
    both ends are shorter."""
    half = entries // 2
    offs = np.arange(-half, half + 1) * 3
    j = np.arange(n)[:, None] + offs
    inside = (j >= 0) & (j < n)
    rowptr = np.concatenate([[0], np.cumsum(inside.sum(1))]).astype(np.int32)
    val = np.broadcast_to(np.where(offs == 0, float(entries), -0.75), inside.shape)[inside]
    return rowptr, j[inside].astype(np.int32), val.copy()


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("entries", [7, 9, 15, 17])
@pytest.mark.parametrize("segments", [1, 32, 33, 128, 129])
def test_matches_oracle(gpu, segments, entries, precision):
    torch = gpu
    n = (segments - 1) * SEGMENT + 777
    dt = np.float64 if precision == "f64" else np.float32
    print(f"[cg-rows] segments={segments} entries={entries} {precision}", flush=True)
    rowptr, col, val = banded(n, entries)
    val = val.astype(dt)
    b = O.uniform(n, 21, -1.0, 1.0, dt)
    x = torch.zeros(n, dtype=torch.float64 if precision == "f64" else torch.float32, device="cuda")
    res = P.cg_solve("csr", n, torch.from_numpy(b).cuda(), x, tol=1e-12, max_iter=3, precision=precision,
                     rowptr=torch.from_numpy(rowptr).cuda(), col=torch.from_numpy(col).cuda(),
                     val=torch.from_numpy(val).cuda(), nnz=len(col))
    if precision == "f64":
        want_x, want_hist, want_k = O.cg(0, n, rowptr, col, val, 0, b, 1e-12, True, 3)
    else:
        want_x, want_hist, want_k = O.cg_f32(0, n, rowptr, col, val, 0, b, float(np.float32(1e-12) ** 2), True, 3)
    assert res.iterations == want_k == 3
    assert np.array_equal(res.history, want_hist)
    assert np.array_equal(x.cpu().numpy(), want_x)
