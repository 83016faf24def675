"""Irregular CSR systems in the workgroup forms of the persistent CG kernel (four,
two and one groups of 256 lanes to a segment of 4096 rows, for DIA by the number
of segments, for CSR by the entries per row as well): hub rows that the grid splits, rows on either side of the split
length, zero and nonzero starts, FP64, FP32 and refinement, caches on and off.
A few iterations against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P
from perks_amd import _lib as L

pytestmark = pytest.mark.gpu

SEGMENT = 4096
# last rows of a partly filled segment: 5 segments; 257 and 513 of them (256 CUs)
ROWS = {4: 4 * SEGMENT + 77, 2: 256 * SEGMENT + 77, 1: 512 * SEGMENT + 77}


def matrix(n, seed):
    """Symmetric and diagonally dominant: a path, one random link a row, and hub
    rows of 64 to 9000 links (with the path's, on either side of 64 and 4096
    entries) in the first, a middle and the last segment."""
    rng = np.random.default_rng(seed)
    rows = [np.arange(n - 1), np.arange(n)]
    cols = [np.arange(1, n), rng.integers(0, n, size=n)]
    for hub, degree in ((5, 9000), (SEGMENT + 1, 62), (SEGMENT + 9, 70), (n // 2, 4200), (n - 2, 500)):
        rows.append(np.full(degree, hub))
        cols.append(rng.choice(n, size=degree, replace=False))
    r, c = np.concatenate(rows), np.concatenate(cols)
    pair = np.unique(np.minimum(r, c) * np.int64(n) + np.maximum(r, c))
    lo, hi = pair // n, pair % n
    v = -rng.uniform(1e-3, 1.0, size=len(pair))
    lo, hi, v = lo[lo != hi], hi[lo != hi], v[lo != hi]
    diag = 1.0 + np.bincount(lo, -v, n) + np.bincount(hi, -v, n)
    i = np.arange(n)
    r, c, v = np.concatenate([lo, hi, i]), np.concatenate([hi, lo, i]), np.concatenate([v, v, diag])
    order = np.argsort(r * np.int64(n) + c)
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    return rowptr, c[order].astype(np.int32), v[order]


@pytest.fixture(scope="module", params=sorted(ROWS))
def system(gpu, request):
    groups = request.param
    n = ROWS[groups]
    cus = P.query_device().cu_count
    nseg = -(-n // SEGMENT)
    assert groups == (4 if nseg <= cus else 2 if nseg <= 2 * cus else 1)
    rowptr, col, val = matrix(n, groups)
    lens = np.diff(rowptr)
    assert (lens > 4096).sum() >= 2 and (lens > 64).sum() >= 4 and lens[5] > 4096 and lens[n - 2] > 64
    return groups, n, rowptr, col, val


def device(torch, rowptr, col, val):
    return dict(rowptr=torch.from_numpy(rowptr).cuda(), col=torch.from_numpy(col).cuda(),
                val=torch.from_numpy(val).cuda(), nnz=len(col))


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("x0", ["zero", "nonzero"])
@pytest.mark.parametrize("cache", [True, False])
def test_irregular_rows_match_oracle(gpu, system, precision, x0, cache):
    torch = gpu
    groups, n, rowptr, col, val = system
    iters = 4
    dt = np.float64 if precision == "f64" else np.float32
    print(f"[cg-irregular] groups={groups} {precision} x0={x0} cache={cache}", flush=True)
    val = val.astype(dt)
    b = O.uniform(n, 11, -1.0, 1.0, dt)
    start = O.uniform(n, 12, -0.5, 0.5, dt) if x0 == "nonzero" else np.zeros(n, dt)
    x = torch.from_numpy(start.copy()).cuda()
    tol = 1e-12
    res = P.cg_solve("csr", n, torch.from_numpy(b).cuda(), x, tol=tol, max_iter=iters, precision=precision,
                     x0_is_zero=(x0 == "zero"), cache_vector=cache, cache_matrix=cache,
                     **device(torch, rowptr, col, val))
    if precision == "f64":
        want_x, want_hist, want_k = O.cg(0, n, rowptr, col, val, 0, b, tol, True, iters, x0=start)
    else:
        want_x, want_hist, want_k = O.cg_f32(0, n, rowptr, col, val, 0, b, float(np.float32(tol) * np.float32(tol)),
                                             True, iters, x0=start)
    assert res.code == L.ERR_NOT_CONVERGED and res.long_rows == (np.diff(rowptr) > 64).sum()
    assert res.iterations == want_k == iters
    assert np.array_equal(res.history, want_hist)
    assert np.array_equal(x.cpu().numpy(), want_x)


@pytest.mark.parametrize("fmt", ["csr", "dia"])
def test_refinement_matches_oracle(gpu, system, fmt):
    torch = gpu
    groups, n, rowptr, col, val = system
    print(f"[cg-irregular] groups={groups} refinement {fmt}", flush=True)
    if fmt == "csr":
        dev, host = device(torch, rowptr, col, val), (0, n, rowptr, col, val, 0)
    else:
        offs, dval = O.poisson7_dia(n, 1, 1)
        dev, host = dict(offsets=offs, val=torch.from_numpy(dval).cuda()), (1, n, None, offs, dval, 7)
    b = O.uniform(n, 13, -1.0, 1.0)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    res = P.cg_solve(fmt, n, torch.from_numpy(b).cuda(), x, tol=1e-12, precision="f32_refine", inner_tol=1e-3,
                     max_inner=5, max_outer=2, **dev)
    want_x, want_hist, want_total, want_outer = O.cg_f32_refine(*host, b, 1e-12, True, 1e-3, 5, 2)
    assert res.outer_iterations == want_outer and res.iterations == want_total
    assert np.array_equal(res.history, want_hist)
    assert np.array_equal(x.cpu().numpy(), want_x)


@pytest.mark.parametrize("fmt", ["csr", "dia"])
def test_f32_poisson_matches_oracle(gpu, system, fmt):
    torch = gpu
    groups, n = system[:2]
    print(f"[cg-irregular] groups={groups} f32 poisson {fmt}", flush=True)
    if fmt == "csr":
        rowptr, col, val = O.poisson7_csr(n, 1, 1)
        val = val.astype(np.float32)
        dev, host = device(torch, rowptr, col, val), (0, n, rowptr, col, val, 0)
    else:
        offs, val = O.poisson7_dia(n, 1, 1)
        val = val.astype(np.float32)
        dev, host = dict(offsets=offs, val=torch.from_numpy(val).cuda()), (1, n, None, offs, val, 7)
    b = O.uniform(n, 14, -1.0, 1.0, np.float32)
    x = torch.zeros(n, dtype=torch.float32, device="cuda")
    res = P.cg_solve(fmt, n, torch.from_numpy(b).cuda(), x, tol=1e-12, max_iter=4, precision="f32", **dev)
    want_x, want_hist, want_k = O.cg_f32(*host, b, float(np.float32(1e-12) ** 2), True, 4)
    assert res.iterations == want_k == 4
    assert np.array_equal(res.history, want_hist)
    assert np.array_equal(x.cpu().numpy(), want_x)
