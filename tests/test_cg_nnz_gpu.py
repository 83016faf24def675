"""CSR solves take the matrix's end from rowptr[n].  The nnz of the matrix
struct may count the arrays' capacity, or be 0: the FP64 and FP32 solves give
the same bits.  (A row's wide loads stop at that end, which decides what the
last rows of the matrix read.)"""
import numpy as np
import pytest

import oracle as O
import perks_amd as P
from perks_amd import _lib as L

pytestmark = pytest.mark.gpu


# 3 rows (fewer entries than one wide load); one segment; segments that no cache holds
@pytest.mark.parametrize("dims", [(3, 1, 1), (16, 16, 15), (160, 160, 150)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_nnz_of_the_struct_changes_nothing(gpu, dims, precision):
    torch = gpu
    dt = np.float32 if precision == "f32" else np.float64
    n = int(np.prod(dims))
    rowptr, col, val = O.poisson7_csr(*dims)
    val = val.astype(dt)
    b_host = O.uniform(n, 5, -1.0, 1.0, dt)
    b = torch.from_numpy(b_host).cuda()
    iters = 2 if n < 8 else 4  # three unknowns are solved in three
    if precision == "f64":
        want_x, want_hist, _ = O.cg(0, n, rowptr, col, val, 0, b_host, 1e-30, True, iters)
    else:
        want_x, want_hist, _ = O.cg_f32(0, n, rowptr, col, val, 0, b_host, float(np.float32(1e-20) ** 2), True, iters)
    slack = 64  # entries behind the matrix that a solve may not use
    dcol = torch.from_numpy(np.concatenate([col, np.full(slack, n - 1, np.int32)])).cuda()
    dval = torch.from_numpy(np.concatenate([val, np.full(slack, np.nan, dt)])).cuda()
    drow = torch.from_numpy(rowptr).cuda()
    for nnz in (len(col), len(col) + slack, 0):
        print(f"[cg-nnz] {precision} dims={dims} nnz={nnz} of {len(col)}", flush=True)
        x = torch.zeros(n, dtype=torch.float32 if precision == "f32" else torch.float64, device="cuda")
        res = P.cg_solve("csr", n, b, x, rowptr=drow, col=dcol, val=dval, nnz=nnz, tol=1e-30 if dt == np.float64 else 1e-20,
                         max_iter=iters, precision=precision)
        assert res.code in (0, L.ERR_NOT_CONVERGED)
        assert np.array_equal(res.history, want_hist)
        assert np.array_equal(x.cpu().numpy(), want_x)
