"""The persistent CG kernel's workgroup forms: four, two or one groups of 256
lanes to a segment of 4096 rows, by the number of segments.  A few iterations
on either side of each line, history and solution (whose update runs one phase
behind) bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P
from perks_amd import _lib as L

pytestmark = pytest.mark.gpu


def system(torch, fmt, dims):
    n = int(np.prod(dims))
    if fmt == "csr":
        rowptr, col, val = O.poisson7_csr(*dims)
        dev = dict(rowptr=torch.from_numpy(rowptr).cuda(), col=torch.from_numpy(col).cuda(),
                   val=torch.from_numpy(val).cuda(), nnz=len(col))
        return n, dev, (0, n, rowptr, col, val, 0)
    offs, val = O.poisson7_dia(*dims)
    return n, dict(offsets=offs, val=torch.from_numpy(val).cuda()), (1, n, None, offs, val, 7)


# 1 segment, less one row group; full; 2; 256 and 257 of them (256 CUs); 512 and 513
@pytest.mark.parametrize("fmt", ["csr", "dia"])
@pytest.mark.parametrize("dims", [(17, 16, 15), (16, 16, 16), (4097, 1, 1), (1024, 1024, 1), (1048577, 1, 1),
                                  (2048, 1024, 1), (2097153, 1, 1)])
@pytest.mark.parametrize("iterations", [1, 6])
def test_group_forms_match_oracle(gpu, fmt, dims, iterations):
    torch = gpu
    print(f"[cg-groups] {fmt} dims={dims} iterations={iterations}", flush=True)
    n, dev, host = system(torch, fmt, dims)
    b_host = O.uniform(n, 7, -1.0, 1.0)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    res = P.cg_solve(fmt, n, torch.from_numpy(b_host).cuda(), x, tol=1e-30, max_iter=iterations, **dev)
    want_x, want_hist, want_k = O.cg(*host, b_host, 1e-30, True, iterations)
    assert res.code == L.ERR_NOT_CONVERGED and res.iterations == want_k == iterations
    assert np.array_equal(res.history, want_hist)
    assert np.array_equal(x.cpu().numpy(), want_x)
