"""The stored values' gradient (k_sampled_outer) at the edges of its split: rows with none, one,
eight (a row's lanes), nine and many stored entries, one to 33 right-hand sides (eight in
flight together), a leading dimension past the rows. Against the definition in NumPy, within
r eps times the sum of |u v| (the bound of a sum of r products in any order)."""
import numpy as np
import pytest
import scipy.sparse as sp

import spand_public_amd as S
from spand_public_amd.problems import CSC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 700])
@pytest.mark.parametrize("nrhs", [1, 7, 8, 9, 16, 33])
def test_sampled_outer(n, nrhs):
    torch = pytest.importorskip("torch")
    print(f"case outer n={n} nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(100 * n + nrhs)
    M = np.zeros((n, n))
    for i in range(n):
        k = min(n, [1, 8, 9, 0, 5, 17, n][i % 7])
        M[i, rng.choice(n, k, replace=False)] = 1.0
    A = sp.csc_matrix(M)
    A.sort_indices()
    ld = n + 3
    u, v = rng.standard_normal((nrhs, ld)), rng.standard_normal((nrhs, ld))
    du, dv = torch.from_numpy(u).cuda(), torch.from_numpy(v).cuda()
    out = torch.full((A.nnz,), float("nan"), dtype=torch.float64, device="cuda")
    m = S.Matrix(CSC(n, A.indptr, A.indices, A.data))
    m.sampled_outer_device(du.data_ptr(), dv.data_ptr(), nrhs, ld, -2.0, out.data_ptr())
    cols = np.repeat(np.arange(n), np.diff(A.indptr))
    p = u[:, A.indices] * v[:, cols]
    bound = 2.0 * (nrhs + 1) * np.finfo(np.float64).eps * np.abs(p).sum(0)
    assert (np.abs(out.cpu().numpy() + 2.0 * p.sum(0)) <= bound).all()
