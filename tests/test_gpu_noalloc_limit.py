"""How many columns the static workspace of the allocation-free apply holds, on the example that
its descriptions give: 64^3, 12 levels, tol 1e-2."""
import ctypes as C

import numpy as np
import pytest

import spand_public_amd as S
from spand_public_amd import _lib
from spand_public_amd.problems import linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [S.FP32, S.FP64])
def test_nine_columns_fit_and_ten_do_not(prec):
    torch = pytest.importorskip("torch")
    print(f"case noalloc limit prec={prec}", flush=True)
    A = neglapl(64, 3)
    t = S.Tree(12)
    t.set_use_geo(True)
    t.set_Xcoo(linspace_nd(64, 3))
    t.set_tol(1e-2)
    t.set_precision(prec)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    B = torch.tensor(np.random.default_rng(1).standard_normal((10, A.n)), device="cuda")
    x, ref = B.clone(), B.clone()
    torch.cuda.synchronize()
    solve = _lib.lib().spand_solve_device_noalloc
    assert solve(t._h, C.c_void_p(x.data_ptr()), 10, A.n, None) == 1  # SPAND_ERR_ARG
    assert solve(t._h, C.c_void_p(x.data_ptr()), 9, A.n, None) == 0
    t.solve_device(ref.data_ptr(), 9, A.n)
    torch.cuda.synchronize()
    assert torch.equal(x, ref) and torch.equal(x[9], B[9])
