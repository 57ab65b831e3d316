"""A batch of more LU pivots than a launch has workgroups along y (65,536): a tridiagonal
nonsymmetric matrix with 131,072 leaves, eliminated in one batch, and as many separators,
scaled in another. The solution's residual: GMRES leaves ||M^{-1} r|| <= 1e-10 ||M^{-1} b||, and
M is about A, an upwind difference (diagonal 12, -11 behind, -1 ahead) of condition below 24
for the exact one-dimensional flow part; 1e-8 leaves a factor of four."""
import numpy as np
import pytest

import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, symmetric_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
def test_more_pivots_than_a_grid_has_rows(prec):
    n, nl = 270000, 18
    print(f"case getrf batch n={n} levels={nl} prec={prec}", flush=True)
    A, X = convdiff(n, 1), linspace_nd(n, 1)
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_precision(prec)
    t.set_symm_kind("GEN")
    t.set_tol(1e-2)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    assert t.level_tune()[0]["n_elim"] > 65536
    b = np.random.default_rng(7).standard_normal(n)
    x, info = S.gmres(A, b, t, iters=60, restart=30, tol=1e-10)
    assert info["status"] == 0 and np.linalg.norm(A.matvec(x) - b) <= 1e-8 * np.linalg.norm(b)
