"""The preconditioner apply at the edges of its kernel: 16 outputs a chunk, 16 inner positions a
step, column groups of 4, 16 and 32, phases shared by one workgroup or spread over the device.

Against the CPU oracle's solve (SPD and GEN, FP64: 1e-12 relative, the bound of the other
parity tests); any column count gives each column the same bits as alone (FP64, FP32, and the
adjoint apply), because a column's sums do not depend on the others."""
import numpy as np
import pytest

import oracle
import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu


def tree(A, X, nl, tol, prec=S.FP64, symm="SPD", skip=0):
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_tol(tol)
    t.set_skip(skip)
    t.set_precision(prec)
    if symm != "SPD":
        t.set_symm_kind(symm)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    return t


# (edge, dimension, levels, tol, skip): one-cluster tree, short ragged clusters, every rank
# zero or full, levels without scaling (their children are copied, not multiplied)
SHAPES = [(3, 2, 1, 0.0, 0), (13, 2, 4, 1e-1, 0), (17, 2, 4, 0.0, 0), (9, 3, 5, 1e-2, 0), (12, 3, 5, 1e-2, 2),
          (33, 2, 5, 1e-2, 5), (19, 3, 6, 10.0, 0)]


@pytest.mark.parametrize("symm", ["SPD", "GEN"])
@pytest.mark.parametrize("n,d,nl,tol,skip", SHAPES)
def test_apply_matches_oracle(n, d, nl, tol, skip, symm):
    print(f"case apply {symm} {d}D n={n} levels={nl} tol={tol} skip={skip}", flush=True)
    A, X = (neglapl(n, d) if symm == "SPD" else convdiff(n, d)), linspace_nd(n, d)
    o, _ = oracle.setup_tree(A, X, nl, tol, skip=skip, symm=symm)
    o.factorize()
    g = tree(A, X, nl, tol, symm=symm, skip=skip)
    B = np.random.default_rng(3).standard_normal((A.n, 5))
    xg = g.solve(B)
    for j in range(5):
        xo = o.solve(B[:, j])
        assert np.linalg.norm(xg[:, j] - xo) <= 1e-12 * np.linalg.norm(xo)
    # the adjoint: <M^{-1} b, c> = <b, M^{-T} c>
    C = np.random.default_rng(4).standard_normal((A.n, 5))
    y = g.solve_transpose(C)
    lhs, rhs = (xg * C).sum(0), (B * y).sum(0)
    scale = np.linalg.norm(xg, axis=0) * np.linalg.norm(C, axis=0)
    assert np.all(np.abs(lhs - rhs) <= 1e-12 * scale)


@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
@pytest.mark.parametrize("symm", ["SPD", "GEN"])
def test_apply_columns_do_not_depend_on_their_number(symm, prec):
    print(f"case apply widths {symm} prec={prec}", flush=True)
    n, d, nl = 14, 3, 6
    A, X = (neglapl(n, d) if symm == "SPD" else convdiff(n, d)), linspace_nd(n, d)
    g = tree(A, X, nl, 1e-2, prec=prec, symm=symm)
    B = np.random.default_rng(5).standard_normal((A.n, 64))
    full, fullt = g.solve(B), g.solve_transpose(B)
    for w in (1, 3, 4, 5, 16, 17, 32, 33, 63):
        assert np.array_equal(g.solve(B[:, :w]), full[:, :w]), w
        assert np.array_equal(g.solve_transpose(B[:, :w]), fullt[:, :w]), w
