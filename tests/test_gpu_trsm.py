"""Triangular solves (k_trsm) at the edges of their tiles: a band matrix of 2 n + w rows, two
interior clusters of about n + w / 2 and n - w / 2 rows around a separator of w, so that such
triangles are applied to panels of w rows or columns (right solves, and for LU left solves that gather
permuted rows of another block). Triangles around the 32-row diagonal blocks and the 16-row
tiles below them and on both sides of the chunk widths' bounds (128, 256), w around the 16- and
32-wide tiles and the chunk widths themselves. FP64 against the CPU oracle: the same operations on every
element in the same order, so every stored block is equal bit for bit. FP32: blocks within
4 (n + 8) eps of the oracle's in norm (substitution's n eps times the condition of a
diagonally dominant triangle, below 3, and the pivot's own rounding)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
import spand_public_amd as S
from spand_public_amd.problems import CSC, linspace_nd, symmetric_graph

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (5, 3), (15, 17), (31, 1), (32, 16), (33, 15), (33, 33), (47, 31), (48, 32), (49, 48), (64, 64),
         (65, 65), (97, 63), (127, 49), (128, 31), (129, 33), (161, 96), (255, 32), (256, 16), (259, 17), (300, 40)]


def band(n, w, symmetric):
    N = 2 * n + w
    rng = np.random.default_rng(1000 * n + w)
    M = np.triu(np.tril(rng.standard_normal((N, N)), w), -w)
    if symmetric:
        M = M + M.T
    M += np.diag(2.0 * np.abs(M).sum(1))
    M *= np.exp(rng.uniform(-1, 1, N))[:, None] if not symmetric else 1.0
    A = sp.csc_matrix(M)
    A.sort_indices()
    return CSC(N, A.indptr, A.indices, A.data)


def blocks(t):
    ops = t.ops()
    out = []
    for i in range(len(ops)):
        if ops[i, 0] not in (7, 8) and ops[i, 5] * ops[i, 6]:
            d = t.op_data(i, ops[i])
            out.append((ops[i, 0], np.tril(d["M"]) if ops[i, 0] == 0 else d["M"], d.get("U"), d.get("p")))
    return ops, out


def both(n, w, symm, prec):
    A = band(n, w, symm == "SPD")
    X = linspace_nd(A.n, 1)
    o, _ = oracle.setup_tree(A, X, 2, 0.0, symm=symm)
    o.factorize()
    t = S.Tree(2)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_precision(prec)
    t.set_symm_kind(symm)
    t.set_tol(0.0)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    (oo, ob), (go, gb) = blocks(o), blocks(t)
    assert np.array_equal(oo, go)
    assert ob
    b = np.random.default_rng(n).standard_normal(A.n)
    return ob, gb, o.solve(b), t.solve(b)


@pytest.mark.parametrize("symm", ["SPD", "GEN"])
@pytest.mark.parametrize("n,w", SIZES)
def test_fp64_equals_oracle(n, w, symm):
    print(f"case trsm fp64 n={n} w={w} {symm}", flush=True)
    ob, gb, xo, xg = both(n, w, symm, S.FP64)
    for a, b in zip(ob, gb):
        assert np.array_equal(a[1], b[1])
        if a[0] == 1:
            assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])
    assert np.linalg.norm(xo - xg) <= 1e-12 * np.linalg.norm(xo)


@pytest.mark.parametrize("symm", ["SPD", "GEN"])
@pytest.mark.parametrize("n,w", SIZES)
def test_fp32_close_to_oracle(n, w, symm):
    print(f"case trsm fp32 n={n} w={w} {symm}", flush=True)
    ob, gb, xo, xg = both(n, w, symm, S.FP32)
    bound = 4 * (n + 8) * np.finfo(np.float32).eps
    for a, b in zip(ob, gb):
        assert np.linalg.norm(a[1] - b[1]) <= bound * np.linalg.norm(a[1])
    assert np.linalg.norm(xo - xg) <= bound * np.linalg.norm(xo)
