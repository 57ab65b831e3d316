"""FP32 triangular solves on the matrix cores (v_mfma_f32_16x16x4f32), bit for bit: the panels of
a leaf are A L^{-T} (SPD), A U^{-1} and L^{-1} P^T A (LU), every entry the ordered chain of fused
multiply-adds that the scalar recurrence takes: for k ascending x_k = a_k (1 / l_kk) (right) or
a_k / l_kk (left), a_i = fma(-x_k, l_ik, a_i). The oracle is the C library's fmaf on the stored
triangles and the assembled blocks."""
import ctypes as C
import ctypes.util

import numpy as np
import pytest
import scipy.sparse as sp

import spand_public_amd as S
from spand_public_amd.problems import CSC, linspace_nd, symmetric_graph

pytestmark = pytest.mark.gpu


def solve(L, B, left):
    """B L^{-T} row by row, or L^{-1} B column by column, in FP32, each multiply-add rounded once."""
    fmaf = C.CDLL(ctypes.util.find_library("m")).fmaf
    fmaf.restype, fmaf.argtypes = C.c_float, [C.c_float] * 3
    n = len(L)
    X = (B.T if left else B).copy()
    l = L.tolist()
    for row in range(len(X)):
        x = X[row].tolist()
        for k in range(n):
            b = np.float32(x[k]) / L[k, k] if left else np.float32(x[k]) * (np.float32(1) / L[k, k])
            x[k] = b = float(b)
            for i in range(k + 1, n):
                x[i] = fmaf(-b, l[i][k], x[i])
        X[row] = x
    return X.T if left else X


def same(X, Y):
    X, Y = np.ascontiguousarray(X, np.float32), np.ascontiguousarray(Y, np.float32)
    return X.shape == Y.shape and np.array_equal(X.view(np.int32), Y.view(np.int32))


# (rows of the leaf, rows of the separator): full and ragged tiles of 16 rows by 32 indices below
# diagonal blocks of 32; tiny scales a corner of the block into the subnormals
@pytest.mark.parametrize("n,w,tiny", [(33, 1, 0), (47, 17, 0), (64, 16, 0), (80, 33, 0), (97, 20, 0), (64, 16, 1),
                                      (80, 33, 1)])
@pytest.mark.parametrize("symm", ["SPD", "GEN"])
def test_fp32_panels_equal_the_scalar_chain(symm, n, w, tiny):
    print(f"case trsm bits {symm} n={n} w={w} tiny={tiny}", flush=True)
    N = 2 * n + w
    rng = np.random.default_rng(1000 * n + w)
    M = np.triu(np.tril(rng.standard_normal((N, N)), w), -w).astype(np.float32).astype(np.float64)
    if symm == "SPD":
        M = M + M.T
    M += np.diag(2.0 * np.abs(M).sum(1))
    if tiny:
        sep = slice(n, n + w)
        M[sep, :n] *= 2.0 ** -130
        M[:n, sep] *= 2.0 ** -130
    A = sp.csc_matrix(M)
    A.sort_indices()
    t = S.Tree(2)
    t.set_use_geo(True)
    t.set_Xcoo(linspace_nd(N, 1))
    t.set_precision(S.FP32)
    t.set_symm_kind(symm)
    t.set_tol(0.0)
    A = CSC(N, A.indptr, A.indices, A.data)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    ops, perm = t.ops(), t.get_assembly_perm()
    start = {int(r[0]): (int(r[6]), int(r[4])) for r in t.get_clusters() if r[0] <= 2}
    scaling = {int(ops[i, 1]): t.op_data(i, ops[i]) for i in np.flatnonzero(ops[:, 0] <= 1) if ops[i, 5]}
    seen = set()
    for i in np.flatnonzero(ops[:, 7] == 0):
        typ, c, nb = (int(v) for v in ops[i, :3])
        if typ not in (2, 4, 5) or not ops[i, 5] * ops[i, 6]:
            continue
        f = scaling[c]
        mine, other = (perm[start[q][0]:start[q][0] + start[q][1]] for q in (c, nb))
        X = t.op_data(i, ops[i])["M"]
        if typ == 5:
            L, B = np.tril(f["M"]), M[np.ix_(mine, other)][f["p"]]
        else:
            L, B = np.triu(f["U"]).T if typ == 4 else np.tril(f["M"]), M[np.ix_(other, mine)]
        assert X.any() and same(X, solve(L.astype(np.float32), B.astype(np.float32), typ == 5)), (typ, c)
        seen.add(typ)
    assert seen == ({2} if symm == "SPD" else {4, 5})
