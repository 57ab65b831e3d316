"""LU pivots of the panel kernels (k_getrf_panel, k_getrf_trail, k_getrf_split) at their edges:
one dense pivot of exactly n rows, around multiples of the panel width and of the update's
columns, one size for each number of rows a thread holds, and one that they leave to the
one-workgroup kernel (FP32). FP64 against the CPU oracle: the same
operations on every element in the same order, so L, U and the permutation are equal bit for
bit. FP32: L U = P^T A within n eps times |L| |U| (the bound of an LU as computed)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
import spand_public_amd as S
from spand_public_amd.problems import CSC, linspace_nd, symmetric_graph

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 9, 31, 32, 33, 40, 63, 64, 65, 91, 96, 97, 127, 128, 129, 160, 161, 255, 321, 1023, 1056, 1057, 2050, 2081]


def dense(n, kind):
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n))
    if kind == "ties":  # equal magnitudes (the first one is the pivot) and exact zeros in U
        M = np.round(M) + np.diag(np.where(np.arange(n) % 3 == 0, 0.0, 4.0))
    if kind == "dominant":  # no interchange at all
        M += 4.0 * n * np.eye(n)
    return M


def csc(M):
    A = sp.csc_matrix(M)
    A.sort_indices()
    return CSC(len(M), A.indptr, A.indices, A.data)


def lu_op(t):
    ops = t.ops()
    i = int(np.flatnonzero(ops[:, 0] == 1)[0])
    return t.op_data(i, ops[i])


def factor(M, prec):
    n = len(M)
    t = S.Tree(1)
    t.set_use_geo(True)
    t.set_Xcoo(linspace_nd(n, 1))
    t.set_precision(prec)
    t.set_symm_kind("GEN")
    A = csc(M)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    return t


@pytest.mark.parametrize("kind", ["random", "ties", "dominant"])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_oracle(n, kind):
    if (n > 1100 and kind != "random") or (n < 7 and kind == "ties"):  # rounded to a singular one
        pytest.skip("one matrix for the large sizes, a nonsingular one for the smallest")
    M = dense(n, kind)
    print(f"case getrf fp64 n={n} {kind}", flush=True)
    o, _ = oracle.setup_tree(csc(M), linspace_nd(n, 1), 1, 0.0, symm="GEN")
    o.factorize()
    a, b = lu_op(o), lu_op(factor(M, S.FP64))
    assert np.array_equal(a["p"], b["p"])
    assert np.array_equal(a["M"], b["M"]) and np.array_equal(a["U"], b["U"])


@pytest.mark.parametrize("n", [n for n in SIZES if n >= 31] + [4097])
def test_fp32_factors(n):
    M = dense(n, "random").astype(np.float32).astype(np.float64)
    print(f"case getrf fp32 n={n}", flush=True)
    d = lu_op(factor(M, S.FP32))
    bound = (n + 8) * np.finfo(np.float32).eps * (np.abs(d["M"]) @ np.abs(d["U"]))
    assert sorted(d["p"]) == list(range(n))
    assert (np.abs(d["M"] @ d["U"] - M[d["p"]]) <= bound).all()
