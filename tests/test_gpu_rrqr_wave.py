"""The persistent RRQR (one wavefront per slab) at the edges of its kernel forms: clusters just
below and above each number of rows a form holds, with one slab and with many.

Against the per-step launches of the same tree: both take every sum in the same order, so the
op sequence, the kept ranks and every stored block are equal bit for bit, in both precisions.
(The per-step path is compared with the oracle elsewhere.)"""
import numpy as np
import pytest

import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu


def factor(A, X, nl, tol, prec, symm, monkeypatch, persistent):
    monkeypatch.setenv("SPAND_RRQR_REG", "0")
    monkeypatch.setenv("SPAND_RRQR_STEPPED_MIN_ROWS", "0")
    monkeypatch.setenv("SPAND_RRQR_STEPPED_MIN_ELEMS", "0")
    monkeypatch.setenv("SPAND_RRQR_PERSISTENT", "1" if persistent else "0")
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_tol(tol)
    t.set_precision(prec)
    if symm != "SPD":
        t.set_symm_kind(symm)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    return t


# (edge, dimension, levels, tol, symm): rows up to about edge^2 / 2 in 3D, edge / 2 in 2D
CASES = [(9, 2, 3, 0.0, "SPD"), (60, 2, 3, 1e-3, "SPD"), (66, 2, 3, 0.0, "SPD"), (8, 3, 3, 1e-2, "SPD"),
         (9, 3, 3, 1e-2, "GEN"), (10, 3, 3, 1e-3, "SPD"), (14, 3, 3, 1e-2, "SPD"), (16, 3, 3, 1e-1, "GEN"),
         (17, 3, 3, 1e-2, "SPD"), (20, 3, 3, 1e-2, "SPD"), (23, 3, 3, 1e-1, "SPD"), (28, 3, 3, 1e-1, "SPD"),
         (32, 3, 3, 1e-1, "SPD")]


@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
@pytest.mark.parametrize("n,d,nl,tol,symm", CASES)
def test_persistent_equals_per_step(n, d, nl, tol, symm, prec, monkeypatch):
    A, X = (neglapl(n, d) if symm == "SPD" else convdiff(n, d)), linspace_nd(n, d)
    a = factor(A, X, nl, tol, prec, symm, monkeypatch, True)
    print(f"case rrqr wave {symm} {d}D n={n} tol={tol} prec={prec} rows {max(r['rows_max'] for r in a.level_tune())} "
          f"cols {max(r['cols_max'] for r in a.level_tune())}", flush=True)
    b = factor(A, X, nl, tol, prec, symm, monkeypatch, False)
    ia, ib = a.ops(), b.ops()
    assert np.array_equal(ia, ib)
    for i in np.flatnonzero(ia[:, 0] <= 6):
        if ia[i, 5] * ia[i, 6]:
            da, db = a.op_data(i, ia[i]), b.op_data(i, ib[i])
            for k in da:
                assert np.array_equal(da[k], db[k]), (i, k)
