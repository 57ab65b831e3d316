"""The Orthogonal ops folded into their clusters' scaling at factorization (W = Q^T L^{-1})."""
import numpy as np
import pytest

import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu
ORTHOGONAL = 6


def factor(n, d, nl, tol, prec, symm):
    A = neglapl(n, d) if symm == "SPD" else convdiff(n, d)
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(linspace_nd(n, d))
    t.set_tol(tol)
    t.set_precision(prec)
    t.set_symm_kind(symm)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    return A, t


@pytest.mark.parametrize("symm", ["SPD", "GEN"])
@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
def test_the_folds_temporaries_are_given_back(symm, prec, monkeypatch):
    """One device allocation per block keeps every block, so the two modes differ by what the
    fold gave back: at least Ve (m x k), S (k x k) and a Z (k x m) per op and side."""
    print(f"case fold memory {symm} prec={prec}", flush=True)
    _, t = factor(16, 3, 6, 1e-2, prec, symm)
    ops = t.ops()
    m, k = (ops[ops[:, 0] == ORTHOGONAL][:, c].astype(np.int64) for c in (5, 6))
    assert len(m) > 20 and k.sum() > 0
    kept = t.factor_info()["arena_bytes"]
    monkeypatch.setenv("SPAND_ARENA_CHUNK_BYTES", "0")
    _, u = factor(16, 3, 6, 1e-2, prec, symm)
    sides = 1 if symm == "SPD" else 2
    esz = 8 if prec == S.FP64 else 4
    assert u.factor_info()["arena_bytes"] - kept >= esz * int(((1 + sides) * m * k + k * k).sum())
    b = np.random.default_rng(1).standard_normal(16 ** 3)
    assert np.array_equal(t.solve(b), u.solve(b))
