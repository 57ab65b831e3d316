"""The slab RRQR, persistent and per-step, on a matrix with a NaN: a column whose norm is not a
number is never the pivot, and the QR ends when no other is left. Both forms take every other
sum in the same order, so the kept ranks and the stored blocks of the level are equal bit for
bit, the NaNs in the same places."""
import numpy as np
import pytest

import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, symmetric_graph

pytestmark = pytest.mark.gpu


def factor(A, X, nl, prec, monkeypatch, persistent):
    for k in ("REG", "STEPPED_MIN_ROWS", "STEPPED_MIN_ELEMS"):
        monkeypatch.setenv(f"SPAND_RRQR_{k}", "0")
    monkeypatch.setenv("SPAND_RRQR_PERSISTENT", "1" if persistent else "0")
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_tol(1e-3)
    t.set_precision(prec)
    t.set_symm_kind("GEN")
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    return t


@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
@pytest.mark.parametrize("n,d", [(24, 2), (40, 2), (10, 3), (14, 3), (17, 3)])
def test_nan_columns_are_not_pivots(n, d, prec, monkeypatch):
    nl = 3
    print(f"case rrqr nan {d}D n={n} prec={prec}", flush=True)
    A, X = convdiff(n, d), linspace_nd(n, d)
    probe = factor(A, X, nl, prec, monkeypatch, False)
    ids, level = probe.get_dof2ID(), {int(r[0]): int(r[1]) for r in probe.get_clusters()}
    # an entry between two neighbouring clusters that level 0 sparsifies, the last of them
    cols = np.repeat(np.arange(A.n), np.diff(A.colptr))
    a, b = ids[A.rowval], ids[cols]
    up = np.array([level[int(i)] > 0 for i in ids])
    at = np.flatnonzero((a != b) & up[A.rowval] & up[cols])
    assert len(at)
    A.nzval[at[np.argmax(np.minimum(a[at], b[at]))]] = np.nan
    p, q = (factor(A, X, nl, prec, monkeypatch, on) for on in (True, False))
    ip, iq = p.ops(), q.ops()
    ip, iq = ip[ip[:, 7] == 0], iq[iq[:, 7] == 0]
    assert np.array_equal(ip, iq)
    orth = np.flatnonzero(ip[:, 0] == 6)
    assert (ip[orth, 6] > 1).any()
    for i in np.flatnonzero(ip[:, 0] <= 6):
        if ip[i, 5] * ip[i, 6]:
            dp, dq = p.op_data(i, ip[i]), q.op_data(i, iq[i])
            for k in dp:
                assert np.array_equal(dp[k], dq[k], equal_nan=True), (i, k)
