"""Every form of the persistent RRQR, bit for bit against the per-step launches (which take every
sum in the same order): the fine and the dense form at each number of rows per lane, clusters
that spread over the XCDs (no XCD holds their slabs, so they exchange through memory), and
waves in several launches. The forms are asked for through SPAND_RRQR_DENSE, the launches
through a lower number of slabs a launch (SPAND_RRQR_SLABS)."""
import numpy as np
import pytest
import scipy.sparse as sp

import spand_public_amd as S
from spand_public_amd.problems import CSC, convdiff, linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu


def factor(A, X, nl, tol, prec, symm, monkeypatch, **env):
    for k in ("REG", "STEPPED_MIN_ROWS", "STEPPED_MIN_ELEMS"):
        monkeypatch.setenv(f"SPAND_RRQR_{k}", "0")
    for k, v in env.items():
        monkeypatch.setenv(f"SPAND_RRQR_{k}", str(v))
    t = S.Tree(nl)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_tol(tol)
    t.set_precision(prec)
    t.set_symm_kind(symm)
    t.set_profiling(True)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    t.factorize()
    for k in env:
        monkeypatch.delenv(f"SPAND_RRQR_{k}")
    wave = t.kernel_profile().get("rrqr_wave", {"launches": 0})["launches"]
    return t, t.ops(), wave


def same(a, ia, b, ib):
    assert np.array_equal(ia, ib)
    for i in np.flatnonzero(ia[:, 0] <= 6):
        if ia[i, 5] * ia[i, 6]:
            da, db = a.op_data(i, ia[i]), b.op_data(i, ib[i])
            for k in da:
                assert np.array_equal(da[k], db[k]), (i, k)


def band(N, w, seed):
    """Random symmetric band matrix, a little more than diagonally dominant: on a line, its
    separators have w rows and are coupled across the leaves."""
    rng = np.random.default_rng(seed)
    d = rng.standard_normal((w, N))
    M = sp.diags([d[k, : N - k - 1] for k in range(w)], [-(k + 1) for k in range(w)], format="csc")
    M = M + M.T
    A = sp.csc_matrix(M + sp.diags(1.05 * np.asarray(abs(M).sum(1)).ravel()))
    A.sort_indices()
    return CSC(N, A.indptr, A.indices, A.data)


# rows of the clusters: at and just above each number that a form holds (FP32: 32, 64, 96, 128,
# 192, 256, 384, 512, 768, 1024; FP64: 32, 48, 64, 96, 128, 192, 256, 384, 512)
ROWS = [32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 192, 193, 256, 257, 384, 385, 512]
LONG = [513, 768, 769, 1000]  # FP32 only


@pytest.mark.parametrize("prec,w", [(S.FP64, w) for w in ROWS] + [(S.FP32, w) for w in ROWS + LONG])
def test_each_form_equals_per_step(prec, w, monkeypatch):
    N = int(6.2 * w)  # three separators of w rows
    A, X = band(N, w, w), linspace_nd(N, 1)
    b, ib, _ = factor(A, X, 3, 1e-3, prec, "SPD", monkeypatch, PERSISTENT=0)
    assert b.level_tune()[0]["rows_max"] == w
    assert (ib[ib[:, 0] == 6][:, 6] > w // 4).any()  # many steps
    for dense in (0, 1):
        print(f"case rrqr form prec={prec} rows={w} dense={dense}", flush=True)
        a, ia, wave = factor(A, X, 3, 1e-3, prec, "SPD", monkeypatch, DENSE=dense)
        assert wave > 0
        same(a, ia, b, ib)


@pytest.mark.parametrize("prec", [S.FP64, S.FP32])
@pytest.mark.parametrize("n,d,nl,tol,symm", [(12, 3, 4, 1e-2, "SPD"), (16, 3, 5, 1e-2, "GEN"), (20, 3, 5, 1e-1, "SPD"),
                                             (60, 2, 4, 1e-3, "SPD")])
@pytest.mark.parametrize("dense", [0, 1])
def test_spread_and_chunked_launches_equal_per_step(n, d, nl, tol, symm, prec, dense, monkeypatch):
    A, X = (neglapl(n, d) if symm == "SPD" else convdiff(n, d)), linspace_nd(n, d)
    b, ib, _ = factor(A, X, nl, tol, prec, symm, monkeypatch, PERSISTENT=0)
    _, _, whole = factor(A, X, nl, tol, prec, symm, monkeypatch, DENSE=dense)
    cols = max(r["cols_max"] for r in b.level_tune())
    launches = []
    # from one that the largest cluster just fits (64 columns a slab at most, 4 at least), where every
    # cluster of more than an eighth of it spreads, to one that holds a few of them an XCD
    for cap in ((cols + 3) // 4, 2 * cols, 8 * cols):
        print(f"case rrqr spread {symm} {d}D n={n} prec={prec} dense={dense} slabs={cap}", flush=True)
        a, ia, wave = factor(A, X, nl, tol, prec, symm, monkeypatch, DENSE=dense, SLABS=cap)
        same(a, ia, b, ib)
        launches.append(wave)
    assert whole > 0 and launches[0] >= whole
