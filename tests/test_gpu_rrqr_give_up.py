"""A wait of the persistent RRQR that gives up costs time, not the factorization: with the bound
lowered to one poll the waits fail, every workgroup returns, and factorize does its work again
with one launch per pivot step. The result is the oracle's, the flag says so, and the tree's later
factorizations keep to the per-step launches."""
import numpy as np
import pytest

import oracle
import spand_public_amd as S
from spand_public_amd.problems import convdiff, linspace_nd, neglapl, symmetric_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("symm", ["SPD", "GEN"])
@pytest.mark.parametrize("everywhere", [False, True])
def test_give_up_is_redone_per_step(symm, everywhere, monkeypatch):
    print(f"case rrqr give up {symm} everywhere={everywhere}", flush=True)
    A, X = (neglapl(20, 3) if symm == "SPD" else convdiff(20, 3)), linspace_nd(20, 3)
    if everywhere:  # every cluster on the slab path
        for k in ("REG", "STEPPED_MIN_ROWS", "STEPPED_MIN_ELEMS"):
            monkeypatch.setenv(f"SPAND_RRQR_{k}", "0")
    t = S.Tree(7)
    t.set_use_geo(True)
    t.set_Xcoo(X)
    t.set_tol(1e-2)
    t.set_symm_kind(symm)
    t.partition(symmetric_graph(A))
    t.assemble(A)
    assert "persistent_rrqr_gave_up" not in t.status_flags()
    monkeypatch.setenv("SPAND_RRQR_SPIN_MAX", "1")
    t.set_profiling(True)
    t.factorize()
    assert t.status_flags()["persistent_rrqr_gave_up"]
    monkeypatch.delenv("SPAND_RRQR_SPIN_MAX")
    o, _ = oracle.setup_tree(A, X, 7, 1e-2, symm=symm)
    o.factorize()
    b = np.random.default_rng(5).standard_normal(A.n)
    xo = o.solve(b)
    for again in (False, True):
        if again:
            t.profile_reset()
            t.factorize()
            assert t.kernel_profile().get("rrqr_wave", {"launches": 0})["launches"] == 0
        assert np.array_equal(o.ops(), t.ops())
        assert np.linalg.norm(xo - t.solve(b)) <= 1e-12 * np.linalg.norm(xo)
