"""Solve-pair statistics: a pair counts when its kernels did work.  The counts
compared are whole numbers."""
import numpy as np
import pytest

import luspice_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [333, 3000])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_only_pairs_that_ran_are_counted(n, prec):
    print("case: pair statistics", n, prec, flush=True)
    c = L.mna("sized", n=n, lr=0.02, seed=7)
    B = L.Batch(c)
    assert B.refactor(prec)["rc"] == 0
    B.kernel_stats(reset=True)
    pairs = 0
    for rhs in (c.rhs, np.zeros(c.n), 2.0 * c.rhs, np.zeros(c.n), np.zeros(c.n), c.rhs):
        before = B.kernel_stats()
        x, rep = B.solve(rhs)
        assert rep["rc"] == 0, rep
        after = B.kernel_stats()
        pairs += rep["inner_total"]
        assert after["tri_count"] == pairs, (after, rep)
        if not rhs.any():
            assert rep["inner_total"] == 0 and not x.any()
            assert after["fwd_ms"] == before["fwd_ms"] and after["bwd_ms"] == before["bwd_ms"]
        else:
            assert after["fwd_ms"] > before["fwd_ms"] and after["bwd_ms"] > before["bwd_ms"]
    B.trisolve(c.rhs)
    assert B.kernel_stats()["tri_count"] == pairs + 1
    B.close()
