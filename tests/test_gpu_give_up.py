"""A refactor whose dependency waits give up: the poll limit is set to its
smallest from the host (LSP_REFACTOR_ROUNDS), so the waits end early, the launch
drains and the report names the wait.  Columns, dependencies and codes are whole
numbers; the solution after it within 1e-6 of the oracle (the pass line of every
solution test here)."""
import re

import numpy as np
import pytest

import luspice_amd as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _dense(n):
    """One supernode: every wait is on the values of the column's last run."""
    rng = np.random.default_rng(3)
    A = rng.uniform(-1, 1, (n, n)) + 2 * n * np.eye(n)
    r, c = np.indices((n, n))
    return L.Circuit(n, r.ravel(), c.ravel(), A.ravel(), rng.uniform(-1, 1, n), q=np.arange(n))


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("kind", ["dense", "c0"])
def test_report_names_the_wait(c0, c0_q, monkeypatch, kind, prec):
    print("case: waits given up", kind, prec, flush=True)
    c = _dense(400) if kind == "dense" else L.Circuit(c0.n, c0.row, c0.col, c0.val, c0.rhs, q=c0_q)
    opts = {"tail_max": -1}
    with monkeypatch.context() as m:
        m.setenv("LSP_REFACTOR_ROUNDS", "0")
        B = L.Batch(c, **opts)
    for k in range(2):
        rep = B.refactor(prec)
        assert rep["rc"] == -6, rep
        got = re.search(r"column (-?\d+) waiting on (-?\d+) (.*) epoch (-?\d+) polls (\d+)", rep["error"])
        assert got, rep
        col, dep, epoch, polls = int(got[1]), int(got[2]), int(got[4]), int(got[5])
        assert 0 <= dep < col < c.n and epoch == 1 + k and polls >= 1, rep
        if kind == "dense":
            assert got[3] == "by its values", rep
    B.close()
    B = L.Batch(c, **opts)
    assert B.refactor(prec)["rc"] == 0
    x, rep = B.solve(c.rhs)
    assert rep["rc"] == 0, rep
    rc, xo, _, _ = O.cpu_lu_ref(c.n, c.row, c.col, c.val, c.q, c.rhs)
    assert rc == -1 and np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)
    B.close()
