"""Masked refactors that alternate precisions: a circuit outside the mask keeps
its factors, its dense block among them, whatever set the others write.

The factors compared are the same memory read twice, so they are equal bit for
bit; so are the solutions of the direct solves, which read nothing else.
"""
import numpy as np
import pytest

import luspice_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep,other", [("fp64", "fp32"), ("fp32", "fp64")])
@pytest.mark.parametrize("new_values", [False, True])
def test_masked_circuit_keeps_its_factors(keep, other, new_values):
    print("case: keep", keep, "other", other, "new values", new_values, flush=True)
    circ = [L.mna("sized", n=n, lr=0.02, seed=n) for n in (700, 1300)]
    for c in circ:
        c.q = L.colamd(c)
    B = L.Batch(circ, tail_density=0.3)
    assert all(B.info(i)["tail_T"] > 64 for i in range(2))
    rhs = np.random.default_rng(1).uniform(-1, 1, B.total_n)
    assert B.refactor(keep)["rc"] == 0
    F, x = B.export_factors(1), B.trisolve(rhs)
    if new_values:
        B.set_values(np.concatenate([c.val for c in circ]) * 1.25)
    B.set_active([0, 1])
    assert B.refactor(other)["rc"] == 0
    B.set_active([1, 0])
    assert B.refactor(keep)["rc"] == 0
    B.set_active(None)
    G, y = B.export_factors(1), B.trisolve(rhs)
    assert np.array_equal(F["Lx"], G["Lx"]) and np.array_equal(F["Ux"], G["Ux"])
    a = circ[0].n
    assert np.array_equal(x[a:], y[a:])
    if not new_values:
        assert np.linalg.norm(x[:a] - y[:a]) <= 1e-10 * np.linalg.norm(x[:a])
    B.close()
