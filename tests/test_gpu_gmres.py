"""GMRES-IR launch sequence at the iteration counts where its kernels change.

A factor-only diagonal shift makes the preconditioner weak, so the solves take
more inner iterations than the product's kernel sums dot products for (four)
and, with a short restart length, several cycles; a step graph records fewer
iterations than such a circuit needs and goes on eagerly.  Tolerances: the true
residual is computed on the host from the caller's values (convergence stops
at 1e-10; an accepted solve may stop at 1e-9), x within 1e-6 of the fp64 oracle
(the pass line of every solution test here).
"""
import numpy as np
import pytest

import luspice_amd as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _residual(c, x):
    r = c.rhs - np.bincount(c.row, c.val * x[c.col], c.n)
    return np.linalg.norm(r) / np.linalg.norm(c.rhs)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("inner,outer", [(3, 40), (4, 40), (5, 40), (9, 20), (50, 7)])
def test_weak_preconditioner_converges(c0, c0_q, inner, outer, prec):
    print("case: gmres inner", inner, "outer", outer, prec, flush=True)
    c = L.Circuit(c0.n, c0.row, c0.col, c0.val, c0.rhs, q=c0_q)
    B = L.Batch(c, factor_shift=1e-2, ir_inner=inner, ir_outer=outer)
    assert B.refactor(prec)["rc"] == 0
    x, rep = B.solve(c.rhs)
    assert rep["rc"] == 0 and rep["fallback"] == 0, rep
    assert rep["inner_total"] >= 4, rep          # otherwise this case shows nothing
    if inner == 3:
        assert rep["outer"] >= 2, rep
    assert _residual(c, x) <= 1e-9
    assert abs(rep["max_rel_res"] - _residual(c, x)) <= 1e-12 + 0.1 * rep["max_rel_res"]
    rc, xo, _, _ = O.cpu_lu_ref(c.n, c.row, c.col, c.val, c0_q, c.rhs)
    assert rc == -1 and np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


def test_zero_right_hand_side_and_masked_circuits(c0, c0_q):
    """b = 0 converges at once with x = 0; masked circuits keep their x."""
    print("case: gmres zero rhs and mask", flush=True)
    c = L.Circuit(c0.n, c0.row, c0.col, c0.val, c0.rhs, q=c0_q)
    d = L.mna("sized", n=333, lr=0.02, seed=7)
    B = L.Batch([c, d, c])
    assert B.refactor("fp32")["rc"] == 0
    rhs = np.concatenate([c.rhs, d.rhs, np.zeros(c.n)])
    x, rep = B.solve(rhs)
    assert rep["rc"] == 0, rep
    assert np.all(x[c.n + d.n:] == 0.0)
    assert _residual(c, x[:c.n]) <= 1e-9 and _residual(d, x[c.n:c.n + d.n]) <= 1e-9
    B.set_rhs(rhs)
    assert B.solve_device()["rc"] == 0
    B.set_active([0, 1, 0])
    B.set_rhs(2.0 * rhs)
    rep = B.solve_device()
    assert rep["rc"] == 0 and rep["converged"] == 1, rep
    y = B.get_x()
    assert np.array_equal(y[:c.n], x[:c.n]) and np.array_equal(y[c.n + d.n:], x[c.n + d.n:])
    assert np.linalg.norm(y[c.n:c.n + d.n] - 2.0 * x[c.n:c.n + d.n]) <= 1e-8 * np.linalg.norm(y[c.n:c.n + d.n])


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_graph_step_goes_on_past_its_recorded_iterations(c0, c0_q, prec):
    print("case: graph continuation", prec, flush=True)
    c = L.Circuit(c0.n, c0.row, c0.col, c0.val, c0.rhs, q=c0_q)
    easy = L.mna("sized", n=150, lr=0.02, seed=3)
    B = L.Batch([c, easy], factor_shift=1e-2)
    rhs = np.concatenate([c.rhs, easy.rhs])
    for k in range(3):                            # recorded once, replayed
        B.set_rhs(rhs * (1.0 + k))
        rr, sr = B.graph_step(prec)
        assert rr["rc"] == 0 and sr["rc"] == 0 and sr["converged"] == 2, (rr, sr)
        assert sr["inner_total"] > 4, sr
        x = B.get_x() / (1.0 + k)
        assert _residual(c, x[:c.n]) <= 1e-9 and _residual(easy, x[c.n:]) <= 1e-9
        assert B.refactor(prec)["rc"] == 0        # eager work between replays
        xe, se = B.solve(rhs)
        assert se["rc"] == 0
        assert np.linalg.norm(x - xe) <= 1e-6 * np.linalg.norm(xe)
