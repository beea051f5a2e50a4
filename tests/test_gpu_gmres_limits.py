"""GMRES-IR at the limits of its options: no cycle at all, and vectors of many
reduction chunks."""
import numpy as np
import pytest

import luspice_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_no_cycle_leaves_x_at_zero(prec):
    """ir_outer = 0 asks for no refinement: x = 0 with its residual, not converged."""
    print("case: ir_outer 0", prec, flush=True)
    c = L.mna("sized", n=700, lr=0.02, seed=5)
    B = L.Batch(c, ir_outer=0, fallback_fp64=0)
    assert B.refactor(prec)["rc"] == 0
    for _ in range(2):
        x, rep = B.solve(c.rhs)
        assert not x.any()
        assert rep["rc"] == -8 and rep["outer"] == 0 and rep["inner_total"] == 0 and rep["converged"] == 0, rep
        assert rep["max_rel_res"] == 1.0, rep
    x, rep = B.solve(np.zeros(c.n))
    assert rep["rc"] == 0 and rep["converged"] == 1 and not x.any(), rep
    B.close()


@pytest.mark.parametrize("sizes,chunk", [((3000,), 1), ((3000, 333, 2500), 1), ((3000,), 2), ((3000,), 512)])
@pytest.mark.parametrize("inner", [3, 40])
def test_many_reduction_chunks(sizes, chunk, inner):
    """Chunks of 1 and 2 rows: the parts of a sum are added up by a launch of
    their own (9 and 2.25 million reads a sum at 3000 rows); 512 rows: by the
    kernels that need them.  Residuals on the host from the caller's values: a
    solve that reports convergence met 1e-9, and reported it to rounding."""
    print("case: reduction chunks", sizes, chunk, inner, flush=True)
    circ = [L.mna("sized", n=n, lr=0.02, seed=n) for n in sizes]
    B = L.Batch(circ, chunk_rows=chunk, ir_inner=inner, ir_outer=60, factor_shift=1e-3)
    for prec in ("fp32", "fp64"):
        B.set_active(None)
        assert B.refactor(prec)["rc"] == 0
        rhs = np.concatenate([c.rhs for c in circ])
        for mask in (None, [1] + [0] * (len(sizes) - 1)):
            B.set_active(mask)
            x, rep = B.solve(rhs)
            assert rep["rc"] == 0 and rep["fallback"] == 0, rep
            assert rep["inner_total"] >= 5, rep
            o, worst = 0, 0.0
            for i, c in enumerate(circ):
                if mask is None or mask[i]:
                    v = x[o:o + c.n]
                    r = c.rhs - np.bincount(c.row, c.val * v[c.col], c.n)
                    worst = max(worst, np.linalg.norm(r) / np.linalg.norm(c.rhs))
                o += c.n
            assert worst <= 1e-9 and abs(worst - rep["max_rel_res"]) <= 1e-12 + 0.1 * worst, (worst, rep)
    B.close()


@pytest.mark.parametrize("inner", [64, 65, 130])
@pytest.mark.parametrize("chunk", [0, 16])
def test_long_cycles(inner, chunk):
    """Cycles of at most and of more than 64 steps (back substitution by the
    update itself or by a launch of its own), beside a circuit that takes few.
    Residuals as above; the second circuit's solution within 1e-6 of its own
    solve (the pass line of every solution test here)."""
    print("case: long cycles", inner, chunk, flush=True)
    circ = [L.mna("sized", n=n, lr=0.02, seed=n) for n in (1500, 300)]
    B = L.Batch(circ, chunk_rows=chunk, ir_inner=inner, ir_outer=60, factor_shift=0.1)
    assert B.refactor("fp64")["rc"] == 0
    rhs = np.concatenate([c.rhs for c in circ])
    x, rep = B.solve(rhs)
    assert rep["rc"] == 0 and rep["fallback"] == 0, rep
    assert rep["inner_total"] > inner, rep            # a full cycle of `inner` steps, then another
    o, worst = 0, 0.0
    for c in circ:
        v = x[o:o + c.n]
        r = c.rhs - np.bincount(c.row, c.val * v[c.col], c.n)
        worst = max(worst, np.linalg.norm(r) / np.linalg.norm(c.rhs))
        o += c.n
    assert worst <= 1e-9 and abs(worst - rep["max_rel_res"]) <= 1e-12 + 0.1 * worst, (worst, rep)
    A = L.Batch(circ[1])
    assert A.refactor("fp64")["rc"] == 0
    y, _ = A.solve(circ[1].rhs)
    assert np.linalg.norm(x[circ[0].n:] - y) <= 1e-6 * np.linalg.norm(y)
    A.close()
    B.close()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_many_reduction_chunks_in_a_graph(prec):
    """The launches that add up the parts are recorded with the step: every
    replay meets the residual line of the eager solve, eager work between them."""
    print("case: reduction chunks in a graph", prec, flush=True)
    c = L.mna("sized", n=3000, lr=0.02, seed=3)
    B = L.Batch(c, chunk_rows=1)
    for k in range(4):
        B.set_rhs(c.rhs * (1.0 + k))
        rr, sr = B.graph_step(prec)
        assert rr["rc"] == 0 and sr["rc"] == 0 and sr["converged"] == 1, (rr, sr)
        x = B.get_x() / (1.0 + k)
        r = c.rhs - np.bincount(c.row, c.val * x[c.col], c.n)
        assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(c.rhs)
        y, se = B.solve(c.rhs)
        assert se["rc"] == 0 and np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
    B.close()
