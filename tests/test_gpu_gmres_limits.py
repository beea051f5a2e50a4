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
