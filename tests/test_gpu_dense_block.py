"""Dense trailing block at the orders where its 64 x 64 tiles begin and end.

The block's order is forced through the options (tail_max with a density that
every block meets), and every factor entry is compared with the oracle's.
fp64: the oracle differs in summation order only, so the tolerances are those
of the existing factor parity test.  fp32 storage: the sparse columns are
stored in fp32 and read back, so entries carry a few times 2^-24 of the
column's largest intermediate value; 1e-4 of the column maximum is far above
that and far below any misplaced tile.
"""
import numpy as np
import pytest

import luspice_amd as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(F, R, n, rtol, atol):
    assert np.array_equal(F["pinv"], R["pinv"])
    assert np.array_equal(F["Lp"], R["Lp"]) and np.array_equal(F["Up"], R["Up"])
    for k in range(n):
        for p, i, x in (("Lp", "Li", "Lx"), ("Up", "Ui", "Ux")):
            s = slice(R[p][k], R[p][k + 1])
            of, orr = np.argsort(F[i][s], kind="stable"), np.argsort(R[i][s], kind="stable")
            assert np.array_equal(F[i][s][of], R[i][s][orr])
            np.testing.assert_allclose(F[x][s][of], R[x][s][orr], rtol=rtol, atol=atol * np.abs(R[x][s]).max())


@pytest.mark.parametrize("T", [64, 65, 127, 128, 129, 193, 256, 300])
def test_dense_block_orders(c0, c0_q, T):
    print("case: dense block of order", T, flush=True)
    B = L.Batch(L.Circuit(c0.n, c0.row, c0.col, c0.val, c0.rhs, q=c0_q), tail_max=T, tail_density=1e-9)
    assert B.info()["tail_T"] == T
    R = O.lu_factor(c0.n, c0.row, c0.col, c0.val, c0_q)
    for prec, rtol, atol in (("fp64", 1e-10, 1e-12), ("fp32", 1e-4, 1e-4), ("fp64", 1e-10, 1e-12)):
        rep = B.refactor(prec)
        assert rep["rc"] == 0, rep
        _check(B.export_factors(0), R, c0.n, rtol, atol)


def test_dense_blocks_of_uneven_order_in_one_launch(c0, c0_q):
    """Blocks of 1 to 5 panels in one batch, one circuit masked out: its
    factors stay those of the launch before."""
    print("case: uneven dense blocks", flush=True)
    circ = [L.mna("sized", n=n, lr=0.02, seed=40 + n) for n in (260, 700, 1300, 2100)]
    for c in circ:
        c.q = L.colamd(c)
    B = L.Batch(circ, tail_density=0.3)
    orders = [B.info(i)["tail_T"] for i in range(len(circ))]
    assert len({(t + 63) // 64 for t in orders}) >= 3, orders
    assert B.refactor("fp64")["rc"] == 0
    before = B.export_factors(2)
    B.set_active([1, 1, 0, 1])
    assert B.refactor("fp64")["rc"] == 0
    after = B.export_factors(2)
    assert np.array_equal(before["Lx"], after["Lx"]) and np.array_equal(before["Ux"], after["Ux"])
    for i, c in enumerate(circ):
        _check(B.export_factors(i), O.lu_factor(c.n, c.row, c.col, c.val, c.q), c.n, 1e-9, 1e-11)
