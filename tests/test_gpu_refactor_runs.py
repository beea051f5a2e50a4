"""Refactor updates at the run widths and row counts where their paths change.

The first w columns are dense among themselves and couple to r border
unknowns, so the border's columns apply a run of w columns with r rows below
it, and the border, which fills in, is itself a supernode of r columns whose
columns wait for one another in turn.  With a small LDS slice the columns live
in global scratch.  No dense trailing block.

Tolerances: the update sums run in fp64, so in exact order-free terms
|L U - P A Q| <= gamma |L| |U| entry by entry with gamma = 2 n 2^-53; fp32
storage rounds each entry of L and of U once more (relative 2^-24 each), so
gamma = 2 n 2^-53 + 3 * 2^-24 covers both factors and their product.
"""
import numpy as np
import pytest

import luspice_amd as L

pytestmark = pytest.mark.gpu


def _matrix(w, r, seed):
    rng = np.random.default_rng(seed)
    n = w + r
    A = np.zeros((n, n))
    A[:w, :w] = rng.uniform(-1, 1, (w, w))
    A[w:, :w] = rng.uniform(-1, 1, (r, w))
    A[:w, w:] = rng.uniform(-1, 1, (w, r))
    A[np.arange(n), np.arange(n)] = 2.0 * n + rng.uniform(0, 1, n)
    return A


def _dense(F, n):
    Lm, U = np.zeros((n, n)), np.zeros((n, n))
    for k in range(n):
        s = slice(F["Lp"][k], F["Lp"][k + 1])
        Lm[F["Li"][s], k] = F["Lx"][s]
        s = slice(F["Up"][k], F["Up"][k + 1])
        U[F["Ui"][s], k] = F["Ux"][s]
    return Lm, U


@pytest.mark.parametrize("w,r", [(1, 1), (1, 63), (2, 64), (3, 65), (4, 61), (5, 60), (4, 129), (8, 256), (9, 257),
                                 (10, 65), (17, 130), (25, 40), (26, 513), (63, 64), (64, 1), (65, 70)])
def test_runs(w, r):
    A = _matrix(w, r, 100 * w + r)
    n = w + r
    row, col = np.nonzero(A)
    c = L.Circuit(n, row.astype(np.int32), col.astype(np.int32), A[row, col], np.ones(n),
                  q=np.arange(n, dtype=np.int32))
    for cap in (0, -32):
        B = L.Batch(c, tail_max=-1, lds_cap=cap)
        for prec, extra in (("fp64", 0.0), ("fp32", 3 * 2.0 ** -24), ("fp64", 0.0)):
            print("case: run", w, "rows", r, "cap", cap, prec, flush=True)
            rep = B.refactor(prec)
            assert rep["rc"] == 0, rep
            F = B.export_factors(0)
            Lm, U = _dense(F, n)
            assert np.array_equal(F["pinv"], np.arange(n))
            np.fill_diagonal(Lm, 1.0)
            bound = (2 * n * 2.0 ** -53 + extra) * (np.abs(Lm) @ np.abs(U)) + 1e-300
            assert (np.abs(Lm @ U - A) <= bound).all(), np.max(np.abs(Lm @ U - A) / bound)
        B.close()
