"""One-workgroup triangular solves: the schedule on the CPU, the kernel on the GPU.

GPU tolerance: fp64 substitution solves (L + dL)(U + dU) x = P b with
|dL| <= n u |L| and |dU| <= n u |U|, so with the same factors on both sides the
residual of L U x = P b is at most 3 n 2^-53 |L| |U| |x| per entry.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(os.path.dirname(HERE), "luspice_amd", "csrc", "host")


@pytest.fixture(scope="module")
def emulator(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("local") / "local_solve")
    srcs = [os.path.join(HERE, "local_solve.cpp")] + \
        [os.path.join(HOST, f) for f in ("symbolic.cpp", "mna.cpp", "csc.cpp", "colamd.cpp")]
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", HOST, "-o", exe] + srcs, check=True)
    return exe


@pytest.mark.parametrize("kind,tail", [(0, 0), (0, 300), (40, 0), (200, 0), (3000, 0), (3000, 1000), (8000, 4000)])
def test_schedule(emulator, kind, tail):
    r = subprocess.run([emulator, str(kind), str(tail)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr


def test_schedule_catches_a_planted_mistake(emulator):
    r = subprocess.run([emulator, "3000", "0", "1"], capture_output=True, text=True, timeout=300)
    assert r.returncode != 0 and "FAIL" in r.stdout, r.stdout


def _residual_ok(F, b, x, q, n):
    import scipy.sparse as sp
    Lm = sp.csc_matrix((F["Lx"], F["Li"], F["Lp"]), shape=(n, n))
    U = sp.csc_matrix((F["Ux"], F["Ui"], F["Up"]), shape=(n, n))
    z = x[q]
    pb = np.empty(n)
    pb[F["pinv"]] = b
    res = np.abs(Lm @ (U @ z) - pb)
    bound = 3 * n * 2.0 ** -53 * (abs(Lm) @ (abs(U) @ np.abs(z))) + 1e-300
    return np.max(res / bound)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,opts", [((20, 65, 200), {}), ((1020,), {}), ((1020,), {"tail_max": -1}),
                                        ((4999,), {"tail_max": -1}), ((3000, 40, 8192, 8400), {})])
def test_solve_against_factors(sizes, opts):
    """Alone, without a dense block (wide supernodes), and beside circuits of
    the task queue (more than 8192 unknowns)."""
    import luspice_amd as L
    print("case: sizes", sizes, opts, flush=True)
    circ = [L.mna("sized", n=n, lr=0.02, seed=9 + n) for n in sizes]
    for c in circ:
        c.q = L.colamd(c)
    B = L.Batch(circ, **opts)
    assert B.refactor("fp64")["rc"] == 0
    rhs = np.random.default_rng(5).uniform(-1, 1, B.total_n)
    for _ in range(2):                                   # a second solve reuses the work arrays
        x = B.trisolve(rhs)
        o = 0
        for i, c in enumerate(circ):
            F = B.export_factors(i)
            worst = _residual_ok(F, rhs[o:o + c.n], x[o:o + c.n], np.asarray(c.q), c.n)
            assert worst <= 1.0, (c.n, worst)
            o += c.n
    B.close()
