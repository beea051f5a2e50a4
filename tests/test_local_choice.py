"""Which circuits are solved by one workgroup each: the choice on the CPU at
batches where both ways were timed, and the kernel at its size limits, on batches
that are checked to go there.

GPU tolerance: substitution in fp64 on the stored factors solves (L + dL)(U + dU)
x = P b with |dL| <= n u |L| and |dU| <= n u |U| (u = 2^-53, whatever the factors'
storage), so the residual of L U x = P b is at most 3 n u |L| |U| |x| per entry.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(os.path.dirname(HERE), "luspice_amd", "csrc", "host")


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("choice") / "local_choice")
    srcs = [os.path.join(HERE, "local_choice.cpp")] + \
        [os.path.join(HOST, f) for f in ("symbolic.cpp", "mna.cpp", "csc.cpp", "colamd.cpp")]
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", HOST, "-o", exe] + srcs, check=True)

    def run(groups, tail_max=0):
        args = [str(v) for g in groups for v in g]
        r = subprocess.run([exe, str(tail_max)] + args, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr
        return [ch == "1" for ch in r.stdout.strip()]
    return run


def _spread(lo, hi, count):
    return [(int(n), 7, 1) for n in np.unique(np.exp(np.linspace(np.log(lo), np.log(hi), count)).astype(int))]


@pytest.mark.parametrize("groups,one_workgroup", [
    ([(200, 5, 1)], True),                  # alone: few tasks a level
    ([(1000, 5, 1)], True),
    ([(5000, 5, 1)], False),                # alone: many
    ([(8000, 5, 1)], False),
    ([(8000, 5, 32)], False),
    ([(8000, 5, 64)], True),                # the queue's task rate
    (_spread(100, 5000, 24), False),        # mixed: what the largest costs alone
    (_spread(100, 5000, 64), False),
    (_spread(2000, 8000, 48), False),
    (_spread(100, 5000, 256), True),
    ([(8400, 5, 1)], False),                # does not fit
])
def test_choice_where_both_ways_were_timed(choice, groups, one_workgroup):
    assert choice(groups) == [one_workgroup] * sum(g[2] for g in groups)


def test_circuits_that_do_not_fit_stay_in_the_queue(choice):
    got = choice([(9000, 5, 1), (3000, 5, 96)])
    assert not got[0] and all(got[1:])
    assert not any(choice([(9000, 5, 1), (3000, 5, 2)]))


def _residual(F, b, x, q, n):
    import scipy.sparse as sp
    Lm = sp.csc_matrix((F["Lx"], F["Li"], F["Lp"]), shape=(n, n))
    U = sp.csc_matrix((F["Ux"], F["Ui"], F["Up"]), shape=(n, n))
    z = x[q]
    pb = np.empty(n)
    pb[F["pinv"]] = b
    res = np.abs(Lm @ (U @ z) - pb)
    return np.max(res / (3 * n * 2.0 ** -53 * (abs(Lm) @ (abs(U) @ np.abs(z))) + 1e-300))


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,tail_max", [((8192, 8191), 0), ((4999, 4997), -1)])
def test_one_workgroup_solves_at_their_limits(choice, sizes, tail_max):
    """The most unknowns that fit, and wide supernodes without a dense block, in
    batches of copies large enough for the rule.  (Copies' factors differ by
    rounding: a refactor sums its dependencies as they become ready.)  Solves with
    the same factors are alike bit for bit."""
    import luspice_amd as L
    print("case: sizes", sizes, "tail_max", tail_max, flush=True)
    copies = 24
    assert all(choice([(n, 9 + n, copies) for n in sizes], tail_max))
    circ = []
    for n in sizes:
        c = L.mna("sized", n=n, lr=0.02, seed=9 + n)
        assert c.n == n
        c.q = L.colamd(c)
        circ += [c] * copies
    B = L.Batch(circ, tail_max=tail_max)
    part = [np.random.default_rng(n).uniform(-1, 1, n) for n in sizes]
    rhs = np.concatenate([np.tile(p, copies) for p in part])
    for prec in ("fp64", "fp32"):
        assert B.refactor(prec)["rc"] == 0
        x = B.trisolve(rhs)
        assert np.array_equal(x, B.trisolve(rhs))            # a second solve reuses the work arrays
        o = 0
        for i, n in enumerate(sizes):
            c = circ[i * copies]
            for k in (0, copies - 1):
                v = x[o + k * n:o + (k + 1) * n]
                worst = _residual(B.export_factors(i * copies + k), part[i], v, np.asarray(c.q), n)
                assert worst <= 1.0, (prec, n, k, worst)
            o += copies * n
    B.close()
