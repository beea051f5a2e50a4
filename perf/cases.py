"""Work that users of the framework have it do, as measurable cases.

A case is a dict of plain values:

  call     newton_host    one Newton step with the program's data on the host: values in, refactor,
                          GMRES-IR solve, x out (what the request loop does per cohort step)
           newton_device  the same step with values and right-hand side already in HBM, x left there
           newton_graph   the device step on the batch's own arenas, replayed as one HIP graph (batched Newton)
           direct         forward + backward solve with factors that are kept, a new right-hand side
                          per call (linear transient: the matrix does not change between time steps)
           spmv           y = A x, vectors in HBM
  circuit  c0, c1         the 1020-unknown circuit and the 316 x 316 power grid (n = 99 906)
           sized          one circuit of n unknowns, 2 % long-range branches
           grid           one circuit of n unknowns, grid edges only
           mix            `count` circuits, n log-uniform in [nmin, nmax], in one batch
  prec     fp32 | fp64    factor storage (for spmv: storage of the matrix values)

Patterns are the generators'; `prepare` draws values and vectors from its seed.
"""
import functools
import math

import numpy as np
import torch  # before luspice_amd: both then share one HIP runtime

import luspice_amd as L
from luspice_amd import _native as N
from luspice_amd import workloads as W


def listed():
    return [
        # smallest request of the serving range, all data on the host: launches and latency only
        {"name": "newton_n200_fp64_host", "call": "newton_host", "circuit": "sized", "n": 200, "prec": "fp64"},
        # the reference's own scale of circuit (n about 1000), mixed precision, data on the host
        {"name": "newton_c0_fp32_host", "call": "newton_host", "circuit": "c0", "n": 1020, "prec": "fp32"},
        # the largest circuit of the batched mix alone on the GPU, an odd size, data in HBM
        {"name": "newton_n4999_fp32", "call": "newton_device", "circuit": "sized", "n": 4999, "prec": "fp32"},
        # a cohort of the request loop: 17 circuits below 2k unknowns stepping together
        {"name": "cohort17_fp32_host", "call": "newton_host", "circuit": "mix", "count": 17, "nmin": 200, "nmax": 1999,
         "prec": "fp32"},
        # the headline benchmark: refactor + solve of the power grid, mixed and fp64
        {"name": "newton_c1_fp32", "call": "newton_device", "circuit": "c1", "n": 99906, "prec": "fp32"},
        {"name": "newton_c1_fp64", "call": "newton_device", "circuit": "c1", "n": 99906, "prec": "fp64"},
        # time stepping of the linear power grid: solves with kept factors
        {"name": "direct_c1_fp64", "call": "direct", "circuit": "c1", "n": 99906, "prec": "fp64"},
        # batched Newton over 512 uneven circuits, one graph per step, mixed and fp64
        {"name": "newton_mix512_fp32_graph", "call": "newton_graph", "circuit": "mix", "count": 512, "nmin": 100,
         "nmax": 5000, "prec": "fp32"},
        {"name": "newton_mix512_fp64_graph", "call": "newton_graph", "circuit": "mix", "count": 512, "nmin": 100,
         "nmax": 5000, "prec": "fp64"},
        # SpMV of one large matrix with fp32 values, and of a whole batch with fp64 values
        {"name": "spmv_c1_fp32", "call": "spmv", "circuit": "c1", "n": 99906, "prec": "fp32"},
        {"name": "spmv_mix512_fp64", "call": "spmv", "circuit": "mix", "count": 512, "nmin": 100, "nmax": 5000,
         "prec": "fp64"},
    ]


def draw(rng):
    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    circuit = rng.choice(["sized", "sized", "grid", "mix", "mix"])
    prec = rng.choice(["fp32", "fp64"])
    if circuit == "mix":
        nmin = logint(100, 1000)
        case = {"call": rng.choice(["newton_host", "newton_device", "newton_graph", "newton_graph", "direct", "spmv"]),
                "circuit": "mix", "count": logint(3, 400), "nmin": nmin, "nmax": logint(max(400, nmin), 5000)}
    else:
        n = logint(100, 5000) if circuit == "sized" else logint(3000, 90000)
        case = {"call": rng.choice(["newton_host", "newton_device", "newton_graph", "direct", "spmv"]),
                "circuit": circuit, "n": n}
    # one direct solve with fp32 factors is a preconditioner, not a solution: programs keep fp64 factors for it
    case["prec"] = "fp64" if case["call"] == "direct" else prec
    return case


@functools.lru_cache(maxsize=None)
def _circuits(circuit, n, count, nmin, nmax):
    """The patterns, base values and column orders: what a program has before its first step."""
    if circuit == "mix":
        return W.newton_mix(count, nmin, nmax)
    if circuit in ("c0", "c1"):
        c = L.mna(circuit, seed=int(circuit[1]))
    else:
        c = L.mna("sized", n=n, lr=0.02 if circuit == "sized" else 0.0, seed=5)
    c.q = L.colamd(c)
    return [c]


def _of(case):
    return _circuits(case["circuit"], case.get("n", 0), case.get("count", 0), case.get("nmin", 0), case.get("nmax", 0))


def _inputs(case, seed):
    """Values (every circuit's, in order) and right-hand sides of one step."""
    cs = _of(case)
    if case["circuit"] in ("c1", "grid"):
        # a resistive grid at another operating point: D A D keeps it symmetric, as conductances are
        c = cs[0]
        rng = np.random.default_rng(seed)
        d = np.exp(rng.normal(0.0, 0.05, c.n))
        return c.val * d[c.row] * d[c.col], rng.uniform(-1.0, 1.0, c.n)
    # a Newton step: every value times lognormal(0, 0.1), right-hand side uniform in [-1, 1]
    return W.step_inputs(cs, 0, seed=seed)


def prepare(case, seed):
    vals, rhs = _inputs(case, seed)
    B = L.Batch(_of(case))
    s = {"call": case["call"], "prec": case["prec"], "batch": B, "report": N.SolveReport()}
    if case["call"] == "newton_host":
        s.update(vals=vals, rhs=rhs)
        return s
    s["vals"] = torch.from_numpy(vals).cuda()
    s["rhs"] = torch.from_numpy(rhs).cuda()
    s["x"] = torch.empty_like(s["rhs"])
    if case["call"] in ("direct", "spmv"):
        B.set_values(vals)
        L.device_sync()  # vals goes with this call
    if case["call"] == "direct":
        _ok(B.refactor(case["prec"]))
    return s


def _ok(report):
    if report["rc"] != 0:
        raise RuntimeError(str(report))


def run(s):
    B, call = s["batch"], s["call"]
    if call == "newton_host":
        B.set_values(s["vals"])
        _ok(B.refactor(s["prec"]))
        x, report = B.solve(s["rhs"])
        _ok(report)
        return x
    rhs, x = s["rhs"].data_ptr(), s["x"].data_ptr()
    if call == "spmv":
        N.check(N.lib.lsp_batch_spmv(B._h, rhs, x, 1, L.prec_code(s["prec"])), "spmv")
    elif call == "direct":
        N.check(N.lib.lsp_batch_trisolve(B._h, rhs, x, 1), "trisolve")
    elif call == "newton_graph":
        B.set_values_device(s["vals"].data_ptr())
        B.set_rhs(rhs)
        _ok(B.graph_step(s["prec"])[1])
        N.check(N.lib.lsp_batch_get_x(B._h, N.C.cast(x, N.c_double_p)), "get_x")
    else:
        B.set_values_device(s["vals"].data_ptr())
        _ok(B.refactor(s["prec"]))
        N.check(N.lib.lsp_batch_solve(B._h, rhs, x, 1, N.C.byref(s["report"])), "solve")
    return s["x"]


@functools.lru_cache(maxsize=None)
def _counts(circuit, n, count, nmin, nmax):
    """Unknowns, entries, factor entries (both triangles) and left-looking updates."""
    B = L.Batch(_circuits(circuit, n, count, nmin, nmax), upload=False)
    info = [B.info(i) for i in range(len(B.circuits))]
    return tuple(sum(i[k] for i in info) for k in ("n", "nnz")) + (
        sum(i["lnnz"] + i["unnz"] for i in info), sum(i["n_updates"] for i in info))


def work(case):
    n, nnz, lu, updates = _counts(case["circuit"], case.get("n", 0), case.get("count", 0), case.get("nmin", 0),
                                  case.get("nmax", 0))
    v = 4 if case["prec"] == "fp32" else 8
    if case["call"] == "spmv":  # values, column ids, row pointers, x, y
        return {"bytes": nnz * (v + 4) + 4 * n + 16 * n, "flops": 2 * nnz}
    solve = {"bytes": lu * (v + 4) + 8 * n + 24 * n, "flops": 2 * lu}  # factors and their row ids once, b, x
    if case["call"] == "direct":
        return solve
    # values in, factors out (row ids read), one solve, one residual
    return {"bytes": 12 * nnz + lu * (v + 4) + 12 * n + solve["bytes"] + 12 * nnz + 20 * n,
            "flops": 2 * updates + solve["flops"] + 2 * nnz}


def _dense(n, row, col, val, b):
    """Solution by dense LU with one refinement step, on the GPU where there is one."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    A = torch.zeros(n * n, dtype=torch.float64, device=dev)
    A.index_add_(0, torch.from_numpy(row.astype(np.int64) * n + col).to(dev), torch.from_numpy(val).to(dev))
    A = A.view(n, n)
    r = torch.from_numpy(b).to(dev)
    lu, piv = torch.linalg.lu_factor(A)
    x = torch.linalg.lu_solve(lu, piv, r[:, None])
    x = x + torch.linalg.lu_solve(lu, piv, r[:, None] - A @ x)
    return x[:, 0].cpu().numpy()


def _banded(c, val, b):
    """Solution of a grid circuit by block-tridiagonal elimination with one refinement step.

    Grid nodes come in row order and each source unknown right after its node, so the half bandwidth is
    one grid row and the sources in it; a block holds that many unknowns and never parts a source from its node."""
    n = c.n
    off = c.row != c.col
    source = np.ones(n, bool)
    source[c.row[~off]] = False  # a source row has no diagonal entry
    at = np.arange(n, dtype=np.float64)
    s = source[c.row] & off
    at[c.row[s]] = c.col[s] + 0.5
    order = np.argsort(at, kind="stable")
    inv = np.empty(n, np.int64)
    inv[order] = np.arange(n)
    r, q = inv[c.row], inv[c.col]
    width = int(np.abs(r - q).max())
    cut = [0]
    while cut[-1] < n:
        e = min(n, cut[-1] + width)
        while e < n and source[order[e]]:
            e += 1
        cut.append(e)
    block = np.searchsorted(np.array(cut), np.arange(n), side="right") - 1
    by = np.argsort(block[r], kind="stable")
    start = np.searchsorted(block[r][by], np.arange(len(cut)))

    def tile(i, j):
        e = by[start[i]:start[i + 1]]
        e = e[block[q[e]] == j]
        m = np.zeros((cut[i + 1] - cut[i], cut[j + 1] - cut[j]))
        np.add.at(m, (r[e] - cut[i], q[e] - cut[j]), val[e])
        return m

    nb = len(cut) - 1
    gain, diag, lower = [], [], []
    for i in range(nb):
        d = tile(i, i)
        lower.append(tile(i, i - 1) if i else None)
        if i:
            d = d - lower[i] @ gain[i - 1]
        diag.append(d)
        gain.append(np.linalg.solve(d, tile(i, i + 1)) if i + 1 < nb else None)

    def solve(rhs):
        y = []
        for i in range(nb):
            t = rhs[cut[i]:cut[i + 1]]
            y.append(np.linalg.solve(diag[i], t - lower[i] @ y[i - 1] if i else t))
        for i in range(nb - 2, -1, -1):
            y[i] = y[i] - gain[i] @ y[i + 1]
        return np.concatenate(y)

    bp = b[order]
    x = solve(bp)
    x = x + solve(bp - np.bincount(r, val * x[q], n))
    out = np.empty(n)
    out[order] = x
    return out


def exact(case, seed):
    vals, rhs = _inputs(case, seed)
    out, a, v = [], 0, 0
    for c in _of(case):
        val, b = vals[a:a + c.nnz], rhs[v:v + c.n]
        a, v = a + c.nnz, v + c.n
        if case["call"] == "spmv":
            out.append(np.bincount(c.row, val * b[c.col], c.n))
        elif case["circuit"] in ("c1", "grid"):
            out.append(_banded(c, val, b))
        else:
            out.append(_dense(c.n, c.row, c.col, val, b))
    x = np.concatenate(out)
    # host calls answer with an array, device calls with a tensor: the same values either way
    return x if case["call"] == "newton_host" else torch.from_numpy(x)
