"""The work that users of this framework have it do, as cases whose time can be measured.

Three kinds of call, over the sizes of the repository's own benchmark and tests:

* ``solve``: one LP, ``cuOptSolve`` through ``cuopt_amd.c_api`` on a problem and settings that the program
  keeps, to a tolerance (as users ask for it) or for a fixed budget of iterations;
* ``batch``: many uneven LPs, ``cuOptAmdBatchSolve``;
* ``unrolled``: the differentiable map ``cuopt_amd.autograd.UnrolledPDHG``, forward alone (inference) or with
  its backward pass (training).

LPs come from the families of ``cuopt_amd/generators.py``, drawn on the GPU so that inputs are quick to make.
"""

import math

import numpy as np
import torch

from cuopt_amd import c_api
from cuopt_amd.autograd import UnrolledPDHG
from cuopt_amd.generators import LP

INF = float("inf")


def listed():
    return [
        # A planning or teaching model of some dozens of rows, solved on demand with the default presolve:
        # launches, allocations and host work count, not arithmetic.
        _solve("solve_tiny_fp64", "random", 50, 125, "fp64", 1e-4, presolve=True),
        # The benchmark's small LP in the reference's arithmetic, to the usual tolerance.
        _solve("solve_2k_fp64", "random", 2000, 5000, "fp64", 1e-4),
        # The same LP in FP32-mixed refined to an accurate solution.
        _solve("solve_2k_fp32_accurate", "random", 2000, 5000, "fp32_mixed", 1e-8),
        # Transportation: 20 000 sources, 50 000 sinks, 50 arcs a source (1 M variables), accurate.
        _solve("transport_fp32_accurate", "transport", 70_000, 1_000_000, "fp32_mixed", 1e-8),
        # The headline workload: Zipf rows, up to half a million nonzeros in one, in both precisions.
        _solve("skewed_fp32", "skewed", 500_000, 1_000_000, "fp32_mixed", 1e-4),
        _solve("skewed_fp64", "skewed", 500_000, 1_000_000, "fp64", 1e-4),
        # A long banded (multi-period) model under a fixed budget of iterations, 16 M nonzeros.
        _solve("banded_fp32_budget", "banded", 1_000_000, 2_000_000, "fp32_mixed", 1e-8, iterations=400),
        # Scenario batches of uneven LPs, 50 to 2 000 rows.
        _batch("batch_fp32", 1024, 50, 2000, "fp32_mixed", 1e-4),
        _batch("batch_fp64", 512, 50, 2000, "fp64", 1e-4),
        # Training through the solver: the benchmark's shape, loss and gradients of 500 steps.
        _unrolled("unrolled_train_fp32", 20_000, 50_000, 64, 500, "fp32_mixed", True),
        # A double-precision training step with a ragged batch.
        _unrolled("unrolled_train_fp64", 5000, 12_500, 24, 200, "fp64", True),
        # Inference of a small layer for a few objectives.
        _unrolled("unrolled_infer_fp32", 2000, 5000, 16, 200, "fp32_mixed", False),
    ]


def _solve(name, family, m, n, precision, tol, iterations=0, presolve=False):
    return {"name": name, "kind": "solve", "family": family, "m": m, "n": n, "precision": precision, "tol": tol,
            "iterations": iterations, "presolve": presolve}


def _batch(name, count, m_min, m_max, precision, tol):
    return {"name": name, "kind": "batch", "count": count, "m_min": m_min, "m_max": m_max, "precision": precision,
            "tol": tol}


def _unrolled(name, m, n, batch, steps, precision, train):
    return {"name": name, "kind": "unrolled", "m": m, "n": n, "batch": batch, "steps": steps, "precision": precision,
            "train": train}


def _between(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    precision = rng.choice(["fp64", "fp32_mixed"])
    kind = rng.choice(["random", "random", "skewed", "transport", "banded", "batch", "batch", "unrolled", "unrolled",
                       "unrolled"])
    if kind == "random":
        m = _between(rng, 50, 20_000)
        case = _solve("", kind, m, int(2.5 * m), precision, rng.choice([1e-4, 1e-8]), presolve=rng.random() < 0.25)
    elif kind == "skewed":
        m = _between(rng, 20_000, 400_000)
        case = _solve("", kind, m, 2 * m, precision, 1e-4)
    elif kind == "transport":
        sources = _between(rng, 1000, 15_000)
        case = _solve("", kind, sources + int(2.5 * sources), 50 * sources, precision, 1e-4)
    elif kind == "banded":
        m = _between(rng, 50_000, 800_000)
        case = _solve("", kind, m, 2 * m, precision, 1e-8, iterations=rng.choice([100, 200, 400]))
    elif kind == "batch":
        m_max = _between(rng, 200, 2000)
        case = _batch("", _between(rng, 16, 500), 50, m_max, precision, 1e-4)
    else:
        m = _between(rng, 500, 20_000)
        case = _unrolled("", m, int(2.5 * m), _between(rng, 1, 64), rng.randrange(100, 301), precision,
                         rng.random() < 0.6)
    del case["name"]
    return case


# ---- inputs -----------------------------------------------------------------------------------------------------


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rng(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed) & 0x7FFFFFFF), np.random.default_rng(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=_device(), dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=_device(), dtype=torch.float64)


def _csr(rows, vals, m):
    """CSR of entries that come in column order: (row pointers, the entries' order by row) as numpy and torch."""
    order = torch.sort(rows, stable=True)[1]
    ptr = np.zeros(m + 1, np.int64)
    np.cumsum(torch.bincount(rows, minlength=m).cpu().numpy(), out=ptr[1:])
    return ptr, order, vals[order].cpu().numpy()


def _random_lps(ms, seed, upper=10.0, k=8):
    """Random equality LPs of ms[i] rows and 2.5 ms[i] columns, k nonzeros a column at distinct rows, with a
    built-in optimal pair (the law of generators.random_lp); all drawn together."""
    g, rng = _rng(seed)
    ms = np.asarray(ms, np.int64)
    ns = (2.5 * ms).astype(np.int64)
    m0, n0 = np.concatenate([[0], np.cumsum(ms)]), np.concatenate([[0], np.cumsum(ns)])
    M, N = int(m0[-1]), int(n0[-1])
    of_col = torch.from_numpy(np.repeat(np.arange(len(ms)), ns)).to(_device())
    height = torch.from_numpy(ms).to(_device())[of_col].double()[:, None]
    rows = (_rand(g, N, k) * height).long()
    while True:
        s = torch.sort(rows, dim=1)[0]
        dup = (s[:, 1:] == s[:, :-1]).any(dim=1)
        if not bool(dup.any()):
            break
        rows = torch.where(dup[:, None], (_rand(g, N, k) * height).long(), rows)
    rows = (rows + torch.from_numpy(m0[:-1]).to(_device())[of_col][:, None]).reshape(-1)
    first = torch.from_numpy(n0[:-1]).to(_device())[of_col]
    cols = (torch.arange(N, device=_device()) - first).repeat_interleave(k)  # within the LP
    ptr, order, val = _csr(rows, _randn(g, N * k), M)
    idx = cols[order].int().cpu().numpy()
    row_of = np.repeat(np.arange(M), np.diff(ptr))
    col_of = idx + n0[:-1][np.repeat(np.arange(len(ms)), ms)][row_of]
    x = np.where(rng.random(N) < 0.6, rng.random(N), 0.0)
    y = rng.standard_normal(M)
    b = np.bincount(row_of, weights=val * x[col_of], minlength=M)
    c = np.bincount(col_of, weights=val * y[row_of], minlength=N) + np.where(x == 0.0, rng.random(N), 0.0)
    lps = []
    for i in range(len(ms)):
        r, q, z = slice(m0[i], m0[i + 1]), slice(n0[i], n0[i + 1]), slice(ptr[m0[i]], ptr[m0[i + 1]])
        lps.append(LP(m=int(ms[i]), n=int(ns[i]), row_offsets=(ptr[m0[i]:m0[i + 1] + 1] - ptr[m0[i]]).astype(np.int32),
                      col_indices=idx[z], values=val[z], c=c[q], con_lb=b[r], con_ub=b[r].copy(),
                      var_lb=np.zeros(ns[i]), var_ub=np.full(ns[i], upper)))
    return lps


def _batch_lps(case, seed):
    """Sizes by the log-uniform law, in mixed order, the same for every seed."""
    at = (np.random.RandomState(0).permutation(case["count"]) + 0.5) / case["count"]
    return _random_lps((case["m_min"] * (case["m_max"] / case["m_min"]) ** at).astype(np.int64), seed)


def _skewed_lp(m, n, seed):
    """Rows by a truncated Zipf law (exponent 1.1), 1 + Poisson(4) entries a column, half = and half <= rows, with
    a built-in optimal pair (the law of generators.skewed_lp)."""
    g, rng = _rng(seed)
    per = 1 + torch.poisson(torch.full((n,), 4.0, device=_device(), dtype=torch.float64), generator=g).long()
    cols = torch.arange(n, device=_device()).repeat_interleave(per)
    cdf = np.cumsum(np.arange(1, m + 1, dtype=np.float64) ** -1.1)
    rows = torch.searchsorted(torch.from_numpy(cdf / cdf[-1]).to(_device()), _rand(g, cols.numel()), right=True)
    key = torch.unique(cols * m + rows.clamp_(max=m - 1))  # one entry per place, in column order
    cols, rows = key // m, key % m
    ptr, order, val = _csr(rows, _randn(g, key.numel()), m)
    idx = cols[order].int().cpu().numpy()
    row_of = np.repeat(np.arange(m), np.diff(ptr))
    x = np.where(rng.random(n) < 0.6, rng.random(n), 0.0)
    y = rng.standard_normal(m)
    y[m // 2:] = 0.0
    b = np.bincount(row_of, weights=val * x[idx], minlength=m)
    c = np.bincount(idx, weights=val * y[row_of], minlength=n) + np.where(x == 0.0, rng.random(n), 0.0)
    ub = b + np.where(np.arange(m) < m // 2, 0.0, rng.random(m))
    lb = np.where(np.arange(m) < m // 2, b, -INF)
    return LP(m=m, n=n, row_offsets=ptr.astype(np.int32), col_indices=idx, values=val, c=c, con_lb=lb, con_ub=ub,
              var_lb=np.zeros(n), var_ub=rng.uniform(1.0, 100.0, n))


def _transport_lp(m, n, seed, arcs=50):
    """`arcs` arcs a source to random sinks (every sink has one), supply rows <=, demand rows =, as
    generators.transportation_lp with demands by the number of arcs and half as much supply again, so that every
    draw is feasible."""
    g, rng = _rng(seed)
    sources = n // arcs
    sinks = m - sources
    dest = (_rand(g, sources, arcs) * sinks).long()
    dest = dest.sort(dim=1)[0]
    for _ in range(8):  # distinct sinks for all but a few sources
        dup = (dest[:, 1:] == dest[:, :-1]).any(dim=1)
        dest = torch.where(dup[:, None], (_rand(g, sources, arcs) * sinks).long().sort(dim=1)[0], dest)
    dest = dest.reshape(-1).cpu().numpy()
    missing = np.flatnonzero(np.bincount(dest, minlength=sinks) == 0)
    dest[rng.permutation(n)[: missing.size]] = missing
    row = torch.from_numpy(np.stack([np.repeat(np.arange(sources), arcs), sources + dest], axis=1).reshape(-1)).to(_device())
    ptr, order, val = _csr(row, torch.ones(2 * n, device=_device(), dtype=torch.float64), m)
    idx = (order // 2).int().cpu().numpy()
    supply = rng.uniform(10.0, 100.0, sources)
    into = np.bincount(dest, minlength=sinks)
    demand = into * rng.uniform(0.5, 1.5, sinks)
    demand *= supply.sum() / (1.5 * demand.sum())
    return LP(m=m, n=n, row_offsets=ptr.astype(np.int32), col_indices=idx, values=val,
              c=rng.integers(1, 101, n).astype(np.float64), con_lb=np.concatenate([np.full(sources, -INF), demand]),
              con_ub=np.concatenate([supply, demand]), var_lb=np.zeros(n), var_ub=np.full(n, INF))


def _banded_lp(m, n, seed, width=16):
    """Equality LP whose row i has `width` neighbouring columns around 2 i (the law of generators.banded_lp)."""
    g, _ = _rng(seed)
    d = torch.arange(-(width // 2), width - width // 2, device=_device())
    cols = ((2 * torch.arange(m, device=_device())[:, None] + d[None, :]) % n).sort(dim=1)[0]
    val = _randn(g, m, width)
    b = (val * _rand(g, n)[cols]).sum(dim=1).cpu().numpy()
    return LP(m=m, n=n, row_offsets=np.arange(0, (m + 1) * width, width, dtype=np.int64).astype(np.int32),
              col_indices=cols.int().reshape(-1).cpu().numpy(), values=val.reshape(-1).cpu().numpy(),
              c=_randn(g, n).cpu().numpy(), con_lb=b, con_ub=b.copy(), var_lb=np.zeros(n), var_ub=np.full(n, 10.0))


def _one_lp(case, seed):
    family, m, n = case["family"], case["m"], case["n"]
    if family == "random":
        return _random_lps([m], seed)[0]
    return {"skewed": _skewed_lp, "transport": _transport_lp, "banded": _banded_lp}[family](m, n, seed)


def _unrolled_inputs(case, seed):
    """The LP, and the tensors that a layer in front of the solver hands over: one objective a batch member, the
    right-hand side, and the training target, in the precision of the model."""
    lp = _random_lps([case["m"]], seed)[0]
    g, _ = _rng(seed + 1)
    dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
    c = torch.from_numpy(lp.c).to(_device()) + 0.1 * _randn(g, case["batch"], lp.n)
    b = torch.from_numpy(lp.con_lb).to(_device())
    return lp, c.to(dtype), b.to(dtype), _rand(g, case["batch"], lp.n).to(dtype)


RIDGE, EVERY = 1e-3, 45


def prepare(case, seed):
    if case["kind"] == "unrolled":
        lp, c, b, target = _unrolled_inputs(case, seed)
        op = UnrolledPDHG(lp, ridge=RIDGE, steps=case["steps"], checkpoint_every=EVERY, precision=case["precision"])
        train = case["train"]
        return {"kind": "unrolled", "op": op, "c": c.requires_grad_(train), "b": b.requires_grad_(train),
                "target": target, "train": train}
    if case["kind"] == "batch":
        return {"kind": "batch", "problems": [c_api.Problem(lp) for lp in _batch_lps(case, seed)], "tol": case["tol"],
                "precision": case["precision"]}
    problem = c_api.Problem(_one_lp(case, seed))
    settings = c_api.make_settings(tol=case["tol"], precision=case["precision"],
                                   iteration_limit=case["iterations"] or None, presolve=case["presolve"])
    return {"kind": "solve", "problem": problem, "settings": settings}


# ---- the pass ---------------------------------------------------------------------------------------------------


def run(state):
    if state["kind"] == "solve":
        r = c_api.solve_problem(state["problem"], state["settings"])
        return {"x": r.x, "y": r.y, "z": r.reduced_cost, "objectives": np.array([r.primal_objective, r.dual_objective]),
                "status": r.status, "iterations": r.iterations}
    if state["kind"] == "batch":
        rs = c_api.batch_solve(state["problems"], tol=state["tol"], precision=state["precision"])
        return {"x": np.concatenate([r.x for r in rs]), "y": np.concatenate([r.y for r in rs]),
                "z": np.concatenate([r.reduced_cost for r in rs]),
                "objectives": np.array([[r.primal_objective, r.dual_objective] for r in rs]),
                "status": np.array([r.status for r in rs]), "iterations": np.array([r.iterations for r in rs])}
    op, c, b = state["op"], state["c"], state["b"]
    if not state["train"]:
        with torch.no_grad():
            x, y = op(c, b)
        return {"x": x, "y": y}
    x, y = op(c, b)
    loss = ((x - state["target"]) ** 2).sum()
    gc, gb = torch.autograd.grad(loss, [c, b])
    return {"x": x.detach(), "y": y.detach(), "gc": gc, "gb": gb}


# ---- what a pass cannot do without ------------------------------------------------------------------------------

#: Entries a column of each family, and iterations that its LPs typically take, by tolerance.
_ENTRIES = {"random": 8, "skewed": 4.75, "transport": 2, "banded": 8}
_ITERATIONS = {("random", 1e-4): 650, ("random", 1e-8): 2200, ("skewed", 1e-4): 1000, ("transport", 1e-4): 800,
               ("transport", 1e-8): 3100}


def _iteration(m, n, nnz, sv):
    """Bytes and operations of one PDHG iteration: both products and the vectors they update."""
    return 2 * nnz * (sv + 4) + 4 * (m + n + 2) + sv * (8 * n + 6 * m), 4.0 * nnz + 12.0 * (m + n)


def work(case):
    sv = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "unrolled":
        m, n, B = case["m"], case["n"], case["batch"]
        nnz = 8 * n
        step = 2 * nnz * (4 + sv) + 4 * (m + n + 2) + sv * (2 * (m + n) + B * (6 * n + 4 * m))
        flops = 4.0 * nnz * B
        times = 3 if case["train"] else 1  # forward, and for the gradients the states again and their adjoints
        return {"bytes": times * case["steps"] * step, "flops": times * case["steps"] * flops}
    if case["kind"] == "batch":
        lo, hi = case["m_min"], case["m_max"]
        m = (hi - lo) / math.log(hi / lo)  # mean of the log-uniform law
        b, f = _iteration(m, 2.5 * m, 20 * m, sv)
        k = case["count"] * _ITERATIONS["random", case["tol"]]
        return {"bytes": k * b, "flops": k * f}
    m, n = case["m"], case["n"]
    b, f = _iteration(m, n, _ENTRIES[case["family"]] * n, sv)
    k = case["iterations"] or _ITERATIONS[case["family"], case["tol"]]
    return {"bytes": k * b, "flops": k * f}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------


def exact(case, seed):
    if case["kind"] == "unrolled":
        return _exact_unrolled(case, seed)
    # A run in 24 bits stops at a check of its own, and one that presolve has changed follows another path.
    if case["kind"] != "solve" or case["presolve"] or (case["precision"] != "fp64" and not case["iterations"]):
        return None
    x, y, z, objectives = _stable3(_one_lp(case, seed), case["tol"], case["iterations"] or 10 ** 9)
    return {"x": x, "y": y, "z": z, "objectives": objectives, "status": None, "iterations": None}


def _matrices(lp):
    dev = _device()
    rows = torch.from_numpy(np.repeat(np.arange(lp.m), np.diff(lp.row_offsets))).to(dev)
    cols = torch.from_numpy(lp.col_indices).to(dev).long()
    vals = torch.from_numpy(lp.values).to(dev)
    order = torch.sort(cols, stable=True)[1]
    tptr = torch.zeros(lp.n + 1, dtype=torch.long, device=dev)
    tptr[1:] = torch.cumsum(torch.bincount(cols, minlength=lp.n), 0)
    ptr = torch.from_numpy(lp.row_offsets).to(dev).long()

    def both(v):
        return (torch.sparse_csr_tensor(ptr, cols, v, size=(lp.m, lp.n)),
                torch.sparse_csr_tensor(tptr, rows[order], v[order], size=(lp.n, lp.m)))

    return rows, cols, vals, both


def _start_vector(m):
    """m standard normals by Marsaglia's polar method on a Mersenne twister with seed 1."""
    words = np.frombuffer(np.random.RandomState(1).bytes(4 * (8 * m + 4096)), "<u4").astype(np.float64)
    u = np.minimum((words[0::2] + words[1::2] * 2.0 ** 32) / 2.0 ** 64, 1.0 - 2.0 ** -53)
    a, b = 2.0 * u[0::2] - 1.0, 2.0 * u[1::2] - 1.0
    r = a * a + b * b
    ok = (r <= 1.0) & (r != 0.0)
    a, b, r = a[ok], b[ok], r[ok]
    f = np.sqrt(-2.0 * np.log(r) / r)
    return np.stack([b * f, a * f], axis=1).reshape(-1)[:m]


def _stable3(lp, tol, limit):
    """Reflected restarted Halpern PDHG (restarts and primal weight of cuPDLPx), from zero, to `tol` on the
    original problem or for `limit` iterations: the point at its last check."""
    dev = _device()
    rows, cols, vals, both = _matrices(lp)
    A, AT = both(vals)
    t = lambda v: torch.from_numpy(v).to(dev)  # noqa: E731
    c, lb, ub, lc, uc = t(lp.c), t(lp.var_lb), t(lp.var_ub), t(lp.con_lb), t(lp.con_ub)
    dr, dc = torch.ones(lp.m, dtype=torch.float64, device=dev), torch.ones(lp.n, dtype=torch.float64, device=dev)
    for sweep in range(11):
        a = (vals * dr[rows] * dc[cols]).abs()
        if sweep < 10:
            rv = torch.zeros_like(dr).scatter_reduce(0, rows, a, "amax", include_self=True)
            cv = torch.zeros_like(dc).scatter_reduce(0, cols, a, "amax", include_self=True)
        else:
            S, ST = both(a)
            rv, cv = S @ torch.ones_like(dc), ST @ torch.ones_like(dr)
        dr = torch.where(rv > 0, dr / rv.clamp(min=1e-300).sqrt(), dr)
        dc = torch.where(cv > 0, dc / cv.clamp(min=1e-300).sqrt(), dc)
    S, ST = both(vals * dr[rows] * dc[cols])

    def bound_norm(lo, up):
        sq = lambda v, keep: torch.where(keep & v.isfinite(), v * v, torch.zeros_like(v)).sum()  # noqa: E731
        return float((sq(lo, lo != up) + sq(up, up == up)).sqrt())

    b_norm, c_norm = bound_norm(lc, uc), float(c.norm())
    beta, gamma = 1.0 / (bound_norm(lc * dr, uc * dr) + 1.0), 1.0 / (float((c * dc).norm()) + 1.0)
    cs, l, u, sl, su = c * dc * gamma, lb / dc * beta, ub / dc * beta, lc * dr * beta, uc * dr * beta
    q = t(_start_vector(lp.m))
    for _ in range(5000):  # sigma_max squared
        q = q / q.norm()
        w = S @ (ST @ q)
        s2 = q.dot(w)
        done = float((w - s2 * q).norm()) < 1e-4
        q = w
        if done:
            break
    eta = 0.998 / math.sqrt(float(s2))
    omega = best_omega = 1.0
    x = torch.zeros_like(cs).clamp(l, u)
    x0, xh, sk = torch.zeros_like(cs), torch.zeros_like(cs), torch.zeros_like(cs)
    y = torch.zeros_like(sl)
    y0, yh = y.clone(), y.clone()
    trial, best_gap, err_sum = INF, INF, 0.0
    fpe = fpe0 = math.nan
    after_restart = periodic = None  # terms of the fixed-point error since the last check
    k = kr = 0
    restart = False

    def every(k):  # iterations between checks at k
        s = 10
        while k >= 100 * s:
            s *= 10
        return s

    def error(terms):
        ny, inter, nx = (float(v) for v in terms)
        return math.sqrt(nx * omega + ny / omega + 2.0 * inter * eta)

    def finite(v):
        return torch.where(v.isfinite(), v, torch.zeros_like(v))

    while True:
        if k % 200 == 0 or k % every(k) == 0:
            xo, yo, zo = xh * dc / beta, yh * dr / gamma, sk / dc / gamma
            ax, r = A @ xo, c - AT @ yo
            l2p, l2d = float((ax - torch.maximum(lc, torch.minimum(ax, uc))).norm()), float((r - zo).norm())
            po = float(xo.dot(c))
            do = float(zo.dot(xo) + (yo.clamp(min=0) * finite(lc) + yo.clamp(max=0) * finite(uc)).sum())
            gap, size = abs(po - do), abs(po) + abs(do)
            if after_restart is not None:
                fpe = fpe0 = error(after_restart)
            if periodic is not None:
                fpe = error(periodic)
            after_restart = periodic = None
            good = l2d <= tol * (1 + c_norm) and l2p <= tol * (1 + b_norm) and gap <= tol * (1 + size)
            if (k > 1 and good) or k >= limit:
                return xo, yo, zo, np.array([po, do])
            restart = False
            if k > 0 and k % 200 == 0:
                restart = k == 200 or fpe <= 0.2 * fpe0 or (fpe <= 0.8 * fpe0 and fpe > trial) or kr >= 0.36 * k
                trial = fpe
            if restart:
                px, py = float((x0 - xh).norm()), float((y0 - yh).norm())
                rel = (l2d / (1 + c_norm)) / (l2p / (1 + b_norm)) if l2p else INF
                if min(px, py) > 1e-16 and max(px, py) < 1e12 and 1e-8 < rel < 1e8:
                    err = math.log(py) - math.log(px) - math.log(omega)
                    err_sum = 0.3 * err_sum + err
                    omega *= math.exp(0.99 * err + 0.01 * err_sum)
                else:
                    omega, err_sum = best_omega, 0.0
                if abs(math.log10(rel)) < best_gap:
                    best_gap, best_omega = abs(math.log10(rel)), omega
                x, x0, y, y0 = xh, xh, yh, yh
                kr, trial = 0, INF
        tau, sigma, w = eta / omega, eta * omega, (kr + 1.0) / (kr + 2.0)
        aty = ST @ y
        moved = x - tau * (cs - aty)
        xp = torch.maximum(torch.minimum(moved, u), l)
        xb = 2.0 * xp - x
        v = y / sigma - S @ xb
        yp = (v - torch.maximum(-su, torch.minimum(v, -sl))) * sigma
        yb = 2.0 * yp - y
        if restart or (k + 1) % 200 == 0:
            terms = ((yb - y) ** 2).sum(), (ST @ yb - aty).dot(xb - x), ((xb - x) ** 2).sum()
            after_restart, periodic = (terms, periodic) if restart else (after_restart, terms)
        restart = False
        k, kr = k + 1, kr + 1
        if k % 200 == 0 or (k + 1) % every(k + 1) == 0:  # the point that the next check looks at
            xh, yh, sk = xp, yp, (xp - moved) / tau
        x, y = w * xb + (1.0 - w) * x0, w * yb + (1.0 - w) * y0


def _exact_unrolled(case, seed):
    lp, c, b, target = _unrolled_inputs(case, seed)
    _, _, vals, both = _matrices(lp)
    A, AT = both(vals)
    c, b, target = c.double().t(), b.double()[:, None], target.double().t()
    q = 1.0 + 0.5 * torch.sin(0.7 * torch.arange(lp.m, device=_device(), dtype=torch.float64) + 0.3)
    s2 = 0.0
    for it in range(2000):  # sigma_max squared
        q = A @ (AT @ (q / q.norm()))
        before, s2 = s2, float(q.norm())
        if it > 10 and abs(s2 - before) <= 1e-10 * s2:
            break
    eta = 0.998 / math.sqrt(s2)
    prox = 1.0 / (1.0 + eta * RIDGE)
    lo = torch.from_numpy(lp.var_lb).to(_device())[:, None]
    up = torch.from_numpy(lp.var_ub).to(_device())[:, None]
    x = torch.zeros_like(c).clamp(lo, up)
    y = torch.zeros(lp.m, c.shape[1], dtype=torch.float64, device=_device())
    inside = []
    for _ in range(case["steps"]):
        xp = torch.maximum(torch.minimum((x - eta * (c - AT @ y)) * prox, up), lo)
        y = y - eta * (A @ (2.0 * xp - x) - b)
        x = xp
        if case["train"]:
            inside.append((xp > lo) & (xp < up))
    if not case["train"]:
        return {"x": x.t(), "y": y.t()}
    ax, ay, gc, gb = 2.0 * (x - target), torch.zeros_like(y), torch.zeros_like(c), torch.zeros_like(y)
    for free in reversed(inside):
        gb += eta * ay
        gxb = -eta * (AT @ ay)
        gw = torch.where(free, (ax + 2.0 * gxb) * prox, torch.zeros_like(ax))
        gc -= eta * gw
        ax = gw - gxb
        ay = ay + eta * (A @ gw)
    return {"x": x.t(), "y": y.t(), "gc": gc.t(), "gb": gb.sum(dim=1)}
