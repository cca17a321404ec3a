"""The work a user of this library has it do, as cases to be timed.

Every case is one triangular factor (or a batch of them) that a program keeps
as a plan, and one call on it: a solve, a solve of several right-hand sides,
an FP32 solve refined in FP64, a batch of uneven factors, or the whole way
from a new factor to its first solution.  The factors are the library's three
families (rbsptrsv.gen), made on the GPU from a seed:

  banded    n rows, 8 draws per row from the 2000 columns before it: deep,
            narrow level sets with irregular dependencies
  grid      lower part of a five-point operator with varying coefficients on
            nx x ny points in natural order: nx + ny - 1 level sets
  powerlaw  row lengths from Zipf(2) up to 512, columns anywhere before the
            row: few, wide level sets

each forward (lower factor) or backward (its transpose).
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "recblock-sptrsv_amd"))

from rbsptrsv import Batch, Plan  # noqa: E402

WINDOW, DRAWS, KMAX = 2000, 8, 512
TOL = 1e-12  # of the refined solves


def listed():
    return [
        # the smallest calls: a small factor inside an outer iteration, where
        # the launches are the time
        {"name": "small_banded_3000", "op": "solve", "family": "banded", "nx": 3000, "ny": 1,
         "lower": True, "rhs": 1},
        # a small grid's upper factor, odd and ragged sides
        {"name": "grid_333x217_back", "op": "solve", "family": "grid", "nx": 333, "ny": 217,
         "lower": False, "rhs": 1},
        # the three factors of the benchmark at their sizes, one right-hand
        # side per call as a preconditioner is applied
        {"name": "banded_100000", "op": "solve", "family": "banded", "nx": 100_000, "ny": 1,
         "lower": True, "rhs": 1},
        {"name": "grid_1500x1500", "op": "solve", "family": "grid", "nx": 1500, "ny": 1500,
         "lower": True, "rhs": 1},
        {"name": "powerlaw_4000000", "op": "solve", "family": "powerlaw", "nx": 4_000_000, "ny": 1,
         "lower": True, "rhs": 1},
        # block Krylov methods and serving: several right-hand sides per call
        {"name": "powerlaw_300001_back_rhs5", "op": "solve", "family": "powerlaw", "nx": 300_001,
         "ny": 1, "lower": False, "rhs": 5},
        {"name": "banded_100000_rhs32", "op": "solve", "family": "banded", "nx": 100_000, "ny": 1,
         "lower": True, "rhs": 32},
        {"name": "grid_1000x1000_rhs16", "op": "solve", "family": "grid", "nx": 1000, "ny": 1000,
         "lower": True, "rhs": 16},
        # FP32 solves refined in FP64
        {"name": "grid_1201x733_f32ir", "op": "f32ir", "family": "grid", "nx": 1201, "ny": 733,
         "lower": True, "rhs": 1},
        # many resident factors of uneven size, 1..32 right-hand sides each
        {"name": "batch_64_fp64", "op": "batch", "family": "banded", "nx": 200_000, "ny": 64,
         "lower": True, "rhs": 32},
        {"name": "batch_24_f32ir", "op": "batch_f32ir", "family": "banded", "nx": 80_000, "ny": 24,
         "lower": True, "rhs": 32},
        # a factor that changes every outer step: plan, one solve, gone
        {"name": "setup_grid_500x500", "op": "setup", "family": "grid", "nx": 500, "ny": 500,
         "lower": True, "rhs": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["solve", "solve", "solve", "multi", "multi", "f32ir", "batch",
                     "batch_f32ir", "setup"])
    case = {"op": op, "family": rng.choice(["banded", "grid", "powerlaw"]), "ny": 1,
            "lower": rng.random() < 0.6, "rhs": 1}
    hi = {"solve": 2_200_000, "multi": 300_000, "f32ir": 900_000, "setup": 250_000}.get(op, 0)
    if op.startswith("batch"):
        case.update(family="banded", nx=_log_int(rng, 3000, 100_000), ny=rng.randint(4, 40),
                    rhs=rng.randint(1, 32))
        return case
    if op == "multi":
        case.update(op="solve", rhs=_log_int(rng, 2, 32))
    if case["family"] == "grid":
        n = math.exp(rng.uniform(math.log(2000), math.log(hi)))
        nx = _log_int(rng, max(8, n ** 0.5 / 2), n ** 0.5 * 2)
        case.update(nx=nx, ny=max(8, int(n / nx)))
    else:
        # a banded factor of n rows is a chain of n / 100 level sets
        case["nx"] = _log_int(rng, 1000, min(hi, 300_000) if case["family"] == "banded" else hi)
    return case


# ------------------------------------------------------------------ factors

def _csc(rows, cols, vals, n):
    """(colptr, rowidx, val) of distinct entries, rows ascending per column."""
    order = torch.argsort(cols * n + rows)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=rows.device)
    ptr[1:] = torch.cumsum(torch.bincount(cols, minlength=n), 0)
    return ptr.int(), rows[order].int(), vals[order].contiguous()


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, dtype=torch.float64, device=g.device) * (hi - lo) + lo


def _factor(case, g, n=None):
    """Lower factor of the case's family (n: a batch member's size), or its
    transpose."""
    dev, family = g.device, case["family"]
    if family == "grid":
        nx, ny = case["nx"], case["ny"]
        n = nx * ny
        i = torch.arange(n, device=dev)
        west, south = i[i % nx != 0], i[i >= nx]
        rows = torch.cat([west, south])
        cols = torch.cat([west - 1, south - nx])
        off = -_uniform(g, rows.numel(), 0.5, 1.5)
        diag = _uniform(g, n, 3.2, 4.8)
    else:
        n = n or case["nx"]
        i = torch.arange(n, device=dev)
        if family == "banded":
            cnt = torch.full((n,), DRAWS, device=dev)
            cnt[0] = 0
            low = (i - WINDOW).clamp(min=0)
        else:
            k = torch.arange(1, KMAX, dtype=torch.float64, device=dev)
            cdf = torch.cumsum(6 / math.pi ** 2 / k ** 2, 0)
            cnt = torch.searchsorted(cdf, _uniform(g, n, 0.0, 1.0)) + 1
            cnt = torch.minimum(cnt, i)
            low = torch.zeros_like(i)
        r = torch.repeat_interleave(i, cnt)
        u = _uniform(g, r.numel(), 0.0, 1.0)
        c = low[r] + (u * (r - low[r])).long()
        key = torch.unique(r * n + c)
        rows, cols = key // n, key % n
        if family == "banded":
            off = _uniform(g, rows.numel(), -0.1, 0.1) / DRAWS
            diag = _uniform(g, n, 2.0, 3.0)
        else:
            off = _uniform(g, rows.numel(), -1.0, 1.0)
            diag = 1.0 + torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, rows, off.abs())
    rows, cols, vals = torch.cat([rows, i]), torch.cat([cols, i]), torch.cat([off, diag])
    return _csc(rows, cols, vals, n) if case["lower"] else _csc(cols, rows, vals, n)


def _rhs(g, n, k):
    b = _uniform(g, n * k, -1.0, 1.0)
    return b if k == 1 else b.view(k, n).t()  # column-major (n, k)


def _batch_sizes(case):
    """Rows and right-hand sides of a batch's factors: log-uniform up to nx,
    1..rhs, the same for every seed."""
    r = random.Random("%d %d %d" % (case["nx"], case["ny"], case["rhs"]))
    return [(_log_int(r, 1000, case["nx"]), r.randint(1, case["rhs"])) for _ in range(case["ny"])]


def _inputs(case, seed):
    """[(colptr, rowidx, val, b)]: one factor, or a batch's."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["op"].startswith("batch"):
        return [_factor(case, g, n) + (_rhs(g, n, k),) for n, k in _batch_sizes(case)]
    f = _factor(case, g)
    return [f + (_rhs(g, f[0].numel() - 1, case["rhs"]),)]


class _Member:
    """A factor of a batch, as rbsptrsv.Batch takes it."""

    def __init__(self, colptr, rowidx, val, substitution):
        self.colptr, self.rowidx, self.val = colptr, rowidx, val
        self.substitution = substitution


def prepare(case, seed):
    facs = _inputs(case, seed)
    op, subst = case["op"], 0 if case["lower"] else 1
    state = {"op": op, "subst": subst}
    if op.startswith("batch"):
        members = [_Member(cp, ri, v, subst) for cp, ri, v, _ in facs]
        state["bs"] = [b for _, _, _, b in facs]
        state["xs"] = [torch.empty_like(b) for b in state["bs"]]
        state["plan"] = Batch(members, mixed=op == "batch_f32ir", tune_rhs=case["rhs"])
    else:
        cp, ri, v, state["b"] = facs[0]
        if op == "setup":
            state["factor"] = (cp, ri, v)
            return state
        state["x"] = torch.empty_like(state["b"])
        state["plan"] = Plan(cp, ri, v, subst, mixed=op == "f32ir", tune_rhs=case["rhs"])
    return state


def run(state):
    op = state["op"]
    if op == "solve":
        return state["plan"].solve(state["b"], x=state["x"])
    if op == "f32ir":
        return state["plan"].solve_f32ir(state["b"], x=state["x"], tol=TOL)[0]
    if op == "batch":
        return state["plan"].solve(state["bs"], xs=state["xs"])
    if op == "batch_f32ir":
        return state["plan"].solve_f32ir(state["bs"], xs=state["xs"], tol=TOL)[0]
    cp, ri, v = state["factor"]
    plan = Plan(cp, ri, v, state["subst"])
    x = plan.solve(state["b"])
    plan.close()
    return x


def _entries(case, n):
    """Expected entries of a factor with n rows, the diagonal included."""
    if case["family"] == "grid":
        return 3 * n - case["nx"] - case["ny"]
    if case["family"] == "banded":
        return 9 * n
    zipf = sum(1 / k for k in range(1, KMAX)) * 6 / math.pi ** 2 + KMAX * 6 / math.pi ** 2 / (KMAX - 0.5)
    return int((1 + zipf) * n)


def work(case):
    """Matrix once (value, column, row pointer), b read and x written; two
    operations per entry and right-hand side."""
    if case["op"].startswith("batch"):
        sizes = _batch_sizes(case)
    else:
        sizes = [(case["nx"] * case["ny"], case["rhs"])]
    nbytes = sum(12 * _entries(case, n) + 4 * (n + 1) + 16 * n * k for n, k in sizes)
    flops = sum(2 * _entries(case, n) * k for n, k in sizes)
    return {"bytes": nbytes, "flops": flops}


# -------------------------------------------------------------------- exact

def _substitute(colptr, rowidx, val, b):
    """x of the triangular system by substitution, one level set at a time,
    in 64 bits."""
    n, dev = colptr.numel() - 1, b.device
    ptr, rows = colptr.long(), rowidx.long()
    cols = torch.repeat_interleave(torch.arange(n, device=dev), ptr[1:] - ptr[:-1])
    diag = torch.empty(n, dtype=torch.float64, device=dev)
    on = rows == cols
    diag[rows[on]] = val[on]
    rows, vals = rows[~on], val[~on]
    cnt = torch.bincount(cols[~on], minlength=n)
    start = torch.cumsum(cnt, 0) - cnt
    rem = torch.bincount(rows, minlength=n)
    acc = b.clone().reshape(n, -1)
    x = torch.empty_like(acc)
    front = torch.nonzero(rem == 0).flatten()
    while front.numel():
        x[front] = acc[front] / diag[front, None]
        c = cnt[front]
        u = torch.repeat_interleave(front, c)
        e = torch.arange(u.numel(), device=dev) - torch.repeat_interleave(torch.cumsum(c, 0) - c, c) + start[u]
        v = rows[e]
        acc.index_add_(0, v, -vals[e, None] * x[u])
        rem.index_add_(0, v, torch.full_like(v, -1))
        v = torch.unique(v)
        front = v[rem[v] == 0]
    return x.reshape(b.shape)


def exact(case, seed):
    xs = [_substitute(*f) for f in _inputs(case, seed)]
    return xs if case["op"].startswith("batch") else xs[0]
