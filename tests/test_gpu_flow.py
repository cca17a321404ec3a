"""The flow schedule (rows in level order over all compute units, each waiting
for its own dependencies), which the tuner picks for wide levels.

x within relative 1e-10 of the oracle's substitution and a relative residual
below 1e-12, forward and backward, for rows of every class (1, 2, 4 entries
per lane, 1 .. 64 lanes per row, several rounds) and every column count of a
launch; the columns of a call agree bit for bit with single solves.
"""
import ctypes

import numpy as np
import pytest

from helpers import csc_from_deps, rel_err, residual
from rbsptrsv import gen

pytestmark = pytest.mark.gpu

X_TOL = 1e-10
RES_TOL = 1e-12


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a device"
    return torch


def _is_flow(p):
    # (the level schedule fits none of the factors this is asked of: more
    # rows than its ring, columns anywhere before the row)
    return p.info().schedule == 2 and p.trace() is None


def _classes(n, seed):
    """Four levels of n rows whose lengths run through every class of rows:
    level k reads n / 2 rows of level k - 1 in turn."""
    lens = [1, 2, 3, 4, 5, 8, 9, 16, 17, 33, 64, 65, 128, 129, 255, 256, 257, 700]
    deps = {}
    for k in range(1, 4):
        for i in range(n):
            L = min(lens[(i + k) % len(lens)], n)
            deps[k * n + i] = sorted({(k - 1) * n + (i * 7 + j * 3) % n for j in range(L)})
    return csc_from_deps(4 * n, deps, seed=seed, diag=50.0)


CASES = [
    ("powerlaw-60000", lambda: gen.powerlaw(60000, seed=5)),
    ("powerlaw-20001", lambda: gen.powerlaw(20001, seed=6)),
    ("random-40000", lambda: gen.random_lower(40000, 6, seed=7)),
    ("classes-1025", lambda: _classes(1025, 1)),
    ("classes-5000", lambda: _classes(5000, 2)),
]


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("name,make", CASES, ids=[c[0] for c in CASES])
def test_flow_solve_matches_oracle(oracle, torch, name, make, lower):
    from rbsptrsv import Plan
    f = make() if lower else make().transpose()
    p = Plan.from_factor(f)
    print("flow", name, lower, "picked" if _is_flow(p) else "other", flush=True)
    K = 9
    B = gen.rhs(f.n, seed=5, k=K)
    rp, ci, v = f.csr()
    single = []
    for j in range(K):
        x = p.solve(torch.as_tensor(B[:, j].copy(), device="cuda")).cpu().numpy()
        xo = oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j])
        assert rel_err(x, xo) < X_TOL
        assert residual(f, x, B[:, j]) < RES_TOL
        single.append(x)
    for k in (2, 3, 4, 5, 8, 9):
        X = p.solve(torch.as_tensor(np.ascontiguousarray(B[:, :k].T), device="cuda").t())
        for j in range(k):
            assert np.array_equal(X[:, j].cpu().numpy().view(np.int64), single[j].view(np.int64))
    p.check()
    p.close()


def test_flow_schedule_is_picked(torch):
    from rbsptrsv import Plan
    for f in (gen.powerlaw(60000, seed=5), gen.powerlaw(60000, seed=5).transpose()):
        p = Plan.from_factor(f)
        assert _is_flow(p)
        p.close()


def test_flow_overlap_and_noalloc(torch):
    """x over b (the same array, shifted by a few rows, shifted by a column),
    a leading dimension above n, and the allocation-free entry point: all
    equal to single solves bit for bit."""
    from rbsptrsv import Plan
    from rbsptrsv._lib import check, lib
    f = gen.powerlaw(60000, seed=5)
    n, k = f.n, 11
    p = Plan.from_factor(f)
    assert _is_flow(p)
    B = torch.as_tensor(np.ascontiguousarray(gen.rhs(n, seed=6, k=k).T), device="cuda")
    want = torch.stack([p.solve(B[j].contiguous()) for j in range(k)])
    pad = torch.zeros(k + 1, n + 13, dtype=torch.float64, device="cuda")
    pad[:k, :n] = B
    x = p.solve(pad.t()[:n, :k], x=pad.t()[:n, :k])          # in place
    assert torch.equal(x.t(), want)
    pad[:k, :n] = B
    x = p.solve(pad.t()[:n, :k], x=pad.t()[:n, 1:k + 1])     # a column further
    assert torch.equal(x.t(), want)
    for shift in (1, -3):
        buf = torch.zeros(n + 8, dtype=torch.float64, device="cuda")
        b, y = buf[4:4 + n], buf[4 + shift:4 + shift + n]
        b.copy_(B[0])
        p.solve(b, x=y)
        assert torch.equal(y, want[0]), shift
    y = torch.empty_like(B)
    for x in (y, B):
        check(lib().rb_solve_noalloc(p._h, ctypes.c_void_p(B.data_ptr()), n,
                                     ctypes.c_void_p(x.data_ptr()), n, k, None))
        assert torch.equal(x, want)
    p.check()
    p.close()


def test_flow_special_values(oracle, torch):
    """An infinite and a NaN right-hand side entry spread to the rows that
    depend on them and to no other."""
    from rbsptrsv import Plan
    f = gen.powerlaw(60000, seed=5)
    b = gen.rhs(f.n, seed=9)
    b[50000], b[55000] = np.inf, np.nan
    rp, ci, v = f.csr()
    xo = oracle.sptrsv_serial(rp, ci, v, f.n, 0, b)
    p = Plan.from_factor(f)
    assert _is_flow(p)
    x = p.solve(torch.as_tensor(b, device="cuda")).cpu().numpy()
    p.check()
    p.close()
    fine = np.isfinite(xo)
    assert np.array_equal(fine, np.isfinite(x)) and fine[:50000].all()
    assert rel_err(x[fine], xo[fine]) < X_TOL


def test_flow_captured_into_a_graph(torch):
    """Replays of a captured solve, with eager work in between, equal the
    eager solve bit for bit."""
    from rbsptrsv import Plan
    f = gen.powerlaw(60000, seed=5)
    p = Plan.from_factor(f)
    assert _is_flow(p)
    b = torch.as_tensor(gen.rhs(f.n, seed=3), device="cuda")
    x = torch.empty_like(b)
    want = p.solve(b).clone()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        p.solve(b, x=x, stream=st)
    for r in range(4):
        x.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, want), r
        assert torch.equal(p.solve(b), want)
    p.check()
    p.close()
