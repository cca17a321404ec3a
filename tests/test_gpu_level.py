"""The level schedule (one workgroup per part and column, x in an LDS ring),
which the tuner picks for deep, narrow factors.

x within relative 1e-10 of the oracle's substitution and a relative residual
below 1e-12 at the edges of its tiles: 64-lane steps, several lanes per row
(more than 8 entries), blocks of 256 rows through rings of 1024 rows and
more, storage in the caller's order and in solve order.  Columns of one call
agree bit for bit with single solves.
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


def _early(n, far):
    """A chain of n rows whose every 100th row also reads a row without
    dependencies `far` rows back, with rows nobody reads in between."""
    deps = {}
    for i in range(1, n):
        if i % 7 == 3 or i % 100 == 50:
            continue  # no dependencies
        deps[i] = [i - 1 if (i - 1) % 7 != 3 and (i - 1) % 100 != 50 else i - 2]
        if i % 100 == 0 and i >= far + 50:
            deps[i].append(i // 100 * 100 - far + 50)
        deps[i] = sorted({c for c in deps[i] if 0 <= c < i})
    return csc_from_deps(n, deps, seed=3)


def _one_long(n, length):
    """A band with one row of `length` entries."""
    deps = {i: sorted({max(0, i - 1), max(0, i - 5), max(0, i - 60)}) for i in range(1, n)}
    deps[n - 1] = list(range(n - 1 - length, n - 1))
    return csc_from_deps(n, deps, seed=4)


CASES = [("banded%d" % n, lambda n=n: gen.banded(n, seed=n, window=w), w)
         for n, w in [(1, 5), (2, 5), (63, 20), (64, 20), (65, 20), (255, 100), (256, 100),
                      (257, 100), (1024, 300), (1025, 300), (5000, 300), (17001, 900),
                      (17001, 2000)]]
CASES = [(name + "w%d" % w, make) for name, make, w in CASES] + [
    ("long-rows", lambda: gen.random_lower(3000, 40, seed=1)),
    ("long-rows-window", lambda: gen.random_lower(9000, 20, seed=2, window=150)),
    ("powerlaw", lambda: gen.powerlaw(6000, seed=3)),
    ("row-512", lambda: _one_long(2000, 512)),
    ("row-513", lambda: _one_long(2000, 513)),
    ("early-rows", lambda: _early(9000, 1500)),
    ("strip", lambda: gen.laplacian(37, 300)),
    ("strip-wide", lambda: gen.laplacian(300, 37)),
    ("diagonal", lambda: csc_from_deps(700, {})),
]


def _is_level(p):
    return p.info().schedule == 2 and p.trace() is None


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("name,make", CASES, ids=[c[0] for c in CASES])
def test_level_solve_matches_oracle(oracle, torch, name, make, lower):
    from rbsptrsv import Plan
    f = make() if lower else make().transpose()
    p = Plan.from_factor(f)
    print("level", name, lower, "picked" if _is_level(p) else "other", flush=True)
    k = 3
    B = gen.rhs(f.n, seed=5, k=k)
    rp, ci, v = f.csr()
    X = p.solve(torch.as_tensor(np.ascontiguousarray(B.T), device="cuda").t())
    for j in range(k):
        xo = oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j])
        x = X[:, j].cpu().numpy()
        assert rel_err(x, xo) < X_TOL
        assert residual(f, x, B[:, j]) < RES_TOL
        x1 = p.solve(torch.as_tensor(B[:, j].copy(), device="cuda")).cpu().numpy()
        assert np.array_equal(x.view(np.int64), x1.view(np.int64))
    p.check()
    p.close()


def test_level_schedule_is_picked(torch):
    from rbsptrsv import Plan
    for f in (gen.banded(20000, seed=4), gen.banded(20000, seed=4).transpose(),
              gen.powerlaw(6000, seed=3)):
        p = Plan.from_factor(f)
        assert _is_level(p)
        p.close()


@pytest.mark.parametrize("make", [lambda: gen.banded(9000, seed=2),
                                  lambda: gen.banded(30000, seed=2).transpose()],
                         ids=["caller-order", "solve-order"])
def test_level_columns_overlap_and_noalloc(torch, make):
    """40 columns, x over b (the same array, and shifted by a few rows), a
    leading dimension above n, and the allocation-free entry point: all equal
    to single solves bit for bit."""
    from rbsptrsv import Plan
    from rbsptrsv._lib import check, lib
    f = make()
    n, k = f.n, 40
    p = Plan.from_factor(f)
    assert _is_level(p)
    B = torch.as_tensor(np.ascontiguousarray(gen.rhs(n, seed=6, k=k).T), device="cuda")
    want = torch.stack([p.solve(B[j].contiguous()) for j in range(k)])
    assert torch.equal(p.solve(B.t()).t(), want)
    pad = torch.zeros(k, n + 13, dtype=torch.float64, device="cuda")
    pad[:, :n] = B
    x = p.solve(pad.t()[:n], x=pad.t()[:n])          # in place
    assert torch.equal(x.t(), want)
    for shift in (1, -3):
        buf = torch.zeros(n + 8, dtype=torch.float64, device="cuda")
        b, y = buf[4:4 + n], buf[4 + shift:4 + shift + n]
        b.copy_(B[0])
        p.solve(b, x=y)
        assert torch.equal(y, want[0]), shift
    y = torch.empty_like(B)
    check(lib().rb_solve_noalloc(p._h, ctypes.c_void_p(B.data_ptr()), n,
                                 ctypes.c_void_p(y.data_ptr()), n, k, None))
    assert torch.equal(y, want)
    p.check()
    p.close()


def test_level_special_values(oracle, torch):
    """An infinite and a NaN right-hand side entry spread to the rows that
    depend on them and to no other."""
    from rbsptrsv import Plan
    f = gen.banded(5000, seed=8, window=40)
    b = gen.rhs(f.n, seed=9)
    b[3000], b[4000] = np.inf, np.nan
    rp, ci, v = f.csr()
    xo = oracle.sptrsv_serial(rp, ci, v, f.n, 0, b)
    p = Plan.from_factor(f)
    if not _is_level(p):  # a near thing between two schedules' timings here
        pytest.skip("the tuner picked the chain-following schedule")
    x = p.solve(torch.as_tensor(b, device="cuda")).cpu().numpy()
    p.close()
    fine = np.isfinite(xo)
    assert np.array_equal(fine, np.isfinite(x)) and fine[:3000].all()
    assert rel_err(x[fine], xo[fine]) < X_TOL


@pytest.mark.parametrize("lower", [True, False])
def test_level_refinement(torch, lower):
    from rbsptrsv import Plan
    for f in (gen.banded(9000, seed=2), gen.random_lower(6000, 12, seed=5, window=200),
              gen.laplacian(37, 200)):
        f = f if lower else f.transpose()
        p = Plan.from_factor(f, mixed=True)
        B = gen.rhs(f.n, seed=7, k=3)
        X, it, rel = p.solve_f32ir(torch.as_tensor(np.ascontiguousarray(B.T), device="cuda").t(),
                                   tol=1e-12)
        print("refinement", f.name, lower, it, rel, _is_level(p), flush=True)
        assert rel <= 1e-12
        for j in range(3):
            assert residual(f, X[:, j].cpu().numpy(), B[:, j]) < RES_TOL
        p.close()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("lower", [True, False])
def test_level_batch(torch, lower, mixed):
    """Uneven factors with 0 .. 40 columns, an empty one among them."""
    from rbsptrsv import Batch
    sizes = [(1, 1), (300, 0), (4000, 5), (257, 40), (0, 0), (9000, 2), (64, 33)]
    facs = [gen.banded(n, seed=i + 1, window=600) if n else
            gen.Factor(0, np.zeros(1, np.int32), np.zeros(0, np.int32), np.zeros(0), True)
            for i, (n, _) in enumerate(sizes)]
    if not lower:
        facs = [f.transpose() if f.n else gen.Factor(0, f.colptr, f.rowidx, f.val, False)
                for f in facs]
    bt = Batch(facs, mixed=mixed, tune_rhs=8)
    rng = np.random.default_rng(3)
    Bs = [rng.uniform(-1, 1, (k, f.n)) for f, (_, k) in zip(facs, sizes)]
    bs = [torch.as_tensor(B, device="cuda").t() if len(B) else None for B in Bs]
    for _ in range(2):
        xs = bt.solve_f32ir(bs, tol=1e-12)[0] if mixed else bt.solve(bs)
        for f, B, x in zip(facs, Bs, xs):
            for j in range(len(B)):
                assert residual(f, x[:, j].cpu().numpy(), B[j]) < RES_TOL
    bt.close()
