"""The level and flow schedules asked for by name, so that the edges of their
tiles are reached whatever the tuner would pick, and the failure path of every
kernel with a bounded wait."""
import numpy as np
import pytest

import test_gpu_flow
import test_gpu_level
from helpers import csc_from_deps, rel_err, residual
from rbsptrsv import SCHED_AUTO, SCHED_FLOW, SCHED_FUSED, SCHED_LEVEL, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a device"
    return torch


def _matches_oracle(oracle, torch, f, schedule, columns):
    from rbsptrsv import Plan
    p = Plan.from_factor(f, schedule=schedule)
    assert p.schedule() == schedule
    B = gen.rhs(f.n, seed=5, k=max(columns)).reshape(f.n, -1)
    rp, ci, v = f.csr()
    single = []
    for j in range(B.shape[1]):
        x = p.solve(torch.as_tensor(B[:, j].copy(), device="cuda")).cpu().numpy()
        assert rel_err(x, oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j])) < 1e-10
        assert residual(f, x, B[:, j]) < 1e-12
        single.append(x)
    for k in columns:
        b = torch.as_tensor(np.ascontiguousarray(B[:, :k].T), device="cuda")
        X = p.solve(b.t()).t().cpu().numpy()
        for j in range(k):
            assert np.array_equal(X[j].view(np.int64), single[j].view(np.int64))
    p.check()
    p.close()


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("name,make", test_gpu_level.CASES,
                         ids=[c[0] for c in test_gpu_level.CASES])
def test_level(oracle, torch, name, make, lower):
    from rbsptrsv import Plan, RbError
    f = make() if lower else make().transpose()
    print("level", name, lower, flush=True)
    if np.diff(f.csr()[0]).max() - 1 > 512:
        with pytest.raises(RbError) as e:
            Plan.from_factor(f, schedule=SCHED_LEVEL)
        assert e.value.status == 1
        return
    _matches_oracle(oracle, torch, f, SCHED_LEVEL, [3])


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("name,make", test_gpu_flow.CASES + [
    ("one-row", lambda: csc_from_deps(1, {})),
    ("diagonal", lambda: csc_from_deps(700, {})),
    ("chain", lambda: csc_from_deps(300, {i: [i - 1] for i in range(1, 300)})),
], ids=lambda v: v if isinstance(v, str) else "")
def test_flow(oracle, torch, name, make, lower):
    f = make() if lower else make().transpose()
    print("flow", name, lower, flush=True)
    _matches_oracle(oracle, torch, f, SCHED_FLOW, [2, 3, 4, 5, 8, 9])


@pytest.mark.parametrize("n", [20001, 60000])
def test_flow_groups(oracle, torch, n):
    """Groups of 8 columns side by side in a launch, up to four of them."""
    _matches_oracle(oracle, torch, gen.powerlaw(n, seed=5), SCHED_FLOW,
                    [7, 15, 16, 17, 24, 25, 31, 32, 33, 40])


def test_level_special_values(oracle, torch):
    """An infinite and a NaN right-hand side entry spread to the rows that
    depend on them and to no other."""
    from rbsptrsv import Plan
    f = gen.banded(5000, seed=8, window=40)
    b = gen.rhs(f.n, seed=9)
    b[3000], b[4000] = np.inf, np.nan
    xo = oracle.sptrsv_serial(*f.csr(), f.n, 0, b)
    p = Plan.from_factor(f, schedule=SCHED_LEVEL)
    x = p.solve(torch.as_tensor(b, device="cuda")).cpu().numpy()
    p.close()
    fine = np.isfinite(xo)
    assert np.array_equal(fine, np.isfinite(x)) and fine[:3000].all()
    assert rel_err(x[fine], xo[fine]) < 1e-10


@pytest.mark.parametrize("k", [1, 3, 19])
@pytest.mark.parametrize("name,make,schedule", [
    ("flow", lambda: gen.powerlaw(60000, seed=5), SCHED_FLOW),
    # (several waves, so that one has to wait for another)
    ("staged", lambda: gen.laplacian(700, 300), SCHED_FUSED),
])
def test_watchdog_trip(torch, name, make, schedule, k):
    """Bounded waits that give up after one poll: x all NaN, the check reports
    it and clears it; another plan on the factor is unaffected.  Every kernel
    exits normally."""
    from rbsptrsv import Plan, RbError
    f = make()
    b = torch.as_tensor(np.ascontiguousarray(gen.rhs(f.n, seed=2, k=k).reshape(f.n, k).T),
                        device="cuda")
    print("watchdog", name, k, flush=True)
    p = Plan.from_factor(f, schedule=schedule, watchdog_spins=1)
    for _ in range(2):
        x = p.solve(b.t() if k > 1 else b[0])
        with pytest.raises(RbError) as e:
            p.check()
        assert e.value.status == 8
        assert bool(torch.isnan(x).all())
        p.check()
    p.close()
    q = Plan.from_factor(f, schedule=schedule)
    y = q.solve(b.t() if k > 1 else b[0])
    q.check()
    q.close()
    y = y.reshape(f.n, k) if k == 1 else y
    for j in range(k):
        assert residual(f, y[:, j].cpu().numpy(), b[j].cpu().numpy()) < 1e-12


def test_watchdog_trip_staged_refinement(torch):
    from rbsptrsv import Plan, RbError
    f = gen.laplacian(700, 300)
    b = torch.as_tensor(gen.rhs(f.n, seed=2), device="cuda")
    print("watchdog staged refinement", flush=True)
    p = Plan.from_factor(f, schedule=SCHED_FUSED, mixed=True, watchdog_spins=1)
    for _ in range(2):
        x = p.solve_f32ir(b, tol=1e-12, max_iter=2, report=False)[0]
        with pytest.raises(RbError) as e:
            p.check()
        assert e.value.status == 8
        assert bool(torch.isnan(x).all())
    p.close()


@pytest.mark.parametrize("make", [lambda: gen.powerlaw(60000, seed=5),
                                  lambda: gen.banded(20000, seed=4)], ids=["wide", "deep"])
def test_tuner_leaves_out_what_trips(torch, make):
    """With waits that give up at once the tuner keeps a schedule that does
    not wait, or the block walk; the solve is right or reported, never wrong."""
    from rbsptrsv import Plan, RbError
    f = make()
    b = gen.rhs(f.n, seed=2)
    p = Plan.from_factor(f, schedule=SCHED_AUTO, watchdog_spins=1)
    assert p.schedule() not in (SCHED_FLOW, SCHED_FUSED)
    x = p.solve(torch.as_tensor(b, device="cuda"))
    try:
        p.check()
    except RbError:
        assert bool(torch.isnan(x).all())
    else:
        assert residual(f, x.cpu().numpy(), b) < 1e-12
    p.close()


def test_not_for_batches(torch):
    from rbsptrsv import Batch, RbError
    facs = [gen.banded(500, seed=i, window=40) for i in range(3)]
    with pytest.raises(RbError) as e:
        Batch(facs, schedule=SCHED_FLOW)
    assert e.value.status == 1
    bt = Batch(facs, schedule=SCHED_LEVEL)
    assert bt.schedule() == SCHED_LEVEL
    bs = [torch.as_tensor(gen.rhs(500, seed=i), device="cuda") for i in range(3)]
    for f, b, x in zip(facs, bs, bt.solve(bs)):
        assert residual(f, x.cpu().numpy(), b.cpu().numpy()) < 1e-12
    bt.close()


def test_batch_factors_do_not_move_each_others_rows(torch):
    """Rows that no other reads, at the head of a factor behind the odd tail of
    a much deeper one: they keep to their own factor's levels, so that the
    batch still fits its rings in the caller's order and needs no union columns
    (2 x 80,100 rows x 16 columns, 20 MB)."""
    from rbsptrsv import Batch
    head, tail = 200, gen.banded(19800, seed=3, window=600)
    cp, ri, v = tail.colptr.astype(np.int64), tail.rowidx, tail.val
    second = gen.Factor(
        head + tail.n, np.concatenate([np.arange(head), head + cp]).astype(np.int32),
        np.concatenate([np.arange(head), head + ri]).astype(np.int32),
        np.concatenate([np.full(head, 2.0), v]), True)
    facs = [gen.banded(60100, seed=2), second]
    bt = Batch(facs, schedule=SCHED_LEVEL)
    rng = np.random.default_rng(1)
    bs = [torch.as_tensor(rng.uniform(-1, 1, (16, f.n)), device="cuda").t() for f in facs]
    xs = [torch.empty_like(b.t()).t() for b in bs]
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    bt.solve(bs, xs=xs)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 10 << 20
    for f, b, x in zip(facs, bs, xs):
        assert residual(f, x[:, 0].cpu().numpy(), b[:, 0].cpu().numpy()) < 1e-12
    bt.close()
