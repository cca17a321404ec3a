"""A batch whose solutions lie over right-hand sides: the same x, bit for bit,
as into memory of their own."""
import numpy as np
import pytest

from rbsptrsv import gen

pytestmark = pytest.mark.gpu

SIZES = [(3000, 3), (3000, 3), (700, 1), (9000, 4)]


@pytest.fixture(scope="module")
def batch():
    import torch
    from rbsptrsv import Batch
    bt = Batch([gen.banded(n, seed=i + 1, window=600) for i, (n, _) in enumerate(SIZES)],
               tune_rhs=4)
    rng = np.random.default_rng(5)
    Bs = [torch.as_tensor(rng.uniform(-1, 1, (k, n)), device="cuda") for n, k in SIZES]
    want = [x.t().clone() for x in bt.solve([B.t() for B in Bs])]
    yield torch, bt, Bs, want
    bt.close()


def _same(xs, want):
    return [bool((x == w).all()) for x, w in zip(xs, want)]


def _two(batch, b0, x0, b1, x1, W0, W1):
    """Factors 0 and 1 (alike in size) with these right-hand sides and
    solutions, (k, n); the others on memory of their own."""
    torch, bt, Bs, want = batch
    xs = [x0.t(), x1.t()] + [torch.empty_like(B).t() for B in Bs[2:]]
    bt.solve([b0.t(), b1.t()] + [B.t() for B in Bs[2:]], xs=xs)
    assert all(_same([x.t() for x in xs], [W0, W1] + want[2:]))


def test_batch_solutions_exchanged(batch):
    torch, bt, Bs, want = batch
    b0, b1 = Bs[0].clone(), Bs[1].clone()
    _two(batch, b0, b1, b1, b0, want[0], want[1])


def test_batch_shared_rhs(batch):
    """One b for two factors, the x of one over it."""
    torch, bt, Bs, want = batch
    b = Bs[0].clone()
    other = torch.empty_like(b)
    xs = bt.solve([b.t(), b.t(), None, None])
    W = [x.t().clone() for x in xs[:2]]
    for x0, x1 in ((b, other), (other, b)):
        b.copy_(Bs[0])
        _two(batch, b, x0, b, x1, W[0], W[1])


@pytest.mark.parametrize("shift", [1, -1, 0])
@pytest.mark.parametrize("rows", [0, 5])
def test_batch_shifted(batch, shift, rows):
    """x a column before or after b, and a few rows off."""
    torch, bt, Bs, want = batch
    n, k = SIZES[0]
    buf = torch.zeros((k + 2) * (n + 16), dtype=torch.float64, device="cuda")

    def at(col, row):
        o = col * (n + 16) + row
        return buf.as_strided((k, n), (n + 16, 1), o)

    b, x = at(1, 0), at(1 + shift, rows)
    b.copy_(Bs[0])
    _two(batch, b, x, Bs[1], torch.empty_like(Bs[1]), want[0], want[1])


def test_batch_other_leading_dimension(batch):
    torch, bt, Bs, want = batch
    n, k = SIZES[0]
    buf = torch.zeros(k * (n + 40), dtype=torch.float64, device="cuda")
    for lb, lx in ((n, n + 40), (n + 40, n)):
        b, x = buf.as_strided((k, n), (lb, 1)), buf.as_strided((k, n), (lx, 1))
        b.copy_(Bs[0])
        _two(batch, b, x, Bs[1], torch.empty_like(Bs[1]), want[0], want[1])


def test_batch_row_blocks_in_place(batch):
    """All factors in place on the rows of one matrix, column by column apart."""
    torch, bt, Bs, want = batch
    N = sum(n for n, _ in SIZES)
    M = torch.zeros(max(k for _, k in SIZES), N, dtype=torch.float64, device="cuda")
    views, o = [], 0
    for (n, k), B in zip(SIZES, Bs):
        views.append(M[:k, o:o + n])
        views[-1].copy_(B)
        o += n
    bt.solve([v.t() for v in views], xs=[v.t() for v in views])
    assert all(_same(views, want))
