"""x over b by whole columns, for more columns than one pass takes: the same
x, bit for bit, as into memory of its own, or the call is refused."""
import ctypes

import numpy as np
import pytest

from rbsptrsv import gen

pytestmark = pytest.mark.gpu

K = 70
FACTORS = {
    "level": (lambda: gen.banded(9000, seed=2), 0),
    "level-solve-order": (lambda: gen.banded(30000, seed=2).transpose(), 0),
    "flow": (lambda: gen.powerlaw(60000, seed=5), 0),
    "blocked": (lambda: gen.powerlaw(6000, seed=3), 1),
    "fused": (lambda: gen.laplacian(300, 40), 2),
}


@pytest.fixture(scope="module", params=list(FACTORS))
def plan(request):
    import torch
    from rbsptrsv import Plan
    make, schedule = FACTORS[request.param]
    f = make()
    p = Plan.from_factor(f, schedule=schedule)
    B = torch.as_tensor(np.random.default_rng(4).uniform(-1, 1, (K, f.n)), device="cuda")
    want = torch.stack([p.solve(B[j].contiguous()) for j in range(K)])
    print(request.param, flush=True)
    yield torch, p, f.n, B, want
    p.check()
    p.close()


def _call(entry, p, b, ldb, x, ldx, k=K):
    from rbsptrsv._lib import lib
    return getattr(lib(), entry)(p._h, ctypes.c_void_p(b), ldb, ctypes.c_void_p(x), ldx, k, None)


@pytest.mark.parametrize("entry", ["rb_solve", "rb_solve_noalloc"])
@pytest.mark.parametrize("shift", [1, -1, 3, -40])
def test_columns_shifted(plan, entry, shift):
    """x `shift` columns after b, and five rows besides."""
    torch, p, n, B, want = plan
    for rows in (0, 5):
        buf = torch.zeros((K + abs(shift) + 1) * n, dtype=torch.float64, device="cuda")
        o = max(0, -shift) * n
        b, x = buf[o:o + K * n], buf[o + shift * n + rows:][:K * n]
        b.copy_(B.flatten())
        assert _call(entry, p, b.data_ptr(), n, x.data_ptr(), n) == 0
        assert torch.equal(x.view(K, n), want), rows


@pytest.mark.parametrize("entry", ["rb_solve", "rb_solve_noalloc"])
@pytest.mark.parametrize("ldb,ldx,first", [(1, 2, 0), (2, 1, 0), (2, 1, 35), (1, 2, -1)])
def test_other_leading_dimension(plan, entry, ldb, ldx, first):
    """b's columns ldb * n apart, x's ldx * n, the first of x `first` columns
    after the first of b."""
    torch, p, n, B, want = plan
    buf = torch.zeros((2 * K + 40) * n, dtype=torch.float64, device="cuda")
    o = max(0, -first) * n
    b = buf[o:].as_strided((K, n), (ldb * n, 1))
    x = buf[o + first * n:].as_strided((K, n), (ldx * n, 1))
    b.copy_(B)
    st = _call(entry, p, b.data_ptr(), ldb * n, x.data_ptr(), ldx * n)
    if st == 0:
        assert torch.equal(x, want)
    else:  # refused, and nothing written
        assert (ldb, first) == (2, 35) and st == 1 and torch.equal(b, B)
