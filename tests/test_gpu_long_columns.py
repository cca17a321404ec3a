"""The level analysis and the block storage of factors with columns and rows
longer than one thread takes (a wave takes them), and with frontiers at the
edges of the paths (one node per thread, two, the workgroup's width, the grid):
the same order, levels, block levels and block statistics as the oracle, bit
for bit."""
import numpy as np
import pytest

from helpers import csc_from_deps, residual
from rbsptrsv import gen

pytestmark = pytest.mark.gpu

COLUMN = [3, 4, 5, 15, 16, 17, 18, 63, 64, 65, 66, 131, 1030]
ROW = [31, 32, 33, 64, 65, 128, 129, 300]


def _levels(widths, seed):
    """Levels of the given widths; the first nodes of a level have columns of
    every length in COLUMN, the first rows rows of every length in ROW (as
    far as the level above has room)."""
    rng = np.random.default_rng(seed)
    deps, start, base = {}, 0, widths[0]
    for k in range(1, len(widths)):
        w, above = widths[k], widths[k - 1]
        for j in range(w):
            deps[base + j] = {start + int(rng.integers(above))}
        for c, n in enumerate(COLUMN[:above]):
            for j in rng.permutation(w)[:n]:
                deps[base + int(j)].add(start + c)
        for j, n in enumerate(ROW[:w]):
            deps[base + j].update(start + int(i) for i in rng.permutation(above)[:n])
        start, base = base, base + w
    return csc_from_deps(base, {i: sorted(d) for i, d in deps.items()}, seed=seed, diag=40.0)


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("widths", [
    [1, 40, 1023, 1024, 1025, 1], [2047, 2048, 2049, 5], [3000, 4096, 4097, 700, 64]])
@pytest.mark.parametrize("lv", [1, 3])
def test_analysis_matches_oracle(oracle, widths, lower, lv):
    import torch
    from rbsptrsv import Plan
    f = _levels(widths, seed=sum(widths))
    if not lower:
        f = f.transpose()
    print("long columns", widths, lower, lv, flush=True)
    re, part, bnz, an = oracle.full_pipeline(f.colptr, f.rowidx, f.val, f.n, f.substitution, lv)
    p = Plan.from_factor(f, lv=lv)
    li, lp = p.levels()
    assert np.array_equal(lp, re["levelPtr"]) and np.array_equal(li, re["levelItem"])
    bl = p.blocks()
    assert np.array_equal(bl["blk_nnz"], bnz)
    for k in ("method", "nlv", "nnzr", "m_new", "lenmax", "longrow", "longlen"):
        assert np.array_equal(bl[k], an[k]), k
    for t in range(1 << lv):
        lvp, lvi, _ = p.tri_levels(t)
        assert np.array_equal(lvp, an["lvptr_local"][t])
        assert np.array_equal(lvi, an["lvitem_local"][t])
    b = gen.rhs(f.n, seed=2)
    x = p.solve(torch.as_tensor(b, device="cuda")).cpu().numpy()
    p.check()
    assert residual(f, x, b) < 1e-12
    p.close()
