"""The refinement's residual from x held in LDS: rows at the edges of its
blocks, of the entries a thread keeps and of the widest window it takes (and
one column beyond, which goes to the general kernel), columns around a group,
in a batch with a different number of columns for every factor."""
import numpy as np
import pytest

from helpers import csc_from_deps, rel_err, residual
from rbsptrsv import gen

pytestmark = pytest.mark.gpu


def _reach(n, rows_of, reach, seed):
    """n rows with row i's entries spread over the reach columns before it."""
    deps = {}
    for i in range(1, n):
        k = min(rows_of[i % len(rows_of)], i, reach)
        lo = max(0, i - reach)
        deps[i] = sorted({lo + int((i - lo - 1) * t / max(1, k - 1)) for t in range(k)})
    return csc_from_deps(n, deps, seed=seed, diag=60.0)


# a block of rows and what they reach fit 7,680 columns: 1,024 + 6,656
CASES = [
    ("blocks", 2049, [1, 2, 3], 700),
    ("ten", 3000, [9, 10, 11, 0], 1500),
    ("long", 2500, [4, 40, 5], 2000),
    ("widest", 9000, [3], 6656),
    ("beyond", 9000, [3], 6657),
]


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("name,n,rows_of,reach", CASES, ids=[c[0] for c in CASES])
def test_refined_solve_matches_oracle(oracle, name, n, rows_of, reach, lower):
    import torch
    from rbsptrsv import Plan
    f = _reach(n, rows_of, reach, seed=n)
    f = f if lower else f.transpose()
    print("residual", name, lower, flush=True)
    rp, ci, v = f.csr()
    B = gen.rhs(f.n, seed=4, k=17)
    p = Plan.from_factor(f, mixed=True)
    for k in (1, 7, 8, 9, 17):
        b = torch.as_tensor(np.ascontiguousarray(B[:, :k].T), device="cuda")
        x = torch.full_like(b, 3.0)   # what x held does not matter
        X = p.solve_f32ir(b.t() if k > 1 else b[0], x=x.t() if k > 1 else x[0])[0]
        X = X.cpu().numpy().reshape(n, k)
        for j in range(k):
            xo = oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j])
            assert rel_err(X[:, j], xo) < 1e-10
            assert residual(f, X[:, j], B[:, j]) < 1e-12
    p.check()
    p.close()


# groups of 1, 2, 4 and 8 columns to a workgroup (so many that at least 192
# workgroups are left), too few workgroups for it (48), and the longest row it
# takes and one more
@pytest.mark.parametrize("n,rows_of,ks", [
    (3000, [3], (15, 16, 17)),
    (25000, [3, 9], (1, 2, 7, 8, 9)),
    (60000, [2], (1, 4, 9, 24)),
    (200000, [3], (1, 8, 9)),
    (50000, [3] * 40 + [31], (1, 9)),
    (50000, [3] * 40 + [32], (1, 9)),
], ids=lambda v: str(v[-1]) if isinstance(v, list) else str(v).replace(" ", ""))
def test_residual_groups(oracle, n, rows_of, ks):
    import torch
    from rbsptrsv import Plan
    f = _reach(n, rows_of, 700, seed=n)
    print("residual groups", n, rows_of[-1], flush=True)
    rp, ci, v = f.csr()
    B = gen.rhs(f.n, seed=4, k=max(ks))
    p = Plan.from_factor(f, mixed=True)
    for k in ks:
        b = torch.as_tensor(np.ascontiguousarray(B[:, :k].T), device="cuda")
        X = p.solve_f32ir(b.t())[0].t().cpu().numpy()
        for j in range(k):
            assert residual(f, X[j], B[:, j]) < 1e-12
        assert rel_err(X[k - 1], oracle.sptrsv_serial(rp, ci, v, f.n, 0, B[:, k - 1])) < 1e-10
    p.check()
    p.close()
