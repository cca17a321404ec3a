"""Rectangular grids whose chains end in the first waves while new ones begin
beside the last (a wave more for every group of 64 chains): the fused
schedule's solves match the oracle, at widths around whole waves, with one
and several columns, in FP64 and refined FP32."""
import numpy as np
import pytest

from helpers import rel_err, residual
from rbsptrsv import gen

pytestmark = pytest.mark.gpu

GRIDS = [(64, 200), (65, 66), (65, 129), (70, 500), (128, 129), (129, 260), (217, 333),
         (66, 3000)]


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_sideways_grids_match_oracle(oracle, nx, ny, lower):
    import torch
    from rbsptrsv import Plan
    # chains run along x; the other direction walks the other way
    f = gen.laplacian(nx, ny) if lower else gen.laplacian(ny, nx).transpose()
    print("chain waves", nx, ny, lower, flush=True)
    rp, ci, v = f.csr()
    B = gen.rhs(f.n, seed=4, k=9)
    Xo = np.stack([oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j])
                   for j in range(9)])
    b = torch.as_tensor(np.ascontiguousarray(B.T), device="cuda")
    p = Plan.from_factor(f, schedule=2)
    single = []
    for j in range(3):
        single.append(p.solve(b[j].contiguous()).cpu().numpy())
        assert rel_err(single[j], Xo[j]) < 1e-10
        assert residual(f, single[j], B[:, j]) < 1e-12
    for k in (2, 9):
        X = p.solve(b[:k].t()).t().cpu().numpy()
        for j in range(k):
            assert rel_err(X[j], Xo[j]) < 1e-10
            if j < 3:
                assert np.array_equal(X[j].view(np.int64), single[j].view(np.int64))
    p.check()
    p.close()
