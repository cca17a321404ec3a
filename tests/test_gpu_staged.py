"""The fused schedule's staged form (one-sided grids): step counts around a
block (16 steps) and the ring (64), one and several waves, FP64 with one and
three columns and refined FP32, against the oracle."""
import numpy as np
import pytest

from helpers import rel_err, residual
from rbsptrsv import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("ny", [2, 64, 130])
@pytest.mark.parametrize("nx", [2, 15, 16, 33, 62, 63, 64, 65, 127, 200])
def test_staged_grids_match_oracle(oracle, nx, ny, lower):
    import torch
    from rbsptrsv import Plan
    f = gen.laplacian(nx, ny)
    f = f if lower else f.transpose()
    print("staged", nx, ny, lower, flush=True)
    rp, ci, v = f.csr()
    B = gen.rhs(f.n, seed=4, k=3)
    Xo = [oracle.sptrsv_serial(rp, ci, v, f.n, f.substitution, B[:, j]) for j in range(3)]
    b = torch.as_tensor(np.ascontiguousarray(B.T), device="cuda")
    p = Plan.from_factor(f, schedule=2, mixed=True)
    single = [p.solve(b[j].contiguous()).cpu().numpy() for j in range(3)]
    X = p.solve(b.t()).t().cpu().numpy()
    R = p.solve_f32ir(b.t())[0].t().cpu().numpy()
    for j in range(3):
        assert rel_err(single[j], Xo[j]) < 1e-10
        assert residual(f, single[j], B[:, j]) < 1e-12
        assert np.array_equal(X[j].view(np.int64), single[j].view(np.int64))
        assert rel_err(R[j], Xo[j]) < 1e-10
    p.check()
    p.close()
