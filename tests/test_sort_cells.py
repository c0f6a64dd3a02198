"""The rebuild of a small fluid in grids of many cells, on both sides of the number of cells (3 x 2^20)
to which one kernel (k_sort) takes the whole rebuild, and of its blocks' first turn over the scan's
tiles (2^20): rates right after rebuilds against the oracle.  Tolerance as in test_gpu_parity.py:
1e-12 norm-wise per column."""
import math

import numpy as np
import pytest

from conftest import gpu_available
from test_brick_kernel import fluid_block

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


def boxed(tp, fluid, cells):
    """The fluid in a box of at most (and about) `cells` cells."""
    nd = fluid.ndims
    R = 2 * fluid.smoothing_length
    cs = [1.0400125 * R / (4 if d == 0 else 2) for d in range(nd)]
    side = int(round(cells ** (1 / nd)))
    n = [side] * nd
    n[0] = cells // side ** (nd - 1)
    domain = ([-0.2] * nd, [-0.2 + (n[d] - 3.5) * cs[d] for d in range(nd)])
    count = math.prod(math.ceil((domain[1][d] - domain[0][d]) / cs[d] + 2.0) + 1 for d in range(nd))
    assert 0.97 * cells < count <= cells
    return tp.Semidiscretization(fluid, domain=domain)


@pytest.mark.parametrize("nd,n", [(2, (60, 30)), (3, (20, 18, 16))])
@pytest.mark.parametrize("cells", [(1 << 20) - 20000, (1 << 20) + 60000, 3 << 20, (3 << 20) + 150000])
def test_rebuilds_in_large_grids_match_oracle(tp, orc, nd, n, cells):
    import torch
    fluid = fluid_block(tp, nd, n, tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0))
    semi = boxed(tp, fluid, cells)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(8)
    u = u[rng.permutation(u.shape[0])]
    v[:, :nd] = rng.normal(0.0, 0.5, size=(v.shape[0], nd))
    for repeat in range(3):
        ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
        vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(nd + 1):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            assert err <= 1e-12, f"column {col}, kick {repeat}: {err:.3e}"
        u = u + rng.uniform(-0.2, 0.2, size=u.shape) * 0.02   # beyond the skin
    semi.close()
