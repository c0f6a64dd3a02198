"""The mixed-precision pair loop (Target32) against the oracle: with and without viscosity, one
brick and many, coincident particles and particles closer than sqrt(eps) R (which the relation
leaves out).  The bounds are those of test_mixed_precision.py's single kick: a few FP32 roundings
times the cancellation in the sums."""
import numpy as np
import pytest

from conftest import gpu_available
from test_brick_kernel import fluid_block

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


@pytest.mark.parametrize("nd,n,alpha", [
    (2, (2, 2), 0.02), (2, (37, 21), 0.0), (2, (120, 90), 0.02),
    (3, (5, 4, 3), 0.02), (3, (30, 23, 16), 0.0), (3, (48, 48, 48), 0.02),
])
def test_mixed_pairs_match_oracle(tp, orc, nd, n, alpha):
    import torch
    fluid = fluid_block(tp, nd, n, tp.ArtificialViscosityMonaghan(alpha=alpha, beta=0.0) if alpha else None)
    semi = tp.Semidiscretization(fluid, precision="mixed")
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(21)
    v[:, :nd] = rng.normal(0.0, 0.5, size=(v.shape[0], nd))
    v[:, nd] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=v.shape[0])
    u[1] = u[0]                                # coincident
    u[3] = u[2] + 1e-10 * 2 * fluid.smoothing_length
    ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    for repeat in range(2):                    # with the rebuild, then on the lists as they are
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(nd + 1):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            assert err <= (1e-5 if col == nd else 1e-4), (col, repeat, err)
    semi.close()
