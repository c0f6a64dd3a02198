"""Bricks of fluids whose masses do not fit their spacing (a thousandth of it), on both sides of the
number of particles to which bricks shrink: rates against the oracle, 1e-12 norm-wise per column
as in test_gpu_parity.py."""
import numpy as np
import pytest

from conftest import gpu_available
from test_brick_kernel import fluid_block

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


@pytest.mark.parametrize("n", [(20, 18, 16), (80, 72, 72)])
def test_light_particles_match_oracle(tp, orc, n):
    import torch
    fluid = fluid_block(tp, 3, n, tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0))
    fluid.mass[:] *= 1e-3
    semi = tp.Semidiscretization(fluid)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(21)
    v[:, :3] = rng.normal(0.0, 0.5, size=(v.shape[0], 3))
    ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    dv = torch.full_like(vd, float("nan"))
    tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
    semi.synchronize()
    got = dv.cpu().numpy()
    for col in range(4):
        err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
        assert err <= 1e-12, f"column {col}: {err:.3e}"
    semi.close()
