"""The rebuild chain (k_links, k_scan, k_gather<1>, one kernel k_sort up to 2^17 particles): kicks
right after it against the oracle, at fluids of one item and the edges of the items of 1024
particles, of more particles than the items take in one turn, and on both sides of 2^17; in a
caller's order without any locality, with cells of many members (a cluster in one cell) and with
the particles moved beyond the skin before every kick; and the sorted order, stable whatever
order the atomics were served in: the same kick twice from scratch gives the same bits.
Tolerance as in test_gpu_parity.py: 1e-12 norm-wise per column."""
import math

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

RTOL = 1e-12


@pytest.mark.parametrize("search", ["lists", "cells"])
@pytest.mark.parametrize("nd,n", [
    (2, (1, 1)), (3, (7, 9, 1)), (2, (32, 32)), (2, (41, 25)),   # 1, 63, 1024, 1025
    (3, (41, 41, 40)),                                          # 67,240: over 64 items of 1024
    (2, (512, 256)), (2, (331, 396)),                           # 2^17 and just above
])
def test_kicks_after_rebuilds_match_oracle(tp, orc, nd, n, search):
    import torch
    dx = 0.02
    g = (0.0, -9.81) if nd == 2 else (0.0, -9.81, 0.0)
    se = tp.StateEquationCole(sound_speed=20 * math.sqrt(9.81 * 0.6), reference_density=1000.0,
                              exponent=7.0, clip_negative_pressure=False)
    ic = tp.RectangularShape(dx, n, (0.0,) * nd, density=1000.0, coordinates_perturbation=0.01, seed=3)
    fluid = tp.WeaklyCompressibleSPHSystem(
        ic, tp.ContinuityDensity(), se, tp.WendlandC2Kernel(nd), 1.2 * dx, acceleration=g,
        viscosity=tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0),
        density_diffusion=tp.DensityDiffusionMolteniColagrossi(delta=0.1))
    states, first = [], None
    for attempt in range(2):
        semi = tp.Semidiscretization(fluid, pair_search=search)
        v0, u0 = semi.initial_state()
        v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
        rng = np.random.default_rng(8)
        u = u[rng.permutation(u.shape[0])]
        v[:, :nd] = rng.normal(0.0, 0.5, size=(v.shape[0], nd))
        v[:, nd] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=v.shape[0])
        if u.shape[0] > 1000:                     # forty particles within a tenth of a spacing
            u[::25][:40] = u[0] + rng.uniform(-0.05, 0.05, size=(40, nd)) * dx
        got = []
        for repeat in range(3):
            vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
            dv = torch.full_like(vd, float("nan"))
            tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
            semi.synchronize()
            got.append(dv.cpu().numpy())
            if attempt == 0:
                ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
                for col in range(nd + 1):
                    err = np.abs(got[-1][:, col] - ref[:, col]).max() / max(np.abs(ref[:, col]).max(), 1e-300)
                    assert err <= RTOL, f"column {col}, kick {repeat}: {err:.3e}"
            u = u + rng.uniform(-0.4, 0.4, size=u.shape) * dx
        semi.close()
        states.append(got)
    for a, b in zip(*states):
        assert np.array_equal(a, b)
