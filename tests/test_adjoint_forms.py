"""The pullback of a kick in the forms of the right-hand side that test_adjoint.py leaves out:
no viscosity, a quadratic term (beta), no density diffusion; brick lists, int lists and the cell
walk.  <dv_bar, J s> from the oracle's dual kick against <J^T dv_bar, s>, as there, relative to
the sum of the terms' magnitudes and to its bound 1e-10."""
import math

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


@pytest.mark.parametrize("nd,n,visc,delta,kw", [
    (2, (24, 17), None, 0.1, {}),
    (2, (24, 17), dict(alpha=0.02, beta=1.5), 0.0, {}),
    (3, (12, 9, 7), dict(alpha=0.0, beta=1.5), 0.1, {}),
    (3, (12, 9, 7), dict(alpha=0.02, beta=0.0), 0.0, dict(pair_search="cells")),
    (3, (12, 9, 7), dict(alpha=0.02, beta=1.5), 0.1, dict(pair_search="lists", cell_divisions=3)),
])
def test_pullback_forms_match_dual_tangents(tp, orc, nd, n, visc, delta, kw):
    import torch
    from trixiparticles_jl_amd import adjoint as ad
    dx = 0.02
    g = (0.0, -9.81) if nd == 2 else (0.0, -9.81, 0.0)
    se = tp.StateEquationCole(sound_speed=20 * math.sqrt(9.81 * 0.6), reference_density=1000.0,
                              exponent=7.0, clip_negative_pressure=False)
    ic = tp.RectangularShape(dx, n, (0.0,) * nd, density=1000.0, coordinates_perturbation=0.05, seed=3)
    fluid = tp.WeaklyCompressibleSPHSystem(
        ic, tp.ContinuityDensity(), se, tp.WendlandC2Kernel(nd), 1.2 * dx, acceleration=g,
        viscosity=tp.ArtificialViscosityMonaghan(**visc) if visc else None,
        density_diffusion=tp.DensityDiffusionMolteniColagrossi(delta=delta) if delta else None)
    semi = tp.Semidiscretization(fluid, **kw)
    P = orc.params_from_semi(semi)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(11)
    nf = v.shape[0]
    v[:, :nd] = rng.normal(0.0, 0.3, size=(nf, nd))
    v[:, nd] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=nf)
    dv_bar = rng.normal(size=v.shape)
    dv_bar[:, nd] *= 1e-2
    vb, ub, pb = ad.kick_vjp(semi, torch.from_numpy(dv_bar).cuda(), torch.from_numpy(v).cuda(),
                             torch.from_numpy(u).cuda())
    vb, ub = vb.cpu().numpy(), ub.cpu().numpy()
    sp = np.zeros((3, 4))
    sp[0, 0] = sp[1, 1] = sp[2, 2] = 1.0
    sv, su = np.zeros((4, nf, nd + 1)), np.zeros((4, nf, nd))
    _, tan = orc.dual_kick(P, v, u, fluid.mass, None, None, sp, sv, su)
    active = (bool(visc), bool(delta), True)
    for k in range(3):
        terms = dv_bar * tan[k]
        if active[k]:
            assert abs(terms.sum() - float(pb[k])) <= 1e-10 * np.abs(terms).sum(), k
    sv[0, :, :nd] = rng.normal(size=(nf, nd))
    sv[1, :, nd] = rng.normal(size=nf)
    su[2] = rng.normal(size=(nf, nd))
    sv[3], su[3] = rng.normal(size=(nf, nd + 1)), rng.normal(size=(nf, nd))
    _, tan = orc.dual_kick(P, v, u, fluid.mass, None, None, None, sv, su)
    for k in range(4):
        terms = dv_bar * tan[k]
        got = (vb * sv[k]).sum() + (ub * su[k]).sum()
        assert abs(terms.sum() - got) <= 1e-10 * np.abs(terms).sum(), k
    semi.close()
