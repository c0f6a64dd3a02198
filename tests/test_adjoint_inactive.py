"""The parameter partials of terms that the right-hand side does not have: without a viscosity the
derivative along alpha is zero, without density diffusion the one along delta, as in the oracle's
dual kick; for the pullback of one kick and through a trajectory, with Verlet lists and cells."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


@pytest.mark.parametrize("nd,dx", [(2, 0.02), (3, 0.05)])
@pytest.mark.parametrize("search", ["lists", "cells"])
@pytest.mark.parametrize("term", ["viscosity", "density_diffusion"])
def test_partials_of_absent_terms_are_zero(tp, orc, nd, dx, search, term):
    import torch
    from trixiparticles_jl_amd import adjoint as ad
    db = tp.dam_break(nd, dx)
    setattr(db.fluid_system, term, None)
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, pair_search=search)
    v, u = semi.initial_state()
    rng = np.random.default_rng(7)
    v[:, :nd] = torch.from_numpy(rng.normal(0.0, 0.3, size=(v.shape[0], nd))).cuda()
    dv_bar = torch.from_numpy(rng.normal(size=tuple(v.shape))).cuda()
    dv_bar[:, nd] *= 1e-2
    k = 0 if term == "viscosity" else 1

    _, _, pb = ad.kick_vjp(semi, dv_bar, v, u)
    sp = np.zeros((3, 4))
    sp[0, 0] = sp[1, 1] = sp[2, 2] = 1.0
    vh, uh = v.cpu().numpy(), u.cpu().numpy()
    wall = db.boundary_system
    _, tan = orc.dual_kick(orc.params_from_semi(semi), vh, uh, db.fluid_system.mass,
                           wall.coordinates.T.copy(), wall.boundary_model.hydrodynamic_mass, sp,
                           np.zeros((4, *vh.shape)), np.zeros((4, *uh.shape)))
    assert not tan[k].any()
    assert pb[k] == 0.0
    for i in {0, 1, 2} - {k}:                   # the terms that are there keep theirs
        terms = dv_bar.cpu().numpy() * tan[i]
        assert abs(terms.sum() - pb[i]) <= 1e-10 * np.abs(terms).sum(), i

    _, _, _, pb = ad.gradient(semi, v, u, u + 0.01 * dx, 1e-5, 3, checkpoint_every=2)
    assert pb[k] == 0.0
    assert all(pb[i] != 0.0 for i in {0, 1, 2} - {k})
    semi.close()
