"""Fluid outside the grid box: the evaluated pairs and the rates of blocks that stand out of the box
on every side, by less and by more than a box length, against the oracle (1e-12 norm-wise per
column, as in test_gpu_parity.py); and particles without a position (NaN), which the cell list
puts into its first cell and which reach no other particle."""
import math

import numpy as np
import pytest

from conftest import gpu_available
from test_brick_kernel import fluid_block

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

RTOL = 1e-12
DX = 0.02


def rates(tp, semi, v, u):
    import torch
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    dv = torch.full_like(vd, float("nan"))
    tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
    semi.synchronize()
    return dv.cpu().numpy()


def state(semi, nd):
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(21)
    v[:, :nd] = rng.normal(0.0, 0.5, size=(v.shape[0], nd))
    v[:, nd] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=v.shape[0])
    return v, u


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nd,n", [(2, (60, 40)), (3, (20, 18, 16))])
@pytest.mark.parametrize("lo,hi", [(0.0, 0.5), (0.3, 0.6), (0.45, 0.55), (-0.4, 1.1)])
def test_fluid_outside_the_box_matches_oracle(tp, orc, nd, n, lo, hi, precision):
    """The box from lo to hi of the block's extent."""
    fluid = fluid_block(tp, nd, n, tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0))
    ext = np.array(n) * DX
    semi = tp.Semidiscretization(fluid, domain=(lo * ext, hi * ext), precision=precision)
    v, u = state(semi, nd)
    ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
    off_ref, idx_ref = orc.neighbors(nd, 2 * fluid.smoothing_length, u, u)
    rows = np.repeat(np.arange(u.shape[0]), np.diff(off_ref))
    for repeat in range(2):                    # with the rebuild, then on the lists as they are
        got = rates(tp, semi, v, u)
        for col in range(nd + 1):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            tol = RTOL if precision == "fp64" else 1e-5 if col == nd else 1e-4
            assert err <= tol, f"column {col}, kick {repeat}: {err:.3e}"
        off, idx = tp.kick_pairs(semi, tp.native.PAIR_FLUID_FLUID)
        assert np.array_equal(np.diff(off) + 1, np.diff(off_ref))
        assert np.array_equal(idx.astype(np.int64), idx_ref[rows != idx_ref])
    semi.close()


@pytest.mark.parametrize("nd,dx", [(2, 0.02), (3, 0.05)])
def test_particles_without_a_position_reach_no_other(tp, nd, dx):
    db = tp.dam_break(nd, dx)
    lo, hi = tp.Semidiscretization(db.fluid_system, db.boundary_system).domain
    lo = lo + 3.5 * dx                         # the first cell beside the fluid's and walls' corner
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, domain=(lo, hi))
    v, u = state(semi, nd)
    away = u.copy()
    lost = [1, u.shape[0] // 2]
    away[lost] = 1e3 + np.arange(2).reshape(2, 1) * 10.0
    ref = rates(tp, semi, v, away)
    pw_ref = semi.update_pressures()[1].copy()
    u[lost] = math.nan
    keep = np.setdiff1d(np.arange(u.shape[0]), lost)
    for repeat in range(2):
        got = rates(tp, semi, v, u)
        assert np.isfinite(got[keep]).all()
        for col in range(nd + 1):
            err = np.abs(got[keep, col] - ref[keep, col]).max() / np.abs(ref[keep, col]).max()
            assert err <= RTOL, f"column {col}, kick {repeat}: {err:.3e}"
        pw = semi.update_pressures()[1]
        assert np.abs(pw - pw_ref).max() <= RTOL * np.abs(pw_ref).max()
    semi.close()
