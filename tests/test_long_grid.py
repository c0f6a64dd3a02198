"""Grids of more than 32,767 cells along x: a long flume, and blocks of fluid at both ends of a long
box and across its 32,768th cell, whose lists hold cell numbers beyond 16 bits.  Rates against the
oracle (1e-12 norm-wise per column, as in test_gpu_parity.py) and the evaluated pairs against its
neighbour relation, at the build of the lists and on the lists as they are."""
import math

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

RTOL = 1e-12


def check(tp, orc, semi, fluid, wall, v, u):
    import torch
    nd = u.shape[1]
    R = 2 * fluid.smoothing_length
    xw = wall.coordinates.T.copy() if wall is not None else None
    mw = wall.boundary_model.hydrodynamic_mass if wall is not None else None
    ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, xw, mw)
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    for repeat in range(2):
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(nd + 1):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            assert err <= RTOL, f"column {col}, kick {repeat}: {err:.3e}"
        for pair, xa, xb in ((tp.native.PAIR_FLUID_FLUID, u, u), (tp.native.PAIR_FLUID_WALL, u, xw),
                             (tp.native.PAIR_WALL_FLUID, xw, u)):
            if xa is None or xb is None:
                continue
            off, _ = tp.kick_pairs(semi, pair)
            roff, _ = orc.neighbors(nd, R, xa, xb)
            itself = 1 if pair == tp.native.PAIR_FLUID_FLUID else 0  # the kick leaves it out
            assert np.array_equal(np.diff(off) + itself, np.diff(roff)), f"pair {pair}, kick {repeat}"


@pytest.mark.parametrize("length,xdiv", [(420.0, 0), (215.0, 8)])
def test_long_flume(tp, orc, length, xdiv):
    db = tp.dam_break(2, 0.02, fluid_size=(length, 0.12), tank_size=(length, 0.2))
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, x_cell_divisions=xdiv)
    lo, hi = semi.domain
    R = 2 * db.fluid_system.smoothing_length
    assert (hi[0] - lo[0]) / (1.05 * R / (xdiv or 4)) > 32767
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    v[:, :2] = np.random.default_rng(5).normal(0.0, 0.3, size=(v.shape[0], 2))
    check(tp, orc, semi, db.fluid_system, db.boundary_system, v, u)
    semi.close()


@pytest.mark.parametrize("nd,n", [(2, (60, 20)), (3, (30, 9, 8))])
def test_blocks_along_a_long_box(tp, orc, nd, n):
    dx = 0.02
    g = (0.0, -9.81) if nd == 2 else (0.0, -9.81, 0.0)
    se = tp.StateEquationCole(sound_speed=20 * math.sqrt(9.81 * 0.6), reference_density=1000.0,
                              exponent=7.0, clip_negative_pressure=False)
    ic = tp.RectangularShape(dx, n, (0.0,) * nd, density=1000.0, coordinates_perturbation=0.01, seed=3)
    fluid = tp.WeaklyCompressibleSPHSystem(
        ic, tp.ContinuityDensity(), se, tp.WendlandC2Kernel(nd), 1.2 * dx, acceleration=g,
        viscosity=tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0),
        density_diffusion=tp.DensityDiffusionMolteniColagrossi(delta=0.1))
    cell = 2.4 * dx * 1.04 / 8                       # with the default skin
    length = 40000 * cell
    lo = [-0.1] * nd
    hi = [length] + [0.3] * (nd - 1)
    semi = tp.Semidiscretization(fluid, x_cell_divisions=8, domain=(lo, hi))
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(5)
    v[:, :nd] = rng.normal(0.0, 0.3, size=(v.shape[0], nd))
    width = n[0] * dx
    starts = (0.0, 32768 * cell - 0.1 - width / 6, length - width / 3 - 0.1)
    third = np.minimum((u[:, 0] / (width / 3)).astype(int), 2)
    u[:, 0] += np.array(starts)[third] - third * (width / 3)
    assert third.min() == 0 and third.max() == 2
    check(tp, orc, semi, fluid, None, v, u)
    semi.close()
