"""The brick kernels' pipeline over bricks and their pair terms, against the oracle: fewer
bricks than blocks, one brick for some blocks and two for others, several per block; every
viscosity form; both density calculators; pairs that the relation leaves out (coincident
particles and particles closer than sqrt(eps) R).  Tolerance as in test_gpu_parity.py: 1e-12
norm-wise per column."""
import math

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

RTOL = 1e-12


def fluid_block(tp, nd, n_per_dim, viscosity, summation=False, diffusion=None, dx=0.02, seed=3):
    g = (0.0, -9.81) if nd == 2 else (0.0, -9.81, 0.0)
    se = tp.StateEquationCole(sound_speed=20 * math.sqrt(9.81 * 0.6), reference_density=1000.0,
                              exponent=7.0, clip_negative_pressure=False)
    ic = tp.RectangularShape(dx, n_per_dim, (0.0,) * nd, density=1000.0,
                             coordinates_perturbation=0.01, seed=seed)
    return tp.WeaklyCompressibleSPHSystem(
        ic, tp.SummationDensity() if summation else tp.ContinuityDensity(), se,
        tp.WendlandC2Kernel(nd), 1.2 * dx, acceleration=g, viscosity=viscosity,
        density_diffusion=diffusion or tp.DensityDiffusionMolteniColagrossi(delta=0.1))


VISCOSITY = {"none": None, "alpha": dict(alpha=0.02, beta=0.0), "beta": dict(alpha=0.02, beta=1.5)}


# bricks of about 6.9 x 7.5 x 7.5 (3D) or 20 x 20 (2D) spacings, smaller ones for fluids that
# would not fill 256 blocks with these (below about 74,000 or 77,000 particles)
@pytest.mark.parametrize("nd,n,visc,kind", [
    (3, (5, 4, 3), "alpha", "continuity"),
    (3, (30, 23, 16), "none", "continuity"),
    (3, (30, 23, 16), "beta", "continuity"),
    (3, (48, 48, 48), "alpha", "continuity"),      # 343 bricks and more: up to two per block
    (3, (70, 60, 60), "alpha", "continuity"),      # three and more per block
    (3, (48, 48, 48), "beta", "summation"),
    (3, (30, 23, 16), "none", "summation"),
    (3, (44, 42, 39), "alpha", "continuity"),      # just below and above full bricks
    (3, (44, 42, 41), "alpha", "continuity"),
    (3, (48, 48, 48), "alpha", "antuono"),
    (2, (37, 21), "beta", "continuity"),
    (2, (420, 380), "alpha", "continuity"),        # 399 bricks and more
    (2, (420, 380), "none", "summation"),
    (2, (120, 90), "beta", "antuono"),
    (2, (300, 250), "alpha", "continuity"),
])
def test_bricks_match_oracle(tp, orc, nd, n, visc, kind):
    import torch
    kw = VISCOSITY[visc]
    fluid = fluid_block(tp, nd, n, tp.ArtificialViscosityMonaghan(**kw) if kw else None,
                        summation=kind == "summation",
                        diffusion=tp.DensityDiffusionAntuono(delta=0.1) if kind == "antuono" else None)
    semi = tp.Semidiscretization(fluid)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(21)
    v[:, :nd] = rng.normal(0.0, 0.5, size=(v.shape[0], nd))
    if v.shape[1] > nd:
        v[:, nd] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=v.shape[0])
    if kind == "continuity":
        u[1] = u[0]                            # coincident
        u[3] = u[2] + 1e-10 * 2 * fluid.smoothing_length
    dv_ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    for repeat in range(2):                    # with the rebuild, then on the lists as they are
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(got.shape[1]):
            err = np.abs(got[:, col] - dv_ref[:, col]).max() / np.abs(dv_ref[:, col]).max()
            assert err <= RTOL, f"column {col}, kick {repeat}: {err:.3e}"
    semi.close()


# cells per compact support along y and z / x, skin: short and long rows, one and four cells of
# reach, lists of up to about 200 entries, and (3D, three cells) bricks that do not stage
@pytest.mark.parametrize("nd,dx,div,xdiv,skin", [
    (2, 0.02, 1, 1, 0.04), (2, 0.02, 4, 8, 0.04), (2, 0.02, 2, 3, 0.6),
    (3, 0.04, 1, 1, 0.04), (3, 0.04, 1, 8, 0.04), (3, 0.04, 2, 8, 0.04), (3, 0.04, 2, 1, 0.04),
    (3, 0.04, 2, 4, 0.45), (3, 0.04, 3, 4, 0.04),
])
def test_listed_pairs_match_bruteforce(tp, orc, nd, dx, div, xdiv, skin):
    import torch
    db = tp.dam_break(nd, dx)
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, cell_divisions=div,
                                 x_cell_divisions=xdiv, skin=skin, pair_search="lists")
    v0, u0 = semi.initial_state()
    u = u0.cpu().numpy().copy()
    rng = np.random.default_rng(4)
    R = 2 * db.fluid_system.smoothing_length
    u += rng.uniform(-0.3, 0.3, size=u.shape) * dx     # a disordered fluid
    dv = torch.empty_like(v0)
    move = rng.normal(size=u.shape)
    move *= 0.45 * skin * R / np.linalg.norm(move, axis=1, keepdims=True)
    xw = db.boundary_system.coordinates.T.copy()
    for x in (u, u + move):                            # the build, then within half the skin
        tp.kick(dv, v0, torch.from_numpy(x).cuda(), {"semi": semi}, 0.0)
        for pair, xa, xb in ((tp.native.PAIR_FLUID_FLUID, x, x), (tp.native.PAIR_FLUID_WALL, x, xw),
                             (tp.native.PAIR_WALL_FLUID, xw, x)):
            off, idx = tp.kick_pairs(semi, pair)
            roff, ridx = orc.neighbors(nd, R, xa, xb, brute=True)
            if pair == tp.native.PAIR_FLUID_FLUID:     # the kick leaves the particle itself out
                rows = np.repeat(np.arange(roff.size - 1), np.diff(roff))
                keep = rows != ridx
                roff = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=roff.size - 1))])
                ridx = ridx[keep]
            assert np.array_equal(off, roff), f"pair {pair}: counts differ"
            assert np.array_equal(idx.astype(np.int64), ridx), f"pair {pair}: sets differ"
    semi.close()
