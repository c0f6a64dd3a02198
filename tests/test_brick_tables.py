"""Bricks whose offset tables are the largest: 3D with two cell divisions and eight along x, and
DensityDiffusionAntuono with three cell divisions.  They stage (mixed precision and
SummationDensity on the lists, which need that, are accepted) whatever the number of particles,
with bricks of full size too, and the rates match the oracle: 1e-12 norm-wise per column as in
test_gpu_parity.py, the bounds of test_mixed_pairs.py for mixed precision."""
import numpy as np
import pytest

from conftest import gpu_available
from test_brick_kernel import fluid_block

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

# bricks have their full size from about 74,000 particles, in mixed precision 148,000
SMALL, FULL = (14, 12, 10), (60, 56, 56)


@pytest.mark.parametrize("n", [SMALL, FULL])
@pytest.mark.parametrize("kind,div,xdiv,precision,search", [
    ("continuity", 2, 8, "fp64", "lists"), ("continuity", 2, 8, "mixed", "auto"),
    ("summation", 2, 8, "fp64", "lists"), ("antuono", 3, 0, "fp64", "lists"),
    ("antuono", 3, 8, "fp64", "lists"),
])
def test_largest_tables_match_oracle(tp, orc, n, kind, div, xdiv, precision, search):
    import torch
    fluid = fluid_block(tp, 3, n, tp.ArtificialViscosityMonaghan(alpha=0.02, beta=0.0),
                        summation=kind == "summation",
                        diffusion=tp.DensityDiffusionAntuono(delta=0.1) if kind == "antuono" else None)
    semi = tp.Semidiscretization(fluid, cell_divisions=div, x_cell_divisions=xdiv,
                                 precision=precision, pair_search=search)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(21)
    v[:, :3] = rng.normal(0.0, 0.5, size=(v.shape[0], 3))
    if v.shape[1] > 3:
        v[:, 3] *= 1.0 + rng.uniform(-2e-3, 2e-3, size=v.shape[0])
    ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, fluid.mass, None, None)
    vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
    for repeat in range(2):                    # with the rebuild, then on the lists as they are
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(got.shape[1]):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            tol = 1e-12 if precision == "fp64" else 1e-5 if col == 3 else 1e-4
            assert err <= tol, f"column {col}, kick {repeat}: {err:.3e}"
    semi.close()


@pytest.mark.parametrize("n", [SMALL, FULL])
@pytest.mark.parametrize("kind,precision", [("continuity", "mixed"), ("summation", "fp64")])
def test_three_divisions_stay_refused(tp, n, kind, precision):
    """3D bricks with three cell divisions do not stage, so what needs them is refused, for a small
    fluid (whose bricks are smaller) too."""
    fluid = fluid_block(tp, 3, n, None, summation=kind == "summation")
    semi = tp.Semidiscretization(fluid, cell_divisions=3, precision=precision, pair_search="lists")
    with pytest.raises(tp.native.TpsphError):
        semi.handle
    semi.close()
