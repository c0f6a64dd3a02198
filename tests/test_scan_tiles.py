"""The scan over many cells: kicks of 3D dam breaks whose grids lie below and above the 2^19 cells at
which its tiles change, with the cell search (small fluids take the scan by itself there) and with
Verlet lists above 2^17 particles, twice with a rebuild, against the oracle.  Tolerance as in
test_gpu_parity.py: 1e-12 norm-wise per column."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]

RTOL = 1e-12


@pytest.mark.parametrize("dx,search", [(0.025, "cells"), (0.0175, "cells"), (0.012, "lists")])
def test_kicks_match_oracle_on_large_grids(tp, orc, dx, search):
    import torch
    db = tp.dam_break(3, dx)
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, pair_search=search)
    v0, u0 = semi.initial_state()
    v, u = v0.cpu().numpy().copy(), u0.cpu().numpy().copy()
    rng = np.random.default_rng(6)
    v[:, :3] = rng.normal(0.0, 0.3, size=(v.shape[0], 3))
    for repeat in range(2):
        ref, *_ = orc.kick(orc.params_from_semi(semi), v, u, db.fluid_system.mass,
                           db.boundary_system.coordinates.T,
                           db.boundary_system.boundary_model.hydrodynamic_mass)
        vd, ud = torch.from_numpy(v).cuda(), torch.from_numpy(u).cuda()
        dv = torch.full_like(vd, float("nan"))
        tp.kick(dv, vd, ud, {"semi": semi}, 0.0)
        semi.synchronize()
        got = dv.cpu().numpy()
        for col in range(4):
            err = np.abs(got[:, col] - ref[:, col]).max() / np.abs(ref[:, col]).max()
            assert err <= RTOL, f"column {col}, kick {repeat}: {err:.3e}"
        u = u + rng.uniform(-0.2, 0.2, size=u.shape) * dx   # beyond the skin
    semi.close()
