"""Walls without fluid through the C ABI: the kick of such a handle gives every wall particle the
values of empty Adami sums, as the oracle does, with Verlet lists and cells, also after a handle
with fluid has left its contents in the device's memory; and tpsph_kick_noalloc accepts it."""
import ctypes as C

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X")]


@pytest.mark.parametrize("nd,dx", [(2, 0.02), (3, 0.06)])
@pytest.mark.parametrize("search", ["lists", "cells"])
def test_walls_without_fluid(tp, orc, nd, dx, search):
    import torch
    lib = tp.native.load()
    db = tp.dam_break(nd, dx)
    semi = tp.Semidiscretization(db.fluid_system, db.boundary_system, pair_search=search)
    v, u = semi.initial_state()
    dv = torch.empty_like(v)
    tp.kick(dv, v, u, {"semi": semi}, 0.0)
    semi.synchronize()
    P = orc.params_from_semi(semi)
    p = semi.params()
    semi.close()

    xw = np.ascontiguousarray(db.boundary_system.coordinates.T)
    mw = np.ascontiguousarray(db.boundary_system.boundary_model.hydrodynamic_mass)
    _, _, pw_ref, rw_ref = orc.kick(P, np.zeros((0, nd + 1)), np.zeros((0, nd)), np.zeros(0), xw, mw)
    wx, wm = torch.from_numpy(xw).cuda(), torch.from_numpy(mw).cuda()
    h = C.c_void_p()
    tp.native.check(lib.tpsph_create(C.byref(p), 0, db.n_wall, None, wx.data_ptr(), wm.data_ptr(),
                                     None, C.byref(h)))
    for _ in range(2):
        tp.native.check(lib.tpsph_kick(h, None, None, None, 0.0), h)
        pw, rw = np.full(db.n_wall, np.nan), np.full(db.n_wall, np.nan)
        tp.native.check(lib.tpsph_get_pressures(h, None, pw.ctypes.data, rw.ctypes.data), h)
        assert np.array_equal(pw, pw_ref)
        assert np.abs(rw - rw_ref).max() <= 1e-12 * np.abs(rw_ref).max()
    off = np.full(db.n_wall + 1, -1, dtype=np.int64)
    tp.native.check(lib.tpsph_kick_pairs_csr(h, tp.native.PAIR_WALL_FLUID, off.ctypes.data, None, 0), h)
    assert not off.any()
    lib.tpsph_destroy(h)

    rc = lib.tpsph_kick_noalloc(C.byref(p), 0, db.n_wall, None, wx.data_ptr(), wm.data_ptr(), None,
                                None, None, 0.0, None)
    assert rc == 0, lib.tpsph_last_error(None).decode()
    torch.cuda.synchronize()
