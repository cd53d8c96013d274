"""The phase-contrast voxel update in its two workgroup widths (k_icd_lines_pc: 16 waves
a line up to a line per CU, 4 above) against the oracle's, slices z mod 3 = 0, 1, 2 in
turn: those of one turn share neither detector rows nor prior terms.  Tolerances are
the line kernel's: the FP32 sums of theta run in another order, 1e-4 of the largest
value."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from conftest import TINY
from test_gpu_phase_contrast import _pair, make_pc_scan, pc  # noqa: F401
from timbir_python_amd import xt_abi, xt_hip

pytestmark = pytest.mark.gpu

# 8, 16, 32 and 64 row lanes; fewer views than view groups; voxels of two bins, whose
# footprints reach the last candidate bins
CFGS = [dataclasses.replace(TINY, name="pc_nz5", N_z=5, num_threads=5, seed=41),
        dataclasses.replace(TINY, name="pc_nz12", N_z=12, num_threads=4, seed=42),
        dataclasses.replace(TINY, name="pc_nz20", N_z=20, N_p=7, num_threads=10, seed=43),
        dataclasses.replace(TINY, name="pc_nz40", N_xy=16, N_z=40, N_p=24, num_threads=8, seed=44),
        dataclasses.replace(TINY, name="pc_two", N_xy=16, mult_xy=2.0, num_threads=2, seed=45)]


@pytest.mark.parametrize("cfg", CFGS, ids=lambda c: c.name)
@pytest.mark.parametrize("lines", [1, 300])
@pytest.mark.parametrize("parity,Iter", [(0, 1), (1, 2)])
def test_pc_pass_per_voxel(parity, Iter, lines, cfg, pc, scan_root, oracle32, oracle64a):  # noqa: F811
    print(f"[gpu] phase-contrast pass {cfg.name} lines={lines} parity={parity}", flush=True)
    path, info = make_pc_scan(cfg, scan_root, oracle64a, "pcgrp")
    eng, (S, O, T) = _pair(cfg, path, oracle32)
    xt_hip.set_option(xt_hip.OPT_PASS, 2)
    xt_hip.set_option(xt_hip.OPT_LINES, lines)
    try:
        vol = (0.7 * info["phantom"]).astype(np.float32)
        vol[:, :, :4, :] = 0  # zero rows: zero-skipping paths
        H = oracle32.detector_response(S, O, T)
        E = np.zeros((S.N_p, S.N_r, S.N_t), np.float32)
        et, ht = xt_abi.PtrTree(E), xt_abi.PtrTree(H)
        oracle32.set_object(O, vol)
        eng.set_volume(vol)
        oracle32.lib.oracle_init_error_sino(C.byref(S), C.byref(O), C.byref(T), ht.ptr, et.ptr)
        Eg = E.copy()
        bs, nb = O.N_z // T.num_z_blocks, T.num_z_blocks
        zs = [z for z in range(O.N_z) if (min(z // bs, nb - 1) & 1) == parity]
        zs.sort(key=lambda z: (z % 3, z))
        rng = np.random.default_rng(Iter)
        tot_o = tot_g = 0.0
        for n in range(12):
            # the centre, the first column and the zero rows among them
            y, x = [(O.N_y // 2, O.N_x // 2), (O.N_y // 2, 0), (1, O.N_x // 2)][n] if n < 3 else (
                rng.integers(0, O.N_y), rng.integers(0, O.N_x))
            ys, xs = np.array([y], np.int32), np.array([x], np.int32)
            for z in zs:
                mb = np.zeros((O.N_y, O.N_x), np.float32)
                mt, zc = xt_abi.PtrTree(mb), C.c_int64(0)
                tot_o += oracle32.lib.oracle_update_lines(
                    C.byref(S), C.byref(O), C.byref(T), et.ptr, ht.ptr, 0, z, z, 1,
                    xs.ctypes.data, ys.ctypes.data, Iter, C.byref(zc), mt.ptr, 0)
            tot_g += xt_hip.update_lines_parity(eng, Eg, xs, ys, Iter, parity)[1]
        xo, xg = oracle32.get_object(O), eng.volume()
        scale = np.abs(xo).max()
        print(f"  max |dx| {np.abs(xg - xo).max() / scale:.3e} e {np.abs(Eg - E).max():.3e}")
        assert np.abs(xo - vol).max() > 1e-3 * scale
        assert np.abs(xg - xo).max() <= 1e-4 * scale
        assert np.abs(Eg - E).max() <= 1e-4 * np.abs(E).max()
        assert abs(tot_g - tot_o) <= 1e-4 * abs(tot_o)
    finally:
        xt_hip.set_option(xt_hip.OPT_PASS, 0)
        xt_hip.set_option(xt_hip.OPT_LINES, 0)
        eng.close()
        oracle32.free(S, O, T)
