"""The batched voxel-update passes (k_icd_plane, k_icd_step: XT_OPT_PASS 2) against the
oracle's voxel update on the same lines.

One line per step is the reference's sequential loop; n lines per step all read the
same error sinogram, so each line's change is the oracle's for that line alone and e
takes the sum of their changes.  Tolerances are the line kernel's per-voxel ones: the
FP32 sums of theta run in another order, 1e-4 of the largest value."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from conftest import SMALL, TINY
from test_gpu_parity import NZ32, NZ64, WIDE3, WIDE6, _pair, _print_case
from timbir_python_amd import xt_abi, xt_hip

pytestmark = pytest.mark.gpu

# an odd number of one-slice blocks; a last block of four slices; blocks of two slices;
# the detector a bin wider than a multiple of the 64 bins a workgroup takes at a time
ODD5 = dataclasses.replace(TINY, name="odd5", N_z=5, num_threads=5, seed=31)
LAST4 = dataclasses.replace(TINY, name="last4", N_z=7, num_threads=2, seed=32)
WIDE65 = dataclasses.replace(TINY, name="bins129", N_xy=86, N_p=30, N_z=4, num_threads=1, seed=33)


def _slices(O, T, parity):
    """The parity's slices in the order of the update: red-black, even slices first (the
    slices of a line share no sinogram entries)."""
    nb = T.num_z_blocks
    bs = O.N_z // nb
    zs = [z for z in range(O.N_z) if (min(z // bs, nb - 1) & 1) == parity]
    return [z for z in zs if z % 2 == 0] + [z for z in zs if z % 2]


# SMALL without its table and the voxels wider than two bins: columns computed in the pass
@pytest.mark.parametrize("cfg,atable", [(c, 1) for c in (TINY, SMALL, NZ32, NZ64, ODD5, LAST4, WIDE65,
                                                          WIDE3, WIDE6)] + [(SMALL, 0)],
                         ids=lambda c: getattr(c, "name", f"atable{c}"))
@pytest.mark.parametrize("lines", [1, 20])
@pytest.mark.parametrize("parity,Iter", [(0, 1), (1, 2)])
def test_batched_pass_per_voxel(parity, Iter, lines, cfg, atable, scan_root, oracle32):
    _print_case(f"batched pass lines={lines} parity={parity} Iter={Iter}", cfg)
    path, info, eng, (S, O, T) = _pair(cfg, scan_root, oracle32)
    xt_hip.set_option(xt_hip.OPT_PASS, 2)
    xt_hip.set_option(xt_hip.OPT_LINES, lines)
    xt_hip.set_option(xt_hip.OPT_ATABLE, atable)
    try:
        vol = (0.7 * info["phantom"]).astype(np.float32)
        vol[:, :, :4, :] = 0  # zero rows: zero-skipping paths
        oracle32.set_object(O, vol)
        eng.set_volume(vol)
        H = oracle32.detector_response(S, O, T)
        E0 = np.zeros((S.N_p, S.N_r, S.N_t), np.float32)
        e0, ht = xt_abi.PtrTree(E0), xt_abi.PtrTree(H)
        oracle32.lib.oracle_init_error_sino(C.byref(S), C.byref(O), C.byref(T), ht.ptr, e0.ptr)
        rng = np.random.default_rng(Iter)
        # lines at least two apart: those of one step are no neighbours of one another
        ys, xs = (a.ravel() for a in np.meshgrid(np.arange(0, O.N_y, 2), np.arange(1, O.N_x, 2)))
        pick = rng.permutation(ys.size)[:lines if lines > 1 else 30]
        ys, xs = ys[pick].astype(np.int32), xs[pick].astype(np.int32)
        Eo, xo = E0.astype(np.float64), vol.copy()
        tot_o = 0.0
        E = E0.copy()
        et = xt_abi.PtrTree(E)
        for i in range(len(ys)):
            if lines > 1:  # every line of the step from the same start
                E[:] = E0
                oracle32.set_object(O, vol)
            before = E.astype(np.float64)
            for z in _slices(O, T, parity):
                mb = np.zeros((O.N_y, O.N_x), np.float32)
                mt, zc = xt_abi.PtrTree(mb), C.c_int64(0)
                tot_o += oracle32.lib.oracle_update_lines(
                    C.byref(S), C.byref(O), C.byref(T), et.ptr, ht.ptr, 0, z, z, 1,
                    xs[i:].ctypes.data, ys[i:].ctypes.data, Iter, C.byref(zc), mt.ptr, 0)
            Eo += E.astype(np.float64) - before
            xo[0, :, ys[i], xs[i]] = oracle32.get_object(O)[0, :, ys[i], xs[i]]
        Eg = E0.copy()
        mag_g, tot_g = xt_hip.update_lines_parity(eng, Eg, xs, ys, Iter, parity)
        xg = eng.volume()
        scale = np.abs(xo).max()
        print(f"  max |dx| {np.abs(xg - xo).max() / scale:.3e} e {np.abs(Eg - Eo).max():.3e}")
        assert np.abs(xo - vol).max() > 1e-3 * scale
        on = np.isin(np.arange(O.N_z), _slices(O, T, parity))
        assert np.array_equal(xg[:, ~on], vol[:, ~on])
        assert np.abs(xg - xo).max() <= 1e-4 * scale
        assert np.abs(Eg - Eo).max() <= 1e-4 * np.abs(Eo).max()
        # the update map holds each line's changes as the volume shows them (the changes are
        # a thousandth of the voxels, so the oracle's own are known to a few of their ulps only)
        np.testing.assert_allclose(mag_g, np.abs(xg - vol)[0].sum(0), rtol=1e-5, atol=1e-12)
        assert abs(tot_g - tot_o) <= 1e-4 * abs(tot_o)
    finally:
        xt_hip.set_option(xt_hip.OPT_PASS, 0)
        xt_hip.set_option(xt_hip.OPT_LINES, 0)
        xt_hip.set_option(xt_hip.OPT_ATABLE, 1)
        eng.close()
        oracle32.free(S, O, T)
