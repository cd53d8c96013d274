"""The filtered backprojection where its kernels' splits end: bins not a multiple of the
filter's 16 (and fewer than 16), 4 and 1 slices per thread, idle slice lanes, fewer
views than the ring guess's 8 view groups.  Against oracle/fbp_oracle.py as at the
other sizes: FP32 sums in another order, 1e-4 of the largest value."""
import dataclasses

import numpy as np
import pytest

from conftest import TINY, make_scan
from test_gpu_fbp import host_fbp
from timbir_python_amd import xt_hip

pytestmark = pytest.mark.gpu

CFGS = [dataclasses.replace(TINY, name="fbp_b12", N_xy=12, N_z=5, N_p=5, num_threads=1, seed=51),
        dataclasses.replace(TINY, name="fbp_b30", N_xy=30, N_z=12, N_p=33, num_threads=4, seed=52),
        dataclasses.replace(TINY, name="fbp_b97", N_xy=97, N_z=20, N_p=64, num_threads=2, seed=53),
        dataclasses.replace(TINY, name="fbp_z64", N_xy=20, N_z=64, N_p=24, num_threads=8, seed=54)]


@pytest.mark.parametrize("cfg", CFGS, ids=lambda c: c.name)
def test_fbp_edges(cfg, scan_root):
    path, _ = make_scan(cfg, scan_root, "fbpedge")
    print(f"[gpu] fbp {cfg.name}", flush=True)
    with xt_hip.Engine(path, cfg.cli_args()) as eng:
        want = host_fbp(eng)
        with xt_hip.Icd(eng) as icd:
            icd.fbp()
            icd.download()
        got = eng.volume()
    err = np.abs(got - want).max() / np.abs(want).max()
    print(f"  max |gpu - oracle| / max |oracle| = {err:.2e}")
    assert err <= 1e-4
