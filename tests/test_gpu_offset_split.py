"""The ring-offset update at the edges of its split (view chunks of 8 or more, 32 or 256
pixels a combine workgroup) against the formula in 64 bits (F/XT_ICD_update.c:666-759).
The sums are FP64; e and d are rounded to float32 once, so 4 ulps of their largest value
bound the difference."""
import numpy as np
import pytest

from test_zz_no_alloc import _Hip
from timbir_python_amd import xt_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 3, 1), (7, 5, 7), (8, 33, 1), (57, 31, 2), (64, 32, 8),
                                   (65, 257, 3), (90, 4100, 8), (40, 8192, 5)])
@pytest.mark.parametrize("zero_mean", [True, False])
def test_offset_split(shape, zero_mean):
    rng = np.random.default_rng(shape[1])
    w = rng.uniform(1e3, 1e4, shape).astype(np.float32)
    e = (rng.standard_normal(shape) / np.sqrt(w)).astype(np.float32)
    e[rng.random(shape) < 0.02] += 1.0
    d = rng.uniform(-0.01, 0.01, shape[1:]).astype(np.float32)
    E, W, D = e.astype(float), w.astype(float), d.astype(float)
    small = E * E * W < 16.0
    num = np.where(small, E * W, 0.4 * np.sqrt(W) * np.sign(E)).sum(0)
    den = np.where(small, W, 0.4 * np.sqrt(W) / np.abs(E)).sum(0)
    gamma = (D + num / den).sum() / (1 / den).sum() if zero_mean else 0.0
    step = (num - gamma) / den
    hip = _Hip()
    try:
        te, tw, td = (hip.upload(a) for a in (e, w, d))
        xt_hip.offset_update_noalloc(*shape, 4.0, 0.1, zero_mean, te, tw, td)
        eg, dg = hip.download(te, e), hip.download(td, d)
    finally:
        hip.free()
    ulp = np.finfo(np.float32).eps
    assert np.abs(eg - (E - step)).max() <= 4 * ulp * np.abs(E - step).max()
    assert np.abs(dg - (D + step)).max() <= 4 * ulp * np.abs(D + step).max()
