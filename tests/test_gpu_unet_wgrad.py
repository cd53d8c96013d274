"""The network's gradients where the weight-gradient kernel's tiles (8 voxels along d1,
8 x 8 or 16 x 4 over d0 and d2) end inside, at and beyond the volume, on every level,
against oracle/unet_oracle.py.  Tolerances are those of the 16 x 16 x 8 case: GPU and
oracle differ by FP32 summation order and the bf16 rounding flips it causes, relative
L2 error <= 3e-2 for a block's gradient and 1e-3 for the loss; the outermost voxels of
these volumes carry a tenth of a gradient or more."""
import numpy as np
import pytest

import unet_oracle as uo
from test_gpu_unet import SCALE, _params, _volume, rel
from timbir_python_amd import xt_hip

pytestmark = pytest.mark.gpu


# 8x24x40: rounding flips in the forward pass reach 3.05e-2 in one block of the coarsest
# level (15 voxels), the same with a kernel that gathers every operand from memory; the
# two kernels' gradients differ by 2.1e-7 there
@pytest.mark.parametrize(
    "shape", [(8, 8, 8), (24, 40, 8), (40, 8, 24),
              pytest.param((8, 24, 40), marks=pytest.mark.xfail(reason="forward rounding flips")),
              (72, 16, 16)], ids=lambda s: "x".join(map(str, s)))
def test_gradients_at_tile_edges(shape):
    print(f"[gpu] unet gradients {shape}", flush=True)
    p = _params(6)
    x, t = _volume(7, shape)
    with xt_hip.UNet(shape, SCALE, seed=0, train=True) as net:
        net.set_params(p)
        loss, g = net.loss_grad(x, t, want_grad=True)
    wl, wg = uo.UNet(p, SCALE, bf16=True).loss_grad(x, t)
    assert abs(loss - wl) / wl <= 1e-3
    errs = {name: rel(g[sl], wg[sl]) for name, sl in uo.layer_slices()}
    print(f"  worst gradient block: {max(errs.items(), key=lambda e: e[1])}")
    assert max(errs.values()) <= 3e-2, errs


@pytest.mark.parametrize("shape", [(8, 8, 32), (24, 24, 16), (80, 16, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_forward_at_tile_edges(shape):
    """32, 16 and 64 voxels along d2: every width of the marching convolution's tile, rows
    past the volume, several segments of d0 (the gradients' shapes have 8 along d2).
    Relative L2 error of the network's own part <= 1e-2, as at 16 x 16 x 8."""
    print(f"[gpu] unet forward {shape}", flush=True)
    p = _params(8)
    x, _ = _volume(9, shape)
    with xt_hip.UNet(shape, SCALE, seed=0) as net:
        net.set_params(p)
        got = net.forward(x)
    want = uo.UNet(p, SCALE, bf16=True).forward(x)
    e = rel((got.astype(np.float64) - x) * SCALE, (want - x) * SCALE)
    print(f"  rel L2 of the residual: {e:.2e}")
    assert e <= 1e-2
