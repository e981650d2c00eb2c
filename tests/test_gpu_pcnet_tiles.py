"""Network gradients on images that cut the kernels' tiles: one 8 x 8 image,
levels one pixel wide, widths around the 64-pixel convolution tile and the
16, 32 and 64-pixel tiles of the weight gradient, more pixel tiles than
blocks of partial sums, and fractional masks.  Against the oracle with the
tolerances of test_gpu_pcnet.py (bf16 operands on both sides, FP32 against
FP64 sums)."""
import numpy as np
import pytest

import mdgpu
from oracle import pcnet as N
from test_gpu_pcnet import _ctx, _data, _pad4, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(8, 8), (8, 136), (136, 8), (72, 64), (64, 72), (24, 520)])
def test_gradients_on_ragged_images(H, W):
    ctx = _ctx()
    P = N.init_params(3)
    ctx.pcnet_set_params(N.flatten(P))
    x, t, _ = _data(H, W, H + W)
    mask = np.random.default_rng(1).uniform(0.0, 1.5, (H, W, 4)).astype(np.float32)
    loss = ctx.pcnet_grad(x, _pad4(t), mask)
    y, A = N.forward(P, x)
    lo, dy = N.loss_grad(y, t, mask[..., :3])
    G = N.backward(P, A, dy)
    assert abs(loss - lo) <= 2e-3 * lo
    g, o = ctx.pcnet_get_params(grads=True)[1], 0
    for (ci, co), (gw, gb) in zip(N.LAYERS, G):
        n = 9 * ci * co
        assert rel(g[o:o + n], gw) < 1e-2
        assert rel(g[o + n:o + n + co], gb) < 1e-2
        o += n + co


def test_accumulated_gradient_over_many_tiles():
    """More 128-pixel tiles than partials (blocks loop over tiles), and the
    second call adding to the first."""
    H, W = 256, 520
    ctx = _ctx()
    ctx.pcnet_set_params(N.flatten(N.init_params(4)))
    x, t, mask = _data(H, W, 9)
    m = np.repeat(mask[..., None], 4, axis=2).astype(np.float32)
    ctx.pcnet_grad(x, _pad4(t), m)
    g1 = ctx.pcnet_get_params(grads=True)[1].copy()
    ctx.pcnet_grad(x, _pad4(t), m, accumulate=True)
    g2 = ctx.pcnet_get_params(grads=True)[1]
    assert np.array_equal(g2, 2.0 * g1)          # the same sums twice, exactly doubled
    ctx2 = _ctx()
    ctx2.pcnet_set_params(N.flatten(N.init_params(4)))
    ctx2.pcnet_grad(x[::-1].copy(), _pad4(t)[::-1].copy(), m[::-1].copy())
    assert np.isfinite(ctx2.pcnet_get_params(grads=True)[1]).all()
