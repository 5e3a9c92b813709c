"""The weight-gradient kernels on grids whose sides are no multiples of their
8 x 4 x 4 tiles and on every channel block they have (16 or 32 output channels
by 16 or 32 input channels), against the FP64 oracle."""
import numpy as np
import pytest

import unet_oracle as U

pytestmark = pytest.mark.gpu


def _bf16(a):
    u = np.asarray(a, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    return (u.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("channels,shape", [((16, 48), (20, 12, 28)), ((32, 48), (12, 20, 4)),
                                            ((32, 64, 16), (12, 4, 20)), ((16, 16), (4, 4, 4)),
                                            ((32, 32), (36, 20, 12))])
def test_weight_gradients_at_tile_edges(channels, shape):
    import pic_gpu as pg

    ctx = pg.Context(*shape, [0, 0, 0], [1.0, 1.0, 1.0])
    ctx.unet_create(channels, seed=5)
    p = U.init_params(channels, seed=7).astype(np.float32)
    ctx.unet_set_params(p)
    rng = np.random.default_rng(sum(shape))
    dims = shape[::-1]
    x = np.stack([rng.normal(size=dims), np.zeros(dims)], axis=-1)
    t = rng.normal(size=dims)
    _, g = ctx.unet_loss_grad(x.astype(np.float32), t.astype(np.float32))
    _, ref = U.loss_grad(_bf16(p).astype(np.float64), x, t, channels)
    off = 0
    for ci, co, taps in U.layer_specs(channels):
        nw = co * taps * ci
        # activations and their gradients are rounded to BF16 (2^-8 relative)
        # in each of the layers on the way
        for a, b in ((g[off:off + nw], ref[off:off + nw]), (g[off + nw:off + nw + co], ref[off + nw:off + nw + co])):
            assert np.linalg.norm(a - b) <= 2.0 ** -8 * 16 * np.linalg.norm(b), (ci, co, taps)
        off += nw + co
    ctx.close()
