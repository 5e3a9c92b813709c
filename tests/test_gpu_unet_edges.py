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


@pytest.mark.parametrize("channels,shape", [((16, 16), (12, 4, 20)), ((32, 16), (20, 12, 4))])
def test_fp32_operands_keep_their_24_bits(channels, shape):
    """The input layer's X and the output layer's dY are FP32: with one voxel of
    them nonzero a gradient is one product of BF16 and FP32, and the three BF16
    parts of the FP32 factor add up with at most two roundings (2^-23 each)."""
    import pic_gpu as pg

    ctx = pg.Context(*shape, [0, 0, 0], [1.0, 1.0, 1.0])
    ctx.unet_create(channels, seed=5)
    specs, dims, V = U.layer_specs(channels), shape[::-1], int(np.prod(shape))
    first = specs[0][1] * 54 + specs[0][1]
    last = 27 * channels[0] + 1
    rng = np.random.default_rng(V)
    at = [(0, 0, 0), tuple(n - 1 for n in dims), tuple(n // 2 for n in dims), (dims[0] // 3, 0, dims[2] - 1)]
    # input layer: with zero weights its output, and the gradient there, do not depend on x
    p = _bf16(U.init_params(channels, seed=7)).astype(np.float32)
    p[:54 * channels[0]] = 0
    p[54 * channels[0]:first] = rng.uniform(0.5, 1.0, channels[0])
    ctx.unet_set_params(p)
    t = rng.normal(size=dims).astype(np.float32)
    for v in at:
        for c in range(2):
            val = np.float32(rng.uniform(0.1, 0.9))
            g = []
            for f in (np.float32(0.5), val):
                x = np.zeros(dims + (2,), np.float32)
                x[v + (c,)] = f
                g.append(ctx.unet_loss_grad(x, t)[1][:54 * channels[0]].astype(np.float64))
            assert np.count_nonzero(g[0]) > 0
            want = g[0] / 0.5 * float(val)
            assert np.all(np.abs(g[1] - want) <= 2.0 ** -22 * np.abs(want)), (v, c)
    # output layer: constant activations h, dy = -t / V at one voxel
    p = np.zeros_like(p)
    h = _bf16(rng.uniform(0.5, 1.5, channels[0])).astype(np.float32)
    dec = p.size - last - channels[0]
    p[dec:dec + channels[0]] = h
    ctx.unet_set_params(p)
    for v in at:
        t = np.zeros(dims, np.float32)
        t[v] = rng.uniform(1.0, 2.0)
        g = ctx.unet_loss_grad(np.zeros(dims + (2,), np.float32), t)[1][-last:].astype(np.float64)
        dy = -float(t[v]) / V
        assert abs(g[-1] - dy) <= 2.0 ** -22 * abs(dy)
        inside = np.zeros(27, bool)
        for k in range(27):
            o = (v[0] + k // 9 - 1, v[1] + k // 3 % 3 - 1, v[2] + k % 3 - 1)
            inside[k] = all(0 <= a < n for a, n in zip(o, dims))
        want = np.where(inside[:, None], g[-1] * h.astype(np.float64)[None, :], 0.0)
        assert np.all(np.abs(g[:-1].reshape(27, -1) - want) <= 2.0 ** -22 * np.abs(want)), v
        t[v] = np.inf  # stays one
        g = ctx.unet_loss_grad(np.zeros(dims + (2,), np.float32), t)[1][-last:]
        assert np.all(np.isneginf(g[:-1].reshape(27, -1)[inside])) and np.isneginf(g[-1])
    ctx.close()
