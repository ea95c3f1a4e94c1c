"""The network's convolutions on a film large enough that the coarse levels take
the splits that smaller ones never reach: 65,536 pixels and more at level 3, so
waves that keep all four tiles of 64 output channels (plain, pooled, masked and
through the pool), all three of 48 through the pool, and 96 channels in pairs.
No level's height is a whole number of tiles. Bands of rows at the top, in the
middle and at the bottom are recomputed in float64 from the tensors that the
device stored."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L
from oracle import net as N
from tests.test_net_gpu import random_params, say, synthetic_accum

pytestmark = pytest.mark.gpu

W, H = 2048, 2056  # level 2: 512 x 514, level 3: 256 x 257


def bands(h):
    return [(0, 11), (h // 2 - 5, h // 2 + 6), (h - 11, h)]


def conv_rows(x, r0, r1, *weights):
    """Rows [r0, r1) of the 3 x 3 convolution of x."""
    lo = max(r0 - 1, 0)
    return N.conv3x3(x[:, lo:r1 + 1].astype(np.float64), *weights)[:, r0 - lo:r1 - lo]


@pytest.fixture(scope="module")
def net(gpu):
    film, ref = L.Film(gpu, W, H), L.Film(gpu, W, H)
    film.upload(synthetic_accum(W, H, 81))
    ref.upload(synthetic_accum(W, H, 82))
    net = L.LearnedDenoiser(gpu, seed=5)
    net.set_params(random_params(81))
    say(f"net kernels case: 1 crop {W}x{H}")
    net.forward_backward([film], [ref], W, H)
    return net


def pooled(x):
    x = x.astype(np.float64)
    return N.to_bf16(0.25 * (x[:, ::2, ::2] + x[:, ::2, 1::2] + x[:, 1::2, ::2] + x[:, 1::2, 1::2]))


def test_forward_at_the_coarse_levels(net):
    """Bounds as in the test of the small shapes: 2^-8 of the value for BF16's
    rounding and a flip of it, 2^-13 of the terms' magnitude for the sums."""
    params = N.unpack(net.params().astype(np.float64))
    out = {i: net.tensor(i + 1) for i in range(3, 10)}
    for i in range(4, 10):
        wt, b = N.to_bf16(params[i][0]), params[i][1]
        h = out[i].shape[1]
        for r0, r1 in bands(h):
            lo, hi = max(r0 - 1, 0), min(r1 + 1, h)
            if i in (4, 6):
                x = pooled(out[i - 1][:, 2 * lo:2 * hi])
            elif i == 8:
                up = out[7][:, lo // 2:(hi + 1) // 2].repeat(2, 1).repeat(2, 2)[:, lo % 2:lo % 2 + hi - lo]
                x = np.concatenate([up, out[5][:, lo:hi]], -1)
            else:
                x = out[i - 1][:, lo:hi]
            want = np.maximum(conv_rows(x, r0 - lo, r1 - lo, wt, b), 0)
            size = conv_rows(np.abs(x), r0 - lo, r1 - lo, np.abs(wt), np.abs(b))
            got = out[i][:, r0:r1]
            assert got.any(), (i, r0)
            assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -13 * size + 1e-30), (i, r0)


def test_input_gradients_at_the_coarse_levels(net):
    params = N.unpack(net.params().astype(np.float64))
    d = {i: net.tensor(i + 1, gradient=True) for i in range(3, 10)}
    for i in (9, 7, 6, 5, 4):
        back = N.to_bf16(params[i][0])[::-1].transpose(0, 2, 1)
        below, h = i - 1, d[i].shape[1]
        act = net.tensor(below + 1)
        for r0, r1 in bands(h):
            g, size = conv_rows(d[i], r0, r1, back), conv_rows(np.abs(d[i]), r0, r1, np.abs(back))
            slack = 2.0 ** -8 * np.abs(g) + 2.0 ** -13 * size
            a, b = r0, r1
            if i in (4, 6):  # through the pool, and the skip's share: the first channels are the layer below's
                a, b = 2 * r0, 2 * r1
                up = lambda t: t.repeat(2, 1).repeat(2, 2)
                skip = {6: 8, 4: 10}[i]
                sb = N.to_bf16(params[skip][0])[::-1].transpose(0, 2, 1)
                c = N.LAYERS[skip - 1][1]
                ds = d[8] if skip == 8 else net.tensor(11, gradient=True)
                sg, ss = conv_rows(ds, a, b, sb)[..., c:], conv_rows(np.abs(ds), a, b, np.abs(sb))[..., c:]
                g, slack = 0.25 * up(g) + sg, 0.25 * up(slack) + 2.0 ** -8 * np.abs(sg) + 2.0 ** -13 * ss
            mask = act[:, a:b] > 0
            got = d[below][:, a:b].astype(np.float64)
            assert np.all(got[~mask] == 0) and got.any(), (i, r0)
            assert np.all(np.abs(got - g * mask) <= (slack + 2.0 ** -8 * np.abs(g)) * mask + 1e-30), (i, r0)
