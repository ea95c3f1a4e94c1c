"""The network's kernels one by one, at the sizes where their tilings can go
wrong: each layer's result recomputed in float64 from the tensors the device
itself stored, so only that kernel's own accumulation remains."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L
from oracle import net as N
from tests.test_net_gpu import films, random_params, say

pytestmark = pytest.mark.gpu

LAYER_INPUT = ["x", "l0", "p0", "l2", "p1", "l4", "p2", "l6", "c2", "l8", "c1", "l10", "c0", "l12", "l13"]

# (crop width, height, crops): the coarsest level 16 pixels wide and one row
# high; 48 pixels wide; heights that end inside a tile at every level; several
# tiles per slice.
SHAPES = [(128, 8, 1), (128, 24, 3), (256, 40, 2), (384, 8, 2), (512, 136, 4)]


def run_backward(gpu, w, h, n, seed):
    ins, _ = films(gpu, w, h, [seed + k for k in range(n)])
    refs, _ = films(gpu, w, h, [seed + 50 + k for k in range(n)])
    net = L.LearnedDenoiser(gpu, seed=seed)
    net.set_params(random_params(seed))
    say(f"net kernels case: {n} crops {w}x{h}")
    net.forward_backward(ins, refs, w, h)
    acts = N.activations_from_layers(net.tensor(0).astype(np.float64), [net.tensor(i + 1) for i in range(15)], bf16=True)
    return net, acts


@pytest.mark.parametrize("w,h,n", SHAPES)
def test_weight_gradients_of_stored_tensors(gpu, w, h, n):
    """dW and db of every layer against the same sums in float64. The device
    adds exact BF16 products in FP32 along chains of fewer than 256 additions
    (tiles of a slice, shares of a tile, slices), each off by at most 2^-24 of
    the partial sum, which is at most the sum of the terms' magnitudes."""
    net, acts = run_backward(gpu, w, h, n, 61)
    grads = net.params(gradients=True).astype(np.float64)
    off = 0
    for i, (ci, co, _) in enumerate(N.LAYERS):
        x = acts[LAYER_INPUT[i]]
        d = net.tensor(i + 1, gradient=True).astype(np.float64)
        _, hh, ww, _ = d.shape
        pad = np.pad(x, ((0, 0), (1, 1), (1, 1), (0, 0)))
        dm = d.reshape(-1, co)
        for t in range(9):
            xs = pad[:, t // 3:t // 3 + hh, t % 3:t % 3 + ww].reshape(-1, ci)
            got = grads[off + t * ci * co:off + (t + 1) * ci * co].reshape(ci, co)
            bound = 2.0 ** -16 * (np.abs(xs).T @ np.abs(dm)) + 1e-30
            worst = np.max(np.abs(got - xs.T @ dm) / bound)
            assert worst <= 1.0, (i, t, worst)
        off += 9 * ci * co
        assert np.all(np.abs(grads[off:off + co] - dm.sum(0)) <= 2.0 ** -16 * np.abs(dm).sum(0) + 1e-30), i
        off += co


@pytest.mark.parametrize("w,h,n", SHAPES)
def test_convolutions_of_stored_tensors(gpu, w, h, n):
    """Every layer's output, and every gradient that the next layer's input
    gradient, pools and concatenations make of it, recomputed in float64 from
    the tensors the device stored. BF16 rounds to 2^-9 of the value; a flip of
    that rounding, or one more rounding of a summand, adds as much again, and
    the FP32 sums of at most 1440 products 2^-13 of the terms' magnitude."""
    net, acts = run_backward(gpu, w, h, n, 71)
    params = N.unpack(net.params().astype(np.float64))
    for i, (ci, co, relu) in enumerate(N.LAYERS):
        wt, b = N.to_bf16(params[i][0]), params[i][1]
        want = N.conv3x3(acts[LAYER_INPUT[i]], wt, b)
        size = N.conv3x3(np.abs(acts[LAYER_INPUT[i]]), np.abs(wt), np.abs(b))
        if relu:
            want = np.maximum(want, 0)
        got = acts[f"l{i}"]
        assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -13 * size + 1e-30), i

    def input_grad(i):
        d = net.tensor(i + 1, gradient=True).astype(np.float64)
        back = N.to_bf16(params[i][0])[::-1].transpose(0, 2, 1)
        return N.conv3x3(d, back), N.conv3x3(np.abs(d), np.abs(back))

    skips = {}
    for i in range(14, 0, -1):
        g, size = input_grad(i)
        slack = 2.0 ** -8 * np.abs(g) + 2.0 ** -13 * size
        below = i - 1
        if i in (8, 10, 12):
            c = N.LAYERS[below][1]
            skips[i] = (g[..., c:], slack[..., c:])
            quads = lambda t: sum(t[:, y::2, x::2, :c] for y in (0, 1) for x in (0, 1))
            g, slack = quads(g), quads(slack)
        elif i in (2, 4, 6):
            up = lambda t: t.repeat(2, 1).repeat(2, 2)
            sg, ss = skips[{2: 12, 4: 10, 6: 8}[i]]
            g, slack = 0.25 * up(g) + sg, 0.25 * up(slack) + ss
        mask = acts[f"l{below}"] > 0
        got = net.tensor(below + 1, gradient=True).astype(np.float64)
        assert np.all(got[~mask] == 0), i
        assert np.all(np.abs(got - g * mask) <= (slack + 2.0 ** -8 * np.abs(g)) * mask + 1e-30), i
