"""The a-trous filter's tiles at the sizes where they can go wrong: films
narrower than a tile or than a stride's halo, odd sides, every stride with
tiles and without, a first pass that is also the last, and the options and
heights that keep to the untiled passes."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L
from tests.test_net_gpu import as_float16, synthetic_accum

pytestmark = pytest.mark.gpu

# (width, height, iterations, sigma_normal)
CASES = [(1, 1, 4, 64.0), (3, 130, 4, 64.0), (130, 3, 4, 64.0), (64, 16, 1, 64.0), (65, 17, 2, 64.0), (127, 67, 3, 64.0),
         (200, 129, 4, 64.0), (97, 133, 6, 64.0), (70, 40, 4, 0.0), (70, 40, 5, 8.0),
         (3, 200000, 4, 64.0), (3, 200001, 4, 64.0)]


@pytest.mark.parametrize("w,h,iterations,sigma_normal", CASES)
def test_matches_the_oracle(gpu, oracle, w, h, iterations, sigma_normal):
    """A weight's exponent is off by at most about 2e-5 (64 times the hardware
    log2's 2^-22, and the rounding of terms up to 30), so a weight by 2e-5 of
    itself and a pass's weighted mean by twice that of the largest colour; the
    oracle's own floats are off as much. Six passes stay below 5e-4."""
    print(f"a-trous case {w}x{h} x {iterations}, normal stop {sigma_normal}", flush=True)
    acc = synthetic_accum(w, h, 1000 * w + h)
    film, out = L.Film(gpu, w, h), L.Film(gpu, w, h)
    film.upload(acc)
    p = L.DenoiseParams(iterations, sigma_normal, 0.08, 4.0, 0.1)
    L.Denoiser(gpu).run(film, out, p)
    got = as_float16(out.download()).reshape(h, w, 16)
    a = as_float16(acc).reshape(h, w, 16)
    inv = np.float32(1) / a[..., 3:4]
    alb = np.maximum(a[..., 4:7] * inv, np.float32(1e-3))
    nrm, dep = a[..., 8:11] * inv, a[..., 7] * inv[..., 0]
    want = oracle.denoise(a[..., 0:3] * inv, alb, nrm, dep, p)
    assert np.max(np.abs(got[..., 0:3] - want)) <= 5e-4 * np.max(np.abs(want))
    np.testing.assert_array_equal(got[..., 3], 1.0)
    np.testing.assert_array_equal(got[..., 4:7], alb)
    np.testing.assert_array_equal(got[..., 7], dep)
    np.testing.assert_array_equal(got[..., 8:11], nrm)
    assert not got[..., 11:].any()


def test_a_batch_filters_each_film_as_alone(gpu):
    """Films of uneven sizes filtered in shared launches (more than one launch
    holds) reach the network exactly as each alone."""
    sizes = [(256, 24), (128, 8), (130, 40), (300, 9)] * 5
    films = []
    for k, (w, h) in enumerate(sizes):
        f = L.Film(gpu, w, h)
        f.upload(synthetic_accum(w, h, k))
        films.append(f)
    print("a-trous case: 20 films in one batch", flush=True)
    net = L.LearnedDenoiser(gpu, seed=3)
    net.forward_backward(films, films, 128, 8)
    batch = net.tensor(0)
    for k, f in enumerate(films):
        net.forward_backward([f], [f], 128, 8)
        np.testing.assert_array_equal(net.tensor(0)[0], batch[k])
