"""The a-trous filter's weights at the bottom of the float range, and the
tiled passes against the untiled ones bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L
from tests.test_net_gpu import as_float16

pytestmark = pytest.mark.gpu

# Films of more rows keep to the untiled passes.
MOST_TILED_ROWS = 200_000


def filtered(gpu, acc, w, h, params):
    film, out = L.Film(gpu, w, h), L.Film(gpu, w, h)
    film.upload(acc)
    L.Denoiser(gpu).run(film, out, params)
    return as_float16(out.download()).reshape(h, w, 16)


def plain_film(w, h, length, seed):
    """One surface seen under noise: averaged normals all of one length."""
    rng = np.random.default_rng(seed)
    a = np.zeros(w * h, L.ACCUM)
    a["samples"] = 1.0
    a["albedo"] = 0.5
    a["radiance"] = 0.25 + 0.5 * rng.random((w * h, 3))
    a["normal"] = np.float32(length) * np.array([0.0, 0.6, 0.8], np.float32)
    a["depth"] = 3.0
    return a


@pytest.mark.parametrize("h", [40, MOST_TILED_ROWS + 1], ids=["tiles", "untiled"])
@pytest.mark.parametrize("squared", [0.256, 0.26, 0.27, 0.285])
def test_short_averaged_normals_are_filtered(gpu, oracle, squared, h):
    """With a normal stop of 64, normals of squared length l weigh l^64, which
    stays a normal float down to l = 2^(-126/64) = 0.2555; the kernel's factor
    of at least 2^-8 leaves a subnormal. All 25 taps count there.

    The luminance stop is far above the colours' spread, so a pass's taps have
    the kernel's weights up to 1e-3, times one common factor. A weight is off
    by the rounding of an exponent near 126 (1e-5 of itself) and by at most
    2^-150 as a subnormal, against a sum of at least 0.47 * 2^-126 (a
    corner's); 25 of these are 6e-6 of the sum. With a colour spread of 1 and
    as much for the oracle, four passes stay below 1.3e-4. A pixel left as it
    was differs by some 0.3."""
    w = 7
    print(f"a-trous case {w}x{h}, squared normals {squared}", flush=True)
    acc = plain_film(w, h, np.sqrt(squared), 7)
    p = L.DenoiseParams(4, 64.0, 0.08, 1.0e4, 0.1)
    got = filtered(gpu, acc, w, h, p)
    rows = min(h, 140)  # the oracle's; those that see its end are left out
    a = as_float16(acc).reshape(h, w, 16)[:rows]
    want = oracle.denoise(a[..., 0:3], a[..., 4:7], a[..., 8:11], a[..., 7], p)
    seen = slice(0, rows if rows == h else rows - 31)
    assert np.abs(want - a[..., 0:3])[seen].max() > 0.1, "the oracle filters"
    assert np.abs(got[..., 0:3][:rows] - want)[seen].max() <= 2.5e-4


@pytest.mark.parametrize("iterations,sigmas", [(1, (64.0, 0.08, 4.0, 0.1)), (4, (64.0, 0.08, 4.0, 0.1)),
                                               (6, (64.0, 0.08, 4.0, 0.1)), (4, (128.0, 1.0, 0.5, 0.02)),
                                               (4, (0.5, 0.01, 40.0, 10.0))])
def test_tiles_equal_the_untiled_passes(gpu, iterations, sigmas):
    """The same rows in a film that is tiled and in one that is too tall for
    tiles: every bit the same, away from the rows that see the extra ones."""
    w, h = 9, MOST_TILED_ROWS
    print(f"a-trous case {w} x {h} and {h + 1}, {iterations} passes, stops {sigmas}", flush=True)
    rng = np.random.default_rng(11)
    n = w * (h + 1)
    y, x = np.divmod(np.arange(n), w)
    a = np.zeros(n, L.ACCUM)
    a["samples"] = 1.0 + (x + y) % 4
    spp = a["samples"].astype(np.float64)[:, None]
    facet = np.stack([np.sin(y // 37 + 0.2 * x), np.cos(y // 11), 1.5 + 0 * x], -1)
    facet /= np.linalg.norm(facet, axis=1, keepdims=True)
    length = 0.5 + 0.5 * rng.random((n, 1)) ** 0.2
    a["normal"] = facet * length * (rng.random((n, 1)) > 0.01) * spp
    a["albedo"] = (0.05 + 0.9 * ((y // 13 + x // 3) % 5 / 4.0))[:, None] * spp * np.array([1.0, 0.7, 0.4])
    a["depth"] = (2.0 + np.sin(y / 50.0) + 0.05 * rng.random(n)) * spp[:, 0]
    light = (1.0 + np.cos(y / 9.0) + 0.02)[:, None] * rng.gamma(2.0, 0.5, (n, 3))
    a["radiance"] = light * a["albedo"]
    p = L.DenoiseParams(iterations, *sigmas)
    tiled = filtered(gpu, a[:w * h], w, h, p)
    untiled = filtered(gpu, a, w, h + 1, p)
    reach = 2 * (2 ** iterations - 1) + 1  # of the passes, and of the deviation
    same = slice(0, h - reach)
    assert np.isfinite(tiled).all()
    np.testing.assert_array_equal(tiled[same].view(np.uint32), untiled[same].view(np.uint32))


@pytest.mark.parametrize("sigmas", [(64.0, -4.0e-39, 4.0, 0.1), (64.0, 0.08, -40.0, 0.1), (64.0, 0.08, 4.0, -1.0)],
                         ids=["depth", "luminance", "albedo"])
def test_stops_that_are_not_positive(gpu, oracle, sigmas):
    """They are accepted and take the untiled passes: as part of a tile a pixel
    outside the film could get a weight (the depth stop's term there, 10 over
    -4e-38, is infinite, where every pixel of this film has none). One surface
    of one depth and albedo, so the taps' weights are the kernel's times the
    luminance stop's; bounds as for films of any kind: a weight off by 2e-5 of
    itself, a pass's mean by twice that of the largest colour."""
    w, h = 20, 13
    print(f"a-trous case {w}x{h}, stops {sigmas}", flush=True)
    acc = plain_film(w, h, 1.0, 3)
    acc["depth"] = 10.0
    p = L.DenoiseParams(4, *sigmas)
    got = filtered(gpu, acc, w, h, p)
    a = as_float16(acc).reshape(h, w, 16)
    want = oracle.denoise(a[..., 0:3], a[..., 4:7], a[..., 8:11], a[..., 7], p)
    assert np.isfinite(want).all() and np.abs(want - a[..., 0:3]).max() > 0.1
    assert np.abs(got[..., 0:3] - want).max() <= 5e-4 * np.abs(want).max()
