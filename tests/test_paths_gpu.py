"""Renders of few paths, traced a path per thread: the film and the ray counts
must be those of the wavefront stages, which a render with per-kernel times
keeps to. Sizes lie on both sides of the path count where one takes over
(131,072 on 256 CUs), with one batch and several, one bounce and many, and well
above it, where every render keeps to the stages."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L

pytestmark = pytest.mark.gpu

# (scene, width, height, samples, bounces, samples per batch)
CASES = [("box-c1", 1, 1, 1, 8, 0), ("box-c1", 37, 29, 3, 1, 0), ("box-c1", 362, 362, 1, 8, 0),
         ("box-c1", 363, 363, 1, 8, 0), ("cornell-mesh", 512, 256, 1, 8, 0), ("cornell-mesh", 513, 257, 1, 2, 0),
         ("cornell-mesh", 640, 360, 4, 8, 0), ("instances-small", 400, 401, 4, 12, 0),
         ("cornell-mesh", 300, 200, 7, 6, 2), ("instances-small", 96, 64, 9, 12, 4), ("glass-box", 700, 500, 2, 16, 0),
         # instanced scenes of 2^18 paths a batch and more, one band and two
         ("instances-small", 640, 512, 2, 12, 0), ("instances-small", 513, 512, 1, 5, 0),
         ("instances-small", 700, 401, 3, 6, 1), ("instance-forest", 800, 600, 4, 16, 0)]


@pytest.mark.parametrize("scene_name,w,h,samples,depth,per_batch", CASES)
@pytest.mark.parametrize("sampler", [L.SAMPLER_SOBOL, L.SAMPLER_INDEPENDENT])
def test_film_equals_the_stages(gpu, scene_name, w, h, samples, depth, per_batch, sampler):
    print(f"path case {scene_name} {w}x{h}x{samples}, {depth} bounces", flush=True)
    blob = L.Blob(scene_name)
    scene = L.Scene(gpu, blob)
    u = blob.uniforms(w, h, samples=samples, max_depth=depth, sampler=sampler)
    films = []
    for profile in (1, 0, 0):
        film = L.Film(gpu, w, h)
        st = L.render_wavefront(gpu, scene, u, samples, film, L.WavefrontConfig(per_batch, 0, 0, 0, 0, profile))
        films.append((film.download(), st.extension_rays, st.shadow_rays))
    for other in films[1:]:
        assert np.array_equal(films[0][0].view(np.uint32), other[0].view(np.uint32))
        assert films[0][1:] == other[1:]
