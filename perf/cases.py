"""The work that programs built on lucida_amd have it do, as cases to be timed.

Seven paths, each through the package's public entry points:

  render   one frame of a scene into a film (render_wavefront): a preview of a
           tiny box, an interactive frame of a mesh, a final frame of a scene
           of a million triangles, and an instanced field under a sky
  batch    a queue of mixed render requests in one call (render_batch)
  lbvh     the LBVH of a mesh that is on the device (lucida_lbvh_build_device)
  treelet  the tree that long renders trace, on the device
           (lucida_bvh_build_treelet_device)
  atrous   the a-trous filter of a film (Denoiser.run)
  denoise  the learned denoiser of a film (LearnedDenoiser.denoise)
  train    one training step of the learned denoiser (LearnedDenoiser.train_step)

Sizes come from the benchmark, the request stream, the training loop and the
tests of this repository. Scenes, cameras, frame seeds, films and weights are
made from the case's seed.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

import lucida_amd as L

DEV = "cuda:0"
_GPU = None


def _gpu() -> L.Gpu:
    """The program's one device context."""
    global _GPU
    if _GPU is None:
        torch.zeros(1, device=DEV)
        _GPU = L.Gpu(0)
    return _GPU


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # A thumbnail or the first pass of an interactive view: the smallest
        # render, a handful of triangles, one sample; latency is all of it.
        {"name": "render-box-160x90x1", "path": "render", "scene": "box-c1", "frequency": 0, "treelet": False,
         "width": 160, "height": 90, "spp": 1, "depth": 8, "sobol": True},
        # An interactive frame of a mesh of 10,252 triangles, independent sampler.
        {"name": "render-mesh-640x360x4", "path": "render", "scene": "cornell-mesh", "frequency": 0,
         "treelet": False, "width": 640, "height": 360, "spp": 4, "depth": 8, "sobol": False},
        # The benchmark's frame: 1.05M triangles, 16 samples, 8 bounces.
        {"name": "render-sphere-1024x1024x16", "path": "render", "scene": "sphere-c2", "frequency": 229,
         "treelet": True, "width": 1024, "height": 1024, "spp": 16, "depth": 8, "sobol": True},
        # 4,096 instances of glass and metal under an environment map, 12
        # bounces, at an ordinary frame size.
        {"name": "render-instances-960x540x4", "path": "render", "scene": "instances-c3", "frequency": 0,
         "treelet": True, "width": 960, "height": 540, "spp": 4, "depth": 12, "sobol": True},
        # A rendering service's queue: requests of uneven size over three scenes.
        {"name": "batch-20", "path": "batch", "jobs": 20, "depth": 8},
        # A small mesh rebuilt each time it is edited: launches and latency.
        {"name": "lbvh-4k", "path": "lbvh", "frequency": 13},
        # The benchmark's mesh, 1,049,844 triangles.
        {"name": "lbvh-1050k", "path": "lbvh", "frequency": 229},
        # The restructured tree of the request stream's meshes (82,944
        # triangles) doubled twice: 328,704 triangles, three rounds.
        {"name": "treelet-329k", "path": "treelet", "frequency": 128, "rounds": 3},
        # The filter on a full frame of odd sides.
        {"name": "atrous-1279x719", "path": "atrous", "width": 1279, "height": 719, "iterations": 4, "samples": 4},
        # The learned denoiser on a preview and on the benchmark's film.
        {"name": "denoise-384x216", "path": "denoise", "width": 384, "height": 216, "samples": 2},
        {"name": "denoise-1024x1024", "path": "denoise", "width": 1024, "height": 1024, "samples": 16},
        # The training loop's step: eight films of 256 x 256.
        {"name": "train-8x256x256", "path": "train", "width": 256, "height": 256, "film": 256, "count": 8},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    path = rng.choice(["render", "render", "batch", "lbvh", "treelet", "atrous", "denoise", "train"])
    if path == "render":
        scene = rng.choice(["box-c1", "cornell-mesh", "sphere-c2", "instances-c3"])
        w, h = _log_int(rng, 96, 1024), _log_int(rng, 64, 1024)
        most = {"instances-c3": 2_000_000}.get(scene, 12_000_000)  # paths
        spp = min(_log_int(rng, 1, 64), max(1, most // (w * h)))
        return {"path": path, "scene": scene, "frequency": _log_int(rng, 16, 229) if scene == "sphere-c2" else 0,
                "treelet": scene == "instances-c3" or (scene == "sphere-c2" and rng.random() < 0.7),
                "width": w, "height": h, "spp": spp, "depth": rng.randint(4, 12 if scene == "instances-c3" else 8),
                "sobol": rng.random() < 0.7}
    if path == "batch":
        return {"path": path, "jobs": rng.randint(4, 20), "depth": rng.randint(4, 8)}
    if path == "lbvh":
        return {"path": path, "frequency": _log_int(rng, 6, 229)}
    if path == "treelet":
        return {"path": path, "frequency": _log_int(rng, 6, 128), "rounds": rng.randint(1, 3)}
    if path == "atrous":
        return {"path": path, "width": _log_int(rng, 96, 1279), "height": _log_int(rng, 64, 719),
                "iterations": rng.randint(3, 5), "samples": _log_int(rng, 1, 64)}
    if path == "denoise":
        return {"path": path, "width": 128 * rng.randint(1, 8), "height": 8 * _log_int(rng, 12, 128),
                "samples": _log_int(rng, 1, 64)}
    w, h = 128 * rng.randint(1, 2), 8 * rng.randint(12, 32)
    return {"path": path, "width": w, "height": h, "film": rng.randint(256, 320), "count": rng.randint(2, 8)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


class _FilmArray:
    """A film's device records as an array; it keeps the film, and so its
    memory, for as long as a view of it is held."""

    def __init__(self, film: L.Film):
        self.film = film
        ptr = L.lib().lucida_film_device_ptr(film._h)
        self.__cuda_array_interface__ = {"shape": (film.height, film.width, 16), "typestr": "<f4",
                                         "data": (ptr, False), "version": 2}


def _film_view(film: L.Film) -> torch.Tensor:
    """The film's device records, (height, width, 16) float32, no copy."""
    view = torch.as_tensor(_FilmArray(film), device=DEV)
    assert view.shape == (film.height, film.width, 16) and view.data_ptr() == L.lib().lucida_film_device_ptr(film._h)
    return view


def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _view(width: int, height: int, seed: int) -> dict:
    """What a camera sees, as images in 64 bits: facets with their own normals,
    depths and textured albedos under smooth light, one in ten dark."""
    g = _generator(seed)
    y, x = torch.meshgrid(torch.arange(height, device=DEV, dtype=torch.float64) / height,
                          torch.arange(width, device=DEV, dtype=torch.float64) / width, indexing="ij")
    cells = 24
    px, py = _rand(g, cells), _rand(g, cells)
    dist = (x[..., None] - px) ** 2 + (y[..., None] - py) ** 2
    cell = dist.argmin(-1)
    n = torch.nn.functional.normalize(_rand(g, cells, 3) * 2 - 1, dim=-1)
    bump = torch.stack([torch.sin(40 * x), torch.cos(31 * y), torch.ones_like(x)], -1) * 0.02
    normal = torch.nn.functional.normalize(n[cell] + bump, dim=-1)
    base, slope = 2 + 6 * _rand(g, cells), _rand(g, cells, 2) - 0.5
    depth = base[cell] + slope[cell][..., 0] * x + slope[cell][..., 1] * y
    albedo = (0.1 + 0.85 * _rand(g, cells, 3))[cell] * (0.75 + 0.25 * torch.sign(torch.sin(60 * x) * torch.sin(60 * y)))[..., None]
    light = (0.05 + 1.5 * _rand(g, cells, 3))[cell] * (1.1 + torch.sin(5 * x + 3 * y))[..., None]
    light = torch.where((_rand(g, cells) < 0.1)[cell][..., None], 0.01 * light, light)
    return {"light": light, "albedo": albedo, "normal": normal, "depth": depth}


def _records(view: dict, samples: int, seed: int) -> torch.Tensor:
    """A film's sums after `samples` noisy samples per pixel of that view."""
    g = _generator(seed)
    mean = view["light"] * view["albedo"]
    k = 0.6 * samples  # a pixel's samples vary a little more than their mean
    noise = torch._standard_gamma(torch.full_like(mean[..., :1], k), generator=g) / k
    fire = 1 + 20 * (_rand(g, *mean.shape[:2], 1) < 0.001)
    rad = mean * noise * fire
    h, w = mean.shape[:2]
    rec = torch.zeros(h, w, 16, device=DEV, dtype=torch.float64)
    rec[..., 0:3] = rad * samples
    rec[..., 3] = samples
    rec[..., 4:7] = view["albedo"] * samples
    rec[..., 7] = view["depth"] * samples
    rec[..., 8:11] = view["normal"] * samples
    rec[..., 12:15] = rad * rad * (1.0 + (0.0 if samples == 1 else 1 / 0.6)) * samples
    return rec.float()


def _film(records: torch.Tensor) -> L.Film:
    film = L.Film(_gpu(), records.shape[1], records.shape[0])
    _film_view(film).copy_(records)
    torch.cuda.synchronize()
    return film


def _weights(seed: int) -> np.ndarray:
    """Weights of a network part way through its training: the fresh
    network's, and an output layer that is no longer zero."""
    rng = np.random.default_rng(seed)
    parts = []
    for k, (cin, cout, _) in enumerate(L.NET_LAYERS):
        used_in, used_out = (15 if k == 0 else cin), (3 if k == len(L.NET_LAYERS) - 1 else cout)
        std = math.sqrt(2.0 / (9 * used_in)) * (0.1 if used_out == 3 else 1.0)
        w = np.zeros((9, cin, cout), np.float32)
        w[:, :used_in, :used_out] = rng.standard_normal((9, used_in, used_out), dtype=np.float32) * np.float32(std)
        b = np.zeros(cout, np.float32)
        b[:used_out] = rng.standard_normal(used_out, dtype=np.float32) * np.float32(0.02)
        parts += [w.ravel(), b]
    return np.concatenate(parts)


# The queue's requests: (scene, side, samples).
_REQUESTS = [(0, 128, 64), (1, 256, 4), (2, 512, 1), (0, 256, 16), (1, 128, 16), (2, 256, 4), (0, 512, 4), (1, 512, 4),
             (2, 128, 1), (0, 128, 1), (1, 256, 16), (2, 512, 4), (0, 256, 1), (1, 128, 64), (2, 256, 16), (0, 512, 1),
             (1, 512, 16), (2, 128, 4), (0, 128, 4), (1, 256, 1)]


def _prepare_mesh(case: dict, seed: int) -> dict:
    """A displaced sphere in its room on the device, and the tree's arrays."""
    a = L.Blob("sphere-c2", seed=1 + seed % 100_000, frequency=case["frequency"]).arrays()
    n = len(a["triangles"])
    tris = torch.from_numpy(a["triangles"].view(np.int32).reshape(n, 4)).to(DEV)
    pos = torch.from_numpy(a["positions"]).to(DEV)
    return {"tris": tris, "pos": pos, "n": n,
            "nodes": torch.zeros(2 * n - 1, 8, dtype=torch.int32, device=DEV),
            "order": torch.zeros(n, dtype=torch.int32, device=DEV),
            "sorted": torch.zeros(n, 4, dtype=torch.int32, device=DEV)}


def prepare(case: dict, seed: int):
    gpu, path = _gpu(), case["path"]
    st = {"case": case}
    if path == "render":
        # another seed is another frame, and another displaced sphere
        blob = L.Blob(case["scene"], seed=1 + seed % 100_000, frequency=case["frequency"])
        st["scene"] = L.Scene(gpu, blob, treelet=case["treelet"])
        st["film"] = L.Film(gpu, case["width"], case["height"])
        st["uniforms"] = blob.uniforms(case["width"], case["height"], samples=case["spp"], max_depth=case["depth"],
                                       frame_seed=seed,
                                       sampler=L.SAMPLER_SOBOL if case["sobol"] else L.SAMPLER_INDEPENDENT)
    elif path == "batch":
        blobs = [L.Blob("box-c1")] + [L.Blob("sphere-c2", seed=1 + (seed + k) % 100_000, frequency=64) for k in (0, 1)]
        scenes = [L.Scene(gpu, b, treelet=True) for b in blobs]
        st["jobs"] = []
        for k, (si, side, spp) in enumerate(_REQUESTS[:case["jobs"]]):
            u = blobs[si].uniforms(side, side, samples=spp, max_depth=case["depth"], frame_seed=seed + k)
            st["jobs"].append((scenes[si], u, spp, L.Film(gpu, side, side)))
    elif path in ("lbvh", "treelet"):
        st.update(_prepare_mesh(case, seed))
    elif path in ("atrous", "denoise"):
        view = _view(case["width"], case["height"], seed)
        st["film"] = _film(_records(view, case["samples"], seed + 1))
        st["out"] = L.Film(gpu, case["width"], case["height"])
        if path == "atrous":
            st["filter"] = L.Denoiser(gpu)
            st["params"] = L.DenoiseParams(case["iterations"], 64.0, 0.08, 4.0, 0.1)
        else:
            st["net"] = L.LearnedDenoiser(gpu)
            st["net"].set_params(_weights(seed))
    else:
        st["net"] = L.LearnedDenoiser(gpu)
        st["net"].set_params(_weights(seed))
        ins, refs, st["crops"] = _training_films(case, seed)
        st["ins"], st["refs"] = [_film(r) for r in ins], [_film(r) for r in refs]
    torch.cuda.synchronize()
    return st


def _training_films(case: dict, seed: int):
    """The batch's input and target records and its crops: inputs of 1 to 256
    samples, targets of 4,096."""
    rng = random.Random(seed)
    ins, refs, crops = [], [], []
    for k in range(case["count"]):
        view = _view(case["film"], case["film"], seed + 3 * k)
        ins.append(_records(view, 1 << rng.randint(0, 8), seed + 3 * k + 1))
        refs.append(_records(view, 4096, seed + 3 * k + 2))
        crops.append((rng.randint(0, case["film"] - case["width"]), rng.randint(0, case["film"] - case["height"])))
    return ins, refs, crops


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(st):
    case, gpu = st["case"], _gpu()
    path = case["path"]
    if path == "render":
        st["film"].clear()
        L.render_wavefront(gpu, st["scene"], st["uniforms"], case["spp"], st["film"])
        return _film_view(st["film"])
    if path == "batch":
        for _, _, _, film in st["jobs"]:
            film.clear()
        L.render_batch(gpu, st["jobs"])
        return [_film_view(film) for _, _, _, film in st["jobs"]]
    if path in ("lbvh", "treelet"):
        count, n = C.c_size_t(), st["n"]
        out = (st["nodes"].data_ptr(), C.byref(count), st["order"].data_ptr(), st["sorted"].data_ptr(), None)
        if path == "lbvh":
            L._check(L.lib().lucida_lbvh_build_device(gpu._h, st["tris"].data_ptr(), n, st["pos"].data_ptr(), *out))
        else:
            L._check(L.lib().lucida_bvh_build_treelet_device(gpu._h, st["tris"].data_ptr(), n, st["pos"].data_ptr(),
                                                             case["rounds"], *out))
        # the nodes past the count are the zeros they were made with
        return {"nodes": st["nodes"], "count": count.value, "order": st["order"], "triangles": st["sorted"]}
    if path == "atrous":
        st["filter"].run(st["film"], st["out"], st["params"])
        return _film_view(st["out"])
    if path == "denoise":
        st["net"].denoise(st["film"], st["out"])
        return _film_view(st["out"])
    loss = st["net"].train_step(st["ins"], st["refs"], case["width"], case["height"], st["crops"])
    return {"loss": loss, "gradients": st["net"].params(gradients=True)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

_LEVEL_PIXELS = [4.0 ** -lvl for lvl in L.NET_LEVEL]


def _net_flops(pixels: float) -> float:
    return sum(2.0 * 9 * cin * cout * s for (cin, cout, _), s in zip(L.NET_LAYERS, _LEVEL_PIXELS)) * pixels


def _scene_size(case: dict) -> tuple[int, float]:
    """Triangles, and the bytes of the scene's tables."""
    scene = case["scene"]
    tris = {"box-c1": 10, "cornell-mesh": 10_252, "instances-c3": 9_680}.get(scene, 20 * case["frequency"] ** 2 + 1024)
    # a triangle's edges, indices, vertices (half a vertex each) and two nodes
    return tris, tris * (48.0 + 16 + 24 + 64) + (4096 * 128 + 2048 * 1024 * 20 if scene == "instances-c3" else 0)


def _path_flops(tris: int, depth: int) -> float:
    """A path's operations: half its bounces taken, each with a closest-hit and
    a shadow walk of about log2(triangles) node pairs (48 operations), two
    triangle tests and one shading."""
    return 0.5 * depth * (2 * (48 * max(1.0, math.log2(tris)) + 2 * 45) + 600)


def work(case: dict) -> dict:
    path = case["path"]
    if path == "render":
        tris, table = _scene_size(case)
        pixels = case["width"] * case["height"]
        return {"bytes": table + 64.0 * pixels, "flops": pixels * case["spp"] * _path_flops(tris, case["depth"])}
    if path == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for si, side, spp in _REQUESTS[:case["jobs"]]:
            w = work({"path": "render", "scene": "box-c1" if si == 0 else "sphere-c2", "frequency": 64, "width": side,
                      "height": side, "spp": spp, "depth": case["depth"]})
            total = {k: total[k] + w[k] for k in total}
        return total
    if path in ("lbvh", "treelet"):
        n = 20 * case["frequency"] ** 2 + 1024
        # triangles and vertices in; order, sorted triangles and about 1.4 n nodes out
        return {"bytes": n * (16.0 + 8 + 4 + 16 + 1.4 * 32),
                "flops": n * (100.0 + (case["rounds"] * 2000.0 if path == "treelet" else 0.0))}
    if path == "atrous":
        px = case["width"] * case["height"]
        return {"bytes": 112.0 * px, "flops": px * (case["iterations"] * 25 * 25.0 + 60)}
    if path == "denoise":
        px = case["width"] * case["height"]
        return {"bytes": 128.0 * px + 4.0 * L.LearnedDenoiser.param_count(), "flops": _net_flops(px) + px * 2600.0}
    px = case["count"] * case["width"] * case["height"]
    film = case["count"] * case["film"] ** 2
    return {"bytes": 64.0 * film + 64.0 * px + 28.0 * L.LearnedDenoiser.param_count(),
            "flops": 3 * _net_flops(px) + film * 2600.0}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------

_LUM = (0.2126, 0.7152, 0.0722)


def _lum(c):
    return c[..., 0] * _LUM[0] + c[..., 1] * _LUM[1] + c[..., 2] * _LUM[2]


def _shift(img, dy: int, dx: int):
    """img moved so that [y, x] holds [y + dy, x + dx], and where that exists."""
    h, w = img.shape[:2]
    out, ok = torch.zeros_like(img), torch.zeros(h, w, device=img.device, dtype=torch.bool)
    ys, xs = slice(max(0, -dy), min(h, h - dy)), slice(max(0, -dx), min(w, w - dx))
    if ys.start < ys.stop and xs.start < xs.stop:
        out[ys, xs] = img[ys.start + dy:ys.stop + dy, xs.start + dx:xs.stop + dx]
        ok[ys, xs] = True
    return out, ok


def _atrous64(rec, iterations: int):
    """The filter in 64 bits: (colour times albedo, albedo, normal, depth)."""
    rec = rec.double()
    inv = 1 / rec[..., 3:4].clamp(min=1)
    albedo = (rec[..., 4:7] * inv).clamp(min=1e-3)
    normal, depth = rec[..., 8:11] * inv, (rec[..., 7:8] * inv)[..., 0]
    color = rec[..., 0:3] * inv / albedo
    al = _lum(albedo)
    lum = _lum(color)
    count, total, square = torch.zeros_like(lum), torch.zeros_like(lum), torch.zeros_like(lum)
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            v, ok = _shift(lum, dy, dx)
            count, total, square = count + ok, total + v, square + v * v
    dev = (square / count - (total / count) ** 2).clamp(min=0).sqrt()
    kernel = (1 / 16, 1 / 4, 3 / 8, 1 / 4, 1 / 16)
    ca = al.clamp(min=1e-3)
    sd, sl, sa = 0.08 * depth.abs().clamp(min=1e-3), 4.0 * dev.clamp(min=1e-4), 0.1 * ca
    for level in range(iterations):
        lum = _lum(color)
        num, den = torch.zeros_like(color), torch.zeros_like(lum)
        for ky in range(5):
            for kx in range(5):
                dy, dx = (ky - 2) << level, (kx - 2) << level
                packed, ok = _shift(torch.cat([color, lum[..., None], normal, depth[..., None], al[..., None]], -1), dy, dx)
                nd = (normal * packed[..., 4:7]).sum(-1).clamp(min=0)
                e = (depth - packed[..., 7]).abs() / sd + (lum - packed[..., 3]).abs() / sl + (ca - packed[..., 8]).abs() / sa
                wt = torch.where(ok, kernel[kx] * kernel[ky] * nd ** 64 * torch.exp(-e), torch.zeros_like(e))
                num, den = num + packed[..., 0:3] * wt[..., None], den + wt
        color = torch.where(den[..., None] > 0, num / den.clamp(min=1e-300)[..., None], color)
    return color * albedo, albedo, normal, depth


def _features64(rec):
    """The network's input channels and the estimate that it corrects."""
    base = _atrous64(rec, 4)[0]
    rec = rec.double()
    inv = 1 / rec[..., 3:4].clamp(min=1)
    albedo, rad = (rec[..., 4:7] * inv).clamp(min=1e-3), rec[..., 0:3] * inv
    depth = (rec[..., 7:8] * inv).clamp(min=0)
    var = _lum((rec[..., 12:15] * inv - rad * rad).clamp(min=0))[..., None]
    log_base = torch.log1p((base / albedo).clamp(min=0))
    feat = torch.cat([torch.log1p((rad / albedo).clamp(min=0)), albedo, rec[..., 8:11] * inv, depth / (1 + depth),
                      torch.log1p((var * inv).sqrt() / _lum(albedo)[..., None]),
                      torch.log2(rec[..., 3:4].clamp(min=1)) / 16, log_base, torch.zeros_like(depth)], -1)
    return feat, log_base, albedo


def _net64(x, params):
    """The network on (n, h, w, 16) features, as products of shifted images."""
    def conv(k, x):
        w, b = params[k]
        n, h, wd, _ = x.shape
        pad = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        out = b + sum(pad[:, t // 3:t // 3 + h, t % 3:t % 3 + wd].reshape(n * h * wd, -1) @ w[t] for t in range(9))
        out = out.reshape(n, h, wd, -1)
        return out.relu() if L.NET_LAYERS[k][2] else out

    def pool(x):
        n, h, w, c = x.shape
        return x.reshape(n, h // 2, 2, w // 2, 2, c).mean((2, 4))

    def up(x, skip):
        return torch.cat([x.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], -1)

    s0 = conv(1, conv(0, x))
    s1 = conv(3, conv(2, pool(s0)))
    s2 = conv(5, conv(4, pool(s1)))
    y = conv(7, conv(6, pool(s2)))
    y = conv(9, conv(8, up(y, s2)))
    y = conv(11, conv(10, up(y, s1)))
    return conv(14, conv(13, conv(12, up(y, s0))))


def _params64(seed: int, grad: bool):
    flat, at, out = torch.from_numpy(_weights(seed)).to(DEV, torch.float64), 0, []
    for cin, cout, _ in L.NET_LAYERS:
        w = flat[at:at + 9 * cin * cout].reshape(9, cin, cout).clone().requires_grad_(grad)
        b = flat[at + 9 * cin * cout:at + (9 * cin + 1) * cout].clone().requires_grad_(grad)
        at += (9 * cin + 1) * cout
        out.append((w, b))
    return out


def exact(case: dict, seed: int):
    path = case["path"]
    if path in ("atrous", "denoise"):
        rec = _records(_view(case["width"], case["height"], seed), case["samples"], seed + 1)
        out = torch.zeros(*rec.shape, device=DEV, dtype=torch.float64)
        if path == "atrous":
            color, albedo, normal, depth = _atrous64(rec, case["iterations"])
        else:
            feat, log_base, albedo = _features64(rec)
            with torch.no_grad():
                y = _net64(feat[None], _params64(seed, False))[0]
            color = torch.expm1((y[..., 0:3] + log_base).clamp(min=0)) * albedo
            inv = 1 / rec.double()[..., 3:4].clamp(min=1)
            normal, depth = rec.double()[..., 8:11] * inv, (rec.double()[..., 7:8] * inv)[..., 0]
        out[..., 0:3], out[..., 3], out[..., 4:7], out[..., 7], out[..., 8:11] = color, 1, albedo, depth, normal
        return out
    if path == "train":
        ins, refs, crops = _training_films(case, seed)
        feats, bases, targets = [], [], []
        for rec, ref, (x0, y0) in zip(ins, refs, crops):
            feat, log_base, albedo = _features64(rec)
            ref = ref.double()
            target = torch.log1p((ref[..., 0:3] / ref[..., 3:4] / albedo).clamp(min=0))
            cut = (slice(y0, y0 + case["height"]), slice(x0, x0 + case["width"]))
            feats.append(feat[cut])
            bases.append(log_base[cut])
            targets.append(target[cut])
        params = _params64(seed, True)
        y = _net64(torch.stack(feats), params)[..., 0:3]
        loss = (y + torch.stack(bases) - torch.stack(targets)).square().mean()
        loss.backward()
        return {"loss": loss.detach(), "gradients": torch.cat([t.grad.reshape(-1) for p in params for t in p])}
    return None  # a render's paths and a build's integers have no such value
