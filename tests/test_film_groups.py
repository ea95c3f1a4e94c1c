"""Films of a batch that share a filter launch: the rule, compiled for the host
(lucida_amd/csrc/film_groups.hpp, tests/film_groups_check.cpp), and on the
device films of shapes that it keeps apart."""
from __future__ import annotations

import shutil
import subprocess
import tempfile
from pathlib import Path

import numpy as np
import pytest

from conftest import ROOT


def test_a_launch_covers_little_beside_its_films():
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host C++ compiler")
    with tempfile.TemporaryDirectory() as d:
        exe = Path(d) / "film_groups_check"
        subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", f"-I{ROOT / 'lucida_amd' / 'csrc'}",
                        str(ROOT / "tests" / "film_groups_check.cpp"), "-o", str(exe)], check=True)
        out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok")


@pytest.mark.gpu
def test_wide_and_tall_films_are_filtered_each_as_alone(gpu):
    import lucida_amd as L
    from tests.test_net_gpu import synthetic_accum
    films = []
    for k, (w, h) in enumerate([(8192, 16), (8192, 24), (128, 4096), (130, 4096), (256, 8), (8192, 8)]):
        f = L.Film(gpu, w, h)
        f.upload(synthetic_accum(w, h, k))
        films.append(f)
    print("film group case: wide and tall films in one batch", flush=True)
    net = L.LearnedDenoiser(gpu, seed=3)
    net.forward_backward(films, films, 128, 8)
    batch = net.tensor(0)
    for k, f in enumerate(films):
        net.forward_backward([f], [f], 128, 8)
        np.testing.assert_array_equal(net.tensor(0)[0], batch[k])
