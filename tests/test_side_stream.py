"""Work on a second stream is joined on every way out of its scope
(lucida_amd/csrc/side_stream.hpp, the denoiser's weight gradients), and the
denoiser's backward pass leaves the second stream to it. Compiled for the
host with stand-ins for the HIP calls (tests/side_stream_check.cpp)."""
from __future__ import annotations

import re
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

from conftest import ROOT

CSRC = ROOT / "lucida_amd" / "csrc"


def test_every_way_out_joins():
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host C++ compiler")
    with tempfile.TemporaryDirectory() as d:
        exe = Path(d) / "side_stream_check"
        subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", "-I/opt/rocm/include",
                        str(ROOT / "tests" / "side_stream_check.cpp"), "-o", str(exe)], check=True)
        out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok")


def test_the_backward_pass_leaves_its_second_stream_to_it():
    text = (CSRC / "net.hip").read_text()
    body = text[text.index("static lucida_status net_backward"):]
    body = body[:body.index("\n}\n")]
    assert re.search(r"SideStream \w+\(s, ", body)
    assert "hipEventRecord" not in body and "hipStreamWaitEvent" not in body
