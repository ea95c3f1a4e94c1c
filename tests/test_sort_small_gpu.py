"""The one-workgroup sort and the line to the sort over the device (8,192
keys), against a stable sort on the host: lengths around a wave, a block and
the line, and keys that put everything into one digit."""
from __future__ import annotations

import numpy as np
import pytest

import lucida_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 4404, 8191, 8192, 8193, 20000])
@pytest.mark.parametrize("family", ["random", "equal", "low", "high", "descending"])
def test_matches_a_stable_sort(gpu, n, family):
    rng = np.random.default_rng(n)
    keys = {"random": lambda: rng.integers(0, 1 << 32, n), "equal": lambda: np.full(n, 0xFFFFFFFF),
            "low": lambda: rng.integers(0, 3, n), "high": lambda: rng.integers(0, 3, n) << 30,
            "descending": lambda: np.arange(n)[::-1]}[family]().astype(np.uint32)
    print(f"sort case: {n} keys, {family}", flush=True)
    vals = rng.integers(0, 1 << 32, n).astype(np.uint32)
    k, v = L.LbvhBuilder(gpu).sort(keys, vals)
    order = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(k, keys[order])
    np.testing.assert_array_equal(v, vals[order])
