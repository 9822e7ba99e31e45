"""Ray queries go to the device in parts of at least 2^17 rays: every ray's hit is the one it has in a
batch of its own part, for batches around the part sizes, and for callers on several threads, which
share the context's buffers one call at a time.  Hits are compared bit for bit."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import tinypt_amd as T
from parity_scenes import PARITY_CASES
from trace_checks import path_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["mesh_small", "instanced_small"])
def test_parts_and_threads(gpu_ctx, name):
    sc = PARITY_CASES[name][0]()
    base = path_rays(sc, np.random.default_rng(3), 20_000)
    ds = T.DeviceScene(sc, gpu_ctx)
    ref = ds.trace_closest(base)

    def check(n, shift):
        idx = (np.arange(n) * 7 + shift) % len(base)
        got = ds.trace_closest(base[idx])
        for key, v in ref.items():
            np.testing.assert_array_equal(got[key], v[idx], err_msg=f"{key} {n}")

    for n in (1, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, (1 << 19) - 3, (1 << 19) + 5, 3 << 18):
        check(n, 0)
    with ThreadPoolExecutor(4) as pool:
        for f in [pool.submit(check, n, k) for k, n in enumerate((1000, 300_000, 5, 140_001, 64, 600_000))]:
            f.result()
    assert len(ds.trace_closest(base[:0])["t"]) == 0
