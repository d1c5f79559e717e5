"""Device-built trees at the sizes where the builder's lists, appended to block
by block, start a block, end one or hold a single entry: hits of random rays
against the oracle, bit for bit."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi
from scenes import random_rays

pytestmark = pytest.mark.gpu


def _soup(n, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, size=(n, 1, 3))
    v = (c + rng.normal(scale=0.6 / n ** (1.0 / 3.0), size=(n, 3, 3))).astype(np.float32).reshape(-1, 3)
    return v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("width", [8, 4])
@pytest.mark.parametrize("n", [2, 3, 64, 65, 257, 1024, 1025, 1026, 2049, 8191, 8192, 8193, 65537])
def test_list_edges(renderer, n, width):
    v, t = _soup(n, n)
    rays = random_rays(3000, n + 1, np.zeros(3), 1.3)
    ref = O.closest_hits([O.Mesh(v, t)], rays)
    slot = renderer.upload_mesh(v, t, width=width, builder=ffi.BUILD_DEVICE)
    try:
        got = renderer.trace_rays([slot], rays)
    finally:
        renderer.remove_mesh(slot)
    for k in ("obj", "tri", "t", "u", "v"):
        assert np.array_equal(got[k].view(np.uint32), ref[k].view(np.uint32)), k
    if n >= 1024:
        assert (ref["tri"] != 0xFFFFFFFF).any()
