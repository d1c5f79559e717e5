"""Voxel rays walked by groups of lanes: grids whose rays do not fill a wave's
round, hit lists ranked by counting and by sorting (more than 128 hits), rays
with ties in t, and both BVH widths, against the oracle byte for byte."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi

pytestmark = pytest.mark.gpu


def _slabs(n, twice=False):
    """n parallel unit squares x = 0.02 k (each given twice: every hit ties with another)."""
    v, t = [], []
    for k in range(n):
        b = len(v)
        x = np.float32(0.02) * np.float32(k)
        v += [[x, 0, 0], [x, 1, 0], [x, 1, 1], [x, 0, 1]]
        for _ in range(2 if twice else 1):
            t += [[b, b + 1, b + 2], [b, b + 2, b + 3]]
    return np.array(v, np.float32), np.array(t, np.uint32)


def _check(renderer, v, t, dim, colors=None, **kw):
    slot = renderer.upload_mesh(v, t, **kw)
    try:
        if colors is not None:
            renderer.set_mesh_colors(slot, vertex_colors=colors)
        dims, data = renderer.voxelize(slot, dim)
        rdims, ref = O.voxelize(O.Mesh(v, t, vertex_colors=colors), dim)
        assert dims == rdims
        assert np.array_equal(data, ref), int((data != ref).sum())
        assert data.any()
    finally:
        renderer.remove_mesh(slot)


@pytest.mark.parametrize("dim", [1, 2, 3, 7, 33])
@pytest.mark.parametrize("width, builder", [(8, ffi.BUILD_HOST), (4, ffi.BUILD_HOST), (8, ffi.BUILD_DEVICE)])
def test_grids_around_a_round(renderer, dim, width, builder):
    v, t = J.torus(60, 30, seed=4)
    colors = np.random.default_rng(1).uniform(0, 1, size=(len(v), 3)).astype(np.float32)
    _check(renderer, v, t, dim, colors, width=width, builder=builder)


@pytest.mark.parametrize("n, twice", [(31, False), (32, False), (33, False), (127, False), (129, False), (300, True)])
def test_hit_counts_around_the_list_sizes(renderer, n, twice):
    v, t = _slabs(n, twice)
    colors = np.random.default_rng(2).uniform(0, 1, size=(len(v), 3)).astype(np.float32)
    _check(renderer, v, t, 16, colors)
