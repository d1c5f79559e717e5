"""Scenes with a top-level BVH in every tail mode: lanes that take objects' and
top-level entries from one another, single-ray waves to full ones, stacks that
spill, both BVH widths, against the oracle (which loops over every object).

Bar as in test_gpu_scenes.py: G-buffers and hits bit-exact, RGBA within 1 LSB."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi
from scenes import random_rays
from test_gpu_scenes import _assert_parity, _frame, _remove, _render_both, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, spread, width, builder", [
    (17, 0.3, 8, ffi.BUILD_HOST),  # every ray passes through most boxes
    (40, 2.0, 4, ffi.BUILD_HOST),
    (300, 2.5, 8, ffi.BUILD_DEVICE),
])
def test_tail_modes(renderer, n, spread, width, builder):
    slots, meshes = _scene(renderer, n, 200 + n, spread, small=True, width=width, builder=builder)
    base = renderer.get_tuning()
    frames = [_frame(slots, spread, ffi.SHADING | ffi.SHADOW | ffi.DIRECTIONAL_LIGHT, w=w, h=h)
              for w, h in ((1, 1), (9, 5), (160, 120))]
    rays = random_rays(5000, 31, np.zeros(3), spread + 1.0)
    rays[7, 3] = np.nan
    rays[9, 0] = np.inf
    ref, ref_any = O.closest_hits(meshes, rays), O.any_hits(meshes, rays)
    try:
        for depth in (8, 16):
            for mode in range(5):
                renderer.set_tuning(**dict(base, coop_tail=mode, stack_depth=depth))
                label = "%d objects, tail mode %d, depth %d" % (n, mode, depth)
                print(label, flush=True)
                for fr in frames:
                    g, im, og, oim, _ = _render_both(renderer, meshes, fr)
                    _assert_parity(g, im, og, oim, "%s, %dx%d" % (label, fr.width, fr.height))
                got = renderer.trace_rays(slots, rays)
                for k in ("obj", "tri", "t", "u", "v"):
                    assert np.array_equal(got[k].view(np.uint32), ref[k].view(np.uint32)), (label, k)
                assert np.array_equal(renderer.any_hit(slots, rays), ref_any), label
    finally:
        renderer.set_tuning(**base)
        _remove(renderer, slots)
