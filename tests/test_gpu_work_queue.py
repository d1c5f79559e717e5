"""The trace kernels' work queue: every ray of a launch is taken exactly once
at the sizes where its bands are empty, uneven or cut (fewer tiles than bands,
one tile more or less than a multiple), and where a wave takes two tiles per
atomic (4.2M rays and more), with the results of the oracle or of smaller
launches, bit for bit."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from scenes import compare_gbuffers, random_rays

pytestmark = pytest.mark.gpu


def _same(a, b):
    for k in ("obj", "tri"):
        assert np.array_equal(a[k], b[k]), k
    for k in ("t", "u", "v"):
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


@pytest.mark.parametrize("n", [1, 63, 64, 65, 447, 511, 512, 513, 577, 4097])
def test_ray_counts_around_the_bands(renderer, n):
    v, t = J.torus(40, 24, seed=2)
    slot = renderer.upload_mesh(v, t)
    m = O.Mesh(v, t)
    rays = random_rays(n, 5, np.zeros(3), 1.4)
    try:
        got = renderer.trace_rays([slot], rays)
        ref = O.closest_hits([m], rays)
        _same(got, ref)
        assert np.array_equal(renderer.any_hit([slot], rays) != 0, ref["obj"] != 0xFFFFFFFF)
    finally:
        renderer.remove_mesh(slot)


def test_two_tiles_per_atomic(renderer):
    v, t = J.torus(40, 24, seed=2)
    slot = renderer.upload_mesh(v, t)
    n = 4600001
    rays = np.tile(random_rays(46001, 9, np.zeros(3), 1.4), (100, 1))[:n]
    rays[:, 0] += np.linspace(0.0, 0.1, n, dtype=np.float32)
    try:
        whole = renderer.trace_rays([slot], rays)
        cut = n // 2 + 37
        parts = [renderer.trace_rays([slot], rays[:cut]), renderer.trace_rays([slot], rays[cut:])]
        _same(whole, {k: np.concatenate([p[k] for p in parts]) for k in whole})
        assert (whole["obj"] != 0xFFFFFFFF).any()
    finally:
        renderer.remove_mesh(slot)


@pytest.mark.parametrize("w, h", [(8, 8), (57, 9), (64, 64), (131, 67)])
def test_small_frames_around_the_bands(renderer, w, h):
    v, t = J.torus(60, 30, seed=3)
    slot = renderer.upload_mesh(v, t, db_id=J.make_db_id(1, 0))
    m = O.Mesh(v, t, db_id=J.make_db_id(1, 0))
    diag, pivot = J.scene_framing(v)
    cs, ci = J.orbit_camera(3.0, 0.4, 0.5)
    mc, cav = J.make_matcap(0)
    renderer.set_matcap(mc, cav)
    tg = renderer.create_target(w, h)
    fr = J.make_frame(w, h, J.camera_with_vertical_fov(60.0), cs, ci, pivot, diag, [slot],
                      flags=J.ffi.EDGES | J.ffi.SHADING | J.ffi.SHADOW)
    try:
        g, _ = renderer.render(fr, tg)
        og, _, _ = O.render([m], fr, mc, cav)
        assert not any(compare_gbuffers(g, og).values())
    finally:
        renderer.destroy_target(tg)
        renderer.remove_mesh(slot)
