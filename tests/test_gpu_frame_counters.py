"""A frame's counters, work queue and stage times whatever ran before it on the
context: shaded and unshaded frames, ray queries, batches, empty scenes."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi
from scenes import random_rays, torus_scene

pytestmark = pytest.mark.gpu

KEYS = ("primary_rays", "hits", "shadow_rays", "shadowed")


@pytest.mark.parametrize("split_passes", [0, 1])
@pytest.mark.parametrize("w, h", [(1, 1), (65, 9), (320, 200)])
def test_counters_after_anything(renderer, w, h, split_passes):
    v, t, cam, cs, ci, pivot, diag, light = torus_scene(60, 30, seed=6)
    mesh = O.Mesh(v, t, db_id=J.make_db_id(1, 0))
    mc, cav = J.make_matcap(0)
    renderer.set_matcap(mc, cav)
    base = renderer.get_tuning()
    slot = renderer.upload_mesh(v, t, db_id=J.make_db_id(1, 0))
    flags = ffi.SHADING | ffi.SHADOW | ffi.DIRECTIONAL_LIGHT
    fr = J.make_frame(w, h, cam, cs, ci, pivot, diag, [slot], flags=flags, light_dir=light)
    empty = J.make_frame(w, h, cam, cs, ci, pivot, diag, [], flags=flags, light_dir=light)
    tg = renderer.create_target(w, h)
    rays = random_rays(300, 5, np.zeros(3), 1.6)
    ref, _, want = O.render([mesh], fr, mc, cav)
    ref_hits = O.closest_hits([mesh], rays)

    def stats():
        s = renderer.stats()
        return [s[k] for k in KEYS], s

    full = [want[k] for k in KEYS]
    none = [0] * 4
    try:
        renderer.set_tuning(**dict(base, split_passes=split_passes))
        steps = [
            (lambda: renderer.render(fr, tg), full),
            (lambda: renderer.render(fr, tg, ffi.STAGE_TRACE), full),
            (lambda: renderer.render(fr, tg, ffi.STAGE_SHADE), none),
            (lambda: renderer.render(empty, tg), [w * h, 0, 0, 0]),
            (lambda: renderer.trace_rays([slot], rays), None),
            (lambda: renderer.render_batch([fr], [tg]), full),
        ]
        for a in steps:
            for b in steps:
                renderer.reset_timings()
                a[0]()
                got = b[0]()
                c, s = stats()
                assert b[1] is None or c == b[1], (steps.index(a), steps.index(b), c)
                if b is steps[0]:
                    assert np.array_equal(got[0]["object_id"], ref["object_id"])
                    assert s["trace_ms"] > 0 and s["shade_ms"] > 0
                    assert (s["shadow_ms"] > 0) == bool(split_passes)
                    tm = renderer.timings()
                    assert tm["trace_ms"][-1] == np.float32(s["trace_ms"])
                    assert tm["shade_ms"][-1] == np.float32(s["shade_ms"])
                if b is steps[4]:
                    assert np.array_equal(got["tri"], ref_hits["tri"])
    finally:
        renderer.set_tuning(**base)
        renderer.destroy_target(tg)
        renderer.remove_mesh(slot)
