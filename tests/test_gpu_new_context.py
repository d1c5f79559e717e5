"""A context that has rendered nothing has no counts, whatever the memory that
it was given held before, and an error that some other call left behind on the
thread does not keep it from being made."""
import ctypes

import numpy as np
import pytest

import j3d_amd as J

pytestmark = pytest.mark.gpu


def test_counters_start_at_zero():
    v, t = J.icosphere(1, seed=1)
    diag, pivot = J.scene_framing(v)
    cs, ci = J.orbit_camera(3.0, 0.5, 0.4)
    for n in (21, 42, 64, 128):
        with J.Renderer(0) as r:  # allocations full of ones and of another context's counts, given back
            for _ in range(40):
                r.upload_points(np.full((n, 3), -np.nan, np.float32), colors=np.full(n, 0xFFFFFFFF, np.uint32))
            r.set_matcap(*J.make_matcap(0))
            slot = r.upload_mesh(v, t)
            fr = J.make_frame(64, 48, J.camera_with_vertical_fov(60.0), cs, ci, pivot, diag, [slot])
            tg = r.create_target(64, 48)
            r.set_counting(True)
            r.render(fr, tg)
            r.render(fr, tg, stages=J.ffi.STAGE_TRACE)
            assert r.stats()["primary_rays"] == 64 * 48
        with J.Renderer(0) as r:
            counts = {k: x for k, x in r.stats().items() if not k.endswith("_ms")}
            assert all(not np.any(x) for x in counts.values()), (n, counts)


def test_an_error_left_behind_by_another_call():
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipSetDevice(9999) != 0 and hip.hipPeekAtLastError() != 0
    try:
        with J.Renderer(0) as r:
            assert r.stats()["primary_rays"] == 0
    finally:
        hip.hipGetLastError()  # clears it
