"""The network's stage time of a learned frame: the network's, also on the frame
that allocates the target's tile-order buffers."""
import numpy as np
import pytest

import j3d_amd as J
from j3d_amd import ffi
from test_mlp_oracle import random_params

pytestmark = pytest.mark.gpu


def test_network_time_without_allocations(renderer):
    v, t = J.torus(120, 60, seed=6)
    slot = renderer.upload_mesh(v, t, db_id=J.make_db_id(1, 0))
    diag, pivot = J.scene_framing(v)
    cs, ci = J.orbit_camera(3.0, 0.9, 0.4)
    renderer.set_matcap(*J.make_matcap(0))
    w, h = 1280, 720
    renderer.set_proposal(slot, random_params(3), [0.0, 0.0, 0.0, 1.5])
    small, full = (0, 0, 1023, 511), (0, 0, w - 1, h - 1)
    first, later = [], []
    try:
        for _ in range(9):
            tg = renderer.create_target(w, h)

            def ms(rect):
                fr = J.make_frame(w, h, J.camera_with_vertical_fov(60.0), cs, ci, pivot, diag, [slot],
                                  flags=ffi.EDGES | ffi.LEARNED, margin=0.05, rect=rect)
                renderer.render(fr, tg, readback=False)
                return renderer.stats()["mlp_ms"]

            ms(small)
            first.append(ms(full))  # the larger rectangle's buffers take the place of the first frame's
            later.append(ms(full))
            renderer.destroy_target(tg)
        # the same launch: its times differ by a few percent
        assert 0 < np.median(later) and np.median(first) <= 1.15 * np.median(later), (first, later)
    finally:
        renderer.remove_mesh(slot)
