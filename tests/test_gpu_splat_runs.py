"""Point clouds large enough to be merged by runs (4,000,000 points and more,
with smaller ones beside them), against the oracle, bit for bit: at the rule's
edge, in scan order, in random order (the table of a run fills up and points go
to memory by themselves) and with every point in a handful of pixels."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi

pytestmark = pytest.mark.gpu


def _sphere(n, order, seed):
    rng = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.float64)
    z = 1.0 - 2.0 * (i + 0.5) / n
    phi = i * (2.0 * np.pi * np.sqrt(n) / n)
    rho = np.sqrt(1.0 - z * z)
    p = np.stack([rho * np.cos(phi), rho * np.sin(phi), z], 1) * (1.0 + 0.01 * rng.normal(size=(n, 1)))
    if order == "random":
        p = p[rng.permutation(n)]
    elif order == "one_spot":
        p = p * 0.001
    p = p.astype(np.float32)
    p[rng.integers(0, n, 1000)] = p[rng.integers(0, n, 1000)]  # ties at other indices
    p[rng.integers(0, n, 20)] = np.nan
    return {"xyz": p, "colors": rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32),
            "db_id": J.make_db_id(2, seed)}


@pytest.mark.parametrize("n, order, w, h", [(3999999, "scan", 320, 200), (4000000, "scan", 1280, 719),
                                            (4000001, "random", 1280, 719), (4300007, "one_spot", 320, 200)])
def test_large_clouds_match_oracle(renderer, n, order, w, h):
    clouds = [_sphere(n, order, 1), _sphere(5000, "random", 2)]
    ids = [renderer.upload_points(c["xyz"], colors=c["colors"], db_id=c["db_id"]) for c in clouds]
    cam = J.camera_with_vertical_fov(60.0)
    cs, ci = J.orbit_camera(2.6, 0.7, 0.4)
    P, _ = J.projection(cam, w, h)
    fr = J.make_frame(w, h, cam, cs, ci, np.zeros(3, np.float32), 2.0, [], flags=ffi.EDGES)
    renderer.set_matcap(*J.make_matcap(0))
    tg = renderer.create_target(w, h)
    try:
        g0, im0 = renderer.render(fr, tg)
        renderer.splat_points(tg, P, ci, ffi.EDGES, ids)
        g1, im1 = renderer.read_target(tg)
        og, oim = O.splat_points(g0, im0, P, ci, ffi.EDGES, clouds)
        assert np.array_equal(g1.view(np.uint8), og.view(np.uint8))
        assert np.array_equal(im1, oim)
        assert (g1["db_id"] == clouds[0]["db_id"]).any()
    finally:
        renderer.destroy_target(tg)
        for c in ids:
            renderer.remove_points(c)
