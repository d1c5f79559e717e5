"""The training step's update kernel: the sum of the blocks' partial gradients
at row counts around its staging (1, one full stage, one row more, a ragged
last stage), and the packed network that a step writes next to its parameters."""
import numpy as np
import pytest

import j3d_amd as J
import oracle as O
from j3d_amd import ffi
from test_mlp_oracle import NORM, random_labels, random_params, random_rays

pytestmark = pytest.mark.gpu


# rays per gradient block: 4 chunks of 32
@pytest.mark.parametrize("blocks", [1, 127, 128, 129, 201, 256])
def test_gradient_sum_over_blocks(renderer, blocks):
    n = 128 * blocks - 5
    p = random_params(71)
    rays, lab = random_rays(72, n, NORM), random_labels(73, n)
    g, loss = renderer.mlp_gradients(p, NORM, rays, lab)
    go, lo = O.mlp_gradients(p, NORM, rays, lab, bf16=True)
    # bf16 operands on both sides: an activation next to a rounding boundary moves
    # by 2^-8 of its value; few rays do not average that away (3e-2 at 1 block)
    tol = 3e-2 if blocks == 1 else 1e-2
    assert np.linalg.norm(g - go) <= tol * np.linalg.norm(go)
    assert abs(loss - lo) <= 2e-3 * max(1.0, abs(lo))


@pytest.mark.parametrize("n_rays, batch", [(4096, 1024), (20000, 16384), (50001, 33024)])
def test_trained_network_is_the_packed_parameters(renderer, n_rays, batch):
    # the proposals of a frame come from the network as the steps packed it;
    # set_proposal packs the same parameters anew
    v, t = J.torus(80, 40, seed=6)
    slot = renderer.upload_mesh(v, t, db_id=J.make_db_id(1, 0))
    diag, pivot = J.scene_framing(v)
    cs, ci = J.orbit_camera(3.0, 0.9, 0.4)
    renderer.set_matcap(*J.make_matcap(0))
    tg = renderer.create_target(160, 90)
    fr = J.make_frame(160, 90, J.camera_with_vertical_fov(60.0), cs, ci, pivot, diag, [slot],
                      flags=J.ffi.EDGES | ffi.LEARNED, margin=0.05)
    try:
        rep = renderer.train_proposal(slot, n_rays=n_rays, batch=batch, epochs=2, seed=4, n_validation=0)
        assert np.isfinite(rep["loss_last"])
        renderer.render(fr, tg)
        trained = renderer.read_proposal(tg)
        params, norm = renderer.get_proposal(slot)
        renderer.set_proposal(slot, params, norm)
        renderer.render(fr, tg)
        packed = renderer.read_proposal(tg)
        assert np.array_equal(trained.view(np.uint32), packed.view(np.uint32))
        # every group moved
        assert np.all(np.isfinite(params)) and np.abs(params).max() > 0
    finally:
        renderer.destroy_target(tg)
        renderer.remove_mesh(slot)
