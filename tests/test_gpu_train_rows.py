"""Every block's partial gradient is in the sum: the labels of one block at an
edge of the update kernel's staging (its first and last rows, the first row of
a later stage) are scaled until that block's part is a large share of the
gradient.  The share is checked on the oracle: losing the row moves the
gradient by several times the tolerance."""
import numpy as np
import pytest

import oracle as O
from test_mlp_oracle import NORM, random_labels, random_params, random_rays

CASES = [(1, 0), (127, 126), (128, 0), (128, 127), (129, 128), (201, 127), (201, 200), (256, 128), (256, 255)]
RAYS = 128  # rays of a gradient block
# bf16 operands on both sides, a gradient led by 128 rays: the bound that one block of rays has
TOL = 3e-2
_cache = {}


def _case(blocks, row):
    """(parameters, rays, labels, the oracle's gradient, the row's part of it)"""
    if (blocks, row) not in _cache:
        n = RAYS * blocks - 5
        p, rays, lab = random_params(71), random_rays(72, n, NORM), random_labels(73, n)
        part = slice(RAYS * row, min(n, RAYS * (row + 1)))
        lab[part, 0] *= np.float32(200.0 if blocks > 1 else 1.0)
        g, _ = O.mlp_gradients(p, NORM, rays, lab, bf16=True)
        gr, _ = O.mlp_gradients(p, NORM, rays[part], lab[part], bf16=True)
        _cache[blocks, row] = p, rays, lab, g, gr * np.float32((part.stop - part.start) / n)
    return _cache[blocks, row]


@pytest.mark.parametrize("blocks, row", CASES)
def test_a_lost_row_would_show(blocks, row):
    _, _, _, g, part = _case(blocks, row)
    assert np.linalg.norm(part) >= 5.0 * TOL * np.linalg.norm(g)


@pytest.mark.gpu
@pytest.mark.parametrize("blocks, row", CASES)
def test_every_row_is_summed(renderer, blocks, row):
    p, rays, lab, g, _ = _case(blocks, row)
    got, _ = renderer.mlp_gradients(p, NORM, rays, lab)
    assert np.linalg.norm(got - g) <= TOL * np.linalg.norm(g)
