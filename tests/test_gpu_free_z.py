"""A flat periodic system bounds no particle's z, and beside a 2D system that is
not flat its z counts in the distances: tiles may then be far taller than a
cell, more than the matrix-core filter's error bound covers.  The sets are those
of a brute force over the minimum images in x and y."""
import numpy as np
import pytest

import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [32, 64])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("height", [0.0, 0.9, 1.4, 3.0, 20.0, 200.0])
def test_tall_tiles(height, precision, T):
    rng = np.random.default_rng(1)
    n, box = 900, 5.0
    x = rng.random((n, 3)) * box
    x[:, 2] = height * (rng.random(n) - 0.5)
    y = rng.random((50, 3)) * np.array([3.0, 3.0, 0.5])
    b = sp.Batch(precision)
    b.set_tile(T)
    i = b.add(x, 1.0, (0, 0, 0), (box, box, 0), periodic=True, m=1.0)
    b.add(y, 1.0, (0, 0, 0), (3, 3, 0.5), m=1.0)  # 2D, not flat
    b.build_cells()
    d = x[:, None, :] - x[None]
    d[..., :2] -= box * np.round(d[..., :2] / box)
    near = (d[..., 0] ** 2 + d[..., 1] ** 2) + d[..., 2] ** 2 <= 1.0
    np.fill_diagonal(near, False)
    got = np.zeros_like(near)
    p = b.neighbour_pairs(i)
    got[p[:, 0], p[:, 1]] = True
    assert len(p) == near.sum() and np.array_equal(got, near)
