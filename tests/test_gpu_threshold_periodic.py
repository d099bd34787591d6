"""Neighbour sets at the acceptance threshold in periodic boxes of three cells
per axis, whose cells are up to 4/3 h wide: the tiles' boxes are larger than
any other system's, so the candidate filter's sums are too.  Pairs from cell
corners outwards and across the seams; the sets are the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu

# Relative distances from the threshold in r: exact ties, one ulp beside them,
# inside the filter's error (3e-5 in r^2), around its band (4e-5 in r^2) and
# around the FP32 test's (1e-4 in r^2).
EPS = [0.0, 1e-16, 3e-16, 1e-13, 1e-10, 1e-8, 1e-6, 5e-6, 1e-5, 1.5e-5, 1.9e-5, 2.0e-5, 2.1e-5,
       4e-5, 5e-5, 1e-4]


def threshold_cloud(dim, h, box, n, seed):
    """n points, each with a partner at r = h (1 +- eps): a third anywhere, a
    third beside cell corners with the partner along the diagonal, and an
    eighth of all along an axis."""
    rng = np.random.default_rng(seed)
    cell = box / 3.0
    a = np.zeros((n, 3))
    d = np.zeros((n, 3))
    a[:, :dim] = rng.random((n, dim)) * box
    d[:, :dim] = rng.normal(size=(n, dim))
    k = n // 3
    a[:k, :dim] = cell * rng.integers(0, 4, (k, dim)) + 1e-3 * h * rng.normal(size=(k, dim))
    d[:k, :dim] = rng.choice([-1.0, 1.0], size=(k, dim)) * (1.0 + 0.2 * rng.normal(size=(k, dim)))
    d[k: k + n // 8] = 0.0
    d[k: k + n // 8, 0] = 1.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    eps = np.array(EPS)[np.arange(n) % len(EPS)] * rng.choice([-1.0, 1.0], size=n)
    return np.concatenate([a, a + d * (h * (1.0 + eps))[:, None]])


@pytest.mark.parametrize("T", [16, 32, 64])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("h", [1.0, 0.0192, 1023.9])
def test_three_cell_boxes(dim, h, precision, T):
    box = 3.999 * h
    x = threshold_cloud(dim, h, box, 1200 if dim == 2 else 2500, 3)
    lo, hi = np.zeros(3), np.zeros(3)
    hi[:dim] = box
    b = sp.Batch(precision)
    b.set_tile(T)
    i = b.add(x, h, lo, hi, periodic=True, m=1.0)
    b.build_cells()
    o = O.OracleSystem(h, lo, hi, periodic=True)
    o.load(x, np.zeros_like(x), None, None, np.zeros(len(x)))
    o.create_cell_list()
    cg, hg = b.neighbour_digest(i)
    co, ho = o.neighbour_digest()
    assert np.array_equal(cg, co) and np.array_equal(hg, ho)
