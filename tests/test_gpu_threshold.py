"""Neighbour sets at the acceptance threshold for every tile size: the matrix
cores only filter the candidates (T = 32 and 64), and pairs close to r == h
are settled by the FP64 predicate, so the sets are the oracle's, bit for bit,
whatever the scale of h."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu

# Relative distances from the threshold: exact ties and one ulp beside them,
# inside the filter's error (2e-5 in r^2), inside and around its band (4e-5 in
# r^2, 2e-5 in r), and around the FP32 test's (1e-4 in r^2).
EPS = [0.0, 1e-16, 3e-16, 1e-13, 1e-10, 1e-8, 1e-6, 5e-6, 1e-5, 1.9e-5, 2.0e-5, 2.1e-5, 4e-5,
       5e-5, 1e-4]


def threshold_cloud(dim, h, n, seed):
    """Random points, each with a partner at r = h (1 +- eps)."""
    rng = np.random.default_rng(seed)
    a = np.zeros((n, 3))
    a[:, :dim] = rng.random((n, dim)) * 4.0 * h + h
    d = np.zeros((n, 3))
    d[:, :dim] = rng.normal(size=(n, dim))
    d[: n // 8] = 0.0
    d[: n // 8, 0] = 1.0  # along an axis: exact ties
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    eps = np.array(EPS)[np.arange(n) % len(EPS)] * rng.choice([-1.0, 1.0], size=n)
    return np.concatenate([a, a + d * (h * (1.0 + eps))[:, None]])


@pytest.mark.parametrize("T", [16, 32, 64])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("h", [1.0, np.nextafter(1.0, 0.0), 0.0192, 3.7e4])
def test_threshold_sets(dim, h, precision, T):
    x = threshold_cloud(dim, h, 1200 if dim == 2 else 2500, 3)
    hi = np.zeros(3)
    hi[:dim] = 6.0 * h
    g = sp.ParticleSystem(sp.Box(0.0, 0.0, 0.0, *hi), h, precision)
    g.set_tile(T)
    g.add_particles(x)
    o = O.OracleSystem(h, np.zeros(3), hi)
    o.load(x, np.zeros_like(x), None, None, np.zeros(len(x)))
    sp.create_cell_list(g)
    o.create_cell_list()
    cg, hg = sp.neighbour_digest(g)
    co, ho = o.neighbour_digest()
    assert np.array_equal(cg, co) and np.array_equal(hg, ho)
