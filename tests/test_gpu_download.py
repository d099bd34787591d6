"""Field downloads of every size class (one pinned copy, parts moved by the
caller's thread, parts moved by several threads) return what was set, from
several threads at once too."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu

MB = 1 << 17  # doubles


def system(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3))
    g = sp.ParticleSystem(sp.Box(0.0, 0.0, 0.0, 1.0, 1.0, 1.0), 0.25, "fp64")
    g.add_particles(x)
    return g, x, rng


# One field of n doubles and one of 3 n: around one pinned block (1 MB), a
# whole round of parts (4 MB) and the size from which threads share the work
# (24 MB, parts of 4 MB).
@pytest.mark.parametrize("n", [1, 7, MB - 1, MB, MB + 1, 4 * MB - 1, 4 * MB + 1, 8 * MB,
                               8 * MB + 1, 24 * MB - 1, 24 * MB, 24 * MB + 1, 28 * MB + 12345])
def test_sizes(n):
    g, x, rng = system(n, n)
    rho = rng.random(n)
    g.set("rho", rho)
    assert np.array_equal(g.get("rho"), rho)
    assert np.array_equal(g.get("x"), x)
    g.close()


def test_threads():
    def work(k):
        g, x, rng = system(300000 + 900001 * k, k)
        for _ in range(3):
            P = rng.random(len(x))
            g.set("P", P)
            assert np.array_equal(g.get("P"), P)
            assert np.array_equal(g.get("x"), x)
        g.close()
        return True

    with ThreadPoolExecutor(4) as ex:
        assert all(ex.map(work, range(4)))
