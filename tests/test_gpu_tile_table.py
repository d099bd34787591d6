"""The tile table on both sides of the grid size from which a thread takes
eight cells instead of one (2^17 cells in 2D, 2^18 in 3D): neighbour sets, orders and removals
are the oracle's, with the last block full, nearly empty and cut inside a
thread's cells."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [8, 32])
@pytest.mark.parametrize("cells", [(512, 256, 1), (131071, 1, 1), (131073, 1, 1), (513, 256, 1),
                                   (1, 133121, 1), (64, 64, 32), (65, 64, 32), (51, 52, 53),
                                   (64, 64, 64), (65, 64, 64), (131071, 1, 3), (67, 71, 73),
                                   (1030, 1021, 1)])
def test_both_tables(cells, T):
    n = 12000
    rng = np.random.default_rng(sum(cells) + T)
    hi = np.array([c - 0.5 for c in cells])  # inside the last cell
    if cells[2] == 1:
        hi[2] = 0.0
    x = rng.random((n, 3)) * hi
    x[: n // 2] = np.minimum(x[: n // 2], rng.random((n // 2, 3)) * 30.0)  # a dense corner
    x[n // 2: n // 2 + 500] = hi - np.minimum(hi, rng.random((500, 3)) * 3.0)  # and the last cells
    out = rng.choice(n, size=n // 30, replace=False)
    x[out, 1] = hi[1] + 1.0
    g = sp.ParticleSystem(sp.Box(0.0, 0.0, 0.0, *hi), 1.0, "fp64")
    g.set_tile(T)
    g.add_particles(x, rho=np.arange(n) + 1.0)
    o = O.OracleSystem(1.0, np.zeros(3), hi)
    o.load(x, np.zeros_like(x), np.arange(n) + 1.0, None, np.zeros(n))
    assert tuple(g.key_geometry()[1]) == cells
    for _ in range(2):  # the second build starts from the first one's order
        assert sp.create_cell_list(g) == n - len(out)
        o.create_cell_list()
        assert np.array_equal(g.get("rho"), o.field("rho"))
        counts, hashes = sp.neighbour_digest(g)
        co, ho = o.neighbour_digest()
        assert np.array_equal(counts, co) and np.array_equal(hashes, ho)
    g.set_tile(64 if T == 8 else 8)  # the table of the same cell list again
    counts, hashes = sp.neighbour_digest(g)
    assert np.array_equal(counts, co) and np.array_equal(hashes, ho)
