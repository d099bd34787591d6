"""The cell build's scans and tile table over grids of every shape, and how
the pair passes hand out their tiles: every tile is worked exactly
once whatever the number of tiles against the blocks the chip holds (a wave
is dealt its first tile, or four in 2D, and takes the rest from the queues),
and the wave's pair counts add up over the copies of the counters."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


def cloud(n, dim, per_cell, seed):
    """n uniform points of a box of about n / per_cell cells of side 1."""
    cells = max(1, int(round((n / per_cell) ** (1.0 / dim))))
    rng = np.random.default_rng(seed)
    x = np.zeros((n, 3))
    x[:, :dim] = rng.random((n, dim)) * cells
    hi = np.zeros(3)
    hi[:dim] = cells
    return x, hi


# With T = 8 and ~8 particles per cell a system has n / 5 to n / 8 tiles: from
# one tile over fewer than the 6144-8192 resident blocks, about as many, and
# several per block to more than four per block.
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim,n", [(2, 1), (2, 9), (2, 700), (2, 40000), (2, 47000), (2, 260000),
                                   (3, 11), (3, 41000), (3, 90000)])
def test_every_tile_once(dim, n, precision):
    x, hi = cloud(n, dim, 8, n)
    g = sp.ParticleSystem(sp.Box(0.0, 0.0, 0.0, *hi), 1.0, precision)
    g.set_tile(8)
    g.add_particles(x)
    o = O.OracleSystem(1.0, np.zeros(3), hi)
    o.load(x, np.zeros_like(x), None, None, np.zeros(n))
    sp.create_cell_list(g)
    o.create_cell_list()
    counts, hashes = sp.neighbour_digest(g)
    co, ho = o.neighbour_digest()
    assert np.array_equal(counts, co) and np.array_equal(hashes, ho)
    # c = 0 and dt = 0: nothing moves, so every step has the same pairs
    pairs = sp.step(g, 3, scheme="wcsph_se", m=1.0, rho0=1.0, hs=0.5)
    dens, force = g.step_pairs()
    assert pairs == dens == force == 3 * int(co.sum())


# Grids cut by the bricks of the tile table on every side, and grids of more
# than 64 scan blocks (131,072 buckets) and tile blocks (65,536 cells), past
# one look back along the chain; a sparse cloud, some particles outside.
@pytest.mark.parametrize("T", [8, 64])
@pytest.mark.parametrize("cells,n", [((1, 1, 1), 40), ((4, 4, 4), 900), ((5, 7, 9), 4000),
                                     ((3, 13, 1), 500), ((17, 8, 1), 2000), ((90, 61, 31), 9000),
                                     ((640, 411, 1), 30000), ((70, 83, 59), 20000)])
def test_grid_shapes(cells, n, T):
    rng = np.random.default_rng(n + T)
    hi = np.array([c - 0.5 for c in cells])  # inside the last cell
    if cells[2] == 1:
        hi[2] = 0.0
    x = rng.random((n, 3)) * hi
    out = rng.choice(n, size=n // 20 + 1, replace=False)
    x[out, 0] = hi[0] + 1.0 + rng.random(len(out))
    x[out[0]] = np.nan
    if cells[2] == 1:
        x[:, 2] = 0.0
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
