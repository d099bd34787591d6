"""The removals that the build's last kernel replays: one thread per system of
its first block, in rounds of 256 systems, after the block's part of the tile
table.  The orders are those of a replay of the reference's swap with the end
(src/core.jl:72-81) on the host."""
import numpy as np
import pytest

import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


def replayed(x, hi):
    """The particles that stay, in the reference's order after the removal."""
    order = list(range(len(x)))
    gone = np.nonzero(~np.all((x >= 0.0) & (x <= hi), axis=1))[0]
    end = len(order)
    for r in gone[::-1]:
        end -= 1
        order[r] = order[end]
    return x[order[:end]]


@pytest.mark.parametrize("nsys", [1, 2, 255, 256, 257, 600])
def test_removals_of_many_systems(nsys):
    rng = np.random.default_rng(nsys)
    hi = np.array([4.0, 4.0, 0.0])
    b = sp.Batch("fp64")
    xs = []
    for k in range(nsys):
        x = np.zeros((20 + k % 7, 3))
        x[:, :2] = rng.random((len(x), 2)) * (5.0 if k % 3 else 4.0)  # every third keeps all
        xs.append(x)
        b.add(x, 1.0, (0, 0, 0), hi, m=1.0)
    b.build_cells()
    for k in range(nsys):
        assert np.array_equal(b.get(k, "x"), replayed(xs[k], hi)), k


@pytest.mark.parametrize("leaving", [1, 777, 19999, 20000])
def test_removals_with_a_long_tile_table(leaving):
    """A table of 250 blocks; from one particle to all of them leave."""
    rng = np.random.default_rng(leaving)
    n, hi = 20000, np.array([39.5, 39.5, 39.5])
    x = rng.random((n, 3)) * hi
    out = rng.choice(n, leaving, replace=False)
    x[out, rng.integers(0, 3, leaving)] = 50.0
    s = sp.ParticleSystem(sp.Box(0, 0, 0, *hi), 1.0, "fp64")
    s.add_particles(x)
    assert sp.create_cell_list(s) == n - leaving
    want = replayed(x, hi)
    assert np.array_equal(s.get("x"), want)
    counts, _ = sp.neighbour_digest(s)
    d = want[:50, None, :] - want[None, :, :]  # (50 particles against all, by brute force)
    r = np.sqrt((d[..., 0] ** 2 + d[..., 1] ** 2) + d[..., 2] ** 2)
    assert np.array_equal(counts[:50], (r <= 1.0).sum(1) - 1)
