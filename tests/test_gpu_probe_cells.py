"""The cells a probe leaves out because they are out of reach: sums stay the
oracle's, bit for bit, for probes on cell faces and corners, beside and far
outside the box, at exact r == h ties, on grids so small that cells alias,
and at coordinates where a cell's face is not a round number."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [1.0, 0.0379, 250.0])
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 2), (2, 5, 1), (6, 5, 4), (9, 7, 1)])
@pytest.mark.parametrize("shift", [0.0, -3.3, 1.0e6])
def test_probe_cells(cells, h, shift):
    rng = np.random.default_rng(sum(cells))
    flat = cells[2] == 1
    lo = np.full(3, shift * h)
    hi = lo + np.array(cells) * h * 0.9999
    if flat:
        lo[2] = hi[2] = 0.0
    n = 3000
    x = lo + rng.random((n, 3)) * (hi - lo)
    corner = np.floor(x[:400] / h) * h  # on cell corners, where inside
    x[:400] = np.where((corner >= lo) & (corner <= hi), corner, x[:400])
    v = rng.normal(size=(n, 3))
    typ = (rng.random(n) < 0.3).astype(float)
    g = sp.ParticleSystem(sp.Box(*lo, *hi), h, "fp64")
    g.add_particles(x, v=v, type=typ)
    o = O.OracleSystem(h, lo, hi)
    o.load(x, v, None, None, typ)
    sp.create_cell_list(g)
    o.create_cell_list()
    tie = np.zeros(3)
    tie[0] = h
    probes = np.concatenate([
        lo - h + rng.random((400, 3)) * (hi - lo + 2.0 * h),
        np.round((lo + rng.random((200, 3)) * (hi - lo)) / h) * h,
        x[:200] + tie, x[200:300] - tie,
        lo + rng.normal(size=(50, 3)) * 50.0 * h])
    if flat:
        probes[::2, 2] = 0.0
    a = sp.probe_sums(g, probes, True, m=1.0)
    b = o.probe_sum(probes, 1.0, True)
    assert np.array_equal(a, b, equal_nan=True)
