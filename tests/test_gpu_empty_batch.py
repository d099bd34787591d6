"""Calls on a batch that holds no system: one that never held any, and one
whose systems have all been retired.  The tile size can be set and tuned, the
steps do nothing, and systems that join afterwards run as in a new batch."""
import numpy as np
import pytest

import smoothedparticles_hip as sp
from smoothedparticles_hip import states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("emptied", [False, True])
def test_batch_without_systems(emptied, precision):
    st = states.dam_break(2, 0.05)
    b = sp.Batch(precision)
    if emptied:
        ids = [b.add_state(st), b.add_state(st)]
        b.init_rho0()
        b.step(2)
        for i in ids:
            b.retire(i)
        b.step(1)  # the retired particles leave their cells
    b.build_cells()
    assert b.size() == (0, 0)
    for T in (8, 16, 32, 64, 0):
        b.set_tile(T)
    assert b.autotune() in (8, 16, 32, 64)
    assert b.step(3) == 0
    b.set_tile(16)

    def run(batch):
        i = batch.add_state(st)
        batch.init_rho0()
        pairs = batch.step(4)
        return pairs, [batch.get(i, f) for f in ("x", "v", "rho", "P")]

    other = sp.Batch(precision)
    other.set_tile(16)
    pairs, fields = run(b)
    want, wanted = run(other)
    assert pairs == want > 0
    for f, w in zip(fields, wanted):
        assert np.array_equal(f, w)
