"""Unary operators on a handle that holds several systems (a batch handle is a
handle of sph.h): the call's parameters are the first system's, call by call,
and the others keep their own."""
import numpy as np
import pytest

import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsys", [1, 2, 3])
def test_unary_parameters_of_each_call(nsys):
    rng = np.random.default_rng(nsys)
    b = sp.Batch("fp64")
    own_dt = [0.5, 0.25, 0.125]
    ids, v, a = [], [], []
    for k in range(nsys):
        n = 40 + 300 * k
        x = np.zeros((n, 3))
        x[:, :2] = rng.random((n, 2)) * 3.0
        v.append(rng.normal(size=(n, 3)))
        a.append(rng.normal(size=(n, 3)))
        ids.append(b.add(x, 1.0, (0, 0, 0), (3, 3, 0), v=v[-1], m=1.0, rho0=1.0, dt=own_dt[k]))
        b.set(ids[-1], "a", a[-1])
    # the same parameters twice, others, and the first ones again
    for dt in (2.0, 2.0, 0.75, 2.0):
        sp.apply_unary(b, sp.kick, m=1.0, rho0=1.0, dt=dt)
        for k, i in enumerate(ids):
            v[k] = v[k] + (dt if k == 0 else own_dt[k]) * a[k]
            assert np.array_equal(b.get(i, "v"), v[k])
