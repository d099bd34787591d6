"""The FP64 pair values where their square root and quotient could go wrong:
coincident particles (r = 0), separations far below h, pairs at r = h, and
several scales of h, against the oracle within the FP64 path's stated
tolerances (density and continuity 1e-12, force 1e-11 of the largest)."""
import numpy as np
import pytest

import oracle as O
import smoothedparticles_hip as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("h", [1.0, 0.0096, 3.0e5, 1.0e-9])
def test_small_and_zero_distances(dim, h):
    rng = np.random.default_rng(5 + dim)
    n = 600
    a = np.zeros((n, 3))
    a[:, :dim] = (0.5 + 3.0 * rng.random((n, dim))) * h
    d = np.zeros((n, 3))
    d[:, :dim] = rng.normal(size=(n, dim))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = np.concatenate([np.zeros(100), h * 10.0 ** rng.uniform(-15, -3, 300), np.full(100, h),
                        h * rng.random(100)])
    x = np.concatenate([a, a + d * r[:, None]])
    v = np.zeros_like(x)
    v[:, :dim] = rng.normal(size=(2 * n, dim))
    rho = 1000.0 * (1.0 + 0.1 * rng.random(2 * n))
    P = 1.0e4 * rng.normal(size=2 * n)
    lo, hi = np.zeros(3), np.zeros(3)
    hi[:dim] = 5.0 * h
    kw = dict(m=1000.0 * (h / 4.8) ** dim, rho0=1000.0, c=50.0, alpha=0.05, hs=h / 2.0, mu=1.0e-3,
              nu=1.0e-6, dt=1e-5)
    g = sp.ParticleSystem(sp.Box(*lo, *hi), h, "fp64")
    g.add_particles(x, v=v, rho=rho, P=P, type=np.zeros(2 * n))
    o = O.OracleSystem(h, lo, hi)
    o.load(x, v, rho, P, np.zeros(2 * n))
    assert sp.create_cell_list(g) == o.create_cell_list()  # (a few partners lie outside the box)
    sp.apply(g, sp.internal_force, **kw)
    o.internal_force(**kw)
    sp.apply(g, sp.balance_of_mass, **kw)
    o.balance_of_mass(**kw)
    sp.apply(g, sp.find_rho0, self=True, **kw)
    o.density_sum_rho0(True, **kw)

    def off(field, of):
        return np.max(np.abs(g.get(field) - of)) / np.max(np.abs(of))

    assert np.all(np.isfinite(g.get("a"))) and np.all(np.isfinite(g.get("rho0")))
    assert off("a", o.field("a")) <= 1e-11
    assert off("Drho", o.field("Drho")) <= 1e-12
    assert np.max(np.abs(g.get("rho0") / o.field("rho0") - 1.0)) <= 1e-12


@pytest.mark.parametrize("field,value", [("rho", np.inf), ("rho", -1000.0), ("v", np.inf),
                                         ("v", -np.inf), ("v", np.nan)])
def test_non_finite_quotients(field, value):
    """One particle with an infinite density (its pairs' viscous quotients are
    0), one that makes the mean density of a pair 0 (infinite quotients), or a
    velocity that is no number: the accelerations are finite, infinite and NaN
    where the oracle's are, the finite ones within 1e-11 of the largest."""
    rng = np.random.default_rng(11)
    n, h = 200, 0.5
    x = 0.05 + 0.9 * rng.random((n, 3))
    v = rng.normal(size=(n, 3))
    rho = np.full(n, 1000.0)
    P = 1.0e4 * rng.normal(size=n)
    if field == "rho":
        rho[7] = value
    else:
        v[7, 0] = value
    kw = dict(m=1.0, rho0=1000.0, c=50.0, alpha=0.05, hs=h / 2.0, mu=0.0, nu=0.0, dt=1e-5)
    g = sp.ParticleSystem(sp.Box(0, 0, 0, 1, 1, 1), h, "fp64")
    g.add_particles(x, v=v, rho=rho, P=P, type=np.zeros(n))
    o = O.OracleSystem(h, np.zeros(3), np.ones(3))
    o.load(x, v, rho, P, np.zeros(n))
    assert sp.create_cell_list(g) == o.create_cell_list()
    sp.apply(g, sp.internal_force, **kw)
    o.internal_force(**kw)
    got, want = g.get("a"), o.field("a")
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    if fin.any():
        assert np.max(np.abs(got[fin] - want[fin])) <= 1e-11 * np.max(np.abs(want[fin]))
