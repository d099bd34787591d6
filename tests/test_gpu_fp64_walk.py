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
