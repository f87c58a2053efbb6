"""The arithmetic and kernel forms the flux launches choose between give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(shape, seed):
    """Conservative hydrodynamic state of order one with jumps, gas at rest and smooth parts."""
    r = np.random.default_rng(seed)
    n = int(np.prod(shape))
    w = np.zeros((n, 8))
    rho = np.where(np.arange(n) % 37 < 18, 1.0, .4) + .2 * r.random(n)
    p = np.where(np.arange(n) % 23 < 11, 1.0, .3) + .1 * r.random(n)
    w[:, 0], w[:, 4] = rho, p / .4
    for c in range(1, len(shape) + 1):
        v = np.where(r.random(n) < .3, 0., r.uniform(-1.5, 1.5, n))
        w[:, c] = rho * v
        w[:, 4] += .5 * rho * v * v
    return w.reshape(shape + (8,))


def _fluxes(grid, subgrid, solver, boundary):
    from astrea_amd.plan import Plan
    dims = grid.ndim - 1
    plan = Plan(dims, subgrid, solver, "ssprk(3,3)",
                [dict(n0=grid.shape[0], n1=grid.shape[1] if dims == 2 else 1, boundary=boundary, dx=1 / 64, gamma=1.4,
                      cfl=.4, t_end=1e9)], varmask=0x13 if dims == 1 else 0x17, compat="physical")
    plan.load([grid])
    out = [plan.evolve_space(parity=q) for q in (0, 1)]
    plan.close()
    return out


@pytest.mark.parametrize("shape", [(5,), (243,), (700,), (17, 11), (64, 35)], ids=str)
@pytest.mark.parametrize("solver", ["llf", "hllc"])
@pytest.mark.parametrize("subgrid,boundary", [("plm", "edge"), ("ppm", "wrap"), ("ppm", "edge")])
def test_short_divisions_and_roots_give_the_general_bits(shape, solver, subgrid, boundary):
    """Density, pressure and velocity times powers of two scale every operation
    of the update exactly, so the fluxes of a scaled state are the scaled
    fluxes, bit for bit.  The state of order one is solved with the short
    divisions and roots, the scaled ones lie outside their range (density and
    pressure of 2^-70 or 2^70; pressure of 2^-140 with velocities of 2^-70;
    one cell outside, so that only its own tile or wave leaves the range) and
    are solved with the general ones."""
    base = _grid(shape, 3)
    ref = _fluxes(base, subgrid, solver, boundary)
    for a, c in ((-70, 0), (70, 0), (0, -70)):  # exponents of density and velocity
        g = base.copy()
        scale = [a] + 3 * [a + c] + [a + 2 * c]  # rho, momenta, energy
        g[..., :5] = np.ldexp(g[..., :5], scale)
        got = _fluxes(g, subgrid, solver, boundary)
        for q in (0, 1):
            for ax in range(len(shape)):
                want = np.ldexp(ref[q][ax]["flux"][..., :5], [s + c for s in scale])
                assert np.array_equal(got[q][ax]["flux"][..., :5], want), (a, c, q, ax)
                assert got[q][ax]["eigmax"] == np.ldexp(ref[q][ax]["eigmax"], c)
