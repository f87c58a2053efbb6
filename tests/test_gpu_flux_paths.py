"""The arithmetic and kernel forms the flux launches choose between give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(shape, seed, mhd=False):
    """Conservative state of order one with jumps, gas at rest and smooth parts (and a field)."""
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
    for c in (5, 6) if mhd else ():
        w[:, c] = .4 + .2 * r.random(n)
        w[:, 4] += .5 * w[:, c] ** 2
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


@pytest.mark.parametrize("shape", [(512, 513), (126, 2050), (2, 130000), (4000, 63), (64, 4100)], ids=str)
@pytest.mark.parametrize("subgrid,solver,boundary", [("ppm", "hllc", "wrap"), ("plm", "hllc", "edge"),
                                                     ("weno5", "llf", "edge")])
def test_marching_flux_equals_the_tiles(shape, subgrid, solver, boundary):
    """Fluxes and eigmax of a plan large enough for the marching flux launch
    against the allocation-free entry point, which runs the 2D tiles: sides
    that are one tile wide, one more, one less, shorter than a stencil."""
    import torch
    from astrea_amd.plan import Plan
    from tests.test_zz_no_alloc import _static_call
    plan = Plan(2, subgrid, solver, "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1], boundary=boundary, dx=1 / 512, gamma=1.4, cfl=.4, t_end=1e9)],
                varmask=0x17)
    plan.load([torch.from_numpy(_grid(shape, 5)).cuda()])
    for parity in (0, 1):
        ref = plan.evolve_space(parity)
        rc, f0, f1, eig = _static_call(plan, parity)
        assert rc == 0
        assert torch.equal(f0, ref[0]["raw"]) and torch.equal(f1, ref[1]["raw"])
        assert eig == [ref[0]["eigmax"], ref[1]["eigmax"]]
    plan.close()


@pytest.mark.parametrize("subgrid,solver,timestep,boundary,mhd", [
    ("ppm", "hllc", "ssprk(3,3)", "edge", False), ("plm", "llf", "rk4", "wrap", False),
    ("weno5", "hlld", "ssprk(3,3)", "wrap", True), ("ppm", "hlld", "rk4", "edge", True),
    ("plm", "hllc", "euler", "edge", False), ("plm", "hllc", "ssprk(2,2)", "edge", False),
    ("plm", "llf", "ssprk(4,3)", "edge", False), ("plm", "llf", "ssprk(5,3)", "wrap", False),
    ("ppm", "hllc", "ssprk(5,4)", "wrap", False), ("plm", "hllc", "ssprk(10,4)", "edge", False),
    ("plm", "hlld", "ssprk(10,4)", "wrap", True)])
def test_marching_batch_equals_its_problems_alone(subgrid, solver, timestep, boundary, mhd):
    """Three steps of a ragged batch, large enough together for the marching
    launch and the 1024-cell combination tiles, against each problem alone on
    the 2D tiles (and, but for the largest, 256-cell combination tiles), bit
    for bit."""
    import torch
    from astrea_amd.plan import Plan
    shapes = [(5, 7), (64, 63), (62, 126), (2, 9), (130, 33), (77, 205), (63, 64), (200, 3), (455, 480)]
    probs = [dict(n0=a, n1=b, boundary=boundary, dx=1 / max(a, b), gamma=1.4, cfl=.3, t_end=1e9) for a, b in shapes]
    grids = [torch.from_numpy(_grid(s, 11 + i, mhd)).cuda() for i, s in enumerate(shapes)]

    def run(ps, gs):
        plan = Plan(2, subgrid, solver, timestep, ps, varmask=0x77 if mhd else 0x17, magnetic_2d=mhd,
                    compat="physical")
        plan.load(gs)
        plan.reset()
        plan.step(3)
        out, st = plan.state.clone(), plan.status()
        offs = plan.offsets + [plan.total]
        plan.close()
        return [out[:, offs[i]:offs[i + 1]] for i in range(len(ps))], st
    both, st = run(probs, grids)
    for i in range(len(shapes)):
        (one,), (s1,) = run(probs[i:i + 1], grids[i:i + 1])
        assert torch.equal(torch.nan_to_num(both[i]), torch.nan_to_num(one)), shapes[i]
        assert st[i] == s1, shapes[i]


@pytest.mark.parametrize("shape", [(1,), (255,), (257,), (8, 32), (9, 31), (7, 33), (1, 70), (50, 2)], ids=str)
@pytest.mark.parametrize("subgrid,boundary", [("ppm", "wrap"), ("ppm", "edge"), ("plm", "edge")])
def test_snapshot_at_tile_edges_and_unaligned_buffers(shape, subgrid, boundary):
    """The snapshot of grids around one tile of the conversion kernel, into a
    16-byte aligned buffer and into one that is not, against the oracle's
    conversion of the same state."""
    import torch
    from astrea_amd.plan import Plan
    from oracle import astrea_oracle as O
    dims = len(shape)
    g = _grid(shape, 9)
    plan = Plan(dims, subgrid, "llf", "euler",
                [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary=boundary, dx=.1, gamma=1.4, cfl=.4,
                      t_end=1.)], varmask=0x13 if dims == 1 else 0x17)
    plan.load([g])
    s = O.Scheme(dimension=dims, subgrid=subgrid, boundary=boundary, gamma=1.4, dx=.1)
    w = O.to_prim(g, s)
    want = w if dims == 1 else np.ascontiguousarray(w.transpose(1, 0, 2))
    n = int(np.prod(shape)) * 8
    for skip in (0, 1):
        buf = torch.full((n + 2,), np.nan, dtype=torch.float64, device="cuda")
        out = buf[skip:skip + n].view(shape[::-1] + (8,))
        assert np.array_equal(plan.snapshot(0, out=out).cpu().numpy(), want)
        assert bool(torch.isnan(buf[:skip]).all()) and bool(torch.isnan(buf[skip + n:]).all())
    plan.close()


@pytest.mark.parametrize("flattener", ["off", "astrea"])
@pytest.mark.parametrize("boundary", ["wrap", "edge"])
@pytest.mark.parametrize("shapes", [((31, 9), (32, 8), (33, 7)), ((64, 4), (65, 5), (63, 3)), ((2, 3), (97, 130))], ids=str)
def test_shared_faces_match_each_cell_for_itself(shapes, boundary, flattener):
    """The PPM reconstruction with its faces shared between cells, against the
    fused sweep, which forms them per cell: bit for bit around its tiles."""
    import torch
    from astrea_amd.plan import Plan
    probs = [dict(n0=a, n1=b, boundary=boundary, dx=1 / max(a, b), gamma=1.4, cfl=.3, t_end=1e9) for a, b in shapes]
    grids = [torch.from_numpy(_grid(s, 21 + i)).cuda() for i, s in enumerate(shapes)]
    outs = []
    for fuse in (False, True):
        plan = Plan(2, "ppm", "hllc", "ssprk(3,3)", probs, varmask=0x17, flattener=flattener, compat="physical",
                    fuse2d=fuse)
        plan.load(grids)
        plan.reset()
        plan.step(3)
        outs.append((plan.state.clone(), plan.status()))
        plan.close()
    assert torch.equal(torch.nan_to_num(outs[0][0]), torch.nan_to_num(outs[1][0]))
    assert outs[0][1] == outs[1][1]


@pytest.mark.parametrize("tile_s", [0, 115])
@pytest.mark.parametrize("solver,flattener,av", [("hllc", "off", False), ("llf", "astrea", False), ("hllc", "astrea", True)])
@pytest.mark.parametrize("boundary", ["wrap", "edge"])
def test_one_dimensional_ppm_around_its_tiles(boundary, solver, flattener, av, tile_s):
    """1D PPM fluxes and wave speeds of grids around one and two tiles and far
    below one, against the oracle.  The kernel orders its operations as the
    oracle does, so only the last bits of a library root or power may differ:
    1e-14 of the largest flux, some 45 units in the last place."""
    from astrea_amd.plan import Plan
    from oracle import astrea_oracle as O
    for n in (2, 5, 114, 115, 116, 231, 242, 243, 244, 247, 487):
        g = _grid((n,), 31 + n)
        plan = Plan(1, "ppm", solver, "ssprk(3,3)",
                    [dict(n0=n, boundary=boundary, dx=1 / 64, gamma=1.4, cfl=.4, t_end=1e9)], varmask=0x13,
                    flattener=flattener, av=av, tile_s=tile_s)
        plan.load([g])
        got = plan.evolve_space(0)[0]
        plan.close()
        s = O.Scheme(dimension=1, subgrid="ppm", solver=solver, boundary=boundary, gamma=1.4, cfl=.4, dx=1 / 64,
                     flattener=flattener, av=av)
        want = O.evolve_space(g, s)[0]
        assert np.abs(got["flux"] - want["flux"]).max() <= 1e-14 * np.abs(want["flux"]).max(), n
        assert abs(got["eigmax"] - want["eigmax"]) <= 1e-14 * want["eigmax"], n


@pytest.mark.parametrize("shape,subgrid,boundary", [((5,), "plm", "edge"), ((128,), "ppm", "wrap"), ((300,), "ppm", "edge"),
                                                    ((510, 515), "ppm", "wrap"), ((516, 520), "plm", "wrap")], ids=str)
def test_short_divisions_and_roots_of_hlld_give_the_general_bits(shape, subgrid, boundary):
    """Velocity and field times a power of two and pressure times its square
    scale every operation exactly (the density cannot be scaled: the solver's
    inner states mix momenta and velocities, as the reference's, whose p* leaves
    a velocity out, so that the energy flux does not scale either).  The state of
    order one runs in the short arithmetic, the scaled ones lie outside its range
    and run in the general one.  The 2D grids are large enough for the marching
    launch."""
    from astrea_amd.plan import Plan
    dims = len(shape)
    base = _grid(shape, 5, mhd=True)
    if dims == 1:
        base[..., 5] = .75
        base[..., 7] = .3 * np.sin(np.arange(shape[0]))
        base[..., 4] += .6
    names = (0, 1, 2, 3, 5, 6, 7) if dims == 1 else (0, 1, 2, 5, 6)

    def fluxes(g):
        plan = Plan(dims, subgrid, "hlld", "ssprk(3,3)",
                    [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary=boundary, dx=1 / 64, gamma=1.4, cfl=.4,
                          t_end=1e9)], varmask=0xFF if dims == 1 else 0x77, magnetic_2d=dims == 2, compat="physical")
        plan.load([g])
        out = [plan.evolve_space(parity=q) for q in (0, 1)]
        plan.close()
        return out
    ref = fluxes(base)
    for c in (-60, -40, 20, 60):
        scale = [0] + 3 * [c] + [2 * c] + 3 * [c]  # rho, momenta, energy, field
        got = fluxes(np.ldexp(base, scale))
        for q in (0, 1):
            for ax in range(dims):
                want = np.ldexp(ref[q][ax]["flux"], [s + c for s in scale])
                for i in names:
                    # strong shocks have roots of negative densities, and NaNs, in both
                    assert np.array_equal(got[q][ax]["flux"][..., i], want[..., i], equal_nan=True), (c, q, ax, i)
                assert got[q][ax]["eigmax"] == np.ldexp(ref[q][ax]["eigmax"], c)


@pytest.mark.parametrize("shape", [(30,), (243,), (33, 9), (70, 40)], ids=str)
@pytest.mark.parametrize("subgrid", ["weno3", "weno5", "weno7"])
def test_short_divisions_of_the_weno_weights_give_the_general_bits(shape, subgrid):
    """One cell of huge velocity takes its
    tile's weights to the general arithmetic; the interfaces whose stencils do
    not reach it keep their bits."""
    base = _grid(shape, 41)
    far = base.copy()
    at = tuple(n // 2 for n in shape)
    rho = far[at][0]
    far[at][1] = rho * 2.0 ** (70 if subgrid != "weno7" else 9)
    far[at][4] += .5 * far[at][1] ** 2 / rho
    ref, got = _fluxes(base, subgrid, "hllc", "edge"), _fluxes(far, subgrid, "hllc", "edge")
    for ax in range(len(shape)):
        f, g = (x[0][ax]["flux"].reshape(shape[ax] + 1, -1, 8) for x in (ref, got))
        keep = np.abs(np.arange(len(f)) - at[ax] - .5) > 8  # conversion, stencil and interface reach less
        for t in range(f.shape[1]):
            sel = keep if len(shape) == 1 or abs(t - at[1 - ax]) <= 8 else np.ones_like(keep)
            assert np.array_equal(f[sel, t], g[sel, t]), (ax, t)


@pytest.mark.parametrize("shape", [(3, 5), (8, 64), (9, 65), (7, 63), (17, 130)], ids=str)
@pytest.mark.parametrize("boundary", ["wrap", "edge"])
def test_corner_reconstruction_around_its_tiles(shape, boundary):
    """Two Euler steps of 2D MHD on grids around one tile of the corner
    reconstruction (64 columns of 8 rows, either way round) against the oracle's
    constrained transport: 1e-13 of each component's largest value, some 450
    units in the last place for two steps."""
    from astrea_amd.plan import Plan
    from oracle import astrea_oracle as O
    a, b = shape
    dx = 1 / max(shape)
    g = np.zeros(shape + (8,))
    x, y = np.meshgrid((np.arange(a) + .5) * dx, (np.arange(b) + .5) * dx, indexing="ij")
    g[..., 0] = 1 + .2 * np.sin(7 * x + 3 * y)
    g[..., 1], g[..., 2] = g[..., 0] * .3 * np.cos(5 * y), g[..., 0] * .2 * np.sin(4 * x)
    g[..., 5], g[..., 6] = .4 + .2 * np.sin(6 * y), .3 * np.cos(5 * x)
    g[..., 4] = 2.5 + .3 * np.cos(9 * x) + .5 * (g[..., 1] ** 2 + g[..., 2] ** 2) / g[..., 0] + .5 * (
        g[..., 5] ** 2 + g[..., 6] ** 2)
    plan = Plan(2, "plm", "hlld", "euler",
                [dict(n0=a, n1=b, boundary=boundary, dx=dx, gamma=1.4, cfl=.2, t_end=1e9, max_steps=2)],
                varmask=0x77, magnetic_2d=True)
    plan.load([g])
    plan.reset()
    st = plan.run(2)[0]
    out = plan.unpack(0)
    plan.close()
    s = O.Scheme(dimension=2, subgrid="plm", solver="hlld", timestep="euler", boundary=boundary, gamma=1.4, cfl=.2,
                 dx=dx, magnetic_2d=True)
    ref = O.run(g, s, 1e9, max_steps=2).grid
    assert st["steps"] == 2 and not st["failed"]
    out = out.cpu().numpy() if hasattr(out, "cpu") else np.asarray(out)
    for i in range(8):
        assert np.abs(out[..., i] - ref[..., i]).max() <= 1e-13 * max(np.abs(ref[..., i]).max(), 1.), i


@pytest.mark.parametrize("shape", [(4000, 63), (63, 4000)], ids=str)
@pytest.mark.parametrize("subgrid", ["plm", "ppm"])
def test_marching_llf_writes_the_last_interface_from_the_last_tile(shape, subgrid):
    """A side of 63 cells splits into tiles of 31 and 32: the first one's last
    lane reaches interface 63, which only the second may write (periodic: the
    first has not the neighbour's radius there)."""
    import torch
    from astrea_amd.plan import Plan
    from tests.test_zz_no_alloc import _static_call
    plan = Plan(2, subgrid, "llf", "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1], boundary="wrap", dx=1 / 512, gamma=1.4, cfl=.4, t_end=1e9)], varmask=0x17)
    plan.load([torch.from_numpy(_grid(shape, 5)).cuda()])
    for parity in (0, 1):
        ref = plan.evolve_space(parity)
        rc, f0, f1, eig = _static_call(plan, parity)
        assert rc == 0
        assert torch.equal(f0, ref[0]["raw"]) and torch.equal(f1, ref[1]["raw"])
        assert eig == [ref[0]["eigmax"], ref[1]["eigmax"]]
    plan.close()


SPLIT_WENO = {((60,), "weno3"): "87ec14056994", ((60,), "weno5"): "f6f5dbaacdd6", ((60,), "weno7"): "37495a2602b1",
              ((19, 23), "weno3"): "28637c7286e8", ((19, 23), "weno5"): "ccc6b3d22937", ((19, 23), "weno7"): "6ec2d1575ab7"}


@pytest.mark.parametrize("shape,subgrid", SPLIT_WENO, ids=str)
def test_split_weno_keeps_its_rounding(shape, subgrid):
    """Split precision contracts multiplications into additions, so that its
    last bits follow the source form of the WENO weights: the fluxes' bytes
    (SHA-256, zeros made positive) are those of the form it was brought up with."""
    import hashlib
    from astrea_amd.plan import Plan
    dims = len(shape)
    plan = Plan(dims, subgrid, "llf", "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary="wrap", dx=1 / 64, gamma=1.4, cfl=.4, t_end=1e9)],
                varmask=0x13 if dims == 1 else 0x17, precision="split")
    plan.load([_grid(shape, 41)])
    out = plan.evolve_space(0)
    plan.close()
    got = hashlib.sha256(b"".join((out[ax]["flux"] + 0.).tobytes() for ax in out)).hexdigest()
    assert got.startswith(SPLIT_WENO[shape, subgrid])


@pytest.mark.parametrize("n", [60, 300, 700])
@pytest.mark.parametrize("subgrid", ["plm", "ppm", "weno3", "weno5", "weno7"])
def test_split_wave_speed_is_the_same_with_every_solver(n, subgrid):
    """The 1D wave speed of a stage comes from its interface states alone:
    split-precision HLLC, HLLD and LLF plans report the same one, bit for bit."""
    from astrea_amd.plan import Plan
    g = _grid((n,), 41, mhd=True)
    g[..., 5] = .75
    speed = {}
    for solver, mask in (("llf", 0x13), ("hllc", 0x13), ("llf", 0xFF), ("hllc", 0xFF), ("hlld", 0xFF)):
        q = g.copy()
        if mask == 0x13:
            q[..., 5:] = 0
        plan = Plan(1, subgrid, solver, "ssprk(3,3)",
                    [dict(n0=n, boundary="wrap", dx=1 / 64, gamma=1.4, cfl=.4, t_end=1e9)], varmask=mask, precision="split")
        plan.load([q])
        speed[solver, mask] = plan.evolve_space(0)[0]["eigmax"]
        plan.close()
    assert speed["hllc", 0x13] == speed["llf", 0x13]
    assert speed["hllc", 0xFF] == speed["hlld", 0xFF] == speed["llf", 0xFF]


@pytest.mark.parametrize("shape,subgrid,boundary", [((300,), "ppm", "edge"), ((300,), "ppm", "wrap"),
                                                    ((512, 513), "plm", "wrap"), ((513, 512), "ppm", "edge")], ids=str)
def test_hlld_with_a_field_along_the_sweep_that_carries_the_fast_wave(shape, subgrid, boundary):
    """A uniform field along x and a sound speed below the Alfven speed: the
    solver's rho (s - u)(s - s_M) - Bn^2 vanishes exactly wherever the gas is
    uniform, and fv.divide gives zero.  Short divisions (states of order one)
    against the general ones (the same states with velocity and field times
    2^-60 and pressure times 2^-120, which scales every operation exactly)."""
    from astrea_amd.plan import Plan
    dims, n = len(shape), int(np.prod(shape))
    cs2 = np.float64(1.4 * 2.0 ** -8)  # density, field 1
    cs2 = np.sqrt(cs2) ** 2
    cf = np.sqrt(.5 * (cs2 + 1. + np.sqrt((cs2 + 1.) ** 2 - 4 * cs2)))
    assert cf * cf - 1. == 0.
    at = np.arange(shape[0]).reshape((-1,) + (1,) * (dims - 1)) + np.zeros(shape)
    base = np.zeros(shape + (8,))
    base[..., 0] = np.where(at % 64 < 50, 1., .5)
    base[..., 1] = base[..., 0] * np.where(at % 96 < 40, .25, 0.)
    base[..., 5] = 1.
    base[..., 4] = np.where(at % 128 < 100, 2.0 ** -8, 2.0 ** -7) / .4 + .5 + .5 * base[..., 1] ** 2 / base[..., 0]
    out = []
    for c in (0, -60):
        plan = Plan(dims, subgrid, "hlld", "ssprk(3,3)",
                    [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary=boundary, dx=1 / 64, gamma=1.4, cfl=.4,
                          t_end=1e9)], varmask=0xFF if dims == 1 else 0x77, magnetic_2d=dims == 2, compat="physical")
        plan.load([np.ldexp(base, [0] + 3 * [c] + [2 * c] + 3 * [c])])
        out.append([plan.evolve_space(parity=q) for q in (0, 1)])
        plan.close()
    for q in (0, 1):
        for ax in range(dims):
            f, g = (o[q][ax]["flux"] for o in out)
            for i, s in enumerate([0] + 3 * [-60] + [None] + 3 * [-60]):
                if s is not None:  # the energy flux does not scale (p* leaves a velocity out)
                    assert np.isfinite(f[..., i]).all()
                    assert np.array_equal(g[..., i], np.ldexp(f[..., i], s - 60)), (q, ax, i)


def _smooth(shape, seed, mhd=False):
    """Conservative state of order one with moderate waves only (and a field):
    every interface is a weak one."""
    r = np.random.default_rng(seed)
    x, y = np.meshgrid(*((np.arange(n) + .5) / n for n in shape), indexing="ij")

    def wave(a, kx, ky):
        return a * np.sin(2 * np.pi * (kx * x + ky * y) + r.uniform(0, 2 * np.pi))
    g = np.zeros(shape + (8,))
    g[..., 0] = 1.2 + wave(.1, 1, 2)
    v = [.2 + wave(.1, 1, 1), -.1 + wave(.1, 2, 1)]
    b = [.3 + wave(.1, 0, 1), .25 + wave(.1, 1, 0)] if mhd else [0 * x, 0 * x]
    for c in (0, 1):
        g[..., 1 + c], g[..., 5 + c] = g[..., 0] * v[c], b[c]
    g[..., 4] = (1. + wave(.1, 2, 1)) / .4 + .5 * (g[..., 0] * (v[0] ** 2 + v[1] ** 2) + b[0] ** 2 + b[1] ** 2)
    return g


FORMS = [("plm", "llf", "wrap"), ("ppm", "hllc", "edge"), ("weno5", "hllc", "wrap"), ("plm", "hlld", "edge"),
         ("ppm", "hlld", "wrap"), ("weno5", "hlld", "edge"), ("weno5", "hlld", "wrap")]


@pytest.mark.parametrize("subgrid,solver,boundary", FORMS)
def test_narrow_problems_march_beside_a_large_one(subgrid, solver, boundary):
    """Two steps of a batch that a large problem takes to the marching launch,
    against each problem alone, which for all but the large one are the 2D
    tiles: bit for bit, finite, and the state has moved."""
    import torch
    from astrea_amd.plan import Plan
    mhd = solver == "hlld"
    shapes = [(5, 7), (64, 63), (62, 126), (2, 9), (130, 33), (1, 50), (63, 64), (200, 3), (290, 280), (1100, 1000)]
    probs = [dict(n0=a, n1=b, boundary=boundary, dx=1 / max(a, b), gamma=1.4, cfl=.3, t_end=1e9) for a, b in shapes]
    grids = [torch.from_numpy(_smooth(s, 11 + i, mhd)).cuda() for i, s in enumerate(shapes)]

    def run(ps, gs):
        plan = Plan(2, subgrid, solver, "ssprk(3,3)", ps, varmask=0x77 if mhd else 0x17, magnetic_2d=mhd,
                    compat="physical")
        plan.load(gs)
        plan.reset()
        first = plan.state.clone()
        plan.step(2)
        out, st = plan.state.clone(), plan.status()
        assert bool(torch.isfinite(out).all()) and not any(s["failed"] for s in st)
        offs = plan.offsets + [plan.total]
        plan.close()
        return [out[:, offs[i]:offs[i + 1]] for i in range(len(ps))], st, first
    both, st, first = run(probs, grids)
    assert not torch.equal(torch.cat(both, 1), first)
    for i in range(len(shapes) - 1):
        (one,), (s1,), _ = run(probs[i:i + 1], grids[i:i + 1])
        assert torch.equal(both[i], one), shapes[i]
        assert st[i] == s1, shapes[i]


@pytest.mark.parametrize("subgrid,solver", [("ppm", "hllc"), ("plm", "llf"), ("weno5", "hlld")])
def test_a_batch_keeps_its_bits_when_large_problems_end(subgrid, solver):
    """A batch whose problems end one after another, largest first, so that its
    flux launches split anew and then turn to the 2D tiles; twice from the
    start, the second time with the graphs of the first."""
    import torch
    from astrea_amd import batch
    from astrea_amd.plan import Plan
    mhd = solver == "hlld"
    shapes, steps = [(1100, 1000), (700, 650), (128, 100), (64, 300)], [2, 5, 11, 16]
    probs = [dict(n0=a, n1=b, boundary="wrap", dx=1 / 512, gamma=1.4, cfl=.3, t_end=1e9, max_steps=k)
             for (a, b), k in zip(shapes, steps)]
    grids = [torch.from_numpy(_smooth(s, 5 + i, mhd)).cuda() for i, s in enumerate(shapes)]

    def run(ps, gs, use_graph, times):
        plan = Plan(2, subgrid, solver, "ssprk(3,3)", ps, varmask=0x77 if mhd else 0x17, magnetic_2d=mhd,
                    compat="physical")
        out = []
        for _ in range(times):
            plan.load(gs)
            plan.reset()
            torch.cuda.synchronize()
            st, _, _ = batch.run(plan, chunk=2, use_graph=use_graph)
            out.append((plan.state.clone(), st))
        offs = plan.offsets + [plan.total]
        plan.close()
        return out, offs
    runs, offs = run(probs, grids, True, 2)
    runs += run(probs, grids, False, 1)[0]
    for i, k in enumerate(steps):
        (one, (s1,)), = run(probs[i:i + 1], grids[i:i + 1], False, 1)[0]
        assert s1["steps"] == k and not s1["failed"] and bool(torch.isfinite(one).all())
        for state, st in runs:
            assert torch.equal(state[:, offs[i]:offs[i + 1]], one), shapes[i]
            assert st[i] == s1


def _flux_us(shapes, subgrid, solver, ends=None):
    """Time of a step's flux launches, after the problems with an end have reached it."""
    import torch
    from astrea_amd.plan import Plan
    mhd = solver == "hlld"
    probs = [dict(n0=a, n1=b, boundary="wrap", dx=1 / max(a, b), gamma=1.4, cfl=.3, t_end=1e9,
                  max_steps=(ends[i] if ends else -1)) for i, (a, b) in enumerate(shapes)]
    plan = Plan(2, subgrid, solver, "ssprk(3,3)", probs, varmask=0x77 if mhd else 0x17, magnetic_2d=mhd, compat="physical")
    plan.load([torch.from_numpy(_smooth(s, 5, mhd)).cuda() for s in shapes])
    plan.reset()
    plan.step(2)
    if ends:
        plan.compact()
    best = np.inf
    for _ in range(4):
        plan.profile(200)
        plan.step(2)
        best = min(best, sum(ms for kind, (ms, _) in plan.profile_read().items() if "flux" in kind) / 2 * 1e3)
    plan.profile(0)
    assert not any(s["failed"] for s in plan.status())
    plan.close()
    return best


@pytest.mark.parametrize("subgrid,solver", [("ppm", "hllc"), ("plm", "llf"), ("weno5", "hlld")])
def test_a_small_problem_is_as_fast_beside_large_ones_that_have_ended(subgrid, solver):
    """The flux launches of a 96^2 problem left of a batch take the time of that
    problem alone (both forms' lines for the 2048^2 one took 2.4 to 3.2 times
    it), and 3/2 of it at most."""
    alone = _flux_us([(96, 96)], subgrid, solver)
    left = _flux_us([(2048, 2048), (96, 96)], subgrid, solver, ends=[2, -1])
    assert left <= 1.5 * alone, (left, alone)


@pytest.mark.parametrize("subgrid,solver", [("ppm", "hllc"), ("plm", "hllc"), ("weno5", "hlld")])
@pytest.mark.parametrize("shapes", [[(2, 130000)], [(16, 16)] * 1000], ids=["2x130000", "1000x16x16"])
def test_narrow_problems_are_not_slower_for_being_many(shapes, subgrid, solver):
    """Flux launches on sides that leave a wave's lanes idle: twice the cells
    take at most 2.2 times as long (the marching launch, which a number of cells
    alone once chose, took 2.6 to 3.0 times as long as the tiles of half)."""
    half = [(2, 65000)] if len(shapes) == 1 else shapes[::2]
    whole, part = _flux_us(shapes, subgrid, solver), _flux_us(half, subgrid, solver)
    assert whole <= 2.2 * part, (whole, part)


@pytest.mark.parametrize("shape", [(160, 160), (161, 159), (159, 161), (7, 3500), (3400, 31), (100001,), (100352,)], ids=str)
@pytest.mark.parametrize("subgrid,boundary", [("ppm", "wrap"), ("ppm", "edge"), ("plm", "edge")])
def test_large_snapshots_at_tile_edges_and_unaligned_buffers(shape, subgrid, boundary):
    """Snapshots large enough for the tiled conversion, of whole tiles and one
    cell more or less, against the oracle's conversion of the same state."""
    test_snapshot_at_tile_edges_and_unaligned_buffers(shape, subgrid, boundary)


def _snapshot_us(shape, subgrid, mhd):
    import torch
    from astrea_amd.plan import Plan
    dims = len(shape)
    plan = Plan(dims, subgrid, "llf", "euler", [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary="wrap", dx=.1,
                                                     gamma=1.4, cfl=.4, t_end=1.)],
                varmask=(0xFF if mhd else 0x13) if dims == 1 else (0x77 if mhd else 0x17))
    plan.load([torch.ones(shape + (8,), dtype=torch.float64, device="cuda")
               * torch.tensor([1., .1] + (dims == 2) * [.1] + (dims == 1) * [0.] + [0., 3.] + 3 * [0.], device="cuda")])
    out = plan.snapshot(0)
    best = np.inf
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(40):
            plan.snapshot(0, out=out)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) / 40 * 1e3)
    plan.close()
    return best


@pytest.mark.parametrize("subgrid,mhd", [("ppm", False), ("ppm", True), ("plm", False)])
def test_thin_snapshots_do_not_pay_for_whole_tiles(subgrid, mhd):
    """The snapshot of a domain two cells high takes at most twice the time of
    the same cells in a square (the tiles, which it fills to a sixteenth, took 3
    to 8 times)."""
    thin, square = _snapshot_us((70000, 2), subgrid, mhd), _snapshot_us((374, 374), subgrid, mhd)
    assert thin <= 2 * square, (thin, square)


@pytest.mark.parametrize("gamma", [-1.4, .6, 1 + 2. ** -52, 5 / 3, 40., 2. ** 70])
@pytest.mark.parametrize("shape", [(60,), (24, 20)], ids=str)
@pytest.mark.parametrize("solver", ["llf", "hllc"])
def test_any_adiabatic_index_takes_the_arithmetic_it_needs(shape, solver, gamma):
    """Fluxes and wave speed against the oracle for indices that the short
    divisions and roots do not cover (a negative one has sound speeds whose
    square is negative, and the wave speed of complex eigenvalues) and at the
    ends of those they do: 1e-13 of the largest flux of a component, some 450
    units in the last place for a library root of numpy's and its sums."""
    from astrea_amd.plan import Plan
    from oracle import astrea_oracle as O
    dims = len(shape)
    g = _grid(shape, 17)
    kin = .5 * (g[..., 1:4] ** 2).sum(-1) / g[..., 0]
    p = .4 * (g[..., 4] - kin)
    g[..., 4] = p / (gamma - 1) + kin
    plan = Plan(dims, "plm", solver, "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary="wrap", dx=1 / 64, gamma=gamma, cfl=.4,
                      t_end=1e9)], varmask=0x13 if dims == 1 else 0x17)
    plan.load([g])
    got = plan.evolve_space(0)
    plan.close()
    with np.errstate(all="ignore"):
        want = O.evolve_space(g, O.Scheme(dimension=dims, subgrid="plm", solver=solver, boundary="wrap", gamma=gamma, cfl=.4,
                                          dx=1 / 64))
    for ax in range(dims):
        f, h = got[ax]["flux"], want[ax]["flux"]
        assert np.array_equal(np.isnan(f), np.isnan(h))
        for c in range(8):
            top = np.nanmax(np.abs(h[..., c]), initial=0.)
            assert np.nanmax(np.abs(f[..., c] - h[..., c]), initial=0.) <= 1e-13 * top, (ax, c)
        e, w = got[ax]["eigmax"], want[ax]["eigmax"]
        assert (np.isnan(e) and np.isnan(w)) or abs(e - w) <= 1e-13 * w, (e, w)


@pytest.mark.parametrize("subgrid,boundary", [("ppm", "edge"), ("weno5", "wrap")])
def test_many_tubes_keep_the_bits_of_each(subgrid, boundary):
    """1D HLLD of more tubes than two workgroups per CU, in the general
    divisions, against each kind of tube alone, in the short ones."""
    import torch
    from astrea_amd.plan import Plan
    n = [130, 700, 1601, 257]
    tubes = []
    for i, m in enumerate(n):
        x = np.arange(m) / m
        g = np.zeros((m, 8))
        g[:, 0] = 1 + .1 * np.sin(7 * x + i)
        g[:, 1:4] = g[:, :1] * np.stack([.2 * np.cos(5 * x), .1 * np.sin(9 * x), .1 + 0 * x], 1)
        g[:, 5:] = np.stack([.75 + 0 * x, .3 * np.cos(6 * x), .2 * np.sin(8 * x)], 1)
        g[:, 4] = (1 + .1 * np.cos(4 * x)) / .4 + .5 * (g[:, 1:4] ** 2).sum(1) / g[:, 0] + .5 * (g[:, 5:] ** 2).sum(1)
        tubes.append(torch.from_numpy(g).cuda())

    def run(which):
        plan = Plan(1, subgrid, "hlld", "ssprk(3,3)",
                    [dict(n0=n[i], boundary=boundary, dx=1 / n[i], gamma=1.4, cfl=.4, t_end=1e9) for i in which],
                    varmask=0xFF)
        plan.load([tubes[i] for i in which])
        plan.reset()
        plan.step(3)
        out, st, offs = plan.state.clone(), plan.status(), plan.offsets + [plan.total]
        plan.close()
        assert bool(torch.isfinite(out).all()) and not any(s["failed"] for s in st)
        return [out[:, offs[k]:offs[k + 1]] for k in range(len(which))], st
    which = [i % 4 for i in range(100)]  # 25 x (2 + 6 + 13 + 3) tiles
    both, st = run(which)
    for i in range(4):
        (one,), (s1,) = run([i])
        for k in (i, 96 + i):
            assert torch.equal(both[k], one) and st[k] == s1


def _hlld_keeps_the_short_form(g):
    """Whether HLLD of neighbouring cells' states along the first axis (gamma =
    1.4) stays in the short divisions' range: star densities positive, the
    fast speeds' discriminants not negative, divisors not tiny."""
    rho = g[..., 0]
    u, b = g[..., 1:4] / rho[..., None], g[..., 5:8]
    p = .4 * (g[..., 4] - .5 * rho * (u ** 2).sum(-1) - .5 * (b ** 2).sum(-1))
    cs2, ca2, cax2 = 1.4 * p / rho, (b ** 2).sum(-1) / rho, b[..., 0] ** 2 / rho
    disc = (cs2 + ca2) ** 2 - 4 * cs2 * cax2
    cf = np.sqrt(.5 * (cs2 + ca2 + np.sqrt(np.maximum(disc, 0))))
    left, right = slice(None, -1), slice(1, None)
    rl, rr, ul, ur = rho[left], rho[right], u[left][..., 0], u[right][..., 0]
    lo, c = np.minimum(ul, ur), np.maximum(cf[left], cf[right])
    sl, sr = lo - c, lo + c
    bl, br = .5 * (b[left] ** 2).sum(-1), .5 * (b[right] ** 2).sum(-1)
    den = rl * (sl - ul) - rr * (sr - ur)
    sm = (p[right] - p[left] + rl * ul * (sl - ul) - rr * ur * (sr - ur) + br - bl) / den
    rls, rrs = rl * (sl - ul) / (sl - sm), rr * (sr - ur) / (sr - sm)
    return (disc[left] >= 0) & (disc[right] >= 0) & (rls > 2. ** -90) & (rrs > 2. ** -90) & (np.abs(den) > 2. ** -90)


@pytest.mark.parametrize("shape,subgrid,boundary", [((128,), "ppm", "wrap"), ((300,), "ppm", "wrap"),
                                                    ((700, 640), "ppm", "wrap"), ((640, 700), "plm", "edge")], ids=str)
def test_short_hlld_of_weak_waves_gives_the_general_bits(shape, subgrid, boundary):
    """As for strong shocks above, where nearly every wave of 64 lanes is solved
    in the general form after all: here the waves are weak, so that the state of
    order one stays in the short form, as its range evaluated on the host shows
    (1D, and the marching launch in 2D)."""
    from astrea_amd.plan import Plan
    dims = len(shape)
    if dims == 2:
        base = _smooth(shape, 3, mhd=True)
    else:
        base = _smooth(shape + (1,), 3, mhd=True)[:, 0]
        x = 2 * np.pi * np.arange(shape[0]) / shape[0]
        base[..., 3] = base[..., 0] * .1 * np.cos(x)
        base[..., 5], base[..., 7] = .75, .2 * np.sin(x)
        base[..., 4] += .7
    assert _hlld_keeps_the_short_form(base).all()
    if dims == 2:
        swap = base.swapaxes(0, 1)[..., [0, 2, 1, 3, 4, 6, 5, 7]]
        assert _hlld_keeps_the_short_form(swap).all()
    names = (0, 1, 2, 3, 5, 6, 7) if dims == 1 else (0, 1, 2, 5, 6)

    def fluxes(g):
        plan = Plan(dims, subgrid, "hlld", "ssprk(3,3)",
                    [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary=boundary, dx=1 / 64, gamma=1.4, cfl=.4,
                          t_end=1e9)], varmask=0xFF if dims == 1 else 0x77, magnetic_2d=dims == 2, compat="physical")
        plan.load([g])
        out = [plan.evolve_space(parity=q) for q in (0, 1)]
        plan.close()
        return out
    ref, got = fluxes(base), fluxes(np.ldexp(base, [0] + 3 * [-60] + [-120] + 3 * [-60]))
    for q in (0, 1):
        for ax in range(dims):
            f, g = ref[q][ax]["flux"], got[q][ax]["flux"]
            assert np.isfinite(f).all()
            for i in names:
                assert np.array_equal(g[..., i], np.ldexp(f[..., i], [0, -60, -60, -60, 0, -60, -60, -60][i] - 60)), (q, ax, i)


@pytest.mark.parametrize("subgrid,solver,boundary", [("ppm", "hllc", "wrap"), ("plm", "hllc", "edge"), ("weno5", "llf", "edge")])
def test_one_cell_outside_the_short_range_at_a_marching_size(subgrid, solver, boundary):
    """A transverse velocity of 2^-120 in one cell of a gas otherwise at rest
    across takes the lines that see it out of the short range, and only those:
    the marching launch against the 2D tiles, bit for bit."""
    import torch
    from astrea_amd.plan import Plan
    from tests.test_zz_no_alloc import _static_call
    g = _smooth((700, 640), 5)
    g[..., 4] -= .5 * g[..., 2] ** 2 / g[..., 0]
    g[..., 2] = 0.
    for at in ((333, 211), (0, 639)):
        g[at][2] = g[at][0] * 2. ** -120
    plan = Plan(2, subgrid, solver, "ssprk(3,3)",
                [dict(n0=700, n1=640, boundary=boundary, dx=1 / 512, gamma=1.4, cfl=.4, t_end=1e9)], varmask=0x17)
    plan.load([torch.from_numpy(g).cuda()])
    for parity in (0, 1):
        ref = plan.evolve_space(parity)
        rc, f0, f1, eig = _static_call(plan, parity)
        assert rc == 0
        assert bool(torch.isfinite(ref[0]["raw"]).all()) and bool(torch.isfinite(ref[1]["raw"]).all())
        assert torch.equal(f0, ref[0]["raw"]) and torch.equal(f1, ref[1]["raw"])
        assert eig == [ref[0]["eigmax"], ref[1]["eigmax"]]
    plan.close()


@pytest.mark.parametrize("subgrid,boundary", [("plm", "edge"), ("ppm", "wrap"), ("weno5", "edge"), ("weno5", "wrap")])
@pytest.mark.parametrize("shape", [(700, 640), (640, 505)], ids=str)
def test_marching_hlld_against_the_oracle(shape, subgrid, boundary):
    """HLLD fluxes and wave speeds of a grid large enough for the marching
    launch against the oracle's: 1e-13 of each component's largest flux, some
    450 units in the last place."""
    from astrea_amd.plan import Plan
    from oracle import astrea_oracle as O
    g = _smooth(shape, 9, mhd=True)
    plan = Plan(2, subgrid, "hlld", "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1], boundary=boundary, dx=1 / 512, gamma=1.4, cfl=.4, t_end=1e9)],
                varmask=0x77, magnetic_2d=True)
    plan.load([g])
    got = plan.evolve_space(0)
    plan.close()
    want = O.evolve_space(g, O.Scheme(dimension=2, subgrid=subgrid, solver="hlld", boundary=boundary, gamma=1.4, cfl=.4,
                                      dx=1 / 512, magnetic_2d=True))
    for ax in (0, 1):
        f, h = got[ax]["flux"], want[ax]["flux"]
        assert np.isfinite(f).all()
        for c in range(8):
            assert np.abs(f[..., c] - h[..., c]).max() <= 1e-13 * np.abs(h[..., c]).max(), (ax, c)
        assert abs(got[ax]["eigmax"] - want[ax]["eigmax"]) <= 1e-13 * want[ax]["eigmax"]


@pytest.mark.parametrize("flattener", ["off", "astrea"])
@pytest.mark.parametrize("boundary", ["wrap", "edge"])
@pytest.mark.parametrize("shapes", [((31, 9), (32, 8), (33, 7)), ((64, 4), (65, 5), (63, 3)), ((2, 3), (97, 130))], ids=str)
def test_shared_faces_of_smooth_states_match_each_cell_for_itself(shapes, boundary, flattener):
    """As above with a state that stays finite for the three steps, which are
    compared as they are."""
    import torch
    from astrea_amd.plan import Plan
    probs = [dict(n0=a, n1=b, boundary=boundary, dx=1 / max(a, b), gamma=1.4, cfl=.3, t_end=1e9) for a, b in shapes]
    grids = [torch.from_numpy(_smooth(s, 21 + i)).cuda() for i, s in enumerate(shapes)]
    outs = []
    for fuse in (False, True):
        plan = Plan(2, "ppm", "hllc", "ssprk(3,3)", probs, varmask=0x17, flattener=flattener, compat="physical",
                    fuse2d=fuse)
        plan.load(grids)
        plan.reset()
        plan.step(3)
        outs.append((plan.state.clone(), plan.status()))
        plan.close()
    assert bool(torch.isfinite(outs[0][0]).all()) and not any(s["failed"] for s in outs[0][1])
    assert torch.equal(outs[0][0], outs[1][0])
    assert outs[0][1] == outs[1][1]


def test_reset_leaves_lists_that_are_whole_alone():
    """Resetting a plan whose problems are all in the device's tile lists takes at
    most half the time of one whose lists have to be restored, copy by copy."""
    import time
    import torch
    from astrea_amd.plan import Plan
    plan = Plan(2, "plm", "hllc", "ssprk(3,3)",
                [dict(n0=n, n1=n, boundary="wrap", dx=1 / n, gamma=1.4, cfl=.3, t_end=1e9, max_steps=k)
                 for n, k in ((700, 1), (64, -1))], varmask=0x17, compat="physical")
    plan.load([torch.from_numpy(_smooth((n, n), 5)).cuda() for n in (700, 64)])
    plan.reset()

    def reset_us(dirty):
        best = np.inf
        for _ in range(8):
            if dirty:
                plan.step(1)
                plan.compact()
            torch.cuda.synchronize()
            t = time.perf_counter()
            plan.reset()
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t) * 1e6)
        return best
    restored, whole = reset_us(True), reset_us(False)
    plan.step(1)
    assert [s["active"] for s in plan.status()] == [False, True] or [s["steps"] for s in plan.status()] == [1, 1]
    plan.close()
    assert whole <= .5 * restored, (whole, restored)


@pytest.mark.parametrize("subgrid", ["plm", "weno3"])
def test_wave_speed_of_many_tiles_costs_a_first_stage_little(subgrid):
    """The first stage's launch, which gathers the wave speed of 2900 tiles, takes
    at most 1.1 times the average of all three stages (1.2 times it where every
    tile wrote to the one address), and the speed is the tiles' largest."""
    import torch
    from astrea_amd.plan import Plan
    n = 700035
    x = np.arange(n) / n
    g = np.zeros((n, 8))
    g[:, 0], g[:, 1] = 1 + .1 * np.sin(7 * x), .2 * np.cos(5 * x)
    g[:, 4] = 2.5 + .2 * np.cos(30 * x)
    at = 500000
    g[at, 4] = 4.  # the fastest cell, in the middle of a tile
    us, speed = {}, {}
    for rk in ("euler", "ssprk(3,3)"):
        plan = Plan(1, subgrid, "hllc", rk, [dict(n0=n, boundary="wrap", dx=1 / n, gamma=1.4, cfl=.3, t_end=1e9)], varmask=0x13)
        plan.load([torch.from_numpy(g).cuda()])
        speed[rk] = plan.evolve_space(0)[0]["eigmax"]
        plan.reset()
        plan.step(2)
        best = np.inf
        for _ in range(5):
            plan.profile(200)
            plan.step(2)
            ms, count = plan.profile_read()["sweep1d"]
            best = min(best, ms / count)
        plan.profile(0)
        plan.close()
        us[rk] = best * 1e3
    small = Plan(1, subgrid, "hllc", "euler", [dict(n0=41, boundary="edge", dx=1 / n, gamma=1.4, cfl=.3, t_end=1e9)], varmask=0x13)
    small.load([g[at - 20:at + 21]])
    assert speed["euler"] == speed["ssprk(3,3)"] == small.evolve_space(0)[0]["eigmax"]
    small.close()
    assert us["euler"] <= 1.1 * us["ssprk(3,3)"], us


SPLIT_HLLD = {((60,), "plm"): "285ce27e560a", ((60,), "ppm"): "487d14b5de47", ((300,), "weno5"): "3ba9833e3e57",
              ((19, 23), "pcm"): "73f03d578263", ((19, 23), "plm"): "3b2d59b985a6", ((40, 33), "ppm"): "d1326fd141be",
              ((40, 33), "weno5"): "c2f3e79e1a82"}


@pytest.mark.parametrize("shape,subgrid", SPLIT_HLLD, ids=str)
def test_split_hlld_keeps_its_rounding(shape, subgrid):
    """Split precision contracts multiplications into additions, so that the
    last bits of HLLD follow its order of operations: the bytes (SHA-256, zeros
    made positive) of the state after three steps are those of the order it was
    brought up with."""
    import hashlib
    import torch
    from astrea_amd.plan import Plan
    dims = len(shape)
    g = _smooth(shape if dims == 2 else shape + (1,), 41, mhd=True)
    plan = Plan(dims, subgrid, "hlld", "ssprk(3,3)",
                [dict(n0=shape[0], n1=shape[1] if dims == 2 else 1, boundary="wrap", dx=1 / 64, gamma=1.4, cfl=.4, t_end=1e9)],
                varmask=0xFF if dims == 1 else 0x77, magnetic_2d=dims == 2, compat="physical", precision="split")
    plan.load([g.reshape(shape + (8,))])
    plan.reset()
    plan.step(3)
    state = plan.state.cpu()
    assert bool(torch.isfinite(state).all()) and not plan.status()[0]["failed"]
    plan.close()
    assert hashlib.sha256((state + 0.).numpy().tobytes()).hexdigest().startswith(SPLIT_HLLD[shape, subgrid])


def test_wave_speed_of_few_tiles_costs_a_first_stage_little():
    """A forward Euler step of 448 flux tiles takes at most .385 of an SSPRK(3,3)
    step, whose other two stages gather no wave speed (.361 measured; .407 where
    tiles that few read the speed before they add their own)."""
    import time
    import torch
    from astrea_amd.plan import Plan
    g, us = torch.from_numpy(_smooth((336, 207), 9)).cuda(), {}
    for rk in ("euler", "ssprk(3,3)"):
        plan = Plan(2, "plm", "hllc", rk, [dict(n0=336, n1=207, boundary="wrap", dx=1 / 336, gamma=1.4, cfl=.3, t_end=1e9)],
                    varmask=0x17)
        plan.load([g])
        plan.reset()
        stream, best = torch.cuda.Stream(), np.inf
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            plan.step_graph(16)
            for _ in range(8):
                stream.synchronize()
                t = time.perf_counter()
                plan.step_graph(16)
                stream.synchronize()
                best = min(best, time.perf_counter() - t)
        us[rk] = best / 16e-6
        assert not plan.status()[0]["failed"]
        plan.close()
    assert us["euler"] <= .385 * us["ssprk(3,3)"], us
