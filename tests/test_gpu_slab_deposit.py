"""The grid-copy deposit of the 2.5D calculators where its split changes: one node row per
slab, one to four slabs, the last slab cut short, the widest rows, the first grids that take
the tile sort instead, line densities of 1 to 4096 bins, and bunches around one workgroup's
and one part's particles.  Against the oracle, with the bars of test_gpu_sc.py."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2
from test_gpu_sc import _bunches

pytestmark = pytest.mark.gpu


def _coords(n, seed, ax=3e-3, ay=2.5e-3):
    r = np.random.default_rng(seed)
    c = r.standard_normal((6, n)) * np.array([ax, 1e-3, ay, 1e-3, 30.0, 1e-3])[:, None]
    return c


# 150 KiB of LDS: 148 rows of 128 nodes in one slab, 149 in two; 256 x 256 in four, 300 x 256
# in the tile sort; rows of 512 nodes are the widest, 513 go to the tile sort
GRIDS = [(3, 3, 4), (3, 512, 2), (4, 5, 1), (5, 300, 3), (147, 128, 16), (151, 128, 16),
         (200, 150, 100), (256, 256, 64), (300, 256, 8), (40, 513, 8), (70, 512, 8),
         (20, 24, 4096), (290, 64, 32)]


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("grid", GRIDS)
def test_step_on_every_split(grid, weights):
    import spacecharge
    n = 40_011
    c = _coords(n, 3)
    b, ob = _bunches(c)
    if weights:
        m = np.random.default_rng(2).uniform(0.5e8, 1.5e8, n)
        b.setMacroSizes(m)
        ob = O.Bunch(c, macrosize=1e8, kin_energy=1.0, msize=m)
    calc, ocalc = spacecharge.SpaceChargeCalc2p5Drb(*grid), O.SC2p5Drb(*grid)
    calc.trackBunch(b, 0.5, 0.1)
    ocalc.trackBunch(ob, 0.5, 0.1)
    out = b.getCoordinates()
    assert rel_l2(calc.getRhoGrid().array(), ocalc.grid(0)[0]) < 1e-12
    assert rel_l2(calc.getPhiGrid().array(), ocalc.grid(1)[0]) < 1e-12
    assert rel_l2(calc.getLongGrid().array(), ocalc.grid(2)[0]) < 1e-12
    m, om = calc.getMoments(), ocalc.moments()
    # the y position of a moment is xMin + iy * dx (as the reference has it): the terms reach
    # max(nx, ny) steps of dx
    span = (ocalc.grid(0)[1][1] - ocalc.grid(0)[1][0]) * max(grid[0], grid[1]) / (grid[0] - 1)
    assert np.allclose(m[:2], om[:2], rtol=0, atol=1e-13 * span)
    assert np.allclose(m[2:], om[2:], rtol=1e-12, atol=0)
    for k in (1, 3):
        assert rel_l2(out[k] - c[k], ob.coords[k] - c[k]) < 1e-10, k


# padded lengths 1024 to 4096 (the longest lines transform in place), on an axis of the copies'
# split, of the tile sort and of both
@pytest.mark.parametrize("grid", [(1100, 40, 64), (40, 1100, 64), (1025, 3, 1), (3, 2048, 4096),
                                  (2048, 9, 8), (1030, 1024, 16), (600, 260, 8)])
@pytest.mark.parametrize("plain", [False, True])
def test_step_on_long_axes(grid, plain):
    import spacecharge
    n = 30_011
    c = _coords(n, 4)
    b, ob = _bunches(c)
    if plain:
        calc, ocalc = spacecharge.SpaceChargeCalc2p5D(*grid), O.SC2p5D(*grid)
    else:
        calc, ocalc = spacecharge.SpaceChargeCalc2p5Drb(*grid), O.SC2p5Drb(*grid)
    args = (0.5,) if plain else (0.5, 0.1)
    calc.trackBunch(b, *args)
    ocalc.trackBunch(ob, *args)
    out = b.getCoordinates()
    for g in range(3):
        a = (calc.getRhoGrid(), calc.getPhiGrid(), calc.getLongGrid())[g].array()
        assert rel_l2(a, ocalc.grid(g)[0]) < 1e-12, g
    for k in (1, 3):
        assert rel_l2(out[k] - c[k], ob.coords[k] - c[k]) < 1e-10, k


@pytest.mark.parametrize("n", [2, 3, 1023, 1024, 1025, 2049, 262_145, 600_003])
def test_bunch_sizes_on_one_calculator(n):
    """Growing and shrinking bunches: the copies of an earlier, larger step are not read."""
    import spacecharge
    calc, ocalc = spacecharge.SpaceChargeCalc2p5Drb(160, 130, 24), O.SC2p5Drb(160, 130, 24)
    for size in (n, 700, n):
        c = _coords(size, size)
        b, ob = _bunches(c)
        calc.trackBunch(b, 0.5, 0.1)
        ocalc.trackBunch(ob, 0.5, 0.1)
        b.getCoordinates()
        assert rel_l2(calc.getRhoGrid().array(), ocalc.grid(0)[0]) < 1e-12
        assert rel_l2(calc.getLongGrid().array(), ocalc.grid(2)[0]) < 1e-12
        assert rel_l2(calc.getPhiGrid().array(), ocalc.grid(1)[0]) < 1e-12


@pytest.mark.parametrize("grid", [(3, 3, 4), (40, 600, 8), (64, 48, 16), (200, 150, 20),
                                  (30, 512, 4), (90, 20, 4)])
def test_green_rebuild_with_the_deposit(grid):
    """SpaceChargeCalc2p5D: the Green function rebuilt inside the deposit and column passes
    (and by the tile-sorted step for rows of 600 nodes), then kept, then rebuilt."""
    import spacecharge
    calc, ocalc = spacecharge.SpaceChargeCalc2p5D(*grid), O.SC2p5D(*grid)
    for k, (ax, ay) in enumerate([(3e-3, 3e-3), (6e-3, 2e-3), (6e-3, 2e-3), (1e-3, 4e-3)]):
        c = _coords(20_000, 50 + k, ax, ay)
        b, ob = _bunches(c)
        calc.trackBunch(b, 0.4)
        ocalc.trackBunch(ob, 0.4)
        out = b.getCoordinates()
        assert calc.getState()[3] == ocalc.state()[3]
        assert rel_l2(calc.getRhoGrid().array(), ocalc.grid(0)[0]) < 1e-12
        assert rel_l2(calc.getPhiGrid().array(), ocalc.grid(1)[0]) < 1e-12
        for q in (1, 3):
            assert rel_l2(out[q] - c[q], ob.coords[q] - c[q]) < 1e-10


@pytest.mark.parametrize("npts,nm", [(8, 1), (64, 0), (64, 16), (68, 31), (200, 33), (1000, 5),
                                      (20_475, 2), (20_476, 2), (30_000, 5)])
def test_boundary_sizes(npts, nm):
    """The boundary's correction for fewer points than lanes, one to seventeen rounds of rows
    per wave, no modes, and the most points that a workgroup's LDS holds and more, on a grid
    whose nodes end within a workgroup."""
    import spacecharge
    bnd = spacecharge.Boundary2D(npts, nm, "Ellipse", 0.05, 0.04)
    obnd = O.Boundary2D(npts, nm, "Ellipse", 0.05, 0.04)
    calc, ocalc = spacecharge.SpaceChargeCalc2p5D(45, 37, 8), O.SC2p5D(45, 37, 8)
    c = _coords(30_000, 7)
    b, ob = _bunches(c)
    calc.trackBunch(b, 0.5, bnd)
    ocalc.trackBunch(ob, 0.5, obnd)
    out = b.getCoordinates()
    # many modes fit few points badly conditioned: the projector's rounding, the same on both
    # sides, is then amplified by the order of the sum over the points (lane sums here)
    bar = 1e-12 if nm <= 16 else 1e-7
    assert rel_l2(calc.getPhiGrid().array(), ocalc.grid(1)[0]) < bar
    for k in (1, 3):
        assert rel_l2(out[k] - c[k], ob.coords[k] - c[k]) < 100 * bar


SLABS, TILES = (32, 24, 8), (40, 600, 8)


@pytest.mark.parametrize("between,grid,plain", [
    ("bunch", SLABS, False), ("bunch", TILES, False), ("bunch", SLABS, True),
    ("bunch", TILES, True), ("potential", SLABS, False), ("potential", TILES, False),
    ("batch", SLABS, False), ("batch_first", SLABS, False), ("replay", SLABS, False)])
def test_kick_waits_while_its_calculator_is_used(between, grid, plain):
    """A calculator writes its state, potential and line density again (another bunch's step,
    findPotential, a batch it belongs to) while a kick of it still waits: the kick is that of
    its own step, as when the bunch is read in between."""
    import spacecharge
    import teapot_base as TPB
    import _obnative as N
    from batch import BunchBatch
    from workloads import PIPE_RADIUS
    outs = []
    for eager in (False, True):
        first, second = (_bunches(_coords(n, 90, ax))[0]
                         for n, ax in ((9001, 3e-3), (20_011, 6e-3)))
        calc = (spacecharge.SpaceChargeCalc2p5D(*grid) if plain
                else spacecharge.SpaceChargeCalc2p5Drb(*grid))
        step = ((lambda b: calc.trackBunch(b, 0.5)) if plain
                else (lambda b: calc.trackBunch(b, 0.5, PIPE_RADIUS)))
        read = (lambda b: b.getCoordinates()) if eager else (lambda b: None)
        if between == "bunch":
            step(first)
            TPB.drift(first, 0.3)
            read(first)
            step(second)
        elif between == "potential":
            step(first)
            read(first)
            rho = np.random.default_rng(1).uniform(0, 1e9, grid[:2])
            phi = np.empty_like(rho)  # (the solver's own box)
            N.call("ob_sc2p5drb_find_potential", calc._h, N.dptr(rho), -1.0, 1.0, -1.0, 1.0,
                   N.dptr(phi))
        else:
            bb = BunchBatch([second], [calc])
            if between == "replay":
                bb.capture(lambda: bb.calculator().trackBunch(bb.bunch(), 0.5, PIPE_RADIUS))
            if between == "batch_first":
                bb.calculator().trackBunch(bb.bunch(), 0.5, PIPE_RADIUS)
                read(second)
                step(first)
            else:
                step(first)
                read(first)
                if between == "replay":
                    bb.replay(1)
                else:
                    bb.calculator().trackBunch(bb.bunch(), 0.5, PIPE_RADIUS)
        outs.append([first.getCoordinates(), second.getCoordinates()])
    for lazy, now in zip(*outs):
        for k in range(6):
            assert rel_l2(lazy[k], now[k]) < 1e-12, k
