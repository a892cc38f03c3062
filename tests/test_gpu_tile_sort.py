"""The tile sort of the 3D calculators where its path changes: tile counts around the limit
of the scan inside the scatter, bunches around one workgroup's and one work item's particles,
one z node, and the way back to user order, with and without macrosizes.  The tiled deposit
against the particle-order one of the same calculator: the same terms in another order, so rho
agrees to n eps / 2 of the largest node at worst and to sqrt(n) eps in the mean."""
import numpy as np
import pytest

from test_gpu_sc import _bunches

pytestmark = pytest.mark.gpu


def _coords(n, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((6, n)) * np.array([3e-3, 1e-3, 2.5e-3, 1e-3, 0.3, 1e-3])[:, None]


# 8 x 8 x 16 boxes: 64 x 64 x 256 nodes are 1024 tiles (scan in the scatter), 64 x 64 x 257
# and 72 x 64 x 256 more (scan launch)
GRIDS = [(64, 64, 256), (64, 64, 257), (72, 64, 256), (3, 3, 1), (9, 17, 2), (33, 8, 40)]


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("n", [2, 511, 513, 1025, 40_011])
@pytest.mark.parametrize("grid", GRIDS)
def test_sorted_deposit_and_order(grid, n, weights):
    import spacecharge
    c = _coords(n, n)
    b, _ = _bunches(c)
    if weights:
        b.setMacroSizes(np.random.default_rng(2).uniform(0.5e8, 1.5e8, n))
    calc, plain = spacecharge.SpaceChargeCalc3D(*grid), spacecharge.SpaceChargeCalc3D(*grid)
    plain.setDepositMode(False)
    for _ in range(3):  # (counters and rho are left clear for the next step)
        calc.trackBunch(b, 0.0)
    # a kick of length 0 leaves the bunch as it was, back in user order
    assert np.array_equal(b.getCoordinates(), c)
    if weights:
        assert np.array_equal(b.getMacroSizes(),
                              np.random.default_rng(2).uniform(0.5e8, 1.5e8, n))
    plain.trackBunch(b, 0.0)
    rho, ref = calc.getRhoGrid().array(), plain.getRhoGrid().array()
    assert np.abs(rho - ref).max() <= n * 1.2e-16 * np.abs(ref).max() + 4e-16 * np.abs(ref).max()
    assert np.isclose(rho.sum(), ref.sum(), rtol=1e-13)


def test_rho_is_kept_when_a_step_is_refused():
    import spacecharge
    c = _coords(500, 1)
    b, _ = _bunches(c)
    calc = spacecharge.SpaceChargeCalc3D(16, 16, 16)
    calc.trackBunch(b, 0.0)
    rho = calc.getRhoGrid().array().copy()
    flat, _ = _bunches(c * np.array([0, 1, 1, 1, 1, 1.])[:, None])
    with pytest.raises(Exception, match="zero extent"):
        calc.trackBunch(flat, 0.0)
    assert np.array_equal(calc.getRhoGrid().array(), rho)


MAPS = {"none": [], "short": [("drift", 0.5), ("quad1", 0.2, 0.7), ("bend1", 0.5, 0.05)],
        "level2": [("soln", 0.3, 0.2)], "long": [("quad1", 0.2, 0.3), ("drift", 0.3)] * 140}


@pytest.mark.parametrize("calc_name,grid", [("3d", (32, 30, 40)), ("3d", (16, 16, 2)),
                                            ("3d", (16, 16, 1)), ("slice", (32, 30, 9))])
@pytest.mark.parametrize("maps", sorted(MAPS))
def test_kick_waits_for_the_maps(calc_name, grid, maps):
    """The kick in one launch with the maps after it: as when the bunch is read in between, for
    two bunches of one calculator, a calculator that goes before they are read, and another
    calculator's step in between."""
    import teapot_base as TPB
    import spacecharge
    cls = (spacecharge.SpaceChargeCalc3D if calc_name == "3d"
           else spacecharge.SpaceChargeCalcSliceBySlice2D)
    coords = [_coords(20_011, 5), _coords(3_001, 6)]
    lazy, eager = ([_bunches(c)[0] for c in coords] for _ in range(2))
    other = [spacecharge.SpaceChargeCalc2p5Drb(16, 16, 8) for _ in range(2)]
    for which, bunches in enumerate((lazy, eager)):
        calc = cls(*grid)
        # (one step each: the box of a second one has its limits at the extreme particles, and
        # the last bit of a coordinate then decides whether they are deposited)
        for b in bunches:
            calc.trackBunch(b, 0.3)
            if which:
                b.getCoordinates()
            for op in MAPS[maps]:
                getattr(TPB, op[0])(b, *op[1:])
        other[which].trackBunch(bunches[0], 0.3, 0.1)
        del calc
    for b, e, c in zip(lazy, eager, coords):
        o1, o2 = b.getCoordinates(), e.getCoordinates()
        for k in range(6):
            # the particle order, and with it rho's rounding, differs: the bar of
            # test_gpu_sc.py for a sorted against a particle-order deposit
            assert np.abs(o1[k] - o2[k]).max() <= 1e-12 * np.abs(o2[k]).max(), k
            if k in (1, 3):  # (one node in z and slices: no dE kick)
                assert not np.array_equal(o1[k], c[k])


@pytest.mark.parametrize("n", [65_536, 65_537, 262_144, 262_145])
def test_item_sizes(n):
    """Work items of 256, 512 and 1024 particles, at the limits between them, most particles in
    one tile."""
    import spacecharge
    c = _coords(n, 8) * np.where(np.random.default_rng(9).random(n) < 0.9, 0.05, 1.0)
    b, _ = _bunches(c)
    calc, plain = spacecharge.SpaceChargeCalc3D(40, 40, 40), spacecharge.SpaceChargeCalc3D(40, 40, 40)
    plain.setDepositMode(False)
    b2, _ = _bunches(c)
    calc.trackBunch(b, 0.3)
    plain.trackBunch(b2, 0.3)
    rho, ref = calc.getRhoGrid().array(), plain.getRhoGrid().array()
    assert np.abs(rho - ref).max() <= n * 1.2e-16 * np.abs(ref).max()
    o1, o2 = b.getCoordinates(), b2.getCoordinates()
    for k in range(6):
        assert np.abs(o1[k] - o2[k]).max() <= 1e-12 * np.abs(o2[k]).max(), k
