"""Batches whose grids take the grid-copy deposit: one to four slabs, from five particles to
several parts a bunch, more bunches than the chip has CUs, a grid and a number of nodes that
send the whole batch to the tile sort, buffers that a calculator moves between two steps, macrosizes, and graph
replays.  Against each bunch on its own, with the bars of test_gpu_batch.py."""
import numpy as np
import pytest

from helpers import rel_l2
from test_gpu_batch import _lattice, _setup, _single

pytestmark = pytest.mark.gpu

CASES = {
    "slabs": ([5000, 70_003, 40_000, 131_073], [(16, 16, 8), (200, 150, 24), (256, 256, 4),
                                                (300, 64, 16)]),
    "few": ([5, 9, 1025, 2049], [(3, 3, 1), (5, 7, 2), (64, 64, 32), (33, 20, 5)]),
    "many": ([400 + 7 * k for k in range(280)], [(8 + k % 9, 8 + k % 5, 4) for k in range(280)]),
    "one": ([262_147], [(128, 128, 64)]),
    "bins": ([5000, 400_003, 30_000, 2000], [(16, 16, 256), (64, 64, 4096), (40, 30, 257),
                                             (8, 8, 65)]),
    "tiles": ([5000, 9000], [(32, 32, 16), (400, 400, 8)]),
    "nodes": ([2000 + 300 * k for k in range(11)], [(256, 256, 8)] * 8 + [(20, 30, 4)] * 3),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_against_single_bunches(case):
    from batch import BunchBatch
    sizes, grids = CASES[case]
    ref, refb = _single(1, sizes, grids)
    bunches, calcs = _setup(sizes, grids)
    bb = BunchBatch(bunches, calcs)
    _lattice(bb.calculator(), 1).trackBunch(bb.bunch())
    bb.synchronize()
    for k, b in enumerate(bunches):
        out = b.getCoordinates()
        for j in range(6):
            assert rel_l2(out[j], ref[k][j]) < 1e-9, (k, j)


@pytest.mark.parametrize("weights", [False, True])
def test_replays_and_a_moved_buffer(weights):
    """Replays equal direct cells; a calculator that tracks a larger bunch of its own in
    between moves its copies, and the next step finds them."""
    import spacecharge
    from batch import BunchBatch
    from workloads import make_bunch, gaussian_coords, PIPE_RADIUS
    sizes, grids = [20_000, 50_001], [(64, 64, 32), (200, 150, 16)]
    outs = []
    for replayed in (False, True):
        bunches, calcs = _setup(sizes, grids)
        if weights:
            for k, b in enumerate(bunches):
                b.setMacroSizes(np.random.default_rng(k).uniform(0.5e8, 1.5e8, sizes[k]))
        bb = BunchBatch(bunches, calcs)
        lat = _lattice(bb.calculator(), 1)
        lat.trackBunch(bb.bunch())
        if replayed:
            bb.capture(lambda: lat.trackBunch(bb.bunch()))
            for _ in range(3):
                bb.replay(1)
                bb.synchronize()
        else:
            for _ in range(3):
                lat.trackBunch(bb.bunch())
        for b in bunches:
            b.getCoordinates()  # (the waiting kicks read the calculators)
        big = make_bunch(gaussian_coords(600_000, seed=9))
        calcs[0].trackBunch(big, 0.1, PIPE_RADIUS)
        lat.trackBunch(bb.bunch())
        bb.synchronize()
        outs.append([b.getCoordinates() for b in bunches])
    for a, b in zip(*outs):
        for j in range(6):
            assert rel_l2(a[j], b[j]) < 1e-9, j


def _weights(n, seed):
    return np.random.default_rng(seed).uniform(0.5e8, 1.5e8, n)


def _set_weights(bunches, calcs):
    for k, b in enumerate(bunches):
        b.setMacroSizes(_weights(b.getSize(), 60 + k))


def _drop_weights(bunches, calcs):
    bunches[1].removePartAttr("macrosize")


def _macrosize(bunches, calcs):
    bunches[0].macroSize(3 * bunches[0].macroSize())


def _long_avg(bunches, calcs):
    calcs[1].setLongAveragingPointsN(7)


CHANGES = {"set": _set_weights, "removed": _drop_weights, "macrosize": _macrosize,
           "long_avg": _long_avg}


@pytest.mark.parametrize("grids", [[(64, 64, 32), (200, 150, 16)], [(64, 64, 32), (400, 400, 16)]])
@pytest.mark.parametrize("change", sorted(CHANGES))
def test_attributes_changed_between_steps(change, grids):
    """What a step reads of its bunches and calculators beside the coordinates, changed after
    the batch has tracked: the next cell is that of the bunches alone, a cell captured before
    the change is refused, one captured after it repeats the direct one."""
    from batch import BunchBatch
    from _obnative import OrbitError
    sizes = [20_000, 50_001]
    weighted = change == "removed"
    alone, acalcs = _setup(sizes, grids)
    batched, bcalcs = _setup(sizes, grids)
    if weighted:
        _set_weights(alone, acalcs)
        _set_weights(batched, bcalcs)
    lats = [_lattice(c, 1) for c in acalcs]
    bb = BunchBatch(batched, bcalcs)
    lat = _lattice(bb.calculator(), 1)
    lat.trackBunch(bb.bunch())
    bb.capture(lambda: lat.trackBunch(bb.bunch()))
    for b, la in zip(alone, lats):
        la.trackBunch(b)
    for bunches, calcs in ((alone, acalcs), (batched, bcalcs)):
        CHANGES[change](bunches, calcs)
    with pytest.raises(OrbitError, match="capture again"):
        bb.replay(1)
    lat.trackBunch(bb.bunch())
    bb.capture(lambda: lat.trackBunch(bb.bunch()))
    bb.replay(1)
    bb.synchronize()
    for k, (a, b, la) in enumerate(zip(alone, batched, lats)):
        la.trackBunch(a)
        la.trackBunch(a)
        ref, out = a.getCoordinates(), b.getCoordinates()
        for j in range(6):
            assert rel_l2(out[j], ref[j]) < 1e-9, (k, j)


def test_weights_set_one_by_one():
    """partAttrValue keeps the values on the host until the next step, as for a bunch alone."""
    from batch import BunchBatch
    sizes, grids = [3000, 5000], [(32, 32, 16), (16, 16, 8)]
    alone, acalcs = _setup(sizes, grids)
    batched, bcalcs = _setup(sizes, grids)
    lats = [_lattice(c, 1) for c in acalcs]
    bb = BunchBatch(batched, bcalcs)
    lat = _lattice(bb.calculator(), 1)
    for replayed in (False, True):
        for bunches in (alone, batched):
            bunches[0].addPartAttr("macrosize")
            for i in range(sizes[0]):
                bunches[0].partAttrValue("macrosize", i, 0, 1e7 * (1 + (i + replayed) % 5))
        if replayed:  # (the attribute is there already: the captured cell takes new values)
            bb.replay(1)
        else:
            lat.trackBunch(bb.bunch())
            bb.capture(lambda: lat.trackBunch(bb.bunch()))
        bb.synchronize()
        for k, (a, b, la) in enumerate(zip(alone, batched, lats)):
            la.trackBunch(a)
            ref, out = a.getCoordinates(), b.getCoordinates()
            for j in range(6):
                assert rel_l2(out[j], ref[j]) < 1e-9, (replayed, k, j)


def test_weights_of_a_bunch_brought_back_to_user_order():
    """A weighted bunch that a 3D calculator has left sorted joins a batch; a read puts it back
    in user order between two cells: coordinates and weights stay together."""
    import spacecharge
    from batch import BunchBatch
    sizes, grids = [30_011, 9000], [(64, 64, 32), (33, 20, 5)]
    outs = []
    for read in (False, True):
        bunches, calcs = _setup(sizes, grids)
        for k, b in enumerate(bunches):
            b.setMacroSizes(_weights(sizes[k], k) ** 2 * 1e-8)
            # (a kick of length 0 sorts the bunch and changes nothing else)
            spacecharge.SpaceChargeCalc3D(32, 32, 16).trackBunch(b, 0.0)
        bb = BunchBatch(bunches, calcs)
        lat = _lattice(bb.calculator(), 1)
        lat.trackBunch(bb.bunch())
        if read:
            for b in bunches:
                b.getCoordinates()
        lat.trackBunch(bb.bunch())
        bb.synchronize()
        outs.append([b.getCoordinates() for b in bunches])
    for a, b in zip(*outs):
        for j in range(6):
            assert rel_l2(b[j], a[j]) < 1e-9, j


def test_objects_that_go_during_a_capture():
    """A bunch is in a reference cycle with its synchronous particle, so the collector may free
    it, and a calculator, while a cell is being recorded: their end waits for the recording's."""
    import gc
    import spacecharge
    from batch import BunchBatch
    from workloads import gaussian_coords, make_bunch, PIPE_RADIUS
    sizes, grids = [3000, 5000], [(32, 32, 16), (16, 16, 8)]
    ref, _ = _single(2, sizes, grids)
    bunches, calcs = _setup(sizes, grids)
    bb = BunchBatch(bunches, calcs)
    lat = _lattice(bb.calculator(), 1)
    lat.trackBunch(bb.bunch())
    other = [make_bunch(gaussian_coords(2000, seed=3)), spacecharge.SpaceChargeCalc2p5Drb(8, 8, 4),
             spacecharge.SpaceChargeCalc3D(8, 8, 8), spacecharge.Boundary2D(16, 3, "Circle", 0.1)]
    other.append(BunchBatch([make_bunch(gaussian_coords(900, seed=4))]))
    other[1].trackBunch(other[0], 0.1, PIPE_RADIUS)

    def cell():
        other.clear()
        gc.collect()
        lat.trackBunch(bb.bunch())

    bb.capture(cell)
    bb.replay(1)
    bb.synchronize()
    for k, b in enumerate(bunches):
        out = b.getCoordinates()
        for j in range(6):
            assert rel_l2(out[j], ref[k][j]) < 1e-9, (k, j)


def test_a_batch_that_goes_while_it_records():
    """Its recording goes with it, and with that the maps and steps recorded: the bunches are
    left as they were, and track alone."""
    import _obnative as N
    from batch import BunchBatch
    from workloads import PIPE_RADIUS
    sizes, grids = [3000, 5000], [(32, 32, 16), (16, 16, 8)]
    bunches, calcs = _setup(sizes, grids)
    ref, rcalcs = _setup(sizes, grids)
    bb = BunchBatch(bunches, calcs)
    for b in ref:
        b.getCoordinates()
    N.call("ob_batch_capture_begin", bb._h)
    bb.calculator().trackBunch(bb.bunch(), 0.5, PIPE_RADIUS)
    bb.trackSequence([("drift", 0.7)])
    bb.__del__()
    for b, c, r, rc in zip(bunches, calcs, ref, rcalcs):
        assert np.array_equal(b.getCoordinates(), r.getCoordinates())
        c.trackBunch(b, 0.5, PIPE_RADIUS)
        rc.trackBunch(r, 0.5, PIPE_RADIUS)
        out, want = b.getCoordinates(), r.getCoordinates()
        for j in range(6):
            assert rel_l2(out[j], want[j]) < 1e-12, j
