"""Batches whose grids take the grid-copy deposit: one to four slabs, from five particles to
several parts a bunch, more bunches than the chip has CUs, a grid that sends the whole batch to
the tile sort, buffers that a calculator moves between two steps, macrosizes, and graph
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
    "tiles": ([5000, 9000], [(32, 32, 16), (400, 400, 8)]),
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
