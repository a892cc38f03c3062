"""Map programs at the edges of a launch: lengths around what the small and the large form of
the kernel arguments hold, the queue's own limit, programs whose shared coefficients change
midway (RingRF moves the synchronous momentum, dE kicks move dp/p), and every op kind in one
program.  Bit for bit against the oracle, map by map (soln and RingRF to a rounding)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

KINDS = [("drift", 0.3), ("quad1", 0.2, 0.7), ("quad1", 0.2, -0.7), ("quad2", 0.1),
         ("quadfringeIN", 0.6), ("quadfringeOUT", 0.6), ("multp", 2, 0.4, 0), ("multp", 3, 0.4, 1),
         ("multp", 0, 1e-4, 0), ("multpfringeIN", 2, 1.0, 0), ("multpfringeOUT", 3, 1.0, 1),
         ("multpfringeIN", 0, 0.01, 0), ("multpfringeOUT", 1, 0.5, 0), ("wrapbunch", 180.0),
         ("rotatexy", 0.3), ("kick", 1e-4, -1e-4, 1e-5), ("kick", 1e-4, 0.0, 0.0),
         ("bend1", 0.5, 0.05), ("bend3", 0.05), ("bend4", 0.05), ("bendfringeIN", 10.0),
         ("bendfringeOUT", 10.0), ("wedgerotate", 0.1, 0), ("wedgerotate", 0.1, 1),
         ("wedgedrift", 0.1, 0), ("wedgedrift", 0.1, 1), ("wedgebend", 0.1, 0, 10.0, 4),
         ("wedgebendCF", 0.1, 1, 10.0, 2, [1, 2], [0.1, 0.2], [0, 1], 4), ("soln", 0.3, 0.2),
         ("RingRF", 100.0, 1, 1e-5, 0.0, 1), ("RingRF", 100.0, 2, 1e-5, 0.3, 1), ("bend2", 0.2)]


def _coords(n, seed=4):
    r = np.random.default_rng(seed)
    return r.standard_normal((6, n)) * np.array([3e-3, 5e-4, 3e-3, 5e-4, 40.0, 1e-3])[:, None]


def _check(ops, n=513):
    import teapot_base as TPB
    from workloads import make_bunch
    c = _coords(n)
    b, ob = make_bunch(c), O.Bunch(c, macrosize=1e10, kin_energy=1.0)
    for op in ops:
        getattr(TPB, op[0])(b, *op[1:])
        ob.apply(*op)
    out = b.getCoordinates()
    if any(op[0] in ("soln", "RingRF") for op in ops):
        # their sin and cos differ from the oracle's in the last bit (2^-53 of the kick); the
        # maps after them magnify that by less than 1e3
        for k in range(6):
            scale = np.abs(ob.coords[k]).max()
            assert np.isfinite(scale) and np.abs(out[k] - ob.coords[k]).max() <= 1e-12 * scale, k
        return
    for k in range(6):
        assert np.array_equal(out[k], ob.coords[k]), (k, np.abs(out[k] - ob.coords[k]).max())


def test_every_op_in_one_program_and_twice():
    exact = [op for op in KINDS if op[0] not in ("soln", "RingRF")]
    _check(exact)
    _check(exact[::-1] + exact)
    _check(KINDS + KINDS[::-1])


# drift: 2 words, bend1: 11; the small form holds 48 words, the large 440, the queue 256 ops
@pytest.mark.parametrize("op,count", [(("drift", 0.01), m) for m in
                                      (1, 23, 24, 25, 219, 220, 221, 255, 256, 257, 600)] +
                         [(("bend1", 0.1, 0.01), m) for m in (4, 5, 39, 40, 41, 81)])
def test_program_lengths(op, count):
    _check([op] * count, n=65)


@pytest.mark.parametrize("steps", [131_069, 131_072, 262_147])
def test_wedgebend_of_many_steps(steps):
    _check([("drift", 0.01)] * 240 + [("wedgebendCF", 0.1, 1, 10.0, 1, [1], [0.1], [0], steps),
                                      ("wedgebend", 0.1, 0, 10.0, steps), ("drift", 0.1)], n=33)


@pytest.mark.parametrize("seed", range(4))
def test_random_programs(seed):
    r = np.random.default_rng(seed)
    # (strong maps in long random chains overflow: fewer of the nonlinear ones)
    ops = [KINDS[i] for i in r.integers(0, len(KINDS), 40)]
    _check(ops)


def test_coefficients_change_within_a_program():
    rf = ("RingRF", 100.0, 1, 1e-5, 0.4, 1)
    ops = []
    for k in range(12):
        ops += [("drift", 0.1), ("quad1", 0.2, 0.5), rf, ("bend3", 0.02), ("kick", 0.0, 0.0, 1e-5),
                ("quadfringeIN", 0.5), ("wedgerotate", 0.05, 0), ("quad2", 0.1)]
    _check(ops)
