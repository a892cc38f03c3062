"""The diagnostics' reductions where their row counts, masked lanes and column counts change:
bunch sizes around a wave, a workgroup, a second particle per thread and the full grid of
workgroups, against sums in extended precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 64: a wave, 256: a workgroup, 2 * 256: two rows, 1024 * 256: the largest grid, twice that:
# the second particle of a thread
SIZES = [1, 2, 63, 65, 255, 257, 513, 8 * 256 + 1, 262_144, 262_145, 524_289]


def _coords(n):
    r = np.random.default_rng(n)
    c = r.normal(0.0, 1e-3, (6, n))
    c += np.array([1e-3, -2e-4, 5e-4, 1e-4, 0.3, 1e-3])[:, None]
    return c


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("n", SIZES)
def test_moments_extrema_and_radius(n, weights):
    import _obnative as N
    from orbit_utils import BunchExtremaCalculator
    from workloads import make_bunch
    c = _coords(n)
    b = make_bunch(c)
    w = np.random.default_rng(1).uniform(0.5, 2.0, n) if weights else np.ones(n)
    if weights:
        b.setMacroSizes(w)
    s = np.zeros(28)
    N.call("ob_bunch_moments", b._h, N.dptr(s))
    cols = [w] + [w * v for v in c] + [w * c[i] * c[j] for i in range(6) for j in range(i, 6)]
    # FP64 sums of n values in any order: relative error at most (log2-like depth) * 2^-53 of
    # the sum of magnitudes; n / 1024 sequential adds per thread are below 1e-12
    for k, v in enumerate(cols):
        e = v.astype(np.longdouble)
        assert abs(s[k] - float(e.sum())) <= 1e-13 * float(np.abs(e).sum()) + 1e-300, k
    out = np.zeros(12)
    N.call("ob_bunch_extrema", b._h, N.dptr(out))
    assert np.array_equal(out[0::2], c.min(axis=1)) and np.array_equal(out[1::2], c.max(axis=1))
    r = np.sqrt((c[0] - c[0].mean()) ** 2 + (c[2] - c[2].mean()) ** 2).max()
    # the mean's rounding moves the radius by an ulp or two of the coordinates
    assert abs(BunchExtremaCalculator().extremaR(b) - r) <= 1e-15 * n ** 0.5 + 1e-12 * r


@pytest.mark.parametrize("order", range(1, 13))
@pytest.mark.parametrize("n,weights", [(1, True), (257, False), (300_001, True)])
def test_power_sums_of_every_order(n, weights, order):
    import _obnative as N
    from workloads import make_bunch
    c = _coords(n)
    b = make_bunch(c)
    m = np.random.default_rng(1).uniform(0.5, 2.0, n) if weights else None
    if weights:
        b.setMacroSizes(m)
    xb, yb = 0.7, 1.3
    prm = np.array([1e-4, -2e-4, 0.5, 1.9, 0.77, xb, yb, 1.0])
    out = np.zeros(order * (order + 3) // 2 + 2)
    N.call("ob_bunch_xy_moments", b._h, order, N.dptr(prm), N.dptr(out))
    dx = (c[0] - 0.5 * c[5] / 1.9 / 0.77 - 1e-4).astype(np.longdouble)
    dy = (c[2] + 2e-4).astype(np.longdouble)
    fx, fy = (m * dx, m * dy) if weights else (dx, dy)
    k = 0
    for j in range(order):
        for i in range(order + 1 - j):
            t = fx ** i * fy ** j
            f = 1.0 / (xb ** i * yb ** j) + (1.0 if weights else 0.0)
            # a product of i + j factors and n terms: under 100 roundings of 2^-53 each
            assert abs(out[k] - float(t.sum()) * f) <= 1e-13 * float(np.abs(t).sum()) * f + 1e-300
            k += 1
    stray = float((dx ** 2 * dy ** order).sum()) if (order >= 2 and not weights) else 0.0
    assert abs(out[k] - stray) <= 1e-13 * float(np.abs(dx ** 2 * dy ** order).sum())
    assert out[k + 1] == pytest.approx(float(m.sum()) if weights else n, rel=1e-13)


@pytest.mark.parametrize("nz", [1, 2, 15, 16, 17, 257, 4096, 4097])
@pytest.mark.parametrize("n", [1, 257, 140_001])
def test_profile_of_every_width(n, nz):
    import spacecharge
    from workloads import make_bunch
    c = _coords(n)
    b = make_bunch(c, intensity=float(n))
    lo, hi = c[0].min() - 1e-4, c[0].max() + 1e-4
    g = spacecharge.Grid1D(nz, lo, hi)
    g.binBunch(b, 0)
    a = g.array()
    dz = (hi - lo) / nz
    ref = np.zeros(nz)
    if nz == 1:
        ref[0] = n
    else:
        i = ((c[0] - lo) / dz - 0.5).astype(np.int64)
        f = (c[0] - (lo + (i + 0.5) * dz)) / dz
        left = f < 0
        i0, ip = np.where(left, i - 1, i) % nz, np.where(left, i, i + 1) % nz
        w0 = np.where(left, -f, 1 - f)
        np.add.at(ref, i0, w0)
        np.add.at(ref, ip, 1 - w0)
    # weights from the same formulas; a bin adds up to n of them in another order
    assert np.abs(a - ref).max() <= 1e-12 * max(1.0, ref.max())


def test_deleted_particles_are_counted():
    """Deleting twice, adding after a deletion, deleting all: compress removes what was deleted
    and nothing more, however often it is called."""
    from workloads import make_bunch
    c = np.random.default_rng(1).standard_normal((6, 9)) * 1e-3
    b = make_bunch(c)
    for i in (3, 3, 7):
        b.deleteParticleFast(i)
    b.addParticle(*[1e-3] * 6)
    b.compress()
    b.compress()
    keep = [0, 1, 2, 4, 5, 6, 8]
    assert b.getSize() == 8
    assert np.array_equal(b.getCoordinates()[:, :7], c[:, keep])
    for i in range(8):
        b.deleteParticleFast(i)
    b.compress()
    assert b.getSize() == 0
    b.addParticle(*[1e-3] * 6)
    b.compress()
    assert b.getSize() == 1
