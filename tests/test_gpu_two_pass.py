"""The two-pass form at the edges of pass 1 (two cells and four rows a thread) and of the loads pass 2
makes ahead: the derivative volumes against the same FP32 operations in numpy, bit for bit, zero
outside their ranges, and one step over tile heights and chunk depths of a plane and more.  Odd row
lengths, an odd border (a store of one cell at each end), rows not a multiple of four, a single
updated plane, unequal spacings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11
L = np.array([0.8, -0.2, 0.0380952380952381, -0.0035714285714285713], np.float32)


def der1(f, axis, h):
    """Der1 of derivatives.h:47 along an axis, float32 operations in its order (edges wrap)."""
    t = None
    for k in range(4):
        v = L[k] * (np.roll(f, -k - 1, axis) - np.roll(f, k + 1, axis))
        t = v if t is None else t + v
    return t * (np.float32(1.0) / np.float32(h))


@pytest.mark.parametrize("dom,bord,d", [
    ((33, 17, 9), 4, (12.5, 12.5, 12.5)),
    ((64, 16, 1), 4, (12.5, 10.0, 8.0)),
    ((1, 1, 21), 5, (12.5, 12.5, 12.5)),
    ((70, 30, 5), 7, (9.0, 12.5, 11.0)),
    ((259, 3, 2), 5, (12.5, 12.5, 12.5)),
])
def test_volumes_and_tiles(fl, dom, bord, d):
    nx, ny, nz = dom
    shape = (nz + 2 * bord, ny + 2 * bord, nx + 2 * bord)
    r = np.random.RandomState(nx)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    fields = [f32(-1, 1) for _ in range(4)]  # pp pc qp qc, the halo cells too
    sz, sy, sx = shape
    in_x = (slice(None), slice(None), slice(bord, sx - bord))
    in_y = (slice(None), slice(bord, sy - bord), slice(bord, sx))
    first = None
    for tiles in ((12, 0), (4, 1), (8, 3), (16, 0)):
        g = fl.Driver(variant="twopass", tiles=tiles)
        g.initialize(shape, d, DT, m, fields=fields, bord=bord)
        g.propagate(1)
        for k, (f, ax, rng) in enumerate([(1, 2, in_x), (1, 1, in_y), (3, 2, in_x), (3, 1, in_y)]):
            ref = np.zeros(shape, np.float32)
            ref[rng] = der1(fields[f], ax, d[2 - ax])[rng]
            assert np.array_equal(g.derivative_volume(k), ref), (tiles, k)
        got = [g.field(k) for k in ("pc", "qc")]
        g.finalize()
        assert not np.array_equal(got[0], fields[0])
        first = first or got
        for a, b in zip(got, first):
            assert np.array_equal(a, b), tiles
