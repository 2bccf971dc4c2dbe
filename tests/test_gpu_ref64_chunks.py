"""The FP64 step over chunk depths that its rule for small grids gives: two planes, a last chunk of
one, and chunks longer than the ten unrolled planes (more than 64 two-plane chunks), bit for bit
against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11


@pytest.mark.parametrize("dom", [(5, 9, 2), (34, 3, 3), (3, 2, 129), (2, 3, 700)])
def test_ref64_chunks(fl, oracle, dom):
    nx, ny, nz = dom
    shape = (nz + 8, ny + 8, nx + 8)
    r = np.random.RandomState(nz)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    st, d = 40, (12.5, 10.0, 8.0)  # the wave reaches several chunks up and down
    isrc = fl.index(shape, 4 + nx // 2, 4 + ny // 2, 4 + nz // 2)
    wav = r.standard_normal(st).astype(np.float32)
    ref = oracle.run("der1der1", shape, 4, d, DT, st, isrc, oracle.precompute(m, "f64"), fp="f64", src=wav)
    g = fl.Ref64(shape, d, DT, m)
    try:
        g.run(st, isrc, src=wav)
        got = {k: g.field(k) for k in ("pp", "pc", "qp", "qc")}
    finally:
        g.destroy()
    assert np.abs(ref["pc"]).max() > 0
    for k in got:
        assert np.array_equal(got[k], ref[k]), k
