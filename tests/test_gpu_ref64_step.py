"""The one-pass FP64 step at the edges of its tiles and chunks, bit for bit against the FP64
oracle: one column or row beyond whole 32 x 8 tiles, chunks shorter and longer than the ten
unrolled planes, a wider border, unequal spacings, and a source cell that no step stores."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11  # a float: the oracle takes dt in double, the library as a float


@pytest.mark.parametrize("dom,bord,d,src", [
    ((33, 9, 8), 4, (12.5, 12.5, 12.5), "inside"),
    ((32, 8, 9), 4, (12.5, 10.0, 8.0), "inside"),
    ((31, 17, 41), 6, (12.5, 12.5, 12.5), "inside"),
    ((65, 7, 27), 4, (9.0, 12.5, 11.0), "halo"),
    ((1, 1, 1), 4, (12.5, 12.5, 12.5), "inside"),
])
def test_ref64_step_edges(fl, oracle, dom, bord, d, src):
    nx, ny, nz = dom
    shape = (nz + 2 * bord, ny + 2 * bord, nx + 2 * bord)
    r = np.random.RandomState(nx)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    isrc = fl.index(shape, bord + nx // 2, bord + ny // 2, bord + nz // 2 if src == "inside" else bord - 2)
    st, rec = 13, bord + nz // 2
    wav = r.standard_normal(st).astype(np.float32)
    ref = oracle.run("der1der1", shape, bord, d, DT, st, isrc, oracle.precompute(m, "f64"), fp="f64",
                     rec_iz=rec, rec_every=2, src=wav)
    g = fl.Ref64(shape, d, DT, m, bord=bord)
    try:
        g.run(5, isrc, src=wav[:5], rec_iz=rec, rec_every=0)
        g.run(st - 5, isrc, it0=5, src=wav[5:], rec_iz=rec, rec_every=2, max_traces=st // 2)
        got = {k: g.field(k) for k in ("pp", "pc", "qp", "qc")}
        tr = g.traces()
    finally:
        g.destroy()
    assert np.abs(ref["pc"]).max() > 0
    for k in got:
        assert np.array_equal(got[k], ref[k]), k
    assert np.array_equal(tr, ref["traces"][2:])  # steps 6, 8, 10, 12
