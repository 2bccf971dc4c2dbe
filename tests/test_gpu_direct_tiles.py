"""The direct form at the edges of its 64 x 16 tiles and z chunks, bit for bit against the original
oracle: one column or row beyond whole tiles, fewer than four columns, an odd border, a depth
of one plane and of several chunks, unequal spacings, receivers on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11


@pytest.mark.parametrize("dom,bord,d", [
    ((65, 17, 9), 4, (12.5, 12.5, 12.5)),
    ((64, 16, 8), 4, (12.5, 10.0, 8.0)),
    ((3, 1, 33), 5, (12.5, 12.5, 12.5)),
    ((67, 31, 1), 7, (9.0, 12.5, 11.0)),
    ((1, 15, 70), 4, (12.5, 12.5, 12.5)),
])
def test_direct_tile_edges(fl, oracle, dom, bord, d):
    nx, ny, nz = dom
    shape = (nz + 2 * bord, ny + 2 * bord, nx + 2 * bord)
    r = np.random.RandomState(nx)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    fields = [f32(-1, 1) for _ in range(4)]  # the halo cells too
    st, rec = 4, bord + nz // 2
    isrc = fl.index(shape, bord + nx // 2, bord + ny // 2, rec)
    wav = r.standard_normal(st).astype(np.float32)
    ref = oracle.run("original", shape, bord, d, DT, st, isrc, oracle.precompute(m), fields=fields, rec_iz=rec,
                     rec_every=2, src=wav)
    g = fl.Driver(variant="direct")
    g.initialize(shape, d, DT, m, fields=fields, bord=bord)
    g.record_traces(rec, 2, st // 2)
    g.run(st, isrc, src=wav, graph_chunk=0)
    got, tr = {k: g.field(k) for k in ("pp", "pc", "qp", "qc")}, g.traces()
    g.finalize()
    for k in got:
        assert np.array_equal(got[k], ref[k]), k
    assert np.array_equal(tr, ref["traces"])
