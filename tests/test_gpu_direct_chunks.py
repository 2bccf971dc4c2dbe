"""The direct form over the chunk depths of its rule: one plane, a few, and chunks that go round the
ten-plane ring (more than 64 one-plane chunks), bit for bit against the original oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11


@pytest.mark.parametrize("dom", [(5, 9, 7), (66, 17, 3), (3, 2, 129), (2, 3, 700)])
def test_direct_chunks(fl, oracle, dom):
    nx, ny, nz = dom
    shape = (nz + 8, ny + 8, nx + 8)
    r = np.random.RandomState(nz)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    fields = [f32(-1, 1) for _ in range(4)]
    st, d = 4, (12.5, 10.0, 8.0)
    isrc = fl.index(shape, 4 + nx // 2, 4 + ny // 2, 4 + nz // 2)
    wav = r.standard_normal(st).astype(np.float32)
    ref = oracle.run("original", shape, 4, d, DT, st, isrc, oracle.precompute(m), fields=fields, src=wav)
    g = fl.Driver(variant="direct")
    g.initialize(shape, d, DT, m, fields=fields)
    g.run(st, isrc, src=wav, graph_chunk=0)
    got = {k: g.field(k) for k in ("pp", "pc", "qp", "qc")}
    g.finalize()
    assert not np.array_equal(got["pc"], fields[1])
    for k in got:
        assert np.array_equal(got[k], ref[k]), k
