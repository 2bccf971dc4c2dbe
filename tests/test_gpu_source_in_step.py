"""Multi-step runs of the two-pass form, whose steps add the next source sample themselves, against
InsertSource + Propagate for every step (graph_chunk 0), bit for bit: fields and receivers, a run
continued at an odd step, sources at both corners of the update domain and (launched plainly) in
the halo."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE, BORD, D, DT = (26, 30, 43), 5, (12.5, 10.0, 8.0), 2.0 ** -11


@pytest.mark.parametrize("cell", [(5, 5, 5), (37, 24, 20), (3, 10, 10)])  # ix, iy, iz
def test_runs_equal_plain_launches(fl, cell):
    r = np.random.RandomState(3)
    f32 = lambda lo, hi: r.uniform(lo, hi, SHAPE).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    isrc, wav = fl.index(SHAPE, *cell), r.standard_normal(17).astype(np.float32)
    out = []
    for chunk in (0, 4):
        g = fl.Driver(variant="twopass")
        g.initialize(SHAPE, D, DT, m, bord=BORD)
        g.record_traces(9, 3, 5)
        g.run(9, isrc, src=wav[:9], graph_chunk=chunk)
        g.run(8, isrc, it0=9, src=wav[9:], graph_chunk=chunk)
        out.append([g.field(k) for k in ("pp", "pc", "qp", "qc")] + [g.traces()])
        g.finalize()
    assert np.abs(out[0][1]).max() > 0 and np.abs(out[0][4][-1]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
