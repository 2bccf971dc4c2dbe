"""The default tiles (12, 0) leave rows and chunk depth to the grid: for grids and forms where the
choice falls on different tile rows and lane layouts, results equal those of fixed 12-row
tiles bit for bit, single grid and batched, and the shape reported is one the step accepts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = (12.5, 12.5, 12.5)


def _model(fl, n3, absorb):
    m = fl.model_gradient(n3, absorb, seed=31, blob_smin=4.0, blob_smax=10.0, smooth_smin=6.0, smooth_smax=16.0)
    return m, m[0].shape, fl.cfl_dt(m, 12.5, 0.4)


def _run(fl, m, shape, dt, prec, variant, tiles):
    d = fl.Driver(variant=variant, precision=prec, tiles=tiles)
    d.initialize(shape, D, dt, m)
    d.record_traces(9, 2, 6)
    d.run(13, fl.center_index(shape), graph_chunk=4)
    out = [d.field(k) for k in ("pp", "pc", "qp", "qc")] + [d.traces()]
    used = d.tiles()
    d.finalize()
    fl.Driver(tiles=(12, 0))
    return out, used


@pytest.mark.parametrize("variant,prec", [("fused", "fp32"), ("fused", "q16r"), ("fused", "fp32r"), ("fused", "bf16"),
                                          ("twopass", "fp32")])
@pytest.mark.parametrize("n3,absorb", [((1, 2, 3), 4), ((40, 36, 32), 8), ((30, 80, 45), 8), ((110, 64, 90), 12)])
def test_default_tiles_equal_fixed_tiles(fl, variant, prec, n3, absorb):
    m, shape, dt = _model(fl, n3, absorb)
    a, used = _run(fl, m, shape, dt, prec, variant, (12, 0))
    b, _ = _run(fl, m, shape, dt, prec, variant, (12, 9))
    assert used[0] in (4, 8, 12, 16) and 1 <= used[1] <= shape[0] - 8
    assert np.abs(a[1]).max() > 0
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("prec", ["fp32", "fp16r"])
def test_default_batch_tiles_equal_fixed_tiles(fl, prec):
    shots = []
    for n3 in ((20, 33, 17), (64, 20, 41)):
        m, shape, dt = _model(fl, n3, 6)
        shots.append({"model": m, "isource": fl.center_index(shape), "rec_iz": 11})
    out = []
    for tiles in ((12, 0), (12, 9)):
        b = fl.Batch(shots, D, dt, precision=prec, tiles=tiles)
        try:
            b.run(9, graph_chunk=4, rec_every=2, max_traces=4)
            out.append([b.field(k, f) for k in range(2) for f in ("pc", "qp")] + [b.traces(k) for k in range(2)])
            assert b.tiles()[0] in (4, 8, 12, 16)
        finally:
            b.set_tiles(12, 0)
            b.destroy()
    assert np.abs(out[0][0]).max() > 0
    for x, y in zip(*out):
        assert np.array_equal(x, y)
