"""The tile setting: (12, 0) is 12 rows with a depth chosen for the grid, single grid and batched, also where
the automatic setting takes other rows; the automatic setting is one of its own, set by set_auto_tiles and
left by set_tiles.  Fields and receivers of all of them are the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = (12.5, 12.5, 12.5)
GRIDS = (((1, 2, 3), 4), ((40, 36, 32), 8), ((110, 64, 90), 12))


def _model(fl, n3, absorb):
    m = fl.model_gradient(n3, absorb, seed=17, blob_smin=4.0, blob_smax=10.0, smooth_smin=6.0, smooth_smax=16.0)
    return m, m[0].shape, fl.cfl_dt(m, 12.5, 0.4)


def _run(fl, m, shape, dt, prec, variant, setting):
    d = fl.Driver(variant=variant, precision=prec)
    if setting == "auto":
        d.set_tiles(4, 3)
        d.set_auto_tiles()
    else:
        d.set_tiles(*setting)
    try:
        d.initialize(shape, D, dt, m)
        d.record_traces(9, 2, 6)
        d.run(13, fl.center_index(shape), graph_chunk=4)
        return d.tiles(), [d.field(k) for k in ("pp", "pc", "qp", "qc")] + [d.traces()]
    finally:
        d.finalize()
        d.set_auto_tiles()


@pytest.mark.parametrize("variant,prec", [("fused", "fp32"), ("fused", "q16r"), ("fused", "fp32r"), ("fused", "bf16"),
                                          ("twopass", "fp32")])
def test_twelve_rows_are_twelve_rows(fl, variant, prec):
    rows = set()
    for n3, absorb in GRIDS:
        m, shape, dt = _model(fl, n3, absorb)
        twelve, a = _run(fl, m, shape, dt, prec, variant, (12, 0))
        auto, b = _run(fl, m, shape, dt, prec, variant, "auto")
        print(variant, prec, shape, "12 rows", twelve, "automatic", auto, flush=True)
        assert twelve[0] == 12 and 1 <= twelve[1] <= shape[0] - 8
        assert auto[0] in (4, 8, 12, 16) and 1 <= auto[1] <= shape[0] - 8
        rows.add(auto[0])
        assert np.abs(a[1]).max() > 0
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    assert rows - {12}  # the automatic setting is another one on these grids


@pytest.mark.parametrize("prec", ["fp32", "fp16r"])
def test_twelve_rows_batched(fl, prec):
    shots = []
    for n3 in ((20, 33, 17), (64, 20, 41)):
        m, shape, dt = _model(fl, n3, 6)
        shots.append({"model": m, "isource": fl.center_index(shape), "rec_iz": 11})
    out, used = [], []
    for setting in ((12, 0), "auto"):
        b = fl.Batch(shots, D, dt, precision=prec, tiles=(4, 3))
        try:
            if setting == "auto":
                b.set_auto_tiles()
            else:
                b.set_tiles(*setting)
            b.run(9, graph_chunk=4, rec_every=2, max_traces=4)
            used.append(b.tiles())
            out.append([b.field(k, f) for k in range(2) for f in ("pc", "qp")] + [b.traces(k) for k in range(2)])
        finally:
            b.set_auto_tiles()
            b.destroy()
    assert used[0][0] == 12 and used[1][0] in (4, 8, 16)
    assert np.abs(out[0][0]).max() > 0
    for x, y in zip(*out):
        assert np.array_equal(x, y)


def test_autotuned_and_refused_tiles(fl):
    """A tuned shape stays, a refused one changes nothing."""
    m, shape, dt = _model(fl, (40, 36, 32), 8)
    d = fl.Driver(variant="fused", precision="fp32")
    d.set_auto_tiles()
    try:
        d.initialize(shape, D, dt, m)
        auto = d.tiles()
        assert d.L.fl_set_tiles(5, 0) == -1 and d.L.fl_set_tiles(12, -1) == -1
        d.L.fl_clear_error()
        assert d.tiles() == auto
        tuned = d.autotune(1)
        assert d.tiles() == tuned and tuned[1] >= 1
    finally:
        d.finalize()
        d.set_auto_tiles()
        d.set_stream_hints(False)
