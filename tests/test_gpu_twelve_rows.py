"""12-row tiles at fixed depths, with and without the streaming hints, against 8-row tiles without them, bit
for bit: non-zero halo cells, chunk depths with no, one and two whole ten-plane groups and the whole column,
tiles cut by both edges of the update domain, steps in both directions and a captured run, receivers on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11


@pytest.mark.parametrize("variant,prec", [("fused", p) for p in ("fp32", "fp32r", "bf16", "fp16", "fp16r", "q16r")] +
                         [("twopass", "fp32")])
@pytest.mark.parametrize("dom,bord,d", [((35, 19, 31), 4, (12.5, 12.5, 12.5)), ((30, 33, 25), 5, (12.5, 10.0, 8.0))])
def test_twelve_rows_at_fixed_depths(fl, variant, prec, dom, bord, d):
    nx, ny, nz = dom
    shape = (nz + 2 * bord, ny + 2 * bord, nx + 2 * bord)
    r = np.random.RandomState(ny)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    fields = [f32(-1, 1) for _ in range(4)]
    isrc, wav = fl.index(shape, bord + 3, bord + ny - 2, bord + nz // 2), r.standard_normal(4).astype(np.float32)

    def steps(tiles, hints):
        g = fl.Driver(variant=variant, precision=prec, tiles=tiles)
        g.set_stream_hints(hints)
        try:
            g.initialize(shape, d, DT, m, fields=fields, bord=bord)
            assert g.tiles()[0] == tiles[0]
            g.record_traces(bord + nz // 2, 1, 6)
            g.propagate(1)
            g.propagate(2)
            g.run(4, isrc, it0=2, src=wav, graph_chunk=2)
            return [g.field(k) for k in ("pp", "pc", "qp", "qc")] + [g.traces()]
        finally:
            g.finalize()
            g.set_stream_hints(False)
            g.set_auto_tiles()

    ref = steps((8, 9), False)
    assert not np.array_equal(ref[1], fields[1]) and np.isfinite(ref[1]).all()
    for zt in (1, 5, 14, 24, 0, nz):
        for hints in (False, True):
            for k, (a, b) in enumerate(zip(steps((12, zt), hints), ref)):
                assert np.array_equal(a, b), (zt, hints, k)
