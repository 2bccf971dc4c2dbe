"""Tile heights that form Dxx and Dyy at the input plane (4 and 16 rows, FP32 on 8) against 12 rows, which
form them at the output plane: one step upwards and one downwards, bit for bit, over chunk depths
with no, one and several whole ten-plane groups and every length of the rest, on tiles cut by both
edges of the update domain, receivers on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 2.0 ** -11


@pytest.mark.parametrize("prec", ["fp32", "bf16", "fp16", "fp16r", "fp32r", "q16r"])
@pytest.mark.parametrize("dom,bord,d,zts", [
    ((35, 19, 31), 4, (12.5, 12.5, 12.5), (1, 5, 13, 14, 15, 0)),
    ((30, 33, 25), 5, (12.5, 10.0, 8.0), (2, 7, 16, 25)),
])
def test_tile_heights_agree(fl, prec, dom, bord, d, zts):
    nx, ny, nz = dom
    shape = (nz + 2 * bord, ny + 2 * bord, nx + 2 * bord)
    r = np.random.RandomState(nx)
    f32 = lambda lo, hi: r.uniform(lo, hi, shape).astype(np.float32)  # noqa: E731
    m = [f32(1500, 4000), f32(300, 1500), f32(0.1, 0.2), f32(0.0, 0.1), f32(-1, 1), f32(0, 1)]
    fields = [f32(-1, 1) for _ in range(4)]  # the halo cells too

    def steps(tiles):
        g = fl.Driver(variant="fused", precision=prec, tiles=tiles)
        g.set_lane_pairs(False)
        g.initialize(shape, d, DT, m, fields=fields, bord=bord)
        g.record_traces(bord + nz // 2, 1, 2)
        g.propagate(1)
        g.propagate(2)
        out = [g.field(k) for k in ("pp", "pc", "qp", "qc")] + [g.traces()]
        g.finalize()
        g.set_lane_pairs(True)
        return out

    ref = steps((12, 9))
    assert not np.array_equal(ref[1], fields[1])
    for ty in (4, 16) + ((8,) if prec == "fp32" else ()):
        for zt in zts:
            for k, (a, b) in enumerate(zip(steps((ty, zt)), ref)):
                assert np.array_equal(a, b), (ty, zt, k)
