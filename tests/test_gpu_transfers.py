"""Host transfers in chunks of 16 MiB: fields and records of grids whose chunks end inside a row,
cover the whole grid, or leave a short last one, against the host values bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = (12.5, 12.5, 12.5)


# part of a chunk, 2^22 cells (a whole chunk) and a few more or fewer, several chunks
@pytest.mark.parametrize("shape", [(9, 9, 9), (37, 121, 133), (64, 256, 256), (41, 61, 1677), (129, 181, 181)])
def test_fields_round_trip(fl, shape):
    m = fl.model_homogeneous("TTI", shape)
    r = np.random.RandomState(3)
    f = r.standard_normal(shape).astype(np.float32)
    g = r.standard_normal(shape).astype(np.float32)
    d = fl.Driver(variant="fused")
    d.initialize(shape, D, 0.001, m)
    d.set_field("pc", f)
    d.set_field("qc", g)
    d.set_field("pp", g)
    assert np.array_equal(d.field("pc"), f)
    assert np.array_equal(d.update_pointers(), f)
    assert np.array_equal(d.field("qc"), g)
    assert np.array_equal(d.field("pp"), g)
    assert not d.field("qp").any()
    d.finalize()


@pytest.mark.parametrize("prec", ["fp32", "fp32r", "fp16", "bf16", "fp16r", "q16r"])
def test_host_records_over_several_chunks(fl, prec):
    """Records of a grid of several chunks equal, cell by cell, those of the same cells in a
    grid of one chunk: the pack kernel's rows and the chunk boundaries."""
    big = (151, 93, 117)  # 1.6M cells: two chunks or more in every form, ending inside rows
    m = fl.model_gradient((117 - 16, 93 - 16, 151 - 16), 4, seed=5)
    assert m[0].shape == big
    # block floating point: the exponent base is the grid's, so the small grid keeps the fastest cell
    zmax = int(np.unravel_index(np.argmax(m[0] * m[0] * (1 + 2 * m[2])), big)[0])
    z0 = min(max(0, zmax - 5), big[0] - 10)
    out = []
    for lo, hi in ((0, big[0]), (z0, z0 + 10)):
        s = (hi - lo,) + big[1:]
        d = fl.Driver(variant="fused", precision=prec)
        d.initialize(s, D, 0.0008, [a[lo:hi] for a in m])
        r = d.records().reshape(s[0], -1)
        out.append(r)
        d.finalize()
    assert np.array_equal(out[0][z0:z0 + 10], out[1])
    assert out[1].any()
