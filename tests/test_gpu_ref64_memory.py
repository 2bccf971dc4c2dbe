"""The FP64 reference gives back what it allocated: with no grid and no batch set up, the device memory free
after fl_ref64_destroy is that before fl_ref64_create, the buffers of its host transfers (32 MiB)
included; a grid that is set up keeps its transfers working across it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D, DT, SHAPE = (12.5, 12.5, 12.5), 2.0 ** -11, (30, 26, 34)
SLACK = 4 << 20  # the allocator's own granularity


def _ref64(fl, m):
    g = fl.Ref64(SHAPE, D, DT, m)
    g.run(3, fl.center_index(SHAPE), src=np.ones(3, np.float32))
    out = g.field("pc")
    g.destroy()
    return out


def test_destroy_returns_the_transfer_buffers(fl):
    m = fl.model_homogeneous("TTI", SHAPE)
    _ref64(fl, m)  # streams and code objects of a first call
    d = fl.Driver(variant="fused")
    d.initialize(SHAPE, D, DT, m)
    d.finalize()  # returns the buffers of its own transfers
    before = fl.device_memory()[0]
    assert np.abs(_ref64(fl, m)).max() > 0
    assert fl.device_memory()[0] >= before - SLACK


def test_a_grid_keeps_its_transfers(fl):
    m = fl.model_homogeneous("TTI", SHAPE)
    f = np.random.RandomState(2).standard_normal(SHAPE).astype(np.float32)
    d = fl.Driver(variant="fused")
    d.initialize(SHAPE, D, DT, m)
    d.set_field("pc", f)
    held = fl.device_memory()[0]
    _ref64(fl, m)
    assert fl.device_memory()[0] <= held + SLACK  # not taken from the grid
    assert np.array_equal(d.field("pc"), f)
    d.finalize()
