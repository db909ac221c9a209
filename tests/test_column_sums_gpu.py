"""Column sums of the bias gradients (plain, masked, and with the cross-entropy backward) at the edges of
their column groups (8 and 32 wide), row chunks (512) and read-ahead (32), bit for bit: the sums run in
the reference's order."""
import numpy as np
import pytest

from axis_amd import hip
from axis_amd.hip import F32, I64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device(0)


def chunked(g):
    """Rows in order inside chunks of 512, then the chunks in order, in fp32."""
    total = np.zeros(g.shape[1], np.float32)
    for r0 in range(0, g.shape[0], 512):
        part = np.zeros(g.shape[1], np.float32)
        for row in g[r0:r0 + 512]:
            part = part + row
        total = total + part
    return total


# the last takes the masked kernel of operands past the last-level cache
@pytest.mark.parametrize("rows,width", [(1, 9), (31, 8), (33, 7), (512, 33), (513, 4097), (2049, 1025), (1537, 2079),
                                        (8193, 1024), (12000, 1999)])
def test_bias_sums(dev, rows, width):
    print(f"rows={rows} width={width}", flush=True)
    rng = np.random.default_rng(rows + width)
    g = rng.standard_normal((rows, width)).astype(np.float32)
    z = rng.standard_normal((rows, width)).astype(np.float32)
    g[0, 0], z[rows - 1, width - 1] = -0.0, np.nan
    dg, dz = dev.upload(g), dev.upload(z)
    out, masked = dev.empty(width), dev.empty(rows * width)
    dev.call("axis_bias_gradient", dg.vp, None, None, out.vp, I64(rows), I64(width))
    assert np.array_equal(dev.read(out, width).view(np.uint32), chunked(g).view(np.uint32))
    dev.call("axis_bias_gradient", dg.vp, dz.vp, masked.vp, out.vp, I64(rows), I64(width))
    want = np.where(z > 0, g, np.float32(0))
    assert np.array_equal(dev.read(masked, rows * width), want.reshape(-1))
    assert np.array_equal(dev.read(out, width).view(np.uint32), chunked(want).view(np.uint32))


@pytest.mark.parametrize("rows,width", [(3, 5), (100, 31), (512, 1000), (700, 4099), (2000, 1027)])
def test_cross_entropy_backward_with_bias(dev, rows, width):
    print(f"rows={rows} width={width}", flush=True)
    rng = np.random.default_rng(rows)
    p, t = rng.random((rows, width)).astype(np.float32), rng.random((rows, width)).astype(np.float32)
    one = np.array([1.5], np.float32)
    d1, dp, dt = dev.upload(one), dev.upload(p), dev.upload(t)
    out, bias = dev.empty(rows * width), dev.empty(width)
    factor = np.float32(1.0 / rows)
    dev.call("axis_categorical_cross_entropy_backward_mean", d1.vp, F32(factor), dp.vp, dt.vp, out.vp, bias.vp,
             I64(rows), I64(width))
    want = (one[0] * factor) * (p - t)
    assert np.array_equal(dev.read(out, rows * width), want.reshape(-1))
    assert np.array_equal(dev.read(bias, width).view(np.uint32), chunked(want).view(np.uint32))
