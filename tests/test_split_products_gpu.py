"""fp32 products on the bf16 matrix cores (three bf16 planes per operand, gemm_split.hip), at the sizes
where its tiles, loads and slices can go wrong, against float64.

Tolerance, per output: each product of the planes leaves out at most 2^-23 |x| |y|, and the kept ones
are added in fp32 through chains of 6 x 32 products, one add per 32 of them and one per slice, so
|error| <= (192 + k / 32 + slices) * 2^-24 * sum |x| |y| whatever the order inside an instruction.
With at most 512 slices (and the epilogue's roundings) that is below `bound`."""
import ctypes

import numpy as np
import pytest

from axis_amd import hip
from axis_amd.hip import I32, I64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return hip.Device(0)


def bound(x, y, k):
    return (192 + k / 32 + 512) * 2.0 ** -24 * (np.abs(x) @ np.abs(y)) + 1e-37


def run(dev, op, x, y, batch, m, k, n, count, *more):
    dx, dy, out = dev.upload(x), dev.upload(y), dev.empty(count)
    dev.call(op, dx.vp, dy.vp, *more, out.vp, I64(batch), I64(m), I64(k), I64(n))
    return dev.read(out, count)


# 256x128, 128x128, 256x64 and 64x64 tiles: whole, one row / column / reduction element past and short
# of the edges, rows that start on any element, slices of the reduction, batches.
SHAPES = [(1, 4096, 512, 1024), (1, 4097, 513, 1025), (1, 2047, 1023, 1151), (1, 8192, 96, 64), (1, 8191, 97, 65),
          (1, 1024, 1024, 512), (1, 1025, 1021, 511), (1, 512, 512, 512), (3, 500, 260, 316), (2, 1000, 333, 401),
          (1, 130, 8192, 200), (1, 2048, 64, 2048), (1, 2500, 33, 1500)]


@pytest.mark.parametrize("batch,m,k,n", SHAPES)
def test_dense_products(dev, batch, m, k, n):
    print(f"dense batch={batch} m={m} k={k} n={n}", flush=True)
    rng = np.random.default_rng(m + k + n)
    a = rng.standard_normal((batch, m, k)).astype(np.float32)
    b = rng.standard_normal((batch, k, n)).astype(np.float32)
    g = rng.standard_normal((batch, m, n)).astype(np.float32)
    t = lambda v: np.swapaxes(v, 1, 2)
    for op, x, y, xm, ym, depth in (("axis_matmul", a, b, a, b, k), ("axis_matmul_left_backward", g, b, g, t(b), n),
                                    ("axis_matmul_right_backward", a, g, t(a), g, m)):
        xd, yd = xm.astype(np.float64), ym.astype(np.float64)
        want = xd @ yd
        got = run(dev, op, x, y, batch, m, k, n, want.size).reshape(want.shape)
        assert np.all(np.abs(got - want) <= bound(xd, yd, depth)), op
        # and as a whole well inside an fp32 sum's own error
        assert np.linalg.norm(got - want) < 1e-6 * np.linalg.norm(want), op


@pytest.mark.parametrize("m,k,n", [(2048, 512, 1024), (1030, 1001, 515)])
@pytest.mark.parametrize("sx,sy", [(1e-36, 1e20), (1e25, 1e-36), (1e-30, 1e-7), (1e30, 1e5)])
def test_magnitudes_at_the_ends_of_the_range(dev, m, k, n, sx, sy):
    # the planes of operands near the end of the exponent range lose bits: such tiles are computed again
    # (1e30 * 1e5: the largest scale whose sums stay inside fp32)
    rng = np.random.default_rng(m)
    x = (rng.standard_normal((m, k)) * sx).astype(np.float32)
    y = (rng.standard_normal((k, n)) * sy).astype(np.float32)
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    got = run(dev, "axis_matmul", x, y, 1, m, k, n, m * n).reshape(m, n)
    assert np.all(np.abs(got - xd @ yd) <= bound(xd, yd, k))


@pytest.mark.parametrize("m,k,n", [(2048, 512, 1024), (1030, 1001, 515)])
def test_tiny_values_among_ordinary_ones(dev, m, k, n):
    # rows (and single elements) of 1e-36 in tiles that keep the planes: what the low planes lose is below
    # the smallest normal number per element of either operand
    rng = np.random.default_rng(n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = rng.standard_normal((k, n)).astype(np.float32)
    x[::7] *= np.float32(1e-36)
    x[:, ::5] *= np.float32(1e-34)
    y[3::11, ::3] *= np.float32(1e-37)
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    lost = 2.0 ** -126 * (np.abs(xd).sum(1)[:, None] + np.abs(yd).sum(0)[None, :])
    got = run(dev, "axis_matmul", x, y, 1, m, k, n, m * n).reshape(m, n)
    assert np.all(np.abs(got - xd @ yd) <= bound(xd, yd, k) + lost)


@pytest.mark.parametrize("m,k,n", [(2048, 512, 1024), (1030, 1001, 515), (512, 4096, 512)])
def test_values_the_planes_do_not_hold(dev, m, k, n):
    # infinities, NaN and magnitudes that bf16 rounds to infinity give what fp32 products give
    rng = np.random.default_rng(k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = rng.standard_normal((k, n)).astype(np.float32) * np.float32(0.01)
    x[3, 5], x[m - 1, k - 1], x[40, 7], x[200, 0] = np.inf, -np.inf, np.nan, np.float32(3.4e38)
    y[5, 2] = 0.0  # inf * 0
    y[9, n - 1] = np.inf
    with np.errstate(invalid="ignore", over="ignore"):
        want = x.astype(np.float64) @ y.astype(np.float64)
    got = run(dev, "axis_matmul", x, y, 1, m, k, n, m * n).reshape(m, n)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf])
    fine = np.isfinite(want)
    scale = np.abs(np.where(fine, want, 0)).max(axis=1, keepdims=True)
    assert np.all((np.abs(got - np.where(fine, want, 0)) <= 1e-5 * scale)[fine])


def conv64(x, w, k, p):
    b, h, wd, c = x.shape
    n = w.shape[1]
    w4 = w.reshape(c, k, k, n)
    xp = np.pad(x, ((0, 0), (p, p), (p, p), (0, 0)))
    oh, ow = h + 2 * p - k + 1, wd + 2 * p - k + 1
    taps = [(ky, kx, xp[:, ky:ky + oh, kx:kx + ow].reshape(-1, c)) for ky in range(k) for kx in range(k)]
    return sum(v @ w4[:, ky, kx] for ky, kx, v in taps).reshape(b, oh, ow, n), taps


# (batch, height, width, channels, outputs, kernel): tap steps (channels % 32 == 0) and per-lane taps,
# aligned and ragged pixel steps of the weight gradient, column tails, one and several slices
CONVS = [(40, 32, 32, 64, 128, 3), (20, 17, 13, 48, 80, 5), (64, 16, 16, 32, 64, 3), (9, 30, 33, 64, 36, 3),
         (100, 8, 8, 96, 256, 3), (33, 20, 20, 260, 72, 1)]


@pytest.mark.parametrize("b,h,w,c,n,k", CONVS)
@pytest.mark.parametrize("special", [False, True])
def test_convolutions(dev, b, h, w, c, n, k, special):
    print(f"conv b={b} {h}x{w} {c}->{n} k={k} special={special}", flush=True)
    rng = np.random.default_rng(c + n)
    p = k // 2
    x = rng.standard_normal((b, h, w, c)).astype(np.float32)
    wt = (rng.standard_normal((c * k * k, n)) * 0.05).astype(np.float32)
    g = rng.standard_normal((b, h, w, n)).astype(np.float32)
    if special:
        x[1, 2, 3, 4], x[b - 1, h - 1, w - 1, c - 1] = np.inf, np.nan
        g[2, 0, 0, 1] = -np.inf
    geo = (I64(b), I32(h), I32(w), I32(c), I32(n), (I32 * 2)(k, k), (I32 * 2)(1, 1), (I32 * 2)(p, p))
    dx, dw, dg = dev.upload(x), dev.upload(wt), dev.upload(g)
    y, gx, gw = dev.empty(b * h * w * n), dev.empty(x.size), dev.empty(wt.size)
    dev.call("axis_conv2d_forward", dx.vp, None, dw.vp, None, y.vp, *geo)
    dev.call("axis_conv2d_backward_data", dg.vp, dw.vp, gx.vp, *geo)
    dev.call("axis_conv2d_backward_weight", dx.vp, None, dg.vp, gw.vp, *geo)
    x64, w64, g64 = x.astype(np.float64), wt.astype(np.float64), g.astype(np.float64)
    flipped = w64.reshape(c, k, k, n)[:, ::-1, ::-1].transpose(3, 1, 2, 0).reshape(n * k * k, c)
    with np.errstate(invalid="ignore"):
        want_y, taps = conv64(x64, w64, k, p)
        want_x, _ = conv64(g64, np.ascontiguousarray(flipped), k, p)
        want_w = np.zeros((c, k, k, n))
        for ky, kx, v in taps:
            want_w[:, ky, kx] = v.T @ g64.reshape(-1, n)
    for got, want in ((dev.read(y, b * h * w * n), want_y), (dev.read(gx, x.size), want_x),
                      (dev.read(gw, wt.size), want_w)):
        want = want.reshape(-1)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf])
        fine = np.isfinite(want)
        assert np.linalg.norm(got[fine] - want[fine]) < 1e-6 * np.linalg.norm(want[fine])
