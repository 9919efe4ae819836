"""The split-operand 3x3 convolution (csrc/om_conv3_s.hpp) at the sizes and values where it can go wrong: widths that are
no multiple of 4, wide rows (some of which the fp32 kernel takes), partial pixel tiles, both channel blocks, one chunk of channels and
split channels, accumulation, and operands the three-way bf16 split does not carry, against float64 over the zero-padded input.

Tolerance: for edges and values the sequential-accumulation bound k 2^-24 sum |w||x| over the k = 9 Cin terms (the kernel's own
rounding count is lower: one per 16 terms and five per 16 on sums 2^-7 as large), and a rounding of each later addition; for the
precision itself, single products within 2^-23.
"""
import time

import numpy as np
import pytest

import gpu_util

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return gpu_util.Dev()


def conv64(x, w):
    """3x3 / stride 1 / padding 1 in float64: sum over taps of w[:, :, t] times the shifted, zero-padded input."""
    n, ci, h, wd = x.shape
    xp = np.zeros((n, ci, h + 2, wd + 2))
    xp[:, :, 1:-1, 1:-1] = x
    y = np.zeros((n, w.shape[0], h * wd))
    for ky in range(3):
        for kx in range(3):
            y += w[:, :, ky, kx].astype(np.float64) @ xp[:, :, ky:ky + h, kx:kx + wd].reshape(n, ci, -1)
    return y.reshape(n, -1, h, wd)


def turned(w):
    return np.ascontiguousarray(w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3))


# (images, Cin, Cout, H, W): dX exchanges the channels
SHAPES = [(1, 32, 32, 1, 1), (1, 32, 64, 3, 5), (2, 64, 32, 7, 7), (3, 96, 64, 5, 33), (1, 512, 64, 2, 3), (2, 32, 96, 19, 27),
          (40, 64, 64, 15, 17), (9, 32, 160, 31, 33), (300, 32, 32, 3, 3), (2, 32, 64, 4, 185), (1, 64, 32, 3, 189),
          (1, 32, 64, 90, 62), (1, 32, 64, 13, 224), (1, 64, 32, 8, 224), (2, 96, 32, 9, 256), (5, 32, 96, 12, 128), (2, 48, 64, 8, 192)]


@pytest.mark.parametrize("N,Cin,Cout,H,W", SHAPES)
def test_edges(dev, N, Cin, Cout, H, W):
    rng = np.random.default_rng(N + 31 * Cin + 1009 * Cout + 7 * W)
    x = rng.standard_normal((N, Cin, H, W)).astype(np.float32)
    w = rng.standard_normal((Cout, Cin, 3, 3)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    g = rng.standard_normal((N, Cout, H, W)).astype(np.float32)
    X, Wd, B, G = dev.put(x), dev.put(w), dev.put(b), dev.put(g)
    Y, R = dev.empty(g.shape, fill=np.nan), dev.empty(g.shape, fill=np.nan)
    dev.call("om_conv2d_fwd", X, Wd, B, Y, N, Cin, H, W, Cout, 3, 3, 1, 1)
    want = conv64(x, w) + b[:, None, None]
    bound = 9 * Cin * 2.0 ** -24 * conv64(np.abs(x), np.abs(w)) + 2.0 ** -22 * (np.abs(want) + np.abs(b)[:, None, None])
    y = dev.get(Y)
    assert np.all(np.abs(y - want) <= bound)
    dev.call("om_conv2d_relu_fwd", X, Wd, B, R, N, Cin, H, W, Cout, 3, 3, 1, 1)
    assert np.array_equal(dev.get(R), np.where(y > 0, y, np.float32(0)))
    dx0 = rng.standard_normal(x.shape).astype(np.float32)
    DX, DW, DB = dev.put(dx0.copy()), dev.empty(w.shape), dev.empty(b.shape)
    dev.call("om_conv2d_bwd", G, X, Wd, DX, DW, DB, N, Cin, H, W, Cout, 3, 3, 1, 1, 1, 0)
    want = conv64(g, turned(w)) + dx0
    bound = 9 * Cout * 2.0 ** -24 * conv64(np.abs(g), turned(np.abs(w))) + 2.0 ** -22 * (np.abs(want) + np.abs(dx0))
    assert np.all(np.abs(dev.get(DX) - want) <= bound)


@pytest.mark.parametrize("N,Cin,Cout,H,W", [(64, 32, 32, 7, 7), (64, 64, 64, 5, 33), (96, 96, 160, 19, 27), (40, 64, 64, 15, 17),
                                            (24, 32, 64, 4, 185), (32, 256, 64, 3, 5), (32, 64, 64, 56, 56)])
def test_single_products(dev, N, Cin, Cout, H, W):
    """One element in each image, at the borders and inside, so every result is one product of two full significands and shows each
    of the six terms: a lost or misplaced plane leaves 2^-17 or more (test_split_terms.py)."""
    rng = np.random.default_rng(N + W)
    w = gpu_util.full_significands(rng, (Cout, Cin, 3, 3))

    def images(chans):
        x, i = np.zeros((N, chans, H, W), np.float32), np.arange(N)
        rows, cols = np.array([0, H - 1, H // 2, 1 % H])[i % 4], np.array([0, W - 1, W // 2, 7 % W, 8 % W])[i % 5]
        x[i, (i * 7) % chans, rows, cols] = gpu_util.full_significands(rng, N)
        return x

    x, g = images(Cin), images(Cout)
    X, Wd, Y, DX = dev.put(x), dev.put(w), dev.empty(g.shape), dev.empty(x.shape)
    dev.call("om_conv2d_fwd", X, Wd, None, Y, N, Cin, H, W, Cout, 3, 3, 1, 1)
    dev.call("om_conv2d_bwd", dev.put(g), X, Wd, DX, dev.empty(w.shape), None, N, Cin, H, W, Cout, 3, 3, 1, 1, 0, 0)
    for got, want in ((dev.get(Y), conv64(x, w)), (dev.get(DX), conv64(g, turned(w)))):
        assert np.all(np.abs(got - want) <= gpu_util.SPLIT_PRODUCT * np.abs(want))


@pytest.mark.parametrize("N,C,H,W", [(6, 32, 17, 19), (1, 64, 6, 9)])
def test_values_the_split_does_not_carry(dev, N, C, H, W):
    rng = np.random.default_rng(11)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    w = rng.standard_normal((C, C, 3, 3)).astype(np.float32) * np.float32(2.0 ** -8)
    x[0, 1, 0, 0], x[0, 2, 3, W - 1], x[0, 3, 5, 2], x[0, 4, 3, 5] = np.inf, -np.inf, np.nan, 3.4e38
    w[7, 5, 2, 2] = np.inf  # times the zeros around the image: NaN along two edges, as the padded sum has it
    w[9] *= np.float32(1e-36)
    X, Wd, B, Y = dev.put(x), dev.put(w), dev.put(np.zeros(C, np.float32)), dev.empty(x.shape, fill=0)
    with np.errstate(invalid="ignore", over="ignore"):
        for flip in (False, True):
            if flip:
                dev.call("om_conv2d_bwd", X, X, Wd, Y, dev.empty(w.shape), dev.empty((C,)), N, C, H, W, C, 3, 3, 1, 1, 0, 0)
            else:
                dev.call("om_conv2d_fwd", X, Wd, B, Y, N, C, H, W, C, 3, 3, 1, 1)
            wf = turned(w) if flip else w
            want = conv64(x, wf)
            bound = 9 * C * (2.0 ** -24 * conv64(np.abs(x), np.abs(wf)) + 2.0 ** -148)
            got, fin = dev.get(Y), np.isfinite(want)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
            assert np.all(np.abs(got[fin] - want[fin]) <= bound[fin])


@pytest.mark.parametrize("N,C,H,W", [(16, 32, 17, 19), (8, 64, 6, 9)])
@pytest.mark.parametrize("tiny_w", [False, True])
def test_tiny_operands_beside_large_ones(dev, N, C, H, W, tiny_w):
    """Images (or filters) down to the smallest subnormals times filters (images) up to 2^100: every term keeps all its bits.
    The bound is test_edges's, and for sums that are subnormal themselves half a unit of the last place a term."""
    rng = np.random.default_rng(19)
    tiny = np.ldexp(1.0, [-112, -118, -124, -127, -133, -137, -142, -147])
    wide = np.ldexp(1.0, [0, 10, 20, 40, 60, 100])
    si, sf = (wide, tiny) if tiny_w else (tiny, wide)
    x = (rng.standard_normal((N, C, H, W)) * np.resize(si, N)[:, None, None, None]).astype(np.float32)
    w0 = rng.standard_normal((C, C, 3, 3))
    X, Y, B = dev.put(x), dev.empty(x.shape), dev.put(np.zeros(C, np.float32))
    for flip in (False, True):
        w = (w0 * (np.resize(sf, C)[None, :, None, None] if flip else np.resize(sf, C)[:, None, None, None])).astype(np.float32)
        if flip:
            dev.call("om_conv2d_bwd", X, X, dev.put(w), Y, dev.empty(w.shape), dev.empty((C,)), N, C, H, W, C, 3, 3, 1, 1, 0, 0)
        else:
            dev.call("om_conv2d_fwd", X, dev.put(w), B, Y, N, C, H, W, C, 3, 3, 1, 1)
        wf = turned(w) if flip else w
        bound = 9 * C * (2.0 ** -24 * conv64(np.abs(x), np.abs(wf)) + 2.0 ** -150)
        assert np.all(np.abs(dev.get(Y) - conv64(x, wf)) <= bound)


@pytest.mark.parametrize("scale,factor", [(2.0 ** -94, 2), (np.nan, 8)])
def test_no_values_take_a_slow_path(dev, scale, factor):
    """Gradients of confidently classified samples are around e^-65 and cost what others do (the factor 2 is for the clock's
    noise); those of a diverged step run on the fp32 instruction, 2.4 times as long. (Loops over single terms once took 12 and
    30 times as long.)"""
    N, C, H, W = 16, 64, 28, 28
    rng = np.random.default_rng(3)
    x, g = (rng.standard_normal((N, C, H, W)).astype(np.float32) for _ in range(2))
    X, Wt, DX = dev.put(x), dev.put(rng.standard_normal((C, C, 3, 3)).astype(np.float32)), dev.empty(x.shape)
    DW, DB = dev.empty((C, C, 3, 3)), dev.empty((C,))
    best = []
    for s in (1.0, scale):
        G = dev.put(g * np.float32(s))
        times = []
        for _ in range(6):
            dev.get(DB)
            t = time.perf_counter()
            for _ in range(10):
                dev.call("om_conv2d_bwd", G, X, Wt, DX, DW, DB, N, C, H, W, C, 3, 3, 1, 1, 0, 0)
            dev.get(DB)
            times.append(time.perf_counter() - t)
        best.append(min(times))
    assert best[1] <= factor * best[0]


@pytest.mark.parametrize("bad", [np.inf, np.nan, 2.0 ** 105])
def test_a_pixel_does_not_depend_on_its_neighbours(dev, bad):
    """A value the split does not carry changes the sums that it is part of and no bit of another."""
    N, C, H, W = 6, 32, 17, 19
    rng = np.random.default_rng(31)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    w = dev.put(rng.standard_normal((C, C, 3, 3)).astype(np.float32))
    b, y = dev.put(np.zeros(C, np.float32)), dev.empty(x.shape)
    keep = np.ones(x.shape, bool)
    keep[2, :, 4:7, 8:11] = False
    out = []
    for v in (x[2, 3, 5, 9], bad):
        x[2, 3, 5, 9] = v
        X = dev.put(x)
        dev.call("om_conv2d_fwd", X, w, b, y, N, C, H, W, C, 3, 3, 1, 1)
        out.append(dev.get(y)[keep])
        dev.call("om_conv2d_bwd", X, X, w, y, dev.empty((C, C, 3, 3)), None, N, C, H, W, C, 3, 3, 1, 1, 0, 0)
        out.append(dev.get(y)[keep])
    assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[3])
