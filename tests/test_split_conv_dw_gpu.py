"""The split-operand weight gradient of the 3x3 convolutions (csrc/om_conv3_dw_s.hpp) at the sizes and values where it can go
wrong: one pixel, odd numbers of eight-column groups, widths that are no multiple of 4 or 8, column segments, bands past the
last row, slots with one and many items, several channel blocks, accumulation, and operands the three-way bf16 split does not
carry, against float64 over the zero-padded input.

Tolerance: for edges and values the sequential-accumulation bound k 2^-24 sum |g||x| over the k = N H W terms, and a rounding of
the later addition; for the precision itself, single products within 2^-23. The bias gradient is summed in double and rounded
once.
"""
import numpy as np
import pytest

import gpu_util

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return gpu_util.Dev()


def dw64(g, x):
    n, ci, h, w = x.shape
    xp = np.zeros((n, ci, h + 2, w + 2))
    xp[:, :, 1:-1, 1:-1] = x
    out = np.zeros((g.shape[1], ci, 3, 3))
    gf = g.astype(np.float64).reshape(n, g.shape[1], -1)
    for ky in range(3):
        for kx in range(3):
            xs = xp[:, :, ky:ky + h, kx:kx + w].reshape(n, ci, -1)
            out[:, :, ky, kx] = sum(gf[i] @ xs[i].T for i in range(n))
    return out


@pytest.mark.parametrize("N,Cin,Cout,H,W", [
    (4100, 32, 64, 1, 1), (300, 32, 64, 3, 5), (90, 64, 64, 7, 7), (26, 96, 64, 5, 33), (9, 32, 192, 19, 27),
    (40, 64, 64, 15, 17), (6, 32, 64, 4, 185), (1, 32, 128, 90, 62), (450, 32, 64, 3, 3), (4, 32, 64, 16, 112),
    (28, 64, 64, 2, 74), (7, 32, 64, 9, 73), (1, 32, 64, 4001, 1)])
def test_edges(dev, N, Cin, Cout, H, W):
    rng = np.random.default_rng(N + 31 * Cin + 1009 * Cout + 7 * W)
    x = rng.standard_normal((N, Cin, H, W)).astype(np.float32)
    g = rng.standard_normal((N, Cout, H, W)).astype(np.float32)
    w0 = rng.standard_normal((Cout, Cin, 3, 3)).astype(np.float32)
    want, mag, dbw = dw64(g, x), dw64(np.abs(g), np.abs(x)), g.astype(np.float64).sum((0, 2, 3))
    X, G, Wd = dev.put(x), dev.put(g), dev.put(w0)
    for acc in (0, 1):
        DW, DB = dev.put(w0.copy()), dev.empty((Cout,), fill=np.nan)
        dev.call("om_conv2d_bwd", G, X, Wd, None, DW, None if acc else DB, N, Cin, H, W, Cout, 3, 3, 1, 1, 0, acc)
        ref = want + w0 if acc else want
        bound = N * H * W * 2.0 ** -24 * mag + 2.0 ** -22 * (np.abs(ref) + acc * np.abs(w0)) + 2.0 ** -149
        assert np.all(np.abs(dev.get(DW) - ref) <= bound)
        if not acc:
            assert np.all(np.abs(dev.get(DB) - dbw) <= 2.0 ** -23 * np.abs(dbw) + 1e-12)


@pytest.mark.parametrize("N,Cin,Cout,H,W", [(4100, 32, 64, 1, 1), (90, 64, 64, 7, 7), (26, 96, 64, 5, 33), (9, 32, 192, 19, 27), (40, 64, 64, 15, 17),
                                            (6, 32, 64, 4, 185), (4, 32, 64, 16, 112), (450, 32, 64, 3, 3), (7, 32, 64, 9, 73)])
def test_single_products(dev, N, Cin, Cout, H, W):
    """One pixel of g in each output channel, at the borders, at the edges of column groups and segments and inside, so every result is
    one product of two full significands (or the zero beside the image) and shows each of the six terms: a lost or misplaced plane
    leaves 2^-17 or more (test_split_terms.py)."""
    rng = np.random.default_rng(N + W)
    x, g, i = gpu_util.full_significands(rng, (N, Cin, H, W)), np.zeros((N, Cout, H, W), np.float32), np.arange(Cout)
    cols = np.array([0, W - 1, 7, 8, 9, 15, 23, 24, 31, 32, 33, W // 2, W - 2]) % W
    g[i * 5 % N, i, i * 3 % H, cols[i % len(cols)]] = gpu_util.full_significands(rng, Cout)
    DW = dev.empty((Cout, Cin, 3, 3))
    dev.call("om_conv2d_bwd", dev.put(g), dev.put(x), dev.put(np.zeros(DW.shape, np.float32)), None, DW, None, N, Cin, H, W, Cout, 3, 3, 1,
             1, 0, 0)
    want = dw64(g, x)
    assert np.all(np.abs(dev.get(DW) - want) <= gpu_util.SPLIT_PRODUCT * np.abs(want))


def test_values_the_split_does_not_carry(dev):
    N, C, H, W = 61, 64, 6, 11
    rng = np.random.default_rng(11)
    x = rng.standard_normal((N, C, H, W)).astype(np.float32)
    g = rng.standard_normal((N, C, H, W)).astype(np.float32) * np.float32(2.0 ** -8)
    x[0, 1, 0, 0], x[0, 2, 3, W - 1], x[0, 3, 5, 2], x[0, 4, 3, 5] = np.inf, -np.inf, np.nan, 3.4e38
    g[1, 5, 2, 2] = np.inf
    g[2, 6, 0, 0] = np.inf  # beside the zeros around the image: NaN in their taps, as the padded sum has it
    g[:, 9] *= np.float32(1e-36)
    with np.errstate(invalid="ignore", over="ignore"):
        want, mag = dw64(g, x), dw64(np.abs(g), np.abs(x))
        DW, DB = dev.empty((C, C, 3, 3)), dev.empty((C,))
        dev.call("om_conv2d_bwd", dev.put(g), dev.put(x), dev.put(np.zeros((C, C, 3, 3), np.float32)), None, DW, DB, N, C, H,
                 W, C, 3, 3, 1, 1, 0, 0)
        got, fin = dev.get(DW), np.isfinite(want)
        bound = N * H * W * (2.0 ** -23 * mag + 2.0 ** -148)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        assert np.all(np.abs(got[fin] - want[fin]) <= bound[fin])
        assert np.array_equal(dev.get(DB)[[5, 6]], np.float32([np.inf, np.inf]))


# exponents of the tiny operand (the last two pairs: subnormals) and of its partner
@pytest.mark.parametrize("et,ew", [(-115, 26), (-120, 40), (-125, 60), (-135, 100), (-145, 100), (-140, 0)])
def test_tiny_operands_beside_large_ones(dev, et, ew):
    """Operands down to the smallest subnormals times operands up to 2^100, whichever of the two is tiny: every term keeps all
    its bits. The bound is test_edges's, and for sums that are subnormal themselves half a unit of the last place a term."""
    N, Cin, Cout, H, W = 40, 32, 64, 9, 13
    rng = np.random.default_rng(23)
    x0, g0 = (rng.standard_normal((N, c, H, W)).astype(np.float32) for c in (Cin, Cout))
    for ex, eg in ((et, ew), (ew, et)):
        x, g = np.ldexp(x0, ex), np.ldexp(g0, eg)
        DW = dev.empty((Cout, Cin, 3, 3))
        dev.call("om_conv2d_bwd", dev.put(g), dev.put(x), dev.put(np.zeros(DW.shape, np.float32)), None, DW, None, N, Cin, H,
                 W, Cout, 3, 3, 1, 1, 0, 0)
        bound = N * H * W * (2.0 ** -24 * dw64(np.abs(g), np.abs(x)) + 2.0 ** -150)
        assert np.all(np.abs(dev.get(DW) - dw64(g, x)) <= bound), (ex, eg)


@pytest.mark.parametrize("bad", [np.inf, np.nan, 2.0 ** 105])
def test_a_channel_does_not_depend_on_its_neighbours(dev, bad):
    """A value the split does not carry changes its own channels' gradients and no bit of another."""
    N, Cin, Cout, H, W = 40, 32, 64, 9, 13
    rng = np.random.default_rng(37)
    x, g = (rng.standard_normal((N, c, H, W)).astype(np.float32) for c in (Cin, Cout))
    zero, out = np.zeros((Cout, Cin, 3, 3), np.float32), []
    for v, u in ((x[2, 3, 5, 9], g[1, 40, 0, 0]), (bad, bad)):
        x[2, 3, 5, 9], g[1, 40, 0, 0] = v, u
        DW = dev.empty(zero.shape)
        dev.call("om_conv2d_bwd", dev.put(g), dev.put(x), dev.put(zero), None, DW, None, N, Cin, H, W, Cout, 3, 3, 1, 1, 0, 0)
        out.append(np.delete(np.delete(dev.get(DW), 3, 1), 40, 0))
    assert np.array_equal(out[0], out[1])
