"""The split-operand product (csrc/om_gemm_s.hpp) at the sizes and values where it can go wrong: partial tiles in both
directions, K tails and uneven k groups, the last partial quad of columns, split K with its reduce, odd leading
dimensions, operands the three-way bf16 split does not carry (infinities, NaN, values past the scaled range) and tiny ones,
and the sizes on either side of the dispatch's rules, against float64.

Tolerance: for edges and values, where a wrong index shows, the sequential-accumulation bound k 2^-24 |A||B| that
test_gemm_parity holds the product to (the kernel's own rounding count is lower: one per 16 terms and five per 16 on sums
2^-7 as large); for the precision itself, single products within 2^-23 and the measured error of long sums.
"""
import numpy as np
import pytest

import gpu_util

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return gpu_util.Dev()


def product(dev, ta, tb, A, B, m, n, k, ldc=None, c0=None, bias=None, acc=0):
    a, b = dev.put(A), dev.put(B)
    c = dev.put(c0) if c0 is not None else dev.empty((m, n), fill=np.nan)
    dev.call("om_gemm", ta, tb, m, n, k, a, A.shape[1], b, B.shape[1], c, ldc or n,
             dev.put(bias) if bias is not None else None, acc, None)
    return dev.get(c)


def operands(rng, ta, tb, m, n, k, pad=0):
    A = rng.standard_normal((k, m + pad) if ta else (m, k + pad)).astype(np.float32)
    B = rng.standard_normal((n, k + pad) if tb else (k, n + pad)).astype(np.float32)
    A64 = (A[:, :m].T if ta else A[:, :k]).astype(np.float64)
    B64 = (B[:, :k].T if tb else B[:, :n]).astype(np.float64)
    return A, B, A64, B64


LAYOUTS = [(0, 1), (0, 0), (1, 0)]
SHAPES = [(1, 4, 16), (31, 5, 33), (33, 7, 47), (64, 65, 31), (65, 63, 127), (127, 97, 129), (129, 95, 161), (257, 130, 200),
          (96, 255, 513), (70, 66, 4099), (1030, 390, 95), (2050, 258, 321), (4096, 99, 40)]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(dev, ta, tb, m, n, k):
    rng = np.random.default_rng(m + 31 * n + 1009 * k)
    A, B, A64, B64 = operands(rng, ta, tb, m, n, k, pad=3)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((m, n + 1)).astype(np.float32)
    got = product(dev, ta, tb, A, B, m, n, k, ldc=n + 1, c0=c0.copy(), bias=bias, acc=1)
    assert np.array_equal(got[:, n], c0[:, n])  # nothing past the last column
    want = A64 @ B64 + bias + c0[:, :n]
    bound = k * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) + 2.0 ** -22 * (np.abs(bias) + np.abs(c0[:, :n]) + np.abs(want))
    assert np.all(np.abs(got[:, :n] - want) <= bound)


# Every tile shape of the kernel, whole and ragged tiles, split K or not (on 256 CUs).
TILES = [(6144, 1003, 64), (6144, 1024, 64), (3000, 1536, 64), (3072, 1536, 64), (3000, 1003, 64), (3072, 1024, 64), (2050, 1003, 64),
         (1536, 1536, 64), (1500, 1003, 96), (1536, 1024, 96), (2050, 512, 96), (1000, 192, 768), (768, 1536, 384), (1536, 96, 768),
         (64, 37, 96), (64, 37, 512), (256, 384, 384), (384, 192, 768), (64, 37, 64), (64, 37, 391), (1536, 1024, 64), (64, 64, 384)]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", TILES)
def test_single_products(dev, ta, tb, m, n, k):
    """A has one element in each row, so every result is one product of two full significands and shows each of the six terms: a
    lost or misplaced plane leaves 2^-17 or more (test_split_terms.py)."""
    rng = np.random.default_rng(m + n + k)
    at = (np.arange(m) * 29) % k
    A64, a = np.zeros((m, k), np.float32), gpu_util.full_significands(rng, m)
    A64[np.arange(m), at] = a
    B = gpu_util.full_significands(rng, (n, k) if tb else (k, n))
    got = product(dev, ta, tb, np.ascontiguousarray(A64.T) if ta else A64, B, m, n, k)
    want = a.astype(np.float64)[:, None] * (B.T if tb else B)[at]
    assert np.all(np.abs(got - want) <= gpu_util.SPLIT_PRODUCT * np.abs(want))


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(130, 70, 200), (512, 384, 384)])
def test_values_the_split_does_not_carry(dev, ta, tb, m, n, k):
    rng = np.random.default_rng(5)
    A, B, A64, B64 = operands(rng, ta, tb, m, n, k)

    def put(row, col, v):
        A[(col, row) if ta else (row, col)] = v
        A64[row, col] = v

    put(3, 1, np.inf)
    put(m - 1, k - 1, -np.inf)
    put(40, k // 2, np.nan)
    put(70, 9, 3.4e38)  # finite, past the largest bf16
    # one row, and elsewhere one column, of tiny values
    for c in range(k):
        put(100, c, A64[100, c] * 1e-36)
    if tb:
        B[20] *= np.float32(1e-30)
    else:
        B[:, 20] *= np.float32(1e-30)
    B64 = (B.T if tb else B).astype(np.float64)
    A64 = (A.T if ta else A).astype(np.float64)
    # keep the large row's sums inside fp32: its partner values shrink by 2^-10 in every column
    if tb:
        B[:, 9] *= np.float32(2.0 ** -10)
    else:
        B[9] *= np.float32(2.0 ** -10)
    B64 = (B.T if tb else B).astype(np.float64)
    got = product(dev, ta, tb, A, B, m, n, k)
    with np.errstate(invalid="ignore", over="ignore"):
        want = A64 @ B64
        bound = k * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) + 2.0 ** -148 * k
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert np.all(np.abs(got[fin] - want[fin]) <= bound[fin])


@pytest.mark.parametrize("rows,sizes", [(999, [(128, 192), (64, 64)]), (4100, [(384, 384), (1152, 384), (384, 1536)]),
                                        (96, [(64, 128), (192, 64), (128, 64), (64, 64)])])
def test_grouped_weight_gradients(dev, rows, sizes):
    rng = np.random.default_rng(rows)
    items = (dev.pkg.om_linear_dw * len(sizes))()
    keep, want = [], []
    for it, (out, in_) in zip(items, sizes):
        g, x = (rng.standard_normal((rows, s)).astype(np.float32) for s in (out, in_))
        b = [dev.put(g), dev.put(x), dev.empty((out, in_), fill=np.nan), dev.empty((out,), fill=np.nan)]
        keep.append(b)
        it.g, it.x, it.dw, it.db = (t.data_ptr() for t in b)
        it.in_, it.out, it.acc_dw, it.acc_db = in_, out, 0, 0
        want.append((g.astype(np.float64), x.astype(np.float64)))
    dev.call("om_linear_bwd_dw_group", len(sizes), items, rows)
    for b, (g, x) in zip(keep, want):
        assert np.all(np.abs(dev.get(b[2]) - g.T @ x) <= rows * 2.0 ** -24 * (np.abs(g).T @ np.abs(x)))
        s = g.sum(0)
        assert np.all(np.abs(dev.get(b[3]) - s) <= 2.0 ** -23 * np.abs(s) + 1e-12 * np.abs(g).sum(0))  # summed in double


# exponents of the tiny operand (the last two pairs: subnormals) and of its partner
TINY_WIDE = [(-115, 26), (-120, 40), (-125, 60), (-135, 100), (-145, 100), (-140, 0)]


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(130, 71, 203), (512, 384, 384)])
def test_tiny_operands_beside_large_ones(dev, ta, tb, m, n, k):
    """Operands down to the smallest subnormals times operands up to 2^100, whichever of the two is tiny: every term keeps all
    its bits. The bound is test_edges's, and for sums that are subnormal themselves half a unit of the last place a term."""
    rng = np.random.default_rng(17)
    A0, B0, _, _ = operands(rng, ta, tb, m, n, k)
    for pair in TINY_WIDE:
        for ea, eb in (pair, pair[::-1]):
            A, B = np.ldexp(A0, ea), np.ldexp(B0, eb)
            A64, B64 = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
            bound = k * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) + k * 2.0 ** -150
            assert np.all(np.abs(product(dev, ta, tb, A, B, m, n, k) - A64 @ B64) <= bound), (ea, eb)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(130, 71, 203), (512, 384, 384)])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 2.0 ** 105])
def test_a_row_does_not_depend_on_its_neighbours(dev, ta, tb, m, n, k, bad):
    """A value the split does not carry changes its own row (column) of the product and no bit of another."""
    A, B, _, _ = operands(np.random.default_rng(29), ta, tb, m, n, k)
    clean = product(dev, ta, tb, A, B, m, n, k)
    A[(7, 37) if ta else (37, 7)] = bad
    B[(20, 9) if tb else (9, 20)] = bad
    got = product(dev, ta, tb, A, B, m, n, k)
    keep = np.ones((m, n), bool)
    keep[37], keep[:, 20] = False, False
    assert np.array_equal(got[keep], clean[keep])


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(64, 64, 192), (64, 64, 288), (64, 64, 320), (512, 384, 224), (1024, 256, 256), (1024, 256, 320),
                                   (1024, 256, 352), (4096, 384, 288), (4096, 384, 320), (4096, 384, 352), (1024, 96, 160), (1024, 96, 192)])
def test_short_sums_on_both_sides_of_the_rule(dev, ta, tb, m, n, k):
    """Whole tiles with sums around the length up to which the fp32 kernels run, with bias and accumulation."""
    rng = np.random.default_rng(m + k)
    A, B, A64, B64 = operands(rng, ta, tb, m, n, k)
    bias, c0 = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    got = product(dev, ta, tb, A, B, m, n, k, c0=c0.copy(), bias=bias, acc=1)
    want = A64 @ B64 + bias + c0
    bound = k * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) + 2.0 ** -22 * (np.abs(bias) + np.abs(c0) + np.abs(want))
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [(16, 16, 16), (32, 32, 63), (33, 32, 40), (128, 128, 65), (128, 100, 351), (129, 100, 163), (128, 128, 353),
                                   (1024, 1024, 16), (1024, 1024, 17)])
def test_small_products_on_both_sides_of_the_rule(dev, ta, tb, m, n, k):
    """Products around the sizes up to which the guarded fp32 kernel runs, with bias and accumulation."""
    rng = np.random.default_rng(m + k)
    A, B, A64, B64 = operands(rng, ta, tb, m, n, k)
    bias, c0 = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    got = product(dev, ta, tb, A, B, m, n, k, c0=c0.copy(), bias=bias, acc=1)
    want = A64 @ B64 + bias + c0
    bound = k * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) + 2.0 ** -22 * (np.abs(bias) + np.abs(c0) + np.abs(want))
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("k,most", [(384, 1.7e-7), (4096, 4.2e-7)])
def test_sums_are_closer_than_the_fp32_instruction(dev, ta, tb, k, most):
    """The 2-norm error of sums of normal products in one chain: one and a half times what was measured (1.1e-7, 2.7e-7), and below the
    fp32 instruction's (3.5e-7, 1.1e-6), whose sums round once per product or four."""
    m, n = 3072, 1536
    A, B, A64, B64 = operands(np.random.default_rng(k), ta, tb, m, n, k)
    got = product(dev, ta, tb, A, B, m, n, k)[::61].astype(np.float64)
    want = A64[::61] @ B64
    assert np.linalg.norm(got - want) <= most * np.linalg.norm(want)
