"""The six-term product of exactly split fp32 values (csrc/om_split.hpp), modelled on the CPU: the bound that the GPU tests hold
single products to (gpu_util.SPLIT_PRODUCT) is met by all six terms and missed when any of the five small ones is lost.
"""
import numpy as np
import pytest

import gpu_util


def bf16(x):
    """Rounded to the nearest bf16, ties to even."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def split(x):
    h = bf16(x)
    m = bf16(x - h)
    return h, m, bf16(x - h - m)


TERMS = [(1, 1), (2, 0), (0, 2), (1, 0), (0, 1)]


def product(a, b, lost=None):
    """The kernel's order: the small terms one after another in fp32, then added to hh."""
    pa, pb = split(a), split(b)
    low = np.float32(0)
    for t in TERMS:
        if t != lost:
            low = (low + pa[t[0]].astype(np.float64) * pb[t[1]]).astype(np.float32)
    return (pa[0].astype(np.float64) * pb[0]).astype(np.float32) + low


def pairs():
    rng = np.random.default_rng(1)
    a, b = (gpu_util.full_significands(rng, 200000) for _ in range(2))
    near = np.float32(1) + np.arange(1, 1 << 18, 41, dtype=np.float32) * np.float32(2.0 ** -23)  # where parts are largest
    return np.concatenate([a, near]), np.concatenate([b, near[::-1]])


def test_the_split_is_exact():
    a, _ = pairs()
    h, m, l = split(a)
    assert np.array_equal(h.astype(np.float64) + m + l, a.astype(np.float64))


def test_six_terms_meet_the_bound():
    a, b = pairs()
    want = a.astype(np.float64) * b
    assert np.all(np.abs(product(a, b) - want) <= gpu_util.SPLIT_PRODUCT * np.abs(want))


@pytest.mark.parametrize("lost", TERMS)
def test_a_lost_term_misses_it(lost):
    a, b = pairs()
    want = a.astype(np.float64) * b
    assert np.mean(np.abs(product(a, b, lost) - want) > gpu_util.SPLIT_PRODUCT * np.abs(want)) > 0.5
