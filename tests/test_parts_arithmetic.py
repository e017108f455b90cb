"""fp32 products as six products of bf16 parts, in NumPy: the split is exact, the
error of short, sparse and long sums is no larger than that of a chain of fp32
FMAs, it has no bias, and none of the six products can be left out."""
import numpy as np
import pytest

from tests.helpers import fma_chain, rel2, rng

SIX = [(0, 0), (0, 1), (1, 0), (0, 2), (2, 0), (1, 1)]


def bf16(x):
    """Nearest bf16, ties to even (finite x)."""
    u = np.asarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


def split(x):
    h = bf16(x)
    m = bf16(x - h)
    return h, m, bf16(x - h - m)


def parts_sum(a, b, products=SIX, step=16):
    """A [M, K] by B [N, K]: h*h in one fp32 accumulator, the others in a second,
    each rounded after every step of 16."""
    pa, pb = split(a), split(b)
    hi = lo = np.zeros((a.shape[0], b.shape[0]), np.float32)
    for k in range(0, a.shape[1], step):
        for i, j in products:
            t = pa[i][:, k:k + step].astype(np.float64) @ pb[j][:, k:k + step].T.astype(np.float64)
            if (i, j) == (0, 0):
                hi = (hi + t).astype(np.float32)
            else:
                lo = (lo + t).astype(np.float32)
    return hi + lo


def test_split_is_exact():
    r = rng(1)
    x = (r.standard_normal(100000) * np.exp2(r.integers(-100, 120, 100000))).astype(np.float32)
    edge = np.array([1, 0x3F7FFFFF, 0x3F808000, 0x3F808001, 0x3F818000, 0x7F7F7FFF, 0x08800001], np.uint32).view(np.float32)
    for v in (x, -x, edge[1:]):
        h, m, l = split(v)
        assert np.array_equal((h + m) + l, v)
        assert np.all(np.abs(m) <= np.abs(v) * 2.0 ** -8) and np.all(np.abs(l) <= np.abs(v) * 2.0 ** -17)


def _operands(M, N, K, terms, seed):
    r = rng(seed)
    a, b = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((N, K), dtype=np.float32)
    if terms < K:  # a gradient of which `terms` values of each row survive a mask
        a *= np.stack([r.permutation(K) < terms for _ in range(M)])
    return a, b


@pytest.mark.parametrize("K,terms", [(1, 1), (16, 16), (400, 1), (400, 4), (400, 16), (1152, 64), (1152, 1152)])
def test_error_against_a_chain_of_fmas(K, terms):
    """One product: its rounding, 2^-24 / sqrt(12) times the spread of significands,
    and the dropped m*l and l*m (28 % of it): sqrt(1 + 0.28^2) = 1.04."""
    a, b = _operands(128, 160, K, terms, K + terms)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    got, fp32 = rel2(parts_sum(a, b), ref), rel2(fma_chain(a, b), ref)
    assert got <= fp32 * (1.06 if terms == 1 else 1.0), (got, fp32)


@pytest.mark.parametrize("K", [1, 16, 400])
def test_no_bias(K):
    a, b = _operands(128, 160, K, K, 50 + K)
    a, b = np.abs(a), np.abs(b)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    err = (parts_sum(a, b) - ref) / ref
    assert abs(err.mean()) <= 6 * err.std() / np.sqrt(err.size)


@pytest.mark.parametrize("drop", SIX)
def test_every_product_counts(drop):
    """Five products are worse than fp32: h*l alone (2^-18.7 of a product) four times."""
    a, b = _operands(64, 64, 1152, 1152, 9)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    assert rel2(parts_sum(a, b, [p for p in SIX if p != drop]), ref) > 2 * rel2(fma_chain(a, b), ref)
