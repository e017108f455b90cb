"""Large A B^T products of MatMulAlloc (a linear layer's input gradient) on bf16
parts, at tile edges and ragged sizes, and with operands that are not finite,
against the float64 oracle.

Bound per element, as for the convolutions on parts: with S the same sum over
magnitudes, the dropped part products are below 3 * 2^-21 S, and each step of 16
rounds at most eight times by 2^-24 of a partial sum; split-K adds one rounding
per split (at most 16)."""
import numpy as np
import pytest

from oracle import kernels as K
from tests.helpers import download, fma_chain, rel2, release, rng, upload

pytestmark = pytest.mark.gpu

SHAPES = [
    # M, K, N: at least 2e9 products, M > 64, K >= 512 (2048 past 384 rows)
    (65, 5200, 6001),      # one row past a tile, one column past one
    (128, 4096, 3840),     # whole tiles
    (129, 4099, 3901),     # K pads its rows to 4 and its last step to 16
    (384, 512, 10200),     # the shortest dot products
    (385, 2048, 2600),     # and beyond 384 rows
    (200, 100001, 101),    # few columns, long K
]


def _matmul(eng, a, b):
    (M, Kd), N = a.shape, b.shape[0]
    ha, hb = upload(eng, a), upload(eng, b)
    hc = eng.lib.MatMulAlloc(ha, hb, M, Kd, N, 2)
    assert hc, eng.last_error()
    c = download(eng, hc, (M, N))
    release(eng, ha, hb, hc)
    return c


@pytest.mark.parametrize("M,Kd,N", SHAPES)
def test_a_bt_on_parts(eng, M, Kd, N):
    r = rng(M + Kd + N)
    a = r.standard_normal((M, Kd), dtype=np.float32)
    b = r.standard_normal((N, Kd), dtype=np.float32)
    ref = K.matmul(a, b, M, Kd, N, 2)
    S = K.matmul(np.abs(a), np.abs(b), M, Kd, N, 2)
    bound = (3 * 2.0 ** -21 + (8 * (Kd / 16 + 2) + 16) * 2.0 ** -24) * S
    assert np.all(np.abs(_matmul(eng, a, b) - ref) <= bound)


def test_a_bt_not_finite(eng):
    M, Kd, N = 130, 4100, 3800
    r = rng(5)
    a = r.standard_normal((M, Kd), dtype=np.float32)
    b = r.standard_normal((N, Kd), dtype=np.float32)
    a[3, 17], a[129, 4099], b[700, 5], b[3799, 2000] = np.inf, np.nan, -np.inf, np.nan
    b[64, 9] = np.array([0x7F800001], np.uint32).view(np.float32)[0]  # payload in the low half alone
    a[70, 40], b[:, 40], b[700, 40] = 3e38, 1e5, 1.0  # row 70 overflows but beside the infinity
    with np.errstate(all="ignore"):
        ref = K.matmul(a, b, M, Kd, N, 2).astype(np.float32)
    c = _matmul(eng, a, b)
    assert np.array_equal(np.isnan(c), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(c), inf)
    assert np.array_equal(c[inf], ref[inf])
    fin = np.isfinite(ref)
    assert np.max(np.abs(c[fin] - ref[fin])) <= 1e-5 * np.max(np.abs(ref[fin]))


@pytest.mark.parametrize("terms", [1, 4, 64, 4100])
def test_a_bt_error_and_bias_against_fp32_fmas(eng, monkeypatch, terms):
    """As for the convolutions: sums of few and many terms against a chain of fp32
    FMAs (64 rows, 150 columns of the product); one term 1.06.  K is not split: the
    sum of split partials rounds in either arithmetic."""
    monkeypatch.setenv("DCE_TUNE_GEMM", "128,64,16,1")
    M, Kd, N = 130, 4100, 3800
    r = rng(terms)
    a = r.standard_normal((M, Kd), dtype=np.float32)
    b = r.standard_normal((N, Kd), dtype=np.float32)
    if terms < Kd:
        a *= np.stack([r.permutation(Kd) < terms for _ in range(M)])
    part = np.s_[66:130, 3650:3800]
    ref = a[part[0]].astype(np.float64) @ b[part[1]].T.astype(np.float64)
    fp32 = rel2(fma_chain(a[part[0]], b[part[1]]), ref)
    assert rel2(_matmul(eng, a, b)[part], ref) <= (1.06 if terms == 1 else 1.0) * fp32
    a, b = np.abs(a), np.abs(b)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    err = (_matmul(eng, a, b) - ref) / ref
    # 2^-28, a sixteenth of half a unit in the last place, and what a bf16 MFMA cuts
    # off downwards: half of 2^-37 of the accumulator for each of its 16 addends
    assert abs(err.mean()) <= 2.0 ** -28 + terms * 2.0 ** -38


def test_a_bt_largest(eng):
    """Finite values that round to infinity as bf16, with finite products."""
    M, Kd, N = 130, 4100, 3800
    r = rng(23)
    a = r.standard_normal((M, Kd), dtype=np.float32)
    b = r.standard_normal((N, Kd), dtype=np.float32) * np.float32(1e-3)
    a[7, 4099], a[129, 0] = np.finfo(np.float32).max, np.float32(-3.3999e38)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    S = np.abs(a).astype(np.float64) @ np.abs(b).T.astype(np.float64)
    c = _matmul(eng, a, b)
    assert np.all(np.isfinite(c)) and np.all(np.abs(c - ref) <= 64 * 2.0 ** -24 * S)


@pytest.mark.parametrize("scale", [1e-36, 1e-39, 1e-33])
@pytest.mark.parametrize("which", ["a", "b", "row"])
def test_a_bt_tiny(eng, which, scale):
    """Values below the range of three bf16 parts (8e-34), and just above it: fp32's
    bound, one rounding of 2^-24 or 2^-149 a term."""
    M, Kd, N = 130, 4100, 3800
    r = rng(17)
    a = r.standard_normal((M, Kd), dtype=np.float32)
    b = r.standard_normal((N, Kd), dtype=np.float32)
    if which == "a":
        a *= np.float32(scale)
    elif which == "b":
        b *= np.float32(scale)
    else:
        b[3799] *= np.float32(scale)
    ref = a.astype(np.float64) @ b.T.astype(np.float64)
    S = np.abs(a).astype(np.float64) @ np.abs(b).T.astype(np.float64)
    # Kd roundings of random sign, each at most 2^-24 of a partial sum that S bounds
    assert np.all(np.abs(_matmul(eng, a, b) - ref) <= 64 * 2.0 ** -24 * S + Kd * 2.0 ** -149)
