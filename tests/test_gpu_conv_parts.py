"""Conv backward on bf16 parts (dW and dX as six bf16 MFMA products per fp32
product) against the float64 oracle: tile edges, channels that fill no block of
16, strides with their sub-pixel phases, split-K, and operands that are
infinite, NaN, overflowing or tiny.

Bound per element, from the arithmetic: with S the same sum over |a||b| and n
steps of 16 k, the dropped part products are below 2^-21 S each, and a step
rounds the accumulator twice and its inner sum once per product group (6 at
most), all below 2^-24 of a partial sum that S bounds; split-K adds one rounding
per split (at most 256) of the partial sums."""
import ctypes

import numpy as np
import pytest

from oracle import kernels as K
from tests.helpers import download, fma_chain, he, rel2, release, rng, upload

pytestmark = pytest.mark.gpu

CASES = [
    # B, C, H, W, OC, k, s, p, act
    (2, 64, 9, 7, 64, 3, 1, 1, 0),        # one 64-row tile, ragged pixels
    (2, 65, 8, 8, 64, 3, 1, 1, 1),        # one channel past a tile and a block
    (1, 48, 11, 13, 128, 3, 1, 1, 1),
    (3, 37, 13, 9, 70, 5, 1, 2, 0),       # channels padded to 48 and 80
    (2, 33, 7, 7, 129, 3, 1, 0, 1),       # no padding; 129 output rows
    (1, 32, 6, 6, 384, 5, 1, 2, 0),       # few rows, long K
    (2, 128, 5, 5, 130, 3, 1, 1, 0),
    (4, 96, 32, 32, 64, 3, 1, 1, 1),      # split-K dW
    (2, 64, 12, 10, 96, 3, 2, 1, 1),      # stride 2: four phases in one launch
    (2, 40, 13, 11, 70, 5, 2, 2, 0),      # odd image, phases of unequal size
    (1, 64, 1, 9, 64, 3, 2, 1, 0),        # phases with no rows
    (2, 512, 8, 8, 480, 1, 2, 0, 0),      # k < s: three phases no tap reaches
    (2, 64, 14, 14, 64, 4, 3, 1, 1),      # stride 3: one launch per phase
    (2, 512, 6, 6, 480, 1, 1, 0, 1),      # pointwise with a ReLU mask
    (7, 137, 6, 7, 505, 3, 2, 0, 0),      # phases of few pixels and long dot products, split
    (1, 56, 7, 15, 384, 7, 2, 3, 1),      # the same: 16, 12, 12 and 9 taps
]


def _backward(eng, x, w, dy, y, s, p, act, pim=None):
    B, C, H, W = x.shape
    OC, _, k, _ = w.shape
    hs = [upload(eng, a) for a in (dy, x, w)]
    hy = upload(eng, y) if act == 1 else None
    pdf, pdb, pdx = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    eng.lib.ConvBackwardFused(hs[0], hy, hs[1], hs[2], pim, B, C, H, W, OC, k, k, s, p, act, 1, 1, 1,
                              ctypes.byref(pdf), ctypes.byref(pdb), ctypes.byref(pdx))
    assert pdf.value and pdb.value and pdx.value, eng.last_error()
    out = (download(eng, pdf.value, w.shape), download(eng, pdb.value, (OC,)), download(eng, pdx.value, x.shape))
    release(eng, *hs, hy, pdf.value, pdb.value, pdx.value)
    return out


def _inputs(B, C, H, W, OC, k, s, p, act):
    r = rng(77 + B + 3 * C + 5 * H + 7 * OC + 11 * k + s)
    x = r.standard_normal((B, C, H, W)).astype(np.float32)
    w = he(r, (OC, C, k, k), C * k * k)
    OH, OW = K.conv_out_hw(H, W, k, s, p)
    dy = r.standard_normal((B, OC, OH, OW)).astype(np.float32)
    y = r.standard_normal(dy.shape).astype(np.float32)
    return x, w, dy, y


def _check(got, x, w, dy, y, s, p, act):
    OC, C, k, _ = w.shape
    ref = K.conv_backward(dy, y, x, w, s, p, act)
    S = K.conv_backward(np.abs(dy), y, np.abs(x), np.abs(w), s, p, act)
    for name, a, b, t, n in (("dW", got[0], ref[0], S[0], dy.size // OC), ("dX", got[2], ref[2], S[2], OC * k * k)):
        bound = (3 * 2.0 ** -21 + (8 * (n / 16 + 2) + 256) * 2.0 ** -24) * t + 1e-37
        worst = np.max(np.abs(a - b) - bound)
        assert worst <= 0, f"{name}: {worst:.3e} past the bound"
    # db: fp32 sums of at most B*OH*OW values
    assert np.all(np.abs(got[1] - ref[1]) <= (dy.size // OC) * 2.0 ** -24 * S[1] + 1e-37)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("keep", [True, False])
def test_backward_on_parts(eng, case, keep):
    """With the copy of x that the forward keeps, and rebuilt from x."""
    B, C, H, W, OC, k, s, p, act = case
    x, w, dy, y = _inputs(*case)
    pim = ctypes.c_void_p()
    if keep:
        hx, hw, hb = upload(eng, x), upload(eng, w), upload(eng, np.zeros(OC, np.float32))
        hy = eng.lib.ConvForwardFused(hx, hw, hb, B, C, H, W, OC, k, k, s, p, 0, ctypes.byref(pim))
        assert hy, eng.last_error()
        yref = K.conv_forward(x, w, np.zeros(OC, np.float32), s, p, 0)
        assert np.max(np.abs(download(eng, hy, yref.shape) - yref)) <= 1e-4 * np.max(np.abs(yref))
        release(eng, hx, hw, hb, hy)
    _check(_backward(eng, x, w, dy, y, s, p, act, pim.value), x, w, dy, y, s, p, act)


@pytest.mark.parametrize("tile", ["128,128,16,1", "128,64,16,3", "64,128,16,2", "64,64,16,5"])
def test_forced_tiles(eng, monkeypatch, tile):
    monkeypatch.setenv("DCE_TUNE_DW", tile)
    monkeypatch.setenv("DCE_TUNE_DX", tile)
    for case in (CASES[3], CASES[4], CASES[7]):
        x, w, dy, y = _inputs(*case)
        s, p, act = case[6:]
        _check(_backward(eng, x, w, dy, y, s, p, act), x, w, dy, y, s, p, act)


@pytest.mark.parametrize("splits", [1, 2, 5])
@pytest.mark.parametrize("case,var", [
    ((1, 96, 11, 13, 32, 3, 1, 1, 1), "DCE_TUNE_DW"),   # 32 output channels
    ((2, 90, 9, 7, 32, 5, 2, 2, 0), "DCE_TUNE_DW"),
    ((1, 32, 7, 9, 384, 5, 1, 2, 0), "DCE_TUNE_DX"),    # 32 input channels, ragged pixels
    ((2, 32, 11, 10, 300, 3, 2, 1, 1), "DCE_TUNE_DX"),  # their phases
], ids=str)
def test_32_row_tiles(eng, monkeypatch, capfd, case, var, splits):
    monkeypatch.setenv(var, f"32,128,16,{splits}")
    monkeypatch.setenv("DCE_TUNE_LOG", "1")
    x, w, dy, y = _inputs(*case)
    s, p, act = case[6:]
    _check(_backward(eng, x, w, dy, y, s, p, act), x, w, dy, y, s, p, act)
    log = [l for l in capfd.readouterr().err.splitlines() if f"{var} parts" in l]
    assert log and all("-> 32x128" in l for l in log), log


@pytest.mark.parametrize("what", ["inf", "nan", "quiet", "overflow", "tiny", "tiny weights", "few tiny", "denormal", "largest"])
def test_special_values(eng, what):
    """Infinities and NaNs come out where IEEE arithmetic puts them (the tile is
    computed again in fp32), and so do values below the range of three bf16 parts,
    to fp32's own bound: as many roundings of 2^-24, or 2^-149 below 2^-126."""
    case = (2, 64, 9, 10, 80, 3, 1, 1, 0)
    x, w, dy, y = _inputs(*case)
    s, p, act = case[6:]
    if what == "inf":
        dy[0, 5, 4, 4], x[1, 7, 3, 3] = np.inf, -np.inf
    elif what == "nan":
        dy[1, 60, 0, 0] = np.nan
    elif what == "quiet":  # a NaN whose payload sits in the low 16 bits alone
        dy[1, 60, 0, 0] = np.array([0x7F800001], np.uint32).view(np.float32)[0]
    elif what == "overflow":
        dy[0, 3, 2, 2], w[3, :, :, :] = 3e38, 3e5
    elif what == "tiny":
        dy *= np.float32(1e-36)
    elif what == "tiny weights":
        w *= np.float32(3e-35)
    elif what == "few tiny":  # a channel alone: its sums have nothing larger in them
        x[:, 9] *= np.float32(2e-37)
        w[:, 9] *= np.float32(2e-37)
        dy[:, 70] *= np.float32(2e-37)
    elif what == "largest":  # finite, but rounds to infinity as bf16; its products stay finite
        dy[1, 60, 4, 4] = np.finfo(np.float32).max
        x, w = x * np.float32(1e-3), w * np.float32(1e-3)
    else:
        dy *= np.float32(1e-39)
    with np.errstate(all="ignore"):
        ref = K.conv_backward(dy, y, x, w, s, p, act)
    got = _backward(eng, x, w, dy, y, s, p, act)
    for a, b in ((got[0], ref[0]), (got[2], ref[2])):
        with np.errstate(all="ignore"):
            b32 = b.astype(np.float32)
        assert np.array_equal(np.isnan(a), np.isnan(b32))
        assert np.array_equal(np.isinf(a), np.isinf(b32))
        inf = np.isinf(b32)
        assert np.array_equal(a[inf], b32[inf])
        fin = np.isfinite(b32)
        scale = np.max(np.abs(b[fin])) if what != "overflow" else np.maximum(np.abs(b[fin]), 1.0)
        tol = 1e-5
        if "tiny" in what or what in ("denormal", "largest"):
            Sm = K.conv_backward(np.abs(dy), y, np.abs(x), np.abs(w), s, p, act)
            Sm, n = (Sm[0], 180) if a is got[0] else (Sm[2], 720)
            assert np.all(np.abs(a - b) <= (n + 256) * (2.0 ** -24 * Sm + 2.0 ** -149))
        elif what == "overflow":  # sums of huge terms cancel: relative to the sum of magnitudes
            Sm = K.conv_backward(np.abs(dy), y, np.abs(x), np.abs(w), s, p, act)
            Sm = (Sm[0] if a is got[0] else Sm[2])[fin]
            assert np.all(np.abs(a[fin] - b[fin]) <= 1e-5 * Sm + 1e-30)
        else:
            assert np.max(np.abs(a[fin] - b[fin])) <= tol * scale


def _patches(a, k, p):
    """[C][H][W] -> [pixels][(c, kh, kw)] of a stride-1 layer."""
    C, H, W = a.shape
    q = np.pad(a, ((0, 0), (p, p), (p, p)))
    v = np.lib.stride_tricks.sliding_window_view(q, (k, k), (1, 2))
    return np.ascontiguousarray(v.transpose(1, 2, 0, 3, 4).reshape(v.shape[1] * v.shape[2], -1))


@pytest.mark.parametrize("keep", [0, 0.02, 0.25, 1], ids=["one", "2%", "25%", "dense"])
def test_error_and_bias_against_fp32_fmas(eng, keep):
    """Sums of one, few and many terms (a masked gradient) are no further from
    float64 than a chain of fp32 FMAs, and not off to one side.  One term: 1.06,
    its rounding and the dropped products."""
    B, C, H, W, OC, k, s, p = 1, 64, 13, 13, 64, 3, 1, 1
    r = rng(31)
    x = r.standard_normal((B, C, H, W)).astype(np.float32)
    w = he(r, (OC, C, k, k), C * k * k)
    dy = r.standard_normal((B, OC, H, W)).astype(np.float32)
    if keep == 0:
        dy[:] = dy * (np.arange(H * W).reshape(H, W) == 85)
    elif keep < 1:
        dy *= r.random(dy.shape) < keep
    dw, _, dx = _backward(eng, x, w, dy, None, s, p, 0)
    ref = K.conv_backward(dy, dy, x, w, s, p, 0)
    fdw = fma_chain(dy.reshape(OC, -1), _patches(x[0], k, p).T).reshape(w.shape)
    flip = w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3).reshape(C, -1)
    fdx = fma_chain(flip, _patches(dy[0], k, k - 1 - p)).reshape(x.shape)
    for name, got, want, fp32 in (("dW", dw, ref[0], fdw), ("dX", dx, ref[2], fdx)):
        slack = 1.06 if name == "dW" and keep == 0 else 1.0
        assert rel2(got, want) <= slack * rel2(fp32, want), name
    # operands of one sign: nothing cancels a bias
    dw, _, dx = _backward(eng, np.abs(x), np.abs(w), np.abs(dy), None, s, p, 0)
    ref = K.conv_backward(np.abs(dy), dy, np.abs(x), np.abs(w), s, p, 0)
    for name, got, want in (("dW", dw, ref[0]), ("dX", dx, ref[2])):
        on = want > 0
        err = (got[on] - want[on]) / want[on]
        # 2^-28, a sixteenth of half a unit in the last place, and what a bf16 MFMA
        # cuts off downwards: half of 2^-37 of the accumulator for each addend
        assert abs(err.mean()) <= 2.0 ** -28 + OC * k * k * 2.0 ** -38, name


def _bytes(eng, fam):
    n, v = ctypes.c_uint64(), [ctypes.c_double() for _ in range(3)]
    ok = eng.lib.GetProfile(fam.encode(), ctypes.byref(n), *[ctypes.byref(d) for d in v])
    return v[2].value if ok else 0.0


def test_forward_alone_pays_nothing(eng):
    """A forward that may get a backward moves and holds what one without does: its
    own fp32 copy of x (33 channels: 36 in memory, 48 as parts).  The backward
    splits that copy, and only for a dW."""
    B, C, H, W, OC, k, s, p, act = CASES[4]
    x, w, dy, y = _inputs(*CASES[4])
    hx, hw, hb = upload(eng, x), upload(eng, w), upload(eng, np.zeros(OC, np.float32))
    hdy = upload(eng, dy)
    eng.lib.SetProfiling(1)
    try:
        moved = []
        for pim in (None, ctypes.c_void_p()):
            eng.lib.ResetProfile()
            hy = eng.lib.ConvForwardFused(hx, hw, hb, B, C, H, W, OC, k, k, s, p, 0,
                                          None if pim is None else ctypes.byref(pim))
            assert hy, eng.last_error()
            moved.append(_bytes(eng, "nhwc"))
            release(eng, hy)
        assert moved[0] == moved[1] == 4.0 * B * H * W * (C + 36)
        # dX alone (frozen filters)
        eng.lib.ResetProfile()
        pdx = ctypes.c_void_p()
        eng.lib.ConvBackwardFused(hdy, None, hx, hw, pim.value, B, C, H, W, OC, k, k, s, p, 0, 1, 0, 0,
                                  None, None, ctypes.byref(pdx))
        assert pdx.value, eng.last_error()
        assert _bytes(eng, "x_parts") == 0 and _bytes(eng, "nhwc") == 4.0 * (dy.size + dy.size // OC * 144 * 1.5)
        release(eng, pdx.value)
    finally:
        eng.lib.SetProfiling(0)
        eng.lib.ResetProfile()
    # what a handle holds: the pool gets it back when it is released
    eng.lib.DrainPool()
    pim = ctypes.c_void_p()
    hy = eng.lib.ConvForwardFused(hx, hw, hb, B, C, H, W, OC, k, k, s, p, 0, ctypes.byref(pim))
    assert hy and pim.value, eng.last_error()
    before = eng.lib.GetPoolMemory()
    release(eng, pim.value)
    held = eng.lib.GetPoolMemory() - before
    assert 4 * B * H * W * 36 <= held < 1.2 * 4 * B * H * W * 36, held
    release(eng, hx, hw, hb, hdy, hy)


def _dx_splits(capfd):
    return [int(l.split("splits ")[1].split()[0]) for l in capfd.readouterr().err.splitlines() if "DCE_TUNE_DX parts" in l]


@pytest.mark.parametrize("case", [CASES[14], CASES[15]], ids=str)
def test_few_pixels_split_the_phases(eng, monkeypatch, capfd, case):
    """A stride-2 dX whose phases would leave the chip to a few long chains."""
    monkeypatch.setenv("DCE_TUNE_LOG", "1")
    x, w, dy, y = _inputs(*case)
    s, p, act = case[6:]
    _check(_backward(eng, x, w, dy, y, s, p, act), x, w, dy, y, s, p, act)
    splits = _dx_splits(capfd)
    assert len(splits) == 1 and splits[0] > 1, splits


@pytest.mark.parametrize("splits", [2, 3, 7])
def test_split_phases(eng, monkeypatch, splits):
    """Phases of unequal length (one with fewer steps than splits), odd images, a
    row without pixels; phases without taps are not split."""
    monkeypatch.setenv("DCE_TUNE_DX", f"64,128,16,{splits}")
    for case in CASES[8:12] + [CASES[15]]:
        x, w, dy, y = _inputs(*case)
        s, p, act = case[6:]
        _check(_backward(eng, x, w, dy, y, s, p, act), x, w, dy, y, s, p, act)
