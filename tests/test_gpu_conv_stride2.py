"""Input gradient of stride-2 convolutions on fp32 MFMAs against the float64
oracle: large ones, whose four sub-pixel phases share one launch, and small
ones, which gather.  Images of few rows or columns, phases that no tap reaches,
tile edges, few and many channels, filter re-layouts in flat and blocked order.

Bound per element, from the arithmetic: a sum of n fp32 products rounds at most
n + 2 times, each time by at most 2^-24 of a partial sum that the sum over
|dy||w| bounds."""
import ctypes

import numpy as np
import pytest

from oracle import kernels as K
from tests.helpers import download, he, release, rng, upload

pytestmark = pytest.mark.gpu

CASES = [
    # B, C, H, W, OC, k, p, act
    (2, 16, 14, 15, 24, 3, 1, 1),      # phases of unequal size; OC no multiple of 16 (flat order)
    (1, 8, 1, 9, 16, 3, 1, 0),         # one row: two phases have no pixels
    (3, 12, 9, 1, 32, 3, 1, 1),        # one column
    (2, 24, 13, 12, 48, 1, 0, 0),      # k < s: three phases without taps
    (2, 24, 12, 13, 48, 1, 1, 1),      # the same, padded: another phase has the tap
    (4, 17, 32, 32, 33, 2, 0, 0),      # k == s: one tap a phase
    (2, 300, 9, 8, 20, 3, 1, 0),       # three row tiles
    (1, 31, 40, 37, 200, 5, 2, 1),     # 9, 6, 6 and 4 taps; blocked order with a flat remainder
    (1, 30, 9, 9, 384, 5, 2, 0),       # few pixels, long dot products
    (2, 3, 21, 20, 16, 3, 1, 1),       # stride-phase copy of x, transposed G
    (1, 1, 8, 8, 6, 7, 3, 0),
    (8, 16, 64, 64, 16, 3, 1, 0),      # tiles over several images
    # large enough for the phases (2e8 products of the gather, 8e8 for k = 1)
    (24, 24, 57, 56, 32, 3, 1, 1),     # phases of unequal size, blocked order
    (1, 20, 160, 159, 31, 5, 2, 0),    # 9, 6, 6 and 4 taps; channels that fill no tile
    (40, 33, 41, 40, 20, 3, 0, 1),     # two row tiles, flat order
    (1500, 31, 1, 18, 36, 3, 1, 0),    # one row: two phases have no pixels
    (44, 128, 28, 27, 256, 1, 0, 0),   # three phases without taps
    (6, 3, 160, 160, 96, 7, 3, 0),     # three channels: 16-row tiles
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_dx_phases(eng, case):
    B, C, H, W, OC, k, p, act = case
    r = rng(4100 + B + 3 * C + 5 * H + 7 * W + 11 * OC + 13 * k + p)
    x = r.standard_normal((B, C, H, W)).astype(np.float32)
    w = he(r, (OC, C, k, k), C * k * k)
    OH, OW = K.conv_out_hw(H, W, k, 2, p)
    dy = r.standard_normal((B, OC, OH, OW)).astype(np.float32)
    y = r.standard_normal(dy.shape).astype(np.float32)
    hs = [upload(eng, a) for a in (dy, x, w)]
    hy = upload(eng, y) if act == 1 else None
    ref = K.conv_backward(dy, y, x, w, 2, p, act)[2]
    S = K.conv_backward(np.abs(dy), y, x, np.abs(w), 2, p, act)[2]
    for req in ((1, 1, 1), (1, 0, 0)):
        pdf, pdb, pdx = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        eng.lib.ConvBackwardFused(hs[0], hy, hs[1], hs[2], None, B, C, H, W, OC, k, k, 2, p, act, *req,
                                  ctypes.byref(pdf), ctypes.byref(pdb), ctypes.byref(pdx))
        assert pdx.value, eng.last_error()
        got = download(eng, pdx.value, x.shape)
        release(eng, pdf.value, pdb.value, pdx.value)
        worst = np.max(np.abs(got - ref) - (OC * k * k + 2) * 2.0 ** -24 * S)
        assert worst <= 1e-37, f"{worst:.3e} past the bound"
    release(eng, *hs, hy)


@pytest.mark.parametrize("case,phased", [
    ((16, 100, 63, 64, 8, 2, 0, 0), False),   # dot products of 32: the gather
    ((10, 60, 64, 63, 9, 4, 1, 0), True),     # 192
    ((60, 9, 64, 65, 9, 3, 1, 0), True),      # 108, over few channels
], ids=str)
def test_short_dot_products_gather(eng, monkeypatch, capfd, case, phased):
    """The choice logs one tile for the gather and a second one for the phases."""
    monkeypatch.setenv("DCE_TUNE_LOG", "1")
    test_dx_phases(eng, case)
    lines = [l for l in capfd.readouterr().err.splitlines() if "DCE_TUNE_DX" in l]
    assert len(lines) == 2 * (1 + phased), lines  # two calls
