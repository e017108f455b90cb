"""A^T B over at most 256 rows (a linear layer's filter gradient) around the rule
that takes 64 x 128 tiles when the last batch of 128 x 128 ones is not full,
against the float64 oracle.  Bound: K + 2 roundings of a partial sum that S, the
sum over magnitudes, bounds."""
import numpy as np
import pytest

from oracle import kernels as K
from tests.helpers import download, release, rng, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,Kd,N", [
    (2177, 128, 2050),   # 64-row tiles: a last row tile of one row, ragged columns
    (2100, 1, 2100),     # one product per sum
    (2500, 37, 4500),    # K past a step
    (2177, 256, 2048),   # the longest of the rule
    (2177, 257, 2048),   # one past it: 128 x 128
    (4096, 16, 4096),    # full batches: 128 x 128
])
def test_at_b_tiles(eng, M, Kd, N):
    r = rng(M + Kd + N)
    a = r.standard_normal((Kd, M), dtype=np.float32)
    b = r.standard_normal((Kd, N), dtype=np.float32)
    ha, hb = upload(eng, a), upload(eng, b)
    hc = eng.lib.MatMulAlloc(ha, hb, M, Kd, N, 1)
    assert hc, eng.last_error()
    c = download(eng, hc, (M, N))
    release(eng, ha, hb, hc)
    S = K.matmul(np.abs(a), np.abs(b), M, Kd, N, 1)
    assert np.all(np.abs(c - K.matmul(a, b, M, Kd, N, 1)) <= (Kd + 2) * 2.0 ** -24 * S)
