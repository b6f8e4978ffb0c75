"""GPU: the fp32 GEMM on split bf16 operands (sgemm.hip) against fp64 at the edges of its tiles,
slices and dispatch, and on values outside bf16's range.

Bound: an MFMA adds 32 products and the accumulator and rounds to fp32, at worst 2 ulp of the
partial sum (<= 2^-22 sum|x w|); six MFMAs per 32-wide slice, then one addition per wave (8 at
most) and the bias.  The split itself is exact but for terms below 2^-26 |x w|.  So
|got - truth| <= (6 ceil(K / 32) + 10) 2^-22 (sum|x w| + |bias|)."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_helpers import down, empty, say, up
from helpers import SplitMix64
from orator_amd import gemm

pytestmark = pytest.mark.gpu


def _run(x, w, bias):
    M, K = x.shape
    N = w.shape[0]
    out = empty((M, N), np.float32)
    say("sgemm split", M, K, N)
    gemm.LaunchSgemm(up(x), up(w), None if bias is None else up(bias), out, M, K, N, 0)
    return down(out, (M, N))


# one K below a slice; K a slice and a part; the limits of the K classes (255 / 256, 1023 / 1024);
# ragged rows and columns of every tile (32 x 32 with 2, 4 and 8 waves, 32 x 64 and 64 x 64 with 4
# and 8); 16-byte and element loads
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (33, 31, 31), (31, 33, 65), (97, 255, 130),
                                   (290, 64, 1100), (33, 256, 33), (300, 256, 1030),
                                   (700, 512, 2050), (2050, 290, 2047), (130, 1023, 70),
                                   (129, 1024, 257), (520, 1056, 514), (1030, 1024, 1028)])
def test_sgemm_split_edges(M, K, N):
    r = SplitMix64(M + 3 * K + 7 * N)
    x, w, b = r.normal((M, K)), r.normal((N, K)), r.normal((N,))
    got = _run(x, w, b)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    bound = (6 * -(-K // 32) + 10) * 2.0 ** -22 * (np.abs(x64) @ np.abs(w64).T + np.abs(b))
    assert np.all(np.abs(got - (x64 @ w64.T + b)) <= bound)


def test_sgemm_split_special_values():
    """Rows with an infinity, a NaN, the largest finite value (which rounds past bf16's range), an
    overflowing sum, and operands so small that their bf16 terms are subnormal, beside ordinary
    rows; what an fp32 chain gives."""
    r = SplitMix64(5)
    M, K, N = 40, 288, 36
    x, w = r.normal((M, K)), r.normal((N, K))
    x[3, 7] = np.inf
    x[5, 100] = np.nan
    x[9, 200] = np.finfo(np.float32).max
    x[11] = np.float32(1e36)
    x[13] *= np.float32(2.0 ** -124)
    x[17] = 0
    w[2] = np.float32(1e2)
    w[4, 7] = 0
    got = _run(x, w, None)
    with np.errstate(all="ignore"):
        ref = np.zeros((M, N), np.float32)
        for k in range(K):
            ref = (x[:, k, None].astype(np.float64) * w[None, :, k] + ref).astype(np.float32)
    for row in (3, 5, 11):
        np.testing.assert_array_equal(np.isnan(got[row]), np.isnan(ref[row]))
        np.testing.assert_array_equal(np.isposinf(got[row]), np.isposinf(ref[row]))
        np.testing.assert_array_equal(np.isneginf(got[row]), np.isneginf(ref[row]))
    assert np.all(got[17] == 0)
    for row in set(range(M)) - {3, 5, 11, 17}:
        mag = np.abs(x[row].astype(np.float64)) @ np.abs(w.astype(np.float64)).T
        ok = np.isfinite(ref[row])
        np.testing.assert_array_equal(np.isfinite(got[row]), ok)
        # either side within K roundings of the fp64 sum (and of fp32's subnormal spacing)
        err = np.abs(got[row][ok].astype(np.float64) - (x[row].astype(np.float64) @ w.astype(np.float64).T)[ok])
        assert np.all(err <= K * (2.0 ** -23 * mag[ok] + 2.0 ** -149))


def test_sgemm_split_rows_past_32_bit_offsets():
    """K >= 2^24: 64 rows no longer fit 32-bit byte offsets; integer operands, exact sum."""
    K = (1 << 24) + 5
    r = np.random.default_rng(3)
    x = r.integers(-1, 2, (1, K)).astype(np.float32)
    w = r.integers(-1, 2, (2, K)).astype(np.float32)
    got = _run(x, w, None)
    np.testing.assert_array_equal(got, (x.astype(np.int64) @ w.astype(np.int64).T).astype(np.float32))
