"""GPU: the fp32 GEMM on split bf16 operands (sgemm.hip) against fp64 at the edges of its tiles,
slices and dispatch, and on values outside bf16's range.

Bound: an MFMA adds 32 products and the accumulator and rounds to fp32, at worst 2 ulp of the
partial sum (<= 2^-22 sum|x w|); six MFMAs per 32-wide slice, then one addition per wave (8 at
most) and the bias.  The split itself is exact but for products of terms below 2^-24 |x w|.  So
|got - truth| <= (6 ceil(K / 32) + 10) 2^-22 (sum|x w| + |bias|)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gpu_helpers import down, empty, say, up
from helpers import SplitMix64
from orator_amd import gemm
from orator_amd.runtime import Stream, synchronize

pytestmark = pytest.mark.gpu


def _run(x, w, bias):
    M, K = x.shape
    N = w.shape[0]
    out = empty((M, N), np.float32)
    say("sgemm split", M, K, N)
    gemm.LaunchSgemm(up(x), up(w), None if bias is None else up(bias), out, M, K, N, 0)
    return down(out, (M, N))


def _rel(got, ref):
    return np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref)


# one K below a slice; K a slice and a part; the limits of the K classes (255 / 256, 1023 / 1024);
# ragged rows and columns of every tile (32 x 32 with 2, 4 and 8 waves, 32 x 64 and 64 x 64 with 4
# and 8); 16-byte and element loads; the one-wave and two-wave 32 x 64 tiles of K <= 64
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (33, 31, 31), (31, 33, 65), (97, 255, 130),
                                   (290, 64, 1100), (33, 256, 33), (300, 256, 1030),
                                   (700, 512, 2050), (2050, 290, 2047), (130, 1023, 70),
                                   (129, 1024, 257), (520, 1056, 514), (1030, 1024, 1028),
                                   (2049, 31, 1030), (1030, 32, 2050), (2100, 64, 1030),
                                   (2049, 40, 2050), (4100, 64, 1028)])
def test_sgemm_split_edges(M, K, N):
    r = SplitMix64(M + 3 * K + 7 * N)
    x, w, b = r.normal((M, K)), r.normal((N, K)), r.normal((N,))
    got = _run(x, w, b)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    bound = (6 * -(-K // 32) + 10) * 2.0 ** -22 * (np.abs(x64) @ np.abs(w64).T + np.abs(b))
    ref = x64 @ w64.T + b
    assert np.all(np.abs(got - ref) <= bound)
    # the sharper check: without the third terms or the corrections the error is 4e-6 and more
    # (measured with all six products: 2.4e-7 at most)
    assert _rel(got, ref) <= 4e-7


# K split over workgroups: two parts, as many as one round takes, an uneven last one, element loads,
# a tile of one row.  33 outputs at least: the 2-norm of the errors over that of the sums is then
# near their ratio of standard deviations, where a single sum may cancel (one of 70000 products
# that came to 0.62 of its standard deviation was 4.02e-7 off)
@pytest.mark.parametrize("M,K,N", [(126, 2048, 512), (3, 4100, 70), (1, 16384, 40), (70, 3001, 33),
                                   (1, 70000, 33), (250, 2080, 500)])
@pytest.mark.parametrize("act", [0, 2])
def test_sgemm_long_k_on_a_short_grid(M, K, N, act):
    """Error against fp64 as small as the parts of K keep it: 2.4e-7 measured at most (7.3e-7 with
    16384 in one workgroup's eight parts)."""
    r = SplitMix64(M + K + N)
    x, w, b = r.normal((M, K)), r.normal((N, K)), r.normal((N,))
    out = empty((M, N), np.float32)
    say("sgemm long k", M, K, N, act)
    gemm.LaunchSgemm(up(x), up(w), up(b), out, M, K, N, act)
    ref = x.astype(np.float64) @ w.astype(np.float64).T + b
    assert _rel(down(out, (M, N)), np.maximum(ref, 0) if act == 2 else ref) <= 4e-7


def test_sgemm_long_k_under_capture():
    """Captured on a stream without a workspace block: the unsplit form, since nothing can be
    allocated there.  With one: the eager result's bits on every replay."""
    hip = C.CDLL("libamdhip64.so")

    def ok(rc):
        assert rc == 0, rc

    M, K, N = 40, 4096, 96
    r = SplitMix64(4)
    x, w = r.normal((M, K)), r.normal((N, K))
    dx, dw, out = up(x), up(w), empty((M, N), np.float32)
    ref = x.astype(np.float64) @ w.astype(np.float64).T

    def replays(stream):
        graph, run = C.c_void_p(), C.c_void_p()
        h = C.c_void_p(stream.handle)
        ok(hip.hipStreamBeginCapture(h, 0))
        gemm.LaunchSgemm(dx, dw, None, out, M, K, N, 0, stream)
        ok(hip.hipStreamEndCapture(h, C.byref(graph)))
        ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
        got = []
        for _ in range(3):
            out.upload(np.full((M, N), np.nan, np.float32))
            synchronize()
            ok(hip.hipGraphLaunch(run, h))
            got.append(down(out, (M, N)))
        ok(hip.hipGraphExecDestroy(run))
        ok(hip.hipGraphDestroy(graph))
        return got

    say("sgemm long k captured")
    stream = Stream()
    for got in replays(stream):
        assert _rel(got, ref) <= 6e-7  # 3.5e-7 measured unsplit
    gemm.LaunchSgemm(dx, dw, None, out, M, K, N, 0, stream)
    eager = down(out, (M, N))
    for got in replays(stream):
        np.testing.assert_array_equal(got, eager)


@pytest.mark.parametrize("M,K,batch", [(126, 512, 1), (1000, 512, 1), (700, 70, 1), (40, 2048, 1),
                                       (60, 512, 3)])
def test_sgemm_output_over_its_operand(M, K, batch):
    """Output over the input, and over the weight (N = K, M = N): as with an output of its own."""
    r = SplitMix64(M + K)
    x, w = r.normal((batch, M, K)), r.normal((batch, K, K))
    say("sgemm in place", M, K, batch)
    for over in ("in", "weight"):
        m = M if over == "in" else K
        xs = x if over == "in" else r.normal((batch, K, K))
        dx, dw, want = up(xs), up(w), empty((batch, m, K), np.float32)
        gemm.LaunchSgemmBatched(dx, dw, want, m, K, K, 2, batch, m * K, K * K, m * K)
        out = dx if over == "in" else dw
        gemm.LaunchSgemmBatched(dx, dw, out, m, K, K, 2, batch, m * K, K * K, m * K)
        np.testing.assert_array_equal(down(out, (batch, m, K)), down(want, (batch, m, K)))


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


# x and w scaled by powers of two whose products are ordinary numbers: below 2^-103 an operand's
# third bf16 term falls between bf16's subnormals, below 2^-134 all three are zero
@pytest.mark.parametrize("ex,ew", [(-102, 40), (-110, 60), (-118, 40), (-125, 60), (-135, 60),
                                   (-140, 100), (-147, 120), (60, -135), (100, -140), (-118, 0)])
@pytest.mark.parametrize("M,K,N", [(33, 512, 70), (40, 290, 65), (3, 64, 5), (70, 1024, 2050)])
def test_sgemm_operands_outside_the_terms_range(M, K, N, ex, ew):
    """As close to fp64 as the fp32 MFMAs that form these results (2.9e-7 on ordinary operands);
    operands are exact inputs, so only the products and sums round.  Half of x's rows and a third
    of its columns are zero: a zero result must not pass for an exact one."""
    r = SplitMix64(M + K + N)
    x = np.ldexp(r.normal((M, K)), ex).astype(np.float32)
    w = np.ldexp(r.normal((N, K)), ew).astype(np.float32)
    x[1::2] = 0
    x[:, ::3] = 0
    got = _run(x, w, None)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    assert np.all(got[1::2] == 0)
    assert _rel(got, ref) <= 4e-7


def test_sgemm_tiny_operand_beside_ordinary_ones():
    """One tiny and one huge operand in a row of ordinary ones, their product the largest term."""
    r = SplitMix64(8)
    M, K, N = 35, 320, 37
    x, w = r.normal((M, K)), r.normal((N, K))
    x[:, 77] = np.float32(1.2345678 * 2.0 ** -120)
    w[:, 77] = np.float32(1.7 * 2.0 ** 126)
    got = _run(x, w, None)
    assert _rel(got, x.astype(np.float64) @ w.astype(np.float64).T) <= 4e-7


def test_sgemm_finite_near_the_largest_number():
    """Operands whose first terms' product overflows although the product does not."""
    x = np.full((2, 1), np.float32(2.0 ** 64 * (1 - 2.0 ** -20)))
    got = _run(x, x, None)
    np.testing.assert_array_equal(got, x * x.T)
    assert np.all(np.isfinite(got))


def test_sgemm_split_rows_past_32_bit_offsets():
    """K >= 2^24: 64 rows no longer fit 32-bit byte offsets; integer operands, exact sum.  And all
    threes: a single chain rounds each addition above 2^24, parts of K stay exact."""
    K = (1 << 24) + 5
    got = _run(np.full((1, K), 3, np.float32), np.ones((1, K), np.float32), None)
    assert abs(float(got[0, 0]) - 3 * K) <= 2.0 ** -22 * 3 * K
    r = np.random.default_rng(3)
    x = r.integers(-1, 2, (1, K)).astype(np.float32)
    w = r.integers(-1, 2, (2, K)).astype(np.float32)
    got = _run(x, w, None)
    np.testing.assert_array_equal(got, (x.astype(np.int64) @ w.astype(np.int64).T).astype(np.float32))
