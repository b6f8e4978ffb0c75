"""GPU: the bf16 GEMM on tiles loaded straight into LDS (gemm_dma.hip) at the edges of its tiles,
stages, K splits and dispatch.  Operands are small integers (exact in bf16) and every sum stays
below 2^24, so any order of fp32 additions gives the exact integer: equality, no tolerance."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as orc
from gpu_helpers import down, empty, say, up
from orator_amd import asr_gemm, asr_ops

pytestmark = pytest.mark.gpu


def _ints(r, shape, lim):
    return r.integers(-lim, lim + 1, shape).astype(np.float32)


# 64 x 64 tiles: one row pair, ragged rows and columns, one K step, fewer steps than stages, uneven K
# splits; 128 x 128 with 4 stages (one tile per CU at most); 128 x 128 with 2; 256 x 192; K not a
# multiple of 64 and N not of 4 (the register-staged kernel) beside them, and the short K with many
# outputs that go to it too; its 128 x 128 tiles last
@pytest.mark.parametrize("M,K,N", [(2, 64, 4), (63, 128, 60), (65, 192, 68), (130, 320, 516),
                                   (3, 2048, 2044), (65, 4160, 1000), (503, 4160, 2048),
                                   (2000, 64, 2044), (1921, 320, 2044), (2000, 64, 4092),
                                   (1921, 192, 4036), (2040, 64, 12284), (1793, 192, 12100),
                                   (130, 72, 516), (130, 64, 514), (2040, 64, 2048),
                                   (1921, 256, 4096), (2040, 72, 4100), (1921, 200, 6004)])
@pytest.mark.parametrize("bias,act", [(False, 0), (True, 2)])
def test_gemm_dma_exact(M, K, N, bias, act):
    r = np.random.default_rng(M + K + N)
    x, w, b = _ints(r, (M, K), 4), _ints(r, (N, K), 4), _ints(r, (N,), 100)
    out = empty((M, N), np.float32)
    say("gemm dma", M, K, N, bias, act)
    asr_gemm.LinearPre(up(orc.to_bf16(x)), up(orc.to_bf16(w)), up(b) if bias else None, out, M, K, N,
                       act)
    ref = x @ w.T + (b if bias else 0)
    np.testing.assert_array_equal(down(out, (M, N)), np.maximum(ref, 0) if act == 2 else ref)


@pytest.mark.parametrize("M,K,I", [(2, 64, 4), (65, 192, 100), (17, 2048, 64), (503, 128, 6140),
                                   (1921, 64, 1024), (2040, 192, 6140), (2040, 192, 6144)])
def test_gemm_dma_swiglu_bits(M, K, I):
    """The same bits as LinearPre, SwiGLU and the cast, on every tile, where K is split and where
    LinearPre takes the register-staged kernel."""
    r = np.random.default_rng(M + K + I)
    x = up(orc.to_bf16(r.standard_normal((M, K)).astype(np.float32)))
    w = up(orc.to_bf16((r.standard_normal((2 * I, K)) * K ** -0.5).astype(np.float32)))
    gu, got = empty((M, 2 * I), np.float32), empty((M, I), np.uint16)
    say("gemm dma swiglu", M, K, I)
    asr_gemm.LinearPreSwiGLU(x, w, got, M, K, I)
    asr_gemm.LinearPre(x, w, None, gu, M, K, 2 * I, 0)
    g = down(gu, (M, 2 * I))
    act, want = empty((M, I), np.float32), empty((M, I), np.uint16)
    asr_ops.SwiGLU(up(np.ascontiguousarray(g[:, :I])), up(np.ascontiguousarray(g[:, I:])), act, M * I)
    asr_ops.F32ToBf16(act, want, M * I)
    np.testing.assert_array_equal(down(got, (M, I), np.uint16), down(want, (M, I), np.uint16))


@pytest.mark.parametrize("M,K,N", [(2, 64, 4), (63, 128, 60), (65, 192, 68), (130, 320, 516),
                                   (3, 2048, 2044), (65, 4160, 1000), (128, 1024, 4096), (129, 1024, 4096),
                                   (1921, 320, 2044), (130, 72, 516)])
def test_linear_rounds_like_the_cast(M, K, N):
    """fp32 activations rounded inside the GEMM: the bits of F32ToBf16 + LinearPre, ties and both
    infinities among the values."""
    r = np.random.default_rng(M + K + N)
    x = r.standard_normal((M, K)).astype(np.float32)
    tie = r.integers(0, K, M)
    x[np.arange(M), tie] = np.float32(1 + 2.0 ** -8) * r.choice([1, -1, 3], M)
    x[0, 0], x[1, K - 1] = np.inf, -np.inf
    w = up(orc.to_bf16((r.standard_normal((N, K)) * K ** -0.5).astype(np.float32)))
    a, b = empty((M, N), np.float32), empty((M, N), np.float32)
    bias = up(r.standard_normal(N).astype(np.float32))
    say("linear f32", M, K, N)
    asr_gemm.Linear(up(x), w, bias, a, M, K, N, 1)
    xb = empty((M, K), np.uint16)
    asr_ops.F32ToBf16(up(x), xb, M * K)
    asr_gemm.LinearPre(xb, w, bias, b, M, K, N, 1)
    np.testing.assert_array_equal(down(a, (M, N)), down(b, (M, N)))


def test_linear_in_place():
    """Output over the input (K = N): through the cast copy, as before."""
    r = np.random.default_rng(9)
    M, K = 70, 256
    x, w = _ints(r, (M, K), 4), _ints(r, (K, K), 4)
    buf = up(x)
    say("linear in place")
    asr_gemm.Linear(buf, up(orc.to_bf16(w)), None, buf, M, K, K, 0)
    np.testing.assert_array_equal(down(buf, (M, K)), x @ w.T)


@pytest.mark.parametrize("M,K", [(2, 64), (70, 256), (200, 2048)])
def test_swiglu_output_over_the_input(M, K):
    """LinearPreSwiGLU in place (I = K, a grid of fewer tiles than CUs): as with an output apart."""
    r = np.random.default_rng(M + K)
    x = orc.to_bf16(r.standard_normal((M, K)).astype(np.float32))
    w = up(orc.to_bf16((r.standard_normal((2 * K, K)) * K ** -0.5).astype(np.float32)))
    want, buf = empty((M, K), np.uint16), up(x)
    say("gemm dma swiglu in place", M, K)
    asr_gemm.LinearPreSwiGLU(buf, w, want, M, K, K)
    asr_gemm.LinearPreSwiGLU(buf, w, buf, M, K, K)
    np.testing.assert_array_equal(down(buf, (M, K), np.uint16), down(want, (M, K), np.uint16))


def test_linear_pre_output_over_the_input():
    """fp32 outputs over the bf16 input (N = K / 2) on a grid whose K is split."""
    r = np.random.default_rng(11)
    M, K = 503, 2048
    x, w = _ints(r, (M, K), 4), _ints(r, (K // 2, K), 4)
    buf = up(orc.to_bf16(x))
    say("gemm dma linear pre in place")
    asr_gemm.LinearPre(buf, up(orc.to_bf16(w)), None, buf, M, K, K // 2, 0)
    np.testing.assert_array_equal(down(buf, (M, K // 2)), x @ w.T)
