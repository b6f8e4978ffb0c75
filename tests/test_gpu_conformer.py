"""GPU parity: batched SGEMM (gemm.cuh) and the Conformer rel-pos attention core against the
oracle.  fp32 paths: max |g - r| / max(|r|, floor) <= 1e-4."""
from __future__ import annotations

import math

import numpy as np
import pytest

import fp16_model
import oracle_lib as orc
import truth64 as t64
from gpu_helpers import down, empty, say, up
from helpers import SplitMix64, check_fp32, rel_err
from orator_amd import conformer_attn as ca
from orator_amd import gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,inner,cols,batch", [(13, 64, 13, 8), (14, 64, 14, 8)])
def test_sgemm_batched_reference_test(rows, inner, cols, batch):
    """test/unit/model/test_gemm_batched.cu:12-61: index%17/17 and index%13/13 inputs, f64
    brute force, max-abs 1e-4."""
    a = (np.arange(batch * rows * inner) % 17 / 17.0).astype(np.float32).reshape(batch, rows, inner)
    w = (np.arange(batch * cols * inner) % 13 / 13.0).astype(np.float32).reshape(batch, cols, inner)
    dout = empty((batch, rows, cols), np.float32)
    say("sgemm_batched ref", rows, cols)
    gemm.LaunchSgemmBatched(up(a), up(w), dout, rows, inner, cols, 0, batch, rows * inner,
                            cols * inner, rows * cols)
    ref = np.einsum("bmk,bnk->bmn", a.astype(np.float64), w.astype(np.float64))
    assert np.max(np.abs(down(dout, (batch, rows, cols)) - ref)) < 1e-4


@pytest.mark.parametrize("M,K,N,act", [(7, 13, 9, 0), (717, 512, 512, 0), (65, 64, 130, 1),
                                       (100, 33, 70, 2), (5, 2048, 3, 3), (1433, 512, 512, 0),
                                       (717, 512, 2048, 1), (2048, 512, 2048, 0),
                                       (717, 100, 1536, 0), (701, 512, 1530, 2)])
def test_sgemm_bias_act_vs_oracle(M, K, N, act):
    """Every activation over the kernel's classes: K of one slice and a few (13, 33, 64, 100) and of
    many (512) on 32 x 32, 32 x 64 and 64 x 64 tiles, K split over workgroups (5 x 2048 -> 3),
    element loads (K = 13, 33, 100), ragged rows and columns (701 x 512 -> 1530)."""
    r = SplitMix64(M * 3 + K + N)
    a, w, bias = r.normal((M, K)), r.normal((N, K), 1.0 / math.sqrt(K)), r.normal((N,))
    dout = empty((M, N), np.float32)
    say("sgemm", M, K, N, act)
    gemm.LaunchSgemm(up(a), up(w), up(bias), dout, M, K, N, act)
    got = down(dout, (M, N))
    pre = a.astype(np.float64) @ w.astype(np.float64).T + bias
    truth = {0: pre, 1: pre / (1 + np.exp(-pre)), 2: np.maximum(pre, 0), 3: 1 / (1 + np.exp(-pre))}[act]
    assert np.max(np.abs(got - truth)) < 1e-4  # the reference's SGEMM gate
    assert rel_err(got, orc.sgemm(a, w, bias, act), 1.0) <= 1e-5  # unit-scale outputs


def _relpos_inputs(r, T, H, Dk):
    return (r.normal((T, H, Dk)), r.normal((T, H, Dk)), r.normal((T, H, Dk)),
            r.normal((2 * T - 1, H, Dk)), r.normal((H, Dk), 0.3), r.normal((H, Dk), 0.3))


@pytest.mark.parametrize("T,valid", [(1, 1), (2, 2), (3, 2), (126, 125), (717, 717), (400, 333),
                                     (5, 0), (70, 0), (1500, 1400)])
def test_relpos_fp32_vs_oracle(T, valid):
    """Config-4 shape (T = 717: 340 chunk + 1 right context + 188 FIFO + 188 speaker cache),
    the NeMo verification shape (T = 126, valid = 125, tools/verify/cc/verify_conformer.cc),
    tiny T where the rel-shift wraps, and valid = 0 (every key masked with the reference's finite
    -1e30: the softmax averages V over all T keys)."""
    H, Dk = 8, 64
    r = SplitMix64(T * 11 + valid)
    q, k, v, p, u, vb = _relpos_inputs(r, T, H, Dk)
    scale = 1.0 / math.sqrt(Dk)
    ref = orc.relpos_attention(q, k, v, p, u, vb, valid, scale)
    dout = empty(q.shape, np.float32)
    say("relpos fp32", T, valid)
    ca.RelPosAttention(up(q), up(k), up(v), up(p), up(u), up(vb), dout, T, H, Dk, valid, scale)
    # At the 1e-3 floor the device is held to 2x the oracle's distance from the fp64 value (the
    # default): the row softmax calls HIP's expf (OCML's exp, documented at <= 1 ulp) where the
    # oracle calls the C library's expf (<= 0.5 ulp in round-to-nearest), so each weight's
    # exponential error may be twice the oracle's.  The three score / context products add
    # nothing to that: 32 products to a rounding against the oracle's serial chain (relative
    # 2-norm at T = 717, whole core: device 2.3e-7, oracle 7.4e-7).
    check_fp32(down(dout, q.shape), ref, 1e-4,
               truth=orc.relpos_attention_f64(q, k, v, p, u, vb, valid, scale) if valid > 0 else None)


def _to_f16_bits(x):
    return np.ascontiguousarray(x, np.float32).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("T,valid,in_f16", [(717, 717, True), (717, 700, False), (126, 125, True),
                                             (1, 1, True), (33, 20, True), (300, 300, False),
                                             (40, 0, True), (70, 0, False), (1500, 1500, True)])
def test_relpos_fused_vs_oracle(T, valid, in_f16):
    """Fused fp16-MFMA rel-pos attention (fp16 inputs N(0,1)).  fp16
    operands with fp32 accumulation: max abs error <= 2e-2 on unit-scale outputs (the
    bar of the 16-bit modes), judged against the oracle run on the fp16-rounded inputs; and
    within 2x (+2e-5) of the error the kernel's own fp16 roundings predict (tests/fp16_model.py,
    computed before the device runs: ~6e-4 at T = 717)."""
    H, Dk = 8, 64
    r = SplitMix64(T * 13 + valid)
    q, k, v, p, u, vb = _relpos_inputs(r, T, H, Dk)
    q, k, v, p = (x.astype(np.float16).astype(np.float32) for x in (q, k, v, p))
    scale = 1.0 / math.sqrt(Dk)
    ref = orc.relpos_attention(q, k, v, p, u, vb, valid, scale)
    predicted = np.max(np.abs(fp16_model.relpos_attention_f16(q, k, v, p, u, vb, valid, scale)
                              - ref))
    dout = empty(q.shape, np.float32)
    say("relpos fused", T, valid, in_f16)
    ins = [up(_to_f16_bits(x)) if in_f16 else up(x) for x in (q, k, v, p)]
    ca.RelPosAttentionFast(*ins, up(u), up(vb), dout, T, H, Dk, valid, scale, in_f16=in_f16)
    got = down(dout, q.shape)
    err = np.max(np.abs(got - ref))
    print(f"T={T} valid={valid}: max abs {err:.2e}, fp16 model predicts {predicted:.2e}")
    assert err <= 2e-2
    assert err <= 2.0 * predicted + 2e-5


@pytest.mark.parametrize("T,valid", [(717, 529), (33, 20), (70, 0), (1, 1)])
def test_relpos_fused_mixed_inputs_match_fp32(T, valid):
    """in_f16 = 2 (q fp32; k, v, p fp16 bits, what the Conformer layer's fused mode feeds) gives
    bit for bit the in_f16 = 0 result on the fp32 rows those fp16 values round from: both round
    k, v, p to nearest even once and form q + u, q + v in fp32."""
    H, Dk = 8, 64
    r = SplitMix64(T * 29 + valid)
    q, k, v, p, u, vb = _relpos_inputs(r, T, H, Dk)
    scale = 1.0 / math.sqrt(Dk)
    say("relpos fused mixed", T, valid)
    d32, dmix = empty(q.shape, np.float32), empty(q.shape, np.float32)
    ca.RelPosAttentionFast(up(q), up(k), up(v), up(p), up(u), up(vb), d32, T, H, Dk, valid,
                           scale, in_f16=0)
    ca.RelPosAttentionFast(up(q), *(up(_to_f16_bits(x)) for x in (k, v, p)), up(u), up(vb),
                           dmix, T, H, Dk, valid, scale, in_f16=2)
    a, b = down(d32, q.shape), down(dmix, q.shape)
    assert np.isfinite(a).all()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
