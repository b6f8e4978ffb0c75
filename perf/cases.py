"""The work a user of this library has it do, as cases that can be timed and checked.

Sizes are the Qwen3-ASR text decoder's (hidden 2048, 16 query / 8 KV heads of 128, SwiGLU 6144,
vocabulary 151936, 28 layers), the audio tower's attention (16 heads of 64) and the Sortformer's
(d_model 512, FFN 2048, 8 heads; its decoder 8 heads of 24), as the tests and the benchmark use
them, over the lengths a speech program meets: prompts of tens to two thousand tokens, contexts
to 4096, one to sixteen streams, encoder windows from under a second to a full minute."""
from __future__ import annotations

import math

import numpy as np
import torch

from orator_amd import (asr_gemm, audio_attn, conformer_attn, decoder, decoder_attn,
                        sortformer_attn)

DEV = "cuda"
HQ, HKV, DH, PAGE = 16, 8, 128, 16
HIDDEN, INTER = 2048, 6144
THETA, EPS = 1e6, 1e-6
SCALE = 1.0 / math.sqrt(DH)
# (K, N) of the linear layers: the decoder's q, k|v or o, its fused qkv, its down projection, and
# the audio tower's FFN pair (d_model 1024)
LINEARS = ((2048, 2048), (2048, 4096), (6144, 2048), (1024, 4096), (4096, 1024))


def listed():
    return [
        # one layer's attention in one decode step of a single transcription: norm, RoPE, cache
        # append and attention; the smallest call, made 28 times per token
        {"name": "decode_one", "kind": "decode", "B": 1, "L": 1300},
        # the same for a few live streams of different lengths over a paged cache
        {"name": "decode_few", "kind": "decode_paged", "B": 6, "L": 1100},
        # a server's full batch over long contexts: the HBM-bound end
        {"name": "decode_many", "kind": "decode_paged", "B": 16, "L": 4096},
        # prompt attention as the decoder runs it (fp32 mode): 30 s of audio and its prompt
        {"name": "prefill_503", "kind": "prefill", "T": 503, "pos0": 0, "mode": 0, "paged": False},
        # prompt attention of the longest prompt the decoder's default context takes, bf16 mode
        {"name": "prefill_2048", "kind": "prefill", "T": 2048, "pos0": 0, "mode": 1,
         "paged": False},
        # an audio tower FFN projection over one 30 s clip: bias and GELU, fp32 activations
        {"name": "linear_390", "kind": "linear", "M": 390, "K": 1024, "N": 4096, "act": 1,
         "bias": True},
        # the decoder's MLP over the longest prompt: gate|up + SwiGLU, then down
        {"name": "mlp_2048", "kind": "mlp", "M": 2048},
        # a Sortformer encoder layer over a streaming chunk with its caches, fused fp16 attention
        {"name": "conformer_717", "kind": "conformer", "T": 717, "valid": 717, "mode": 1},
        # the same layer over a short padded chunk, everything fp32
        {"name": "conformer_126", "kind": "conformer", "T": 126, "valid": 125, "mode": 0},
        # the audio tower's windowed attention over a 30 s clip
        {"name": "window_390", "kind": "window", "N": 390, "seg": 104},
        # the Sortformer decoder's masked self-attention
        {"name": "mha_717", "kind": "mha", "T": 717, "valid": 700},
        # a whole transcription: the prompt's prefill, then greedy tokens by graph replay
        {"name": "transcribe_503", "kind": "transcribe", "T": 503, "new": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode_paged", "prefill", "prefill", "linear", "mlp",
                       "conformer", "conformer", "window", "mha", "transcribe"))
    if kind == "decode":
        return {"kind": kind, "B": 1, "L": _log(rng, 64, 4096)}
    if kind == "decode_paged":
        return {"kind": kind, "B": rng.randint(2, 16), "L": _log(rng, 128, 4096)}
    if kind == "prefill":
        return {"kind": kind, "T": _log(rng, 24, 2048), "pos0": rng.choice((0, 0, rng.randint(1, 2000))),
                "mode": rng.randint(0, 1), "paged": rng.random() < 0.25}
    if kind == "linear":
        K, N = rng.choice(LINEARS)
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": K, "N": N, "act": rng.randint(0, 1),
                "bias": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 16, 2048)}
    if kind == "conformer":
        T = _log(rng, 16, 1000)
        return {"kind": kind, "T": T, "valid": max(1, T - rng.randint(0, T // 4)),
                "mode": rng.randint(0, 1)}
    if kind == "window":
        return {"kind": kind, "N": _log(rng, 13, 1560), "seg": rng.choice((52, 104, 130))}
    if kind == "mha":
        T = _log(rng, 16, 1000)
        return {"kind": kind, "T": T, "valid": max(1, T - rng.randint(0, T // 3))}
    return {"kind": kind, "T": _log(rng, 32, 503), "new": rng.randint(6, 24)}


# ------------------------------------------------------------------------- inputs ----
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) + 1)


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    x = torch.randn(shape, generator=g, device=DEV, dtype=dtype)
    return x.mul_(std).add_(mean) if (std != 1.0 or mean != 0.0) else x


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _p(t):
    return None if t is None else t.data_ptr()


def _lengths(case, g):
    """Keys each stream attends in this step (the appended one included)."""
    if case["B"] == 1:
        return [case["L"] + 1]
    lo = max(1, case["L"] // 2)
    r = torch.randint(lo, case["L"] + 1, (case["B"],), generator=g, device=DEV).tolist()
    r[0] = case["L"]
    return [n + 1 for n in r]


def _decode_inputs(case, seed):
    g = _gen(seed)
    B = case["B"]
    lens = _lengths(case, g)
    cap = 2048 if case["L"] < 2048 else 4224
    st = {"q": _randn(g, B, HQ, DH, std=2.0), "k": _randn(g, B, HKV, DH, std=2.0),
          "v": _randn(g, B, HKV, DH), "qn": _randn(g, DH, std=0.1, mean=1.0),
          "kn": _randn(g, DH, std=0.1, mean=1.0), "pos": _ints([n - 1 for n in lens]),
          "lens": lens, "B": B, "out": torch.empty(B, HQ, DH, device=DEV)}
    if case["kind"] == "decode_paged":
        cap = -(-(case["L"] + 64) // PAGE) * PAGE  # room for the tokens still to come
        pages = cap // PAGE
        order = torch.randperm(B * pages, generator=g, device=DEV)
        st["table"] = order.reshape(B, pages).to(torch.int32)
        st["pages"] = pages
        rows = B * cap
    else:
        rows = cap
    st["kc"] = _randn(g, rows, HKV, DH, dtype=torch.bfloat16)
    st["vc"] = _randn(g, rows, HKV, DH, dtype=torch.bfloat16)
    st["cap"] = cap
    return st


def _prefill_inputs(case, seed):
    g = _gen(seed)
    T, pos0 = case["T"], case["pos0"]
    cap = max(2048, -(-(T + pos0) // PAGE) * PAGE)
    st = {"q": _randn(g, T, HQ, DH), "out": torch.empty(T, HQ, DH, device=DEV),
          "pos0": _ints([pos0]), "cap": cap, "table": None, "pages": 0,
          "kc": _randn(g, cap, HKV, DH, dtype=torch.bfloat16),
          "vc": _randn(g, cap, HKV, DH, dtype=torch.bfloat16)}
    if case["paged"]:
        st["pages"] = cap // PAGE
        st["table"] = torch.randperm(st["pages"], generator=g, device=DEV).to(torch.int32)
    return st


def _linear_inputs(case, seed):
    g = _gen(seed)
    M, K, N = case["M"], case["K"], case["N"]
    return {"x": _randn(g, M, K), "W": _randn(g, N, K, std=K ** -0.5, dtype=torch.bfloat16),
            "b": _randn(g, N, std=0.1) if case["bias"] else None,
            "out": torch.empty(M, N, device=DEV), "case": dict(case)}


def _mlp_inputs(case, seed):
    g = _gen(seed)
    M = case["M"]
    return {"x": _randn(g, M, HIDDEN, dtype=torch.bfloat16), "M": M,
            "gu": _randn(g, 2 * INTER, HIDDEN, std=HIDDEN ** -0.5, dtype=torch.bfloat16),
            "dn": _randn(g, HIDDEN, INTER, std=INTER ** -0.5, dtype=torch.bfloat16),
            "act": torch.empty(M, INTER, dtype=torch.bfloat16, device=DEV),
            "out": torch.empty(M, HIDDEN, device=DEV)}


D_MODEL, N_HEADS, D_FF, CONV = 512, 8, 2048, 9


def _pos_rows(T):
    """Sinusoids of the relative positions T - 1 .. -(T - 1): [2T - 1, D_MODEL]."""
    pos = np.arange(T - 1, -T, -1, dtype=np.float64)[:, None]
    div = np.exp(np.arange(0, D_MODEL, 2) * (-math.log(10000.0) / D_MODEL))
    pe = np.empty((2 * T - 1, D_MODEL), np.float32)
    pe[:, 0::2], pe[:, 1::2] = np.sin(pos * div), np.cos(pos * div)
    return torch.from_numpy(pe).to(DEV)


def _conformer_weights(g):
    D, F, w = D_MODEL, D_FF, {}
    lin = lambda n, k: _randn(g, n, k, std=k ** -0.5)  # noqa: E731
    vec = lambda n: _randn(g, n, std=0.1)  # noqa: E731
    for p in ("ff1", "ff2"):
        w[f"{p}_w1"], w[f"{p}_b1"], w[f"{p}_w2"], w[f"{p}_b2"] = lin(F, D), vec(F), lin(D, F), vec(D)
    for p in ("ff1", "att", "conv", "ff2", "out"):
        w[f"norm_{p}_w"], w[f"norm_{p}_b"] = _randn(g, D, std=0.1, mean=1.0), vec(D)
    for p in ("q", "k", "v", "out", "pw2"):
        w[f"{p}_w"], w[f"{p}_b"] = lin(D, D), vec(D)
    w["pos_w"], w["pos_bias_u"], w["pos_bias_v"] = lin(D, D), vec(D), vec(D)
    w["pw1_w"], w["pw1_b"] = lin(2 * D, D), vec(2 * D)
    w["dw_w"], w["dw_b"] = _randn(g, D, CONV, std=CONV ** -0.5), vec(D)
    w["bn_w"], w["bn_b"], w["bn_mean"] = _randn(g, D, std=0.1, mean=1.0), vec(D), vec(D)
    w["bn_var"] = 0.5 + torch.rand(D, generator=g, device=DEV)
    return w


def _conformer_inputs(case, seed):
    g = _gen(seed)
    w = _conformer_weights(g)
    return {"w": w, "x0": _randn(g, case["T"], D_MODEL), "pe": _pos_rows(case["T"])}


def _segments(case):
    N, seg = case["N"], case["seg"]
    start = [i // seg * seg for i in range(N)]
    return start, [min(s + seg, N) for s in start]


def _small_attn_inputs(case, seed):
    g = _gen(seed)
    n, h, d = (case["N"], 16, 64) if case["kind"] == "window" else (case["T"], 8, 24)
    st = {x: _randn(g, n, h, d) for x in "qkv"}
    st["out"] = torch.empty(n, h, d, device=DEV)
    st["case"] = dict(case)
    if case["kind"] == "window":
        a, b = _segments(case)
        st["start"], st["end"] = _ints(a), _ints(b)
    return st


HEAD_SHIFT = 4099


def _transcribe_state(case, seed):
    """The 28-layer decoder on random weights.  The head is the embedding table shifted by
    HEAD_SHIFT rows, so token t is followed by t + HEAD_SHIFT with a clear margin, as a trained
    model's confident continuations are."""
    g = _gen(seed)
    cfg = decoder.AsrTextConfig()
    V, qd, kvd = cfg.vocab_size, HQ * DH, HKV * DH
    bf = lambda n, k, s: _randn(g, n, k, std=s, dtype=torch.bfloat16)  # noqa: E731
    gain = lambda n: _randn(g, n, std=0.1, mean=1.0)  # noqa: E731
    embed = bf(V, HIDDEN, 1.0)
    head = torch.roll(embed, HEAD_SHIFT, 0)
    layers = [dict(in_ln=gain(HIDDEN), q_norm=gain(DH), k_norm=gain(DH), post_ln=gain(HIDDEN),
                   qkv_w=bf(qd + 2 * kvd, HIDDEN, 0.015), o_w=bf(HIDDEN, qd, 0.015),
                   gateup_w=bf(2 * INTER, HIDDEN, 0.015), down_w=bf(HIDDEN, INTER, 0.015))
              for _ in range(cfg.num_layers)]
    norm = gain(HIDDEN)
    x = _randn(g, case["T"], HIDDEN)
    x[-1] = embed[1 + int(seed) % 997].float()
    keep = (embed, head, norm, layers)
    addr = [{k: v.data_ptr() for k, v in L.items()} for L in layers]
    torch.cuda.synchronize()
    dec = decoder.AsrTextDecoder(cfg, embed.data_ptr(), norm.data_ptr(), head.data_ptr(), addr)
    return {"dec": dec, "keep": keep, "x": x, "T": case["T"], "new": case["new"]}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "decode_paged"):
        st = _decode_inputs(case, seed)
        st["rope"] = torch.empty(st["cap"], DH // 2, 2, device=DEV)
        decoder_attn.RopeTable(_p(st["rope"]), st["cap"], THETA, _stream())
    elif kind == "prefill":
        st = _prefill_inputs(case, seed)
        st["case"] = dict(case)
    elif kind == "linear":
        st = _linear_inputs(case, seed)
    elif kind == "mlp":
        st = _mlp_inputs(case, seed)
    elif kind == "conformer":
        st = _conformer_inputs(case, seed)
        st["x"], st["case"] = st["x0"].clone(), dict(case)
        st["layer"] = conformer_attn.ConformerLayer({k: _p(v) for k, v in st["w"].items()},
                                                    D_MODEL, N_HEADS, D_FF, CONV)
    elif kind in ("window", "mha"):
        st = _small_attn_inputs(case, seed)
    else:
        st = _transcribe_state(case, seed)
    st["kind"] = kind
    return st


# ----------------------------------------------------------------------- one pass ----
def run(st):
    kind, s = st["kind"], _stream()
    if kind == "decode":
        decoder_attn.GqaDecodeAttnAppendQkNorm(
            _p(st["q"]), _p(st["k"]), _p(st["v"]), _p(st["kc"]), _p(st["vc"]), _p(st["out"]), HQ,
            HKV, DH, _p(st["pos"]), st["cap"], SCALE, _p(st["qn"]), _p(st["kn"]), EPS,
            _p(st["rope"]), st["cap"], s)
        return {"out": st["out"], "kc": st["kc"], "vc": st["vc"]}
    if kind == "decode_paged":
        decoder_attn.GqaDecodeAttnAppendQkNormPaged(
            _p(st["q"]), _p(st["k"]), _p(st["v"]), _p(st["kc"]), _p(st["vc"]), _p(st["table"]),
            st["pages"], PAGE, st["B"] * st["pages"], _p(st["pos"]), _p(st["out"]), st["B"], HQ,
            HKV, DH, SCALE, _p(st["qn"]), _p(st["kn"]), EPS, _p(st["rope"]), st["cap"], s)
        return {"out": st["out"], "kc": st["kc"], "vc": st["vc"]}
    if kind == "prefill":
        decoder_attn.GqaCacheAttnEx(
            _p(st["q"]), None, _p(st["kc"]), _p(st["vc"]), _p(st["table"]), st["pages"],
            PAGE if st["pages"] else 0, _p(st["out"]), st["case"]["T"], HQ, HKV, DH,
            _p(st["pos0"]), st["cap"], SCALE, st["case"]["mode"], s)
        return st["out"]
    if kind == "linear":
        c = st["case"]
        asr_gemm.Linear(_p(st["x"]), _p(st["W"]), _p(st["b"]), _p(st["out"]), c["M"], c["K"],
                        c["N"], c["act"], s)
        return st["out"]
    if kind == "mlp":
        asr_gemm.LinearPreSwiGLU(_p(st["x"]), _p(st["gu"]), _p(st["act"]), st["M"], HIDDEN, INTER, s)
        asr_gemm.LinearPre(_p(st["act"]), _p(st["dn"]), None, _p(st["out"]), st["M"], INTER,
                           HIDDEN, 0, s)
        return {"act": st["act"], "out": st["out"]}
    if kind == "conformer":
        c = st["case"]
        st["x"].copy_(st["x0"])  # the layer works in place
        st["layer"].Forward(_p(st["x"]), c["T"], c["valid"], _p(st["pe"]), s, c["mode"])
        return st["x"]
    if kind == "window":
        n = st["case"]["N"]
        audio_attn.WindowAttention(_p(st["q"]), _p(st["k"]), _p(st["v"]), _p(st["out"]),
                                   _p(st["start"]), _p(st["end"]), n, 16, 64, 0.125, s)
        return st["out"]
    if kind == "mha":
        c = st["case"]
        sortformer_attn.MaskedSelfAttention(_p(st["q"]), _p(st["k"]), _p(st["v"]), _p(st["out"]),
                                            c["T"], 8, 24, c["valid"], 24 ** -0.5, s)
        return st["out"]
    dec = st["dec"]
    dec.Prefill(_p(st["x"]), st["T"], s)
    prompt = dec.CopyLogits()
    tokens = dec.DecodeGreedy(st["T"], st["new"], *decoder.EOS_IDS, stream=s)
    return {"prompt_logits": prompt, "tokens": np.asarray(tokens, np.int32),
            "logits": dec.CopyLogits()}


# ------------------------------------------------------- what a pass cannot do without ----
def work(case):
    kind = case["kind"]
    row = HKV * DH * 2 * 2  # one token's K and V
    if kind in ("decode", "decode_paged"):
        # lengths are spread over [L/2, L] but for the longest
        keys = case["L"] + 1 + (case["B"] - 1) * (0.75 * case["L"] + 1)
        per = (2 * HQ + 2 * HKV) * DH * 4
        return {"bytes": keys * row + case["B"] * per, "flops": 4 * keys * HQ * DH}
    if kind == "prefill":
        T, p = case["T"], case["pos0"]
        pairs = T * p + T * (T + 1) / 2
        return {"bytes": (T + p) * row + 2 * T * HQ * DH * 4, "flops": 4 * pairs * HQ * DH}
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4 * M * K + 2 * K * N + 4 * M * N + (4 * N if case["bias"] else 0),
                "flops": 2 * M * K * N}
    if kind == "mlp":
        M = case["M"]
        return {"bytes": 2 * M * HIDDEN + 2 * 3 * HIDDEN * INTER + 2 * M * INTER + 4 * M * HIDDEN,
                "flops": 2 * M * 3 * HIDDEN * INTER}
    if kind == "conformer":
        T, D, F = case["T"], D_MODEL, D_FF
        params = 4 * D * F + 8 * D * D
        return {"bytes": 4 * (params + (2 * T - 1) * D + 2 * T * D),
                "flops": 2 * T * (4 * D * F + 7 * D * D) + 2 * (2 * T - 1) * D * D
                + 6 * T * case["valid"] * D}
    if kind == "window":
        a, b = _segments(case)
        return {"bytes": 4 * case["N"] * 16 * 64 * 4,
                "flops": 4 * 16 * 64 * sum(e - s for s, e in zip(a, b))}
    if kind == "mha":
        return {"bytes": 4 * case["T"] * 8 * 24 * 4, "flops": 4 * case["T"] * case["valid"] * 8 * 24}
    T, n, L = case["T"], case["new"], 28
    layer = HIDDEN * (4 * HKV * DH + 2 * HQ * DH - 2 * HKV * DH) + 3 * HIDDEN * INTER
    weights, head = 2 * L * layer, 2 * 151936 * HIDDEN
    keys = sum(T + i + 1 for i in range(n))
    return {"bytes": (1 + n) * (weights + head) + L * row * (T + keys) + 4 * T * HIDDEN,
            "flops": 2 * (T + n) * L * layer + (1 + n) * head
            + 4 * L * HQ * DH * (T * (T + 1) / 2 + keys)}


def tolerance(case):
    """Four times or so the distance between two correct forms of the same pass."""
    kind = case["kind"]
    if kind in ("decode", "decode_paged", "window", "mha"):
        return {"rel": 1e-5}
    if kind == "prefill":
        return {"rel": 1e-5} if case["mode"] == 0 else {"rel": 8e-3}
    if kind == "linear":
        return {"rel": 1e-5}
    if kind == "mlp":
        return {"rel": 2e-3}
    if kind == "conformer":
        return {"rel": 1e-5} if case["mode"] == 0 else {"rel": 4e-4}
    return {"rel": 2.5e-2}


# -------------------------------------------------------------- the same in 64 bits ----
def _softmax_av(q, k, v, mask, scale):
    """q [T, H, D], k and v [S, H, D], mask [T, S] of the keys each row attends; float64."""
    s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) * scale
    s = s.masked_fill(~mask, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.transpose(0, 1).contiguous()).transpose(0, 1)


def _bf16(x):
    return x.float().to(torch.bfloat16).double()


def _exact_decode(case, seed):
    st = _decode_inputs(case, seed)
    j = np.arange(DH // 2, dtype=np.float32)
    inv = np.power(np.float64(THETA), (-2.0 * j / DH).astype(np.float64)).astype(np.float32)

    def rope(x, gain, p):
        x = x.double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()
        ang = torch.from_numpy((np.float32(p) * inv).astype(np.float64)).to(DEV)
        a, b = x[..., :DH // 2], x[..., DH // 2:]
        return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()), -1)

    out = torch.empty(st["B"], HQ, DH, dtype=torch.float64, device=DEV)
    for b, n in enumerate(st["lens"]):
        if "table" in st:
            rows = (st["table"][b].long()[:, None] * PAGE + torch.arange(PAGE, device=DEV)).reshape(-1)[:n]
        else:
            rows = torch.arange(n, device=DEV)
        st["kc"][rows[n - 1]] = rope(st["k"][b], st["kn"], n - 1).float().to(torch.bfloat16)
        st["vc"][rows[n - 1]] = st["v"][b].to(torch.bfloat16)
        k, v = st["kc"][rows].double(), st["vc"][rows].double()
        k, v = (x.repeat_interleave(HQ // HKV, 1) for x in (k, v))
        mask = torch.ones(1, n, dtype=torch.bool, device=DEV)
        out[b] = _softmax_av(rope(st["q"][b], st["qn"], n - 1)[None], k, v, mask, SCALE)[0]
    return {"out": out, "kc": st["kc"], "vc": st["vc"]}


def _exact_prefill(case, seed):
    st = _prefill_inputs(case, seed)
    T, p = case["T"], case["pos0"]
    rows = torch.arange(st["cap"], device=DEV)
    if st["table"] is not None:
        rows = (st["table"].long()[:, None] * PAGE + torch.arange(PAGE, device=DEV)).reshape(-1)
    rows = rows[:T + p]
    mask = torch.arange(T + p, device=DEV)[None] <= torch.arange(p, T + p, device=DEV)[:, None]
    out = torch.empty(T, HQ, DH, dtype=torch.float64, device=DEV)
    G = HQ // HKV
    for h in range(HKV):
        k, v = (st[x][rows, h].double()[:, None].expand(-1, G, -1) for x in ("kc", "vc"))
        out[:, h * G:(h + 1) * G] = _softmax_av(st["q"][:, h * G:(h + 1) * G].double(), k, v, mask, SCALE)
    return out


def _exact_conformer(case, seed):
    st = _conformer_inputs(case, seed)
    w = {k: v.double() for k, v in st["w"].items()}
    T, valid, D, H = case["T"], case["valid"], D_MODEL, N_HEADS
    Dk = D // H
    F = torch.nn.functional
    norm = lambda x, p: F.layer_norm(x, (D,), w[f"norm_{p}_w"], w[f"norm_{p}_b"], 1e-5)  # noqa: E731
    lin = lambda x, p: x @ w[f"{p}_w"].T + w[f"{p}_b"]  # noqa: E731

    def ffn(x, p):
        h = F.silu(norm(x, p) @ w[f"{p}_w1"].T + w[f"{p}_b1"])
        return x + 0.5 * (h @ w[f"{p}_w2"].T + w[f"{p}_b2"])

    x = ffn(st["x0"].double(), "ff1")
    y = norm(x, "att")
    q, k, v = (lin(y, n).reshape(T, H, Dk).transpose(0, 1) for n in "qkv")
    pos = (st["pe"].double() @ w["pos_w"].T).reshape(2 * T - 1, H, Dk).permute(1, 2, 0).contiguous()
    u, vb = w["pos_bias_u"].reshape(H, 1, Dk), w["pos_bias_v"].reshape(H, 1, Dk)
    i = torch.arange(T, device=DEV)
    shift = (T - 1 - i[:, None] + i[None]).expand(H, T, T)
    s = (q + u) @ k.transpose(1, 2).contiguous() + ((q + vb) @ pos).gather(2, shift)
    s = (s / math.sqrt(Dk)).masked_fill(i[None, None] >= valid, -math.inf)
    ctx = (torch.softmax(s, -1) @ v).transpose(0, 1).reshape(T, D)
    x = x + lin(ctx, "out")
    a, b = lin(norm(x, "conv"), "pw1").chunk(2, -1)
    c = a * torch.sigmoid(b)
    c[valid:] = 0
    c = F.conv1d(c.T[None], w["dw_w"][:, None], w["dw_b"], padding=(CONV - 1) // 2, groups=D)[0].T
    c = (c - w["bn_mean"]) * torch.rsqrt(w["bn_var"] + 1e-5) * w["bn_w"] + w["bn_b"]
    x = x + lin(F.silu(c), "pw2")
    return norm(ffn(x, "ff2"), "out")


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "decode_paged"):
        return _exact_decode(case, seed)
    if kind == "prefill":
        return _exact_prefill(case, seed)
    if kind == "linear":
        st = _linear_inputs(case, seed)
        y = _bf16(st["x"]) @ st["W"].double().T
        if case["bias"]:
            y = y + st["b"].double()
        return torch.nn.functional.gelu(y) if case["act"] == 1 else y
    if kind == "mlp":
        st = _mlp_inputs(case, seed)
        g, u = (st["x"].double() @ st["gu"].double().T).chunk(2, -1)
        act = torch.nn.functional.silu(g) * u
        return {"act": act, "out": _bf16(act) @ st["dn"].double().T}
    if kind == "conformer":
        return _exact_conformer(case, seed)
    if kind == "window":
        st = _small_attn_inputs(case, seed)
        j = torch.arange(case["N"], device=DEV)[None]
        mask = (j >= st["start"][:, None]) & (j < st["end"][:, None])
        return _softmax_av(*(st[x].double() for x in "qkv"), mask, 0.125)
    if kind == "mha":
        st = _small_attn_inputs(case, seed)
        mask = (torch.arange(case["T"], device=DEV) < case["valid"]).expand(case["T"], -1)
        return _softmax_av(*(st[x].double() for x in "qkv"), mask, 24 ** -0.5)
    return None
