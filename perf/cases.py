"""Performance cases: what a program built on rapidllm_amd has the GPU do.

Each case is one pass through the public entry points (the C ABI bound by
rapidllm_amd.hip, or rapidllm_amd.engine.Engine) at a size the 27B hybrid model or its
tests use: the layers of a decode step at one token, at a verify's four and at batch
widths, the layers of a prompt prefill, and two whole-engine calls.

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs, packed weights and workspaces, on the GPU
  run(state)          one pass; returns its outputs
  work(case)          bytes and operations the pass cannot do without
  tolerance(case)     how far another correct implementation's outputs may be
  exact(case, seed)   the outputs in 64-bit arithmetic with plain torch
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from rapidllm_amd import hip
from rapidllm_amd.engine import Engine
from rapidllm_amd.hip import call
from rapidllm_amd.model import Q_Q4_K, Q_Q6_K, qwen27b_spec

DEV = "cuda"
HEAD = 128    # DeltaNet key and value width
HD = 256      # attention head width
ROT = 64      # rotary dimensions
THETA = 1e7
EPS = 1e-6
CONV = 4      # conv taps

# Row-major [m][n] linears of a layer: DeltaNet in_proj, attention q|gate;k;v, the two
# output projections, MLP gate/up and down; odd ones as the GEMM tests use.
LINEARS = [(16480, 5120), (14336, 5120), (5120, 6144), (34816, 5120), (5120, 17408), (1000, 1152), (4112, 2560)]


def listed():
    return [
        # One token through one DeltaNet layer's recurrent update: the smallest call of a
        # decode step, 48 times per token.
        {"name": "gdn_decode_t1", "kind": "gdn_decode", "T": 1, "nk": 16, "nv": 48},
        # One token through the largest single linear (MLP down): the weight stream that
        # single-user decoding consists of.
        {"name": "fp8_linear_t1", "kind": "fp8_linear", "m": 5120, "n": 17408, "T": 1},
        # An odd batch of sequences through the attention input projection.
        {"name": "fp8_linear_t13", "kind": "fp8_linear", "m": 14336, "n": 5120, "T": 13},
        # One token through the MLP of a GGUF Q4_K model.
        {"name": "q4k_mlp_t1", "kind": "kq_mlp", "q": 4, "H": 5120, "I": 17408, "T": 1},
        # A batch of twelve sequences through the MLP of a GGUF Q6_K model.
        {"name": "q6k_mlp_t12", "kind": "kq_mlp", "q": 6, "H": 5120, "I": 17408, "T": 12},
        # lm_head and greedy choice for the four tokens of a speculative verify.
        {"name": "head_t4", "kind": "head", "V": 248320, "H": 5120, "T": 4},
        # Four verify tokens attending over a long context.
        {"name": "attn_decode_32k", "kind": "attn_decode", "T": 4, "pos": 32000, "nq": 24, "nkv": 4},
        # MLP block (norm, gate/up with SwiGLU, down) over a ragged prompt chunk.
        {"name": "fp8_mlp_prefill", "kind": "fp8_mlp", "H": 5120, "I": 17408, "T": 2011},
        # Attention of a prompt chunk behind an earlier one.
        {"name": "attn_prefill", "kind": "attn_prefill", "T": 1500, "pos": 2500, "nq": 24, "nkv": 4},
        # DeltaNet recurrence of a prompt chunk.
        {"name": "gdn_prefill", "kind": "gdn_prefill", "T": 2011, "nk": 16, "nv": 48},
        # Single-user decoding of a block-FP8 model: 16 steps, then the last logits.
        {"name": "engine_decode_fp8", "kind": "engine_decode", "q": 0, "layers": 16, "B": 1, "steps": 16},
        # A long prompt into a GGUF Q4_K model, up to its logits.
        {"name": "engine_prefill_q4k", "kind": "engine_prefill", "q": 4, "layers": 16, "T": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gdn_decode", "fp8_linear", "kq_mlp", "head", "attn_decode", "fp8_mlp", "attn_prefill",
                       "gdn_prefill", "engine_decode", "engine_prefill"])
    if kind == "gdn_decode":
        nk, nv = rng.choice([(16, 48), (16, 32), (2, 6), (4, 4)])
        return {"kind": kind, "T": rng.randint(1, 8), "nk": nk, "nv": nv}
    if kind == "fp8_linear":
        m, n = rng.choice(LINEARS)
        return {"kind": kind, "m": m, "n": n, "T": rng.randint(1, 16)}
    if kind == "kq_mlp":
        return {"kind": kind, "q": rng.choice([4, 6]), "H": 256 * rng.randint(4, 20), "I": 256 * rng.randint(4, 68),
                "T": rng.randint(1, 16)}
    if kind == "head":
        return {"kind": kind, "V": rng.choice([248320, 151936, 32000]), "H": 128 * rng.randint(8, 40),
                "T": rng.randint(1, 4)}
    if kind == "attn_decode":
        nq, nkv = rng.choice([(24, 4), (24, 4), (12, 2), (6, 1)])
        return {"kind": kind, "T": rng.randint(1, 4), "pos": _log(rng, 1, 36000), "nq": nq, "nkv": nkv}
    if kind == "fp8_mlp":
        return {"kind": kind, "H": 128 * rng.randint(8, 40), "I": 128 * rng.randint(16, 136),
                "T": _log(rng, 17, 2048)}
    if kind == "attn_prefill":
        nq, nkv = rng.choice([(24, 4), (24, 4), (12, 2), (6, 1)])
        return {"kind": kind, "T": _log(rng, 17, 2048), "pos": rng.choice([0, _log(rng, 1, 6000)]), "nq": nq,
                "nkv": nkv}
    if kind == "gdn_prefill":
        nk, nv = rng.choice([(16, 48), (16, 48), (16, 32), (2, 6)])
        return {"kind": kind, "T": _log(rng, 17, 4096), "nk": nk, "nv": nv}
    if kind == "engine_decode":
        return {"kind": kind, "q": rng.choice([0, 4]), "layers": 4 * rng.randint(1, 4), "B": rng.randint(1, 16),
                "steps": rng.randint(2, 16)}
    return {"kind": kind, "q": rng.choice([0, 4]), "layers": 4 * rng.randint(1, 4), "T": _log(rng, 24, 2000)}


# ---------------------------------------------------------------- inputs from the seed


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _ints(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV)


def _acts(g, T, n):
    """Hidden states: unit scale with a few channels an order of magnitude larger, as a
    residual stream has."""
    x = _randn(g, T, n)
    wide = _ints(g, 0, n, max(1, n // 256))
    x[:, wide] *= 12.0
    return x


def _fp8(g, m, n):
    """A block-FP8 weight: normal values, each 128x128 block scaled to e4m3's range."""
    mp, np_ = -(-m // 128) * 128, -(-n // 128) * 128
    w = torch.zeros(mp, np_, device=DEV)
    w[:m, :n] = _randn(g, m, n, std=0.02)
    blk = w.view(mp // 128, 128, np_ // 128, 128)
    scale = blk.abs().amax(dim=(1, 3)) / 448.0
    q = (blk / scale[:, None, :, None]).reshape(mp, np_)[:m, :n]
    return q.to(torch.float8_e4m3fn).contiguous(), scale.contiguous()


def _fp8_f64(w, scale):
    m, n = w.shape
    s = scale.repeat_interleave(128, 0)[:m].repeat_interleave(128, 1)[:, :n]
    return w.to(torch.float32).double() * s.double()


def _fp16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


def _kq_blocks(g, q, m, n):
    """GGUF super-blocks of a weight of standard deviation about 0.02 to 0.05: random
    quants, sub-block scales within a factor of a few of each other, and (Q4_K) mins
    that centre each sub-block."""
    nb = m * (n // 256)
    if q == 4:
        blk = torch.empty(nb, 144, dtype=torch.uint8, device=DEV)
        d = 5e-5 * (1 + torch.rand(nb, generator=g, device=DEV))
        blk[:, 0:2] = _fp16_bytes(d)
        blk[:, 2:4] = _fp16_bytes(d * 7.5)
        sc = _ints(g, 16, 64, nb, 8)
        mn = (sc + _ints(g, -3, 4, nb, 8)).clamp(0, 63)
        # 6-bit packing: bytes 0..3 scales 0..3, 4..7 mins 0..3 (top two bits hold the
        # top bits of entries 4..7), 8..11 the low nibbles of entries 4..7
        blk[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        blk[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
        blk[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
        blk[:, 16:] = torch.randint(0, 256, (nb, 128), generator=g, device=DEV, dtype=torch.uint8)
        return blk
    blk = torch.empty(nb, 210, dtype=torch.uint8, device=DEV)
    blk[:, :192] = torch.randint(0, 256, (nb, 192), generator=g, device=DEV, dtype=torch.uint8)
    sc = _ints(g, 10, 61, nb, 16) * (2 * _ints(g, 0, 2, nb, 16) - 1)
    blk[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
    blk[:, 208:210] = _fp16_bytes(3e-5 * (1 + torch.rand(nb, generator=g, device=DEV)))
    return blk


def _kq_f64(blk, q, m, n):
    nb = blk.shape[0]
    f16 = lambda c: blk[:, c:c + 2].contiguous().view(torch.float16).double()  # noqa: E731  [nb][1]
    if q == 4:
        s = blk[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = blk[:, 16:].view(nb, 4, 1, 32)
        qv = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32).double()
        w = (f16(0) * sc)[:, :, None] * qv - (f16(2) * mn)[:, :, None]
    else:
        ql = blk[:, :128].view(nb, 2, 2, 32).to(torch.int32)
        qh = blk[:, 128:192].view(nb, 2, 1, 32).to(torch.int32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [nb][half][quarter][32]
        sh = torch.tensor([0, 2, 4, 6], device=DEV, dtype=torch.int32).view(1, 1, 4, 1)
        qv = (lo | (((qh >> sh) & 3) << 4)).double() - 32.0
        sc = blk[:, 192:208].contiguous().view(torch.int8).double()
        w = f16(208)[:, :, None] * (sc[:, :, None] * qv.view(nb, 16, 16))
    return w.reshape(m, n)


def _gdn_inputs(c, seed):
    g, nk, nv = _gen(seed), c["nk"], c["nv"]
    cd = 2 * nk * HEAD + nv * HEAD
    return {
        "y": _randn(g, c["T"], cd + 2 * nv),  # in_proj rows: q|k|v channels, a, b
        "A_log": _randn(g, nv, std=0.5),
        "dt": _randn(g, nv, std=0.5),
        "conv_w": _randn(g, cd, CONV, std=0.5),
        "conv": _randn(g, cd, CONV),
        "S": _randn(g, nv, HEAD, HEAD, std=0.02),  # transposed: [head][value][key]
        "cd": cd,
    }


def _attn_inputs(c, seed):
    g, nq, nkv, pos = _gen(seed), c["nq"], c["nkv"], c["pos"]
    ctx = -(-(pos + c["T"]) // 256) * 256
    kv = []
    for _ in range(2):
        a = torch.zeros(nkv, ctx, HD, device=DEV, dtype=torch.float16)
        a[:, :pos] = _randn(g, nkv, pos, HD).to(torch.float16)
        kv.append(a)
    return {
        "Y": _randn(g, c["T"], 2 * nq * HD + 2 * nkv * HD),
        "qn": _randn(g, HD, std=0.1),
        "kn": _randn(g, HD, std=0.1),
        "K": kv[0],
        "V": kv[1],
        "ctx": ctx,
    }


# ---------------------------------------------------------------- states


def _u8(nbytes):
    return torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=DEV)


def _zeros_u8(nbytes):
    return torch.zeros(max(int(nbytes), 16), dtype=torch.uint8, device=DEV)


def _f32(*shape):
    return torch.empty(*shape, device=DEV)


def _pack_fp8(w, scale):
    m, n = w.shape
    L = hip.lib()
    wt, ts = _u8(L.rl_hip_fp8_packed_bytes(m, n)), _f32(L.rl_hip_fp8_tile_scales(m, n))
    call("rl_hip_pack_fp8", w.data_ptr(), scale.data_ptr(), wt.data_ptr(), ts.data_ptr(), m, n, None)
    torch.cuda.synchronize()
    return wt, ts


def _pack_kq(q, blk, m, n):
    t = Q_Q4_K if q == 4 else Q_Q6_K
    w = _u8(hip.lib().rl_hip_kquant_tiled_bytes(t, m, n))
    call("rl_hip_pack_kquant", t, blk.data_ptr(), w.data_ptr(), m, n, None)
    torch.cuda.synchronize()
    return w


def _frag(n, T):
    return _u8(hip.lib().rl_hip_act_frag_bytes(n, T))


def _fp8_linear_inputs(c, seed):
    g = _gen(seed)
    w, s = _fp8(g, c["m"], c["n"])
    return w, s, _acts(g, c["T"], c["n"])


def _kq_mlp_inputs(c, seed):
    g, q, H, I = _gen(seed), c["q"], c["H"], c["I"]
    return _kq_blocks(g, q, I, H), _kq_blocks(g, q, I, H), _kq_blocks(g, q, H, I), _acts(g, c["T"], H)


def _head_inputs(c, seed):
    g = _gen(seed)
    w = torch.empty(c["V"], c["H"], dtype=torch.bfloat16, device=DEV)
    for r in range(0, c["V"], 32768):
        w[r:r + 32768] = _randn(g, min(32768, c["V"] - r), c["H"], std=0.02).to(torch.bfloat16)
    return w, _acts(g, c["T"], c["H"])


def _fp8_mlp_inputs(c, seed):
    g, H, I = _gen(seed), c["H"], c["I"]
    return _fp8(g, I, H), _fp8(g, I, H), _fp8(g, H, I), _randn(g, H, std=0.1), _acts(g, c["T"], H)


def prepare(case, seed):
    c, k, L = case, case["kind"], hip.lib()
    if k in ("gdn_decode", "gdn_prefill"):
        s = dict(_gdn_inputs(c, seed), c=c)
        s["o"] = _f32(c["T"], c["nv"] * HEAD)
        s["conv_out"] = torch.empty_like(s["conv"])
        if k == "gdn_decode":
            s["S_out"] = torch.empty_like(s["S"])
        else:
            s["ws"] = _u8(L.rl_hip_gdn_prefill_workspace_bytes(c["T"], c["nk"], c["nv"], HEAD, HEAD))
        return s
    if k == "fp8_linear":
        w, sc, x = _fp8_linear_inputs(c, seed)
        wt, ts = _pack_fp8(w, sc)
        return {"c": c, "w": wt, "ts": ts, "x": x, "frag": _frag(c["n"], c["T"]), "y": _f32(c["T"], c["m"])}
    if k == "kq_mlp":
        H, I, T = c["H"], c["I"], c["T"]
        t = Q_Q4_K if c["q"] == 4 else Q_Q6_K
        gb, ub, db, x = _kq_mlp_inputs(c, seed)
        gu = _u8(L.rl_hip_kquant_tiled_bytes(t, 2 * I, H))
        call("rl_hip_pack_kquant_gate_up", t, gb.data_ptr(), ub.data_ptr(), gu.data_ptr(), I, H, None)
        torch.cuda.synchronize()
        return {"c": c, "t": t, "gu": gu, "down": _pack_kq(c["q"], db, H, I), "x": x, "h": _f32(T, I),
                "y": _f32(T, H), "ws_gu": _zeros_u8(L.rl_hip_kquant_workspace_bytes(2 * I, H, T)),
                "ws_down": _zeros_u8(L.rl_hip_kquant_workspace_bytes(H, I, T))}
    if k == "head":
        w, x = _head_inputs(c, seed)
        wt = _u8(L.rl_hip_bf16_packed_bytes(c["V"], c["H"]))
        call("rl_hip_pack_bf16", w.data_ptr(), wt.data_ptr(), c["V"], c["H"], None)
        torch.cuda.synchronize()
        T = c["T"]
        return {"c": c, "w": wt, "x": x, "frag": _frag(c["H"], T), "logits": _f32(T, c["V"]),
                "idx": torch.empty(T, dtype=torch.int32, device=DEV), "val": _f32(T),
                "ws": _u8(L.rl_hip_argmax_workspace_bytes(T, c["V"]))}
    if k in ("attn_decode", "attn_prefill"):
        s = _attn_inputs(c, seed)
        nkv, ctx, T = c["nkv"], s["ctx"], c["T"]
        # the caches in the documented fragment orders
        kc = s["K"].view(nkv, ctx // 256, 16, 16, HD // 32, 4, 8).permute(0, 1, 4, 2, 5, 3, 6).contiguous()
        vc = s["V"].view(nkv, ctx // 32, 4, 8, HD // 16, 16).permute(0, 1, 4, 2, 5, 3).contiguous()
        nb = (L.rl_hip_attn_workspace_bytes(nkv, ctx) if k == "attn_decode"
              else L.rl_hip_attn_prefill_workspace_bytes(c["nq"], T))
        return {"c": c, "Y": s["Y"], "qn": s["qn"], "kn": s["kn"], "kc": kc, "vc": vc, "ctx": ctx,
                "pos": torch.tensor([c["pos"]], dtype=torch.int32, device=DEV), "ws": _zeros_u8(nb), "nb": nb,
                "out": _f32(T, c["nq"] * HD)}
    if k == "fp8_mlp":
        H, I, T = c["H"], c["I"], c["T"]
        (gw, gs), (uw, us), (dw, ds), gamma, x = _fp8_mlp_inputs(c, seed)
        gu, gts = _u8(L.rl_hip_fp8_packed_bytes(2 * I, H)), _f32(L.rl_hip_fp8_gate_up_tile_scales(I, H))
        call("rl_hip_pack_fp8_gate_up", gw.data_ptr(), gs.data_ptr(), uw.data_ptr(), us.data_ptr(), gu.data_ptr(),
             gts.data_ptr(), I, H, None)
        down, dts = _pack_fp8(dw, ds)
        return {"c": c, "gu": gu, "gts": gts, "down": down, "dts": dts, "gamma": gamma, "x": x, "fx": _frag(H, T),
                "fh": _frag(I, T), "y": _f32(T, H)}
    # whole engine: device-generated weights of the 27B model's shape, fewer layers
    spec = qwen27b_spec(n_layers=c["layers"], has_mtp=False)
    rng = np.random.Generator(np.random.PCG64(seed))
    old = os.environ.pop("RL_SYNTH_LINEAR", None)
    if c["q"] == 4:
        os.environ["RL_SYNTH_LINEAR"] = "q4_k"
    try:
        B = c.get("B", 1)
        eng = Engine(spec, None, ctx=max(512, c.get("T", 0) + 16), seed=seed & 0xFFFF, max_batch=B)
    finally:
        os.environ.pop("RL_SYNTH_LINEAR", None)
        if old is not None:
            os.environ["RL_SYNTH_LINEAR"] = old
    shape = (c["steps"], B) if k == "engine_decode" else (c["T"],)
    return {"c": c, "eng": eng, "ids": rng.integers(0, spec.vocab, shape).astype(np.int32)}


# ---------------------------------------------------------------- one pass


def run(s):
    c, k = s["c"], s["c"]["kind"]
    p = lambda name: s[name].data_ptr()  # noqa: E731
    if k == "gdn_decode":
        ld, cd, nv = s["cd"] + 2 * c["nv"], s["cd"], c["nv"]
        call("rl_hip_gdn_decode", p("y"), p("y") + 4 * cd, p("y") + 4 * (cd + nv), ld, p("A_log"), p("dt"),
             p("conv_w"), p("conv"), p("conv_out"), p("S"), p("S_out"), p("o"), c["T"], c["nk"], nv, HEAD, HEAD, CONV,
             0, None)
        return {"o": s["o"], "S": s["S_out"], "conv": s["conv_out"]}
    if k == "gdn_prefill":
        ld, cd, nv = s["cd"] + 2 * c["nv"], s["cd"], c["nv"]
        # the state advances in place, as over the chunks of a prompt
        call("rl_hip_gdn_prefill", p("y"), ld, cd, cd + nv, p("A_log"), p("dt"), p("conv_w"), p("conv"),
             p("conv_out"), p("S"), p("o"), p("ws"), s["ws"].numel(), c["T"], c["nk"], nv, HEAD, HEAD, CONV, 0, None)
        return {"o": s["o"], "S": s["S"], "conv": s["conv_out"]}
    if k == "fp8_linear":
        call("rl_hip_pack_act", p("x"), p("frag"), c["n"], c["T"], None)
        call("rl_hip_gemm_fp8_frag", p("w"), p("ts"), p("frag"), p("y"), c["m"], c["n"], c["T"], 0, None)
        return s["y"]
    if k == "kq_mlp":
        H, I, T = c["H"], c["I"], c["T"]
        call("rl_hip_gemm_kquant_swiglu", s["t"], p("gu"), p("x"), p("h"), p("ws_gu"), s["ws_gu"].numel(), I, H, T,
             None)
        call("rl_hip_gemm_kquant", s["t"], p("down"), p("h"), p("y"), p("ws_down"), s["ws_down"].numel(), H, I, T, 0,
             None)
        return {"h": s["h"], "y": s["y"]}
    if k == "head":
        call("rl_hip_pack_act", p("x"), p("frag"), c["H"], c["T"], None)
        call("rl_hip_gemm_bf16_frag", p("w"), p("frag"), p("logits"), c["V"], c["H"], c["T"], 0, None)
        call("rl_hip_argmax_rows", p("logits"), c["T"], c["V"], p("idx"), p("val"), p("ws"), None)
        return {"logits": s["logits"], "idx": s["idx"], "val": s["val"]}
    if k == "attn_decode":
        ld = s["Y"].shape[1]
        call("rl_hip_attn_decode_layer", p("Y"), ld, p("qn"), p("kn"), p("kc"), p("vc"), s["ctx"], p("pos"), c["T"],
             c["nq"], c["nkv"], HD, ROT, THETA, EPS, p("ws"), s["nb"], p("out"), None, None)
        return s["out"]
    if k == "attn_prefill":
        ld = s["Y"].shape[1]
        call("rl_hip_attn_prefill_layer", p("Y"), ld, p("qn"), p("kn"), p("kc"), p("vc"), s["ctx"], p("pos"), c["T"],
             c["nq"], c["nkv"], HD, ROT, THETA, EPS, p("ws"), s["nb"], p("out"), None)
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if k == "fp8_mlp":
        H, I, T = c["H"], c["I"], c["T"]
        call("rl_hip_rmsnorm_pack", p("x"), H, p("gamma"), None, p("fx"), H, T, EPS, None)
        call("rl_hip_gemm_fp8_prefill", p("gu"), p("gts"), p("fx"), p("fh"), 2 * I, H, T, 6, 0, None)
        call("rl_hip_gemm_fp8_prefill", p("down"), p("dts"), p("fh"), p("y"), H, I, T, 0, 0, None)
        return s["y"]
    eng, ids = s["eng"], s["ids"]
    if k == "engine_prefill":
        eng.prefill(ids)
        return eng.copy_logits()
    # the same token sequences from empty states each pass
    if c["B"] == 1:
        eng.reset()
        for t in range(c["steps"]):
            eng.decode_token(int(ids[t, 0]))
            eng.greedy()
        return eng.copy_logits()
    eng.zero_slots(c["B"])
    for t in range(c["steps"]):
        eng.decode_tokens(ids[t], [t] * c["B"])
        eng.copy_greedy_n(c["B"])
    return eng.copy_logits_n(c["B"])


# ---------------------------------------------------------------- work and tolerance

_KQ_BYTES = {4: 144 / 256, 6: 210 / 256}


def _layer_params(spec, delta):
    H, I = spec.hidden, spec.intermediate
    if delta:
        zd = spec.n_v_heads * spec.v_dim
        mix = H * (spec.conv_dim + zd + 2 * spec.n_v_heads) + H * zd
    else:
        mix = H * (2 * spec.n_q + 2 * spec.n_kv) * HD + H * spec.n_q * HD
    return mix + 3 * H * I


def work(case):
    c, k = case, case["kind"]
    T = c.get("T", 1)
    if k in ("gdn_decode", "gdn_prefill"):
        nk, nv = c["nk"], c["nv"]
        cd, S = 2 * nk * HEAD + nv * HEAD, nv * HEAD * HEAD
        return {"bytes": 4 * (T * (cd + 2 * nv + nv * HEAD) + 3 * cd * CONV + 2 * S + 2 * nv),
                "flops": T * (7 * S + 2 * CONV * cd)}
    if k == "fp8_linear":
        m, n = c["m"], c["n"]
        return {"bytes": m * n + 4 * -(-m // 128) * -(-n // 128) + 4 * T * (m + n), "flops": 2 * m * n * T}
    if k == "kq_mlp":
        H, I = c["H"], c["I"]
        return {"bytes": 3 * H * I * _KQ_BYTES[c["q"]] + 4 * T * 2 * (H + I), "flops": 6 * H * I * T}
    if k == "head":
        return {"bytes": 2 * c["V"] * c["H"] + 4 * T * (c["V"] + c["H"]), "flops": 2 * c["V"] * c["H"] * T}
    if k in ("attn_decode", "attn_prefill"):
        nq, nkv, pos = c["nq"], c["nkv"], c["pos"]
        pairs = T * pos + T * (T + 1) // 2
        return {"bytes": 4 * T * (3 * nq + 2 * nkv) * HD + 4 * nkv * (pos + T) * HD, "flops": 4 * pairs * nq * HD}
    if k == "fp8_mlp":
        H, I = c["H"], c["I"]
        return {"bytes": 3 * H * I + 8 * T * H, "flops": 6 * H * I * T}
    spec = qwen27b_spec(n_layers=c["layers"], has_mtp=False)
    nd = 3 * c["layers"] // 4
    lin = nd * _layer_params(spec, True) + (c["layers"] - nd) * _layer_params(spec, False)
    wb = lin * (_KQ_BYTES[4] if c["q"] == 4 else 1.0)
    head = spec.vocab * spec.hidden
    hb = head * (_KQ_BYTES[6] if c["q"] == 4 else 2.0)
    state = nd * 8 * spec.n_v_heads * HEAD * HEAD
    if k == "engine_prefill":
        return {"bytes": wb + hb + state, "flops": 2 * lin * T + 2 * head}
    B = c["B"]
    return {"bytes": c["steps"] * (wb + hb + B * state + 4 * B * spec.vocab), "flops": c["steps"] * 2 * B * (lin + head)}


def tolerance(case):
    # About four times what was measured.  Against 64 bits: the linears, which take
    # activations as 15 or 16 significant bits, 1e-5 (one) to 6e-5 (a K-quant MLP),
    # attention 2e-4 (fp16 probabilities), the recurrence 1e-7 to 2e-7 (32-bit sums in
    # any order stay within 1e-5).  Whole engines: one prompt through the prefill and
    # through the decode kernels, 1e-5 to 3e-5 (block-FP8) and 3e-4 (K-quant).
    q = case.get("q", 0)
    return {
        "gdn_decode": {"rel": 1e-5, "max": 1e-3},
        "gdn_prefill": {"rel": 2e-5, "max": 2e-3},
        "fp8_linear": {"rel": 5e-5, "max": 1e-3},
        "kq_mlp": {"rel": 2.5e-4, "max": 5e-3},
        "head": {"rel": 5e-5, "max": 1e-3},
        "attn_decode": {"rel": 1e-3, "max": 1e-2},
        "attn_prefill": {"rel": 1e-3, "max": 1e-2},
        "fp8_mlp": {"rel": 1e-4, "max": 2e-3},
        "engine_decode": {"rel": 1.5e-3 if q else 2e-4, "max": 1e-2 if q else 1e-3},
        "engine_prefill": {"rel": 1.5e-3 if q else 2e-4, "max": 1e-2 if q else 1e-3},
    }[case["kind"]]


# ---------------------------------------------------------------- 64-bit references


def _silu(x):
    return x * torch.sigmoid(x)


def _l2n(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + EPS)


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + gamma.double())


def _gdn_exact(c, seed):
    s = _gdn_inputs(c, seed)
    T, nk, nv, cd = c["T"], c["nk"], c["nv"], s["cd"]
    y = s["y"].double()
    raw = torch.cat([s["conv"].double()[:, 1:].T, y[:, :cd]], 0)  # the window's last taps, then the tokens
    w = s["conv_w"].double()
    mix = _silu(sum(raw[j:j + T] * w[:, j] for j in range(CONV)))
    win = torch.cat([s["conv"].double().T, y[:, :cd]], 0)[-CONV:].T
    src = torch.arange(nv, device=DEV) // (nv // nk)
    q = _l2n(mix[:, :nk * HEAD].reshape(T, nk, HEAD)[:, src]) / math.sqrt(HEAD)
    kk = _l2n(mix[:, nk * HEAD:2 * nk * HEAD].reshape(T, nk, HEAD)[:, src])
    v = mix[:, 2 * nk * HEAD:].reshape(T, nv, HEAD)
    beta = torch.sigmoid(y[:, cd + nv:])
    g = torch.exp(-torch.exp(s["A_log"].double()) * torch.nn.functional.softplus(y[:, cd:cd + nv] + s["dt"].double()))
    S, o = s["S"].double(), torch.empty(T, nv, HEAD, dtype=torch.float64, device=DEV)
    for t in range(T):
        S = S * g[t][:, None, None]
        d = (v[t] - (S * kk[t][:, None, :]).sum(-1)) * beta[t][:, None]
        S = S + d[:, :, None] * kk[t][:, None, :]
        o[t] = (S * q[t][:, None, :]).sum(-1)
    return {"o": o.reshape(T, nv * HEAD), "S": S, "conv": win.contiguous()}


def _rope(x, pos):
    """x [T][heads][256] at positions pos..: pairs (i, i + 32) of the first 64 dims;
    angles in 32 bits, as the model defines them."""
    half = ROT // 2
    freq = (1.0 / torch.pow(torch.tensor(THETA, dtype=torch.float32),
                            torch.arange(half, dtype=torch.float32) / half)).to(DEV)
    ang = (torch.arange(pos, pos + x.shape[0], device=DEV, dtype=torch.float32)[:, None] * freq).double()[:, None, :]
    a, b = x[..., :half], x[..., half:ROT]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos(), x[..., ROT:]], -1)


def _attn_exact(c, seed):
    s = _attn_inputs(c, seed)
    T, nq, nkv, pos = c["T"], c["nq"], c["nkv"], c["pos"]
    Y = s["Y"].double()
    qg = Y[:, :2 * nq * HD].reshape(T, nq, 2, HD)
    kv = Y[:, 2 * nq * HD:].reshape(T, 2, nkv, HD)
    q = _rope(_rms(qg[:, :, 0], s["qn"]), pos)
    K, V = s["K"].clone(), s["V"].clone()
    K[:, pos:pos + T] = _rope(_rms(kv[:, 0], s["kn"]), pos).transpose(0, 1).to(torch.float16)
    V[:, pos:pos + T] = kv[:, 1].transpose(0, 1).to(torch.float16)
    out = torch.empty(T, nq, HD, dtype=torch.float64, device=DEV)
    seen = torch.arange(pos + T, device=DEV)[None, :] <= torch.arange(pos, pos + T, device=DEV)[:, None]
    for h in range(nq):
        kh, vh = K[h // (nq // nkv), :pos + T].double(), V[h // (nq // nkv), :pos + T].double()
        sc = (q[:, h].contiguous() @ kh.T.contiguous()) / math.sqrt(HD)
        out[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ vh
    out = (out * torch.sigmoid(qg[:, :, 1])).reshape(T, nq * HD)
    return out if c["kind"] == "attn_decode" else {"out": out, "k": None, "v": None}


def exact(case, seed):
    c, k = case, case["kind"]
    if k in ("gdn_decode", "gdn_prefill"):
        return _gdn_exact(c, seed)
    if k in ("attn_decode", "attn_prefill"):
        return _attn_exact(c, seed)
    if k == "fp8_linear":
        w, sc, x = _fp8_linear_inputs(c, seed)
        return x.double() @ _fp8_f64(w, sc).T.contiguous()
    if k == "kq_mlp":
        gb, ub, db, x = _kq_mlp_inputs(c, seed)
        H, I, q, xd = c["H"], c["I"], c["q"], x.double()
        h = _silu(xd @ _kq_f64(gb, q, I, H).T.contiguous()) * (xd @ _kq_f64(ub, q, I, H).T.contiguous())
        return {"h": h, "y": h @ _kq_f64(db, q, H, I).T.contiguous()}
    if k == "head":
        w, x = _head_inputs(c, seed)
        xd = x.double()
        y = torch.cat([xd @ w[r:r + 16384].double().T.contiguous() for r in range(0, c["V"], 16384)], 1)
        val, idx = y.max(1)
        return {"logits": y, "idx": None, "val": val}
    if k == "fp8_mlp":
        gw, uw, dw, gamma, x = _fp8_mlp_inputs(c, seed)
        n = _rms(x.double(), gamma)
        h = _silu(n @ _fp8_f64(*gw).T.contiguous()) * (n @ _fp8_f64(*uw).T.contiguous())
        return h @ _fp8_f64(*dw).T.contiguous()
    return None  # a whole model: its layers are checked one by one
