#!/usr/bin/env python3
"""Benchmark: the Qwen3.6/3.8-27B-shape MTP speculative-verify decode step on one
MI355X, with the block-FP8 GEMM roofline and the reference
CPU path timed beside it.

    python bench.py [--gpus 1] [--steps K] [--warmup W]

Workload (synthetic, random-init, generated on the device): 64 layers (48 Gated
DeltaNet + 16 gated attention), hidden 5120, intermediate 17408, block-FP8 e4m3
linears with 128x128 fp32 scales log-uniform in [1e-3, 1e-1], bf16 embedding and
lm_head (vocab 248320), fp16 KV cache prefilled with N(0,1) to 32768 positions,
a 1-layer MTP stem head.  Timed regions replay the captured HIP graphs with all
inputs resident in HBM:
  T=1 decode step (self-fed), T=4 MTP-verify step, 3-token MTP stem draft.
value = T=1 decode tokens/s.  One JSON line on stdout.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "decode tok/s at T=1 and MTP-verify T=4; achieved HBM GB/s vs MI355X peak"
PEAK_GBS = 8000.0
CTX = 32768
PF_TOKENS = 4096


def measure_gguf_step(spec, K, W):
    """The same C5 step with the layer linears and MTP fc as Q4_K super-blocks and a
    Q6_K lm_head (the tensor mix of a Q4_K_M GGUF; in_proj a/b BF16), random blocks
    generated on the device: T=1 and T=4 step times, the batch-4, -8 and -16 steps
    (sequences at 32K context, one weight pass each) and the weight bytes a T=1 step
    reads."""
    from rapidllm_amd.engine import Engine

    os.environ["RL_SYNTH_LINEAR"] = "q4_k"
    try:
        eng = Engine(spec, None, ctx=CTX + 4096, max_T=4, seed=4321, max_batch=16)
    finally:
        del os.environ["RL_SYNTH_LINEAR"]
    eng.synthetic_context(CTX)
    eng.replicate_slot0(16)
    eng.time_batch(4, W)
    tb4 = eng.time_batch(4, K) / K
    eng.time_batch(8, W)
    tb8 = eng.time_batch(8, K) / K
    eng.time_batch(16, W)
    tb16 = eng.time_batch(16, K) / K
    eng.synthetic_context(CTX)
    eng.time_steps(1, W)
    t1 = eng.time_steps(1, K) / K
    eng.synthetic_context(CTX)
    eng.time_steps(4, W)
    t4 = eng.time_steps(4, K) / K
    # prompt prefill through the chunked path (K-quant linears as fp16 tiles, block-scaled)
    ids = np.random.default_rng(3).integers(0, spec.vocab, PF_TOKENS).astype(np.int32)
    eng.prefill(ids[:600])
    tp = time.perf_counter()
    eng.prefill(ids)
    pf_s = time.perf_counter() - tp
    eng.close()
    H, I, V = spec.hidden, spec.intermediate, spec.vocab
    nk, nv, dk, dv = spec.n_k_heads, spec.n_v_heads, spec.k_dim, spec.v_dim
    conv = 2 * nk * dk + nv * dv
    q4 = lambda m, n: m * (n // 256) * 144
    lin = 0
    for kind in spec.layer_kinds:
        if kind == 0:
            lin += q4(conv, H) + q4(nv * dv, H) + 2 * nv * H * 2 + q4(H, nv * dv)
        else:
            lin += q4(2 * spec.n_q * spec.head_dim + 2 * spec.n_kv * spec.head_dim, H) + q4(H, spec.n_q * spec.head_dim)
        lin += 2 * q4(I, H) + q4(H, I)
    head = V * (H // 256) * 210
    kv = step_bytes(spec, 1, CTX)
    total = lin + head + kv["kv"] + kv["state"]
    return {"workload": "C5 step, Q4_K layer linears + Q6_K lm_head (Q4_K_M mix), 32K context",
            "t1_ms": round(t1, 4), "tok_s": round(1000.0 / t1, 3), "t4_verify_ms": round(t4, 4),
            "t4_over_t1": round(t4 / t1, 4), "t1_bytes": int(total),
            "t1_GBps": round(total / t1 / 1e6, 1), "t1_frac": round(total / t1 / 1e6 / PEAK_GBS, 4),
            "batch4_step_ms": round(tb4, 4), "batch4_tok_s": round(4000.0 / tb4, 3),
            "batch8_step_ms": round(tb8, 4), "batch8_tok_s": round(8000.0 / tb8, 3),
            "batch16_step_ms": round(tb16, 4), "batch16_tok_s": round(16000.0 / tb16, 3),
            "prefill_tokens": PF_TOKENS, "prefill_ms": round(pf_s * 1e3, 1),
            "prefill_tok_s": round(PF_TOKENS / pf_s, 1),
            "prefill_speedup_vs_verify_chunks": round((PF_TOKENS / pf_s) / (4000.0 / t4), 2)}


def measure_wide_batch(spec, K, W):
    """Continuous batches of 8 and 16 sequences at 32K context each (block-FP8): one
    step advances every slot by one token; the engine runs the slots in groups of 8
    rows, one weight pass per group."""
    from rapidllm_amd.engine import Engine

    eng = Engine(spec, None, ctx=CTX + 4096, max_T=4, seed=1234, max_batch=16)
    out = {}
    for B in (8, 16):
        eng.synthetic_context(CTX)
        eng.replicate_slot0(B)
        eng.time_batch(B, W)
        tb = eng.time_batch(B, K) / K
        out[f"batch{B}_step_ms"] = round(tb, 4)
        out[f"batch{B}_tok_s"] = round(1000.0 * B / tb, 3)
    eng.close()
    return out


def graph_breakdown(eng, spec, steps, iters=20):
    """Where the graph-replayed step's time goes: one DeltaNet layer, one attention
    layer (at the synthetic context), layer 0 (whose input is not a folded norm) and
    the step's head and tail (embedding, first norm, lm_head, argmax, acceptance),
    each recorded as a graph of its own launches and replayed `iters` times; their
    sum over the step's layers against the step itself."""
    kinds = spec.layer_kinds
    d = next(i for i in range(1, len(kinds)) if kinds[i] == 0)
    a = next(i for i in range(1, len(kinds)) if kinds[i] == 1)
    n_d = sum(1 for k in kinds[1:] if k == 0)
    n_a = sum(1 for k in kinds[1:] if k == 1)
    out = {}
    for T, step_ms in steps.items():
        eng.time_layer(d, T, 3)
        us = {name: eng.time_layer(i, T, iters) * 1e3
              for name, i in (("delta_layer", d), ("attn_layer", a), ("layer0", 0), ("ends", spec.n_layers))}
        total = us["layer0"] + n_d * us["delta_layer"] + n_a * us["attn_layer"] + us["ends"]
        out[f"t{T}"] = {**{k + "_us": round(v, 2) for k, v in us.items()},
                        "layers_sum_ms": round(total / 1e3, 4), "step_ms": round(step_ms, 4)}
    return out


def step_bytes(spec, T, ctx):
    """Algorithmic HBM bytes of one T-token step: every weight byte once, KV read
    once (+ the T new rows written), recurrent state read once and written once per
    token (rollback snapshots), plus activations in/out of each linear."""
    H, I, V = spec.hidden, spec.intermediate, spec.vocab
    nk, nv, dk, dv = spec.n_k_heads, spec.n_v_heads, spec.k_dim, spec.v_dim
    nq, nkv, hd = spec.n_q, spec.n_kv, spec.head_dim
    conv = spec.conv_dim
    n_d = sum(1 for k in spec.layer_kinds if k == 0)
    n_a = spec.n_layers - n_d

    def fp8(m, n):
        return m * n + 4 * ((m + 127) // 128) * ((n + 127) // 128) + 4 * T * (m + n)

    lin = 0
    lin += n_d * (fp8(conv + nv * dv + 2 * nv, H) + fp8(H, nv * dv))
    lin += n_a * (fp8(2 * nq * hd + 2 * nkv * hd, H) + fp8(H, nq * hd))
    lin += spec.n_layers * (fp8(2 * I, H) + fp8(H, I))
    head = V * H * 2 + 4 * T * (V + H)
    kv = n_a * (2 * nkv * hd * 2 * (ctx + T))
    state = n_d * (nv * dk * dv * 4 * (1 + T) + conv * 4 * 4 * (1 + T))
    return {"linears": lin, "lm_head": head, "kv": kv, "state": state, "total": lin + head + kv + state}


EPI_STORE, EPI_SWIGLU, EPI_PARTIAL, EPI_ADDNORM, EPI_SWIGLU_H = 0, 2, 3, 4, 5
EPI_ADDNORM_BS = 104  # add-norm with the per-block input scale (DeltaNet out_proj)
SPLIT = 4


def gemm_shapes(spec):
    """(m, n, count per step, epilogue) of the block-FP8 GEMM launches in one step,
    as the engine issues them: fused [qkv|z|a|b] and [q|gate;k;v] stores, residual
    GEMMs adding into x with the next RMSNorm's fragments and sums of squares,
    gate/up in half tiles with the SwiGLU epilogue.  The GEMMs reading the residual
    stream (n = hidden) fold its RMSNorm (input sums of squares); the DeltaNet
    out_proj scales each 128-column input block by the head's gated-RMSNorm
    factor."""
    H, I = spec.hidden, spec.intermediate
    nv, dv = spec.n_v_heads, spec.v_dim
    nq, nkv, hd = spec.n_q, spec.n_kv, spec.head_dim
    n_d = sum(1 for k in spec.layer_kinds if k == 0)
    n_a = spec.n_layers - n_d
    a16 = lambda v: (v + 15) // 16 * 16
    m_in = a16(spec.conv_dim) + a16(nv * dv) + 2 * a16(nv)
    return [
        (m_in, H, n_d, EPI_STORE), (H, nv * dv, n_d, EPI_ADDNORM_BS if dv == 128 else EPI_ADDNORM),
        (2 * nq * hd + 2 * nkv * hd, H, n_a, EPI_STORE), (H, nq * hd, n_a, EPI_ADDNORM),
        (2 * I, H, spec.n_layers, EPI_SWIGLU_H), (H, I, spec.n_layers, EPI_ADDNORM),
    ]


def valu_compare(iters=30, rotate_bytes=768 << 20):
    """T=1 block-FP8 GEMV: the matrix-core kernel (rl_hip_time_gemm_fp8, store) and a
    VALU dot-product kernel over the same weight layout (rl_hip_time_gemv_fp8_valu:
    e4m3 -> fp32 conversions, FMAs, shuffle sums), weights cold in HBM, best of 3."""
    import ctypes as C

    from rapidllm_amd import ops, synth
    from rapidllm_amd.hip import DeviceBuffer, call

    r = synth.rng(3)
    s = C_stream()
    out = []
    for m, n in ((16480, 5120), (14336, 5120), (34816, 5120)):
        lin = ops.Fp8Linear(synth.fp8_weight(r, m, n), synth.fp8_scales(r, m, n, 1e-3, 1e-2))
        nb = lin.w.nbytes
        copies = [lin.w] + [DeviceBuffer(nb) for _ in range(max(1, -(-rotate_bytes // nb)) - 1)]
        for c in copies[1:]:
            call("rl_hip_memcpy_d2d", c.ptr, lin.w.ptr, nb, s)
        ptrs = (C.c_void_p * len(copies))(*[c.ptr for c in copies])
        X = r.standard_normal((1, n)).astype(np.float32)
        xd = DeviceBuffer.from_numpy(X)
        frag = ops.act_frag_buffer(n, 1)
        call("rl_hip_pack_act", xd.ptr, frag.ptr, n, 1, s)
        yd = DeviceBuffer(4 * m)
        ms = C.c_float()
        best = {"mfma": 1e9, "valu": 1e9}
        for _ in range(3):
            call("rl_hip_time_gemm_fp8", ptrs, len(copies), lin.ts.ptr, frag.ptr, yd.ptr, None, None, None, None, None,
                 m, n, 1, EPI_STORE, 1, iters, s, C.byref(ms))
            best["mfma"] = min(best["mfma"], ms.value * 1e3)
            call("rl_hip_time_gemv_fp8_valu", ptrs, len(copies), lin.ts.ptr, xd.ptr, yd.ptr, m, n, iters, s,
                 C.byref(ms))
            best["valu"] = min(best["valu"], ms.value * 1e3)
        out.append({"m": m, "n": n, "mfma_us": round(best["mfma"], 2), "valu_us": round(best["valu"], 2),
                    "mfma_GBps": round(nb / best["mfma"] / 1e3, 1), "valu_GBps": round(nb / best["valu"] / 1e3, 1)})
        del lin, copies
    return out


def measure_gemm(spec, T, iters=30, rotate_bytes=768 << 20):
    """Average duration of the block-FP8 GEMM over the step's launch mix: per shape,
    `iters` back-to-back launches from C++ (rl_hip_time_gemm_fp8: HIP events on the
    launch stream around the loop), each with the epilogue the step uses.

    Each shape cycles through enough copies of its packed weight (>= rotate_bytes,
    three times the 256 MB Infinity Cache) that every launch reads its weight from
    HBM, as in the decode step; the cache-resident figure (one copy re-read) is
    reported beside it as "warm_us"."""
    import ctypes as C

    from rapidllm_amd import hip, ops, synth
    from rapidllm_amd.hip import DeviceBuffer, call

    r = synth.rng(5)
    tot_ms = tot_bytes = 0.0
    n_launch = 0
    per = []
    s = C_stream()
    for m, n, count, epi_kind in gemm_shapes(spec):
        block_scale = epi_kind == EPI_ADDNORM_BS
        epi = EPI_ADDNORM if block_scale else epi_kind
        if epi == EPI_SWIGLU_H:
            lin = ops.Fp8GateUp(synth.fp8_weight(r, m // 2, n), synth.fp8_scales(r, m // 2, n),
                                synth.fp8_weight(r, m // 2, n), synth.fp8_scales(r, m // 2, n))
        else:
            lin = ops.Fp8Linear(synth.fp8_weight(r, m, n), synth.fp8_scales(r, m, n))
        nb = lin.w.nbytes
        copies = [lin.w] + [DeviceBuffer(nb) for _ in range(max(1, -(-rotate_bytes // nb)) - 1)]
        for c in copies[1:]:
            call("rl_hip_memcpy_d2d", c.ptr, lin.w.ptr, nb, s)
        X = r.standard_normal((T, n)).astype(np.float32)
        xd = DeviceBuffer.from_numpy(X)
        frag = ops.act_frag_buffer(n, T)
        yd = DeviceBuffer(4 * T * m * SPLIT)
        fo = ops.act_frag_buffer(m // 2 if epi == EPI_SWIGLU_H else m, T) if epi in (EPI_SWIGLU_H, EPI_ADDNORM) else None
        gam = DeviceBuffer.from_numpy(np.zeros(m, np.float32))
        G = hip.lib().rl_hip_norm_group_rows()
        ssq = DeviceBuffer(4 * T * ((m + G - 1) // G))
        bss = DeviceBuffer.from_numpy(np.full((n // 128) * T * 4, 32.0, np.float32)) if block_scale else None
        folded = epi in (EPI_STORE, EPI_SWIGLU_H) and n == spec.hidden
        ssi = DeviceBuffer.from_numpy(np.full((n + G - 1) // G * T, 32.0 * G / 32, np.float32)) if folded else None
        yd.zero(s)
        call("rl_hip_pack_act", xd.ptr, frag.ptr, n, T, s)
        ptrs = (C.c_void_p * len(copies))(*[c.ptr for c in copies])
        one = (C.c_void_p * 1)(lin.w.ptr)
        ms, warm = C.c_float(), C.c_float()
        args = (lin.ts.ptr, frag.ptr, yd.ptr, fo.ptr if fo else None, gam.ptr, ssq.ptr, bss.ptr if bss else None,
                ssi.ptr if ssi else None, m, n, T, epi, SPLIT)
        call("rl_hip_time_gemm_fp8", ptrs, len(copies), *args, len(copies), s, C.byref(ms))  # warm-up
        call("rl_hip_time_gemm_fp8", ptrs, len(copies), *args, iters, s, C.byref(ms))
        call("rl_hip_time_gemm_fp8", one, 1, *args, iters, s, C.byref(warm))
        ms, warm = ms.value, warm.value
        b = m * n + 4 * ((m + 127) // 128) * ((n + 127) // 128) + 4 * T * (m + n)
        label = {0: "store", 5: "swiglu", 3: f"split{SPLIT}", 4: "add+norm", 104: "add+norm+block-scale"}[epi_kind]
        per.append({"m": m, "n": n, "epilogue": label,
                    "per_step": count, "us": round(ms * 1e3, 2), "GBps": round(b / ms / 1e6, 1),
                    "warm_us": round(warm * 1e3, 2), "copies": len(copies)})
        tot_ms += ms * count
        tot_bytes += b * count
        n_launch += count
        del lin, xd, frag, yd, fo, gam, ssq, bss, ssi, copies
    avg_ms = tot_ms / n_launch
    avg_bytes = tot_bytes / n_launch
    return avg_ms, avg_bytes, per


def measure_configs(spec, gemm_t1, gemm_t4, iters=30, rotate_bytes=768 << 20):
    """Per-config kernel lines, each on weights / states read
    from HBM (rotated over >= rotate_bytes), timed with HIP events around
    back-to-back launches from C++.  `gemm_t1` / `gemm_t4` are measure_gemm's
    per-shape results at T=1 / T=4."""
    import ctypes as C

    from rapidllm_amd import ops, synth
    from rapidllm_amd.hip import DeviceBuffer, call

    s = C_stream()
    r = synth.rng(11)
    out = {}

    def frac(b, us):
        return round(b / us / 1e3 / PEAK_GBS, 4)

    # C1: one block-FP8 GEMV, W [17408 x 5120], T = 1
    m, n = 17408, 5120
    W = synth.fp8_weight(r, m, n)
    lin = ops.Fp8Linear(W, synth.fp8_scales(r, m, n))
    nb = lin.w.nbytes
    copies = [lin.w] + [DeviceBuffer(nb) for _ in range(max(1, -(-rotate_bytes // nb)) - 1)]
    for c in copies[1:]:
        call("rl_hip_memcpy_d2d", c.ptr, lin.w.ptr, nb, s)
    xd = DeviceBuffer.from_numpy(r.standard_normal((1, n)).astype(np.float32))
    frag = ops.act_frag_buffer(n, 1)
    yd = DeviceBuffer(4 * m)
    call("rl_hip_pack_act", xd.ptr, frag.ptr, n, 1, s)
    ptrs = (C.c_void_p * len(copies))(*[c.ptr for c in copies])
    ms = C.c_float()
    args = (lin.ts.ptr, frag.ptr, yd.ptr, None, None, None, None, None, m, n, 1, EPI_STORE, SPLIT)
    call("rl_hip_time_gemm_fp8", ptrs, len(copies), *args, len(copies), s, C.byref(ms))
    call("rl_hip_time_gemm_fp8", ptrs, len(copies), *args, iters, s, C.byref(ms))
    b = m * n + 4 * ((m + 127) // 128) * ((n + 127) // 128) + 4 * (m + n)
    us = ms.value * 1e3
    out["c1_fp8_gemv_17408x5120_t1"] = {"us": round(us, 2), "bytes": b, "GBps": round(b / us / 1e3, 1),
                                        "frac": frac(b, us)}
    del lin, copies, xd, frag, yd, ptrs

    # C2: GGUF Q4_K / Q6_K GEMV, W [5120 x 17408], T = 1 (and T = 4, 8)
    m, n = 5120, 17408
    for name, qt, gen, bb in (("q4_k", ops.Q4_K, synth.q4k_blocks, 144), ("q6_k", ops.Q6_K, synth.q6k_blocks, 210)):
        lin = ops.KQuantLinear(qt, gen(r, m, n), m, n)
        nb = lin.w.nbytes
        copies = [lin.w] + [DeviceBuffer(nb) for _ in range(max(1, -(-rotate_bytes // nb)) - 1)]
        for c in copies[1:]:
            call("rl_hip_memcpy_d2d", c.ptr, lin.w.ptr, nb, s)
        ptrs = (C.c_void_p * len(copies))(*[c.ptr for c in copies])
        res = {}
        for T in (1, 4, 8):
            xd = DeviceBuffer.from_numpy(r.standard_normal((T, n)).astype(np.float32))
            yd = DeviceBuffer(4 * T * m)
            ws = ops.kquant_workspace(m, n, T)
            targs = (qt, ptrs, len(copies), xd.ptr, yd.ptr, ws.ptr, ws.nbytes, m, n, T)
            call("rl_hip_time_gemm_kquant", *targs, len(copies), s, C.byref(ms))
            call("rl_hip_time_gemm_kquant", *targs, iters, s, C.byref(ms))
            b = m * (n // 256) * bb + 4 * T * (m + n)
            us = ms.value * 1e3
            res[f"t{T}"] = {"us": round(us, 2), "bytes": b, "GBps": round(b / us / 1e3, 1), "frac": frac(b, us)}
        out[f"c2_{name}_gemv_5120x17408"] = res
        del lin, copies, ptrs

    # C3: one layer's block-FP8 linear set at T = 4 (DeltaNet in_proj, q|gate;k;v,
    # o, gate/up, down): gemm_shapes entries 0, 2, 3, 4, 5 (1 is the DeltaNet
    # out_proj, not in the set)
    res = {}
    for T, per in ((1, gemm_t1), (4, gemm_t4)):
        us = b = 0.0
        for sh in (per[i] for i in (0, 2, 3, 4, 5)):
            us += sh["us"]
            b += sh["m"] * sh["n"] + 4 * ((sh["m"] + 127) // 128) * ((sh["n"] + 127) // 128) + \
                4 * T * (sh["m"] + sh["n"])
        res[f"t{T}"] = {"us": round(us, 2), "bytes": int(b), "GBps": round(b / us / 1e3, 1), "frac": frac(b, us)}
    res["t4_over_t1"] = round(res["t4"]["us"] / res["t1"]["us"], 4)
    out["c3_fp8_linear_set"] = res

    # C4: Gated DeltaNet recurrent decode, T = 4, over 48 layer states
    T, nk, nv, dk, dv, K = 4, spec.n_k_heads, spec.n_v_heads, spec.k_dim, spec.v_dim, spec.conv_k
    conv = spec.conv_dim
    n_d = sum(1 for k in spec.layer_kinds if k == 0)
    Ss = [DeviceBuffer.from_numpy((0.02 * r.standard_normal(nv * dk * dv)).astype(np.float32)) for _ in range(n_d)]
    ld = conv + 2 * nv
    qkv = DeviceBuffer.from_numpy(r.standard_normal((T, ld)).astype(np.float32))
    A_log = DeviceBuffer.from_numpy(r.standard_normal(nv).astype(np.float32))
    dt_b = DeviceBuffer.from_numpy(r.standard_normal(nv).astype(np.float32))
    cw = DeviceBuffer.from_numpy((0.5 * r.standard_normal(conv * K)).astype(np.float32))
    cin = DeviceBuffer.from_numpy(r.standard_normal(conv * K).astype(np.float32))
    cout = DeviceBuffer(4 * conv * K)
    o = DeviceBuffer(4 * T * nv * dv)
    sp = (C.c_void_p * n_d)(*[x.ptr for x in Ss])
    gargs = (sp, n_d, qkv.ptr, qkv.ptr + 4 * conv, qkv.ptr + 4 * (conv + nv), ld, A_log.ptr, dt_b.ptr, cw.ptr,
             cin.ptr, cout.ptr, o.ptr, T, nk, nv, dk, dv, K, 0)
    call("rl_hip_time_gdn", *gargs, 1, s, C.byref(ms))
    call("rl_hip_time_gdn", *gargs, 5, s, C.byref(ms))
    us = ms.value * 1e3
    b = 2 * nv * dk * dv * 4 + 2 * conv * K * 4 + 4 * T * (ld + nv * dv)
    out["c4_deltanet_t4_per_layer"] = {"us": round(us, 2), "bytes": b, "GBps": round(b / us / 1e3, 1),
                                       "frac": frac(b, us), "layers": n_d,
                                       "all_layers_us": round(us * n_d, 1)}
    del Ss
    return out


def cpu_configs(spec, budget_s=6.0):
    """The reference CPU path for configs 1, 2 and 4 on the host cores, timed in the
    same run (oracle/_ref: the reference's own compiled ops; the oracle restatement,
    kind "port", where they were not built).  Median of up to 3 runs per line."""
    from oracle import oracle as O
    from rapidllm_amd import synth

    R = O.ref()
    kind = "reference" if R is not None else "port"
    threads = int(R.ref_num_threads()) if R is not None else 1
    r = synth.rng(21)
    out = {}

    def med(fn):
        ts = []
        t_end = time.time() + budget_s
        while time.time() < t_end and len(ts) < 3:
            t = time.perf_counter()
            fn()
            ts.append(time.perf_counter() - t)
        return float(np.median(ts)) * 1e6, len(ts)

    # C1: ops::gemv_fp8 (scalar, one thread: the reference's only FP8 CPU GEMV)
    m, n = 17408, 5120
    W, sc = synth.fp8_weight(r, m, n), synth.fp8_scales(r, m, n)
    x = r.standard_normal(n).astype(np.float32)
    y = np.empty(m, np.float32)
    if R is not None:
        us, k = med(lambda: R.ref_gemv_fp8(O.P(W, O._u8), O.P(sc), O.P(x), O.P(y), m, n))
    else:
        us, k = med(lambda: O.gemv_fp8(W, sc, x))
    out["c1"] = {"us": round(us, 1), "cores": 1, "kind": kind, "runs": k, "what": "ops::gemv_fp8 17408x5120"}
    del W
    # C2: ops::gemv_q4_k / gemv_q6_k (row-parallel over the reference WorkerPool)
    m, n = 5120, 17408
    x = r.standard_normal(n).astype(np.float32)
    y = np.empty(m, np.float32)
    for name, gen, fr, fo in (("q4_k", synth.q4k_blocks, "ref_gemv_q4_k", O.gemv_q4_k),
                              ("q6_k", synth.q6k_blocks, "ref_gemv_q6_k", O.gemv_q6_k)):
        blk = np.ascontiguousarray(gen(r, m, n)).reshape(-1)
        if R is not None:
            f = getattr(R, fr)
            us, k = med(lambda: f(O.P(blk, O._u8), O.P(x), O.P(y), m, n))
            cores = threads
        else:
            us, k = med(lambda: fo(blk, x, m, n, 8))
            cores = 8
        out[f"c2_{name}"] = {"us": round(us, 1), "cores": cores, "kind": kind, "runs": k,
                             "what": f"ops::gemv_{name} 5120x17408"}
    # C4: per token conv1d_update over the 10240 channels + the delta-rule step over
    # 48 heads (ops::delta_recurrent_step_simd), 4 tokens, one layer; x 48 layers
    nv, dk, dv, conv, K = spec.n_v_heads, spec.k_dim, spec.v_dim, spec.conv_dim, spec.conv_k
    S = (0.02 * r.standard_normal(nv * dk * dv)).astype(np.float32)
    st = r.standard_normal(conv * K).astype(np.float32)
    cw = (0.5 * r.standard_normal(conv * K)).astype(np.float32)
    xs = r.standard_normal((4, conv)).astype(np.float32)
    q = r.standard_normal((4, nv * dk)).astype(np.float32)
    kk = r.standard_normal((4, nv * dk)).astype(np.float32)
    v = r.standard_normal((4, nv * dv)).astype(np.float32)
    beta = (1 / (1 + np.exp(-r.standard_normal((4, nv))))).astype(np.float32)
    gl = (-np.log1p(np.exp(r.standard_normal((4, nv))))).astype(np.float32)
    ycv = np.empty(conv, np.float32)
    o = np.empty(nv * dv, np.float32)

    def layer_ref():
        for t in range(4):
            R.ref_conv1d_update(O.P(xs[t]), O.P(cw), O.P(st), O.P(ycv), conv, K)
            R.ref_delta_step_simd(O.P(S), O.P(q[t]), O.P(kk[t]), O.P(v[t]), O.P(beta[t]), O.P(gl[t]), O.P(o), nv, dk,
                                  dv, 1e-6)

    def layer_port():
        Sm = S.reshape(nv, dk, dv).copy()
        stm = st.reshape(conv, K).copy()
        for t in range(4):
            O.conv1d_update(xs[t], cw.reshape(conv, K), stm)
            O.delta_step(Sm, q[t].reshape(nv, dk), kk[t].reshape(nv, dk), v[t].reshape(nv, dv), beta[t], gl[t])

    us, k = med(layer_ref if R is not None else layer_port)
    n_d = sum(1 for kd in spec.layer_kinds if kd == 0)
    out["c4"] = {"us_per_layer": round(us, 1), "all_layers_us": round(us * n_d, 1),
                 "cores": threads if R is not None else 1, "kind": kind, "runs": k,
                 "what": "4 x (ops::conv1d_update 10240 ch + ops::delta_recurrent_step_simd 48 heads) per layer"}
    out["host"] = host_info(R)
    return out


_stream = None


def C_stream():
    global _stream
    if _stream is None:
        import ctypes as C
        from rapidllm_amd.hip import call
        p = C.c_void_p()
        call("rl_hip_stream_create", C.byref(p))
        _stream = p.value
    return _stream


def copy_probe(mib, reps=10):
    """A plain 16-byte-vector device copy of known size: the scale for the
    FETCH_SIZE / WRITE_SIZE counters (each copy reads and writes mib MiB once)."""
    from rapidllm_amd.hip import DeviceBuffer, Timer, call

    n = mib << 20
    a, b = DeviceBuffer(n), DeviceBuffer(n)
    s = C_stream()
    call("rl_hip_memset", a.ptr, 1, n, s)
    tm = Timer(s)
    tm.start()
    for _ in range(reps):
        call("rl_hip_copy_probe", a.ptr, b.ptr, n, s)
    ms = tm.stop() / reps
    print(json.dumps({"copy_bytes_each_way": n, "us": round(ms * 1e3, 2), "GBps_rd_plus_wr": round(2 * n / ms / 1e6, 1)}))


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "gemm_fp8_t1_mix_traffic.txt")


def measured_traffic():
    """HBM bytes per launch of the roofline kernel, from the committed counter
    summary (rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE, scaled by the copy kernel)."""
    try:
        for line in open(TRAFFIC_FILE):
            if line.startswith("traffic_bytes_per_launch"):
                return int(float(line.split("=")[1]))
    except OSError:
        pass
    return None


def host_info(R=None):
    """The host the CPU lines ran on: logical CPUs (and those this process may use),
    the CPU model string, and the SIMD path the reference's runtime dispatch picked
    (cpu_caps.cpp: AVX-512 F/DQ/BW/VL, else AVX2 + FMA, else scalar)."""
    import ctypes as C

    model, flags = "unknown", set()
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name") and model == "unknown":
                    model = line.split(":", 1)[1].strip()
                elif line.startswith("flags") and not flags:
                    flags = set(line.split(":", 1)[1].split())
    except OSError:
        pass
    if R is not None:
        R.ref_simd_name.restype = C.c_char_p
        isa = R.ref_simd_name().decode()
    else:
        isa = ("avx512f+dq+bw+vl" if {"avx512f", "avx512dq", "avx512bw", "avx512vl"} <= flags
               else "avx2+fma" if {"avx2", "fma"} <= flags else "scalar") + " (from /proc/cpuinfo)"
    return {"nproc": os.cpu_count(), "usable_cpus": len(os.sched_getaffinity(0)), "cpu_model": model,
            "reference_isa": isa}


def cpu_baseline(spec, sbytes_total, ctx=None, budget_s=25.0):
    """The reference's own CPU decode path (oracle/_ref, ops_fused.cpp), one layer of
    each kind at the 27B shape, timed once each (and again while the budget lasts,
    keeping the fastest): fused_delta_decode (block-FP8 in_proj / out_proj, the
    recurrent update), fused_attn_decode at the step's context (FP8 projections,
    attention over an fp32 cache of ctx positions), fused_mlp_decode (three FP8
    GEMVs), and the bf16 lm_head GEMV.  The step is 48 / 16 / 64 / 1 of them
    (session.cpp:325-411, 531-559).  The reference runs gemv_fp8 and attn_decode on
    one thread (scalar loops, ops.cpp:182-194, 575-605) and gemv_bf16 and the
    recurrent step on its WorkerPool (cpu_caps.cpp:123-131, 260-263); `cores` is
    that pool's size.  Without the reference objects the MLP alone is timed on the
    oracle restatement and scaled by bytes (kind "port")."""
    from oracle import oracle as O
    from rapidllm_amd import synth

    ctx = ctx or CTX
    H, I = spec.hidden, spec.intermediate
    nk, nv, dk, dv = spec.n_k_heads, spec.n_v_heads, spec.k_dim, spec.v_dim
    nq, nkv, hd = spec.n_q, spec.n_kv, spec.head_dim
    r = synth.rng(9)

    def lin(m, n):
        w = synth.fp8_weight_wide(r, m, n) if m * n >= 1 << 26 else synth.fp8_weight(r, m, n)
        return w, synth.fp8_scales(r, m, n)

    def vec(n, mean=0.0, sd=0.1):
        return (mean + sd * r.standard_normal(n)).astype(np.float32)

    wg, wu, wd = lin(I, H), lin(I, H), lin(H, I)
    gam = vec(H)
    x0 = r.standard_normal(H).astype(np.float32)
    R = O.ref()
    if R is None:
        times = []
        t_end = time.time() + budget_s
        while time.time() < t_end and len(times) < 3:
            x = x0.copy()
            t = time.perf_counter()
            xn = O.qwen3_rmsnorm(x, gam)
            g = O.gemv_fp8(wg[0], wg[1], xn)
            u = O.gemv_fp8(wu[0], wu[1], xn)
            h = (g / (1 + np.exp(-g.astype(np.float64))) * u).astype(np.float32)
            x += O.gemv_fp8(wd[0], wd[1], h)
            times.append(time.perf_counter() - t)
        t_m = float(min(times))
        mlp_bytes = 3 * H * I
        return {"value": round(mlp_bytes / (t_m * sbytes_total), 6), "unit": "tok/s", "cores": 1, "kind": "port",
                "host": host_info(None),
                "sample": f"oracle restatement of fused_mlp_decode (one 27B MLP layer, {t_m:.2f} s), scaled by "
                          f"bytes to the {sbytes_total/1e9:.2f} GB step"}
    P, u8 = O.P, O._u8
    conv_dim = 2 * nk * dk + nv * dv
    # DeltaNet layer
    dq, dz, da, db, do = lin(conv_dim, H), lin(nv * dv, H), lin(nv, H), lin(nv, H), lin(H, nv * dv)
    A_log, dt_bias, gnorm = vec(nv, 0, 0.5), vec(nv, 0, 0.5), vec(dv, 1.0, 0.1)
    conv_w = vec(conv_dim * spec.conv_k, 0, 0.5)
    S0 = (0.02 * r.standard_normal(nv * dk * dv)).astype(np.float32)
    cs0 = r.standard_normal(conv_dim * spec.conv_k).astype(np.float32)
    # attention layer: projections and a cache of ctx positions (fp32, as the CPU path keeps it)
    aq, ak, av, ao = lin(2 * nq * hd, H), lin(nkv * hd, H), lin(nkv * hd, H), lin(H, nq * hd)
    qn, kn = vec(hd), vec(hd)
    kc = np.zeros((ctx + 1) * nkv * hd, np.float32)
    vc = np.zeros_like(kc)
    kc[: ctx * nkv * hd] = r.standard_normal(ctx * nkv * hd, dtype=np.float32)
    vc[: ctx * nkv * hd] = r.standard_normal(ctx * nkv * hd, dtype=np.float32)
    lm = synth.bf16_random_bits(r, spec.vocab, H)
    logits = np.empty(spec.vocab, np.float32)

    def t_delta():
        x, S, cs = x0.copy(), S0.copy(), cs0.copy()
        t = time.perf_counter()
        R.ref_fused_delta(P(gam), P(dq[0], u8), P(dq[1]), P(dz[0], u8), P(dz[1]), P(da[0], u8), P(da[1]),
                          P(db[0], u8), P(db[1]), P(do[0], u8), P(do[1]), P(A_log), P(dt_bias), P(conv_w), P(gnorm),
                          P(S), P(cs), P(x), H, nk, nv, dk, dv, spec.conv_k, dv, spec.rms_eps)
        return time.perf_counter() - t

    def t_attn():
        x = x0.copy()
        t = time.perf_counter()
        R.ref_fused_attn(P(gam), P(aq[0], u8), P(aq[1]), P(ak[0], u8), P(ak[1]), P(av[0], u8), P(av[1]),
                         P(ao[0], u8), P(ao[1]), P(qn), P(kn), P(kc), P(vc), P(x), H, nq, nkv, hd,
                         spec.rotary_dim, ctx, spec.rope_theta, spec.rms_eps)
        return time.perf_counter() - t

    def t_mlp():
        x = x0.copy()
        t = time.perf_counter()
        R.ref_fused_mlp(P(gam), P(wg[0], u8), P(wg[1]), P(wu[0], u8), P(wu[1]), P(wd[0], u8), P(wd[1]), P(x), H, I,
                        spec.rms_eps)
        return time.perf_counter() - t

    def t_head():
        t = time.perf_counter()
        R.ref_gemv_bf16(P(lm, O._u16), P(x0), P(logits), spec.vocab, H)
        return time.perf_counter() - t

    parts = {"delta": t_delta, "attn": t_attn, "mlp": t_mlp, "lm_head": t_head}
    best = {k: f() for k, f in parts.items()}
    t_end = time.time() + budget_s - sum(best.values())
    while time.time() + sum(best.values()) < t_end:
        for k, f in parts.items():
            best[k] = min(best[k], f())
    n_d = sum(1 for k in spec.layer_kinds if k == 0)
    n_a = spec.n_layers - n_d
    step_s = n_d * best["delta"] + n_a * best["attn"] + spec.n_layers * best["mlp"] + best["lm_head"]
    return {"value": round(1.0 / step_s, 6), "unit": "tok/s", "cores": int(R.ref_num_threads()), "kind": "reference",
            "host": host_info(R),
            "step_s": round(step_s, 2),
            "per_layer_s": {k: round(v, 4) for k, v in best.items()},
            "sample": f"one 27B layer of each kind through the reference's fused CPU decode functions "
                      f"(fused_delta_decode {best['delta']:.3f} s, fused_attn_decode at {ctx} positions "
                      f"{best['attn']:.3f} s, fused_mlp_decode {best['mlp']:.3f} s) and the bf16 lm_head GEMV "
                      f"({best['lm_head']:.3f} s), fastest of repeated runs; step = {n_d} x delta + {n_a} x attn + "
                      f"{spec.n_layers} x mlp + lm_head = {step_s:.1f} s; the FP8 GEMVs and the attention are "
                      f"single-threaded in the reference, gemv_bf16 and the recurrent step use its worker pool"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--layers", type=int, default=64)
    ap.add_argument("--gemm-only", action="store_true",
                    help="time only the block-FP8 GEMM launch mix (the roofline kernel), for counter runs")
    ap.add_argument("--gemm-tokens", type=int, default=1, help="tokens per GEMM launch with --gemm-only (1..4)")
    ap.add_argument("--valu-compare", action="store_true",
                    help="time only the T=1 FP8 GEMV on the matrix cores against a VALU dot-product kernel")
    ap.add_argument("--prefill-only", type=int, default=0,
                    help="time only a prompt prefill of this many tokens (for kernel traces)")
    ap.add_argument("--configs-only", action="store_true",
                    help="run only the per-config kernel lines (configs 1-4), for kernel traces")
    ap.add_argument("--batch-only", type=int, nargs="?", const=4, default=0,
                    help="time only the batch decode step of this many slots (default 4; C5, 32K context "
                         "per slot)")
    ap.add_argument("--step-only", action="store_true",
                    help="time only the T=1 decode and T=4 verify steps (for kernel traces and A/B runs)")
    ap.add_argument("--copy-probe-mb", type=int, default=0,
                    help="run only a plain device copy of this many MiB (counter calibration)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the decode path is single-GPU; see DESIGN.md for how it would shard)", file=sys.stderr)
        sys.exit(2)

    from rapidllm_amd import hip
    from rapidllm_amd.engine import MTP_LAYER, MTP_STEM, Engine
    from rapidllm_amd.model import ModelSpec

    hip.require_gpu()
    spec = ModelSpec(n_layers=args.layers)
    if args.copy_probe_mb:
        copy_probe(args.copy_probe_mb)
        return
    if args.valu_compare:
        print(json.dumps({"t1_gemv_fp8_mfma_vs_valu": valu_compare()}))
        return
    if args.gemm_only:
        g_ms, g_bytes, per = measure_gemm(spec, args.gemm_tokens, iters=args.steps)
        print(json.dumps({"avg_launch_us": round(g_ms * 1e3, 2), "bytes_per_launch": int(g_bytes), "shapes": per}))
        return
    if args.configs_only:
        _, _, per1 = measure_gemm(spec, 1)
        _, _, per4 = measure_gemm(spec, 4)
        cfg = measure_configs(spec, per1, per4)
        if not args.no_cpu:
            cfg["cpu"] = cpu_configs(spec)
        print(json.dumps(cfg))
        return
    if args.prefill_only:
        eng = Engine(spec, None, ctx=max(CTX, args.prefill_only) + 4096, max_T=4, seed=1234)
        ids = np.random.default_rng(3).integers(0, spec.vocab, args.prefill_only).astype(np.int32)
        eng.prefill(ids[:600])
        t0 = time.perf_counter()
        eng.prefill(ids)
        pf_s = time.perf_counter() - t0
        eng.close()
        print(json.dumps({"prefill_tokens": args.prefill_only, "prefill_ms": round(pf_s * 1e3, 1),
                          "prefill_tok_s": round(args.prefill_only / pf_s, 1)}))
        return
    if args.step_only:
        eng = Engine(spec, None, ctx=CTX + 4096, max_T=4, seed=1234)
        res = {}
        for T in (1, 4):
            eng.synthetic_context(CTX)
            eng.time_steps(T, args.warmup)
            res[f"t{T}_ms"] = round(eng.time_steps(T, args.steps) / args.steps, 4)
        eng.close()
        print(json.dumps(res))
        return
    if args.batch_only:
        B = args.batch_only
        eng = Engine(spec, None, ctx=CTX + 4096, max_T=4, seed=1234, max_batch=B)
        eng.synthetic_context(CTX)
        eng.replicate_slot0(B)
        eng.time_batch(B, args.warmup)
        tb = eng.time_batch(B, args.steps) / args.steps
        eng.close()
        print(json.dumps({f"batch{B}_step_ms": round(tb, 4), f"batch{B}_tok_s": round(1000.0 * B / tb, 3)}))
        return
    t0 = time.time()
    eng = Engine(spec, None, ctx=CTX + 4096, max_T=4, seed=1234, max_batch=4)
    build_s = time.time() - t0
    print(f"[bench] engine built in {build_s:.1f}s, {eng.device_bytes/1e9:.2f} GB on device", file=sys.stderr,
          flush=True)

    K, W = args.steps, args.warmup
    # The headline T=1 decode is timed last: the measurements before it (about a
    # second of continuous GPU work) bring the GPU to its steady clocks, which a
    # serving loop runs at; timed from idle, the first ~1 s of steps run up to 7%
    # slower.  Its own window is still W untimed + K timed steps.
    # prompt prefill (chunked path on the prefill GEMM / attention)
    ids = np.random.default_rng(3).integers(0, spec.vocab, PF_TOKENS).astype(np.int32)
    eng.prefill(ids[:600])  # buffers and first-use costs outside the timed call
    t0 = time.perf_counter()
    eng.prefill(ids)
    pf_s = time.perf_counter() - t0
    # Steady clocks for the T=4 window too: straight after the one prompt it reads 6.9-7.05 ms,
    # a second of work later 6.7 (the timed prompt alone gave that while it took longer).
    for _ in range(4):
        eng.prefill(ids)
    # T=4 MTP verify (drafts in the token buffer; acceptance advances 1..4)
    eng.synthetic_context(CTX)
    eng.time_steps(4, W)
    t4 = eng.time_steps(4, K) / K
    # MTP stem draft of 3 tokens
    eng.synthetic_context(CTX)
    eng.time_steps(1, 1)
    eng.time_steps(1, W, mtp_drafts=3)
    tm = eng.time_steps(1, K, mtp_drafts=3) / K
    # the same with the MTP decoder layer (stem + mtp.layers[0] per draft)
    eng.set_mtp_mode(MTP_LAYER)
    eng.time_steps(1, W, mtp_drafts=3)
    tml = eng.time_steps(1, K, mtp_drafts=3) / K
    eng.set_mtp_mode(MTP_STEM)
    # continuous batch of 4 sequences at 32K context each (one weight pass per step)
    eng.synthetic_context(CTX)
    eng.replicate_slot0(4)
    eng.time_batch(4, W)
    tb4 = eng.time_batch(4, K) / K
    # T=1 decode at 32K context (the headline value)
    eng.synthetic_context(CTX)
    eng.time_steps(1, W)
    t1 = eng.time_steps(1, K) / K
    breakdown = graph_breakdown(eng, spec, {1: t1, 4: t4})
    eng.close()
    gguf = measure_gguf_step(spec, K, W)
    wide = measure_wide_batch(spec, K, W)

    b1 = step_bytes(spec, 1, CTX)
    b4 = step_bytes(spec, 4, CTX)
    g_ms, g_bytes, per = measure_gemm(spec, 1)
    _, _, per4 = measure_gemm(spec, 4)
    configs = measure_configs(spec, per, per4)
    roof = {"bound": "hbm", "kernel": "gemm_frag_kernel (block-FP8, T=1 step launch mix, weights read from HBM)",
            "achieved": round(g_bytes / g_ms / 1e6, 1), "peak": PEAK_GBS, "unit": "GB/s",
            "frac": round(g_bytes / g_ms / 1e6 / PEAK_GBS, 4), "traffic": measured_traffic(),
            "bytes_per_launch": int(g_bytes), "avg_launch_us": round(g_ms * 1e3, 2), "shapes": per}
    out = {
        "metric": METRIC,
        "value": round(1000.0 / t1, 3),
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": round(t1, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp8e4m3 x bf16(hi+mid) -> fp32",
        "data": "synthetic (random-init weights generated on device; KV prefilled N(0,1))",
        "config": {"workload": "C5: Qwen3.6-27B-shape hybrid decode step, 64 layers (48 DeltaNet + 16 gated attn), "
                               "block-FP8 linears, bf16 lm_head 248320, fp16 KV at 32768 context, batch 1",
                   "context": CTX, "layers": spec.n_layers},
        "t4_verify_ms": round(t4, 4),
        "t4_over_t1": round(t4 / t1, 4),
        "mtp_draft3_ms": round(tm, 4),
        "mtp_layer_draft3_ms": round(tml, 4),
        "spec_tok_s_full_accept": round(4000.0 / (t4 + tm), 3),
        "spec_tok_s_full_accept_layer": round(4000.0 / (t4 + tml), 3),
        "gguf_q4_k": gguf,
        "batch4_step_ms": round(tb4, 4),
        "batch4_tok_s": round(4000.0 / tb4, 3),
        **wide,
        "prefill_tokens": PF_TOKENS,
        "prefill_ms": round(pf_s * 1e3, 1),
        "prefill_tok_s": round(PF_TOKENS / pf_s, 1),
        "prefill_speedup_vs_verify_chunks": round((PF_TOKENS / pf_s) / (4000.0 / t4), 2),
        "graph_breakdown": breakdown,
        "step_roofline": {"t1_bytes": b1["total"], "t1_GBps": round(b1["total"] / t1 / 1e6, 1),
                          "t1_frac": round(b1["total"] / t1 / 1e6 / PEAK_GBS, 4),
                          "t4_bytes": b4["total"], "t4_GBps": round(b4["total"] / t4 / 1e6, 1),
                          "t4_frac": round(b4["total"] / t4 / 1e6 / PEAK_GBS, 4), "bytes_t1": b1},
        "roofline": roof,
        "configs": configs,
    }
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(spec, b1["total"])
        configs["cpu"] = cpu_configs(spec)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
