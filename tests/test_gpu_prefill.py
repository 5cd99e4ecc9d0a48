"""GPU parity of the prefill path (many prompt tokens per launch) against the CPU
oracle: block-FP8 linears on the matrix cores, 1e-3 relative L2 per token."""
import numpy as np
import pytest

from rapidllm_amd import hip, ops, synth
from rapidllm_amd.hip import DeviceBuffer, call

pytestmark = pytest.mark.gpu

REL_L2 = 1e-3


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("m,n,T", [(64, 512, 1), (300, 1000, 17), (1000, 1536, 64), (129, 640, 100),
                                   (2048, 5120, 256)])
def test_gemm_prefill_vs_oracle(gpu, orc, m, n, T):
    r = synth.rng(300 + m + n + T)
    W = synth.fp8_weight(r, m, n)
    s = synth.fp8_scales(r, m, n)
    X = r.standard_normal((T, n)).astype(np.float32)
    lin = ops.Fp8Linear(W, s)
    Y = ops.linear_prefill(lin, X)
    Yo = orc.gemm_fp8(W, s, X)
    for t in range(T):
        assert rel_l2(Y[t], Yo[t]) <= REL_L2, (m, n, T, t, rel_l2(Y[t], Yo[t]))


@pytest.mark.parametrize("T,I", [(70, 256), (200, 520)])
def test_gemm_prefill_swiglu_half_tiles(gpu, orc, T, I):
    """Prefill SwiGLU (epilogue 5) over the engine's half-tile gate/up packing,
    gate and up with independent block scales; I = 520 ends in a partial 128-row
    scale block."""
    r = synth.rng(43 + I)
    n = 768
    Wg, Wu = synth.fp8_weight(r, I, n), synth.fp8_weight(r, I, n)
    sg, su = synth.fp8_scales(r, I, n), synth.fp8_scales(r, I, n)
    X = r.standard_normal((T, n)).astype(np.float32)
    g = orc.gemm_fp8(Wg, sg, X).astype(np.float64)
    u = orc.gemm_fp8(Wu, su, X).astype(np.float64)
    want = g / (1.0 + np.exp(-g)) * u
    got = ops.linear_prefill(ops.Fp8GateUp(Wg, sg, Wu, su), X, epilogue=5)
    for t in range(T):
        assert rel_l2(got[t], want[t]) <= REL_L2, (t, rel_l2(got[t], want[t]))


@pytest.mark.parametrize("T,I", [(70, 256), (131, 384)])
def test_gemm_prefill_swiglu_to_fragments(gpu, T, I):
    """Epilogue 6 (SwiGLU half tiles written as the next GEMM's bf16 hi + mid
    fragments) is byte-identical to epilogue 5 followed by rl_hip_pack_act."""
    from rapidllm_amd.hip import DeviceBuffer, call
    r = synth.rng(47 + I)
    n = 512
    lin = ops.Fp8GateUp(synth.fp8_weight(r, I, n), synth.fp8_scales(r, I, n), synth.fp8_weight(r, I, n),
                        synth.fp8_scales(r, I, n))
    X = r.standard_normal((T, n)).astype(np.float32)
    xd = DeviceBuffer.from_numpy(X)
    frag = ops.act_frag_buffer(n, T)
    call("rl_hip_pack_act", xd.ptr, frag.ptr, n, T, None)
    yd = DeviceBuffer(4 * T * I)
    call("rl_hip_gemm_fp8_prefill", lin.w.ptr, lin.ts.ptr, frag.ptr, yd.ptr, 2 * I, n, T, 5, I, None)
    want = ops.act_frag_buffer(I, T)
    call("rl_hip_pack_act", yd.ptr, want.ptr, I, T, None)
    got = ops.act_frag_buffer(I, T)
    call("rl_hip_gemm_fp8_prefill", lin.w.ptr, lin.ts.ptr, frag.ptr, got.ptr, 2 * I, n, T, 6, I, None)
    nb = (I // 128) * 16 * 2 * T * 16  # fragment units (block, i, g) x (hi, mid) x T x 16 B
    a = got.numpy(np.uint8, (got.nbytes,))[:nb]
    b = want.numpy(np.uint8, (want.nbytes,))[:nb]
    assert np.array_equal(a, b)


def test_gemm_prefill_add_and_swiglu(gpu, orc):
    r = synth.rng(41)
    T, n, I = 70, 768, 256
    # gate/up interleaved per 16-row tile, as the engine packs them
    Wg, Wu = synth.fp8_weight(r, I, n), synth.fp8_weight(r, I, n)
    sg, su = synth.fp8_scales(r, I, n), synth.fp8_scales(r, I, n)
    W = np.empty((2 * I, n), np.uint8)
    S = np.empty((2 * I // 128, (n + 127) // 128), np.float32)
    for b in range(I // 16):
        W[32 * b:32 * b + 16] = Wg[16 * b:16 * b + 16]
        W[32 * b + 16:32 * b + 32] = Wu[16 * b:16 * b + 16]
    X = r.standard_normal((T, n)).astype(np.float32)
    g = orc.gemm_fp8(Wg, sg, X)
    u = orc.gemm_fp8(Wu, su, X)
    want = g / (1.0 + np.exp(-g.astype(np.float64))) * u
    # the interleaved matrix's 128-row scale blocks mix gate and up rows, so pack
    # it with per-row-tile scales by building the tiles from the two halves
    lin_g, lin_u = ops.Fp8Linear(Wg, sg), ops.Fp8Linear(Wu, su)
    from rapidllm_amd.hip import DeviceBuffer, call
    L = __import__("rapidllm_amd.hip", fromlist=["lib"]).lib()
    w = DeviceBuffer(L.rl_hip_fp8_packed_bytes(2 * I, n))
    ts = DeviceBuffer(4 * L.rl_hip_fp8_tile_scales(2 * I, n))
    tile = 2048 * ((n + 127) // 128)
    nt = (n + 127) // 128
    for b in range(I // 16):
        call("rl_hip_memcpy_d2d", w.ptr + (2 * b) * tile, lin_g.w.ptr + b * tile, tile, None)
        call("rl_hip_memcpy_d2d", w.ptr + (2 * b + 1) * tile, lin_u.w.ptr + b * tile, tile, None)
        call("rl_hip_memcpy_d2d", ts.ptr + 4 * (2 * b) * nt, lin_g.ts.ptr + 4 * b * nt, 4 * nt, None)
        call("rl_hip_memcpy_d2d", ts.ptr + 4 * (2 * b + 1) * nt, lin_u.ts.ptr + 4 * b * nt, 4 * nt, None)
    xd = DeviceBuffer.from_numpy(X)
    frag = ops.act_frag_buffer(n, T)
    yd = DeviceBuffer(4 * T * I)
    call("rl_hip_pack_act", xd.ptr, frag.ptr, n, T, None)
    call("rl_hip_gemm_fp8_prefill", w.ptr, ts.ptr, frag.ptr, yd.ptr, 2 * I, n, T, 2, I, None)
    got = yd.numpy(np.float32, (T, I))
    for t in range(T):
        assert rel_l2(got[t], want[t]) <= REL_L2, t
    # add epilogue: Y0 + W . X
    Y0 = r.standard_normal((T, I)).astype(np.float32)
    got = ops.linear_prefill(lin_g, X, epilogue=1, Y0=Y0)
    for t in range(T):
        assert rel_l2(got[t], Y0[t] + g[t]) <= REL_L2, t


def test_gemm_prefill_matches_decode_gemm(gpu):
    """The prefill kernel and the decode kernel compute the same products; results
    agree to fp32 reassociation (different K-split orders)."""
    r = synth.rng(9)
    m, n, T = 512, 2048, 8
    lin = ops.Fp8Linear(synth.fp8_weight(r, m, n), synth.fp8_scales(r, m, n))
    X = r.standard_normal((T, n)).astype(np.float32)
    a = ops.linear_prefill(lin, X)
    b = ops.linear_T(lin, X)
    assert rel_l2(a, b) <= 1e-5


@pytest.mark.parametrize("T,pos,nq,nkv", [(1, 0, 24, 4), (16, 0, 24, 4), (37, 300, 24, 4), (100, 1000, 24, 4),
                                          (70, 250, 4, 2), (33, 17, 2, 2)])
def test_attn_prefill_vs_oracle(gpu, orc, T, pos, nq, nkv):
    """Causal prefill attention: every token over the cache and the earlier prompt
    tokens, against the per-token oracle (fp16 K/V as the device cache holds them)."""
    from tests.test_gpu_layers import _attn_oracle
    r = synth.rng(60 + pos + T + nq)
    hd = 256
    ctx = ((pos + T + 255) // 256) * 256 + 256
    Y = r.standard_normal((T, 2 * nq * hd + 2 * nkv * hd)).astype(np.float32)
    qn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    kn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    K = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    V = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    cache = ops.AttnCache(nkv, ctx, hd)
    if pos:
        cache.fill(K, V)
    out = ops.attn_prefill_layer(Y, cache, pos, qn, kn, nq, nkv)
    want = _attn_oracle(orc, Y, K, V, pos, qn, kn, nq, nkv)
    for t in range(T):
        assert rel_l2(out[t], want[t]) < 1e-3, (t, rel_l2(out[t], want[t]))


def test_attn_prefill_then_decode(gpu, orc):
    """K/V written by the prefill serve a following decode step: decode at the next
    position after a prefill equals the oracle over the whole sequence."""
    from tests.test_gpu_layers import _attn_oracle
    r = synth.rng(99)
    nq, nkv, hd, pos, T = 24, 4, 256, 200, 40
    ctx = 512
    Y = r.standard_normal((T + 1, 2 * nq * hd + 2 * nkv * hd)).astype(np.float32)
    qn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    kn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    K = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    V = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    cache = ops.AttnCache(nkv, ctx, hd)
    cache.fill(K, V)
    ops.attn_prefill_layer(Y[:T], cache, pos, qn, kn, nq, nkv)
    got = ops.attn_decode_layer(Y[T:], cache, pos + T, qn, kn, nq, nkv)
    want = _attn_oracle(orc, Y, K, V, pos, qn, kn, nq, nkv)
    assert rel_l2(got[0], want[T]) < 1e-3


@pytest.mark.parametrize("chunk", ["512", "2048"])
def test_engine_chunked_prefill_matches_oracle(gpu, orc, monkeypatch, chunk):
    """A 600-token prompt: two prefill chunks (512 + 84, RL_PREFILL_CHUNK=512) or one
    (the default chunk of 2048) through the chunked path,
    the last max_T tokens as a decode step; logits equal the oracle's, decoding and
    speculative generation continue exactly as from a token-by-token prefill."""
    from oracle.oracle import OracleModel
    from rapidllm_amd import model as M
    from rapidllm_amd.engine import Engine
    from tests.test_gpu_engine import margin_ok, mini_spec
    spec = mini_spec()
    W = M.random_weights(spec, seed=3, w_scale=(1e-3, 1e-2))
    monkeypatch.setenv("RL_PREFILL_CHUNK", chunk)
    eng = Engine(spec, W, ctx=1024)
    orc_m = OracleModel(spec, W, ctx=1024)
    rng = np.random.default_rng(5)
    prompt = [int(t) for t in rng.integers(0, spec.vocab, 600)]
    eng.prefill(prompt)
    orc_m.reset()
    for t in prompt:
        g, lg, hd = orc_m.decode(t)
    assert rel_l2(eng.copy_logits(), lg) < 1e-3
    assert rel_l2(eng.copy_last_hidden(), hd) < 1e-3
    if margin_ok(lg):
        assert eng.greedy() == g
    tok = g
    for _ in range(4):
        eng.decode_token(tok)
        g, lg, _ = orc_m.decode(tok)
        assert rel_l2(eng.copy_logits(), lg) < 1e-3
        tok = g
    want, _, _ = orc_m.generate(prompt, 8)
    got, _, _ = eng.generate(prompt, 8, spec_n=3)
    assert got == want


@pytest.mark.parametrize("T,nk,nv,v_tiled", [(1, 16, 48, False), (37, 16, 48, False), (200, 2, 6, True),
                                             (64, 4, 4, False)])
def test_gdn_prefill_vs_oracle(gpu, orc, T, nk, nv, v_tiled):
    """DeltaNet prefill (conv over all tokens, then the recurrence with the state in
    registers) against per-token oracle steps: outputs, final state, final window."""
    from tests.test_gpu_layers import _gdn_case, _gdn_oracle
    r = synth.rng(400 + T + nv)
    case = _gdn_case(r, T, nk, nv, v_tiled)
    o, S, conv = ops.gdn_prefill(*case, nk, nv, v_tiled)
    o_ref, S_ref, conv_ref = _gdn_oracle(orc, *case, nk, nv, v_tiled)
    for t in range(T):
        assert rel_l2(o[t], o_ref[t]) < 1e-3, (t, rel_l2(o[t], o_ref[t]))
    assert rel_l2(S, S_ref) < 1e-4
    assert np.array_equal(conv, conv_ref)


@pytest.mark.parametrize("T,decay", [(700, 0.5), (130, 6.0), (64, -3.0)])
def test_gdn_prefill_chunked_vs_per_token(gpu, orc, monkeypatch, T, decay):
    """The chunked scan (chunks of 64 tokens in WY form) and the per-token scan
    (RL_PF_GDN_CHUNK=0) against the per-token oracle over several chunks and a
    ragged last one: decay 6 makes A_log large enough that g underflows to 0 in
    fp32 on some tokens (the chunk's log-decay sums must not turn into inf - inf),
    decay -3 keeps g near 1 (little forgetting, the state carries over chunks)."""
    from tests.test_gpu_layers import _gdn_case, _gdn_oracle
    nk, nv = 2, 4
    r = synth.rng(900 + T)
    case = list(_gdn_case(r, T, nk, nv, False))
    case[3] = (case[3] + decay).astype(np.float32)  # A_log
    o_ref, S_ref, conv_ref = _gdn_oracle(orc, *case, nk, nv, False)
    for mode in ("1", "0"):
        monkeypatch.setenv("RL_PF_GDN_CHUNK", mode)
        o, S, conv = ops.gdn_prefill(*case, nk, nv, False)
        assert np.isfinite(o).all() and np.isfinite(S).all()
        for t in range(T):
            assert rel_l2(o[t], o_ref[t]) < 1e-3, (mode, t, rel_l2(o[t], o_ref[t]))
        assert rel_l2(S, S_ref) < 1e-4, mode
        assert np.array_equal(conv, conv_ref)


def test_gdn_prefill_chunked_full_shape(gpu, monkeypatch):
    """At the 27B DeltaNet shape (16 k-heads, 48 v-heads) over a full 2048-token
    prefill chunk, the chunked scan and the per-token scan (each pinned to the
    per-token oracle at smaller sizes above) agree on every output row and on the
    final state."""
    from tests.test_gpu_layers import _gdn_case
    T, nk, nv = 2048, 16, 48
    case = _gdn_case(synth.rng(950), T, nk, nv, False)
    monkeypatch.setenv("RL_PF_GDN_CHUNK", "1")
    o1, S1, c1 = ops.gdn_prefill(*case, nk, nv, False)
    monkeypatch.setenv("RL_PF_GDN_CHUNK", "0")
    o0, S0, c0 = ops.gdn_prefill(*case, nk, nv, False)
    assert np.isfinite(o1).all() and np.isfinite(S1).all()
    err = np.linalg.norm(o1 - o0, axis=1) / np.maximum(np.linalg.norm(o0, axis=1), 1e-30)
    assert err.max() < 1e-4, (int(err.argmax()), float(err.max()))
    assert rel_l2(S1, S0) < 1e-5
    assert np.array_equal(c1, c0)


@pytest.mark.parametrize("qt,m,n,T", [(ops.Q4_K, 256, 1024, 70), (ops.Q6_K, 160, 768, 130),
                                      (ops.Q4_K, 5120, 4096, 300)])
def test_kquant_prefill_gemm_vs_oracle(gpu, orc, qt, m, n, T):
    """The K-quant prefill linear: rl_hip_kquant_to_bf16x2 turns the tiled blocks
    into BF16 hi + lo tiles (hi + lo equal the reference's dequantised weight to 16
    significant bits; checked against ops::dequant_q4_k / dequant_q6_k), and the
    BF16 x2 prefill GEMM over them matches the oracle's K-quant GEMV per token."""
    from rapidllm_amd.hip import DeviceBuffer, call
    r = synth.rng(700 + m + T)
    blocks = synth.q4k_blocks(r, m, n) if qt == ops.Q4_K else synth.q6k_blocks(r, m, n)
    lin = ops.KQuantLinear(qt, blocks, m, n)
    mt = (m + 15) // 16
    hi, lo = DeviceBuffer(mt * 16 * n * 2), DeviceBuffer(mt * 16 * n * 2)
    call("rl_hip_kquant_to_bf16x2", qt, lin.w.ptr, hi.ptr, lo.ptr, m, n, None)
    # the split against the exact dequantisation, element by element (first row tile)
    deq = orc.dequant_q4_k if qt == ops.Q4_K else orc.dequant_q6_k
    Wd = deq(np.ascontiguousarray(blocks.reshape(-1)), m * n).reshape(m, n)
    h = hi.numpy(np.uint16, (mt * 16 * n,))
    l = lo.numpy(np.uint16, (mt * 16 * n,))
    nkb = n // 128
    for row in (0, 5, 15):
        for c in (0, 37, 128, n - 1):
            kb, j = c // 128, c % 128
            g, q, e = j // 32, (j % 32) // 8, j % 8
            i = (0 * nkb + kb) * 2048 + q * 512 + 8 * (row + 16 * g) + e
            w = synth.bf16_to_f32(h[i:i + 1])[0] + synth.bf16_to_f32(l[i:i + 1])[0]
            assert abs(w - Wd[row, c]) <= abs(Wd[row, c]) * 2.0 ** -15, (row, c, w, Wd[row, c])
    X = r.standard_normal((T, n)).astype(np.float32)
    xd = DeviceBuffer.from_numpy(X)
    frag = ops.act_frag_buffer(n, T)
    yd = DeviceBuffer(4 * T * m)
    call("rl_hip_pack_act", xd.ptr, frag.ptr, n, T, None)
    call("rl_hip_gemm_bf16_prefill", hi.ptr, lo.ptr, frag.ptr, yd.ptr, m, n, T, 0, m, None)
    got = yd.numpy(np.float32, (T, m))
    gemv = orc.gemv_q4_k if qt == ops.Q4_K else orc.gemv_q6_k
    for t in range(0, T, max(1, T // 7)):
        want = gemv(np.ascontiguousarray(blocks.reshape(-1)), X[t], m, n, 8)
        assert rel_l2(got[t], want) <= REL_L2, (t, rel_l2(got[t], want))


def _f16_to_f32(bits):
    return np.asarray(bits, np.uint16).view(np.float16).astype(np.float32)


@pytest.mark.parametrize("qt,m,n,T,epi", [(ops.Q4_K, 256, 1024, 70, 0), (ops.Q6_K, 160, 768, 130, 1),
                                          (ops.Q4_K, 5120, 4096, 300, 0), (ops.Q6_K, 512, 1280, 64, 5)])
def test_kquant_f16_prefill_gemm_vs_oracle(gpu, orc, qt, m, n, T, epi):
    """The K-quant prefill linears' fp16 form: rl_hip_kquant_to_f16 stores each
    weight of a (16-row tile, 128-column block) as rn16(w / s) with a power-of-two s
    per block (checked against ops::dequant_q4_k / dequant_q6_k to fp16 rounding);
    rl_hip_act_frag_to_f16 turns the bf16 hi + mid fragments into fp16 hi + lo of
    x / xscale without losing a bit; the fp16 prefill GEMM (store, add, and SwiGLU
    over half tiles) matches the oracle's K-quant GEMV per token."""
    from rapidllm_amd.hip import DeviceBuffer, call
    r = synth.rng(800 + m + T)
    blocks = synth.q4k_blocks(r, m, n) if qt == ops.Q4_K else synth.q6k_blocks(r, m, n)
    lin = ops.KQuantLinear(qt, blocks, m, n)
    mt, nkb = (m + 15) // 16, n // 128
    w16 = DeviceBuffer(mt * 16 * n * 2)
    ts = DeviceBuffer(4 * mt * nkb)
    call("rl_hip_kquant_to_f16", qt, lin.w.ptr, w16.ptr, ts.ptr, m, n, None)
    deq = orc.dequant_q4_k if qt == ops.Q4_K else orc.dequant_q6_k
    Wd = deq(np.ascontiguousarray(blocks.reshape(-1)), m * n).reshape(m, n)
    h = _f16_to_f32(w16.numpy(np.uint16, (mt * 16 * n,)))
    sc = ts.numpy(np.float32, (mt, nkb))
    for rt in (0, mt - 1):
        for kb in (0, nkb - 1):
            blk = np.abs(Wd[16 * rt:16 * rt + 16, 128 * kb:128 * kb + 128])
            s = sc[rt, kb]
            mx = blk.max()
            assert s > 0 and (mx == 0 or 2.0 ** 14 <= mx / s < 2.0 ** 15), (rt, kb, s, mx)
            assert s == 2.0 ** np.round(np.log2(s))  # a power of two
    for row in (0, 5, 15, 16 * (mt - 1) + 3):
        for c in (0, 37, 128, n - 1):
            rt, kb, j = row // 16, c // 128, c % 128
            g, q, e = j // 32, (j % 32) // 8, j % 8
            i = (rt * nkb + kb) * 2048 + q * 512 + 8 * (row % 16 + 16 * g) + e
            w = np.float32(h[i]) * sc[rt, kb]
            want = np.float32(Wd[row, c] / sc[rt, kb]).astype(np.float16).astype(np.float32) * sc[rt, kb]
            assert w == want, (row, c, w, Wd[row, c])
    X = (r.standard_normal((T, n)) * np.exp(r.uniform(-6, 6, (T, 1)))).astype(np.float32)
    xd = DeviceBuffer.from_numpy(X)
    frag = ops.act_frag_buffer(n, T)
    call("rl_hip_pack_act", xd.ptr, frag.ptr, n, T, None)
    frag16 = ops.act_frag_buffer(n, T)
    xs = DeviceBuffer(4 * nkb * T)
    call("rl_hip_act_frag_to_f16", frag.ptr, frag16.ptr, xs.ptr, n, T, None)
    # hi + lo (fp16) times the scale equals hi + mid (bf16) exactly, unit by unit
    fb = frag.numpy(np.uint16, (frag.nbytes // 2,)).reshape(nkb * 16, 2 * T, 8)
    f16 = frag16.numpy(np.uint16, (frag16.nbytes // 2,)).reshape(nkb * 16, 2 * T, 8)
    xsv = xs.numpy(np.float32, (nkb, T))
    for t in (0, T - 1):
        bf = synth.bf16_to_f32(fb[:, t]) + synth.bf16_to_f32(fb[:, T + t])
        hl = (_f16_to_f32(f16[:, t]).astype(np.float64) + _f16_to_f32(f16[:, T + t])) * \
            np.repeat(xsv[:, t], 16)[:, None]
        assert np.array_equal(bf.astype(np.float64), hl), t
    mo = m // 2 if epi == 5 else m
    Y0 = r.standard_normal((T, mo)).astype(np.float32)
    yd = DeviceBuffer.from_numpy(Y0)
    call("rl_hip_gemm_f16_prefill", w16.ptr, ts.ptr, frag16.ptr, xs.ptr, yd.ptr, m, n, T, epi, mo, None)
    got = yd.numpy(np.float32, (T, mo))
    gemv = orc.gemv_q4_k if qt == ops.Q4_K else orc.gemv_q6_k
    for t in range(0, T, max(1, T // 7)):
        y = gemv(np.ascontiguousarray(blocks.reshape(-1)), X[t], m, n, 8).astype(np.float64)
        if epi == 5:  # half tiles: rows 16k .. 16k+7 gate, 16k+8 .. 16k+15 up of outputs 8k .. 8k+7
            yt = y.reshape(-1, 2, 8)
            with np.errstate(over="ignore"):
                want = (yt[:, 0] / (1.0 + np.exp(-yt[:, 0])) * yt[:, 1]).reshape(-1)
        else:
            want = y + (Y0[t] if epi == 1 else 0.0)
        assert rel_l2(got[t], want) <= REL_L2, (t, rel_l2(got[t], want))


@pytest.mark.parametrize("quant", ["q4_k", "q6_k", "bf16"])
def test_engine_kquant_chunked_prefill_matches_oracle(gpu, orc, monkeypatch, quant):
    """A GGUF-style model (K-quant layer linears, BF16 a / b rows, Q6_K lm_head), or
    a model with BF16 layer linears, prefills a 300-token prompt through the chunked
    path (two chunks of 256 + the decode-step tail): logits and decoding continue as
    the oracle's."""
    from oracle.oracle import OracleModel
    from rapidllm_amd import model as M
    from rapidllm_amd.engine import Engine
    from tests.test_gpu_engine import margin_ok, mini_spec
    spec = mini_spec()
    lq = {"q4_k": M.Q_Q4_K, "q6_k": M.Q_Q6_K, "bf16": M.Q_BF16}[quant]
    W = M.random_weights(spec, seed=13, linear_quant=lq, head_quant=M.Q_BF16 if quant == "bf16" else M.Q_Q6_K)
    monkeypatch.setenv("RL_PREFILL_CHUNK", "256")
    eng = Engine(spec, W, ctx=1024)
    orc_m = OracleModel(spec, W, ctx=1024)
    rng = np.random.default_rng(15)
    prompt = [int(t) for t in rng.integers(0, spec.vocab, 300)]
    eng.prefill(prompt)
    orc_m.reset()
    for t in prompt:
        g, lg, hd = orc_m.decode(t)
    assert rel_l2(eng.copy_logits(), lg) < 1e-3
    if margin_ok(lg):
        assert eng.greedy() == g
    tok = g
    for _ in range(3):
        eng.decode_token(tok)
        g, lg, _ = orc_m.decode(tok)
        assert rel_l2(eng.copy_logits(), lg) < 1e-3
        tok = g
    eng.close()


@pytest.mark.parametrize("m,n,T,epi", [
    # K split over 8 waves (T <= 32): 2, 4 and 8 row tiles; 10 half column blocks leave
    # a ragged last step, 384 columns waves without one
    (300, 640, 1, 0), (33000, 384, 20, 0), (16480, 256, 32, 1), (544, 384, 31, 5),
    # over 4 (T <= 64): 2, 4, 8 and 10 row tiles
    (300, 640, 33, 0), (9000, 384, 64, 0), (24592, 384, 64, 0), (40000, 256, 50, 5),
    # over 2, and none: 4, 8, 10 and 12 row tiles, ragged last row and token blocks
    (300, 640, 65, 1), (4112, 128, 129, 0), (9000, 384, 200, 5), (33000, 256, 700, 0), (16480, 256, 300, 2),
    (20000, 256, 400, 5), (16480, 256, 520, 0),
    # a second group of eight token blocks, one or two blocks wide
    (300, 640, 1025, 0), (544, 384, 1160, 5)])
def test_gemm_prefill_work_splits(gpu, orc, m, n, T, epi):
    """Every work split of the block-FP8 prefill GEMM (row tiles per workgroup, waves
    along tokens and along K) at the edges of its range, with each epilogue, against the
    oracle on the first and last tokens and those at 32-token boundaries.  Tolerance:
    activations keep 16 significant bits (at most 2^-15 = 3e-5 off per product) and fp32
    sums of at most 640 terms add less than 1e-6; SwiGLU multiplies two such results."""
    r = synth.rng(1100 + m + n + T)
    toks = sorted({0, T // 2, T - 1} | {t for t in (31, 32, 63, 64, 127, 128, 255, 256, 1023, 1024, 1151, 1152) if t < T})
    X = r.standard_normal((T, n)).astype(np.float32)
    Xs = np.ascontiguousarray(X[toks])
    if epi == 5:
        I = m // 2 // 8 * 8
        Wg, Wu = synth.fp8_weight_wide(r, I, n), synth.fp8_weight_wide(r, I, n)
        sg, su = synth.fp8_scales(r, I, n), synth.fp8_scales(r, I, n)
        g = orc.gemm_fp8(Wg, sg, Xs).astype(np.float64)
        with np.errstate(over="ignore"):
            want = g / (1.0 + np.exp(-g)) * orc.gemm_fp8(Wu, su, Xs).astype(np.float64)
        got = ops.linear_prefill(ops.Fp8GateUp(Wg, sg, Wu, su), X, epilogue=5)
    else:
        W, s = synth.fp8_weight_wide(r, m, n), synth.fp8_scales(r, m, n)
        lin = ops.Fp8Linear(W, s)
        y = orc.gemm_fp8(W, s, Xs).astype(np.float64)
        if epi == 2:  # rows 32b .. 32b+15 gate, 32b+16 .. 32b+31 up
            y2 = y.reshape(len(toks), -1, 2, 16)
            with np.errstate(over="ignore"):
                want = (y2[:, :, 0] / (1.0 + np.exp(-y2[:, :, 0])) * y2[:, :, 1]).reshape(len(toks), -1)
            got = ops.linear_prefill(lin, X, epilogue=2)
        else:
            Y0 = r.standard_normal((T, m)).astype(np.float32) if epi == 1 else None
            want = y + (Y0[toks] if epi == 1 else 0.0)
            got = ops.linear_prefill(lin, X, epilogue=epi, Y0=Y0)
    assert np.isfinite(got).all()
    for k, t in enumerate(toks):
        assert rel_l2(got[t], want[k]) <= (2 if epi in (2, 5) else 1) * 3.2e-5, (t, rel_l2(got[t], want[k]))


@pytest.mark.parametrize("quant,hidden,inter,T", [
    # one 128-row and one ragged token block; the MLP's SwiGLU straight into the down
    # projection's fp16 + e4m3 input (768 rows: three 256-row blocks)
    ("fp8", 256, 384, 64), ("fp8", 384, 640, 129), ("fp8", 256, 1024, 260),
    # an intermediate that leaves a partial column block: fp32 SwiGLU rows, then packed
    ("fp8", 256, 328, 191), ("fp8", 128, 136, 65),
    ("q4_k", 256, 512, 64), ("q6_k", 512, 768, 257), ("q4_k", 256, 1280, 127),
    # one token short of the split inputs: the bf16 hi + mid kernels
    ("fp8", 256, 384, 63), ("q4_k", 256, 512, 63)])
def test_engine_prefill_split_inputs(gpu, orc, quant, hidden, inter, T):
    """Prompt chunks of T tokens at the edges of the fp16 + e4m3 prefill linears (64
    tokens and up; every producer of their inputs, in models so small that the linears
    take 128-token blocks of 128 rows, or of 256 with the SwiGLU output: the other work
    splits are in test_gpu_gemm_x.py) against the oracle model.  Tolerance: block-FP8 inputs are 2^-16
    off at most, 3e-5 after a few layers; the K-quant weights as fp16 2^-12, 1e-3."""
    from oracle.oracle import OracleModel
    from rapidllm_amd import model as M
    from rapidllm_amd.engine import Engine
    spec = M.ModelSpec(vocab=512, hidden=hidden, n_layers=4, intermediate=inter, n_k_heads=2, n_v_heads=4, n_q=4,
                       n_kv=2, layer_kinds=[0, 1, 0, 0], has_mtp=False)
    lq = {"fp8": M.Q_FP8, "q4_k": M.Q_Q4_K, "q6_k": M.Q_Q6_K}[quant]
    kw = {"w_scale": (1e-3, 1e-2)} if quant == "fp8" else {"head_quant": M.Q_Q6_K}
    W = M.random_weights(spec, seed=21 + T, linear_quant=lq, **kw)
    eng = Engine(spec, W, ctx=512)
    orc_m = OracleModel(spec, W, ctx=512)
    prompt = [int(t) for t in np.random.default_rng(T).integers(0, spec.vocab, T + 4)]  # the last 4: a decode step
    eng.prefill(prompt)
    orc_m.reset()
    for t in prompt:
        g, lg, hd = orc_m.decode(t)
    bar = 1e-4 if quant == "fp8" else 1e-3
    assert rel_l2(eng.copy_logits(), lg) < bar, rel_l2(eng.copy_logits(), lg)
    assert rel_l2(eng.copy_last_hidden(), hd) < bar
    eng.close()


@pytest.mark.parametrize("quant", ["fp8", "q4_k"])
def test_engine_prefill_mixed_chunks(gpu, orc, monkeypatch, quant):
    """One prompt in chunks of both input forms (100 tokens: fp16 + e4m3; 50: bf16 hi + mid),
    attention and DeltaNet layers, then a second prompt: the forms share buffers.  Bars as in
    test_engine_prefill_split_inputs."""
    from oracle.oracle import OracleModel
    from rapidllm_amd import model as M
    from rapidllm_amd.engine import Engine
    monkeypatch.setenv("RL_PREFILL_CHUNK", "100")
    spec = M.ModelSpec(vocab=512, hidden=256, n_layers=4, intermediate=512, n_k_heads=2, n_v_heads=4, n_q=4, n_kv=2,
                       layer_kinds=[0, 1, 0, 0], has_mtp=False)
    kw = {"w_scale": (1e-3, 1e-2)} if quant == "fp8" else {"head_quant": M.Q_Q6_K}
    W = M.random_weights(spec, seed=77, linear_quant=M.Q_FP8 if quant == "fp8" else M.Q_Q4_K, **kw)
    eng, orc_m = Engine(spec, W, ctx=512), OracleModel(spec, W, ctx=512)
    bar = 1e-4 if quant == "fp8" else 1e-3
    for n, seed in ((154, 1), (254, 2)):
        prompt = [int(t) for t in np.random.default_rng(seed).integers(0, spec.vocab, n)]
        eng.reset()
        eng.prefill(prompt)
        orc_m.reset()
        for t in prompt:
            _, lg, _ = orc_m.decode(t)
        assert rel_l2(eng.copy_logits(), lg) < bar, (n, rel_l2(eng.copy_logits(), lg))
    eng.close()


@pytest.mark.parametrize("T,pos,nq,nkv", [
    (1, 5000, 24, 4), (17, 3000, 24, 4), (33, 0, 6, 1), (64, 4031, 24, 4), (100, 2500, 12, 2), (65, 1800, 8, 8),
    (31, 900, 9, 3),      # a kv head count that does not divide the XCDs
    (1380, 700, 24, 4),   # one full round of workgroups and a split remainder
    (1366, 0, 24, 4)])    # ... whose ranges start at the first position
def test_attn_prefill_split_positions(gpu, T, pos, nq, nkv):
    """Prefill attention where workgroups are split over ranges of positions and merged
    (few tokens over a long context, and the remainder after full rounds), on the first
    and last tokens and those around 32-token blocks, against 64-bit attention over the
    fp16 cache.  Tolerance: probabilities rounded to fp16 (2^-12 each) and a cache entry
    that rounds the other way (2^-11), below 1e-3 of the output."""
    r = synth.rng(70 + pos + T + nq)
    hd, rot, theta = 256, 64, 1e7
    ctx = ((pos + T + 255) // 256) * 256 + 256
    Y = r.standard_normal((T, 2 * nq * hd + 2 * nkv * hd)).astype(np.float32)
    qn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    kn = (r.standard_normal(hd) * 0.1).astype(np.float32)
    K = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    V = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    cache = ops.AttnCache(nkv, ctx, hd)
    if pos:
        cache.fill(K, V)
    out = ops.attn_prefill_layer(Y, cache, pos, qn, kn, nq, nkv)

    def norm_rope(x, g):  # [T][heads][256]
        x = x.astype(np.float64)
        x = x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-6) * (1.0 + g.astype(np.float64))
        freq = (np.float32(1) / np.power(np.float32(theta), np.arange(rot // 2, dtype=np.float32) / (rot // 2)))
        ang = (np.arange(pos, pos + T, dtype=np.float32)[:, None] * freq.astype(np.float32)).astype(np.float64)[:, None]
        a, b = x[..., :rot // 2].copy(), x[..., rot // 2:rot].copy()
        x[..., :rot // 2] = a * np.cos(ang) - b * np.sin(ang)
        x[..., rot // 2:rot] = a * np.sin(ang) + b * np.cos(ang)
        return x

    qg = Y[:, :2 * nq * hd].reshape(T, nq, 2, hd)
    kv = Y[:, 2 * nq * hd:].reshape(T, 2, nkv, hd)
    q = norm_rope(qg[:, :, 0], qn)
    Ka = np.concatenate([K, norm_rope(kv[:, 0], kn).astype(np.float16)]).astype(np.float64)
    Va = np.concatenate([V, kv[:, 1].astype(np.float16)]).astype(np.float64)
    for t in sorted({0, T // 2, T - 1} | {x for x in (15, 16, 31, 32, 1279, 1280, 1343, 1344) if x < T}):
        n = pos + t + 1
        want = np.empty((nq, hd))
        for h in range(nq):
            s = Ka[:n, h * nkv // nq] @ q[t, h] / 16.0
            w = np.exp(s - s.max())
            want[h] = (w / w.sum()) @ Va[:n, h * nkv // nq]
        want /= 1.0 + np.exp(-qg[t, :, 1].astype(np.float64))
        assert rel_l2(out[t], want.reshape(-1)) < 1e-3, (t, rel_l2(out[t], want.reshape(-1)))


@pytest.mark.parametrize("T,pos,nq,nkv", [
    (1, 0, 24, 4), (17, 0, 24, 4), (64, 0, 6, 1), (65, 3, 8, 8), (100, 668, 12, 2),   # 768 keys
    (450, 0, 24, 4), (512, 256, 9, 3), (300, 100, 24, 4), (768, 0, 6, 1),
    (101, 668, 12, 2), (512, 257, 24, 4), (768, 1, 24, 4), (769, 0, 8, 8)])           # one key more
def test_attn_prefill_short_context_in_large_cache(gpu, T, pos, nq, nkv):
    """A chunk over few keys takes the short kernel whatever the cache's capacity: up to 768
    keys the outputs are the bytes that a cache of just those keys gives.  Beyond, two kernels that each round probabilities to fp16 (2^-12) agree within 1e-3."""
    r = synth.rng(90 + pos + T + nq)
    hd = 256
    Y = r.standard_normal((T, 2 * nq * hd + 2 * nkv * hd)).astype(np.float32)
    K = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    V = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    qn, kn = (r.standard_normal(hd).astype(np.float32) * np.float32(0.1) for _ in range(2))
    outs = []
    for ctx in ((pos + T + 255) // 256 * 256, 8192):
        cache = ops.AttnCache(nkv, ctx, hd)
        if pos:
            cache.fill(K, V)
        outs.append(ops.attn_prefill_layer(Y, cache, pos, qn, kn, nq, nkv))
    assert np.isfinite(outs[0]).all()
    if pos + T <= 768:
        assert outs[0].tobytes() == outs[1].tobytes()
    else:
        for t in range(T):
            assert rel_l2(outs[1][t], outs[0][t]) < 1e-3, (t, rel_l2(outs[1][t], outs[0][t]))


@pytest.mark.parametrize("T,pos,nq,nkv", [
    (1, 5000, 24, 4), (17, 3001, 24, 4), (33, 1100, 6, 1), (64, 4031, 24, 4), (100, 2503, 12, 2), (65, 1800, 8, 8),
    (31, 900, 9, 3), (130, 640, 24, 4), (767, 9, 24, 4), (1380, 700, 24, 4)])
@pytest.mark.parametrize("known", [True, False])
@pytest.mark.parametrize("whole_ws", [True, False])
def test_attn_prefill_known_keys_and_small_workspace(gpu, T, pos, nq, nkv, known, whole_ws):
    """The routes of a chunk past 768 keys: the keys known to the host (as in the engine: the
    norm / RoPE pass and the merge of their own) or read on the device, in a workspace of the
    documented size or of the q fragments alone (no split), against single tokens' decode
    attention over the caches that the chunk left.  The decode kernel and the prefill
    kernels each round probabilities to fp16 (2^-12) and norm a token's own q in another order:
    5e-4 each, 1e-3 together.  Nothing is written past the workspace or the output, and a
    second call gives the same bytes."""
    r = synth.rng(130 + pos + T + nq)
    hd, ld, guard = 256, 2 * nq * 256 + 2 * nkv * 256, 4096
    ctx = 8192
    Y = r.standard_normal((T, ld)).astype(np.float32)
    K = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    V = r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32)
    qn, kn = (r.standard_normal(hd).astype(np.float32) * np.float32(0.1) for _ in range(2))
    cache = ops.AttnCache(nkv, ctx, hd)
    cache.fill(K, V)
    nb = hip.lib().rl_hip_attn_prefill_workspace_bytes(nq, T) if whole_ws else nq * -(-T // 16) * 16384 + 256
    ws = DeviceBuffer.from_numpy(np.full(nb + guard, 0xA5, np.uint8))
    ob = 4 * T * nq * hd
    out = DeviceBuffer.from_numpy(np.full(ob + guard, 0xA5, np.uint8))
    args = [DeviceBuffer.from_numpy(a) for a in (Y, qn, kn, np.array([pos], np.int32))]
    got = []
    for _ in range(2):
        call("rl_hip_attn_prefill_layer_keys", args[0].ptr, ld, args[1].ptr, args[2].ptr, cache.k.ptr, cache.vt.ptr, ctx,
             args[3].ptr, T, nq, nkv, hd, 64, 1e7, 1e-6, ws.ptr, nb, out.ptr, pos + T if known else 0, None)
        raw = out.numpy(np.uint8, (ob + guard,))
        assert (raw[ob:] == 0xA5).all() and (ws.numpy(np.uint8, (nb + guard,))[nb:] == 0xA5).all()
        got.append(raw[:ob].tobytes())
    assert got[0] == got[1]
    o = np.frombuffer(got[0], np.float32).reshape(T, nq * hd)
    assert np.isfinite(o).all()
    for t in sorted({0, T // 2, T - 1} | {x for x in (15, 16, 31, 32, 63, 64, 1279, 1280) if x < T}):
        want = ops.attn_decode_layer(Y[t], cache, pos + t, qn, kn, nq, nkv)[0]
        assert rel_l2(o[t], want) < 1e-3, (t, rel_l2(o[t], want))


@pytest.mark.parametrize("T,pos,nq,nkv,bad", [
    (200, 1000, 24, 4, (100, 199)), (900, 1000, 24, 4, (0, 97, 640)), (130, 800, 6, 1, (31, 32)),
    (300, 700, 8, 8, (140, 299)), (70, 4003, 9, 3, (47,)), (1400, 33, 24, 4, (64, 1024, 1399)), (1, 900, 24, 4, (0,))])
@pytest.mark.parametrize("known", [True, False])
def test_attn_prefill_non_finite_v(gpu, T, pos, nq, nkv, bad, known):
    """Infinities and NaN in the V of some tokens (some dims of one kv head), past 768 keys:
    they reach that token's outputs and those after it, in these dims, and leave every other
    output byte as it is without them."""
    r = synth.rng(170 + pos + T + nq)
    hd, ctx = 256, 8192
    Y = r.standard_normal((T, 2 * nq * hd + 2 * nkv * hd)).astype(np.float32)
    K, V = (r.standard_normal((pos, nkv, hd)).astype(np.float16).astype(np.float32) for _ in range(2))
    qn, kn = (r.standard_normal(hd).astype(np.float32) * np.float32(0.1) for _ in range(2))
    kv = nkv - 1
    v0 = 2 * nq * hd + nkv * hd + kv * hd
    Yb = Y.copy()
    Yb[bad[0], v0 + 3] = np.inf
    Yb[bad[0], v0 + 129] = -np.inf
    Yb[bad[-1], v0 + 3] = np.inf
    Yb[bad[-1], v0 + 250] = np.nan
    Yb[bad[-1], v0 + 64] = -1e5  # past fp16's range
    outs = []
    for y in (Y, Yb):
        cache = ops.AttnCache(nkv, ctx, hd)
        cache.fill(K, V)
        ws = DeviceBuffer(hip.lib().rl_hip_attn_prefill_workspace_bytes(nq, T))
        out = DeviceBuffer(4 * T * nq * hd)
        args = [DeviceBuffer.from_numpy(a) for a in (y, qn, kn, np.array([pos], np.int32))]
        call("rl_hip_attn_prefill_layer_keys", args[0].ptr, y.shape[1], args[1].ptr, args[2].ptr, cache.k.ptr, cache.vt.ptr,
             ctx, args[3].ptr, T, nq, nkv, hd, 64, 1e7, 1e-6, ws.ptr, ws.nbytes, out.ptr, pos + T if known else 0, None)
        outs.append(out.numpy(np.float32, (T, nkv, nq // nkv, hd)))
    want = outs[0]
    for t, d, x in ((bad[0], 3, np.inf), (bad[0], 129, -np.inf), (bad[-1], 250, np.nan), (bad[-1], 64, -np.inf)):
        want[t:, kv, :, d] = x
    assert np.array_equal(want.view(np.uint32)[~np.isnan(want)], outs[1].view(np.uint32)[~np.isnan(want)])
    assert np.isnan(outs[1][np.isnan(want)]).all()
