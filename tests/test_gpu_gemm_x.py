"""The engine's prompt linears (fp16 + e4m3 inputs) one launch at a time, against 64-bit
products: every work split of every weight kind and epilogue.

Tolerance.  An input element x is h + l: h = fp16(x / s) is off by at most 2^-11 of itself,
and l holds that remainder in e4m3's 4 bits, off by at most 2^-5 of the power of two above
it: h + l is off by at most 2^-16 of x.  fp16 tiles enter the remainder's pass with 4 bits as
well, 2^-11 * 2^-4 more: 2^-15 + 2^-16 in all.  That is the bar, which a token reaches that
one element dominates (errors of many elements average: 4.9e-6 and 7.3e-6 of the result for
normal inputs); fp32 sums of at most 384 terms add less than 1e-6.  Without the remainder's
pass the error is 2.1e-4, with a wrong one larger.  SwiGLU: d(silu(g) u) <= 1.1 |u dg| +
|silu(g) du| and silu(g) is 0.6 |g| in the mean: 3 times a linear's bar.  Its outputs as the
next input: 2^-16 more."""
import ctypes
import os

import numpy as np
import pytest

from rapidllm_amd import hip, ops, synth
from rapidllm_amd.hip import DeviceBuffer, call

BAR = {0: 2.0 ** -16 + 1e-6, 1: 2.0 ** -15 + 2.0 ** -16 + 1e-6}  # block-FP8, fp16 tiles
STORE, ADD, SWIGLU, SWIGLU_X = 0, 1, 5, 7

# (fp16 tiles, epilogue, m, n, T): ragged row and token blocks, three column blocks in some
CASES = [
    # block-FP8: 128-token blocks of 128, 192 and 256 rows, and two launches
    (0, STORE, 16, 128, 64), (0, ADD, 300, 384, 65), (0, STORE, 16480, 256, 129), (0, ADD, 16368, 256, 1025),
    (0, STORE, 10992, 384, 1025), (0, STORE, 14912, 256, 1300), (0, ADD, 9440, 256, 3000),
    (0, SWIGLU, 80, 328, 100), (0, SWIGLU, 16480, 256, 129), (0, SWIGLU, 10992, 384, 1025), (0, SWIGLU, 16368, 256, 1025),
    (0, SWIGLU_X, 256, 256, 64), (0, SWIGLU_X, 768, 384, 129), (0, SWIGLU_X, 10240, 256, 1100),
    # fp16 tiles: one workgroup per CU, 256- and 128-token blocks
    (1, STORE, 16, 128, 64), (1, ADD, 300, 384, 65), (1, STORE, 16480, 256, 129), (1, ADD, 16480, 256, 257),
    (1, STORE, 16368, 384, 257), (1, ADD, 13120, 256, 513), (1, STORE, 17488, 256, 513),
    # two launches of every pair
    (1, STORE, 16368, 256, 513), (1, ADD, 13120, 256, 1025), (1, STORE, 15248, 256, 1025), (1, ADD, 14352, 256, 1025),
    (1, STORE, 16704, 256, 1025), (1, STORE, 13456, 256, 1025), (1, ADD, 16368, 256, 1025), (1, STORE, 17040, 256, 1025),
    (1, STORE, 16704, 256, 1300), (1, ADD, 16480, 256, 1300), (1, STORE, 26464, 128, 1300), (1, STORE, 24640, 256, 300),
    (1, ADD, 35584, 128, 300),
    (1, SWIGLU, 80, 384, 100), (1, SWIGLU, 16480, 256, 129), (1, SWIGLU, 16480, 256, 257), (1, SWIGLU, 16368, 384, 257),
    (1, SWIGLU, 13120, 256, 513), (1, SWIGLU, 17488, 256, 513), (1, SWIGLU, 16704, 256, 1300),
    (1, SWIGLU_X, 256, 256, 64), (1, SWIGLU_X, 768, 384, 129), (1, SWIGLU_X, 34304, 128, 129),
    (1, SWIGLU_X, 27136, 256, 513)]


def split(fp16, epi, m, T, cus=256):
    out = (ctypes.c_int * 6)()
    call("rl_hip_gemm_x_split", fp16, epi, m, T, cus, out)
    return (out[0], out[1]), (out[3], out[4]) if out[5] else None, out[2], out[5]


def test_cases_take_every_split():
    """CPU: over the shapes of the models' linears and prompts of up to 4096 tokens, no pair
    of launches (and for SwiGLU no kernel) is chosen that no case above takes."""
    if not os.path.exists(hip.LIB_PATH):
        pytest.skip("library not built (python -c 'import __graft_entry__ as g; g.build()')")
    pairs, kernels = set(), set()
    for fp16, epi, m, n, T in CASES:
        a, b, _, _ = split(fp16, epi, m, T)
        pairs.add((fp16, epi == SWIGLU_X, a, b))
        kernels |= {(fp16, epi, k) for k in (a, b) if k}
    for fp16 in (0, 1):
        for T in (64, 100, 128, 129, 256, 300, 512, 700, 1024, 1300, 2044, 2048, 3000, 4092):
            for m in list(range(16, 36864, 304)) + [14336, 16480, 5120, 34816, 10240, 4096]:
                a, b, na, nb = split(fp16, STORE, m, T)
                assert (fp16, False, a, b) in pairs, (fp16, m, T, a, b)
                # the launches cover the rows, each once
                assert 64 * (a[0] * na + (b[0] * (nb - 1) if b else -a[0])) < m <= 64 * (a[0] * na + (b[0] * nb if b else 0))
                assert all((fp16, SWIGLU, k) in kernels for k in (a, b) if k), (fp16, m, T, a, b)
                a, b, _, _ = split(fp16, SWIGLU_X, (m + 255) // 256 * 256, T)
                assert (fp16, True, a, b) in pairs, (fp16, m, T, a, b)


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def weights(r, fp16, m, n):
    """(device tiles, device scales, the weights in float64, rows in tile order)."""
    kb, mt = -(-n // 128), -(-m // 16)
    if not fp16:
        W, s = synth.fp8_weight_wide(r, m, n), synth.fp8_scales(r, m, n)
        lin = ops.Fp8Linear(W, s)
        dense = ops_e4m3(W) * np.repeat(np.repeat(s.astype(np.float64), 128, 0)[:m], 128, 1)[:, :n]
        return lin.w, lin.ts, dense, lin
    # fp16 tiles as rl_hip_kquant_to_f16 leaves them: largest magnitudes in [2^14, 2^15)
    w = (r.standard_normal((mt, 16, kb, 4, 4, 8)) * 2.0 ** 12.5).clip(-32752, 32752).astype(np.float16)  # [rt][row][kb][g][q][e]
    w[mt - 1, m - 16 * (mt - 1):] = 0
    ts = np.exp2(r.integers(-24, -18, (mt, kb))).astype(np.float32)
    dense = (w.astype(np.float64) * ts[:, None, :, None, None, None]).reshape(16 * mt, 128 * kb)[:m, :n]
    return DeviceBuffer.from_numpy(np.ascontiguousarray(w.transpose(0, 2, 4, 3, 1, 5))), DeviceBuffer.from_numpy(ts), dense, None


def ops_e4m3(W):
    table = ops.e4m3_to_f32(np.arange(256, dtype=np.uint8)).astype(np.float64)
    return table[W]


def unpack_x(buf, n, T, toks):
    """The elements of an input in float64 for some tokens."""
    kb = -(-n // 128)
    raw = buf.numpy(np.uint8, (buf.nbytes,))
    h = raw[:256 * kb * T].view(np.float16).reshape(kb, 4, 4, T, 8)[:, :, :, toks].astype(np.float64)
    l8 = raw[256 * kb * T:384 * kb * T].reshape(kb, 2, 4, T, 16)[:, :, :, toks]
    s = raw[384 * kb * T:388 * kb * T].view(np.float32).reshape(kb, T)[:, toks].astype(np.float64)
    hx = h.transpose(3, 0, 2, 1, 4).reshape(len(toks), kb, 128)          # [t][kb][g][i][e]
    lx = ops_e4m3(l8).transpose(3, 0, 2, 1, 4).reshape(len(toks), kb, 128)  # [t][kb][g][c][e]
    return ((hx + lx / 128) * s.T[:, :, None]).reshape(len(toks), 128 * kb)[:, :n]


def inputs(r, T, n):
    """Tokens of different size, a few channels an order of magnitude larger."""
    X = r.standard_normal((T, n)) * np.exp2(r.integers(-6, 7, (T, 1)))
    X[:, r.integers(0, n, max(1, n // 100))] *= 12.0
    return X.astype(np.float32)


def pack(X):
    T, n = X.shape
    x, rows = DeviceBuffer(hip.lib().rl_hip_act_x_bytes(n, T)), DeviceBuffer.from_numpy(X)
    call("rl_hip_pack_act_x", rows.ptr, x.ptr, n, T, None)
    call("rl_hip_device_synchronize")
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("n,T", [(128, 1), (136, 5), (640, 70), (5120, 3)])
def test_pack_act_x(gpu, n, T):
    """Input form: every element within 2^-16 of itself down to 2^-13 of its block's largest,
    below that within half the smallest e4m3 remainder, 2^-29 of the largest; zeros exact."""
    r = synth.rng(n + T)
    X = inputs(r, T, n)
    X[0, :8] = 0.0
    X[:, 1::9] *= np.float32(2.0 ** -12)
    X[:, 2::9] *= np.float32(2.0 ** -18)
    got = unpack_x(pack(X), n, T, list(range(T)))
    err = np.abs(got - X.astype(np.float64))
    blk = np.abs(np.pad(X, ((0, 0), (0, -n % 128)))).reshape(T, -1, 128).max(2).repeat(128, 1)[:, :n]
    assert (err <= np.maximum(2.0 ** -16 * np.abs(X), 2.0 ** -29 * blk)).all()
    assert (got[0, :8] == 0.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n,T", [(128, 64), (768, 70), (5120, 65), (6144, 67)])
def test_norms_to_act_x(gpu, n, T):
    """The layer norm and the gated norm written as an input are the bytes of the norms that
    write fp32 rows (rl_hip_rmsnorm_pack, rl_hip_gated_rmsnorm_pack), packed: no less precise.
    Gates reach far enough down for the exponential's precision to show."""
    r = synth.rng(n + T)
    X, g = inputs(r, T, n), (r.standard_normal(n) * 0.1).astype(np.float32)
    d = [DeviceBuffer.from_numpy(a) for a in (X, g)]
    y, x = DeviceBuffer(4 * T * n), DeviceBuffer(hip.lib().rl_hip_act_x_bytes(n, T))
    used = 388 * (n // 128) * T
    call("rl_hip_rmsnorm_pack", d[0].ptr, n, d[1].ptr, y.ptr, None, n, T, 1e-6, None)
    call("rl_hip_rmsnorm_x", d[0].ptr, d[1].ptr, x.ptr, n, T, 1e-6, None)
    call("rl_hip_device_synchronize")
    want = pack(y.numpy(np.float32, (T, n)))
    assert x.numpy(np.uint8, (x.nbytes,))[:used].tobytes() == want.numpy(np.uint8, (x.nbytes,))[:used].tobytes()
    if n < 256:
        return  # (one head: the norm over all of n)
    Z = (r.standard_normal((T, n)) * 12).astype(np.float32)
    z = DeviceBuffer.from_numpy(Z)
    call("rl_hip_gated_rmsnorm_pack", d[0].ptr, z.ptr, n, d[1].ptr, 128, y.ptr, None, n, T, 1e-6, None)
    call("rl_hip_gated_rmsnorm_x", d[0].ptr, z.ptr, n, d[1].ptr, x.ptr, n, T, 1e-6, None)
    call("rl_hip_device_synchronize")
    want = pack(y.numpy(np.float32, (T, n)))
    assert x.numpy(np.uint8, (x.nbytes,))[:used].tobytes() == want.numpy(np.uint8, (x.nbytes,))[:used].tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("fp16,epi,m,n,T", CASES)
def test_gemm_x(gpu, fp16, epi, m, n, T):
    r = synth.rng(17 * m + n + T + epi)
    w, ts, W, keep = weights(r, fp16, m, n) if fp16 or epi < SWIGLU else gate_up(r, m, n)
    X = inputs(r, T, n)
    toks = sorted({0, T // 2, T - 1} | {t for t in (31, 32, 63, 64, 127, 128, 255, 256, 511, 512, 1023, 1024) if t < T})
    y = X[toks].astype(np.float64) @ W.T
    x = pack(X)
    if epi >= SWIGLU:  # row tiles of 8 gate and 8 up rows
        g, u = y.reshape(len(toks), -1, 2, 8).transpose(2, 0, 1, 3).reshape(2, len(toks), -1)
        y = g / (1 + np.exp(-g.clip(-700))) * u
    mo = y.shape[1]
    Y0 = (r.standard_normal((T, mo)) * np.abs(y).mean()).astype(np.float32) if epi == ADD else None
    yd = DeviceBuffer.from_numpy(Y0) if epi == ADD else DeviceBuffer(4 * T * mo)
    call("rl_hip_gemm_x", fp16, w.ptr, ts.ptr, x.ptr, yd.ptr, None, m, n, T, SWIGLU if epi == SWIGLU_X else epi, 0, None)
    rows = yd.numpy(np.float32, (T, mo))
    assert np.isfinite(rows).all()
    got = rows[toks].astype(np.float64) - (Y0[toks].astype(np.float64) if epi == ADD else 0.0)
    bar = BAR[fp16] * (3 if epi >= SWIGLU else 1) + (2e-7 if epi == ADD else 0.0)  # (the sum's rounding)
    for k, t in enumerate(toks):
        assert rel(got[k], y[k]) < bar, (t, rel(got[k], y[k]))
    if epi == SWIGLU_X:
        # the same numbers as the fp32 rows packed by a pass of their own
        out = DeviceBuffer(hip.lib().rl_hip_act_x_bytes(mo, T))
        call("rl_hip_gemm_x", fp16, w.ptr, ts.ptr, x.ptr, None, out.ptr, m, n, T, epi, 0, None)
        call("rl_hip_device_synchronize")
        used = 388 * (mo // 128) * T
        assert out.numpy(np.uint8, (out.nbytes,))[:used].tobytes() == pack(rows).numpy(np.uint8, (out.nbytes,))[:used].tobytes()
        for k, t in enumerate(toks):
            z = unpack_x(out, mo, T, [t])[0]
            assert rel(z, y[k]) < bar + 2.0 ** -16, (t, rel(z, y[k]))


def gate_up(r, m, n):
    """Block-FP8 gate and up with scales of their own, in half tiles."""
    i = m // 2
    Wg, Wu = synth.fp8_weight_wide(r, i, n), synth.fp8_weight_wide(r, i, n)
    sg, su = synth.fp8_scales(r, i, n), synth.fp8_scales(r, i, n)
    lin = ops.Fp8GateUp(Wg, sg, Wu, su)
    d = [ops_e4m3(w) * np.repeat(np.repeat(s.astype(np.float64), 128, 0)[:i], 128, 1)[:, :n] for w, s in ((Wg, sg), (Wu, su))]
    return lin.w, lin.ts, np.stack([v.reshape(i // 8, 8, n) for v in d], 1).reshape(m, n), lin
