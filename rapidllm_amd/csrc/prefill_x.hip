// prefill_x.hip -- prefill linears over activations split into fp16 + e4m3.
//
// The engine's prompt chunks (T of 64 and more) run their block-FP8 and K-quant linears
// here.  A matrix-core product with 16 significant bits of x needs two passes over the
// weights' operands; with x = hi + mid in bf16 (prefill.hip) both run at the 16-bit
// rate.  fp16 holds 11 of the bits, so the remainder fits e4m3's 4 and its pass runs at
// the 8-bit rate: 3/4 of the matrix-core time and 3/4 of the activation bytes.  Error of a
// product apart from the weights' rounding (normal inputs, channels 12 to 1e6 times as
// large, log-normal ones of sigma 1 to 6): block-FP8 4.7e-6 to 5.1e-6 (bf16 hi + mid, which
// truncates: 8.6e-6 to 1.03e-5), fp16 tiles, whose second pass rounds the weights, too,
// 7.1e-6 to 7.9e-6 (two fp16 passes over the same truncated x: as bf16 hi + mid).
//
// An input of T tokens and n columns (ActX, act_x_bytes):
//   s [kb][T]        power of two per (128-column block, token) that puts the block's
//                    largest |x| / s in [2^12, 2^13)
//   h [kb][i][g][T]  16-byte units, fp16(x / s) of columns 32g + 8i .. + 7
//   l [kb][c][g][T]  16-byte units, e4m3((x / s - h) * 2^7) of columns 32g + 16c .. + 15
// One s serves a block, so elements 2^-14 and more below their block's largest lose bits of
// l (absolute error 2^-29 of the largest), and from 2^-18 on hold the 11 bits of h; bf16 hi +
// mid keep 16 bits of each.  Only an output that the block's large elements do not reach
// (weights of 0) can show it.
// Weights: block-FP8 tiles, decoded to fp16 w * 2^7 for the first pass and taken as they
// are for the second; or the fp16 tiles of rl_hip_kquant_to_f16, taken as they are for
// the first and converted to e4m3(w / 2^7) for the second (the remainder carries 2^-12
// of x, so the 4 bits left of w add 2^-16 of the product).
#include <type_traits>

#include "prefill.h"

using namespace rl;

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;

union H8u {
    f16x8 v;
    uint32_t u[4];
    i32x4 i;
};

// ------------------------------------------------------------- writing inputs

// s for a block of largest magnitude mx; 1 / s is exact
__device__ inline float x_scale(float mx) {
    if (!(mx > 0.f)) return 1.f;
    int e;
    frexpf(mx, &e);
    return ldexpf(1.f, max(e, -100) - 13);
}

// 8 columns (unit col8 of the row) of token t: u = x / s
__device__ inline void write_x8(const ActX& o, int col8, int t, int T, const float (&u)[8]) {
    const int kb = col8 >> 4, jb = (col8 & 15) * 8;
    const int g = jb >> 5, i = (jb >> 3) & 3;
    H8u hh;
    int lo[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const _Float16 v = static_cast<_Float16>(u[4 * d + e]);
            hh.v[4 * d + e] = v;
            r[e] = (u[4 * d + e] - static_cast<float>(v)) * 128.f;
        }
        int p = __builtin_amdgcn_cvt_pk_fp8_f32(r[0], r[1], 0, false);
        lo[d] = __builtin_amdgcn_cvt_pk_fp8_f32(r[2], r[3], p, true);
    }
    o.h[((static_cast<size_t>(kb) * 4 + i) * 4 + g) * T + t] = hh.i;
    *reinterpret_cast<i32x2*>(reinterpret_cast<char*>(o.l + ((static_cast<size_t>(kb) * 2 + (i >> 1)) * 4 + g) * T + t) +
                              8 * (i & 1)) = i32x2{lo[0], lo[1]};
}

// Largest magnitude over the 16 lanes (one 128-column block) a lane belongs to.
__device__ inline float group16_max(float v) {
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    return v;
}

// A lane's 8 columns (unit col8, 16 consecutive lanes = one block) of token t.
__device__ inline void put_x8(const ActX& o, int col8, int t, int T, const float (&x)[8]) {
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
    const float s = x_scale(group16_max(mx)), inv = 1.f / s;
    float u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] = x[e] * inv;
    write_x8(o, col8, t, T, u);
    if ((col8 & 15) == 0) o.s[static_cast<size_t>(col8 >> 4) * T + t] = s;
}

// One wave per token and run of 64 units; n a multiple of 8 (columns past n are zeros).
__global__ __launch_bounds__(256) void pack_x_kernel(const float* __restrict__ X, ActX o, int n, int units, int T) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= T) return;
    for (int u = lane; u < units; u += 64) {
        float v[8];
        if (8 * u < n) {
            const float4* p = reinterpret_cast<const float4*>(X + static_cast<size_t>(t) * n) + 2 * u;
            const float4 a = p[0], b = p[1];
            v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = 0.f;
        }
        put_x8(o, u, t, T, v);
    }
}

// RMSNorm of prefill rows, one wave per token (rmsnorm_wave_kernel's arithmetic), written
// as an ActX and, when frag is given, as bf16 hi + mid fragments too.
template <int NU>
__global__ __launch_bounds__(256) void rmsnorm_x_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                        ActX o, i32x4* __restrict__ frag, int n, int T, float eps) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= T) return;  // whole waves
    const float* xt = x + static_cast<size_t>(t) * n;
    const int nu = n / 8;
    float v[NU][8];
    double ss = 0.0;
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const int u = lane + 64 * k;
        if (u < nu) {
            const float4 a = reinterpret_cast<const float4*>(xt)[2 * u];
            const float4 b = reinterpret_cast<const float4*>(xt)[2 * u + 1];
            v[k][0] = a.x, v[k][1] = a.y, v[k][2] = a.z, v[k][3] = a.w;
            v[k][4] = b.x, v[k][5] = b.y, v[k][6] = b.z, v[k][7] = b.w;
        }
    }
#pragma unroll
    for (int k = 0; k < NU; ++k)
        if (lane + 64 * k < nu)
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += static_cast<double>(v[k][e]) * v[k][e];
    ss = wave_sum_d(ss);
    const float inv = 1.f / sqrtf(static_cast<float>(ss / n) + eps);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const int u = lane + 64 * k;
        if (u >= nu) break;  // n is a multiple of 128: whole blocks leave together
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = v[k][e] * inv * (gamma ? 1.f + gamma[8 * u + e] : 1.f);
        put_x8(o, u, t, T, y);
        if (frag) write_frag8(frag, u, t, T, y);
    }
}

// Gated RMSNorm per 128-wide head (gnorm_pack128_kernel's arithmetic, expf included) as an ActX.
__global__ __launch_bounds__(256) void gnorm_x_kernel(const float* __restrict__ o, const float* __restrict__ z, int ld_z,
                                                      const float* __restrict__ gamma, ActX out,
                                                      int n, int T, float eps) {
    const int t = blockIdx.y, tid = threadIdx.x;
    const int hh = blockIdx.x * 16 + (tid >> 4), u = tid & 15;
    if (hh * 128 >= n) return;  // whole 16-lane groups
    const int c0 = hh * 128 + 8 * u;
    const float4* op = reinterpret_cast<const float4*>(o + static_cast<size_t>(t) * n + c0);
    const float4* zp = reinterpret_cast<const float4*>(z + static_cast<size_t>(t) * ld_z + c0);
    const float4 o0 = op[0], o1 = op[1], z0 = zp[0], z1 = zp[1];
    const float ov[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
    const float zv[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
    double ss = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += static_cast<double>(ov[e]) * ov[e];
    ss = group16_sum_d(ss);
    const float inv = 1.f / sqrtf(static_cast<float>(ss / 128) + eps);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        v[e] = (gamma ? gamma[8 * u + e] : 1.f) * (ov[e] * inv) * (zv[e] / (1.f + expf(-zv[e])));
    put_x8(out, c0 >> 3, t, T, v);
}

// ------------------------------------------------------------------- the GEMM

// All of a wave's loads have arrived and its LDS reads are done; then all waves'.
__device__ inline void full_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }


struct GemmX {
    const uint8_t* W;
    const float* ts;
    ActX x;
    float* Y;
    ActX out;  // epilogue kEpiSwiGLUHX
    int m, n_kb, T, ldy, m_valid, nrb, ntb, epi, vec;
    int rt_base;  // first row tile of the launch
};

// Workgroup: 2 x TG waves; 4R row tiles (64R rows) x 64 TG tokens; wave (rg, tg) owns R
// pairs of row tiles (32-row A operands) and two 32-token B operands, so a converted
// weight fragment feeds both.  A half column block (64 of 128 columns) of weights and
// activations is copied global -> LDS (double buffered, straight, without registers)
// while the previous one is multiplied; one barrier per half block.  The block scales
// multiply each half block's fp32 partial.
// WK 0: block-FP8 tiles; 3: fp16 tiles.  kGuh (WK 0): two scales per tile.
//
// Bound by matrix-core power and issue: 34816 x 5120, 2044 tokens, block-FP8: MFMA units 60%
// busy at 1.8 GHz, 7.6 VALU instructions per MFMA, no LDS conflicts; without any copy into LDS after the first block (timing only) a launch is
// 14% shorter, with every copy hitting the same cache lines 7%.  34816 x 5120, 2044
// tokens, SwiGLU to inputs: block-FP8 1071 us (680 TFLOP/s of useful products; 1200 us
// for the bf16 hi + mid kernel), fp16 tiles 1049 us (2300 us for two fp16 passes on
// 16x16 MFMA).  Registers set the rest: 128 accumulators, so the e4m3 parts of the
// tokens are read again for each row pair, and a spilled variant runs at half speed.
template <int WK, bool kGuh, int R, int TG>
__global__ __launch_bounds__(128 * TG, 2) void gemm_x_kernel(GemmX p) {
    constexpr int NW = 2 * TG, RT = 4 * R;
    constexpr int kAC = WK == 0 ? 1 : 2;                  // 1 KiB chunks per tile and half block
    constexpr int kAQ = (RT * kAC + NW - 1) / NW;         // of them per wave
    constexpr int GW = 16 / TG;                           // token blocks an XCD takes side by side
    __shared__ i32x4 A0[RT * kAC * 64], A1[RT * kAC * 64];  // [tile][chunk][lane of the packed tile]
    __shared__ i32x4 B0[NW * 6 * 64], B1[NW * 6 * 64];      // [32 tokens][4 fp16 steps, 2 e4m3 parts][lane]

    int rb, tb;
    if (!xcd_block(p.nrb, p.ntb, GW, rb, tb)) return;

    const int T = p.T, n_kb = p.n_kb;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = wave / TG, tg = wave % TG;
    const int h = lane >> 5, col = lane & 31;
    const int m_tiles = (p.m + kTileRows - 1) / kTileRows;
    const int rt0 = p.rt_base + rb * RT;
    const int tok0 = tb * 64 * TG + 64 * tg;
    const bool live = tok0 < T;  // wave-uniform
    const int last_hb = 2 * n_kb - 1;

    const uint32_t tileb = static_cast<uint32_t>(n_kb) * (WK == 0 ? 2048u : 4096u);  // bytes per row tile
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.W), 0, static_cast<int>(static_cast<uint32_t>(m_tiles) * tileb), 0x00020000);
    const __amdgpu_buffer_rsrc_t hr =
        __builtin_amdgcn_make_buffer_rsrc(p.x.h, 0, static_cast<int>(static_cast<uint32_t>(n_kb) * 256u * T), 0x00020000);
    const __amdgpu_buffer_rsrc_t lr =
        __builtin_amdgcn_make_buffer_rsrc(p.x.l, 0, static_cast<int>(static_cast<uint32_t>(n_kb) * 128u * T), 0x00020000);
    // B copies: wave w brings tokens 32w .. 32w+31 of the block
    const int bvoff = (h * T + min(tb * 64 * TG + 32 * wave + col, T - 1)) * 16;
    auto dma = [&](int hb_, i32x4* A, i32x4* B) {
        const int hb = min(hb_, last_hb);
#pragma unroll
        for (int q = 0; q < kAQ; ++q) {
            const int ch = min(wave + NW * q, RT * kAC - 1);  // (a clamped wave copies the last chunk again)
            const uint32_t so = static_cast<uint32_t>(min(rt0 + ch / kAC, m_tiles - 1)) * tileb +
                                (static_cast<uint32_t>(hb) * kAC + ch % kAC) * 1024u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(A + ch * 64), 16, 16 * lane, static_cast<int>(so), 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)  // step s = 2i + p: unit row (kb, 2c + i, g = 2p + h)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                hr, (lds_void*)(B + (wave * 6 + s) * 64), 16, bvoff,
                static_cast<int>((static_cast<uint32_t>(hb) * 8u + 4u * (s >> 1) + 2u * (s & 1)) * 16u * T), 0, 0);
#pragma unroll
        for (int s = 0; s < 2; ++s)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                lr, (lds_void*)(B + (wave * 6 + 4 + s) * 64), 16, bvoff,
                static_cast<int>((static_cast<uint32_t>(hb) * 4u + 2u * s) * 16u * T), 0, 0);
    };

    // lane j holds the block scale of the wave's tile j (kGuh: of half j % 2 of tile j / 2)
    constexpr bool k2 = WK == 0 && kGuh;
    const __amdgpu_buffer_rsrc_t tr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.ts), 0, m_tiles * n_kb * (k2 ? 8 : 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(p.x.s, 0, n_kb * T * 4, 0x00020000);
    const int st = min(rt0 + 2 * R * rg + min(k2 ? lane / 2 : lane, 2 * R - 1), m_tiles - 1);
    const int tvoff = k2 ? (st * n_kb * 2 + (lane & 1)) * 4 : st * n_kb * 4;
    const int xvoff = (tok0 + col) * 4;  // (tokens past the last one read other scales, or 0 past the end)
    constexpr float kUnit = WK == 0 ? 1.f / 128.f : 1.f;  // decoded block-FP8 weights are w * 2^7
    struct Sc {
        float w, x[2];
    };
    auto load_f = [](__amdgpu_buffer_rsrc_t r, int voff, int soff) {
        return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    };
    auto load_sc = [&](int kb) {
        Sc s;
        s.w = load_f(tr, tvoff, kb * (k2 ? 8 : 4)) * kUnit;
        s.x[0] = load_f(sr, xvoff, kb * T * 4);
        s.x[1] = load_f(sr, xvoff + 128, kb * T * 4);
        return s;
    };

    f32x16 tot[R][2], acc[2];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) tot[r][n][v] = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[1][v] = 0.f;

    // quarter q of tot[r][n] += (tile scale * x scale) * acc[n]
    auto add_scaled = [&](int r, int n, int q, const Sc& s) {
        const float f =
            __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s.w), k2 ? 4 * r + q : 2 * r + q / 2)) * s.x[n];
#pragma unroll
        for (int v = 4 * q; v < 4 * q + 4; ++v) tot[r][n][v] = fmaf(f, acc[n][v], tot[r][n][v]);
    };
    auto mf16 = [](const H8u& a, const H8u& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, b.v, c, 0, 0, 0);
    };
    auto mf8 = [](const i32x8& a, const i32x8& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
    };
    const int aoff = (2 * R * rg + (col >> 4)) * kAC * 64 + h * 16 + (col & 15);
    const int boff = 2 * tg * 6 * 64 + lane;
    // One half block; s: its scales, sprev: those of the pending acc[1] (the last row pair's
    // second token operand).  The order is pinned: each MFMA is followed by the work that
    // fits under it (a quarter of a finished partial's scaled add, the next fragments).
    auto half = [&](const i32x4* A, const i32x4* B, const Sc& s, const Sc& sprev) {
        H8u af[4], bf[2][4];
        i32x8 a8, b8[2];
        const i32x4* ap = A + aoff;
        const i32x4* bp = B + boff;
        f32x16 z;
#pragma unroll
        for (int v = 0; v < 16; ++v) z[v] = 0.f;
        auto ld8 = [](const i32x4& x, const i32x4& y) { return i32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}; };
        // WK 0: dword d of a8's part p holds 4 weights; step s = 2i + p takes dwords 2i, 2i + 1
        auto cvt16 = [&](int st) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int w = a8[4 * (st & 1) + 2 * (st >> 1) + d];
                af[st].u[2 * d] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 128.f, false));
                af[st].u[2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 128.f, true));
            }
        };
        // WK 3: the e4m3 of af[st]
        auto cvt8 = [&](int st) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                s16x2 c = {0, 0};
                c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(c, f16x2{af[st].v[4 * d], af[st].v[4 * d + 1]}, 128.f, false);
                c = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(c, f16x2{af[st].v[4 * d + 2], af[st].v[4 * d + 3]}, 128.f, true);
                a8[4 * (st & 1) + 2 * (st >> 1) + d] = __builtin_bit_cast(int, c);
            }
        };
        auto ld16 = [&](int r, int st) { af[st].i = ap[(2 * r * kAC + (st >> 1)) * 64 + 32 * (st & 1)]; };
        if constexpr (WK == 0) {
            a8 = ld8(ap[0], ap[32]);
        } else {
#pragma unroll
            for (int st = 0; st < 4; ++st) ld16(0, st);
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int st = 0; st < 4; ++st) bf[n][st].i = bp[(n * 6 + st) * 64];
            if (WK == 3 && n == 0) b8[0] = ld8(bp[4 * 64], bp[5 * 64]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Sc& sp1 = r ? s : sprev;
            const int rp = r ? r - 1 : R - 1;
            // first token operand
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                if constexpr (WK == 0)
                    if (st == 0) cvt16(0);
                acc[0] = mf16(af[st], bf[0][st], st ? acc[0] : z);
                if constexpr (WK == 3) {
                    cvt8(st);
                } else {
                    if (st < 3) cvt16(st + 1);
                    if (st == 1) b8[0] = ld8(bp[4 * 64], bp[5 * 64]);  // (not kept over r: registers)
                }
                if (st) add_scaled(rp, 1, st - 1, sp1);
                __builtin_amdgcn_sched_barrier(0);
            }
            acc[0] = mf8(a8, b8[0], acc[0]);
            b8[1] = ld8(bp[10 * 64], bp[11 * 64]);  // (read for each r: registers)
            add_scaled(rp, 1, 3, sp1);
            __builtin_amdgcn_sched_barrier(0);
            // second; the next row pair's weights follow their last use
            acc[1] = mf16(af[0], bf[1][0], z);
            if constexpr (WK == 3)
                if (r + 1 < R) ld16(r + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            acc[1] = mf8(a8, b8[1], acc[1]);
            if constexpr (WK == 0)
                if (r + 1 < R) a8 = ld8(ap[2 * (r + 1) * 64], ap[2 * (r + 1) * 64 + 32]);
            add_scaled(r, 0, 0, s);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 1; st < 4; ++st) {
                acc[1] = mf16(af[st], bf[1][st], acc[1]);
                if constexpr (WK == 3)
                    if (r + 1 < R) ld16(r + 1, st);
                add_scaled(r, 0, st, s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    dma(0, A0, B0);
    Sc s = load_sc(0), sprev = {0.f, {0.f, 0.f}};
    full_barrier();
    for (int kb = 0; kb < n_kb; ++kb) {
        dma(2 * kb + 1, A1, B1);
        if (live) half(A0, B0, s, sprev);
        full_barrier();
        dma(2 * kb + 2, A0, B0);
        const Sc sn = load_sc(min(kb + 1, n_kb - 1));
        if (live) half(A1, B1, s, s);
        sprev = s;
        s = sn;
        full_barrier();
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) add_scaled(R - 1, 1, q, sprev);

    // lane (h, col) holds rows 8u + 4h + v (u = 0..3, v = 0..3) of each row pair for tokens
    // tok0 + 32 n + col
    const int rtw = rt0 + 2 * R * rg;
    if constexpr (kGuh) {
        // tot[r][n][8j .. 8j+3] becomes the SwiGLU output rows 4h .. 4h+3 of half tile 2r + j
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) tot[r][n][8 * j + v] = silu_fast(tot[r][n][8 * j + v]) * tot[r][n][8 * j + 4 + v];
        if constexpr (R == 4) {
            if (p.epi == kEpiSwiGLUHX) {
                // the workgroup's 128 outputs are one column block of the next input: its
                // largest magnitude per token over both row groups, through LDS
                float* smax = reinterpret_cast<float*>(A0);
                float mx[2] = {0.f, 0.f};
#pragma unroll
                for (int n = 0; n < 2; ++n) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int v = 0; v < 4; ++v) mx[n] = fmaxf(mx[n], fabsf(tot[r][n][8 * j + v]));
                    mx[n] = fmaxf(mx[n], __shfl_xor(mx[n], 32, 64));
                    if (h == 0) smax[(rg * TG + tg) * 64 + 32 * n + col] = mx[n];
                }
                __syncthreads();
                const int ob = rt0 / 16;  // the output's column block
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const int tok = tok0 + 32 * n + col;
                    const float sx = x_scale(fmaxf(mx[n], smax[((1 - rg) * TG + tg) * 64 + 32 * n + col]));
                    const float inv = 1.f / sx;
                    if (tok >= T) continue;
                    if (rg == 0 && h == 0) p.out.s[static_cast<size_t>(ob) * T + tok] = sx;
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const int u8 = 2 * R * rg + 2 * r + j, g = u8 >> 2, i = u8 & 3;
                            union {
                                _Float16 e[4];
                                i32x2 q;
                            } hh;
                            float rr[4];
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                const float u = tot[r][n][8 * j + v] * inv;
                                hh.e[v] = static_cast<_Float16>(u);
                                rr[v] = (u - static_cast<float>(hh.e[v])) * 128.f;
                            }
                            int lo = __builtin_amdgcn_cvt_pk_fp8_f32(rr[0], rr[1], 0, false);
                            lo = __builtin_amdgcn_cvt_pk_fp8_f32(rr[2], rr[3], lo, true);
                            char* hd = reinterpret_cast<char*>(p.out.h + ((static_cast<size_t>(ob) * 4 + i) * 4 + g) * T + tok);
                            *reinterpret_cast<i32x2*>(hd + 8 * h) = hh.q;
                            char* ld = reinterpret_cast<char*>(p.out.l + ((static_cast<size_t>(ob) * 2 + (i >> 1)) * 4 + g) * T + tok);
                            *reinterpret_cast<int*>(ld + 8 * (i & 1) + 4 * h) = lo;
                        }
                }
                return;
            }
        }
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int tok = tok0 + 32 * n + col;
        if (tok >= T) continue;
        float* yrow = p.Y + static_cast<size_t>(tok) * p.ldy;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int rt = rtw + 2 * r;
            if constexpr (kGuh) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (rt + j >= m_tiles) break;
                    float o4[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) o4[v] = tot[r][n][8 * j + v];
                    const int row = (rt + j) * 8 + 4 * h;
                    store_rows4(yrow + row, o4, p.m_valid - row, p.vec, false);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    float o4[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) o4[v] = tot[r][n][4 * u + v];
                    const int row = rt * kTileRows + 8 * u + 4 * h;
                    store_rows4(yrow + row, o4, p.m_valid - row, p.vec, p.epi == kEpiAdd);
                }
            }
        }
    }
}

template <int WK, bool kGuh, int R, int TG>
void launch_gemm_x_cfg(GemmX p, int rt_base, int row_blocks, hipStream_t s) {
    p.rt_base = rt_base;
    p.nrb = row_blocks;
    p.ntb = (p.T + 64 * TG - 1) / (64 * TG);
    hipLaunchKernelGGL((gemm_x_kernel<WK, kGuh, R, TG>), dim3((p.nrb * p.ntb + 7) / 8 * 8), dim3(128 * TG), 0, s, p);
    check_launch("gemm_x_kernel");
}

// Row blocks of 64 r rows from a row tile on, in blocks of 64 tg tokens.
struct XSplit {
    int r = 0, tg = 0, blocks = 0;
};

// The work split: 256, 192 or 128 rows (r = 4, 3, 2) x 256 or 128 tokens (tg = 4, 2) per
// workgroup.  A CU holds one workgroup, and of block-FP8 two of 128 tokens, which is why
// block-FP8 takes no others (their barriers fall at different times: 32768 x 5120, 2048
// tokens, 955 us against 1037 with 256 tokens); a round of workgroups takes about 2r + 1
// units.  A lone 4-wave workgroup on a CU takes 0.65 of that.  When whole rounds leave a
// small remainder of row blocks, those rows are a launch of their own with another split
// (34816 rows, 2044 tokens in fp16 tiles: 5 rounds of 256 x 256 with the last one a quarter
// full).  x_out: outputs in whole column blocks, 256 rows.  The sums of an output do not
// depend on the split.
void gemm_x_split(int wk, bool x_out, int m, int T, int cus, XSplit& first, XSplit& rest) {
    static constexpr XSplit kSplits[] = {{4, 4}, {3, 4}, {2, 4}, {4, 2}, {3, 2}, {2, 2}};
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    auto skip = [&](const XSplit& c) { return (x_out && c.r != 4) || (wk == 0 && c.tg != 2); };
    auto blocks = [](const XSplit& c, int tiles) { return (tiles + 4 * c.r - 1) / (4 * c.r); };
    auto ntb = [&](const XSplit& c) { return (T + 64 * c.tg - 1) / (64 * c.tg); };
    auto slots = [&](const XSplit& c) { return wk == 0 ? 2 * cus : cus; };
    auto cost = [&](const XSplit& c, long wgs) {
        const double unit = (2 * c.r + 1) * (c.tg == 4 ? 1.0 : wk == 0 ? 0.95 : 0.65);
        const long full = wgs / slots(c), rem = wgs % slots(c);
        return unit * (full + (rem == 0 ? 0.0 : wk == 0 && rem <= cus ? 0.65 : 1.0));
    };
    double best = 0;
    for (const XSplit& c : kSplits) {
        if (skip(c)) continue;
        const int nb = blocks(c, m_tiles);
        const long wgs = static_cast<long>(nb) * ntb(c);
        RL_REQUIRE(wgs < (1L << 30), RL_ERR_RANGE, "gemm_x: too many workgroups");
        const double t = cost(c, wgs);
        if (!first.blocks || t < best) {
            best = t;
            first = {c.r, c.tg, nb};
            rest = {};
        }
        const int nb1 = static_cast<int>(wgs / slots(c) * slots(c) / ntb(c));
        if (nb1 == 0 || nb1 == nb) continue;
        for (const XSplit& c2 : kSplits) {
            if (skip(c2)) continue;
            const int nb2 = blocks(c2, m_tiles - nb1 * 4 * c.r);
            // a second launch costs about a third of a unit
            const double t2 = cost(c, static_cast<long>(nb1) * ntb(c)) + cost(c2, static_cast<long>(nb2) * ntb(c2)) + 0.35;
            if (t2 < best) {
                best = t2;
                first = {c.r, c.tg, nb1};
                rest = {c2.r, c2.tg, nb2};
            }
        }
    }
}

template <int WK, bool kGuh>
void launch_gemm_x(const GemmX& p, hipStream_t s) {
    XSplit first, rest;
    gemm_x_split(WK, p.epi == kEpiSwiGLUHX, p.m, p.T, device_cus(), first, rest);
    auto launch = [&](const XSplit& c, int rt_base) {
        if constexpr (WK == 3) {
            if (c.tg == 4) {
                if (c.r == 4) launch_gemm_x_cfg<WK, kGuh, 4, 4>(p, rt_base, c.blocks, s);
                if (c.r == 3) launch_gemm_x_cfg<WK, kGuh, 3, 4>(p, rt_base, c.blocks, s);
                if (c.r == 2) launch_gemm_x_cfg<WK, kGuh, 2, 4>(p, rt_base, c.blocks, s);
                return;
            }
        }
        if (c.r == 4) launch_gemm_x_cfg<WK, kGuh, 4, 2>(p, rt_base, c.blocks, s);
        if (c.r == 3) launch_gemm_x_cfg<WK, kGuh, 3, 2>(p, rt_base, c.blocks, s);
        if (c.r == 2) launch_gemm_x_cfg<WK, kGuh, 2, 2>(p, rt_base, c.blocks, s);
    };
    launch(first, 0);
    if (rest.blocks) launch(rest, first.blocks * 4 * first.r);
}

}  // namespace

namespace rl {

size_t act_x_bytes(int n, int T) {
    const size_t kb = (n + 127) / 128;
    return kb * T * (256 + 128 + 4) + 512;
}

ActX act_x_at(void* mem, int n, int T) {
    const size_t kb = (n + 127) / 128;
    char* c = static_cast<char*>(mem);
    ActX x;
    x.h = reinterpret_cast<i32x4*>(c);
    x.l = reinterpret_cast<i32x4*>(c + kb * T * 256);
    x.s = reinterpret_cast<float*>(c + kb * T * 384);
    return x;
}

bool rmsnorm_x_supported(int n) { return n % 128 == 0 && n <= 64 * 12 * 8; }

void rmsnorm_x(const float* x, const float* gamma, const ActX& out, void* frag, int n, int T, float eps, hipStream_t s) {
    RL_REQUIRE(x && out.h && rmsnorm_x_supported(n) && T >= 1, RL_ERR_RANGE, "rmsnorm_x: bad arguments");
    RL_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0, RL_ERR_RANGE, "rmsnorm_x: rows must be 16-byte aligned");
    const dim3 grid((T + 3) / 4);
    i32x4* f = static_cast<i32x4*>(frag);
    if (n <= 64 * 4 * 8)
        hipLaunchKernelGGL(rmsnorm_x_kernel<4>, grid, dim3(256), 0, s, x, gamma, out, f, n, T, eps);
    else if (n <= 64 * 8 * 8)
        hipLaunchKernelGGL(rmsnorm_x_kernel<8>, grid, dim3(256), 0, s, x, gamma, out, f, n, T, eps);
    else
        hipLaunchKernelGGL(rmsnorm_x_kernel<12>, grid, dim3(256), 0, s, x, gamma, out, f, n, T, eps);
    check_launch("rmsnorm_x_kernel");
}

void gnorm_x(const float* o, const float* z, int ld_z, const float* gamma, const ActX& out, int n, int T, float eps,
             hipStream_t s) {
    RL_REQUIRE(o && z && out.h && n > 0 && n % 128 == 0 && T >= 1 && T <= 65535, RL_ERR_RANGE, "gnorm_x: bad arguments");
    RL_REQUIRE(reinterpret_cast<uintptr_t>(o) % 16 == 0 && reinterpret_cast<uintptr_t>(z) % 16 == 0 && ld_z % 4 == 0,
               RL_ERR_RANGE, "gnorm_x: rows must be 16-byte aligned");
    hipLaunchKernelGGL(gnorm_x_kernel, dim3((n / 128 + 15) / 16, T), dim3(256), 0, s, o, z, ld_z, gamma, out, n, T,
                       eps);
    check_launch("gnorm_x_kernel");
}

void pack_x(const float* X, const ActX& out, int n, int T, hipStream_t s) {
    RL_REQUIRE(X && out.h && n > 0 && n % 8 == 0 && T >= 1, RL_ERR_RANGE, "pack_x: bad arguments");
    RL_REQUIRE(reinterpret_cast<uintptr_t>(X) % 16 == 0, RL_ERR_RANGE, "pack_x: rows must be 16-byte aligned");
    hipLaunchKernelGGL(pack_x_kernel, dim3((T + 3) / 4), dim3(256), 0, s, X, out, n, (n + 127) / 128 * 16, T);
    check_launch("pack_x_kernel");
}

void gemm_x(int wk, const uint8_t* W, const float* ts, const ActX& x, float* Y, int m, int n, int T, int epi, int ldy,
            int m_valid, hipStream_t s, const ActX* out) {
    RL_REQUIRE(wk == 0 || wk == 3, RL_ERR_RANGE, "gemm_x: weight kind");
    RL_REQUIRE(m > 0 && n > 0 && T >= 1 && W && ts && x.h && x.l && x.s, RL_ERR_RANGE, "gemm_x: bad arguments");
    RL_REQUIRE(epi == kEpiStore || epi == kEpiAdd || epi == kEpiSwiGLUH || epi == kEpiSwiGLUHX, RL_ERR_RANGE,
               "gemm_x: epilogue must be store, add or swiglu over half tiles");
    RL_REQUIRE(epi == kEpiSwiGLUHX ? out && out->h : Y != nullptr, RL_ERR_RANGE, "gemm_x: null output");
    if (epi == kEpiSwiGLUH) RL_REQUIRE(m % 16 == 0, RL_ERR_RANGE, "gemm_x swiglu: rows a multiple of 16");
    if (epi == kEpiSwiGLUHX)
        RL_REQUIRE(m % 256 == 0, RL_ERR_RANGE, "gemm_x swiglu to inputs: outputs a multiple of 128");
    const int n_kb = (n + 127) / 128, m_tiles = (m + kTileRows - 1) / kTileRows;
    // the kernel addresses weights and inputs with 32-bit offsets
    RL_REQUIRE(static_cast<size_t>(m_tiles) * n_kb * (wk == 0 ? 2048 : 4096) < (size_t{1} << 32) &&
                   static_cast<size_t>(n_kb) * T * 256 < (size_t{1} << 32),
               RL_ERR_RANGE, "gemm_x: weights and inputs must each stay under 4 GiB");
    GemmX p{};
    p.W = W;
    p.ts = ts;
    p.x = x;
    p.Y = Y;
    if (out) p.out = *out;
    p.m = m;
    p.n_kb = n_kb;
    p.T = T;
    p.ldy = ldy;
    p.m_valid = m_valid;
    p.epi = epi;
    p.vec = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
    const bool guh = epi == kEpiSwiGLUH || epi == kEpiSwiGLUHX;
    if (wk == 0)
        (guh ? launch_gemm_x<0, true> : launch_gemm_x<0, false>)(p, s);
    else
        (guh ? launch_gemm_x<3, true> : launch_gemm_x<3, false>)(p, s);
}

}  // namespace rl

extern "C" {

size_t rl_hip_act_x_bytes(int n, int T) { return rl::act_x_bytes(n, T); }

int rl_hip_pack_act_x(const float* X, void* x, int n, int T, void* stream) {
    return guard([&] {
        RL_REQUIRE(x && n > 0 && T > 0, RL_ERR_RANGE, "pack_act_x: bad arguments");
        rl::pack_x(X, rl::act_x_at(x, n, T), n, T, S(stream));
    });
}

int rl_hip_rmsnorm_x(const float* rows, const float* gamma, void* x, int n, int T, float eps, void* stream) {
    return guard([&] {
        RL_REQUIRE(x && n > 0 && T > 0, RL_ERR_RANGE, "rmsnorm_x: bad arguments");
        rl::rmsnorm_x(rows, gamma, rl::act_x_at(x, n, T), nullptr, n, T, eps, S(stream));
    });
}

int rl_hip_gated_rmsnorm_x(const float* o, const float* z, int ld_z, const float* gamma, void* x, int n, int T, float eps,
                           void* stream) {
    return guard([&] {
        RL_REQUIRE(x && n > 0 && T > 0, RL_ERR_RANGE, "gated_rmsnorm_x: bad arguments");
        rl::gnorm_x(o, z, ld_z, gamma, rl::act_x_at(x, n, T), n, T, eps, S(stream));
    });
}

int rl_hip_gemm_x(int fp16_tiles, const void* w, const float* tile_scale, const void* x, float* Y, void* x_out, int m, int n,
                  int T, int epilogue, int ldy, void* stream) {
    return guard([&] {
        RL_REQUIRE(x && m > 0 && n > 0 && T > 0, RL_ERR_RANGE, "gemm_x: bad arguments");
        const bool to_x = epilogue == rl::kEpiSwiGLUHX;
        RL_REQUIRE(!to_x || x_out, RL_ERR_RANGE, "gemm_x: null output");
        const int mo = to_x || epilogue == rl::kEpiSwiGLUH ? m / 2 : m;
        const rl::ActX out = to_x ? rl::act_x_at(x_out, mo, T) : rl::ActX{};
        rl::gemm_x(fp16_tiles ? 3 : 0, static_cast<const uint8_t*>(w), tile_scale, rl::act_x_at(const_cast<void*>(x), n, T),
                   Y, m, n, T, epilogue, ldy > 0 ? ldy : mo, mo, S(stream), to_x ? &out : nullptr);
    });
}

int rl_hip_gemm_x_split(int fp16_tiles, int epilogue, int m, int T, int cus, int* split) {
    return guard([&] {
        RL_REQUIRE(m > 0 && T > 0 && cus > 0 && split, RL_ERR_RANGE, "gemm_x_split: bad arguments");
        XSplit first, rest;
        gemm_x_split(fp16_tiles ? 3 : 0, epilogue == rl::kEpiSwiGLUHX, m, T, cus, first, rest);
        const int v[6] = {first.r, first.tg, first.blocks, rest.r, rest.tg, rest.blocks};
        for (int k = 0; k < 6; ++k) split[k] = v[k];
    });
}

}  // extern "C"
