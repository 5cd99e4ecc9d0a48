// prefill.hip -- block-FP8 linears over many tokens (prompt prefill), on MFMA.
//
// Same arithmetic as ops::gemv_fp8 (reference src/kernels/ops.cpp:182-194) applied
// to every prompt token, i.e. the reference's prefill linears
// (src/kernels/cuda/cuda_engine.cu:18338-18590 launch_prefill_chunk -> launch_linear
// for T > 8, cuda_engine.cu:12008-12016).  At prefill sizes the work is matrix-core
// bound, not HBM bound; at few tokens it is the weight stream, and waves split K.
//
// Operands: A = weight rows, e4m3 decoded to bf16 by the hardware converter (exact); B =
// tokens of the activation fragments (bf16 hi and mid parts, two MFMAs into the same
// accumulator, so products carry 16 significant bits of x); the 128x128 block scale
// multiplies a column block's fp32 partial.  Weights use the decode GEMM's tiled layout
// (16 rows x 128 columns per 2 KiB tile), activations its fragment layout for T tokens.
//
// Two kernels: gemm_fp8_pf_kernel for the block-FP8 tiles (32x32 MFMA), and
// gemm_prefill_kernel for BF16 and fp16 tiles (16x16 MFMA).
#include <type_traits>

#include "prefill.h"

using namespace rl;

namespace {

constexpr int kPfNT = 2;     // 16-token column tiles per wave
constexpr int kPfTok = 64 * kPfNT;  // tokens per workgroup

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

union Frag8 {
    bf16x8 v;
    f16x8 h;
    uint32_t u[4];
    i32x4 i;
};

__device__ inline void e4m3x4_to_bf16(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const bf16x2_t a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(w), 1.0f, false);
    const bf16x2_t b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(static_cast<int>(w), 1.0f, true);
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, b);
}

// A barrier that waits for this wave's LDS accesses only (loads to registers stay in
// flight across it).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// EPI: 0 store, 1 add (Y += W.x), 2 SwiGLU over interleaved gate/up row tiles
// (even tile = gate rows, odd = up rows of the same 16 outputs; Y row = output row),
// 5 SwiGLU over half tiles (tile k: gate rows 8k..8k+7, up rows 8k..8k+7; scales
// [tile][kb][2]).
// WK: the weight tiles.  1: BF16 (4 KiB tiles of the decode GEMM's BF16 layout, no
// scales).  2: two BF16 matrices W_hi + W_lo (a weight split into 16 significant bits): three MFMAs per step,
// hi.x_hi + hi.x_mid + lo.x_hi.  3: fp16 tiles in the BF16 layout with one
// power-of-two scale per (tile, column block) (the K-quant linears as dequantised
// for prefill), activations as fp16 hi + lo fragments with one power-of-two scale
// per (column block, token): two fp16 MFMAs per step.
// Workgroup: 4 waves, 4 row tiles x 128 tokens; wave w owns tokens 32w .. 32w+31 (two
// 16-token column tiles, so each weight fragment read from LDS feeds four MFMAs).  The
// weight tiles of a column block (16 KiB; 32 KiB for hi + lo) are staged in LDS, double
// buffered, the next block's loads in flight during the MFMAs.
template <int EPI, int WK>
__global__ __launch_bounds__(256) void gemm_prefill_kernel(const uint8_t* __restrict__ W,
                                                           const float* __restrict__ tscale,
                                                           const i32x4* __restrict__ frag, float* __restrict__ Y,
                                                           int m, int n_kb, int T, int ldy, int m_valid,
                                                           const uint8_t* __restrict__ W_lo = nullptr,
                                                           const float* __restrict__ xscale = nullptr) {
    constexpr int kPfRT = 4;      // row tiles per workgroup (fp16 at 8: one wave per SIMD, slower)
    constexpr int kCh = 4;        // 16-B chunks per lane per tile
    constexpr int kTileB = 4096;  // bytes per tile
    constexpr int kMat = WK == 2 ? 2 : 1;           // weight matrices staged
    constexpr int kUnits = kPfRT * kCh * 64 * kMat / 256;  // 16-B staging units per thread
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, col = lane & 15;
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    const int rt0 = blockIdx.x * kPfRT;
    int tokv[kPfNT], tokcv[kPfNT];
#pragma unroll
    for (int nt = 0; nt < kPfNT; ++nt) {
        tokv[nt] = blockIdx.y * kPfTok + (wave * kPfNT + nt) * 16 + col;  // B column of this lane
        tokcv[nt] = min(tokv[nt], T - 1);
    }
    const int NC = 2 * T;
    // the input fragments as a buffer resource (gfx9 raw dword buffer; the host keeps
    // them under 4 GiB) and the byte offset of the unit of (k-step i, lane group g,
    // token) within a column block
    const __amdgpu_buffer_rsrc_t frsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<i32x4*>(frag), 0, static_cast<int>(static_cast<uint32_t>(n_kb) * 16u * 2u * T * 16u), 0x00020000);
    uint32_t boff[kPfNT][4];
#pragma unroll
    for (int nt = 0; nt < kPfNT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) boff[nt][i] = static_cast<uint32_t>((i * 4 + g) * NC + tokcv[nt]) * 16u;

    __shared__ i32x4 wl[2][kMat][kPfRT][kCh][64];  // [buffer][matrix][row tile][16-B chunk][lane]

    // staging: unit u = (matrix, row tile, chunk, lane), kUnits per thread.  Every
    // address is a uniform base for the column block plus a loop-invariant 32-bit
    // lane offset (the host keeps weights and fragments under 4 GiB), so the loads
    // take the scalar-base form with no 64-bit address arithmetic per iteration.
    uint32_t woff[kUnits];
#pragma unroll
    for (int q = 0; q < kUnits; ++q) {
        const int u = tid + 256 * q;
        const int l = u & 63, c = (u >> 6) % kCh, r = (u / (64 * kCh)) % kPfRT;
        const int rt = min(rt0 + r, m_tiles - 1);
        woff[q] = static_cast<uint32_t>(rt) * static_cast<uint32_t>(n_kb * kTileB) + c * 1024 + 16 * l;
    }
    // weights as buffer resources too (non-temporal loads: aux bit 1)
    const int wbytes = static_cast<int>(static_cast<uint32_t>(m_tiles) * static_cast<uint32_t>(n_kb * kTileB));
    const __amdgpu_buffer_rsrc_t wrsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(W), 0, wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t wlrsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(kMat > 1 ? W_lo : W), 0, wbytes, 0x00020000);
    i32x4 stg[kUnits];
    auto stage_load = [&](int kb) {
#pragma unroll
        for (int q = 0; q < kUnits; ++q) {
            const int mat = (tid + 256 * q) / (64 * kCh * kPfRT);
            stg[q] = __builtin_amdgcn_raw_buffer_load_b128(mat ? wlrsrc : wrsrc, static_cast<int>(woff[q]),
                                                           kb * kTileB, 2);
        }
    };
    auto stage_store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kUnits; ++q) {
            const int u = tid + 256 * q;
            wl[buf][u / (64 * kCh * kPfRT)][(u / (64 * kCh)) % kPfRT][(u >> 6) % kCh][u & 63] = stg[q];
        }
    };

    f32x4 tot[kPfNT][kPfRT];
#pragma unroll
    for (int nt = 0; nt < kPfNT; ++nt)
#pragma unroll
        for (int r = 0; r < kPfRT; ++r) tot[nt][r] = f32x4{0.f, 0.f, 0.f, 0.f};

    stage_load(0);
    stage_store(0);
    __syncthreads();
    for (int kb = 0; kb < n_kb; ++kb) {
        const int buf = kb & 1;
        if (kb + 1 < n_kb) stage_load(kb + 1);
        // activation fragments of this lane's token: 4 k-steps x (hi, mid); WK 3: the
        // fp16 hi / lo fragments and the token's block scale
        i32x4 bh[kPfNT][4], bm[kPfNT][4];
        float xs[kPfNT];
        if constexpr (WK == 3) {
#pragma unroll
            for (int nt = 0; nt < kPfNT; ++nt) xs[nt] = xscale[static_cast<size_t>(kb) * T + tokcv[nt]];
        }
        // buffer loads: the column block's offset as the scalar offset, the lane's
        // as the vector offset (no per-load address arithmetic)
        const int kbo = kb * 16 * NC * 16;
#pragma unroll
        for (int nt = 0; nt < kPfNT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bh[nt][i] = __builtin_amdgcn_raw_buffer_load_b128(frsrc, static_cast<int>(boff[nt][i]), kbo, 0);
                bm[nt][i] = __builtin_amdgcn_raw_buffer_load_b128(frsrc, static_cast<int>(boff[nt][i]), kbo + 16 * T, 0);
            }
#pragma unroll
        for (int r = 0; r < kPfRT; ++r) {
            const int rt = min(rt0 + r, m_tiles - 1);
            f32x4 acc[kPfNT];
#pragma unroll
            for (int nt = 0; nt < kPfNT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                Frag8 a, b;
                a.i = wl[buf][0][r][i][lane];
#pragma unroll
                for (int nt = 0; nt < kPfNT; ++nt) {
                    if constexpr (WK == 3) {
                        b.i = bh[nt][i];
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, b.h, acc[nt], 0, 0, 0);
                        b.i = bm[nt][i];
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, b.h, acc[nt], 0, 0, 0);
                    } else {
                        b.i = bh[nt][i];
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[nt], 0, 0, 0);
                        b.i = bm[nt][i];
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[nt], 0, 0, 0);
                    }
                }
                if constexpr (WK == 2) {
                    a.i = wl[buf][1][r][i][lane];
#pragma unroll
                    for (int nt = 0; nt < kPfNT; ++nt) {
                        b.i = bh[nt][i];
                        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[nt], 0, 0, 0);
                    }
                }
            }
            if constexpr (WK == 3) {
                const float sc = tscale[static_cast<size_t>(rt) * n_kb + kb];
#pragma unroll
                for (int nt = 0; nt < kPfNT; ++nt) tot[nt][r] += (sc * xs[nt]) * acc[nt];
            } else {
#pragma unroll
                for (int nt = 0; nt < kPfNT; ++nt) tot[nt][r] += acc[nt];
            }
        }
        if (kb + 1 < n_kb) stage_store(buf ^ 1);
        __syncthreads();
    }

    // lane (g, col) holds rows 4g .. 4g+3 of each row tile for token tokv[nt]
#pragma unroll
    for (int nt = 0; nt < kPfNT; ++nt) {
        const int tok = tokv[nt];
        if (tok >= T) break;
        float* yrow = Y + static_cast<size_t>(tok) * ldy;
        if constexpr (EPI == 5) {
            // lane (g < 2, col) holds gate rows 4g..4g+3; lane + 32 the matching up rows
#pragma unroll
            for (int r = 0; r < kPfRT; ++r) {
                if (rt0 + r >= m_tiles) break;
                const int orow = (rt0 + r) * 8 + 4 * g;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float up = __shfl_xor(tot[nt][r][v], 32, 64);
                    if (g < 2 && orow + v < m_valid) yrow[orow + v] = silu_fast(tot[nt][r][v]) * up;
                }
            }
        } else if constexpr (EPI == 6) {
            // as 5; lanes g = 0 and 1 hold output rows 0..3 and 4..7 of the half tile,
            // one 8-column fragment unit of the next GEMM's input, which lane g = 0
            // writes (the same bf16 hi + mid split as pack_act)
            i32x4* fo = reinterpret_cast<i32x4*>(Y);
#pragma unroll
            for (int r = 0; r < kPfRT; ++r) {
                if (rt0 + r >= m_tiles) break;
                float h8[8];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float up = __shfl_xor(tot[nt][r][v], 32, 64);
                    h8[v] = silu_fast(tot[nt][r][v]) * up;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) h8[4 + v] = __shfl_xor(h8[v], 16, 64);
                if (g == 0) write_frag8(fo, rt0 + r, tok, T, h8);
            }
        } else if constexpr (EPI == 2) {
#pragma unroll
            for (int r = 0; r < kPfRT; r += 2) {
                if (rt0 + r + 1 >= m_tiles) break;
                const int orow = ((rt0 + r) / 2) * kTileRows + 4 * g;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (orow + v < m_valid) yrow[orow + v] = silu_fast(tot[nt][r][v]) * tot[nt][r + 1][v];
            }
        } else {
#pragma unroll
            for (int r = 0; r < kPfRT; ++r) {
                if (rt0 + r >= m_tiles) break;
                const int row = (rt0 + r) * kTileRows + 4 * g;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (row + v >= m_valid) break;
                    if constexpr (EPI == 1)
                        yrow[row + v] += tot[nt][r][v];
                    else
                        yrow[row + v] = tot[nt][r][v];
                }
            }
        }
    }
}



// Block-FP8 linears on 32x32x16 MFMA.
//
// Workgroup: TG x KW waves, RT row tiles (16 rows each) x 32 TG tokens.  Wave (tg, kw)
// owns tokens 32 tg .. 32 tg + 31 for all RT tiles, taken in pairs as 32-row A operands,
// over the half column blocks (64 of a block's 128 columns: the first or second 1 KiB of
// a packed tile) kw, kw + KW, ...; the KW partial results are added in order at the end.
// The weights are staged through LDS (double buffered); a wave's activation fragments
// of one half block sit in registers, the next half's loading meanwhile.  The block
// scale multiplies each half block's fp32 partial.
// kGuh: gate / up half tiles with two scales per tile (epilogues 5 and 6).
template <bool kGuh, int RT, int TG, int KW>
__global__ __launch_bounds__(64 * TG * KW, 2) void gemm_fp8_pf_kernel(const uint8_t* __restrict__ W,
                                                                     const float* __restrict__ tscale,
                                                                     const i32x4* __restrict__ frag,
                                                                     float* __restrict__ Y, int m, int n_kb, int T,
                                                                     int ldy, int m_valid, int nrb, int ntb, int epi,
                                                                     int vec) {
    constexpr int kQ = (RT + TG - 1) / TG;  // tiles a wave stages
    constexpr int R2 = RT / 2;
    int rb, tb;
    if (!xcd_block(nrb, ntb, 8, rb, tb)) return;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tg = wave / KW, kw = wave % KW;
    const int h = lane >> 5, col = lane & 31;
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    const int rt0 = rb * RT;
    const int tok0 = (tb * TG + tg) * 32;
    const int tok = tok0 + col, tokc = min(tok, T - 1);
    const bool live = tok0 < T;  // wave-uniform: a wave past the last token only stages

    const __amdgpu_buffer_rsrc_t frsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<i32x4*>(frag), 0, static_cast<int>(static_cast<uint32_t>(n_kb) * 512u * T), 0x00020000);
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(W), 0, static_cast<int>(static_cast<uint32_t>(m_tiles) * static_cast<uint32_t>(n_kb) * 2048u),
        0x00020000);

    constexpr int kRTp = TG * kQ;           // staged tiles (RT rounded up)
    constexpr int kBuf = KW * kRTp * 64;    // one staging buffer, 16-byte units
    constexpr int kRed = (KW - 1) * TG * R2 * 16 * 16;  // the KW - 1 other partials, 16-byte units
    constexpr int kLds = 2 * kBuf > kRed ? 2 * kBuf : kRed;
    __shared__ i32x4 lds[kLds];  // [buffer][kw][row tile][lane of the packed tile]
    uint32_t woff[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q)
        woff[q] = static_cast<uint32_t>(min(rt0 + tg + TG * q, m_tiles - 1)) * static_cast<uint32_t>(n_kb * 2048) + 16 * lane;
    const int n_hb = 2 * n_kb;
    const int pairs = (n_hb + 2 * KW - 1) / (2 * KW);  // steps, two at a time
    i32x4 stg[kQ];
    auto stage_load = [&](int step) {
        const int so = min(step * KW + kw, n_hb - 1) * 1024;
#pragma unroll
        for (int q = 0; q < kQ; ++q)
            stg[q] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, static_cast<int>(woff[q]), so, 0);
    };
    i32x4* const sbase = lds + (kw * kRTp + tg) * 64 + lane;
    auto stage_store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kQ; ++q) sbase[buf * kBuf + TG * q * 64] = stg[q];
    };
    f32x16 tot[R2];
#pragma unroll
    for (int r = 0; r < R2; ++r)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[r][v] = 0.f;

    stage_load(0);
    stage_store(0);
    if (!live) {  // only stages; the same barriers as the working waves
        lds_barrier();
        for (int st = 1; st <= 2 * pairs; ++st) {
            stage_load(st);
            stage_store(st & 1);
            lds_barrier();
        }
    } else {
        // fragments of half block hb: unit (k-step i, lane group g = 2p + h, token), hi then mid
        const int boff = (2 * T * h + tokc) * 16;
        auto load_b = [&](int step, Frag8 (&b)[2][2][2]) {  // [p][i & 1][hi, mid]
            const uint32_t so = static_cast<uint32_t>(min(step * KW + kw, n_hb - 1)) * 256u * T;
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int part = 0; part < 2; ++part)
                        b[p][i][part].i = __builtin_amdgcn_raw_buffer_load_b128(
                            frsrc, boff, static_cast<int>(so + (128u * i + 64u * p + 16u * part) * T), 0);
        };
        // lane j holds the block scale of tile j (half tiles: of half j % 2 of tile j / 2)
        const int st = min(rt0 + (kGuh ? min(lane / 2, RT - 1) : min(lane, RT - 1)), m_tiles - 1);
        const float* sp = kGuh ? tscale + static_cast<size_t>(st) * n_kb * 2 + (lane & 1)
                               : tscale + static_cast<size_t>(st) * n_kb;
        auto load_s = [&](int step) {
            return sp[static_cast<size_t>(min(step * KW + kw, n_hb - 1) >> 1) * (kGuh ? 2 : 1)];
        };

        f32x16 acc[2];
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[1][v] = 0.f;

        const i32x4* wbase = lds + (kw * kRTp + (col >> 4)) * 64 + h * 16 + (col & 15);
        // quarter q of tot[r] += scale * p
        auto add_scaled = [&](int r, int q, const f32x16& p, float sv) {
            const float sc = __int_as_float(
                __builtin_amdgcn_readlane(__float_as_int(sv), kGuh ? 4 * r + q : 2 * r + q / 2));
#pragma unroll
            for (int v = 4 * q; v < 4 * q + 4; ++v) tot[r][v] = fmaf(sc, p[v], tot[r][v]);
        };
        // One half block.  Each MFMA is followed by the VALU work that fits under it (the
        // conversion of the next fragment, a quarter of the previous tile pair's scaled
        // add) and the order is pinned: left to itself the compiler runs the reads,
        // conversions, MFMAs and adds of a pair one after the other.
        auto half = [&](auto C, const Frag8 (&b)[2][2][2], float sv, float svp) {
            constexpr int o = decltype(C)::value * R2;  // parity of the accumulators
            const i32x4* wp = wbase + decltype(C)::value * kBuf;
            i32x4 raw[2] = {wp[0], wp[32]};
            Frag8 a, a1;
            e4m3x4_to_bf16(static_cast<uint32_t>(raw[0][0]), a.u[0], a.u[1]);
            e4m3x4_to_bf16(static_cast<uint32_t>(raw[0][1]), a.u[2], a.u[3]);
#pragma unroll
            for (int u = 0; u < RT; ++u) {
                const int r = u >> 1, p = u & 1;
                const int rp = r ? r - 1 : R2 - 1;
                const float sp_ = r ? sv : svp;
                f32x16& ac = acc[(r + o) & 1];
                const f32x16& ap = acc[(r + o + 1) & 1];
                if (p == 0) {
                    f32x16 z;
#pragma unroll
                    for (int v = 0; v < 16; ++v) z[v] = 0.f;
                    ac = z;
                }
                ac = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b[p][0][0].v, ac, 0, 0, 0);
                e4m3x4_to_bf16(static_cast<uint32_t>(raw[p][2]), a1.u[0], a1.u[1]);
                if (p == 1) add_scaled(rp, 2, ap, sp_);
                __builtin_amdgcn_sched_barrier(0);
                ac = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b[p][0][1].v, ac, 0, 0, 0);
                e4m3x4_to_bf16(static_cast<uint32_t>(raw[p][3]), a1.u[2], a1.u[3]);
                if (u + 2 < RT) raw[p] = wp[(u + 2) / 2 * 128 + 32 * p];
                if (p == 1) add_scaled(rp, 3, ap, sp_);
                __builtin_amdgcn_sched_barrier(0);
                ac = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1.v, b[p][1][0].v, ac, 0, 0, 0);
                if (u + 1 < RT) e4m3x4_to_bf16(static_cast<uint32_t>(raw[1 - p][0]), a.u[0], a.u[1]);
                if (p == 0) add_scaled(rp, 0, ap, sp_);
                __builtin_amdgcn_sched_barrier(0);
                ac = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1.v, b[p][1][1].v, ac, 0, 0, 0);
                if (u + 1 < RT) e4m3x4_to_bf16(static_cast<uint32_t>(raw[1 - p][1]), a.u[2], a.u[3]);
                if (p == 0) add_scaled(rp, 1, ap, sp_);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        Frag8 b0[2][2][2], b1[2][2][2];
        load_b(0, b0);
        float s0 = load_s(0), svp = 0.f;  // svp: scales of the pending partial acc[1]
        lds_barrier();
        for (int k2 = 0; k2 < pairs; ++k2) {
            const bool in0 = KW == 1 || 2 * k2 * KW + kw < n_hb, in1 = KW == 1 || (2 * k2 + 1) * KW + kw < n_hb;
            stage_load(2 * k2 + 1);
            load_b(2 * k2 + 1, b1);
            const float s1 = load_s(2 * k2 + 1);
            if (in0) half(std::integral_constant<int, 0>{}, b0, s0, svp);
            stage_store(1);
            lds_barrier();
            stage_load(2 * k2 + 2);
            load_b(2 * k2 + 2, b0);
            const float s2 = load_s(2 * k2 + 2);
            if (in1) {
                half(std::integral_constant<int, 1>{}, b1, s1, s0);
                svp = s1;
            } else if (in0) {  // the wave's last half block was the pair's first
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[1][v] = acc[(R2 - 1) & 1][v];
                svp = s0;
            }
            s0 = s2;
            stage_store(0);
            lds_barrier();
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) add_scaled(R2 - 1, q, acc[1], svp);
    }
    if constexpr (KW > 1) {
        // partials of waves kw > 0 through LDS (the staging buffers are free after the
        // last barrier), added by wave kw = 0 in the order of kw
        float* red = reinterpret_cast<float*>(lds);
        if (kw > 0 && live) {
            float* d = red + ((kw - 1) * TG + tg) * (R2 * 16 * 64) + lane;
#pragma unroll
            for (int r = 0; r < R2; ++r)
#pragma unroll
                for (int v = 0; v < 16; ++v) d[(r * 16 + v) * 64] = tot[r][v];
        }
        __syncthreads();
        if (kw > 0) return;
#pragma unroll 1
        for (int k = 1; k < KW; ++k) {
            const float* d = red + ((k - 1) * TG + tg) * (R2 * 16 * 64) + lane;
#pragma unroll
            for (int r = 0; r < R2; ++r)
#pragma unroll
                for (int v = 0; v < 16; ++v) tot[r][v] += d[(r * 16 + v) * 64];
        }
    }
    const bool in = tok < T;  // (no lane leaves: the fragment epilogue exchanges lanes of one token)

    // lane (h, col) holds rows 8u + 4h + v (u = 0..3, v = 0..3) of each 32-row pair
    float* yrow = Y + static_cast<size_t>(tokc) * ldy;
#pragma unroll
    for (int r = 0; r < R2; ++r) {
        const int rt = rt0 + 2 * r;
        if constexpr (kGuh) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (rt + j >= m_tiles) break;
                float o4[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) o4[v] = silu_fast(tot[r][8 * j + v]) * tot[r][8 * j + 4 + v];
                if (epi == kEpiSwiGLUHFrag) {
                    // one 8-column fragment unit of the next GEMM's input per tile: lanes h = 0
                    // write its hi part, lanes h = 1 its mid part (the split of pack_act)
                    float h8[8];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float o = __shfl_xor(o4[v], 32, 64);
                        h8[v] = h ? o : o4[v];
                        h8[4 + v] = h ? o4[v] : o;
                    }
                    union {
                        uint16_t e[8];
                        i32x4 q;
                    } hi, mid;
#pragma unroll
                    for (int e = 0; e < 8; ++e) split_bf16(h8[e], hi.e[e], mid.e[e]);
                    if (in) reinterpret_cast<i32x4*>(Y)[frag_unit(rt + j, tok, T) + (h ? T : 0)] = h ? mid.q : hi.q;
                } else {
                    const int row = (rt + j) * 8 + 4 * h;
                    if (in) store_rows4(yrow + row, o4, m_valid - row, vec, false);
                }
            }
        } else if (epi == kEpiSwiGLU) {
            if (rt + 1 >= m_tiles) break;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float o4[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) o4[v] = silu_fast(tot[r][4 * u + v]) * tot[r][8 + 4 * u + v];
                const int row = (rt / 2) * kTileRows + 8 * u + 4 * h;
                if (in) store_rows4(yrow + row, o4, m_valid - row, vec, false);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float o4[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) o4[v] = tot[r][4 * u + v];
                const int row = rt * kTileRows + 8 * u + 4 * h;
                if (in) store_rows4(yrow + row, o4, m_valid - row, vec, epi == kEpiAdd);
            }
        }
    }
}

// bf16 hi + mid activation fragments -> fp16 hi + lo fragments, one thread per
// (128-column block kb, token t): x = hi + mid (exact, 16 significant bits), scaled
// by a power of two xscale[kb][t] that puts the block's largest |x| in
// [2^14, 2^15), then split into fp16 hi = rn(x / s) and lo = rn(x / s - hi), which
// together hold every bit of x.  Same layout as the input (units (kb, i, g): hi in
// column t, lo in column T + t).
__global__ void act_frag_to_f16_kernel(const i32x4* __restrict__ frag, i32x4* __restrict__ out,
                                       float* __restrict__ xscale, int n_kb, int T) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_kb * T) return;
    const int t = idx % T, kb = idx / T;
    const size_t NC = 2 * static_cast<size_t>(T);
    auto unit = [&](int gi) { return (static_cast<size_t>(kb) * 16 + gi) * NC + t; };
    auto value = [&](const Frag8& h, const Frag8& md, int e) {
        const uint32_t hb = (h.u[e >> 1] >> (16 * (e & 1))) & 0xffffu;
        const uint32_t mb = (md.u[e >> 1] >> (16 * (e & 1))) & 0xffffu;
        return __uint_as_float(hb << 16) + __uint_as_float(mb << 16);
    };
    float mx = 0.f;
    for (int gi = 0; gi < 16; ++gi) {
        Frag8 h, md;
        h.i = frag[unit(gi)];
        md.i = frag[unit(gi) + T];
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(value(h, md, e)));
    }
    float sc = 1.f;
    if (mx > 0.f) {
        int ex;
        frexpf(mx, &ex);
        sc = ldexpf(1.f, ex - 15);
    }
    const float inv = 1.f / sc;
    for (int gi = 0; gi < 16; ++gi) {
        Frag8 h, md, oh, ol;
        h.i = frag[unit(gi)];
        md.i = frag[unit(gi) + T];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = value(h, md, e) * inv;
            const _Float16 vh = static_cast<_Float16>(v);
            oh.h[e] = vh;
            ol.h[e] = static_cast<_Float16>(v - static_cast<float>(vh));
        }
        out[unit(gi)] = oh.i;
        out[unit(gi) + T] = ol.i;
    }
    xscale[static_cast<size_t>(kb) * T + t] = sc;
}

template <bool kGuh, int RT, int TG, int KW>
void launch_fp8_pf_cfg(const uint8_t* W, const float* ts, const i32x4* frag, float* Y, int m, int n_kb, int T, int ldy,
                       int m_valid, int epi, hipStream_t s) {
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    const int nrb = (m_tiles + RT - 1) / RT, ntb = (T + 32 * TG - 1) / (32 * TG);
    const int vec = epi != kEpiSwiGLUHFrag && ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
    RL_REQUIRE(static_cast<long>(nrb) * ntb < (1L << 30), RL_ERR_RANGE, "gemm_prefill: too many workgroups");
    const int wgs = (nrb * ntb + 7) / 8 * 8;
    hipLaunchKernelGGL((gemm_fp8_pf_kernel<kGuh, RT, TG, KW>), dim3(wgs), dim3(64 * TG * KW), 0, s, W, ts, frag, Y, m,
                       n_kb, T, ldy, m_valid, nrb, ntb, epi, vec);
    check_launch("gemm_fp8_pf_kernel");
}

// The work split.  A CU runs eight waves of these kernels.  A step of a workgroup (KW
// half blocks) takes about RT + 3 units of 0.15 us: RT / 2 pairs of 8 MFMAs for each of
// a SIMD's two waves, and the step's fixed latency.  The split with the smallest (rounds
// of workgroups) x (steps) x (RT + 3) is taken; with KW = 2 a CU's eight waves share one
// barrier, which costs about an eighth more where the chip is full (34816 x 5120, 2011
// tokens: 1235 us with KW = 1, 1402 us with KW = 2, both at RT = 10), and pays where it is
// not (5120 x 17408, 512 tokens: 309 us at RT = 10, KW = 1, 228 us at RT = 8, KW = 2).
// With at most 32 (64) tokens the waves that would own absent tokens split K instead:
// 5120 x 17408 at 64 tokens 364 -> 68 us, 34816 x 5120 153 -> 60 us.
template <bool kGuh>
void launch_fp8_pf(const uint8_t* W, const float* ts, const i32x4* frag, float* Y, int m, int n_kb, int T, int ldy,
                   int m_valid, int epi, hipStream_t s) {
    struct Cfg {
        int rt, tg, kw;
        void (*launch)(const uint8_t*, const float*, const i32x4*, float*, int, int, int, int, int, int, hipStream_t);
    };
#define RL_PFC(RT, TG, KW) Cfg{RT, TG, KW, launch_fp8_pf_cfg<kGuh, RT, TG, KW>}
    static const Cfg cfgs[] = {
        RL_PFC(12, 4, 1), RL_PFC(10, 4, 1), RL_PFC(8, 4, 1), RL_PFC(10, 4, 2), RL_PFC(8, 4, 2), RL_PFC(4, 4, 2),
        RL_PFC(10, 2, 4), RL_PFC(8, 2, 4),  RL_PFC(4, 2, 4), RL_PFC(2, 2, 4),  RL_PFC(8, 1, 8),
        RL_PFC(4, 1, 8),  RL_PFC(2, 1, 8)};
#undef RL_PFC
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    const int tg = T <= 32 ? 1 : T <= 64 ? 2 : 4;
    const Cfg* best = nullptr;
    long cost = 0;
    for (const Cfg& c : cfgs) {
        if (c.tg != tg) continue;
        const long wgs = static_cast<long>((m_tiles + c.rt - 1) / c.rt) * ((T + 32 * tg - 1) / (32 * tg));
        const long slots = static_cast<long>(device_cus()) * 8 / (c.tg * c.kw);
        const long t = (wgs + slots - 1) / slots * ((2 * n_kb + c.kw - 1) / c.kw) * (c.rt + 3) * (c.kw == 2 ? 9 : 8);
        if (!best || t < cost) {
            cost = t;
            best = &c;
        }
    }
    best->launch(W, ts, frag, Y, m, n_kb, T, ldy, m_valid, epi, s);
}

}  // namespace

namespace rl {

void gemm_prefill_any(int wk, const uint8_t* W, const uint8_t* W_lo, const float* ts, const void* frag, float* Y,
                      int m, int n, int T, int epi, int ldy, int m_valid, hipStream_t s, const float* xscale) {
    RL_REQUIRE(m > 0 && n > 0 && T >= 1, RL_ERR_RANGE, "gemm_prefill: empty shape");
    RL_REQUIRE(W && frag && Y && ((wk != 0 && wk != 3) || ts) && (wk != 2 || W_lo) && (wk != 3 || xscale),
               RL_ERR_RANGE, "gemm_prefill: null pointer");
    RL_REQUIRE(wk >= 0 && wk <= 3, RL_ERR_RANGE, "gemm_prefill: weight kind");
    RL_REQUIRE(epi == kEpiStore || epi == kEpiAdd || epi == kEpiSwiGLU || epi == kEpiSwiGLUH ||
                   epi == kEpiSwiGLUHFrag,
               RL_ERR_RANGE, "gemm_prefill: epilogue must be store, add or swiglu");
    if (epi == kEpiSwiGLUH) RL_REQUIRE(m % 16 == 0, RL_ERR_RANGE, "gemm_prefill swiglu: rows a multiple of 16");
    if (epi == kEpiSwiGLUHFrag)
        RL_REQUIRE(m % 256 == 0 && m_valid == m / 2, RL_ERR_RANGE,
                   "gemm_prefill swiglu to fragments: outputs a multiple of 128");
    const int m_tiles = (m + kTileRows - 1) / kTileRows;
    if (epi == kEpiSwiGLU) RL_REQUIRE(m % 32 == 0, RL_ERR_RANGE, "gemm_prefill swiglu: rows must be a multiple of 32");
    const int n_kb = (n + 127) / 128;
    // the kernel addresses weights and fragments with 32-bit offsets
    RL_REQUIRE(static_cast<size_t>(m_tiles) * n_kb * (wk == 0 ? 2048 : 4096) < (size_t{1} << 32) &&
                   static_cast<size_t>(n_kb) * 16 * 2 * T * 16 < (size_t{1} << 32),
               RL_ERR_RANGE, "gemm_prefill: weights and input fragments must each stay under 4 GiB");
    if (wk == 0) {
        const bool guh = epi == kEpiSwiGLUH || epi == kEpiSwiGLUHFrag;
        (guh ? launch_fp8_pf<true> : launch_fp8_pf<false>)(W, ts, static_cast<const i32x4*>(frag), Y, m, n_kb, T, ldy,
                                                           m_valid, epi, s);
        return;
    }
    const int rt = 4;
    const dim3 grid((m_tiles + rt - 1) / rt, (T + kPfTok - 1) / kPfTok);
    RL_REQUIRE(grid.y <= 65535, RL_ERR_RANGE, "gemm_prefill: too many tokens");
    const i32x4* fr = static_cast<const i32x4*>(frag);
#define RL_PF(E, K)                                                                                                 \
    if (epi == E && wk == K) {                                                                                      \
        hipLaunchKernelGGL((gemm_prefill_kernel<E == kEpiSwiGLUH ? 5 : E, K>), grid, dim3(256), 0, s, W, ts, fr, Y, m, \
                           n_kb, T, ldy, m_valid, W_lo, xscale);                                                    \
        check_launch("gemm_prefill_kernel");                                                                        \
        return;                                                                                                     \
    }
    RL_PF(kEpiStore, 1) RL_PF(kEpiAdd, 1) RL_PF(kEpiSwiGLU, 1) RL_PF(kEpiSwiGLUH, 1)
    RL_PF(kEpiStore, 2) RL_PF(kEpiAdd, 2) RL_PF(kEpiSwiGLU, 2) RL_PF(kEpiSwiGLUH, 2)
    RL_PF(kEpiStore, 3) RL_PF(kEpiAdd, 3) RL_PF(kEpiSwiGLU, 3) RL_PF(kEpiSwiGLUH, 3)
    RL_PF(kEpiSwiGLUHFrag, 1) RL_PF(kEpiSwiGLUHFrag, 2) RL_PF(kEpiSwiGLUHFrag, 3)
#undef RL_PF
}

void act_frag_to_f16(const void* frag, void* frag16, float* xscale, int n, int T, hipStream_t s) {
    RL_REQUIRE(frag && frag16 && xscale && n > 0 && T >= 1 && frag != frag16, RL_ERR_RANGE,
               "act_frag_to_f16: bad arguments");
    const int n_kb = (n + 127) / 128;
    const int total = n_kb * T;
    hipLaunchKernelGGL(act_frag_to_f16_kernel, dim3((total + 255) / 256), dim3(256), 0, s,
                       static_cast<const i32x4*>(frag), static_cast<i32x4*>(frag16), xscale, n_kb, T);
    check_launch("act_frag_to_f16_kernel");
}

void gemm_fp8_prefill(const uint8_t* W, const float* ts, const void* frag, float* Y, int m, int n, int T, int epi,
                      int ldy, int m_valid, hipStream_t s) {
    gemm_prefill_any(0, W, nullptr, ts, frag, Y, m, n, T, epi, ldy, m_valid, s);
}

}  // namespace rl

extern "C" {

int rl_hip_gemm_fp8_prefill(const uint8_t* w_tiled, const float* tile_scale, const void* frag, float* Y, int m, int n,
                            int T, int epilogue, int ldy, void* stream) {
    return guard([&] {
        const int mv = epilogue == kEpiSwiGLU || epilogue == kEpiSwiGLUH || epilogue == kEpiSwiGLUHFrag ? m / 2 : m;
        rl::gemm_fp8_prefill(w_tiled, tile_scale, frag, Y, m, n, T, epilogue, ldy > 0 ? ldy : mv, mv, S(stream));
    });
}

int rl_hip_gemm_bf16_prefill(const uint16_t* w_tiled, const uint16_t* w_lo_tiled, const void* frag, float* Y, int m,
                             int n, int T, int epilogue, int ldy, void* stream) {
    return guard([&] {
        const int mv = epilogue == kEpiSwiGLU || epilogue == kEpiSwiGLUH || epilogue == kEpiSwiGLUHFrag ? m / 2 : m;
        rl::gemm_prefill_any(w_lo_tiled ? 2 : 1, reinterpret_cast<const uint8_t*>(w_tiled),
                             reinterpret_cast<const uint8_t*>(w_lo_tiled), nullptr, frag, Y, m, n, T, epilogue,
                             ldy > 0 ? ldy : mv, mv, S(stream));
    });
}

int rl_hip_act_frag_to_f16(const void* frag, void* frag16, float* xscale, int n, int T, void* stream) {
    return guard([&] { rl::act_frag_to_f16(frag, frag16, xscale, n, T, S(stream)); });
}

int rl_hip_gemm_f16_prefill(const void* w16, const float* tile_scale, const void* frag16, const float* xscale,
                            float* Y, int m, int n, int T, int epilogue, int ldy, void* stream) {
    return guard([&] {
        const int mv = epilogue == kEpiSwiGLU || epilogue == kEpiSwiGLUH || epilogue == kEpiSwiGLUHFrag ? m / 2 : m;
        rl::gemm_prefill_any(3, static_cast<const uint8_t*>(w16), nullptr, tile_scale, frag16, Y, m, n, T, epilogue,
                             ldy > 0 ? ldy : mv, mv, S(stream), xscale);
    });
}

}  // extern "C"
