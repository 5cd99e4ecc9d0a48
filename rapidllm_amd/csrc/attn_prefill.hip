// attn_prefill.hip -- gated GQA attention over a prompt chunk and the fp16 KV cache.
//
// T tokens at positions p0 .. p0+T-1 (the reference's prefill attention,
// cuda_engine.cu:18338-18590; semantics per token as attn.hip): qk_prep_pf_kernel writes
// K / V to the cache and q as fp16 hi + lo fragments, attn_prefill_kernel streams the
// cache with a running max / sum / output per query (online softmax), and
// attn_merge_kernel adds the parts of the queries whose positions were split.
#include <algorithm>
#include <climits>

#include "attn.h"

using namespace rl;

namespace {

constexpr int kPrepLd = kHD + 4;

// grid (ceil(T / 16) + 1, ceil((nq + 2 nkv) / hpw)), 256 threads: the tokens of one aligned
// group of 16 positions, hpw of the heads [0, nq) q, [nq, nq + nkv) k, then v.  16 lanes per
// token (dims 4 l + 64 k) form the norm; the rows go through LDS so that every store is a
// 16-byte unit of the layouts and the token's RoPE angles are formed once for the
// workgroup's heads.  One wave per (head, token), storing 2-byte elements: 44 us for 1500
// tokens, 24 + 2 x 4 heads.
__global__ __launch_bounds__(256) void qk_prep_pf_kernel(AttnArgs p, i32x4* __restrict__ qp, int hpw) {
    __shared__ float row_s[16][kPrepLd];
    __shared__ float2 ang_s[16][kHD / 2];
    __shared__ float freq_s[kHD / 2];
    const int tid = threadIdx.x, ti = tid >> 4, l16 = tid & 15;
    const int p0 = *p.pos;
    const int base = (p0 & ~15) + 16 * blockIdx.x;  // first position of the group
    const int t_lo = max(base - p0, 0), t_hi = min(base + 16 - p0, p.T);  // its tokens
    if (t_lo >= t_hi) return;
    const int half = p.rot / 2;
    if (tid < half) freq_s[tid] = 1.f / powf(p.theta, static_cast<float>(tid) / static_cast<float>(half));
    __syncthreads();
    for (int k = tid; k < 16 * half; k += 256) {
        const int j = k / half, i = k % half;
        const float ang = static_cast<float>(base + j) * freq_s[i];
        ang_s[j][i] = make_float2(cosf(ang), sinf(ang));
    }
    const int qcols = p.nq * kHD * 2, heads = p.nq + 2 * p.nkv;
    const int ntb = (p.T + 15) / 16;
    const int t = base + ti - p0;
    const bool in = t >= t_lo && t < t_hi;
    const int h1 = min(heads, static_cast<int>(blockIdx.y + 1) * hpw);
    for (int head = blockIdx.y * hpw; head < h1; ++head) {
        const bool is_q = head < p.nq, is_v = head >= p.nq + p.nkv;
        const int off = is_q ? head * 2 * kHD : qcols + (head - p.nq) * kHD;
        float x[4][4];
        double ss = 0.0;
        if (in) {
            const float* src = p.Y + static_cast<size_t>(t) * p.ld_y + off;
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x[k][r] = src[64 * k + 4 * l16 + r];
                    ss += static_cast<double>(x[k][r]) * x[k][r];
                }
        }
        __syncthreads();  // the previous head's rows have been read (and the angles are there)
        if (!is_v) {
            const float* gam = is_q ? p.q_norm : p.k_norm;
            ss = group16_sum_d(ss);
            const float inv = 1.f / sqrtf(static_cast<float>(ss / kHD) + p.eps);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[k][r] = x[k][r] * inv * (gam ? 1.f + gam[64 * k + 4 * l16 + r] : 1.f);
        }
        if (in) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r) row_s[ti][64 * k + 4 * l16 + r] = x[k][r];
        }
        __syncthreads();
        // (token, d) of the group, rotated: dim i < half with dim i + half
        auto value = [&](int j, int d) {
            const float v = row_s[j][d];
            if (is_v || d >= 2 * half) return v;
            if (d < half) return v * ang_s[j][d].x - row_s[j][d + half] * ang_s[j][d].y;
            return row_s[j][d - half] * ang_s[j][d - half].y + v * ang_s[j][d - half].x;
        };
        union {
            _Float16 e[8];
            i32x4 v;
        } hi, lo;
        if (is_v) {
            // 8 positions of one dim per unit, whole units at the group's inside
            uint16_t* vb = p.vt + static_cast<size_t>(head - p.nq - p.nkv) * p.ctx * kHD;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int d = tid, j0 = 8 * q;
                if (base + j0 >= p0 + t_lo && base + j0 + 8 <= p0 + t_hi) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) hi.e[e] = static_cast<_Float16>(row_s[j0 + e][d]);
                    *reinterpret_cast<i32x4*>(vb + v_off(base + j0, d)) = hi.v;
                } else {
                    for (int e = 0; e < 8; ++e) {
                        const int tt = base + j0 + e - p0;
                        if (tt >= t_lo && tt < t_hi)
                            vb[v_off(base + j0 + e, d)] =
                                __builtin_bit_cast(uint16_t, static_cast<_Float16>(row_s[j0 + e][d]));
                    }
                }
            }
            continue;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int u = tid + 256 * q, j = u & 15, d = 8 * (u >> 4);  // token j of the group, dims d .. d + 7
            const int tt = base + j - p0;
            if (tt < t_lo || tt >= t_hi) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = value(j, d + e);
                hi.e[e] = static_cast<_Float16>(v);
                lo.e[e] = static_cast<_Float16>(v - static_cast<float>(hi.e[e]));
            }
            if (!is_q) {
                *reinterpret_cast<i32x4*>(p.kc + static_cast<size_t>(head - p.nq) * p.ctx * kHD + k_off(base + j, d)) = hi.v;
            } else {
                i32x4* o = qp + q_unit(head / p.G, head % p.G, p.G, ntb, tt >> 4) + (d >> 3) * p.G * 32 + (tt & 15);
                o[0] = hi.v;
                o[16] = lo.v;
            }
        }
    }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

// One workgroup: 4 waves x 32 queries of one kv head (wave: one head, 32 tokens), all
// reading the same K and V from LDS, where 64 positions of each (32 KiB) are copied
// straight from the cache, double buffered.  S^T = K . Q^T and O^T = V^T . P^T on 32x32x16
// fp16 MFMA (q as hi + lo, two MFMAs per step): the K rows enter in an order that leaves
// each lane's scores at the positions its P^T operand needs, so the probabilities never
// leave the wave's registers.  The scores of the next 64 positions are computed while the
// current ones go through exp.  One wave per SIMD: q fragments and output take 256
// registers.
// Bound by that wave's chain: 3072 MFMA cycles in about 7000 per 64 positions (2.15 GHz; 1500
// tokens over 4000 positions: the matrix cores are busy 36% of the launch).  With 16
// tokens x 3 heads per workgroup on 16x16 MFMA, K and V from the L2 and P through LDS, 1500
// tokens over 4000 positions took 514 us (24 / 4 heads), 4092 over 32092 11.3 ms; now 244
// us and 4.5 ms.  A running maximum that moves only past 2^8 saves the rescaling but
// rounds the largest probability, otherwise an exact 1 (error 2.06e-4 against 1.93e-4). 
__global__ __launch_bounds__(256, 1) void attn_prefill_kernel(AttnArgs p, const i32x4* __restrict__ qp,
                                                              float* __restrict__ out, int items, PfParts pp,
                                                              int auto_route) {
    if (auto_route && attn_prefill_auto_short(*p.pos + p.T)) return;  // attn_prefill_finish_kernel has it
    __shared__ i32x4 K0[2048], K1[2048];  // [d/32][pos/16][(d/8)%4][pos%16]
    __shared__ i32x4 V0[2048], V1[2048];  // [pos/32][d/16][(pos/8)%4][d%16]
    __shared__ int flag[4];
    // kv head from the XCD (blockIdx % 8), so that its cache is read through one L2 (or
    // two); longest items first
    int kv, idx;
    if (8 % p.nkv == 0) {
        const int per = 8 / p.nkv, x = blockIdx.x % 8;
        kv = x % p.nkv;
        idx = blockIdx.x / 8 * per + x / p.nkv;
    } else {
        kv = blockIdx.x % p.nkv;
        idx = blockIdx.x / p.nkv;
    }
    const int part = idx < pp.unsplit ? 0 : (idx - pp.unsplit) % pp.parts;
    const int si = idx < pp.unsplit ? 0 : (idx - pp.unsplit) / pp.parts;  // split item
    const bool split = idx >= pp.unsplit;
    if (split) idx = pp.unsplit + si;
    if (idx >= items) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, col = lane & 31;
    const int ntb = (p.T + 31) / 32, ntb16 = (p.T + 15) / 16;
    const int entries = p.G * ntb;
    const int e = min((items - 1 - idx) * 4 + wave, entries - 1);  // (extra waves repeat the last entry)
    const int head = kv * p.G + e % p.G, tb = e / p.G;
    const int p0 = *p.pos;
    const int tok = 32 * tb + col;
    const int qpos = p0 + min(tok, p.T - 1);
    const int L = pf_keys(items - 1 - idx, p.G, p.T, p0);  // keys 0 .. L-1 for the workgroup
    const int q_first = p0 + 32 * tb;                       // positions up to here need no mask
    const int wg_first = p0 + 32 * ((items - 1 - idx) * 4 / p.G);  // ... in any wave
    const int nblk = (L + 63) / 64;
    const int parts = split ? pf_parts(pp.parts, nblk) : 1;
    if (part >= parts) return;
    const int blk0 = nblk * part / parts, blk1 = nblk * (part + 1) / parts;
    const float c = 1.44269504f / sqrtf(static_cast<float>(kHD));  // log2(e) / sqrt(hd)

    const uint16_t* kbase = p.kc + static_cast<size_t>(kv) * p.ctx * kHD;
    const uint16_t* vbase = p.vt + static_cast<size_t>(kv) * p.ctx * kHD;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(kbase), 0, static_cast<int>(static_cast<uint32_t>(p.ctx) * kHD * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(vbase), 0, static_cast<int>(static_cast<uint32_t>(p.ctx) * kHD * 2u), 0x00020000);
    auto dma_k = [&](int blk_, i32x4* K) {  // wave w brings d / 32 = 2w, 2w + 1
        const int blk = min(blk_, nblk - 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t so = static_cast<uint32_t>(blk >> 2) * 131072u + (2 * wave + (q >> 2)) * 16384u +
                                static_cast<uint32_t>(blk & 3) * 4096u + (q & 3) * 1024u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (lds_void*)(K + (2 * wave + (q >> 2)) * 256 + (q & 3) * 64), 16,
                                                     16 * lane, static_cast<int>(so), 0, 0);
        }
    };
    auto dma_v = [&](int blk_, i32x4* V) {  // positions past L - 1 come from written groups
        const int blk = min(blk_, nblk - 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int u = wave * 8 + q;
            const int grp = min(2 * blk + (u >> 4), (L - 1) >> 5);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (lds_void*)(V + u * 64), 16, 16 * lane,
                                                     static_cast<int>(static_cast<uint32_t>(grp) * 16384u + (u & 15) * 1024u), 0,
                                                     0);
        }
    };

    H8 qh[16], ql[16];
    {
        const i32x4* qq = qp + q_unit(kv, e % p.G, p.G, ntb16, min(2 * tb + (col >> 4), ntb16 - 1)) + h * p.G * 32 + (col & 15);
#pragma unroll
        for (int st = 0; st < 16; ++st) {
            qh[st].i = qq[st * p.G * 64];
            ql[st].i = qq[st * p.G * 64 + 16];
            // q lives in accumulation registers, which the MFMAs read directly: the output
            // is rescaled by vector instructions and has the others
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                int a, b;
                asm("v_accvgpr_write_b32 %0, %1" : "=a"(a) : "v"(qh[st].i[d]));
                asm("v_accvgpr_write_b32 %0, %1" : "=a"(b) : "v"(ql[st].i[d]));
                qh[st].i[d] = a;
                ql[st].i[d] = b;
            }
        }
    }
    f32x16 o[8], s[2], z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.f;
    float m, l;  // running max of the scaled scores (log2 units), lane's part of the sum

    // K row 8u + 4h' + v of a 32-position tile is position 16 (u / 2) + 8 h' + 4 (u % 2) + v
    const int krow = 8 * ((col >> 2) & 1) + 4 * ((col >> 3) & 1) + (col & 3);
    const int koff = ((col >> 4) * 4 + h) * 16 + krow;
    const int voff = ((col >> 4) * 4 + h) * 16 + (col & 15);

    auto scores = [&](const i32x4* K, f32x16 (&sn)[2]) {
#pragma unroll
        for (int st = 0; st < 16; ++st)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                H8 k;
                k.i = K[koff + (st >> 1) * 256 + (st & 1) * 32 + a * 128];
                sn[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k.v, qh[st].v, st ? sn[a] : z, 0, 0, 0);
                sn[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k.v, ql[st].v, sn[a], 0, 0, 0);
            }
    };
    // s of block blk -> scaled, masked; returns the lane's query's maximum over the block
    auto mask_max = [&](int blk, f32x16 (&sn)[2]) {
        if (64 * blk + 63 > q_first) {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int pos = 64 * blk + 32 * a + 16 * (v >> 3) + 8 * h + (v & 7);
                    if (pos > qpos) sn[a][v] = -INFINITY;
                }
        }
        float x = fmaxf(sn[0][0], sn[1][0]);
#pragma unroll
        for (int v = 1; v < 16; ++v) x = fmaxf(x, fmaxf(sn[0][v], sn[1][v]));
        return fmaxf(x, __shfl_xor(x, 32, 64)) * c;
    };
    auto step = [&](int blk, float mx, const i32x4* Kn, const i32x4* V) {
        const float mn = fmaxf(m, mx);
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
        m = mn;
        f32x16 sn[2];
        scores(Kn, sn);
        H8 pf[4];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float x = __builtin_amdgcn_exp2f(fmaf(s[a][v], c, -m));
                l += x;
                pf[2 * a + (v >> 3)].v[v & 7] = static_cast<_Float16>(x);
            }
#pragma unroll
        for (int q = 0; q < 32; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // VALU
        }
        // the rescaling of one 32-wide slice of the output hides under the MFMAs of another
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            o[dt] *= alpha;
#pragma unroll
            for (int aj = 0; aj < 4; ++aj) {
                H8 vf;
                vf.i = V[voff + (aj >> 1) * 1024 + dt * 128 + (aj & 1) * 32];
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf.v, pf[aj].v, o[dt], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < 32; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 1);
        }
        s[0] = sn[0];
        s[1] = sn[1];
        return mask_max(blk + 1, s);
    };

    // The non-finite V of a block that some query masks: to the outputs of the queries that see
    // their position, and zeros for the product.
    auto clean_v = [&](int blk, i32x4* V) {
        const uint16_t* vh = reinterpret_cast<const uint16_t*>(V);
#pragma unroll 1
        for (int j = 0; j < 64; ++j) {
            const uint16_t* row = vh + (j >> 5) * 8192 + ((j >> 3) & 3) * 128 + (j & 7);
            const uint32_t see = 64 * blk + j <= qpos ? 0xffffu : 0u;
            bool bad = false;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                bad |= (row[(lane >> 2) * 512 + (4 * (lane & 3) + k) * 8] & 0x7c00u) == 0x7c00u;
            if (__ballot(bad) == 0) continue;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int d = 32 * dt + 8 * (v >> 2) + (v & 3);
                    const uint32_t x = row[(d >> 4) * 512 + ((d & 15) + 4 * h) * 8] & see;
                    const float add = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(x)));
                    o[dt][v] += (x & 0x7c00u) == 0x7c00u ? add : 0.f;
                }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll 1
        for (int q = 0; q < 8; ++q) {
            i32x4 x = V[wave * 512 + q * 64 + lane];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t w = static_cast<uint32_t>(x[d]);
                const uint32_t m16 = ((((w & 0x7c007c00u) + 0x04000400u) >> 15) & 0x00010001u) * 0xffffu;
                x[d] = static_cast<int>(w & ~m16);
            }
            V[wave * 512 + q * 64 + lane] = x;
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    // A masked probability is 0, and 0 times an infinity or NaN a NaN: non-finite V of later tokens
    // (or left in the cache behind them) would reach queries that do not see it.  A workgroup
    // with an output that is not finite starts again and takes such values out of the blocks
    // with masks.  That costs the others the check of their outputs and a looser schedule of
    // the loop: 2% (1000 tokens over 9000 positions 426 -> 435 us).  Measured instead: every
    // workgroup scanning its blocks with masks 3 us a call or 7%, a loop of its own for the
    // second pass 4%, a function call for it 13 us (scratch memory).
    int clean_from = INT_MAX;  // the position from which blocks are cleaned: the second pass's
    for (;;) {
        l = 0.f;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt] = z;
        dma_k(blk0, K0);
        dma_k(blk0 + 1, K1);
        dma_v(blk0, V0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        scores(K0, s);
        float mx = mask_max(blk0, s);
        m = fmaxf(mx, -1e30f);  // (a lane whose positions are all masked in this part: probabilities and a sum of 0)
        // block blk: K(blk + 1) and V(blk) are in LDS; K(blk + 2) and V(blk + 1) on their way
        for (int blk = blk0; blk < blk1; blk += 2) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (__builtin_expect(64 * blk + 63 > clean_from, 0)) clean_v(blk, V0);
            dma_k(blk + 2, K0);
            dma_v(blk + 1, V1);
            mx = step(blk, mx, K1, V0);
            if (blk + 1 >= blk1) break;
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (__builtin_expect(64 * blk + 127 > clean_from, 0)) clean_v(blk + 1, V1);
            dma_k(blk + 3, K1);
            dma_v(blk + 2, V0);
            mx = step(blk + 1, mx, K0, V1);
        }
        if (clean_from != INT_MAX) break;
        float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int v = 0; v < 16; ++v) t[v & 3] = fmaf(o[dt][v], 0.f, t[v & 3]);
        const bool any = __ballot((t[0] + t[1]) + (t[2] + t[3]) != 0.f) != 0;
        if (lane == 0) flag[wave] = any;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (__builtin_amdgcn_readfirstlane(flag[0] | flag[1] | flag[2] | flag[3]) == 0) break;
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        clean_from = wg_first;
    }

    l += __shfl_xor(l, 32, 64);
    if (parts > 1) {
        const size_t w = ((static_cast<size_t>(kv) * (items - pp.unsplit) + si) * pp.parts + part) * 4 + wave;
        float* od = pp.o + (w * 32 + col) * kHD;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                *reinterpret_cast<float4*>(od + 32 * dt + 8 * u + 4 * h) =
                    make_float4(o[dt][4 * u], o[dt][4 * u + 1], o[dt][4 * u + 2], o[dt][4 * u + 3]);
        if (h == 0) pp.ml[w * 32 + col] = make_float2(m, l);
        return;
    }
    if (tok >= p.T || (items - 1 - idx) * 4 + wave >= entries) return;
    const float inv = 1.f / l;
    const float* gate = p.Y + static_cast<size_t>(tok) * p.ld_y + static_cast<size_t>(head) * 2 * kHD + kHD;
    float* dst = out + static_cast<size_t>(tok) * (p.nq * kHD) + static_cast<size_t>(head) * kHD;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int d0 = 32 * dt + 8 * u + 4 * h;
            float4 r;
            r.x = o[dt][4 * u] * inv * sigmoid_f(gate[d0]);
            r.y = o[dt][4 * u + 1] * inv * sigmoid_f(gate[d0 + 1]);
            r.z = o[dt][4 * u + 2] * inv * sigmoid_f(gate[d0 + 2]);
            r.w = o[dt][4 * u + 3] * inv * sigmoid_f(gate[d0 + 3]);
            *reinterpret_cast<float4*>(dst + d0) = r;
        }
}

// grid (split items * 4 waves, nkv, 4), 256 threads
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs p, float* __restrict__ out, int items, PfParts pp) {
    merge_parts(p, out, items, pp, blockIdx.x, blockIdx.y, blockIdx.z);
}

}  // namespace

namespace rl {

// q fragments, then the parts of at most kMaxParts workgroups (128 queries each)
constexpr int kMaxParts = 256;
static size_t attn_prefill_q_bytes(int nq, int T) {
    return static_cast<size_t>(nq) * ((T + 15) / 16) * 16 * kHD * 2 * 2 + 256;
}
size_t attn_prefill_workspace_bytes(int nq, int T) {
    return attn_prefill_q_bytes(nq, T) + static_cast<size_t>(kMaxParts) * 128 * (kHD * 4 + 8) + 256;
}

void attn_prefill_layer(const float* Y, int ld_y, const float* q_norm, const float* k_norm, uint16_t* kc,
                        uint16_t* vt, int ctx, const int* pos_dev, int T, int nq, int nkv, int hd, int rot,
                        float theta, float eps, void* ws, size_t ws_bytes, float* out, hipStream_t s, int max_keys) {
    RL_REQUIRE(hd == kHD, RL_ERR_UNSUPPORTED, "attn prefill: head_dim must be 256");
    RL_REQUIRE(nkv > 0 && nq % nkv == 0, RL_ERR_RANGE, "attn prefill: n_q must be a multiple of n_kv");
    const int G = nq / nkv;
    RL_REQUIRE(G >= 1 && G <= 8, RL_ERR_UNSUPPORTED, "attn prefill: n_q/n_kv must be in 1..8");
    RL_REQUIRE(T >= 1 && T <= 65535 * 16, RL_ERR_RANGE, "attn prefill: bad token count");
    RL_REQUIRE(ctx > 0 && ctx % kChunk == 0, RL_ERR_RANGE, "attn prefill: cache capacity must be a multiple of 256");
    RL_REQUIRE(rot >= 2 && rot % 2 == 0 && rot <= hd, RL_ERR_RANGE, "attn prefill: bad rotary dim");
    RL_REQUIRE(Y && kc && vt && pos_dev && ws && out, RL_ERR_RANGE, "attn prefill: null pointer");
    RL_REQUIRE(ws_bytes >= attn_prefill_q_bytes(nq, T), RL_ERR_RANGE, "attn prefill: workspace too small");
    AttnArgs p{};
    p.Y = Y;
    p.ld_y = ld_y;
    p.q_norm = q_norm;
    p.k_norm = k_norm;
    p.kc = kc;
    p.vt = vt;
    p.ctx = ctx;
    p.pos = pos_dev;
    p.T = T;
    p.nq = nq;
    p.nkv = nkv;
    p.G = G;
    p.rot = rot;
    p.theta = theta;
    p.eps = eps;
    i32x4* qp = static_cast<i32x4*>(ws);
    // (the position is on the device: the context is at most the cache's capacity; the
    // kernel below addresses a head's cache with 32-bit offsets)
    if (attn_prefill_is_short(T, max_keys > 0 ? std::min(max_keys, ctx) : ctx) || ctx >= 1 << 23) {
        attn_prefill_short(p, qp, out, s);
        return;
    }
    // a large cache and keys that only the device knows: the kernels choose
    const bool auto_route = max_keys <= 0 && attn_prefill_auto_short(T);
    // four heads per workgroup share the angles once that still leaves two workgroups per CU
    // (1500 tokens: 31 us); with fewer tokens one head each, for the latency
    const int hpw = ((T + 15) / 16) * (nq + 2 * nkv) >= 8 * device_cus() ? 4 : 1;
    if (auto_route) {
        attn_prefill_short_prep(p, qp, s);
    } else {
        hipLaunchKernelGGL(qk_prep_pf_kernel, dim3((T + 15) / 16 + 1, (nq + 2 * nkv + hpw - 1) / hpw), dim3(256), 0, s, p,
                           qp, hpw);
        check_launch("qk_prep_pf_kernel");
    }
    const int items = (G * ((T + 31) / 32) + 3) / 4;  // workgroups per kv head
    // whole rounds of one workgroup per CU take all positions; the rest are split so that
    // they fill a round (with the parts' memory: a workspace of just the q fragments takes
    // every workgroup whole)
    const int cus = std::min(device_cus(), kMaxParts);
    PfParts pp{};
    pp.unsplit = static_cast<int>(static_cast<long>(items) * nkv / cus * cus / nkv);
    const int split = items - pp.unsplit;
    pp.parts = split ? std::max(1, std::min(cus / (split * nkv), 16)) : 1;
    const size_t off = (attn_prefill_q_bytes(nq, T) + 255) / 256 * 256;
    if (pp.parts > 1 && ws_bytes >= off + static_cast<size_t>(split) * nkv * pp.parts * 128 * (kHD * 4 + 8)) {
        pp.ml = reinterpret_cast<float2*>(static_cast<char*>(ws) + off);
        pp.o = reinterpret_cast<float*>(pp.ml + static_cast<size_t>(split) * nkv * pp.parts * 128);
    } else {
        pp.unsplit = items;
        pp.parts = 1;
    }
    const int slots = pp.unsplit + (items - pp.unsplit) * pp.parts;  // workgroups per kv head
    const int per = 8 % nkv == 0 ? 8 / nkv : 1;
    const int wgs = 8 % nkv == 0 ? (slots + per - 1) / per * 8 : slots * nkv;
    hipLaunchKernelGGL(attn_prefill_kernel, dim3(wgs), dim3(256), 0, s, p, qp, out, items, pp,
                       static_cast<int>(auto_route));
    check_launch("attn_prefill_kernel");
    if (auto_route) {
        attn_prefill_auto_finish(p, qp, out, items, pp, s);
    } else if (pp.parts > 1) {
        hipLaunchKernelGGL(attn_merge_kernel, dim3((items - pp.unsplit) * 4, nkv, 4), dim3(256), 0, s, p, out, items, pp);
        check_launch("attn_merge_kernel");
    }
}

}  // namespace rl

extern "C" {

size_t rl_hip_attn_prefill_workspace_bytes(int n_q, int T) { return rl::attn_prefill_workspace_bytes(n_q, T); }

int rl_hip_attn_prefill_layer(const float* Y, int ld_y, const float* q_norm, const float* k_norm, uint16_t* k_cache,
                              uint16_t* vt_cache, int ctx, const int* pos_dev, int T, int n_q, int n_kv, int head_dim,
                              int rotary_dim, float theta, float eps, void* workspace, size_t workspace_bytes,
                              float* out, void* stream) {
    return rl_hip_attn_prefill_layer_keys(Y, ld_y, q_norm, k_norm, k_cache, vt_cache, ctx, pos_dev, T, n_q, n_kv, head_dim,
                                          rotary_dim, theta, eps, workspace, workspace_bytes, out, 0, stream);
}

int rl_hip_attn_prefill_layer_keys(const float* Y, int ld_y, const float* q_norm, const float* k_norm, uint16_t* k_cache,
                                   uint16_t* vt_cache, int ctx, const int* pos_dev, int T, int n_q, int n_kv, int head_dim,
                                   int rotary_dim, float theta, float eps, void* workspace, size_t workspace_bytes,
                                   float* out, int max_keys, void* stream) {
    return guard([&] {
        rl::attn_prefill_layer(Y, ld_y, q_norm, k_norm, k_cache, vt_cache, ctx, pos_dev, T, n_q, n_kv, head_dim,
                               rotary_dim, theta, eps, workspace, workspace_bytes, out, S(stream), max_keys);
    });
}

}  // extern "C"
