// attn.h -- what the decode (attn.hip) and prefill (attn_prefill.hip) attention share.
#pragma once

#include "internal.h"

namespace rl {

constexpr int kHD = 256;
constexpr int kChunk = 256;
constexpr int kMaxPairs = 32;  // G * T query rows per kv head (<= 2 tiles of 16)

union H8 {
    f16x8 v;
    i32x4 i;
    _Float16 h[8];
};

__device__ inline float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }

struct AttnArgs {
    const float* Y;  // fused q(+gate)/k/v projection output, [T][ld_y]
    int ld_y;
    const float* q_norm;
    const float* k_norm;
    uint16_t* kc;  // [nkv][ctx][hd]
    uint16_t* vt;  // [nkv][hd][ctx]
    int ctx;
    const int* pos;  // device: position of token 0
    int T, nq, nkv, G, rot;
    int t_off, T_out;  // outputs: token t goes to column t_off + t of T_out
    float theta, eps;
    i32x4* qf;     // [nkv][8 s][4 g][2*PT ct][16 col] x 16 B
    float* part_o; // [nkv][chunks][kMaxPairs][hd]
    float* part_m; // [nkv][chunks][kMaxPairs]
    float* part_l;
    int max_chunks;
    float* out;     // optional [T][nq*hd]
    i32x4* frag;    // optional o_proj fragments (n = nq*hd)
    // batch decode: nb sequences ("slots") in one launch set.  Slot b's token t is
    // row b*T + t of Y and output column t_off + b*T + t; its cache, position and
    // workspace (qf, partials) sit kv_bstride elements, pos_stride ints and ws_slot
    // bytes after slot b-1's.
    int nb;
    size_t kv_bstride;
    int pos_stride;
    size_t ws_slot;
};

// Arguments of slot b (uniform per workgroup: the offsets stay in scalar registers).
__device__ inline void to_slot(AttnArgs& p, int b) {
    p.kc += b * p.kv_bstride;
    p.vt += b * p.kv_bstride;
    p.pos += b * p.pos_stride;
    p.Y += static_cast<size_t>(b) * p.T * p.ld_y;
    p.qf = reinterpret_cast<i32x4*>(reinterpret_cast<char*>(p.qf) + b * p.ws_slot);
    p.part_o = reinterpret_cast<float*>(reinterpret_cast<char*>(p.part_o) + b * p.ws_slot);
    p.part_m = reinterpret_cast<float*>(reinterpret_cast<char*>(p.part_m) + b * p.ws_slot);
    p.part_l = reinterpret_cast<float*>(reinterpret_cast<char*>(p.part_l) + b * p.ws_slot);
    p.t_off += b * p.T;
}

__host__ __device__ inline int pair_tiles(int G, int T) { return (G * T + 15) / 16; }

// Cache layouts (per kv head, ctx * 256 fp16), in MFMA fragment order so that every
// wave load is one contiguous 1 KiB run (lane l reads 16 B at 16 l), and the 4 waves
// of a chunk workgroup read adjacent runs at every step (one 16 KiB stretch):
//   K: [pos/256][d/32][(pos/16)%16][(d/8)%4][pos%16][d%8] -- A operand of S^T = K . Q^T
//   V: [pos/32][d/16][(pos/8)%4][d%16][pos%8]              -- A operand of O^T = V^T . P^T
__host__ __device__ inline size_t k_off(int pos, int d) {
    return ((((static_cast<size_t>(pos >> 8) * 8 + (d >> 5)) * 16 + ((pos >> 4) & 15)) * 4 + ((d >> 3) & 3)) * 16 +
            (pos & 15)) * 8 +
           (d & 7);
}
__host__ __device__ inline size_t v_off(int pos, int d) {
    return (((static_cast<size_t>(pos >> 5) * 16 + (d >> 4)) * 4 + ((pos >> 3) & 3)) * 16 + (d & 15)) * 8 + (pos & 7);
}

// ---- prefill
//
// The q fragments (16 bytes, 8 dims of a token) of every prefill kernel: qp[kv][t / 16][d / 32]
// [(d / 8) % 4][head of the kv head's G][hi/lo][t % 16].
__host__ __device__ inline size_t q_unit(int kv, int q, int G, int ntb16, int tb16) {
    return ((static_cast<size_t>(kv) * ntb16 + tb16) * 32 * G + q) * 32;  // of d = 0, hi, t % 16 = 0
}

// Split positions.  The chip runs one workgroup per CU, so the workgroups past the last
// full round (all of them, with few tokens) are split into `parts` ranges of positions;
// each range leaves its output, maximum and sum in the workspace.  The split follows from
// T and the head counts; a workgroup lowers the number of parts to what its context fills
// (kMinPartBlocks blocks of 64 positions each).  33 tokens over 8033 positions: 368 -> 62 us.
struct PfParts {
    int unsplit;  // workgroups per kv head that take all positions
    int parts;
    float* o;     // [kv head][split workgroup][part][4 waves][32 queries][256]
    float2* ml;   // [...][4 waves][32 queries]: maximum (log2 units), sum
};
constexpr int kMinPartBlocks = 2;
__device__ inline int pf_parts(int parts, int nblk) { return max(1, min(parts, nblk / kMinPartBlocks)); }
// keys 0 .. L-1 for item i (4 (token block, head) entries) of a kv head
__device__ inline int pf_keys(int i, int G, int T, int p0) {
    const int e_last = min(i * 4 + 3, G * ((T + 31) / 32) - 1);
    return p0 + min(T, 32 * (e_last / G) + 32);
}

// Adds the parts of the split queries: workgroup (bx < split items * 4 waves, kv, bz < 4) of
// 256 threads; each wave adds two queries side by side, lane l dims 4l .. 4l+3, parts in order.
__device__ inline void merge_parts(const AttnArgs& p, float* __restrict__ out, int items, const PfParts& pp, int bx,
                                   int kv, int bz) {
    const int si = bx / 4, wv = bx % 4;
    const int lane = threadIdx.x & 63, q0 = 8 * bz + 2 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = items - 1 - (pp.unsplit + si);
    const int e = item * 4 + wv;
    if (e >= p.G * ((p.T + 31) / 32)) return;
    const int parts = pf_parts(pp.parts, (pf_keys(item, p.G, p.T, *p.pos) + 63) / 64);
    const int head = kv * p.G + e % p.G, tok0 = 32 * (e / p.G) + q0;
    if (parts == 1 || tok0 >= p.T) return;
    const size_t w0 = (static_cast<size_t>(kv) * (items - pp.unsplit) + si) * pp.parts * 4 + wv;
    float M[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
    float4 a[2], g[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float* gate = p.Y + static_cast<size_t>(min(tok0 + j, p.T - 1)) * p.ld_y +
                            static_cast<size_t>(head) * 2 * kHD + kHD + 4 * lane;
        g[j] = make_float4(gate[0], gate[1], gate[2], gate[3]);
        a[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int k = 0; k < parts; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) M[j] = fmaxf(M[j], pp.ml[(w0 + 4 * k) * 32 + q0 + j].x);
    for (int k = 0; k < parts; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float2 ml = pp.ml[(w0 + 4 * k) * 32 + q0 + j];
            const float f = __builtin_amdgcn_exp2f(ml.x - M[j]);
            const float4 o = *reinterpret_cast<const float4*>(pp.o + ((w0 + 4 * k) * 32 + q0 + j) * kHD + 4 * lane);
            l[j] = fmaf(f, ml.y, l[j]);
            a[j].x = fmaf(f, o.x, a[j].x);
            a[j].y = fmaf(f, o.y, a[j].y);
            a[j].z = fmaf(f, o.z, a[j].z);
            a[j].w = fmaf(f, o.w, a[j].w);
        }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int tok = tok0 + j;
        if (tok >= p.T) return;
        const float inv = 1.f / l[j];
        float4 r;
        r.x = a[j].x * inv * sigmoid_f(g[j].x);
        r.y = a[j].y * inv * sigmoid_f(g[j].y);
        r.z = a[j].z * inv * sigmoid_f(g[j].z);
        r.w = a[j].w * inv * sigmoid_f(g[j].w);
        *reinterpret_cast<float4*>(out + static_cast<size_t>(tok) * (p.nq * kHD) + static_cast<size_t>(head) * kHD + 4 * lane) = r;
    }
}

// Which kernel a prompt chunk takes, where the host knows the keys (figures in attn.hip at
// attn_prefill_short_kernel).
__host__ __device__ inline bool attn_prefill_is_short(int T, int keys) {
    return keys <= 768 || (keys <= 1024 && T <= 128);
}
// ... and where it knows only the cache's capacity and the keys follow from the position on the
// device: the chunk's kernels read it and choose.  (The capacity alone sends every short prompt in
// a large cache the long way.)  24 / 4 heads, a cache of 32768 positions, by the capacity and so:
// 64 tokens over 64 keys 30.8 -> 15.1 us, 450 over 450 50.7 -> 37.5, 768 over 768 75.1 -> 58.9;
// longer contexts 33 over 8033 62.2 -> 53.8, 512 over 3512 114.6 -> 115.0, 760 over 3760 201.4 -> 200.3.
__host__ __device__ inline bool attn_prefill_auto_short(int keys) { return keys <= 768; }

// attn.hip: prefill over a short context (qp: the workspace)
void attn_prefill_short(const AttnArgs& p, i32x4* qp, float* out, hipStream_t s);
// The launches before and after attn_prefill_kernel where the device chooses: the short kernel's
// norm / RoPE pass, and the short kernel or the merge.
void attn_prefill_short_prep(const AttnArgs& p, i32x4* qp, hipStream_t s);
void attn_prefill_auto_finish(const AttnArgs& p, const i32x4* qp, float* out, int items, const PfParts& pp, hipStream_t s);

}  // namespace rl
