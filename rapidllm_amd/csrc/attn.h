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

// attn.hip: prefill over a short context (qp: the workspace)
inline bool attn_prefill_is_short(int T, int keys) { return keys <= 768 || (keys <= 1024 && T <= 128); }
void attn_prefill_short(const AttnArgs& p, i32x4* qp, float* out, hipStream_t s);

}  // namespace rl
