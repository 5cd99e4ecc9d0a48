// prefill.h -- what the prompt linears' kernels (prefill.hip, prefill_x.hip) share.
#pragma once

#include "internal.h"

namespace rl {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTileRows = 16;  // weight rows per packed tile

__device__ inline float silu_fast(float x) { return x / (1.f + __expf(-x)); }

// Four consecutive outputs (of which `left` exist): one 16-byte access where the row
// stride and base allow (vec), else one by one.
__device__ inline void store_rows4(float* dst, const float (&o)[4], int left, int vec, bool add) {
    if (vec && left >= 4) {
        float4 r = make_float4(o[0], o[1], o[2], o[3]);
        float4* d = reinterpret_cast<float4*>(dst);
        if (add) {
            const float4 a = *d;
            r = make_float4(a.x + r.x, a.y + r.y, a.z + r.z, a.w + r.w);
        }
        *d = r;
        return;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (v < left) dst[v] = add ? dst[v] + o[v] : o[v];
}

// Workgroup -> (row block of nrb, token block of ntb); false: none left.  Each XCD (blockIdx %
// 8; the grid is a multiple of 8) takes a contiguous run of the order "gw token blocks
// wide, then down the rows", so the workgroups it runs at one time share both weights
// and activations in its L2.
__device__ inline bool xcd_block(int nrb, int ntb, int gw, int& rb, int& tb) {
    const int per = gridDim.x / 8;
    const int lin = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (lin >= nrb * ntb) return false;
    const int grp = lin / (nrb * gw), rem = lin - grp * nrb * gw;
    const int w = min(gw, ntb - grp * gw);
    rb = rem / w;
    tb = grp * gw + rem % w;
    return true;
}

}  // namespace rl
