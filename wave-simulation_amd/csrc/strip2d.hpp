// Arithmetic shared by the row-strip kernels (strip2d.hip) and the resident time loop
// (resident2d.hip): derivatives from a row or a column window, the adjoint's record.
#pragma once

#include <hip/hip_fp16.h>

#include "acq2d.hpp"

namespace wv {
namespace {

// general form: table taps for offsets -H..H
template <int K>
__device__ __forceinline__ float dtab(const float *v, const float *c)
{
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < K; k++) s = __builtin_fmaf(c[k], v[k], s);
    return s;
}

// y derivative at window row i (own row) with the row's table taps c (offsets -H..H)
template <int H, int N>
__device__ __forceinline__ float ydiff(const float (&w)[N], int i, const float *c)
{
    float s = 0.f;
#pragma unroll
    for (int k = 0; k <= 2 * H; k++) s = __builtin_fmaf(c[k], w[i + k - H], s);
    return s;
}

// Record NF fields (f0, f0+1, ...) of the wavefront's strip (S rows x 64
// columns) for the adjoint pass (Rec2D): the maximum over the strip (a DPP
// wavefront reduction) sets each field's FP16 scale; rows are stored in pairs,
// one 32-bit word per lane and pair.
template <int S, int NF>
__device__ __forceinline__ void record_strips(const Rec2D &R, const Layout2D &L, int nshots, int t, int f0, int shot,
                                              int x0, int ya, int lane, const float (&h)[NF][S])
{
    static_assert(S % 2 == 0, "rows are recorded in pairs");
    const bool in = x0 + lane < L.NX;
    float m[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        m[f] = 0.f;
#pragma unroll
        for (int r = 0; r < S; r++)
            if (in && ya + r < L.NY) m[f] = fmaxf(m[f], fabsf(h[f][r]));
    }
#pragma unroll
    for (int f = 0; f < NF; f++) m[f] = wave_max_nonneg(m[f]);
    if (ya >= L.NY) return;  // a strip wholly below the grid (last block row) records nothing
#pragma unroll
    for (int f = 0; f < NF; f++) {
        // strips whose values are all below 1e-30 are stored as zeros (scale 1); above it the
        // scale stays a normal float, so h / scale is finite
        const float sc = m[f] > 1e-30f ? m[f] * (1.f / 32768.f) : 1.f, is = 1.f / sc;
        const long long fs = ((long long)t * 5 + f0 + f) * nshots + shot;
        const long long q = (fs * R.nty + ya / S) * R.nbx + x0 / TILE_X;
        if (lane == 0) R.scale[q] = sc;
        unsigned *w = R.h + q * (S / 2) * TILE_X + lane;
#pragma unroll
        for (int p = 0; p < S / 2; p++) {
            // cells outside the grid store zeros
            const float a = (in && ya + 2 * p < L.NY) ? h[f][2 * p] * is : 0.f;
            const float b = (in && ya + 2 * p + 1 < L.NY) ? h[f][2 * p + 1] * is : 0.f;
            // written once, read once much later: streamed past the caches
            __builtin_nontemporal_store((unsigned)__half_as_ushort(__float2half_rn(a)) |
                                            ((unsigned)__half_as_ushort(__float2half_rn(b)) << 16),
                                        w + p * TILE_X);
        }
    }
}

}  // namespace
}  // namespace wv
