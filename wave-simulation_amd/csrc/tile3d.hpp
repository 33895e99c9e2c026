// Staging of x-z tiles of 3D fields, plane by plane along depth (elastic3d.hip, adjoint3d.hip).
#pragma once

#include "buffer.hpp"
#include "elastic3d.hpp"

namespace wv {

namespace {

constexpr int NTH = TILE_X * BLOCK_Y;

// Thread share of the region [x0-HX, x0+64+HX) x [z0-HZ, z0+TZ+HZ) of one y plane.
template <int HX, int HZ, int TZ>
struct Region {
    static constexpr int RW = TILE_X + 2 * HX;
    static constexpr int RH = TZ + 2 * HZ;
    static constexpr int TOT = RW * RH;
    static constexpr int IT = (TOT + NTH - 1) / NTH;
    float v[IT];
    __device__ __forceinline__ void load(const float *__restrict__ g, const Layout3D &L, int x0, int y, int z0, int tid)
    {
        const long long base = L.at(x0 - HX, y, z0 - HZ);
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = tid + k * NTH;
            if (TOT % NTH == 0 || i < TOT) {
                const int r = i / RW;
                const int c = i - r * RW;
                v[k] = g[base + (long long)r * L.pitch + c];
            }
        }
    }
    __device__ __forceinline__ void store(float (*S)[RW], int tid) const
    {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = tid + k * NTH;
            if (TOT % NTH == 0 || i < TOT) {
                const int r = i / RW;
                const int c = i - r * RW;
                S[r][c] = v[k];
            }
        }
    }
    // rows of an LDS array that every thread's share fits in (surplus threads write padding)
    static constexpr int RHP = (IT * NTH + RW - 1) / RW;
    // the same without a guard (S has RHP rows), so no divergent branch sits between the loads
    // in flight and this store
    __device__ __forceinline__ void store_padded(float (*S)[RW], int tid) const
    {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = tid + k * NTH;
            const int r = i / RW;
            const int c = i - r * RW;
            S[r][c] = v[k];
        }
    }
};

// Byte offsets, within one y plane, of a thread's share of a Region (the same
// for every plane, so they are computed once per block).
template <int HX, int HZ, int TZ>
struct RegionOff {
    using R = Region<HX, HZ, TZ>;
    unsigned o[R::IT];
    __device__ __forceinline__ void init(const Layout3D &L, int x0, int z0, int tid)
    {
#pragma unroll
        for (int k = 0; k < R::IT; k++) {
            const int i = min(tid + k * NTH, R::TOT - 1);  // surplus threads reload the last element
            const int r = i / R::RW, c = i - r * R::RW;
            o[k] = (unsigned)(((z0 - HZ + r + L.H) * L.pitch + (x0 - HX + c + XPAD)) * 4);
        }
    }
};

// One y plane of a field as a buffer resource (plane offsets stay 32-bit for any grid).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const float *f, const Layout3D &L, int y)
{
    return brsrc(f + (long long)(y + L.H) * L.slab, (unsigned)(L.slab * 4));
}

template <int HX, int HZ, int TZ>
__device__ __forceinline__ void load_region(Region<HX, HZ, TZ> &g, const RegionOff<HX, HZ, TZ> &o, const float *f,
                                            const Layout3D &L, int y)
{
    const auto b = plane_rsrc(f, L, y);
#pragma unroll
    for (int k = 0; k < Region<HX, HZ, TZ>::IT; k++) g.v[k] = bload(b, o.o[k], 0);
}

}  // namespace

}  // namespace wv
