// Launchers of the resident time loop for one physics (instantiated per file, resident2d_*.hip).
#pragma once

#include <type_traits>

#include "resident2d_kernel.hpp"

namespace wv {
namespace {

template <typename Kern>
hipError_t res_launch(Kern k, const ResGo &g)
{
    const int threads = g.plan->nwv * 64;
    hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)g.lds);
    if (e != hipSuccess) return e;
    if (g.capacity) {
        int dev = 0, cus = 0, nb = 0;
        if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
        if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
        if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)k, threads, g.lds)) != hipSuccess) return e;
        *g.capacity = nb * cus;
        return hipSuccess;
    }
    Res2DKernArgs ka{*g.L, *g.F, *g.C, *g.T, *g.P, *g.A, *g.X, g.rec};
    void *args[] = {&ka};
    return hipLaunchCooperativeKernel((const void *)k, dim3(g.plan->blocks()), dim3(threads), args, (unsigned)g.lds, g.st);
}

// rows per wavefront: 1, 2, 4 with up to 16 wavefronts per block (128 registers per lane), 4 and 8 with
// up to 8 (the LDS strides are those of the largest tile of a variant)
template <int PHYS, int H, bool REC>
hipError_t res_rows(const ResGo &g)
{
    constexpr int W8 = PHYS == ELASTIC ? 2 : 4;
    switch (g.plan->srow) {
    case 1:
        if constexpr (!REC) return res_launch(res2d<PHYS, H, 1, 1024, 4, false>, g);
        return hipErrorInvalidValue;
    case 2: return res_launch(res2d<PHYS, H, 2, 1024, 4, REC>, g);
    case 4:
        if (g.plan->wmax == 8) return res_launch(res2d<PHYS, H, 4, 512, 4, REC>, g);
        return res_launch(res2d<PHYS, H, 4, 1024, 4, REC>, g);
    case 8: return res_launch(res2d<PHYS, H, 8, 512, W8, REC>, g);
    default: return hipErrorInvalidValue;
    }
}

template <int PHYS, bool REC>
hipError_t res_order(int order, const ResGo &g)
{
    switch (order / 2) {
    case 1: return res_rows<PHYS, 1, REC>(g);
    case 2: return res_rows<PHYS, 2, REC>(g);
    case 3: return res_rows<PHYS, 3, REC>(g);
    case 4: return res_rows<PHYS, 4, REC>(g);
    case 5: return res_rows<PHYS, 5, REC>(g);
    case 6: return res_rows<PHYS, 6, REC>(g);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace wv
