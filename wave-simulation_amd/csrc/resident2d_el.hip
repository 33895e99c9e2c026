// Resident 2D time loop: ELASTIC (see resident2d_kernel.hpp).
#include "resident2d_launch.hpp"

namespace wv {
hipError_t res2d_el(int order, bool rec, const void *go)
{
    const ResGo &g = *(const ResGo *)go;
    return rec ? res_order<ELASTIC, true>(order, g) : res_order<ELASTIC, false>(order, g);
}
}  // namespace wv
