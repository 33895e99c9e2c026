// Resident 2D time loop: ACOUSTIC (see resident2d_kernel.hpp).
#include "resident2d_launch.hpp"

namespace wv {
hipError_t res2d_ac(int order, bool rec, const void *go)
{
    (void)rec;  // the record belongs to the elastic adjoint
    const ResGo &g = *(const ResGo *)go;
    return res_order<ACOUSTIC, false>(order, g);
}
}  // namespace wv
