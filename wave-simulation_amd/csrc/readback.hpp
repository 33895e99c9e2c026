// Results handed out to the host (readback.hip): laid out on the device, copied once.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace wv {

// A padded plane / volume: cell (x, y, z) at off + y * sy + z * sz + x (2D: NZ = 1).
// Grid order, in which callers hold fields: x fastest, then z, then y.
struct PaddedGrid {
    int NX, NY, NZ;
    long long off, sy, sz;
    size_t row() const { return (size_t)NX * NZ; }
};

// Device staging buffer of a handle, of at most kStageBytes (or one trace / one y row): results go
// through it in parts. It grows to what was asked for, and goes with the handle. The lock is held
// for a whole read-back, since threads may read results of one handle side by side.
class Staging {
  public:
    static constexpr size_t kStageBytes = 64u << 20;
    ~Staging()
    {
        if (p_) (void)hipFree(p_);
    }
    // room for `items` of `bytes` each plus `extra`: items fitted (cut to what fits), 0: no memory
    size_t reserve(size_t items, size_t bytes, size_t extra);
    char *data() const { return p_; }
    std::mutex lock;

  private:
    char *p_ = nullptr;
    size_t n_ = 0;
};

// Each call orders itself after the work on `st` and returns with `out` filled.

// out[r][t] = seis[t][r0 + r] for nr traces of a time-major [NT][total] array
hipError_t read_traces(Staging &S, const float *seis, int total, int r0, int nr, int NT, float *out, hipStream_t st);
// a padded array in grid order
hipError_t read_grid(Staging &S, const float *f, const PaddedGrid &g, float *out, hipStream_t st);
hipError_t read_grid(Staging &S, const double *f, const PaddedGrid &g, double *out, hipStream_t st);
// Gradient with respect to vp (0), vs (1) or rho (2) from the gradients with respect to the
// coefficients, through the averaging rules of the coefficient preparation (Modelparameter.cpp:
// 336-639): c[0 .. dim) 1/rho along x, y(, z), then M, mu, and mu averaged in xy(, xz, yz).
// model: vp, vs, rho on the host in grid order.
hipError_t read_model_gradient(Staging &S, int dim, int param, const PaddedGrid &g, const double *const *c,
                               const float *const *model, double *out, hipStream_t st);

}  // namespace wv
