// Results handed out to the host (readback.hip): laid out on the device, copied once.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>

namespace wv {

// A padded plane / volume: cell (x, y, z) at off + y * sy + z * sz + x (2D: NZ = 1).
// Grid order, in which callers hold fields: x fastest, then z, then y.
struct PaddedGrid {
    int NX, NY, NZ;
    long long off, sy, sz;
    size_t row() const { return (size_t)NX * NZ; }
};

// Staging buffer of a handle, of at most kStageBytes (or one trace / one y row): results go through
// it in parts. It is device memory, or, where none is left, pinned host memory that the kernels write
// across the link, so that results can be had from a full device. It grows to what was asked for, and
// goes with the handle. The lock is held for a whole read-back, since threads may read results of one
// handle side by side.
class Staging {
  public:
    static constexpr size_t kStageBytes = 64u << 20;
    ~Staging() { drop(); }
    // room for `items` of `bytes` each plus `extra`: items fitted (cut to what fits), 0: no memory
    size_t reserve(size_t items, size_t bytes, size_t extra)
    {
        items = std::min(items, std::max<size_t>(1, (kStageBytes - std::min(kStageBytes, extra)) / bytes));
        for (; items; items /= 2) {
            const size_t need = items * bytes + extra;
            if (need <= n_) return items;
            drop();
            if (hipMalloc((void **)&p_, need) == hipSuccess) {
                n_ = need;
                return items;
            }
            (void)hipGetLastError();
            p_ = nullptr;
            if (items > 1) continue;
            if (hipHostMalloc((void **)&p_, need, hipHostMallocDefault) == hipSuccess) {
                n_ = need;
                pinned_ = true;
                return items;
            }
            (void)hipGetLastError();
            p_ = nullptr;
        }
        return 0;
    }
    char *data() const { return p_; }
    // between this buffer and the caller's memory, behind the work on `st`
    hipError_t copy_out(void *dst, const void *src, size_t n, hipStream_t st) const
    {
        return copy(dst, src, n, hipMemcpyDeviceToHost, st);
    }
    hipError_t copy_in(void *dst, const void *src, size_t n, hipStream_t st) const
    {
        return copy(dst, src, n, hipMemcpyHostToDevice, st);
    }
    std::mutex lock;

  private:
    hipError_t copy(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t st) const
    {
        if (!pinned_) return hipMemcpyAsync(dst, src, n, kind, st);
        const hipError_t e = hipStreamSynchronize(st);
        if (e == hipSuccess) std::memcpy(dst, src, n);
        return e;
    }
    void drop()
    {
        if (p_) (void)(pinned_ ? hipHostFree(p_) : hipFree(p_));
        p_ = nullptr;
        n_ = 0;
        pinned_ = false;
    }
    char *p_ = nullptr;
    size_t n_ = 0;
    bool pinned_ = false;
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
