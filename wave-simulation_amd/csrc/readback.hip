// Layout changes and the gradient's chain rule for results that go to the host.
//
// A call used to copy whole padded arrays (for a shot's seismograms those of all shots, for a model
// gradient every coefficient's) to the host and pick or combine the values there, on one core. Here
// the device writes exactly what the call returns, in the caller's order, and one copy moves it. What
// bounds a call now is that copy: the kernels read and write a few MB at HBM speed. Per call, before
// and now: one of 64 shots' seismograms (300 traces of 500 steps out of 19,200) 1.6 ms -> 0.05 ms; a
// 144 x 120 x 104 wavefield 1.6 -> 0.44 ms; a model gradient of 600 x 600 cells 7.4 -> 0.37 ms, of
// 96 x 72 x 80 cells 37 -> 0.54 ms.
#include "readback.hpp"

namespace wv {

namespace {

// 64 x 64 tiles through LDS: reads run along the traces of a time step, writes along time
__global__ __launch_bounds__(256) void traces(const float *__restrict__ seis, int total, int r0, int nr, int NT,
                                              float *__restrict__ out)
{
    __shared__ float s[64][65];
    const int tb = blockIdx.x * 64, rb = blockIdx.y * 64, l = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int k = w; k < 64; k += 4)
        if (tb + k < NT && rb + l < nr) s[k][l] = seis[(long long)(tb + k) * total + r0 + rb + l];
    __syncthreads();
    for (int k = w; k < 64; k += 4)
        if (rb + k < nr && tb + l < NT) out[(long long)(rb + k) * NT + tb + l] = s[l][k];
}

// y rows [y0, y0 + ny)
template <typename T>
__global__ __launch_bounds__(256) void pack(const T *__restrict__ f, PaddedGrid g, int y0, int ny,
                                            T *__restrict__ out)
{
    const long long n = (long long)g.NX * g.NZ * ny;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) {
        const long long row = i / g.NX;
        const int x = (int)(i - row * g.NX), y = (int)(row / g.NZ), z = (int)(row - (long long)y * g.NZ);
        out[i] = f[g.off + (y0 + y) * g.sy + z * g.sz + x];
    }
}

struct ChainArgs {
    const double *c[8];
    const float *vp, *vs, *rho;  // of rows [y0 - 1, y0 + ny] as far as the grid has them
};

// One thread per cell gathers what the coefficients of its neighbours contribute to it, in FP64.
template <int DIM>
__global__ __launch_bounds__(256) void chain_rule(int param, PaddedGrid g, int y0, int ny, ChainArgs A,
                                                  double *__restrict__ out)
{
    const long long gs[3] = {1, (long long)g.NX * g.NZ, g.NX};  // steps along x, y, z in grid order
    const long long ps[3] = {1, g.sy, g.sz};                    // in the padded layout
    const long long n = gs[1] * ny, m0 = y0 > 0 ? gs[1] : 0;
    const int len[3] = {g.NX, g.NY, g.NZ};
    auto mu = [&](long long i) {
        const double m = (double)A.rho[i] * A.vs[i] * A.vs[i];
        return m < 1.0 ? 1.0 : m;
    };
    for (long long k = blockIdx.x * 256ll + threadIdx.x; k < n; k += gridDim.x * 256ll) {
        const long long row = k / g.NX, i = k + m0;
        const int yr = (int)(row / g.NZ);
        const int p[3] = {(int)(k - row * g.NX), y0 + yr, (int)(row - (long long)yr * g.NZ)};
        const long long o = g.off + p[1] * g.sy + p[2] * g.sz + p[0];
        const double r = A.rho[i], a = A.vp[i], b = A.vs[i];
        if (param == 0) {
            out[k] = A.c[DIM][o] * 2.0 * r * a;
            continue;
        }
        // mu: itself, and in the harmonic averages that this cell is part of
        double gmu = A.c[DIM + 1][o];
        const double mi = mu(i);
#pragma unroll
        for (int pl = 0; pl < (DIM == 2 ? 1 : 3); pl++) {
            const int a0 = pl == 2 ? 1 : 0, a1 = pl == 0 ? 1 : 2;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int d0 = q & 1, d1 = q >> 1;
                if (p[a0] < d0 || p[a1] < d1) continue;
                const long long j = i - d0 * gs[a0] - d1 * gs[a1];
                const bool in0 = p[a0] - d0 + 1 < len[a0], in1 = p[a1] - d1 + 1 < len[a1];
                double sum = 1.0 / mu(j);
                if (in0) sum += 1.0 / mu(j + gs[a0]);
                if (in1) sum += 1.0 / mu(j + gs[a1]);
                if (in0 && in1) sum += 1.0 / mu(j + gs[a0] + gs[a1]);
                const double w = in0 && in1 ? 0.25 : (in0 || in1 ? 0.5 : 1.0);
                const double m = 1.0 / (w * sum);
                if (m < 4.0) continue;  // the average is set to 0: no dependence
                gmu += A.c[DIM + 2 + pl][o - d0 * ps[a0] - d1 * ps[a1]] * m * m * w / (mi * mi);
            }
        }
        const bool own = r * b * b >= 1.0;  // mu is not clamped
        if (param == 1) {
            out[k] = own ? gmu * 2.0 * r * b : 0.0;
            continue;
        }
        double gr = A.c[DIM][o] * a * a;
        if (own) gr += gmu * b * b;
        // 1 / ((rho_i + rho_next) / 2); the last cell alone
#pragma unroll
        for (int ax = 0; ax < DIM; ax++) {
            if (p[ax] > 0) {
                const double av = 0.5 * ((double)A.rho[i - gs[ax]] + r);
                gr += A.c[ax][o - ps[ax]] * (-0.5 / (av * av));
            }
            if (p[ax] + 1 < len[ax]) {
                const double av = 0.5 * (r + (double)A.rho[i + gs[ax]]);
                gr += A.c[ax][o] * (-0.5 / (av * av));
            } else {
                gr += A.c[ax][o] * (-1.0 / (r * r));
            }
        }
        out[k] = gr;
    }
}

int blocks(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 8192); }

#define TRY(x)                                \
    do {                                      \
        const hipError_t e_ = (x);            \
        if (e_ != hipSuccess) return e_;      \
    } while (0)

template <typename T>
hipError_t read_rows(Staging &S, const T *f, const PaddedGrid &g, T *out, hipStream_t st)
{
    std::lock_guard<std::mutex> hold(S.lock);
    const size_t part = S.reserve(g.NY, g.row() * sizeof(T), 0);
    if (!part) return hipErrorOutOfMemory;
    T *d = (T *)S.data();
    for (size_t y = 0; y < (size_t)g.NY; y += part) {
        const size_t ny = std::min(part, g.NY - y), n = ny * g.row();
        pack<T><<<blocks(n), 256, 0, st>>>(f, g, (int)y, (int)ny, d);
        TRY(hipGetLastError());
        TRY(S.copy_out(out + y * g.row(), d, n * sizeof(T), st));
    }
    return hipStreamSynchronize(st);
}

}  // namespace

hipError_t read_traces(Staging &S, const float *seis, int total, int r0, int nr, int NT, float *out, hipStream_t st)
{
    std::lock_guard<std::mutex> hold(S.lock);
    // 65535 blocks of 64 traces are what the second grid dimension takes
    const size_t part = S.reserve(std::min(nr, 65535 * 64), (size_t)NT * sizeof(float), 0);
    if (!part) return hipErrorOutOfMemory;
    float *d = (float *)S.data();
    for (size_t r = 0; r < (size_t)nr; r += part) {
        const int n = (int)std::min(part, nr - r);
        traces<<<dim3((NT + 63) / 64, (n + 63) / 64), 256, 0, st>>>(seis, total, r0 + (int)r, n, NT, d);
        TRY(hipGetLastError());
        TRY(S.copy_out(out + r * NT, d, (size_t)n * NT * sizeof(float), st));
    }
    return hipStreamSynchronize(st);
}

hipError_t read_grid(Staging &S, const float *f, const PaddedGrid &g, float *out, hipStream_t st)
{
    return read_rows(S, f, g, out, st);
}
hipError_t read_grid(Staging &S, const double *f, const PaddedGrid &g, double *out, hipStream_t st)
{
    return read_rows(S, f, g, out, st);
}

hipError_t read_model_gradient(Staging &S, int dim, int param, const PaddedGrid &g, const double *const *c,
                               const float *const *model, double *out, hipStream_t st)
{
    std::lock_guard<std::mutex> hold(S.lock);
    // a part: its rows of the result and of the model, and the model's rows on either side
    const size_t row = g.row(), halo = 2 * 3 * row * sizeof(float);
    const size_t part = S.reserve(g.NY, row * (sizeof(double) + 3 * sizeof(float)), halo);
    if (!part) return hipErrorOutOfMemory;
    double *d = (double *)S.data();
    float *md = (float *)(d + part * row);
    ChainArgs A{};
    for (int k = 0; k < (dim == 2 ? 5 : 8); k++) A.c[k] = c[k];
    const float **m[3] = {&A.vp, &A.vs, &A.rho};
    for (size_t y = 0; y < (size_t)g.NY; y += part) {
        const size_t ny = std::min(part, g.NY - y);
        const size_t ya = y ? y - 1 : 0, yb = std::min<size_t>(g.NY, y + ny + 1), n = (yb - ya) * row;
        for (int k = 0; k < 3; k++) {
            *m[k] = md + k * (part + 2) * row;
            TRY(S.copy_in((void *)*m[k], model[k] + ya * row, n * sizeof(float), st));
        }
        if (dim == 2)
            chain_rule<2><<<blocks(ny * row), 256, 0, st>>>(param, g, (int)y, (int)ny, A, d);
        else
            chain_rule<3><<<blocks(ny * row), 256, 0, st>>>(param, g, (int)y, (int)ny, A, d);
        TRY(hipGetLastError());
        TRY(S.copy_out(out + y * row, d, ny * row * sizeof(double), st));
    }
    return hipStreamSynchronize(st);
}

}  // namespace wv
