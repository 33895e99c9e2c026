// Resident 2D time loop for gfx950.
//
// One time step of the two-launch kernels moves every field and coefficient of every shot through
// memory twice.  A 2D shot is small next to the chip's own storage (256 CUs with 160 KB of LDS and
// 512 KB of registers each), so this kernel keeps it there: one cooperative launch runs all time
// steps of a run call, a block owns a tile of 64 columns x R rows of one shot, its fields live in
// LDS with an H-wide halo, its coefficients and x taps in registers, and only the CPML memory
// variables of frame tiles (read and written by their own block alone) stay in memory, where they
// hit L2.  A step is
//   velocity-type update, exchange of its halos, stress-type update, sources, exchange, receivers.
//
// Halo exchange.  A block needs the H outermost rows / columns of its four neighbours (no corners:
// every derivative is along one axis).  Each value travels as a 64-bit word (value, tag of the step)
// stored and polled with agent-scope atomics, so a word says by itself whether it has arrived and
// no flag, fence or second round trip follows the data: one exchange of 2048 words per block takes
// about 2 us, 1.0 us of it latency (measured on a 16 x 16 grid of blocks).
// A word's slot is free again when it is written next: a neighbour sends its velocity halos of step
// k + 1 only after it has received this block's stress halos of step k, and those were sent behind
// a block barrier that follows this block's last read of the neighbour's velocity halos of step k
// (likewise for the stress slots).  The exchange after the last step of a shot is therefore kept.
//
// Every wait ends: the launch is cooperative, the blocks meet once before they touch any state and
// give the launch up together when some block has not come in after RES_START_TICKS, and later waits
// end with an error after RES_WAIT_TICKS.  The host asks for the verdict only where it waits for the
// stream anyway, and has the ordinary kernels run the steps of a refused launch then.
//
// Arithmetic: the operations of the row-strip kernels (elastic) and of the tiled ones
// (acoustic, SH, TM-EM) in their order, so a run may change between them at any step.
#pragma once

#include "resident2d.hpp"
#include "strip2d.hpp"

namespace wv {
namespace {

constexpr unsigned long long RES_START_TICKS = 30000000ull;   // 0.3 s of the 100 MHz counter
constexpr unsigned long long RES_WAIT_TICKS = 2000000000ull;  // 20 s

// Fields each phase's result is exchanged for: along x and along y.
template <int PHYS>
struct ResFields;
template <>
struct ResFields<ELASTIC> {  // vx vy sxx syy sxy
    static constexpr int NF = 5, N = 2;
    static constexpr int X[2][2] = {{0, 1}, {2, 4}}, Y[2][2] = {{0, 1}, {4, 3}};
};
template <>
struct ResFields<ACOUSTIC> {  // vx vy p
    static constexpr int NF = 3, N = 1;
    static constexpr int X[2][1] = {{0}, {2}}, Y[2][1] = {{1}, {2}};
};
template <>
struct ResFields<TMEM> {  // hx hy ez
    static constexpr int NF = 3, N = 1;
    static constexpr int X[2][1] = {{1}, {2}}, Y[2][1] = {{0}, {2}};
};
template <>
struct ResFields<SH> {  // vz sxz syz
    static constexpr int NF = 3, N = 1;
    static constexpr int X[2][1] = {{0}, {1}}, Y[2][1] = {{0}, {2}};
};

// A value the compiler must take as new here: what the time loop derives from it (addresses of
// rows, halo words, memory variables) is computed where it is used instead of being kept in
// registers, or spilled, over the whole loop.
__device__ __forceinline__ int fresh_lane(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int fresh_uniform(int v)
{
    asm volatile("" : "+s"(v));
    return v;
}

// Read-only floats at uniform addresses (scalar loads).
typedef const __attribute__((address_space(4))) float *scalar_floats;
__device__ __forceinline__ scalar_floats row_taps(const float *table, int y, int K)
{
    return (scalar_floats)(unsigned long long)(table + (long long)y * K);
}
// ydiff with the taps read through the scalar cache
template <int H, int N>
__device__ __forceinline__ float ydiff_s(const float (&w)[N], int i, scalar_floats c)
{
    float s = 0.f;
#pragma unroll
    for (int k = 0; k <= 2 * H; k++) s = __builtin_fmaf(c[k], w[i + k - H], s);
    return s;
}

__device__ __forceinline__ unsigned agent_load(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The blocks of a launch meet before they touch any state: the last one in (or the first whose
// patience runs out) decides for all.  A launch queued behind a refused one is refused at once, since
// the state is not the one it was meant for; the host runs the steps of all of them.  True: go.
__device__ __forceinline__ bool res_check_in(const Res2DArgs &X, int *s_go)
{
    if (threadIdx.x == 0) {
        const unsigned go = 2 * X.launch, stop = 2 * X.launch + 1;
        const unsigned n = __hip_atomic_fetch_add(X.ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
        const unsigned long long t0 = wall_clock64();
        const unsigned behind = agent_load(X.ctl + 3);
        unsigned v = agent_load(X.ctl + 1);
        unsigned want = behind ? stop : n == X.arrive ? go : 0;
        while (v != go && v != stop) {
            if (!want && wall_clock64() - t0 > RES_START_TICKS) want = stop;
            if (want) {
                if (__hip_atomic_compare_exchange_strong(X.ctl + 1, &v, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT)) {
                    const unsigned first = want == go ? 0 : behind ? behind : X.launch;
                    if (first) __hip_atomic_store(X.ctl + 3, first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(X.host, ((unsigned long long)first << 32) | want, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_SYSTEM);
                    v = want;
                }
            } else {
                __builtin_amdgcn_s_sleep(2);
                v = agent_load(X.ctl + 1);
            }
        }
        *s_go = v == go;
    }
    __syncthreads();
    return *s_go != 0;
}

// H-wide halos of one phase as items of 64 words, one wavefront each: first the x items (side, field,
// group of 64 / H rows: lane = row in the group x column), then the y items (side, field, row: lane
// = column).  Bit 0 of an item is the side it arrives from, so the sender's item is the
// neighbour's with that bit flipped.
template <int PHYS, int H, int PH>
struct ResHalo {
    using RF = ResFields<PHYS>;
    static constexpr int N = RF::N, RPG = TILE_X / H, RW = TILE_X + 2 * H, NJ = 2;
    static constexpr int SH = N == 2 ? 2 : 1;  // bits of (side, field)

    struct Item {
        bool there, live;  // there is a neighbour on that side (uniform); this lane carries a word
        int step;          // its block number less this block's
        int own, halo;  // LDS offsets of this block's border value (sent) and of its halo value (received)
    };
    static __device__ __forceinline__ Item item(int idx, int nx, int R, int FS, int lane, int lrow, int lcol, int bx,
                                                int by, int nbx, int nby)
    {
        Item it;
        const bool x = idx < nx;
        const int j = x ? idx : idx - nx, side = j & 1;  // 0 left / top, 1 right / bottom
        const int f = N == 2 ? (j >> 1) & 1 : 0, g = j >> SH;
        const int fx = f ? RF::X[PH][N - 1] : RF::X[PH][0], fy = f ? RF::Y[PH][N - 1] : RF::Y[PH][0];
        const int pos = x ? bx : by, num = x ? nbx : nby;
        it.there = side ? pos + 1 < num : pos > 0;
        it.step = (x ? 1 : nbx) * (2 * side - 1);
        if (x) {
            const int r = g * RPG + lrow;
            it.live = lrow < RPG && r < R;
            const int base = fx * FS + (r + H) * RW + lcol;
            it.own = base + (side ? TILE_X : H);
            it.halo = base + (side ? TILE_X + H : 0);
        } else {
            it.live = true;
            const int base = fy * FS + g * RW + H + lane;
            it.own = base + (side ? R : H) * RW;
            it.halo = base + (side ? R + H : 0) * RW;
        }
        return it;
    }
    static __device__ __forceinline__ int x_items(int R) { return ((R + RPG - 1) / RPG) << SH; }
    static __device__ __forceinline__ int y_items() { return H << SH; }
};

typedef const __attribute__((address_space(4))) Res2DKernArgs *res_args;
// The launch's arguments, read anew (scalar loads that hit the constant cache).
__device__ __forceinline__ res_args fresh_args(res_args p)
{
    asm volatile("" : "+s"(p));
    return p;
}
#define RES_GLOBAL __attribute__((address_space(1)))

// Cells outside a CPML frame that share a tile or a wavefront with it have a = b = 0 in the tables, which
// leaves a finite derivative as it is but makes an infinite one NaN.  Lanes outside the x frame take no
// part in its update (where the registers are full, 8 rows of three fields, a select on psi costs less: SELX).
// Rows outside the y frame: a select on psi with three fields; with the five of P-SV an a that changes no
// finite derivative, psi being far below half a unit in its last place, and leaves an infinite one as
// it is, with zeros stored for psi (SELY).  us per step, with selects for x and y and without: 1000 x 1000
// elastic 12.1 and 10.9; 428 x 392 TM-EM of 40 shots at order 10 (8 rows) 59.9 and 61.5, 882 x 482 of 5 at
// order 4 (4 rows) 13.7 and 13.6.
constexpr float RES_OUTSIDE_A = 1e-30f;

// Floats of a wavefront's private memory variables: two phases x (x frame, y frame) x NP * S rows.
template <int PHYS, int S>
constexpr int res_psi_wave()
{
    return 4 * (PHYS == ELASTIC ? 2 : 1) * S * TILE_X;
}

// One launch: see the top of this file.  S rows per wavefront, MAXT threads at most per block, REC:
// the elastic derivative sums of every step are recorded for the adjoint pass.
template <int PHYS, int H, int S, int MAXT, int MINW, bool REC>
__global__ __launch_bounds__(MAXT, MINW) void res2d(Res2DKernArgs KA)
{
    using RF = ResFields<PHYS>;
    constexpr int NF = RF::NF, K = 2 * H + 1, RW = TILE_X + 2 * H, NW = S + 2 * H;
    constexpr int RMAX = MAXT / 64 * S, FS = (RMAX + 2 * H) * RW;  // LDS strides of the largest tile: constants
    constexpr int NP = PHYS == ELASTIC ? 2 : 1;   // memory variables per phase and axis
    constexpr bool SELY = PHYS != ELASTIC, SELX = SELY && S == 8;  // see RES_OUTSIDE_A
    constexpr int PV = NP * S >= 4 ? 4 : NP * S;  // floats per access of the private memory variables
    typedef float vpsi __attribute__((ext_vector_type(PV)));
    extern __shared__ float lds[];
    __shared__ int s_go, s_bad;
    const res_args G0 = (res_args)__builtin_amdgcn_kernarg_segment_ptr();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_ = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_;
    const int nwv = KA.X.nwv, nthr = nwv * 64, R = nwv * S;
    float *const sf = lds;
    float *const s_cy = lds + NF * FS;  // [RMAX][4] a_y, b_y, a_y(half), b_y(half)
    if (tid == 0) s_bad = 0;
    if (!res_check_in(KA.X, &s_go)) return;

    // contiguous tiles on one XCD (blocks are dealt to the 8 XCDs round robin)
    const int nblk = gridDim.x, b = blockIdx.x, xcd = b & 7, q8 = nblk >> 3, rem = nblk & 7;
    const int t = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + (b >> 3);
    const int ntile = KA.X.nbx * KA.X.nby, slot = t / ntile, tile = t - slot * ntile;
    const int by = tile / KA.X.nbx, bx = tile - by * KA.X.nbx;
    const int x0 = bx * TILE_X, y0 = by * R, x = x0 + lane, NX = KA.L.NX, NY = KA.L.NY;
    const int ya = y0 + wave * S;                    // first row of the wavefront
    const bool xin = x < NX;
    const Col col = column(KA.L, KA.P, x);
    const int PW = KA.P.on ? KA.P.W : 0, W2 = 2 * PW;
    const bool xframe = PW && (x0 < PW || x0 + TILE_X > NX - PW);  // the tile touches the x frame
    const bool yframe = PW && (ya < PW || ya + S > NY - PW);       // the wavefront's rows touch the y frame
    const bool xf = col.xi >= 0;
    int yrows = 0;  // the wavefront's rows inside the y frame, one bit each
    for (int r = 0; r < S; r++)
        if (frame_index(ya + r, NY, PW, KA.C.free_surface != 0) >= 0) yrows |= 1 << r;
    // rows H and more from both edges share one set of y taps
    const bool inner = ya >= H && ya + S - 1 <= NY - 1 - H;

    float cxf[K], cxb[K];
    load_taps<H>(cxf, KA.T.xf, x);
    load_taps<H>(cxb, KA.T.xb, x);
    for (int e = tid; e < R; e += nthr) {
        const bool on = PW && y0 + e < NY;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float a = on ? (h ? KA.P.ayh : KA.P.ay)[y0 + e] : 0.f, b = on ? (h ? KA.P.byh : KA.P.by)[y0 + e] : 0.f;
            s_cy[4 * e + 2 * h] = SELY || a != 0.f || b != 0.f ? a : RES_OUTSIDE_A;
            s_cy[4 * e + 2 * h + 1] = b;
        }
    }
    // coefficients of the own cells
    constexpr int NC = PHYS == ELASTIC ? 5 : (PHYS == TMEM ? 4 : 3);
    float co[NC][S];
#pragma unroll
    for (int r = 0; r < S; r++) {
        const bool in = ya + r < NY;
        const long long o = KA.L.at(x0, min(ya + r, NY - 1)) + lane;
#pragma unroll
        for (int k = 0; k < NC; k++) co[k][r] = in ? KA.C.c[k][o] : 0.f;
    }
    const bool fs = KA.C.free_surface != 0, abs = KA.C.damp != nullptr;
    unsigned tag = KA.X.tag0;
    bool bad = false;
    constexpr int PSI_WAVE = res_psi_wave<PHYS, S>();
    // this lane's memory variables of phase ph, ax 0 x frame, 1 y frame: variable-major, PV at a time
    auto psi_at = [&](res_args G, int ph, int ax) {
        float *g = G->X.psi + ((long long)t * nwv + fresh_uniform(wave_)) * PSI_WAVE + (2 * ph + ax) * NP * S * TILE_X;
        return (RES_GLOBAL vpsi *)g + (tid & 63);
    };
    auto psi_load = [&](res_args G, int ph, int ax, float (&p)[NP * S]) {
        RES_GLOBAL vpsi *g = psi_at(G, ph, ax);
#pragma unroll
        for (int k = 0; k < NP * S / PV; k++) {
            const vpsi v = g[k * TILE_X];
#pragma unroll
            for (int i = 0; i < PV; i++) p[k * PV + i] = v[i];
        }
    };
    auto psi_store = [&](res_args G, int ph, int ax, const float (&p)[NP * S]) {
        RES_GLOBAL vpsi *g = psi_at(G, ph, ax);
#pragma unroll
        for (int k = 0; k < NP * S / PV; k++) {
            vpsi v;
#pragma unroll
            for (int i = 0; i < PV; i++) v[i] = p[k * PV + i];
            g[k * TILE_X] = v;
        }
    };
    // between the handle's frames and the private layout (start and end of a shot)
    auto psi_move = [&](int shot, bool in) {
#pragma unroll 1
        for (int q = 0; q < 4; q++) {
            const int ph = q >> 1, ax = q & 1, ya = y0 + fresh_uniform(wave_) * S, x = x0 + fresh_lane(tid & 63);
            if (!(ax ? yframe : xframe)) continue;
            float p[NP * S];
            if (!in) psi_load(G0, ph, ax, p);
#pragma unroll
            for (int j = 0; j < NP; j++) {
                const int var = PHYS == ELASTIC ? 2 * ph + j : ph;
#pragma unroll
                for (int r = 0; r < S; r++) {
                    const int yi = frame_index(ya + r, NY, PW, fs);
                    const bool on = ax ? yi >= 0 && xin : xf && ya + r < NY;
                    float *g = ax ? KA.P.psy[var] + ((long long)shot * W2 + max(yi, 0)) * NX + min(x, NX - 1)
                                  : KA.P.psx[var] + ((long long)shot * NY + min(ya + r, NY - 1)) * W2 + max(col.xi, 0);
                    if (in)
                        p[j * S + r] = on ? *g : 0.f;
                    else if (on)
                        *g = p[j * S + r];
                }
            }
            if (in) psi_store(G0, ph, ax, p);
        }
    };

    for (int shot = slot; shot < KA.X.nshots; shot += KA.X.conc) {
        const long long so = (long long)shot * KA.L.plane;
        // fields of the tile and its halo (the padding of the planes is zero)
#pragma unroll 1
        for (int f = 0; f < NF; f++) {
            const float *g = KA.F.f[f] + so;
            for (int row = wave; row < R + 2 * H; row += nwv) {
                const int y = y0 - H + row;
                const bool in = y < NY;
                float *d = sf + f * FS + row * RW;
                d[lane] = in ? g[KA.L.at(x0 - H, y) + lane] : 0.f;
                if (lane < 2 * H) d[TILE_X + lane] = in ? g[KA.L.at(x0 - H, y) + TILE_X + lane] : 0.f;
            }
        }
        psi_move(shot, true);
        // the tile's sources and receivers
        const int sb = (shot * KA.X.nby + by) * KA.X.nbx + bx;
        const int s0 = KA.X.bsrc_ptr[sb], ns = KA.X.bsrc_ptr[sb + 1] - s0;
        const int r0 = KA.X.brec_ptr[sb], nr = KA.X.brec_ptr[sb + 1] - r0;
        auto lds_cell = [&](res_args G, long long cell, int ty, int &o2) {
            // (a plane has fewer than 2^31 floats)
            const int pitch = G->L.pitch, gy = (int)cell / pitch, yy = gy - G->L.ypad, xx = (int)cell - gy * pitch - XPAD;
            const int o = (yy - y0 + H) * RW + (xx - x0 + H);
            int f = velocity_field<PHYS>(ty);
            o2 = -1;
            if (PHYS == ELASTIC && ty == 1) {
                f = 2;
                o2 = 3 * FS + o;
            }
            return f * FS + o;
        };
        auto source = [&](res_args G, int e, int &o1, int &o2) {
            const int id = ((const RES_GLOBAL int *)G->X.bsrc)[s0 + e];
            o1 = lds_cell(G, ((const RES_GLOBAL long long *)G->A.src_cell)[id], ((const RES_GLOBAL int *)G->A.src_type)[id], o2);
            return id;
        };
        auto signal = [&](res_args G, int id, int tt) {
            return ((const RES_GLOBAL float *)G->A.src_sig)[(long long)id * G->A.NT + tt];
        };
        auto receiver = [&](res_args G, int e, int &o1, int &o2) {
            const int id = ((const RES_GLOBAL int *)G->X.brec)[r0 + e];
            o1 = lds_cell(G, ((const RES_GLOBAL long long *)G->A.rec_cell)[id], ((const RES_GLOBAL int *)G->A.rec_type)[id], o2);
            return id;
        };
        auto record_sample = [&](res_args G, int id, int tt, int o1, int o2) {
            float v = sf[o1];
            if (PHYS == ELASTIC && o2 >= 0) {
                v += sf[o2];
                v *= 0.5f;
            }
            ((RES_GLOBAL float *)G->A.seis)[(long long)tt * G->A.rec_total + id] = v;
        };
        // the first source of every lane of wavefront 0 and the first receiver of every thread stay in
        // registers; the source's next sample is loaded a step ahead
        int so1 = 0, so2 = -1, ro1 = 0, ro2 = -1, rid = 0, sid = 0;
        float sv = 0.f;
        if (tid < ns && tid < 64) {
            sid = source(G0, tid, so1, so2);
            sv = signal(G0, sid, KA.X.t0);
        }
        if (tid < nr) rid = receiver(G0, tid, ro1, ro2);
        // memory variables (stress phase under ABS: the damping factors, in px) of the next phase,
        // loaded before the wait for its halos
        // (rows outside the y frame store zeros, and load zeros every time)
        float px[NP * S], py[NP * S];
#pragma unroll
        for (int k = 0; k < NP * S; k++) px[k] = py[k] = 0.f;
        auto load_psi = [&](int ph) {
            const res_args G = fresh_args(G0);
            if (xf) psi_load(G, ph, 0, px);
            if (yframe) psi_load(G, ph, 1, py);
            if (abs && ph == 1) {
                const int ya = y0 + fresh_uniform(wave_) * S;
                const RES_GLOBAL float *g = (const RES_GLOBAL float *)G->C.damp;
#pragma unroll
                for (int r = 0; r < S; r++)
                    px[r] = g[(long long)(min(ya + r, NY - 1) + G->L.ypad) * G->L.pitch + x0 + XPAD + (tid & 63)];
            }
        };
        // a phase's updated memory variables, stored behind its halo words
        auto store_psi = [&](int ph) {
            const res_args G = fresh_args(G0);
            if (xf) psi_store(G, ph, 0, px);
            if (yframe) {
                if constexpr (S > 1 && !SELY) {
#pragma unroll
                    for (int k = 0; k < NP * S; k++) py[k] = yrows >> k % S & 1 ? py[k] : 0.f;
                }
                psi_store(G, ph, 1, py);
            }
        };
        // CPML of the derivative d of every row: memory variable j of a phase, profile full or half
        // (outside the frames: see RES_OUTSIDE_A)
        auto cpml_x = [&](int j, float (&d)[S], bool half) {
            const float a = half ? col.axh : col.ax, b = half ? col.bxh : col.bx;
#pragma unroll
            for (int r = 0; r < S; r++) {
                if constexpr (SELX) {
                    const float p = __builtin_fmaf(a, d[r], b * px[j * S + r]);
                    px[j * S + r] = xf ? p : 0.f;
                    d[r] += px[j * S + r];
                } else {
                    px[j * S + r] = cpml(d[r], px[j * S + r], a, b);
                }
            }
        };
        auto cpml_y = [&](int j, float (&d)[S], bool half, int row) {
#pragma unroll
            for (int r = 0; r < S; r++) {
                const float *cy = s_cy + 4 * (row + r) + (half ? 2 : 0);
                if constexpr (S > 1 && SELY) {
                    const float p = __builtin_fmaf(cy[0], d[r], cy[1] * py[j * S + r]);
                    py[j * S + r] = yrows >> r & 1 ? p : 0.f;
                    d[r] += py[j * S + r];
                } else {
                    py[j * S + r] = cpml(d[r], py[j * S + r], cy[0], cy[1]);
                }
            }
        };
        // y derivative of field f at the wavefront's rows from a column window in registers; INNER: the
        // taps of an inner row for all (`in`), else every row's own (`table`), through the scalar cache
        auto y_rows = [&](auto inner_c, const float *table, const float *in, int f, int lr0, int ya, float (&d)[S]) {
            constexpr bool INNER = decltype(inner_c)::value;
            float w[NW];
#pragma unroll
            for (int i = 0; i < NW; i++) w[i] = sf[f * FS + lr0 + (i - H) * RW];
#pragma unroll
            for (int r = 0; r < S; r++)
                d[r] = ydiff_s<H, NW>(w, r + H,
                                      INNER ? row_taps(in, min(H, NY - 1), K) : row_taps(table, min(ya + r, NY - 1), K));
            __builtin_amdgcn_sched_barrier(0);
        };
        // x derivative of field f
        auto x_rows = [&](const float (&ct)[K], int f, int lr0, float (&d)[S]) {
#pragma unroll
            for (int r = 0; r < S; r++) d[r] = dtab<K>(sf + f * FS + lr0 + r * RW - H, ct);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto send = [&](auto ph) {
            constexpr int PH = decltype(ph)::value;
            using HL = ResHalo<PHYS, H, PH>;
            const res_args G = fresh_args(G0);
            const int lane = fresh_lane(tid & 63), wave = fresh_uniform(wave_), lrow = lane / H, lcol = lane - lrow * H;
            const int nx = HL::x_items(R), n = nx + HL::y_items(), nbx = G->X.nbx, nby = G->X.nby, words = G->X.words;
            RES_GLOBAL unsigned long long *const xch =
                (RES_GLOBAL unsigned long long *)G->X.xch + (long long)t * words + (PH ? G->X.phase1 : 0) + lane;
            for (int idx = wave; idx < n; idx += nwv) {
                const auto it = HL::item(idx, nx, R, FS, lane, lrow, lcol, bx, by, nbx, nby);
                if (!it.there) continue;
                if (it.live) {
                    const unsigned long long w =
                        ((unsigned long long)tag << 32) | (unsigned long long)__float_as_uint(sf[it.own]);
                    __hip_atomic_store(xch + (long long)it.step * words + (idx ^ 1) * 64, w, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        };
        auto recv = [&](auto ph) {
            constexpr int PH = decltype(ph)::value;
            using HL = ResHalo<PHYS, H, PH>;
            constexpr int NJ = HL::NJ;
            const res_args G = fresh_args(G0);
            const int lane = fresh_lane(tid & 63), wave = fresh_uniform(wave_), lrow = lane / H, lcol = lane - lrow * H;
            const int nx = HL::x_items(R), n = nx + HL::y_items(), nbx = G->X.nbx, nby = G->X.nby;
            RES_GLOBAL unsigned long long *const mine =
                (RES_GLOBAL unsigned long long *)G->X.xch + (long long)t * G->X.words + (PH ? G->X.phase1 : 0) + lane;
            for (int base = wave; base < n; base += NJ * nwv) {
                typename HL::Item it[NJ];
                bool want[NJ];
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    const int idx = base + j * nwv;
                    it[j] = HL::item(idx, nx, R, FS, lane, lrow, lcol, bx, by, nbx, nby);
                    want[j] = idx < n && it[j].there;
                }
                unsigned long long v[NJ];
                int spin = 0;
                unsigned long long since = 0;
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (int j = 0; j < NJ; j++)
                        if (want[j])
                            v[j] = __hip_atomic_load(mine + (base + j * nwv) * 64, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int j = 0; j < NJ; j++)
                        if (want[j] && it[j].live) ok = ok && (unsigned)(v[j] >> 32) == tag;
                    if (__all(ok)) break;
                    if ((++spin & 1023) == 0) {
                        if (!since) since = wall_clock64();
                        if (agent_load(G->X.ctl + 2) || wall_clock64() - since > RES_WAIT_TICKS) {
                            s_bad = 1;
                            break;
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    if (want[j] && it[j].live) sf[it[j].halo] = __uint_as_float((unsigned)v[j]);
            }
        };
        // One phase over the wavefront's rows.  All rows are read and computed before the first is
        // written (a write would order every later read behind it), without branches in between;
        // cells outside the grid are computed like the others and not written.  INNER: rows H and
        // more from both edges, whose y taps are one set (the free-surface operators equal the plain
        // ones there); the others read theirs through the scalar cache.
        auto velocity_rows = [&](auto inner_c, float (&rh)[REC ? 2 : 1][S]) {
            const res_args G = fresh_args(G0);
            const int wave = fresh_uniform(wave_), ya = y0 + wave * S;
            const int lr0 = (wave * S + H) * RW + H + fresh_lane(lane);
            float u[S], v[S], a[S], c[S];  // x derivatives u, a; y derivatives v, c
            // one derivative after the other, so that one window's registers are live at a time
            if constexpr (PHYS == ELASTIC) {
                y_rows(inner_c, G->T.yb_v, G->T.yb, 4, lr0, ya, v);
                y_rows(inner_c, G->T.yf_v, G->T.yf, 3, lr0, ya, c);
                x_rows(cxf, 2, lr0, u);
                x_rows(cxb, 4, lr0, a);
            } else if constexpr (PHYS == SH) {
                y_rows(inner_c, G->T.yb_v, G->T.yb, 2, lr0, ya, v);
                x_rows(cxb, 1, lr0, u);
            } else {
                y_rows(inner_c, PHYS == TMEM ? G->T.yf : G->T.yf_v, G->T.yf, 2, lr0, ya, v);
                x_rows(cxf, 2, lr0, u);
            }
            if (SELX ? xframe : xf) {
                cpml_x(0, u, PHYS != SH);
                if constexpr (PHYS == ELASTIC) cpml_x(1, a, false);
            }
            if (yframe) {
                cpml_y(0, v, PHYS != SH && PHYS != ELASTIC, ya - y0);
                if constexpr (PHYS == ELASTIC) cpml_y(1, c, true, ya - y0);
            }
            float n0[S], n1[S];
#pragma unroll
            for (int r = 0; r < S; r++) {
                const int o = lr0 + r * RW;
                n1[r] = 0.f;
                if constexpr (PHYS == ELASTIC) {
                    u[r] += v[r];
                    a[r] += c[r];
                    if constexpr (REC) {
                        rh[0][r] = u[r];
                        rh[1][r] = a[r];
                    }
                    n0[r] = add_scaled(sf[o], u[r], co[2][r]);
                    n1[r] = add_scaled(sf[FS + o], a[r], co[3][r]);
                } else if constexpr (PHYS == ACOUSTIC) {
                    n0[r] = add_scaled(sf[o], u[r], co[1][r]);
                    n1[r] = add_scaled(sf[FS + o], v[r], co[2][r]);
                } else if constexpr (PHYS == TMEM) {
                    n0[r] = add_scaled(sf[o], -v[r], co[3][r]);
                    n1[r] = add_scaled(sf[FS + o], u[r], co[2][r]);
                } else if constexpr (PHYS == SH) {
                    u[r] += v[r];
                    n0[r] = add_scaled(sf[o], u[r], co[0][r]);
                }
            }
#pragma unroll
            for (int r = 0; r < S; r++)
                if (xin && ya + r < NY) {
                    sf[lr0 + r * RW] = n0[r];
                    if (PHYS != SH) sf[FS + lr0 + r * RW] = n1[r];
                }
        };
        auto stress_rows = [&](auto inner_c, float (&rh)[REC ? 3 : 1][S]) {
            const res_args G = fresh_args(G0);
            const int wave = fresh_uniform(wave_), ya = y0 + wave * S;
            const int lr0 = (wave * S + H) * RW + H + fresh_lane(lane);
            float u[S], v[S], a[S], c[S];
            if constexpr (PHYS == ELASTIC) {
                y_rows(inner_c, G->T.yb, G->T.yb, 1, lr0, ya, v);
                y_rows(inner_c, G->T.yf, G->T.yf, 0, lr0, ya, c);
                x_rows(cxb, 0, lr0, u);
                x_rows(cxf, 1, lr0, a);
            } else if constexpr (PHYS == SH) {
                y_rows(inner_c, G->T.yf, G->T.yf, 0, lr0, ya, v);
                x_rows(cxf, 0, lr0, u);
            } else {
                y_rows(inner_c, G->T.yb, G->T.yb, PHYS == ACOUSTIC ? 1 : 0, lr0, ya, v);
                x_rows(cxb, PHYS == ACOUSTIC ? 0 : 1, lr0, u);
            }
            if (SELX ? xframe : xf) {
                cpml_x(0, u, PHYS == SH);
                if constexpr (PHYS == ELASTIC) cpml_x(1, a, true);
            }
            if (yframe) {
                cpml_y(0, v, PHYS == SH, ya - y0);
                if constexpr (PHYS == ELASTIC) cpml_y(1, c, true, ya - y0);
            }
            float n0[S], n1[S], n2[S];
#pragma unroll
            for (int r = 0; r < S; r++) {
                const int o = lr0 + r * RW;
                n1[r] = n2[r] = 0.f;
                if constexpr (PHYS == ELASTIC) {
                    // u: Dx vx, v: Dy vy, a: Dx vy, c: Dy vx
                    float xx = sf[2 * FS + o], yy = sf[3 * FS + o], xy = sf[4 * FS + o];
                    el_normal(xx, yy, u[r], v[r], co[0][r], co[1][r]);
                    c[r] += a[r];
                    if constexpr (REC) {
                        rh[0][r] = u[r];
                        rh[1][r] = v[r];
                        rh[2][r] = c[r];
                    }
                    n0[r] = xx;
                    n1[r] = yy;
                    n2[r] = add_scaled(xy, c[r], co[4][r]);
                } else if constexpr (PHYS == ACOUSTIC) {
                    u[r] += v[r];
                    n0[r] = add_scaled(sf[2 * FS + o], u[r], co[0][r]);
                } else if constexpr (PHYS == TMEM) {
                    u[r] -= v[r];
                    n0[r] = tm_ez(co[0][r], sf[2 * FS + o], co[1][r], u[r]);
                } else if constexpr (PHYS == SH) {
                    n0[r] = add_scaled(sf[FS + o], u[r], co[1][r]);
                    n1[r] = add_scaled(sf[2 * FS + o], v[r], co[2][r]);
                }
            }
            if (PHYS != SH && fs && ya == 0 && xin) {
                if constexpr (PHYS == ELASTIC)
                    el_surface(n0[0], n1[0], u[0], v[0], ((const RES_GLOBAL float *)G->C.fsH)[x],
                               ((const RES_GLOBAL float *)G->C.fsV)[x]);
            }
            if (abs) {
#pragma unroll
                for (int r = 0; r < S; r++) {
                    n0[r] *= px[r];
                    n1[r] *= px[r];
                    n2[r] *= px[r];
                }
            }
            if (PHYS == ACOUSTIC && fs && ya == 0) n0[0] *= 0.f;
            constexpr int F0 = PHYS == SH ? 1 : 2;
#pragma unroll
            for (int r = 0; r < S; r++)
                if (xin && ya + r < NY) {
                    const int o = lr0 + r * RW;
                    sf[F0 * FS + o] = n0[r];
                    if (PHYS == ELASTIC || PHYS == SH) sf[(F0 + 1) * FS + o] = n1[r];
                    if (PHYS == ELASTIC) sf[(F0 + 2) * FS + o] = n2[r];
                }
        };
        using c0 = std::integral_constant<int, 0>;
        using c1 = std::integral_constant<int, 1>;
        // the adjoint's record of a phase's sums
        auto keep = [&](auto first, int tt, const auto &rh) {
            constexpr int F0 = decltype(first)::value, N = F0 ? 3 : 2;
            const int lane = fresh_lane(tid & 63), ya = y0 + fresh_uniform(wave_) * S;
            record_strips<S, N>(KA.R, KA.L, KA.X.nshots, tt, F0, shot, x0, ya, lane, rh);
        };

        load_psi(0);
        __syncthreads();
        for (int st = 0; st < KA.X.nsteps; st++, tag++) {
            const int tt = KA.X.t0 + st;
            {
                float rh[REC ? 2 : 1][S];
                if (inner)
                    velocity_rows(std::true_type{}, rh);
                else
                    velocity_rows(std::false_type{}, rh);
                block_sync_lds();
                send(c0{});
                store_psi(0);
                load_psi(1);
                if constexpr (REC) keep(c0{}, tt, rh);
            }
            recv(c0{});
            block_sync_lds();
            if (s_bad) {
                bad = true;
                break;
            }
            {
                float rh[REC ? 3 : 1][S];
                if (inner)
                    stress_rows(std::true_type{}, rh);
                else
                    stress_rows(std::false_type{}, rh);
                block_sync_lds();
                // ABS of the velocity-type fields, after the stress-type update has read them
                if (abs) {
                    const int lr0 = (fresh_uniform(wave_) * S + H) * RW + H + fresh_lane(tid & 63);
#pragma unroll
                    for (int r = 0; r < S; r++)
                        if (ya + r < NY && xin) {
                            sf[lr0 + r * RW] *= px[r];
                            if (PHYS != SH) sf[FS + lr0 + r * RW] *= px[r];
                        }
                    if (ns == 0) block_sync_lds();
                }
                if (ns > 0) {
                    block_sync_lds();
                    if (wave == 0) {
                        const res_args G = fresh_args(G0);
                        // in list order
                        for (int e0 = 0; e0 < ns; e0 += 64) {
                            if (e0 && e0 + lane < ns) sv = signal(G, source(G, e0 + lane, so1, so2), tt);
                            for (int e = 0; e < min(64, ns - e0); e++) {
                                if (lane == e) {
                                    sf[so1] += sv;
                                    if (so2 >= 0) sf[so2] += sv;
                                }
                                wave_sync();
                            }
                        }
                        if (ns > 64) sid = source(G, lane, so1, so2);
                        if (lane < ns && tt + 1 < G->A.NT) sv = signal(G, sid, tt + 1);
                    }
                    block_sync_lds();
                }
                send(c1{});
                store_psi(1);
                load_psi(0);
                if (tid < nr) record_sample(fresh_args(G0), rid, tt, ro1, ro2);
                for (int e = tid + nthr; e < nr; e += nthr) {
                    const res_args G = fresh_args(G0);
                    int o1, o2;
                    const int id = receiver(G, e, o1, o2);
                    record_sample(G, id, tt, o1, o2);
                }
                if constexpr (REC) keep(std::integral_constant<int, 2>{}, tt, rh);
            }
            recv(c1{});
            block_sync_lds();
            if (s_bad) {
                bad = true;
                break;
            }
        }
        if (bad) {
            if (tid == 0) {
                __hip_atomic_store(KA.X.ctl + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(KA.X.host + 1, (unsigned long long)KA.X.launch, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
            }
            return;
        }
        // the state goes back to memory
#pragma unroll 1
        for (int row = wave; row < R; row += nwv)
#pragma unroll 1
            for (int f = 0; f < NF; f++)
                if (y0 + row < NY && xin)
                    (KA.F.f[f] + so + KA.L.at(x0, y0 + row))[lane] = sf[f * FS + (row + H) * RW + H + lane];
        psi_move(shot, false);
        __syncthreads();  // before the next shot's fields overwrite the tile
    }
}

}  // namespace
}  // namespace wv
