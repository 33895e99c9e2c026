// Host side of the resident 2D time loop: launch plan, acquisition lists, exchange buffer, the
// hand-shake with a launch.
#include <algorithm>
#include <chrono>
#include <mutex>

#include "handle.hpp"
#include "resident2d.hpp"

namespace wv {

hipError_t res2d_el(int order, bool rec, const void *go);
hipError_t res2d_ac(int order, bool rec, const void *go);
hipError_t res2d_tm(int order, bool rec, const void *go);
hipError_t res2d_sh(int order, bool rec, const void *go);

namespace {

hipError_t res_dispatch(int physics, int order, bool rec, const ResGo &g)
{
    switch (physics) {
    case ELASTIC: return res2d_el(order, rec, &g);
    case ACOUSTIC: return res2d_ac(order, rec, &g);
    case TMEM: return res2d_tm(order, rec, &g);
    case SH: return res2d_sh(order, rec, &g);
    default: return hipErrorInvalidValue;
    }
}

size_t res_lds(int physics, int H, int rows)
{
    const int nf = physics == ELASTIC ? 5 : 3;
    return sizeof(float) * ((size_t)nf * (rows + 2 * H) * (TILE_X + 2 * H) + 4ull * rows);
}

}  // namespace

size_t res2d_words(int physics, int H, int rows, int *phase1)
{
    const int n = physics == ELASTIC ? 2 : 1, rpg = TILE_X / H;
    const int items = 2 * n * ((rows + rpg - 1) / rpg) + 2 * n * H;
    *phase1 = items * 64;
    return (size_t)2 * items * 64;
}

static int wv_cu_count()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    return cus;
}

// Blocks of a plan that the device holds at once (0: the plan does not launch there).
static int res_capacity(int physics, int order, const Res2DPlan &p, bool rec)
{
    int cap = 0;
    ResGo g{};
    g.plan = &p;
    g.capacity = &cap;
    g.lds = res_lds(physics, order / 2, p.srow * p.wmax);
    if (res_dispatch(physics, order, rec, g) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    // a block whose wavefronts do not spread evenly over the four SIMDs of a CU may find no place beside
    // another one although registers and LDS would do in sum: count one block per CU then
    const int cus = wv_cu_count();
    if (p.nwv % 4) cap = std::min(cap, cus);
    // Two things the estimate does not know. A block is given LDS in units of 1280 bytes (five blocks of
    // 32,440 bytes do not fit 160 KB); and a SIMD takes six wavefronts of these kernels, whose scalar
    // registers are all in use, where it says seven (1792 blocks of four wavefronts, 1536 come in).
    const size_t lds = (g.lds + 16 + 1279) / 1280 * 1280;
    return std::min(cap, cus * std::min((int)(160 * 1024 / lds), std::max(1, 6 / ((p.nwv + 3) / 4))));
}

// Estimated us per time step of the whole batch: rounds x (exchange, barriers and latency of a step +
// the arithmetic of the rows a CU holds).  Measured (MI355X, order 8; us per round): elastic 64 rows
// per CU 11.9 (one block of 16 x 4 rows; 10.9 since, which leaves the choices as they are) and 12.4 (two of
// 8 x 4), 16 rows 5.7; TM-EM 64 rows 6.4 - 6.7; SH 64 rows 6.0, 128 rows 10.4; acoustic order 4: 4 rows 3.5,
// 64 rows 4.7.
static double res_step_us(int physics, int order, const Res2DPlan &p, int nshots)
{
    const int rounds = (nshots + p.conc - 1) / p.conc, cus = std::max(1, wv_cu_count());
    const double rows = (double)p.rows() * ((p.blocks() + cus - 1) / cus);
    const double per_row = (physics == ELASTIC ? 0.13 : 0.052) * (order + 4) / 12.0;
    return rounds * (3.3 + 0.1 * p.srow + per_row * rows * (p.srow == 8 ? 1.2 : 1.0));
}

// The same of the two-launch kernels: launch gaps and one memory round trip per phase, then their
// traffic.  Measured (us): elastic 1e6 cells 21.8, 1.44e6 31.4, 8e6 107; TM-EM 5.1e6 46, 2.05e7 195;
// SH 0.94e6 15.8; acoustic 4e4 7.5 - 10.5.
static double two_launch_us(int physics, double cells)
{
    return 7.0 + cells * (physics == ELASTIC ? 1.3e-5 : 9.1e-6);
}

Res2DPlan res2d_plan(int physics, int order, const Layout2D &L, int nshots, int srow, int nwv, bool rec, double *gain)
{
    Res2DPlan best;
    *gain = 0.0;
    if (physics != ELASTIC && physics != ACOUSTIC && physics != TMEM && physics != SH) return best;
    const int H = order / 2;
    double best_t = 1e30;
    static const int variants[5][2] = {{1, 16}, {2, 16}, {4, 16}, {4, 8}, {8, 8}};
    for (auto &va : variants) {
        const int S = va[0], wmax = va[1];
        if (srow && S != srow) continue;
        if (res_lds(physics, H, S * wmax) + 1024 > 160 * 1024) continue;
        int cap[17] = {};
        for (int w = 1; w <= wmax; w++) {
            if (nwv && w != nwv) continue;
            Res2DPlan p;
            p.nwv = w;
            p.srow = S;
            p.wmax = wmax;
            const int R = p.rows();
            if (R < H) continue;  // a halo reaches into the next tile only
            p.nbx = (L.NX + TILE_X - 1) / TILE_X;
            p.nby = (L.NY + R - 1) / R;
            p.conc = 1;
            const long long per = (long long)p.nbx * p.nby;
            if (per > 4096) continue;
            cap[w] = res_capacity(physics, order, p, rec);
            if (per > cap[w]) continue;
            const int most = cap[w] / (int)per, rounds = (nshots + most - 1) / most;
            p.conc = (nshots + rounds - 1) / rounds;
            const double t = res_step_us(physics, order, p, nshots);
            if (t < best_t) {
                best_t = t;
                best = p;
            }
        }
    }
    if (best) *gain = two_launch_us(physics, (double)L.NX * L.NY * nshots) / best_t;
    return best;
}

hipError_t launch_res2d(int physics, int order, const Res2DPlan &plan, const Layout2D &L, const Fields2D &F,
                        const Coef2D &C, const Taps &T, const Cpml2D &P, const Acq &A, const Res2DArgs &X,
                        const Rec2D *rec, hipStream_t stream)
{
    ResGo g{};
    g.plan = &plan;
    g.L = &L;
    g.F = &F;
    g.C = &C;
    g.T = &T;
    g.P = &P;
    g.A = &A;
    g.X = &X;
    g.rec = rec ? *rec : Rec2D{};
    g.st = stream;
    g.lds = res_lds(physics, order / 2, plan.srow * plan.wmax);
    return res_dispatch(physics, order, rec != nullptr, g);
}

}  // namespace wv

// A launch and the steps it stands for.
struct Res2DQueued {
    int t0, nsteps;
    unsigned launch;
};

struct Res2DState {
    wv::Res2DPlan plan;
    double gain = 0.0;  // estimated step time of the two-launch kernels over that of the plan
    bool planned = false, lists = false;
    int srow = 0;
    int want_rows = 0, want_waves = 0;  // wv_resident_plan
    std::vector<void *> allocs;      // exchange buffer, control words
    std::vector<void *> acq_allocs;  // lists of the plan's tiles
    int *bsrc_ptr = nullptr, *bsrc = nullptr, *brec_ptr = nullptr, *brec = nullptr;
    unsigned long long *xch = nullptr;
    unsigned *ctl = nullptr;
    float *psi = nullptr;
    unsigned long long *host = nullptr;  // pinned, one for the handle's life: see Res2DArgs
    int words = 0, phase1 = 0;  // exchange words of a block
    unsigned tag = 1, arrived = 0;
    unsigned launches = 0;  // made in the handle's life
    unsigned first = 1;     // the first one since the last wv_reset
    bool off = false;       // the ordinary kernels run the steps until the next wv_reset
    int refused = 0;        // check-ins refused in a row
    std::vector<Res2DQueued> queued;  // launches not known to have gone, in order
    std::mutex lock;                  // of `queued`: results may be read from several threads
    hipEvent_t ev[2] = {};  // per-kernel timing
    bool timed = false;     // the timed run calls went through the resident loop
};

void res2d_destroy(wv_solver *s)
{
    if (!s->res) return;
    s->free_list(s->res->acq_allocs);
    s->free_list(s->res->allocs);
    if (s->res->host) (void)hipHostFree(s->res->host);
    for (hipEvent_t e : s->res->ev)
        if (e) (void)hipEventDestroy(e);
    delete s->res;
    s->res = nullptr;
}

void res2d_acquisition_changed(wv_solver *s)
{
    if (!s->res) return;
    s->free_list(s->res->acq_allocs);
    s->res->lists = false;
}

bool res2d_eligible(const wv_solver *s)
{
    if (s->dim != 2 || s->plain || s->visco) return false;
    if (s->physics != wv::ELASTIC && s->physics != wv::ACOUSTIC && s->physics != wv::TMEM && s->physics != wv::SH)
        return false;
    return s->cfg.tile_y == 0 && (s->cfg.path == WV_PATH_FUSED || (s->cfg.path == WV_PATH_STRIP && s->physics == wv::ELASTIC));
}

// What is known of the queued launches: 0 some verdict is not in (launches that went are taken off), 1 all
// went, 2 some were refused.
static int res_verdicts(Res2DState *r)
{
    std::vector<Res2DQueued> &q = r->queued;
    if (q.empty()) return 1;
    const unsigned long long w = __atomic_load_n(r->host, __ATOMIC_ACQUIRE);
    const unsigned first = (unsigned)(w >> 32), v = (unsigned)w;
    if (v & 1) {
        // (a refusal from before the latest wv_reset concerns none of these)
        if ((int)(first - q.front().launch) >= 0 && v == 2 * q.back().launch + 1) return 2;
        return 0;
    }
    size_t n = 0;
    while (n < q.size() && (int)(v - 2 * q[n].launch) >= 0) n++;
    if (n) r->refused = 0;
    q.erase(q.begin(), q.begin() + n);
    return q.empty() ? 1 : 0;
}

// Waits for the verdicts. 0: all queued launches went; 1: some were refused, and *redo has them in order
// (the loop is off then); < 0: error.
static int res_settle(wv_solver *s, std::vector<Res2DQueued> *redo)
{
    Res2DState *r = s->res;
    int v = res_verdicts(r);
    if (v == 0) {
        HIP_TRY(hipStreamSynchronize(s->st));
        v = res_verdicts(r);
    }
    if (v == 1) return 0;
    std::vector<Res2DQueued> q;
    q.swap(r->queued);
    if (v == 0) return fail(WV_EDEVICE, "the resident time loop ended without a verdict");
    const unsigned first = (unsigned)(__atomic_load_n(r->host, __ATOMIC_ACQUIRE) >> 32);
    for (const Res2DQueued &e : q)
        if ((int)(e.launch - first) >= 0) redo->push_back(e);
    // something else holds the GPU
    r->off = true;
    r->refused++;
    return 1;
}

// The steps of refused launches, with the ordinary kernels, and the checkpoints between them.
static int res_redo(wv_solver *s, const std::vector<Res2DQueued> &q)
{
    for (const Res2DQueued &e : q) {
        int rc = adjoint_checkpoint_again(s, e.t0);
        if (rc) return rc;
        wv::launch_set(s->d_tbase, e.t0, s->st);
        if ((rc = s->enqueue_steps(e.nsteps, false))) return rc;
    }
    return 0;
}

int res2d_settle(wv_solver *s)
{
    if (!s->res) return 0;
    std::lock_guard<std::mutex> hold(s->res->lock);
    std::vector<Res2DQueued> redo;
    int rc = res_settle(s, &redo);
    if (rc == 1 && (rc = res_redo(s, redo)) == 0) {
        HIP_TRY(hipEventRecord(s->ev1, s->st));
        return 1;
    }
    return rc;
}

int res2d_went(wv_solver *s)
{
    if (!s->res) return 0;
    std::lock_guard<std::mutex> hold(s->res->lock);
    std::vector<Res2DQueued> refused;
    return res_settle(s, &refused);
}

bool res2d_queued(wv_solver *s)
{
    if (!s->res) return false;
    std::lock_guard<std::mutex> hold(s->res->lock);
    // (a launch on an idle stream begins within tens of microseconds)
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    int v;
    while ((v = res_verdicts(s->res)) == 0 && std::chrono::steady_clock::now() < until) {
    }
    return v == 0;
}

// The plan for the handle (rows per wavefront as the record's strips when it is written); false:
// the resident loop does not take this problem.
static bool res_plan(wv_solver *s, int srow)
{
    if (!s->res) s->res = new Res2DState();
    Res2DState *r = s->res;
    if (r->off) return false;
    if (r->planned && r->srow == srow) return (bool)r->plan;
    // the queued launches use the buffers of the plan that goes (refused ones: the caller finds the loop
    // off, and settles before it runs anything)
    {
        std::lock_guard<std::mutex> hold(r->lock);
        if (!r->queued.empty() && (hipStreamSynchronize(s->st) != hipSuccess || res_verdicts(r) != 1)) return false;
    }
    s->free_list(r->acq_allocs);
    s->free_list(r->allocs);
    r->lists = false;
    r->plan = wv::res2d_plan(s->physics, s->cfg.spatial_fd_order, s->L, s->cfg.nshots, srow ? srow : r->want_rows,
                             r->want_waves, srow != 0, &r->gain);
    r->planned = true;
    r->srow = srow;
    r->xch = nullptr;
    r->ctl = nullptr;
    r->tag = 1;
    r->arrived = 0;
    return (bool)r->plan;
}

// Floats of a plan's memory variables.
static size_t res_psi(const wv_solver *s, const wv::Res2DPlan &p)
{
    if (s->cfg.damping_boundary != 2) return 0;
    return (size_t)p.blocks() * p.nwv * 4 * (s->physics == wv::ELASTIC ? 2 : 1) * p.srow * wv::TILE_X;
}

// Device bytes that runs of the handle with that many rows per wavefront (0: the planner's choice) will
// want for the loop, for memory plans that divide what is free.
size_t res2d_bytes(wv_solver *s, int srow)
{
    if (!res2d_eligible(s)) return 0;
    double gain = 0.0;
    const wv::Res2DPlan p = wv::res2d_plan(s->physics, s->cfg.spatial_fd_order, s->L, s->cfg.nshots, srow, 0, srow != 0, &gain);
    if (!p) return 0;
    int phase1 = 0;
    size_t n = wv::res2d_words(s->physics, s->H, p.rows(), &phase1) * p.blocks() * sizeof(unsigned long long);
    n += res_psi(s, p) * sizeof(float);
    size_t ids = 2 * (size_t)s->cfg.nshots * p.nby * p.nbx + 2;
    for (const ShotAcq &a : s->shots) ids += a.sidx.size() + a.ridx.size();
    return n + ids * sizeof(int);
}

// The plan's exchange buffer, control words, memory variables and report words: all of them or none.
// False: a handle whose device memory is used up keeps the ordinary kernels, which need none of these.
static bool res_buffers(wv_solver *s)
{
    Res2DState *r = s->res;
    if (r->xch) return true;
    const wv::Res2DPlan &p = r->plan;
    int phase1 = 0;
    const size_t words = wv::res2d_words(s->physics, s->H, p.rows(), &phase1);
    const size_t npsi = res_psi(s, p);
    std::vector<void *> got;
    unsigned long long *xch = nullptr;
    unsigned *ctl = nullptr;
    float *psi = nullptr;
    unsigned long long *host = nullptr;
    if (s->dalloc(&xch, words * p.blocks(), got) || s->dalloc(&ctl, 4, got) ||
        (npsi && s->dalloc(&psi, npsi, got)) ||
        (!r->host && hipHostMalloc((void **)&host, 64, hipHostMallocDefault) != hipSuccess)) {
        (void)hipGetLastError();
        s->free_list(got);
        return false;
    }
    if (host) {
        host[0] = host[1] = 0;
        r->host = host;
    }
    r->allocs = got;
    r->words = (int)words;
    r->phase1 = phase1;
    r->ctl = ctl;
    r->psi = psi;
    r->xch = xch;
    return true;
}

// The acquisition per (shot, tile of the plan): all four lists or none.
static bool res_lists(wv_solver *s)
{
    Res2DState *r = s->res;
    if (r->lists) return true;
    const wv::Res2DPlan &p = r->plan;
    const int R = p.rows();
    const size_t nsb = (size_t)s->cfg.nshots * p.nby * p.nbx;
    std::vector<std::vector<int>> bs(nsb), br(nsb);
    int gs = 0, gr = 0;
    for (int sh = 0; sh < s->cfg.nshots; sh++) {
        auto blk = [&](long long g) {
            const int x = (int)(g % s->L.NX), y = (int)(g / s->L.NX);
            return ((size_t)sh * p.nby + y / R) * p.nbx + x / wv::TILE_X;
        };
        for (long long g : s->shots[sh].sidx) bs[blk(g)].push_back(gs++);
        for (long long g : s->shots[sh].ridx) br[blk(g)].push_back(gr++);
    }
    std::vector<int> bsp(1, 0), bsl, brp(1, 0), brl;
    for (size_t b = 0; b < nsb; b++) {
        bsl.insert(bsl.end(), bs[b].begin(), bs[b].end());
        bsp.push_back((int)bsl.size());
        brl.insert(brl.end(), br[b].begin(), br[b].end());
        brp.push_back((int)brl.size());
    }
    std::vector<void *> got;
    int *q[4] = {};
    if (s->upload(&q[0], bsp, got) || s->upload(&q[1], bsl, got) || s->upload(&q[2], brp, got) ||
        s->upload(&q[3], brl, got)) {
        (void)hipGetLastError();
        s->free_list(got);
        return false;
    }
    r->acq_allocs = got;
    r->bsrc_ptr = q[0];
    r->bsrc = q[1];
    r->brec_ptr = q[2];
    r->brec = q[3];
    r->lists = true;
    return true;
}

// nsteps steps from t0 in one launch.  0: enqueued (timed: done); 1: not (the caller settles and runs the steps
// with the ordinary kernels); < 0: error.
int res2d_run(wv_solver *s, int t0, int nsteps, const wv::Rec2D *rec)
{
    if (!res_plan(s, rec ? s->tile_y / 4 : 0)) return 1;
    Res2DState *r = s->res;
    const wv::Res2DPlan &p = r->plan;
    if (!res_buffers(s) || !res_lists(s)) {
        // no memory
        s->free_list(r->allocs);
        r->xch = nullptr;
        r->planned = false;
        r->off = true;
        return 1;
    }
    wv::Res2DArgs X{};
    X.nwv = p.nwv;
    X.nbx = p.nbx;
    X.nby = p.nby;
    X.conc = p.conc;
    X.nshots = s->cfg.nshots;
    X.t0 = t0;
    X.nsteps = nsteps;
    X.words = r->words;
    X.phase1 = r->phase1;
    X.xch = r->xch;
    X.tag0 = r->tag;
    X.ctl = r->ctl;
    X.launch = ++r->launches;
    r->arrived += (unsigned)p.blocks();
    X.arrive = r->arrived;
    X.host = r->host;
    X.bsrc_ptr = r->bsrc_ptr;
    X.bsrc = r->bsrc;
    X.brec_ptr = r->brec_ptr;
    X.brec = r->brec;
    X.psi = r->psi;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (s->ktiming) {
        for (auto &ev : r->ev)
            if (!ev) HIP_TRY(hipEventCreate(&ev));
        e0 = r->ev[0];
        e1 = r->ev[1];
        HIP_TRY(hipEventRecord(e0, s->st));
    }
    const hipError_t e = wv::launch_res2d(s->physics, s->cfg.spatial_fd_order, p, s->L, s->fields2d(s->cur), s->coef2d(),
                                          s->taps(), s->cpml2d(s->cur), s->acq(), X, rec, s->st);
    if (e != hipSuccess) {
        // nothing ran: leave the counters as the device has them
        r->launches--;
        r->arrived -= (unsigned)p.blocks();
        (void)hipGetLastError();
        return 1;
    }
    const int rounds = (s->cfg.nshots + p.conc - 1) / p.conc;
    r->tag += (unsigned)(rounds * nsteps);
    {
        std::lock_guard<std::mutex> hold(r->lock);
        (void)res_verdicts(r);
        r->queued.push_back({t0, nsteps, X.launch});
    }
    if (!e0) return 0;
    HIP_TRY(hipEventRecord(e1, s->st));
    HIP_TRY(hipEventSynchronize(e1));
    if (const int rc = res2d_went(s)) return rc;
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    s->kms[0] += ms;
    s->klaunch[0] += nsteps;  // counted per time step
    r->timed = true;
    return 0;
}

// Whether the planner expects the resident loop to be the faster one for the handle's run calls.
bool res2d_expected(wv_solver *s, bool rec)
{
    return res_plan(s, rec ? s->tile_y / 4 : 0) && (s->res->want_rows || s->res->want_waves || s->res->gain > 1.05);
}

// A wait inside a resident launch ran out: the state is not valid until wv_reset. (Every call that would go
// on from the state or hand it out asks here first. The report names the launch, so it outlives the buffers
// of a plan, and one from before the reset does not count.)
bool res2d_failed(const wv_solver *s)
{
    if (!s->res || !s->res->host) return false;
    const unsigned launch = (unsigned)__atomic_load_n(s->res->host + 1, __ATOMIC_ACQUIRE);
    return launch && (int)(launch - s->res->first) >= 0;
}

// wv_reset: what went wrong before does not matter any more, in stream order. The loop is tried again after
// a refused check-in (one other kernel may have been the cause, and a refusal costs 0.3 s), but not after
// three of them in a row.
int res2d_reset(wv_solver *s)
{
    Res2DState *r = s->res;
    if (!r) return 0;
    std::lock_guard<std::mutex> hold(r->lock);
    (void)res_verdicts(r);
    r->queued.clear();
    r->first = r->launches + 1;
    if (r->refused < 3) r->off = false;
    if (r->xch) HIP_TRY(hipMemsetAsync(r->ctl + 2, 0, 2 * sizeof(unsigned), s->st));
    return 0;
}

// Bytes that a step of the whole batch moves outside the CUs: halo words (8 bytes, written and read, H deep on
// both sides of every edge between tiles), CPML memory variables (read and written), ABS factors, samples.
// The load and the store of the state at the ends of a run call are not in it.
double res2d_step_bytes(const wv_solver *s)
{
    if (!s->res || !s->res->plan) return 0.0;
    const wv::Res2DPlan &p = s->res->plan;
    const double B = s->cfg.nshots, nf = s->physics == wv::ELASTIC ? 2 : 1, W = s->cfg.boundary_width;
    double bytes = B * 2 * 8 * 2 * nf * 2 * s->H * ((p.nbx - 1.0) * s->cfg.NY + (p.nby - 1.0) * s->cfg.NX);
    if (s->cfg.damping_boundary == 2)
        bytes += B * 8 * 2 * nf * (2 * W * s->cfg.NY + (s->cfg.free_surface ? W : 2 * W) * s->cfg.NX);
    if (s->cfg.damping_boundary == 1) bytes += B * 4 * (double)s->cfg.NX * s->cfg.NY;
    double samples = s->rec_total;
    for (const ShotAcq &a : s->shots) samples += a.sidx.size();
    return bytes + 4 * samples;
}

bool res2d_timed(const wv_solver *s) { return s->res && s->res->timed; }
void res2d_timing_reset(wv_solver *s)
{
    if (s->res) s->res->timed = false;
}

extern "C" int wv_resident_plan(wv_solver *s, int rows, int waves, int *plan)
{
    if (!s || !s->inited) return fail(WV_ESTATE, "not initialised");
    if (!res2d_eligible(s)) return fail(WV_EINVAL, "the resident loop does not take the runs of this handle");
    if ((rows != 0 && rows != 1 && rows != 2 && rows != 4 && rows != 8) || waves < 0 || waves > 16)
        return fail(WV_EINVAL, "rows per wavefront must be 0, 1, 2, 4 or 8, wavefronts 0 to 16");
    if (const int rc = res2d_settle(s); rc < 0) return rc;
    if (!s->res) s->res = new Res2DState();
    Res2DState *r = s->res;
    const int was[2] = {r->want_rows, r->want_waves};
    r->want_rows = rows;
    r->want_waves = waves;
    r->planned = false;
    if (!res_plan(s, 0)) {
        r->want_rows = was[0];
        r->want_waves = was[1];
        r->planned = false;
        return fail(WV_EINVAL, "no such plan of the resident loop fits");
    }
    if (plan) {
        plan[0] = r->plan.srow;
        plan[1] = r->plan.nwv;
        plan[2] = r->plan.conc;
    }
    return WV_OK;
}
