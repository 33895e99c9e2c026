// The resident loop's host side (resident2d.cpp) and the read-backs' staging (readback.hpp) over a stand-in for the HIP runtime: memory comes from
// malloc and can be made to run out at a chosen allocation; launches and copies go to a stream that works
// when it is waited for, or told to, and notes what was run.
//   resident_host <test>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <set>
#include <string>
#include <vector>

#include "handle.hpp"
#include "resident2d.hpp"

#define CHECK(c)                                                                \
    do {                                                                        \
        if (!(c)) {                                                             \
            std::fprintf(stderr, "line %d: not true: %s\n", __LINE__, #c);      \
            std::exit(1);                                                       \
        }                                                                       \
    } while (0)

namespace {

std::set<void *> live;
size_t live_bytes = 0;
int allocations = 0, fail_at = 0;  // the fail_at-th allocation finds no memory (0: none)
size_t device_left = ~(size_t)0;   // largest device allocation that is still to be had
int launches = 0, copies = 0;
bool refuse = false;  // not all blocks of a launch come in
bool give_up = false;  // a launch's wait runs out
wv::Res2DArgs last;    // arguments of the last launch
std::string last_error;

hipError_t give(void **p, size_t n)
{
    if (++allocations == fail_at) return hipErrorOutOfMemory;
    *p = std::calloc(1, n ? n : 1);
    live.insert(*p);
    live_bytes += n;
    return hipSuccess;
}
hipError_t take(void *p)
{
    CHECK(!p || live.erase(p) == 1);
    std::free(p);
    return hipSuccess;
}

// The stream: what is queued, and a note of what was run ("R" resident, "O" ordinary steps, "C" a checkpoint).
std::vector<std::function<void()>> stream;
std::string ran;
void work(size_t n)
{
    for (size_t k = 0; k < n && k < stream.size(); k++) stream[k]();
    stream.erase(stream.begin(), stream.begin() + std::min(n, stream.size()));
}
void note(const char *what, int t0, int n)
{
    ran += std::string(what) + std::to_string(t0) + (n ? "+" + std::to_string(n) : "") + " ";
}
std::string take_notes()
{
    std::string s;
    s.swap(ran);
    return s;
}

hipError_t launch(const wv::ResGo &g)
{
    if (g.capacity) {
        *g.capacity = 256;
        return hipSuccess;
    }
    const wv::Res2DArgs X = *g.X;
    CHECK(X.xch && X.ctl && X.host && X.bsrc_ptr && X.bsrc && X.brec_ptr && X.brec);
    CHECK(X.psi || !g.P->on);
    launches++;
    last = X;
    // the check-in of resident2d_kernel.hpp, all blocks at once
    stream.push_back([X] {
        CHECK(live.count(X.ctl) && live.count(X.xch) && live.count((void *)X.brec));
        X.ctl[0] += X.nbx * X.nby * X.conc;
        CHECK(X.ctl[0] == X.arrive);
        const unsigned behind = X.ctl[3];
        const bool stop = behind || refuse;
        if (stop) X.ctl[3] = behind ? behind : X.launch;
        X.host[0] = stop ? ((unsigned long long)X.ctl[3] << 32) | (2 * X.launch + 1) : 2 * X.launch;
        if (stop) return;
        note("R", X.t0, X.nsteps);
        if (give_up) {
            X.ctl[2] = 1;
            X.host[1] = X.launch;
        }
    });
    return hipSuccess;
}

}  // namespace

int wv_fail(int code, const std::string &msg)
{
    last_error = msg;
    return code;
}
wv_solver::~wv_solver()
{
    (void)hipStreamSynchronize(nullptr);
    res2d_destroy(this);
    free_list(allocs);
}

int step_base = 0;
int wv_solver::enqueue_steps(int n, bool)
{
    const int t0 = step_base;
    stream.push_back([t0, n] { note("O", t0, n); });
    return 0;
}
int adjoint_checkpoint_again(wv_solver *, int t)
{
    stream.push_back([t] { note("C", t, 0); });
    return 0;
}

namespace wv {
void launch_set(int *, int v, hipStream_t) { step_base = v; }
hipError_t res2d_el(int, bool, const void *go) { return launch(*(const ResGo *)go); }
hipError_t res2d_ac(int, bool, const void *go) { return launch(*(const ResGo *)go); }
hipError_t res2d_tm(int, bool, const void *go) { return launch(*(const ResGo *)go); }
hipError_t res2d_sh(int, bool, const void *go) { return launch(*(const ResGo *)go); }
}  // namespace wv

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return n > device_left ? hipErrorOutOfMemory : give(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return give(p, n); }
hipError_t hipFree(void *p)
{
    work(stream.size());  // (hipFree waits for the device)
    return take(p);
}
hipError_t hipHostFree(void *p) { return take(p); }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t)
{
    stream.push_back([p, v, n] { std::memset(p, v, n); });
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    copies++;
    work(stream.size());  // (pageable memory)
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    work(stream.size());
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    static char event;
    *e = (hipEvent_t)&event;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
}

namespace {

void make(wv_solver &s)
{
    s.physics = wv::ELASTIC;
    s.cfg.NX = s.L.NX = 200;
    s.cfg.NY = s.L.NY = 150;
    s.cfg.NZ = 1;
    s.cfg.NT = 1000;
    s.cfg.spatial_fd_order = 8;
    s.H = 4;
    s.cfg.damping_boundary = 2;
    s.cfg.nshots = 2;
    s.variant = V_STRIP;
    s.tile_y = 16;
    s.inited = s.model_ok = true;
    s.shots.resize(2);
    for (ShotAcq &a : s.shots) {
        a.sidx = {75 * 200 + 100};
        a.ridx = {10 * 200 + 30, 140 * 200 + 190};
    }
}

// Whichever allocation fails, nothing is kept of the others, no launch is made with a part of the buffers,
// and the caller is told to run the steps with the ordinary kernels, now and the next time.
void no_memory()
{
    int total = 0;
    {
        wv_solver s;
        make(s);
        CHECK(res2d_run(&s, 0, 100) == 0 && launches == 1);
        total = allocations;
    }
    CHECK(live.empty());
    CHECK(total == 8);  // exchange words, control words, memory variables, report words, four lists
    for (int k = 1; k <= total; k++) {
        allocations = launches = 0;
        fail_at = k;
        {
            wv_solver s;
            make(s);
            CHECK(res2d_run(&s, 0, 100) == 1);
            CHECK(live.size() <= 1);  // (the report words stay with the handle)
            CHECK(res2d_run(&s, 100, 200) == 1);
            CHECK(launches == 0);
        }
        CHECK(live.empty());
    }
}

// A memory plan is told at least what the loop's buffers take, before they are there.
void memory_asked_for()
{
    for (int physics : {wv::ELASTIC, wv::ACOUSTIC, wv::TMEM, wv::SH})
        for (int damping = 0; damping < 3; damping++) {
            live_bytes = 0;
            wv_solver s;
            make(s);
            s.physics = physics;
            s.cfg.damping_boundary = damping;
            const size_t said = res2d_bytes(&s, 0);
            CHECK(live_bytes == 0);
            CHECK(res2d_run(&s, 0, 100) == 0);
            const size_t words = 64 + 4 * sizeof(unsigned);  // report and control words
            CHECK(said >= live_bytes - words && said <= live_bytes);
        }
    wv_solver s;
    make(s);
    s.visco = true;
    CHECK(res2d_bytes(&s, 0) == 0);
}

// Only a launch that ran is reported as the timed kernel.
void timing()
{
    wv_solver s;
    make(s);
    s.ktiming = true;
    refuse = true;
    CHECK(res2d_run(&s, 0, 100) == 1 && launches == 1);
    CHECK(!res2d_timed(&s) && s.klaunch[0] == 0 && take_notes().empty());
    refuse = false;
    wv_solver t;
    make(t);
    t.ktiming = true;
    CHECK(res2d_run(&t, 0, 100) == 0);
    CHECK(res2d_timed(&t) && t.klaunch[0] == 100);
    res2d_timing_reset(&t);
    CHECK(!res2d_timed(&t));
}

// 0 / 1: the steps went through the loop / the ordinary kernels
int run(wv_solver &s, int t0, int n, const wv::Rec2D *rec = nullptr)
{
    const int rc = res2d_run(&s, t0, n, rec);
    return rc ? rc : res2d_settle(&s);
}

// A wait that ran out is reported until wv_reset, through plans given up and made, and not afterwards.
void failure()
{
    wv_solver s;
    make(s);
    const wv::Rec2D rec{};
    CHECK(!res2d_failed(&s));
    CHECK(run(s, 0, 100) == 0 && !res2d_failed(&s));
    give_up = true;
    CHECK(run(s, 100, 100) == 0 && res2d_failed(&s));
    give_up = false;
    CHECK(run(s, 0, 100, &rec) == 0);  // another plan, another set of buffers
    CHECK(res2d_failed(&s));
    CHECK(run(s, 0, 100) == 0);
    CHECK(res2d_failed(&s));
    last.ctl[2] = 1;
    CHECK(res2d_reset(&s) == 0);
    CHECK(!res2d_failed(&s));
    CHECK(run(s, 0, 100) == 0 && !res2d_failed(&s) && last.ctl[2] == 0);
    // a launch from before the reset may still be at it
    give_up = true;
    CHECK(res2d_run(&s, 0, 100) == 0);
    CHECK(res2d_reset(&s) == 0);
    (void)hipStreamSynchronize(nullptr);
    CHECK(last.host[1] == last.launch && !res2d_failed(&s));
    CHECK(run(s, 0, 100) == 0 && res2d_failed(&s));
}

// A refused check-in leaves the steps to the ordinary kernels until wv_reset, three in a row for good.
void refusal()
{
    wv_solver s;
    make(s);
    const wv::Rec2D rec{};
    refuse = true;
    for (int k = 1; k <= 3; k++) {
        CHECK(run(s, 0, 100) == 1 && launches == k);
        CHECK(run(s, 100, 100) == 1 && run(s, 200, 100, &rec) == 1 && launches == k);
        CHECK(res2d_reset(&s) == 0);
    }
    CHECK(run(s, 0, 100) == 1 && launches == 3);
    wv_solver t;
    make(t);
    launches = 0;
    for (int k = 1; k <= 4; k++) {  // not in a row
        refuse = true;
        CHECK(run(t, 0, 100) == 1);
        CHECK(res2d_reset(&t) == 0);
        (void)hipStreamSynchronize(nullptr);
        refuse = false;
        CHECK(run(t, 0, 100) == 0 && launches == 2 * k);
    }
    // the same for want of memory
    wv_solver u;
    make(u);
    fail_at = allocations + 2;
    CHECK(run(u, 0, 100) == 1 && run(u, 0, 100) == 1);
    CHECK(res2d_reset(&u) == 0);
    CHECK(run(u, 0, 100) == 0);
}

// Launches are queued without waiting for any of them, on two handles in turn; the steps of a refused one
// and of all behind it are run with the ordinary kernels, in order and once, when the handle is settled.
void queue()
{
    wv_solver a, b;
    make(a);
    make(b);
    CHECK(run(a, 0, 1) == 0 && run(b, 0, 1) == 0);
    take_notes();
    for (int k = 0; k < 5; k++) CHECK(res2d_run(&a, 10 * k, 10) == 0 && res2d_run(&b, 7 * k, 7) == 0);
    CHECK(stream.size() == 10 && ran.empty());
    CHECK(res2d_queued(&a));
    work(9);
    CHECK(!res2d_queued(&a) && res2d_queued(&b));
    CHECK(res2d_settle(&a) == 0 && stream.size() == 1);  // nothing to wait for
    CHECK(res2d_settle(&b) == 0 && stream.empty());
    CHECK(take_notes() == "R0+10 R0+7 R10+10 R7+7 R20+10 R14+7 R30+10 R21+7 R40+10 R28+7 ");

    // the third of five is refused
    for (int k = 0; k < 5; k++) CHECK(res2d_run(&a, 10 * k, 10) == 0);
    work(2);
    refuse = true;
    work(1);
    refuse = false;
    CHECK(res2d_settle(&a) == 1);
    (void)hipStreamSynchronize(nullptr);
    CHECK(take_notes() == "R0+10 R10+10 C20 O20+10 C30 O30+10 C40 O40+10 ");
    CHECK(res2d_settle(&a) == 0 && res2d_run(&a, 50, 10) == 1);

    // wv_reset drops what is queued, refused or not
    CHECK(res2d_reset(&a) == 0);
    refuse = true;
    CHECK(res2d_run(&a, 0, 10) == 0 && res2d_run(&a, 10, 10) == 0);
    CHECK(res2d_reset(&a) == 0);
    work(3);
    refuse = false;
    CHECK(res2d_run(&a, 0, 10) == 0 && res2d_run(&a, 10, 10) == 0);
    CHECK(res2d_settle(&a) == 0 && take_notes() == "R0+10 R10+10 ");
    refuse = true;
    CHECK(res2d_run(&a, 0, 10) == 0 && res2d_went(&a) == 1 && stream.empty());
    CHECK(res2d_settle(&a) == 0 && take_notes().empty());
    refuse = false;

    // another plan while launches of the old one are queued
    const wv::Rec2D rec{};
    CHECK(res2d_reset(&a) == 0);
    CHECK(res2d_run(&a, 0, 10) == 0 && res2d_run(&a, 10, 10, &rec) == 0);
    CHECK(res2d_settle(&a) == 0 && take_notes() == "R0+10 R10+10 ");
    CHECK(res2d_run(&a, 20, 10, &rec) == 0);
    refuse = true;
    CHECK(res2d_run(&a, 30, 10) == 1 && res2d_settle(&a) == 1);
    (void)hipStreamSynchronize(nullptr);
    CHECK(take_notes() == "C20 O20+10 ");
}

// A division of the work asked for is taken, or refused without a trace.
void plan()
{
    wv_solver s;
    make(s);
    int p[3];
    CHECK(wv_resident_plan(&s, 0, 0, p) == WV_OK);
    const int free_choice[3] = {p[0], p[1], p[2]};
    for (int rows : {1, 2, 4, 8}) {
        CHECK(wv_resident_plan(&s, rows, 8, p) == WV_OK && p[0] == rows && p[1] == 8 && p[2] == 2);
        CHECK(res2d_expected(&s, false) && run(s, 0, 10) == 0 && last.nwv == 8);
    }
    CHECK(wv_resident_plan(&s, 8, 16, p) == WV_EINVAL);  // 8 rows: 8 wavefronts at most
    CHECK(wv_resident_plan(&s, 1, 3, p) == WV_EINVAL);   // lower than a halo
    CHECK(wv_resident_plan(&s, 3, 0, p) == WV_EINVAL && wv_resident_plan(&s, 4, 17, p) == WV_EINVAL);
    CHECK(run(s, 0, 10) == 0 && last.nwv == 8);
    CHECK(wv_resident_plan(&s, 0, 0, nullptr) == WV_OK && run(s, 0, 10) == 0 && last.nwv == free_choice[1]);
    s.cfg.tile_y = 16;
    CHECK(wv_resident_plan(&s, 0, 0, p) == WV_EINVAL);
}

// The bytes reported for a step: every tile sends H rows or columns of its border, two fields per phase, to
// each neighbour, and every cell of the frames moves four memory variables.
void step_bytes()
{
    wv_solver s;
    make(s);
    int p[3];
    CHECK(wv_resident_plan(&s, 4, 8, p) == WV_OK);
    const int R = 32, nbx = 4, nby = 5, H = 4, W = s.cfg.boundary_width = 10;
    double words = 0, psi = 0;
    for (int by = 0; by < nby; by++)
        for (int bx = 0; bx < nbx; bx++) {
            const int rows = std::min(R, 150 - by * R), columns = std::min(64, 200 - bx * 64);
            words += 2 * 2 * H * (((bx > 0) + (bx + 1 < nbx)) * rows + ((by > 0) + (by + 1 < nby)) * columns);
        }
    for (int y = 0; y < 150; y++)
        for (int x = 0; x < 200; x++) psi += 4 * (wv::frame_index(x, 200, W, false) >= 0) + 4 * (wv::frame_index(y, 150, W, false) >= 0);
    const double samples = 2;  // one source per shot; no receivers are set up here
    CHECK(res2d_step_bytes(&s) == 2 * (words * 8 * 2 + psi * 4 * 2) + samples * 4);
}

// Read-backs take what device memory there is, down to one item, then pinned host memory.
void staging()
{
    const size_t M = 1u << 20;
    {
        wv::Staging S;
        CHECK(S.reserve(100, M, 0) == 64);  // cut to the limit
        CHECK(S.reserve(10, M, 0) == 10 && live.size() == 1);
    }
    CHECK(live.empty());
    device_left = 20 * M;
    {
        wv::Staging S;
        CHECK(S.reserve(100, M, 0) == 16);
        CHECK(S.reserve(2, 3 * M, M) == 2);
    }
    device_left = 0;
    {
        wv::Staging S;
        CHECK(S.reserve(100, 3 * sizeof(int), sizeof(int)) == 1);
        CHECK(live.size() == 1);
        const int in[3] = {1, 2, 3};
        int out[3] = {};
        CHECK(S.copy_in(S.data(), in, sizeof(in), nullptr) == hipSuccess);
        CHECK(S.copy_out(out, S.data(), sizeof(out), nullptr) == hipSuccess);
        CHECK(out[0] == 1 && out[2] == 3 && copies == 0);  // (host memory: no device copy)
        device_left = 1000;
        CHECK(S.reserve(10, 12, 4) == 10);  // device memory again
        CHECK(S.copy_out(out, S.data(), sizeof(out), nullptr) == hipSuccess && copies == 1);
    }
    CHECK(live.empty());
    fail_at = allocations + 1;
    wv::Staging S;
    device_left = 0;
    CHECK(S.reserve(1, 8, 0) == 0);
}

}  // namespace

int main(int argc, char **argv)
{
    const std::string t = argc > 1 ? argv[1] : "";
    if (t == "no_memory")
        no_memory();
    else if (t == "memory_asked_for")
        memory_asked_for();
    else if (t == "timing")
        timing();
    else if (t == "failure")
        failure();
    else if (t == "refusal")
        refusal();
    else if (t == "queue")
        queue();
    else if (t == "plan")
        plan();
    else if (t == "step_bytes")
        step_bytes();
    else if (t == "staging")
        staging();
    else
        CHECK(!"a known test");
    std::puts("ok");
    return 0;
}
