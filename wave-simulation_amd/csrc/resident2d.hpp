// Resident 2D time loop (resident2d_*.hip, resident2d.cpp): every time step of a run call in one
// cooperative launch, the wavefields of the shots in flight held in LDS.
#pragma once

#include "wave_internal.hpp"

namespace wv {

// Launch plan: tiles of 64 columns x (nwv * srow) rows, one block each; nbx x nby tiles per
// shot, `conc` shots in flight, the handle's shots taken in rounds of `conc`.
struct Res2DPlan {
    int nwv = 0, srow = 0;  // wavefronts per block, rows per wavefront
    int wmax = 16;          // most wavefronts of the kernel variant (its LDS strides)
    int nbx = 0, nby = 0, conc = 0;
    int rows() const { return nwv * srow; }
    int blocks() const { return nbx * nby * conc; }
    explicit operator bool() const { return nwv > 0; }
};

// Arguments of one launch besides the solver's own tables.
struct Res2DArgs {
    int nwv, nbx, nby, conc, nshots;
    int t0, nsteps;
    int words, phase1;         // exchange words of a block; first one of the stress-type phase
    unsigned long long *xch;   // [block][words]: value in the low half, tag in the high half
    unsigned tag0;             // tag of the launch's first step
    unsigned *ctl;             // [0] blocks arrived (all launches), [1] verdict, [2] a wait ran out,
                               // [3] the launch whose refusal those queued behind it share
    unsigned arrive, launch;   // value of ctl[0] when all blocks of this launch are in; launch number
    unsigned long long *host;  // pinned: [0] the latest verdict: 2 launch (+ 1: refused), and in the high half
                               // the launch whose refusal it shares; [1] the launch whose wait ran out last
    const int *bsrc_ptr, *bsrc, *brec_ptr, *brec;  // acquisition lists per (shot, tile) of this plan
    float *psi;                // memory variables of the resident tiles, [block][wavefront][psi_wave floats]
};

// Everything a launch is handed, one kernel argument: the time loop reads it from the argument
// segment where it needs it instead of keeping it in scalar registers.
struct Res2DKernArgs {
    Layout2D L;
    Fields2D F;
    Coef2D C;
    Taps T;
    Cpml2D P;
    Acq A;
    Res2DArgs X;
    Rec2D R;
};

// What a per-physics launcher (resident2d_*.hip) is asked for.
struct ResGo {
    const Res2DPlan *plan;
    const Layout2D *L;
    const Fields2D *F;
    const Coef2D *C;
    const Taps *T;
    const Cpml2D *P;
    const Acq *A;
    const Res2DArgs *X;
    Rec2D rec;
    hipStream_t st;
    int *capacity;  // not null: report the blocks resident at once instead of launching
    size_t lds;
};

// The plan the estimate prefers (empty: none fits) among those with `srow` rows per wavefront and `nwv` wavefronts
// (0: any), rec: of the kernel that records the derivative sums; *gain = estimated step time of the two-launch
// kernels over the plan's.
Res2DPlan res2d_plan(int physics, int order, const Layout2D &L, int nshots, int srow, int nwv, bool rec, double *gain);
// exchange words of a block; *phase1: first one of the stress-type phase
size_t res2d_words(int physics, int H, int rows, int *phase1);
// Returns the launch status (cooperative launch: every block is resident or nothing runs).
hipError_t launch_res2d(int physics, int order, const Res2DPlan &plan, const Layout2D &L, const Fields2D &F,
                        const Coef2D &C, const Taps &T, const Cpml2D &P, const Acq &A, const Res2DArgs &X,
                        const Rec2D *rec, hipStream_t stream);

}  // namespace wv
