// dg_kernels.hpp -- launch interface between the host runtime (dg_api.hip)
// and the kernels (dg_kernels.hip).
#pragma once
#include "dg_grid.hpp"
#include "dg_math.hpp"

namespace dg {

// Kernel classes for the optional live per-kernel timing (HIP events recorded
// after each launch on the grid's stream).
enum KernelId {
    K_BC, K_CFL, K_HALF, K_PRED_X, K_PRED_Y, K_PRED_Z, K_EMF_PRED, K_FARADAY_HALF, K_WHALF, K_CTU,
    K_FLUX_X, K_FLUX_Y, K_FLUX_Z, K_EMF, K_FARADAY, K_APPLY, K_COUNT
};
static const char* const kKernelNames[K_COUNT] = {
    "boundary", "cfl", "half_states", "pred_sweep_x", "pred_sweep_y", "pred_sweep_z", "emf_pred", "faraday_half",
    "whalf", "ctu_correct", "flux_sweep_x", "flux_sweep_y", "flux_sweep_z", "emf", "faraday", "apply"};

// The step sizes of a step, in device memory: the CFL pass may have found
// them on the device (launch_ctl_* / launch_cfl), so that the host need not
// wait for one step to launch the next.
struct StepDts {
    double full[3], half[3];  // dt / dx, dt / dy, dt / dz and their halves
    int stop, pad;            // set: every kernel of the step leaves at once
};
// Control of a run of steps launched without waiting (dg_advance).  The CFL
// pass of a step commits the one before it: where that one failed, or no time
// is left, it sets `stop` and every later launch of the run does nothing.
constexpr int CTL_RING = 64;  // steps of a run
enum { CTL_NO_SPEED = 1 };    // why: the maximum signal speed is zero
struct StepCtl {
    StepDts t;
    double dt, left, left_next, tol;  // of the step begun last: its dt, the time left before and after it
    unsigned long long err;           // its failure key
    unsigned long long vmax;          // CFL maximum being gathered (FP64 bits)
    int count, why;                   // steps begun; CTL_*
    unsigned ticket, pad;             // workgroups of the CFL pass that have finished
    double ring[CTL_RING];            // dt of each step begun
};

// Everything one unsplit step needs: geometry, physics switches, the current
// and next state, and the scratch arrays of the stages.
struct StepCtx {
    int dim;
    bool mhd, mixed;
    int ctu, cfl_mode;
    bool fused;           // fused sweeps (no half-state arrays) where available
    int march_chunk;      // faces one thread walks in a strided-axis sweep (0: automatic)
    int march_window;     // 1: FP64 walkers run the register-window form of the FP32 build (a check; same results)
    Ext ce, fe;
    Phys ph;
    double d[3];
    StepCtl* ctl;         // step sizes, stop flag and failure word
    int half;             // split sweeps: steps of dt / 2
    double cfl_coeff;
    Soa W, Wn;            // current / next cell state
    double* B[3];         // current face B
    double* Bn[3];        // next face B
    double* Bh[3];        // half-step face B (CTU MHD)
    Soa HS[6];            // xL, xR, yL, yR, zL, zR
    Soa F[3];             // corrector (final) fluxes; reference-structured path: both
    Soa Fp[3];            // predictor fluxes of the fused path
    Soa T[6];             // 3D hydro corner fluxes (reference-structured path: five)
    double* E0[3];        // corner EMF (predictor, then final)
    double* Eh[3];        // half-step reference EMF
    unsigned long long* err;
    double* cflpart;      // per-block CFL maxima of the new state (apply pass), or null
    void (*mark)(void* user, int id);  // per-kernel timing hook (null when off)
    void* mark_user;
};
inline void mark(const StepCtx& c, int id) {
    if (c.mark) c.mark(c.mark_user, id);
}

// One boundary pass (cells or faces of one face/axis of one BC element).
struct BCArgs {
    const StepCtl* ctl;  // of a run of steps (its end is checked before the pass), or null
    Soa W;
    double* B[3];
    Ext ce, fe;
    int dim, nf, kind, side, axis, corners, gated;  // side: 0 negative, 1 positive, 2 both (periodic)
    double st[8];
    int lo[2], hi[2];                           // transverse ranges
};
// A whole boundary list as one launch (k_bc_list): its passes in the list's
// order, at most one per face, every one over the full transverse range.
struct BCPass {
    int axis, side, kind, gated;  // side: 0 negative, 1 positive; kind as dg_bc
    double st[8];
};
// The kernels walk the passes by these bytes, in one word of the arguments:
// read from the passes themselves, each is another line of the argument
// segment to wait for.  (Unrolled over all six with their first words read up
// front, the lines cost 4 us a step.)  With the run's words read together and
// the 1D step's cells before its gate: 1D 1024 cells, 20 steps, 22 us less, 64 x
// 32 x 32 3D MHD, 6 steps, 11 us.
inline unsigned long long bc_head(const BCPass& p) { return (unsigned long long)(p.axis | p.side << 2 | p.kind << 3 | (p.gated ? 1 : 0) << 5); }
struct BCListArgs {
    const StepCtl* ctl;     // as BCArgs
    Soa W;
    double* B[3];
    Ext ce, fe;
    int dim, nf, npass;
    unsigned ncell, nface;  // ghost cells / boundary faces the launch covers
    unsigned long long heads;  // byte q: bc_head of pass q (launch_bc_list)
    BCPass p[6];
};
// Batched 2D MHD patches (CTU + CT).  Every stage of the step is one launch
// over all patches: a block table per work kind maps each workgroup to a
// patch and the first work item it covers.  Pools hold every patch back to
// back: patch p's cell field f of pool X is at X + nfield*oc + f*nc; face
// component c at X + 3*of + c*nfc.
struct PatchDesc {
    int n[2];           // interior cells
    double d[2];        // dx, dy
    long oc, nc;        // cell offset / count (ghosts included)
    long of, nfc;       // face offset / count
    int cls;            // size class (tile table index)
};
enum { BATCH_CLASSES = 4, BATCH_THREADS = 256 };
// per-patch status codes (the values of DG_ERR_CFL / DG_ERR_DT_UNDERFLOW)
enum { BATCH_ERR_CFL = 5, BATCH_ERR_DT = 6 };
// work kinds of a batched step (items per patch in dg_api.hip: batch_items)
enum BatchKind {
    BK_BC,                                   // boundary: ghost cells x 8 fields, then boundary faces x 3 components
    BK_CELLS1,                               // cells [-1, n+1)^2: CFL
    BK_PRED_X, BK_PRED_Y,                    // predictor sweeps (x: faces-per-thread chunks; y: 63 faces per wavefront)
    BK_EDGES,                                // edges [-1, n+2)^2 in tiles: the half-step stages
    BK_FLUX_X, BK_FLUX_Y,                    // corrector sweeps
    BK_FACES,                                // every face (and cell) in tiles: the final stages
    BK_CELLS,                                // every cell: initialize_B_fields
    BK_COUNT
};
struct BlockTable {
    const int* patch;   // per workgroup: patch
    const int* first;   // per workgroup: first work item (a multiple of BATCH_THREADS)
    unsigned nblocks;
};
struct BCPasses {
    unsigned long long heads;
    BCPass p[4];
};
struct BatchArgs {
    const PatchDesc* P;
    int npatch;
    double* W[2];              // cell state pools (8 fields), double-buffered
    double* B[2];              // face-B pools, double-buffered
    double* Fp;                // predictor fluxes, 2 axes x 8 fields
    double* F;                 // corrector fluxes, 2 axes x 8 fields
    double* Bh;                // half-step faces
    double* E0;                // corner EMF
    double* Eh;                // half-step reference EMF
    int* parity;               // per patch: index of the current buffer
    double* dt_last;           // per patch: dt of the last accepted step
    long* steps;               // per patch: accepted steps
    long* fails;               // per patch: rejected attempts
    int* status;               // per patch: 0, or the DG_* code that stopped it
    unsigned long long* err;   // per patch failure key of the current attempt
    unsigned long long* vmax;  // per patch CFL signal speed (FP64 bits)
    unsigned long long* vnext; // per patch: the apply pass's maximum over the interior of the state it wrote (FP64 bits)
    int* cfl_ok;               // per patch: vnext describes the current state (its last attempt was committed)
    double* dt;                // per patch dt of the current attempt
    StepDts* ts;               // per patch dt / dx, dt / dy of the current attempt
    int* halv;                 // per patch halvings since the last accepted step
    int* active;               // per patch: steps in this launch sequence
    Phys ph;
    double cfl_coeff, tol;
    int cfl_mode;
    BCPasses bc;               // outflow or periodic on every face, corner ghosts
    int chunk[BATCH_CLASSES];  // x-sweep faces per thread, per size class
    int ysw[BATCH_CLASSES];    // y-sweep segment width in lanes (64, 32, 16: 63, 31, 15 faces; 0: columns streamed), per size class
    int commit;                // 0: run the step, keep every patch's state and counters (tuning)
    int cls_filter;            // -1: all patches, else only this size class
};

// The kernels are compiled twice (dg_kernels.hip): p64 is the FP64 drop-in
// (no FMA contraction, correctly rounded division and square root); p32 holds
// the mixed form's kernels (FP32 reconstruction and Riemann solves with
// contraction and fast FP32 division / square root; FP64 state, accumulation,
// pressure recovery and CT).  Separate namespaces keep every kernel symbol of
// one build out of the other.
#define DG_LAUNCH_INTERFACE                                                                                     \
    void launch_batch_step(const BatchArgs& a, const BlockTable* bt, bool init_only, bool first, bool last, hipStream_t s); \
    long launch_step(const StepCtx& c, hipStream_t s);  /* returns the CFL maxima left in cflpart */              \
    long launch_split_axis(const StepCtx& c, int ax, Soa in, Soa out, hipStream_t s);  /* one split sweep (hydro) */ \
    void launch_bc(const BCArgs& a, bool faces, hipStream_t s);                                                 \
    bool launch_bc_list(BCListArgs& a, hipStream_t s);                                                          \
    void launch_cfl(const StepCtx& c, unsigned long long* out, bool run, hipStream_t s);                        \
    void launch_cfl_tail(const StepCtx& c, long nparts, unsigned long long* out, bool run, hipStream_t s);      \
    bool launch_bc_tail(BCListArgs& a, const StepCtx& c, long nparts, hipStream_t s);  /* list and tail, in a run */  \
    void launch_ctl_set(const StepCtx& c, double dt, hipStream_t s);        /* one step of size dt */             \
    void launch_ctl_begin(const StepCtx& c, double left, double tol, hipStream_t s);  /* a run of steps */        \
    void launch_ctl_next(const StepCtx& c, hipStream_t s);                  /* its next step, without CFL */      \
    void launch_init_B(int dim, Soa W, double* B, Ext ce, Ext fe, hipStream_t s);                               \
    void launch_divb(int dim, double* B, Ext ce, Ext fe, const double d[3], unsigned long long* out, hipStream_t s); \
    void launch_fill_u64(unsigned long long* p, unsigned long long v, int n, hipStream_t s);                    \
    void launch_aos_to_soa(const double* a, int stride, int nf, Soa soa, long n, hipStream_t s);                \
    void launch_soa_to_aos(Soa soa, int nf, double* a, int stride, long n, hipStream_t s);
// tiles of 8 x 32 points of the 2D constrained-transport passes
inline long ct_tiles(long ni, long nj) { return ((ni + 7) / 8) * ((nj + 31) / 32); }
namespace p64 { DG_LAUNCH_INTERFACE }
namespace p32 { DG_LAUNCH_INTERFACE }

}  // namespace dg
