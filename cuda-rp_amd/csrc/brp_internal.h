// brp_internal.h -- device data layout and kernel entry points of
// libbubbles_rp (the MI355X coupled FDTD + Rayleigh-Plesset step).
//
// HBM layout
//   Every grid array lives in one common frame: logical columns
//   i in [-1, N+1] and rows j in [-1, M+1] (the union of the reference's
//   1m, 2m, 2n extents for simulation.order = 2), row-major, element
//   (i, j) at  (j + 1) * pitch + (i + kCol0).  kCol0 = 64 puts column i = 0
//   on a 256-byte boundary for both float and double, so a wavefront's 64
//   consecutive cells are one aligned 256/512-byte segment.  pitch is a
//   multiple of 64 elements.
//   Fields: vx, vy, p.x, p.y (two buffers, rotated as p / pn), p0 in the
//   precision's field type F (double or float); void fraction in four int64
//   fixed-point buffers (value * 2^60) rotated as f_g / f_gn / f_gm / spare.
//   Bubbles: structure of arrays in FP64, sorted by cell at set-up.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "../../include/bubbles_rp.h"
#include "rp_vfit.h"

namespace brp {

constexpr int kCol0 = 64;
constexpr double kFgScale = 1152921504606846976.0;       // 2^60
constexpr double kFgInvScale = 8.673617379884035e-19;    // 2^-60
constexpr int kMaxEval = 1024;                           // residual slots per step

// Constant parameters of the grid kernels (passed by value).
struct GridParams {
    int N, M;            // interior cells in x and y
    int pitch;           // elements per frame row
    double dx, dy, rdx, rdy;
    double dt;
    double rho_inf, cs_inf;
    double P_inf;
    int pml_x0, pml_x1, pml_y0, pml_y1;
    int plane_v, plane_p, focused_v, focused_p;
    int src_row;         // source row written (pml.y0 == 0 or extension E1)
    int cylindrical;
    double amp, freq, omega;
    int on_wave, off_wave;
    double fp_x, fp_y, fdist;  // control point and focal distance
    int ap_lo, ap_hi, n_elem;  // aperture cells and element count (E4)
    double s3;           // dt * rho_l * c * c   (MixturePressureKernel)
    int ahead = 0;  // queued before the host knows how the step before ends (halted)
};

__host__ __device__ inline int64_t frame_off(int i, int j, int pitch) {
    return (int64_t)(j + 1) * pitch + (i + kCol0);
}

// Bit-exact binning: floor(x * rdx + c) with no FMA contraction
// (BubbleUpdateIndexKernel, bubble_CUDA_kernel.cuh:355-356).
__device__ inline int bin_index(double x, double rdx, double c) {
#pragma clang fp contract(off)
    double v = floor(x * rdx + c);
    return (v >= -1.0e9 && v <= 1.0e9) ? (int)v : -1000000000;
}

// Window of cells where any void-fraction buffer may be nonzero.
struct Window {
    int i0, i1, j0, j1;  // inclusive, within [0, N+1]
};

// What one wavefront of an RP launch did; k_pressure_ghosts, the iteration's
// last kernel, adds the wavefronts' records to the step's scalars.
struct RPTotals {
    unsigned long long sub_sum;  // sub-steps integrated
    unsigned int done, kept;     // bubbles written back; of them, kept
    int sub_max, flags;          // StepScalars::flags bits
    unsigned int end;            // the device's clock when it was done (low word)
};

// The RP launch's work queue has kQueueHeads heads, each on a line of its own:
// head q hands out the batches q, q + kQueueHeads, ... of the queue order.
constexpr int kQueueHeads = 16, kHeadStride = 32;

// Where the phases of a step begin: the velocity update, the bubble motion,
// the first pressure evaluation; in a Picard iteration the queue, the RP
// launch, the fold at the axis and the pressure evaluation; the temperature
// solve.  A phase ends where the next begins, but for the motion and the RP
// launch: the kernel after them may be queued only once the host has read a
// report, so their own workgroups and wavefronts say when they end.
enum Mark { kMarkVelocity, kMarkMotion, kMarkPressure, kMarkQueue, kMarkRP, kMarkFold, kMarkPicard,
            kMarkThermal, kMarks };

// What the host reads after an evaluation: k_pressure_ghosts, the
// evaluation's last kernel, writes it into pinned host memory, seq last.
struct StepReport {
    double resid;                // of this evaluation (Pa)
    int bbox[4];
    int flags, sub_max;
    unsigned long long sub_sum;
    unsigned int done, reused;
    unsigned long long phase[5];
    double focal[2];
    unsigned long long seq;
};

// Device-side per-step scalars written by the kernels.
struct StepScalars {
    int bbox[4];                         // min i, max i, min j, max j of bubble stencils
    int flags;                           // bit 0 nonfinite p / f_g >= 1, bit 1 scatter
                                         // range / nonfinite R, bit 2 sub-step cap
    int sub_max;                         // max RP sub-steps this step
    unsigned long long sub_sum;          // sum of RP sub-steps this step
    unsigned int done;                   // bubbles written back by the RP kernel this step
    unsigned int reused;                 // of them, kept from the previous iteration
    // The step's phases in ticks of the device's constant-rate clock: marks
    // that kernels set, and the phases' sums (brp_get_phase_times' order).
    unsigned long long mark[kMarks], phase[5];
    int halt;                            // the step does not end with the last evaluation
    unsigned long long resid[kMaxEval];  // max |dp0| bit patterns (>= 0 doubles)
    double focal_v[256];                 // per-block maxima of the focal-point search
    int focal_i[256];
};

// Picard iterations go on while the residual over the ambient pressure is
// above this (bubble_CUDA.cu:243).
constexpr double kPicardTol = (double)1.0e-7f;

#if defined(__HIPCC__)
// Whether the step before goes on or has failed, for kernels of the next step
// queued before the host knows: they leave everything as it is.
__device__ inline bool halted(const GridParams &g, const StepScalars *sc) {
    return g.ahead && sc->halt != 0;
}
// Whether a step needs its first Picard iteration, for kernels queued before
// the host knows: its own test (p_inf = 0: the host has decided).
__device__ inline bool picard_needed(const StepScalars *sc, double p_inf) {
    return p_inf == 0.0 || __longlong_as_double((long long)sc->resid[0]) / p_inf > kPicardTol;
}
// One word of a report.  Report words bypass the caches, one by one: a release
// at system scope would write back every dirty line of the XCD's L2 first.
__device__ inline void report_word(unsigned long long *dst, unsigned long long v) {
    __hip_atomic_store(dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The sequence number, after this wavefront's words have arrived.
__device__ inline void report_seq(StepReport *rep, unsigned long long seq) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
    report_word(&rep->seq, seq);
}

// Sets a phase's mark (the kernel's first workgroup, one thread).  The store
// is written out so that the compiler does not take it for one that may
// change what the kernel reads through its other pointers: after it, uniform
// reads would no longer be scalar loads.
__device__ inline void set_mark(StepScalars *sc, Mark m) {
#if defined(__HIP_DEVICE_COMPILE__)
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && threadIdx.y == 0) {
        const unsigned long long now = wall_clock64();
        asm volatile("global_store_dwordx2 %0, %1, off" ::"v"(&sc->mark[m]), "v"(now));
    }
#endif
}
#endif

#if defined(__HIPCC__)
// FP64 contributions of a workgroup's bubble stencils (256 threads) to frame
// arrays, summed in LDS tiles over the workgroup's bounding box and flushed
// with one global atomic per touched cell: bubbles are cell-sorted, so a
// workgroup's stencils cover a small patch, and in dense clouds (hundreds of
// bubbles per cell) per-contribution global atomics on the same addresses
// serialise.  A patch larger than `cap` cells falls back to global atomics
// per contribution.  Every thread calls begin and flush (they synchronise);
// `any` says whether the thread has a stencil, [i0, i1] x [j0, j1].  The box
// is reduced by lane moves: atomics on its four corners run as loops over the
// lanes.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) double lds_double;
#else
typedef double lds_double;  // the host pass only parses kernel bodies
#endif
template <int TILES, int CAP>
struct StencilTiles {
    double t[TILES][CAP];
    int red[4][4];
};
struct TileBox {
    int i0, j0, w, h;  // w, h <= 0: no stencil
    bool binned;
};
template <int TILES, int CAP>
__device__ inline TileBox tiles_begin(StencilTiles<TILES, CAP> &s, bool any, int i0, int i1, int j0,
                                      int j1) {
    int lo_i = any ? i0 : 0x7fffffff, hi_i = any ? i1 : -0x7fffffff;
    int lo_j = any ? j0 : 0x7fffffff, hi_j = any ? j1 : -0x7fffffff;
    for (int off = 32; off > 0; off >>= 1) {
        lo_i = min(lo_i, __shfl_xor(lo_i, off, 64));
        hi_i = max(hi_i, __shfl_xor(hi_i, off, 64));
        lo_j = min(lo_j, __shfl_xor(lo_j, off, 64));
        hi_j = max(hi_j, __shfl_xor(hi_j, off, 64));
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s.red[wv][0] = lo_i;
        s.red[wv][1] = hi_i;
        s.red[wv][2] = lo_j;
        s.red[wv][3] = hi_j;
    }
    __syncthreads();
    for (int k = 0; k < 4; k++) {
        lo_i = min(lo_i, s.red[k][0]);
        hi_i = max(hi_i, s.red[k][1]);
        lo_j = min(lo_j, s.red[k][2]);
        hi_j = max(hi_j, s.red[k][3]);
    }
    TileBox b{lo_i, lo_j, 0, 0, false};
    if (lo_i <= hi_i && lo_j <= hi_j) {
        b.w = hi_i - lo_i + 1;
        b.h = hi_j - lo_j + 1;
        b.binned = (int64_t)b.w * b.h <= CAP;  // workgroup-uniform
    }
    if (b.binned)
        for (int q = 0; q < TILES; q++)
            for (int k = threadIdx.x; k < b.w * b.h; k += 256) s.t[q][k] = 0.0;
    __syncthreads();
    return b;
}
template <int TILES, int CAP>
__device__ inline void tiles_add(StencilTiles<TILES, CAP> &s, int q, const TileBox &b, double *glob,
                                 int pitch, int i, int j, double v) {
    if (b.binned)
        __hip_atomic_fetch_add((lds_double *)&s.t[q][(j - b.j0) * b.w + (i - b.i0)], v,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        atomicAdd(&glob[frame_off(i, j, pitch)], v);
}
template <int TILES, int CAP>
__device__ inline void tiles_flush(StencilTiles<TILES, CAP> &s, const TileBox &b,
                                   double *const (&glob)[TILES], int pitch) {
    if (!b.binned) return;
    __syncthreads();
    for (int k = threadIdx.x; k < b.w * b.h; k += 256) {
        const int64_t o = frame_off(b.i0 + k % b.w, b.j0 + k / b.w, pitch);
        for (int q = 0; q < TILES; q++)
            if (const double v = s.t[q][k]; v != 0.0) atomicAdd(&glob[q][o], v);
    }
}
#endif

// Bubble arrays (device pointers; n padded to a multiple of 256).
struct BubbleArrays {
    int n;
    double *x, *y;
    double *R[2], *Rn[2], *d1R[2], *PG[2], *bdt[2], *re[2];  // RP state, double-buffered
    double *R_t, *Q_B;
    double *PL[3];        // rotating liquid-pressure history
    double *n_B, *R0, *PG0, *calpha;
    double *vx, *vy;      // v_B (= v_L)
    int *sub;             // sub-steps of the last RP call, per bubble
    int *order;           // work-queue order: bubbles with many sub-steps first
    int *key;             // work-queue keys of a step's first Picard iteration
    int *order_tmp;       // partition scratch: the extreme class before its sort
    int *sort_hist;       // partition scratch: 2048 bin counts / offsets of that sort
    int *part;            // partition scratch: per-block extreme and heavy offsets + totals
    int *bbox_blk;        // per-block stencil bounding boxes of k_motion (4 ints each)
    unsigned int *end_blk;  // per block of k_motion: the device's clock at its end (low word)
    RPTotals *totals;     // per wavefront of the RP launch
    unsigned int *heads;  // kQueueHeads work-queue heads, kHeadStride apart, twice
                          // (the second for the extreme entries on lane pairs)
};

// Bubble physics constants shared by every bubble.
struct BubbleParams {
    double PL0, T0, gam, sig, mu, rho, K0, dt0;
    int mbs, mbe, nbs, nbe;
    double dcx, dcy, dcz;   // delta_coef
    double pi4r3, pi;
    int max_substeps;
    int cylindrical;
    int rp_exact;
    int heavy_threshold;    // sub-steps that put a bubble at the queue front
    int extreme_threshold;  // sub-steps that give a bubble a wavefront of its own (at most)
    const double *rp_shared;  // device table of rp_table_values (kRpTable doubles)
};

// The persistent RP kernel's fixed parameters, in device memory: the kernel
// reads them where its refill and write-back code uses them instead of
// holding them in scalar registers across its sub-step loop.
struct RPLaunch {
    GridParams g;
    BubbleParams bp;
    BubbleArrays b;
};

// The shortened-chain sub-step's constant table: the shared constants
// (rp_table_values, 15 doubles, padded to 64), then the piecewise polynomials
// of the thermal-impedance functions V and Y of alpha = s (1 + i)
// (rp_vfit.h, built for the simulation's gam), which the kernels stage in LDS.
constexpr int kRpVOffset = 64;
constexpr int kRpVFunc = kVIntervals * (kVDegree + 1) * 2;  // doubles per function
constexpr int kRpVSize = 2 * kRpVFunc;
constexpr int kRpTable = kRpVOffset + kRpVSize;

// The constants shared by every bubble in the shortened-chain RP sub-step, in
// the field order of RPFastShared (rp_device.h): PL0, gam, mu, rho, 1/rho,
// dt0, 3 gam, 3 (gam - 1), 3 (gam - 1) K0 T0, 2 sig, 4 mu, mu^2,
// -2 sig rho, 4 pi K0, 16 pi mu; then (from kRpVOffset) the V and Y tables.
inline void rp_table_values(const BubbleParams &bp, double v[kRpTable]) {
    v[0] = bp.PL0;
    v[1] = bp.gam;
    v[2] = bp.mu;
    v[3] = bp.rho;
    v[4] = 1.0 / bp.rho;
    v[5] = bp.dt0;
    v[6] = 3.0 * bp.gam;
    v[7] = 3.0 * (bp.gam - 1.0);
    v[8] = 3.0 * (bp.gam - 1.0) * bp.K0 * bp.T0;
    v[9] = 2.0 * bp.sig;
    v[10] = 4.0 * bp.mu;
    v[11] = bp.mu * bp.mu;
    v[12] = -2.0 * bp.sig * bp.rho;
    v[13] = 4.0 * bp.pi * bp.K0;
    v[14] = 16.0 * bp.pi * bp.mu;
    for (int k = 15; k < kRpVOffset; k++) v[k] = 0.0;
    rp_vtable_build(v[7], v + kRpVOffset);
}

}  // namespace brp

// Kernel launchers (kernels_*.hip).  All run on stream s.
namespace brp {
// Velocity and its boundary at time t; clears the step's scalars.
template <typename F>
void launch_velocity(hipStream_t s, const GridParams &g, F *vx, F *vy, const F *p0,
                     const int64_t *fgn, Window w, int first_step, const F *cxa, const F *cxb,
                     const F *cya, const F *cyb, double t, StepScalars *sc, int nslots);
template <typename F>
void launch_pressure_first(hipStream_t s, const GridParams &g, const F *vx, const F *vy,
                           const F *pnx, const F *pny, F *px, F *py, F *p0,
                           const int64_t *fg_cur, const int64_t *fg_n, int64_t *fg_mp,
                           Window w, const F *ax, const F *bx, const F *ay, const F *by,
                           const double *xu, const double *rxp, StepScalars *sc);
template <typename F>
void launch_pressure_picard(hipStream_t s, const GridParams &g, const F *vx, const F *vy,
                            const F *pnx, const F *pny, F *px, F *py, F *p0,
                            const int64_t *fg_k, const int64_t *fg_n, int64_t *fg_prev,
                            Window w, const F *ax, const F *bx, const F *ay, const F *by,
                            const double *xu, const double *rxp, StepScalars *sc, int slot);
template <typename F>
void launch_pressure_ghosts(hipStream_t s, const GridParams &g, F *p0, const double *el_amp,
                            const double *el_phase, double t, int eval, const RPTotals *tot,
                            int n_tot, const int *bbox_blk, const unsigned int *end_blk,
                            int n_bbox, StepScalars *sc, StepReport *rep, unsigned long long seq,
                            unsigned int done_want);
// Whether a Picard iteration's evaluation changes no ghost cell of p0: they
// hold the source row, or nothing, and mirror no wall.
inline bool pressure_ghosts_fixed(const GridParams &g) {
    const bool source = g.src_row && (g.plane_p || g.focused_p);
    return g.pml_x0 && g.pml_x1 && g.pml_y1 && (g.pml_y0 || source);
}
template <typename F>
void launch_motion(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                   const BubbleArrays &b, const F *vx, const F *vy, StepScalars *sc);
// Shape of an RP launch: bound by its longest chains (one workgroup per
// compute unit), with long chains but bound by the work of all bubbles (as
// many workgroups as fit), or without long chains (the same).
enum RPGrid { kRPLean, kRPFull, kRPLight };
// The RP launch of Picard iteration `slot` over the queue order, with the
// gathered pressures of launch_queue_keys in PL[plp].
// Returns the number of wavefronts launched (their records in b.totals).
// p_inf as in picard_needed: where no iteration is needed, the launch and
// launch_queue_keys leave everything as it is.
template <typename F>
int launch_bubble_step(hipStream_t s, const RPLaunch &host, const RPLaunch *dev, int cur,
                        int plm, int pln, int plp, const F *p0, int64_t *fg_target, StepScalars *sc,
                        int slot, RPGrid shape, int cus, int per_cu, double p_inf);
// Whether the launch runs every bubble on a lane pair, and whether it then
// needs no queue (it gathers the pressures itself).
bool bubble_step_pairs(const RPLaunch &host, int cus);
bool bubble_step_unordered(const RPLaunch &host, int cus);
// The device's compute units and the persistent RP kernel's workgroups per
// compute unit (its occupancy limit), queried once per handle.
void rp_grid_query(int device, int *cus, int *per_cu);
int bubble_step_blocks(int n_bubbles, bool lean, int cus, int per_cu);
// The shape of the next RP launch, from the last one's longest chain and its
// sub-steps in all, and the sub-steps from which its bubbles are extreme.
RPGrid bubble_step_grid(int sub_max, double sub_per_launch, int cus);
int bubble_step_extreme(int sub_max, int extreme_threshold);
// Pressure gather of a Picard iteration's bubbles into PL[plp] and its queue
// keys (predicted or previous sub-step counts; -1: the previous iteration's
// results stand).
template <typename F>
void launch_queue_keys(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                       const BubbleArrays &b, const F *p0, int cur, int plp, int slot, int ext,
                       StepScalars *sc, double p_inf);
void launch_order_partition(hipStream_t s, const BubbleArrays &b, const int *key, int threshold,
                            int ext, bool sort, const StepScalars *sc, double p_inf);
void launch_scatter_initial(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                            const BubbleArrays &b, int64_t *fg_target, StepScalars *sc);
// (sc may be null)
void launch_cyl_fold(hipStream_t s, const GridParams &g, int64_t *fg, StepScalars *sc);
// Frozen schedule: record the accepted RP step sizes of the last RP launch
// (same inputs, same sub-step function) and replay them in a later run.
void launch_rp_record(hipStream_t s, const RPLaunch *dev, int n, int cur, int plm, int pln,
                      int plp, const int64_t *off, double *dts, unsigned int *mismatch);
template <typename F>
void launch_rp_replay(hipStream_t s, const RPLaunch *dev, int n, int cur, int plm, int pln,
                      int plp, const F *p0, int64_t *fg_target, StepScalars *sc,
                      const int64_t *off, const double *dts);
// Scatter of the current R_t with accumulation mode 1 (FP64 atomics),
// 2 (compensated FP32 atomics) or 3 (FP32 atomics) into out (zeroed).
void launch_scatter_variant(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                            const BubbleArrays &b, int mode, void *out, int64_t frame);
void launch_scatter_radii(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                          const BubbleArrays &b, const double *Rt, int64_t *fg, StepScalars *sc);
void launch_copy_d(hipStream_t s, double *dst, const double *src, int n);
void launch_bubble_index(hipStream_t s, const GridParams &g, const BubbleArrays &b,
                         double *out, int which);
void launch_zero_scalars(hipStream_t s, StepScalars *sc, int nslots);

// ---- read-back (readback.hip) ----
// A device array as doubles, row-major with nx columns: a rectangle of a frame
// from logical column i0 and row j0, or (kPerm, kPermInt) a bubble array in
// the caller's order.
struct PackSrc {
    enum Kind { kFloat, kDouble, kFixed, kDensity, kSum3, kPerm, kPermInt } kind;
    int64_t nx;
    const void *src, *src2, *src3;  // src2, src3: kSum3
    const int *iperm;               // caller index -> sorted bubble
    int i0, j0, pitch;
    double scale;                   // kDensity: the liquid's density
    const int *perm;                // the inverse of iperm, on the host (null: src is just being made)
};
// Pinned memory of a handle's read-backs: `small` (the handle's) for arrays of
// up to small_doubles values and copies of up to kCopyMax bytes, else a ring of
// slots.  One read-back at a
// time has them: a handle may be read by several threads.
struct HostRing {
    static constexpr int64_t kMaxSmall = 1 << 17;
    static constexpr size_t kCopyMax = 1 << 16;
    std::mutex mu;
    double *small = nullptr;
    int64_t small_doubles = 0;
    double *host = nullptr;
    hipEvent_t ev[8] = {};
    hipError_t reserve();
    void release();  // the ring's slots and events
};
// rows x src.nx values into dst (leading dimension ld); returns when they are
// there.  `device`, the stream's, is current.
hipError_t read_back(hipStream_t s, int device, HostRing &ring, const PackSrc &src, int64_t rows,
                     double *dst, int64_t ld);

// ---- copies (kernels_copy.hip) ----
// Arrays to copy in one launch (16-byte aligned, sizes multiples of 4);
// src null: zeros.
struct CopyPlan {
    static constexpr int kMax = 64;
    int n = 0;
    unsigned tiles = 0;
    unsigned tile0[kMax];
    void *dst[kMax];
    const void *src[kMax];
    size_t bytes[kMax];
    void add(void *d, const void *s, size_t b);
};
void launch_copy_many(hipStream_t s, const CopyPlan &c);
// One rectangle of several frame arrays (elements of 4 or 8 bytes), each into
// a dense buffer.
struct RectPlan {
    int n = 0;
    void *dst[4];
    const void *src[4];
    int elem[4];
    void add(void *d, const void *s, size_t e) {
        dst[n] = d;
        src[n] = s;
        elem[n++] = (int)e;
    }
};
void launch_copy_rects(hipStream_t s, const RectPlan &r, const Window &w, int pitch);

// ---- temperature (kernels_thermal.hip) ----
template <typename F>
void launch_temperature(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                        const BubbleArrays &b, bool bubbles, Window w, double T_inf, double *T,
                        double *dT, double *heat, const int64_t *fg, const int64_t *fgn,
                        int first, const F *px, const F *py, const F *pnx, const F *pny,
                        StepScalars *sc);

void launch_focal_point(hipStream_t s, const GridParams &g, const double *dT, const double *heat,
                        StepScalars *sc, StepReport *rep, unsigned long long seq);

// ---- adjoint (kernels_adjoint.hip) ----
// Adjoint fields, FP64, same frame as the forward fields.
struct AdjField {
    double *p0, *px, *py, *pnx, *pny, *vx, *vy;
};
// A recorded rectangle of a frame array: logical cells [i0, i0 + w) x
// [j0, j0 + h), stored row by row without padding; cells outside read 0.
template <typename T>
struct Rect {
    const T *p;
    int i0, j0, w, h;
    __host__ __device__ bool in(int i, int j) const {
        return (unsigned)(i - i0) < (unsigned)w && (unsigned)(j - j0) < (unsigned)h;
    }
    __device__ T at(int i, int j) const {
        return in(i, j) ? p[(int64_t)(j - j0) * w + (i - i0)] : T(0);
    }
};
template <typename F>
void launch_box_sumsq(hipStream_t s, const GridParams &g, const F *p0, const int box[4],
                      double *out);
template <typename F>
void launch_adj_seed(hipStream_t s, const GridParams &g, Rect<F> p0, double *Lp0,
                     const int box[4], double c);
void launch_adj_pressure_ghosts(hipStream_t s, const GridParams &g, double *L,
                                const double *el_amp, const double *el_phase, double t,
                                double *gA, double *gP);
template <typename F>
// win (may be null = the whole frame): the cells to evaluate; outside them
// the evaluation's adjoint inputs must be zero.
void launch_adj_pressure(hipStream_t s, const GridParams &g, bool first, const AdjField &a,
                         Rect<int64_t> fk, Rect<int64_t> gC, const double *extra, double *Lf,
                         double *LgC, double *LfN, double *LfM, const F *ax, const F *bx,
                         const F *ay, const F *by, const Window *win);
void launch_adj_velocity_ghosts(hipStream_t s, const GridParams &g, double *Lvx, double *Lvy);
template <typename F>
void launch_adj_velocity(hipStream_t s, const GridParams &g, double *Lvx, double *Lvy,
                         const F *p0, Rect<int64_t> fgn, int first, const F *cxa, const F *cxb,
                         const F *cya, const F *cyb, double *Lp0, double *LfC);
// The adjoints that k_adj_bubble reads and adds to (see there).
struct AdjBubble {
    const double *Rt, *Lf, *jac;
    const double *LRe[4];  // null before the step's last iteration
    double *LRs[4], *lPLn, *lPLm;
    const double *lPL_extra;
    double *Lp0, *Lx, *Ly;
};
// What k_adj_motion carries across the step boundary (see there).
struct AdjHistory {
    int picard;
    double *LA, *LB, *lPLn, *lPLm, *LR[4];
};
template <typename F>
void launch_adj_bubble(hipStream_t s, const GridParams &g, const BubbleParams &bp, int n,
                       const double *x, const double *y, const double *n_B, const AdjBubble &A,
                       Rect<F> p0);
template <typename F>
void launch_adj_motion(hipStream_t s, const GridParams &g, const BubbleParams &bp, int n,
                       const double *xs, const double *ys, Rect<F> vx, Rect<F> vy, double *Lvx,
                       double *Lvy, double *Lx, double *Ly, const AdjHistory &H);
// One Picard iteration of one step for the RP Jacobians of the reverse
// sweep: the step's RP start state and pressure history, the iteration's
// gathered pressure and the forward's sub-step counts (taped), and where its
// Jacobian columns go (35 x nb doubles when last, else 7 x nb).
struct JacSlot {
    const double *rp[6];  // R, Rn, d1R, PG, dt, re at the step's start
    const double *PLm, *PLn, *PLp;
    const int *sub;
    double *jac;
    int last;  // the step's last Picard iteration
};
constexpr int kJacCols = 7, kJacColsLast = 35;
// The Jacobians of n_slots iterations (slots in device memory), in the
// kernel's order (ord: n_slots x nb indices, bins: kAdjJacBins ints, head: two
// counters, buf: adj_rp_jac_buf_doubles(max_blocks) doubles of reverse-mode
// states); replays whose sub-step count differs from the taped one are
// counted in *mismatch.
constexpr int kAdjJacBins = 8193;
void launch_adj_rp_jacobians(hipStream_t s, const BubbleParams &bp, const BubbleArrays &b,
                             double dt_mix, const JacSlot *slots, int n_slots, unsigned *ord,
                             int *bins, unsigned *head, unsigned *mismatch, double *buf,
                             int max_blocks);
// Workgroups of the Jacobian kernel one compute unit holds (its occupancy),
// and the reverse-mode state buffer a grid of `blocks` workgroups needs.
int adj_rp_jac_per_cu();
size_t adj_rp_jac_buf_doubles(int blocks);
}  // namespace brp
