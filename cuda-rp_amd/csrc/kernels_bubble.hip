// kernels_bubble.hip -- Lagrangian bubble kernels for gfx950.
//
// One bubble per lane.  Bubbles are stored sorted by cell, so the B x B
// scatter stencils of neighbouring lanes hit the same few cells; the
// void-fraction accumulation is int64 fixed point (value * 2^60): integer
// atomics are associative, so the scatter is bit-reproducible in any order
// (the FP64 CAS loop of the reference, bubble_CUDA_kernel.cuh:95-114, is not).
#include "brp_internal.h"
#include "rp_device.h"
#include "rp_fast.h"

#include <math.h>

#include <algorithm>

namespace brp {
namespace {

constexpr int kMaxBand = 8;

// smooth_delta_x / smooth_delta_y (bubble_CUDA_kernel.cuh:214-222)
__device__ inline double delta_w(double coef_x, double coef_k, int pos, double h, double b) {
#pragma clang fp contract(off)
    return coef_x * (1.0 + cos(coef_k * (((double)pos - 0.5) * h - b)));
}

// A stencil's weights along one axis, each cosine taken once.  NB = 2: the
// usual band, known at compile time, so that the stencil's loops unroll and
// its loads and cosines overlap; NB = 0: any band up to kMaxBand.  (The
// gather took the inner axis's cosines again for every outer one:
// k_queue_keys over 2^22 bubbles 70 -> 51 us, 2^20 22.8 -> 17.)
template <int NB>
struct Weights {
    double w[NB ? NB : kMaxBand];
    __device__ Weights(double coef_x, double coef_k, int first, int nb, double h, double b) {
        if constexpr (NB > 0) {
#pragma unroll
            for (int a = 0; a < NB; a++) w[a] = delta_w(coef_x, coef_k, first + a, h, b);
        } else {
            for (int a = 0; a < nb; a++) w[a] = delta_w(coef_x, coef_k, first + a, h, b);
        }
    }
    __device__ double operator[](int a) const { return w[a]; }
};

__device__ inline int64_t to_fixed(double v, bool *bad) {
    double s = v * kFgScale;
    if (!(fabs(s) < 4.611686018427388e18)) {  // |v| < 4, NaN rejected
        *bad = true;
        return 0;
    }
    return (int64_t)__double2ll_rn(s);
}

// Block-wide reduction of (min, max) pairs into this block's slot of out
// (4 ints), and when it was done; k_pressure_ghosts folds the slots into sc->bbox.  One plain
// store per block instead of device-scope atomics on four shared addresses, which
// serialise across the whole grid.
__device__ inline void block_bbox(int imin, int imax, int jmin, int jmax, int *out,
                                  unsigned int *end) {
    const unsigned int now = (unsigned int)wall_clock64();  // (its latency passes meanwhile)
    for (int off = 32; off > 0; off >>= 1) {
        imin = min(imin, __shfl_xor(imin, off, 64));
        imax = max(imax, __shfl_xor(imax, off, 64));
        jmin = min(jmin, __shfl_xor(jmin, off, 64));
        jmax = max(jmax, __shfl_xor(jmax, off, 64));
    }
    __shared__ int red[4][4];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[0][w] = imin;
        red[1][w] = imax;
        red[2][w] = jmin;
        red[3][w] = jmax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
        for (int k = 1; k < nw; k++) {
            imin = min(imin, red[0][k]);
            imax = max(imax, red[1][k]);
            jmin = min(jmin, red[2][k]);
            jmax = max(jmax, red[3][k]);
        }
        out[4 * blockIdx.x + 0] = imin;
        out[4 * blockIdx.x + 1] = imax;
        out[4 * blockIdx.x + 2] = jmin;
        out[4 * blockIdx.x + 3] = jmax;
        end[blockIdx.x] = now;
    }
}

// BubbleInterpolationVelocityKernel + v_B <- v_L + BubbleMotionKernel
// (bubble_CUDA_kernel.cuh:398-468, 1282-1297), fused per bubble; also the
// bounding box of the new scatter stencils for the Picard window.
// Bound by its eight cosines rather than its 96 bytes a bubble (2^22 bubbles:
// 131 us with the band known at run time only, 112 with NB = 2; 80 to move
// the bytes).
template <typename F, int NB>
__global__ __launch_bounds__(256) void k_motion(GridParams g, BubbleParams bp, BubbleArrays b,
                                                 const F *__restrict__ vx,
                                                 const F *__restrict__ vy, StepScalars *sc) {
    const bool stop = halted(g, sc);  // tested where it writes: the load's time passes meanwhile
    set_mark(sc, kMarkMotion);
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    int imin = 0x7fffffff, imax = -0x7fffffff, jmin = 0x7fffffff, jmax = -0x7fffffff;
    if (idx < b.n) {
        const double x = b.x[idx], y = b.y[idx];
        const int ibmx = bin_index(x, g.rdx, 1.0), ibmy = bin_index(y, g.rdy, 1.0);
        const int ibnx = bin_index(x, g.rdx, 0.5), ibny = bin_index(y, g.rdy, 0.5);
        // the four weight sets (x at ibm / ibn columns, y at ibn / ibm rows),
        // each evaluated once
        const int nb = NB ? NB : bp.mbe - bp.mbs + 1;
        const Weights<NB> wxm(bp.dcx, bp.dcy, ibmx + bp.nbs, nb, g.dx, x);
        const Weights<NB> wxn(bp.dcx, bp.dcy, ibnx + bp.mbs, nb, g.dx, x);
        const Weights<NB> wyn(bp.dcx, bp.dcz, ibny + bp.mbs, nb, g.dy, y);
        const Weights<NB> wym(bp.dcx, bp.dcz, ibmy + bp.nbs, nb, g.dy, y);
        double vLx = 0.0, vLy = 0.0;
#pragma unroll
        for (int a = 0; a < nb; a++) {
            const int i = ibmx + bp.nbs + a;
#pragma unroll
            for (int c = 0; c < nb; c++) {
                const int j = ibny + bp.mbs + c;
                if (i >= -1 && i <= g.N + 1 && j >= 0 && j <= g.M + 1)
                    vLx += (double)vx[frame_off(i, j, g.pitch)] * wxm[a] * wyn[c];
            }
        }
#pragma unroll
        for (int a = 0; a < nb; a++) {
            const int i = ibnx + bp.mbs + a;
#pragma unroll
            for (int c = 0; c < nb; c++) {
                const int j = ibmy + bp.nbs + c;
                if (i >= 0 && i <= g.N + 1 && j >= -1 && j <= g.M + 1)
                    vLy += (double)vy[frame_off(i, j, g.pitch)] * wxn[a] * wym[c];
            }
        }
        if (!stop) {
            b.vx[idx] = vLx;
            b.vy[idx] = vLy;
        }
        double nx, ny;
        {
#pragma clang fp contract(off)
            nx = x + vLx * g.dt;
            ny = y + vLy * g.dt;
        }
        if (!stop) {
            b.x[idx] = nx;
            b.y[idx] = ny;
        }
        const int kx = bin_index(nx, g.rdx, 0.5), ky = bin_index(ny, g.rdy, 0.5);
        imin = max(kx + bp.mbs, 0);
        imax = min(kx + bp.mbe, g.N + 1);
        jmin = max(ky + bp.mbs, 0);
        jmax = min(ky + bp.mbe, g.M + 1);
        if (imin > imax || jmin > jmax) {
            imin = 0x7fffffff;
            imax = -0x7fffffff;
            jmin = 0x7fffffff;
            jmax = -0x7fffffff;
        }
    }
    if (stop) return;
    block_bbox(imin, imax, jmin, jmax, b.bbox_blk, b.end_blk);
}

// A bubble's volume per cell area, the quantity the scatter spreads
// (VoidFractionReverseLookupKernel, bubble_CUDA_kernel.cuh:576-619).
__device__ inline double fg_temp_of(const GridParams &g, const BubbleParams &bp, double n_B,
                                    double R, double x) {
#pragma clang fp contract(off)
    double v = bp.pi4r3 * n_B * (R * R * R) * g.rdx * g.rdy;
    if (bp.cylindrical) v = bp.pi4r3 * n_B * (R * R * R) * g.rdx * g.rdy / x;
    return v;
}

// Gather of p0 at a bubble (BubbleInterpolationScalarKernel,
// bubble_CUDA_kernel.cuh:361-395) and the bubble's B x B stencil weights.
template <int NB, typename F>
__device__ inline double gather_band(const GridParams &g, const BubbleParams &bp, const F *p0,
                                     double x, double y, int ibnx, int ibny) {
    const int nb = NB ? NB : bp.mbe - bp.mbs + 1;
    const Weights<NB> Dx(bp.dcx, bp.dcy, ibnx + bp.mbs, nb, g.dx, x);
    const Weights<NB> Dy(bp.dcx, bp.dcz, ibny + bp.mbs, nb, g.dy, y);
    double PL = 0.0;
#pragma unroll
    for (int a = 0; a < nb; a++) {
        const int i = ibnx + bp.mbs + a;
#pragma unroll
        for (int c = 0; c < nb; c++) {
            const int j = ibny + bp.mbs + c;
            if (i >= 0 && i <= g.N + 1 && j >= 0 && j <= g.M + 1) {
#pragma clang fp contract(off)
                PL += (double)p0[frame_off(i, j, g.pitch)] * Dx[a] * Dy[c];
            }
        }
    }
    return PL;
}
template <typename F>
__device__ inline double gather_p0(const GridParams &g, const BubbleParams &bp, const F *p0,
                                   double x, double y, int ibnx, int ibny) {
    return bp.mbe - bp.mbs == 1 ? gather_band<2>(g, bp, p0, x, y, ibnx, ibny)
                                : gather_band<0>(g, bp, p0, x, y, ibnx, ibny);
}

// Per-wavefront aggregation of the void-fraction scatter in LDS: an
// open-addressing table of (frame offset, int64 sum) pairs.  A lane adds its
// stencil's contributions to the table; the wavefront flushes the table to
// the grid with one global atomic per distinct cell when it is half full and
// when the wavefront ends.  Bubbles reach a wavefront in batches of
// consecutive cell-sorted indices, so its table sees few distinct cells: with
// clustered bubbles (thousands per cell) this replaces thousands of
// same-address device atomics by one, and int64 addition keeps the result
// identical in any order.  A contribution that finds no slot in kAggProbe
// probes goes to the grid directly.
constexpr int kAggSlots = 512;  // per wavefront (a power of two)
constexpr int kAggProbe = 16;
struct WaveAgg {
    unsigned long long val[kAggSlots];
    int key[kAggSlots];  // frame offset, -1 when empty
    int count;           // occupied slots
};

__device__ inline void agg_clear(WaveAgg &A, int lane) {
    for (int k = lane; k < kAggSlots; k += 64) {
        A.key[k] = -1;
        A.val[k] = 0ull;
    }
    if (lane == 0) A.count = 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) unsigned long long lds_u64_t;
#else
typedef unsigned long long lds_u64_t;  // the host pass only parses kernel bodies
#endif
__device__ inline lds_u64_t *lds_u64(unsigned long long *p) { return (lds_u64_t *)p; }

__device__ inline void agg_add(WaveAgg &A, int cell, unsigned long long q, int64_t *fg) {
    int h = (int)(((unsigned)cell * 2654435761u) >> 23) & (kAggSlots - 1);
    for (int probe = 0; probe < kAggProbe; probe++) {
        const int k = atomicCAS(&A.key[h], -1, cell);
        if (k == -1) atomicAdd(&A.count, 1);
        if (k == -1 || k == cell) {
            __hip_atomic_fetch_add(lds_u64(&A.val[h]), q, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
            return;
        }
        h = (h + 1) & (kAggSlots - 1);
    }
    atomicAdd((unsigned long long *)&fg[cell], q);
}

// Whole wavefront: the table's sums to the grid, then an empty table.
__device__ inline void agg_flush(WaveAgg &A, int lane, int64_t *fg) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = lane; k < kAggSlots; k += 64) {
        const int c = A.key[k];
        if (c >= 0) {
            const unsigned long long v = A.val[k];
            if (v) atomicAdd((unsigned long long *)&fg[c], v);
        }
    }
    agg_clear(A, lane);
}

// VoidFractionReverseLookupKernel's per-bubble scatter (bubble_CUDA_kernel.cuh:
// 576-619): fg_temp times the B x B smooth-delta weights, as int64 fixed
// point, added to the wavefront's table.
template <int NB>
__device__ inline void scatter_band(const GridParams &g, const BubbleParams &bp, double x,
                                    double y, int ibnx, int ibny, double fg_temp, WaveAgg &A,
                                    int64_t *fg, bool *bad) {
    const int nb = NB ? NB : bp.mbe - bp.mbs + 1;
    const Weights<NB> wx(bp.dcx, bp.dcy, ibnx + bp.mbs, nb, g.dx, x);
    const Weights<NB> wy(bp.dcx, bp.dcz, ibny + bp.mbs, nb, g.dy, y);
    for (int a = 0; a < nb; a++) {
        const int i = ibnx + bp.mbs + a;
        for (int c = 0; c < nb; c++) {
            const int j = ibny + bp.mbs + c;
            if (i >= 0 && i <= g.N + 1 && j >= 0 && j <= g.M + 1) {
                double v;
                {
#pragma clang fp contract(off)
                    v = fg_temp * wx[a] * wy[c];
                }
                const int64_t q = to_fixed(v, bad);
                if (q != 0) agg_add(A, (int)frame_off(i, j, g.pitch), (unsigned long long)q, fg);
            }
        }
    }
}
__device__ inline void scatter_bubble_agg(const GridParams &g, const BubbleParams &bp, double x,
                                          double y, int ibnx, int ibny, double fg_temp,
                                          WaveAgg &A, int64_t *fg, bool *bad) {
    if (bp.mbe - bp.mbs == 1)
        scatter_band<2>(g, bp, x, y, ibnx, ibny, fg_temp, A, fg, bad);
    else
        scatter_band<0>(g, bp, x, y, ibnx, ibny, fg_temp, A, fg, bad);
}

__device__ inline unsigned long long lanemask_lt(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// A wavefront's record of an RP launch (RPTotals), one plain store.
__device__ inline void rp_launch_totals(RPTotals *tot, int lane, int sub_max,
                                        unsigned long long sub_sum, unsigned int done,
                                        unsigned int kept, bool bad, bool capped) {
    const unsigned int now = (unsigned int)wall_clock64();  // (its latency passes meanwhile)
    for (int off = 32; off > 0; off >>= 1) {
        sub_max = max(sub_max, __shfl_xor(sub_max, off, 64));
        sub_sum += __shfl_xor(sub_sum, off, 64);
        done += __shfl_xor(done, off, 64);
        kept += __shfl_xor(kept, off, 64);
    }
    const int flags = (__ballot(bad) ? 2 : 0) | (__ballot(capped) ? 4 : 0);
    if (lane == 0)
        tot[blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)] =
            RPTotals{sub_sum, done, kept, sub_max, flags, now};
}

// The next batch of `size` entries of a wavefront from the queue of n (whole
// wavefront).  `head` (wave-uniform) is the head it draws from; when that has
// run out, one read of all heads finds another that has not, or that the
// queue is empty (returns false).  One head for all wavefronts hands out a
// batch every 14 ns, which bounds a launch of short chains: 2^20 bubbles with
// 11 sub-steps each, in batches of 64, 260 us a launch with one head, 211 us
// with sixteen.
__device__ inline bool queue_batch(unsigned int *heads, int lane, int n, int size, int &head,
                                   int &next, int &end) {
    while (head >= 0) {
        unsigned int k = 0;
        if (lane == 0) k = atomicAdd(&heads[head * kHeadStride], 1u);
        k = __builtin_amdgcn_readfirstlane(k);
        const long long base = ((long long)k * kQueueHeads + head) * size;
        if (base < n) {
            next = (int)base;
            end = min((int)base + size, n);
            return true;
        }
        bool alive = false;
        if (lane < kQueueHeads) {
            const unsigned int h = __hip_atomic_load(&heads[lane * kHeadStride], __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            alive = ((long long)h * kQueueHeads + lane) * size < n;
        }
        const unsigned long long m = __ballot(alive);
        // the first live head after this one, in a circle (a head that has
        // run out stays so: this ends)
        const unsigned long long up = m & ~((2ull << head) - 1);
        head = m ? __ffsll((long long)(up ? up : m)) - 1 : -1;
    }
    return false;
}

// Where a wavefront of k_bubble_persistent takes its bubbles from and how it
// holds them: long ones on lane pairs, the others a lane each, its last ones
// on lane pairs again.
enum RPPhase { kOnPairs, kOnLanes, kSpread };

// The integration state of lane src, in every lane.
__device__ inline void spread_lane(RPLaneF<double> &L, RPFastConst &k, int src) {
    double *p[] = {&L.Rp,   &L.Rn,  &L.d1R,  &L.PG,      &L.Rt,     &L.PC0, &L.PC1, &L.PC2,
                   &L.dtL,  &L.remain, &L.time, &L.SumHeat, &L.SumVis,
                   &k.iR0,  &k.PG0, &k.iPG0, &k.calpha_irho, &k.PG0R03, &k.T0_PG0R03, &k.A0, &k.B0};
#pragma unroll
    for (double *q : p) *q = __shfl(*q, src, 64);
    L.counter = __shfl(L.counter, src, 64);
}

// One Picard iteration for every bubble, fused (after k_queue_keys gathered
// PL_p, BubbleInterpolationScalarKernel, kernel.cuh:361-395):
//   BubbleRadiusKernel              (RP from the step's start state, 471-554)
//   VoidFractionReverseLookupKernel (scatter R_t into fg_target, 576-619)
// A bubble whose key is -1 keeps the previous iteration's results (the same
// inputs) and is only scattered.
//
// Persistent kernel with lane-level work refill.  The number of RP sub-steps
// differs by orders of magnitude between bubbles (about 11 at rest, thousands
// through an inertial collapse), so one bubble per lane would run each
// wavefront at the pace of its slowest lane.  Here every lane integrates one
// sub-step per loop pass; lanes whose bubbles reached the sync time are
// written back and refilled with the next bubbles once half of them have
// finished.  Bubbles are handed to wavefronts in
// batches of 64 consecutive (cell-sorted) indices through sixteen atomic counters
// per Picard iteration, so a wavefront costs the sum, not the max, of its
// lanes' sub-steps.  Per bubble the arithmetic is exactly that of the
// reference kernel, so results do not depend on the schedule.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const RPLaunch crpl;  // scalar-loadable
#else
typedef const RPLaunch crpl;  // the host pass only parses kernel bodies
#endif
// The launch parameters, through a pointer opaque to the optimiser so that
// each use site loads what it needs (scalar loads) rather than the kernel
// keeping every field live across the sub-step loop.
__device__ inline crpl *rpl(const RPLaunch *p) {
    crpl *q = (crpl *)p;
    asm volatile("" : "+s"(q));
    return q;
}

// PAIRS (launches with long chains): the queue's extreme entries after the
// dedicated ones run on lane pairs of the shared wavefronts, 32 to a wavefront
// (spread thinner over all of them they leave lanes idle and end no sooner:
// 1, 8, 16, 24 or 32 at least to a wavefront, ms for 16 steps of 2^22 bubbles:
// 189 / 188 / - / 178 / 178, 10 of 65 536: 46.7 / 42.3 / 40.5 / 39.6 / 40.5),
// before the others are taken a lane each; and once the queue is empty a wavefront with at most 32 bubbles left
// moves them onto lane pairs.  A pair does a sub-step in 0.7 of a lane's time,
// and a chain of the 257th rank is nearly as long as the first: RP launch of
// 2^20 bubbles 2142 -> 1476 us, 30 011 1640 -> 1460, 65 536 1207 -> 1110; 2^22
// in clouds (with the full grid; the average of 20 steps) 3.00 -> 2.50 ms, 2.10
// since the queue keys tell a step's first launch its long chains.  At most 256
// VGPRs, so that two wavefronts fit a SIMD; held to that by the attribute for
// two the compiler spills nine, and a launch without long chains took 12 %
// more.
//
// A shared wavefront holds at most `quota` bubbles (64 but for a population
// too small to give every wavefront 64), takes as many from the queue at a
// time, and leaves the sub-step loop to write back and refill when half of
// them have finished (4096^2 clustered on the lean grid, quota 64, ms per step
// for 16 / 24 / 32 / 40 / 48 finished lanes: 24.5 / 23.3 / 23.0 / 23.2 / 24.2;
// 2048^2 equal within 1 % from 24 to 48).
template <typename F, bool FAST, bool PAIRS>
__global__ __launch_bounds__(256) void k_bubble_persistent(const RPLaunch *kp, int max_substeps,
                                                            const double *rp_shared, int cur,
                                                            int plm, int pln, int plp,
                                                            int64_t *__restrict__ fg_target,
                                                            StepScalars *sc, int quota,
                                                            int solo_cap) {
    set_mark(sc, kMarkRP);
    const int lane = threadIdx.x & 63;
    const int nxt = cur ^ 1;
    __shared__ WaveAgg agg_all[4];  // 25 KB: one table per wavefront
    __shared__ __align__(16) double vtab[FAST ? kRpVSize : 1];  // 50 KB: the V and Y tables
    WaveAgg &agg = agg_all[threadIdx.x >> 6];
    agg_clear(agg, lane);
    // The shared RP constants go through LDS into vector registers, held for
    // the whole kernel (two wavefronts per SIMD still fit): read
    // from the constant table instead, each sub-step waited on its scalar
    // loads (no scalar registers are free to hold them).
    __shared__ double shc[16];
    if (FAST) {
        rp_vtab_stage(rp_shared, vtab);
        if (threadIdx.x < 15) shc[threadIdx.x] = rp_shared[threadIdx.x];
        __syncthreads();
    }
    RPFastShared fsh{};
    if (FAST) {
        const ldouble *t = (const ldouble *)shc;
        fsh = RPFastShared{t[0], t[1], t[2],  t[3],  t[4],  t[5],  t[6], t[7],
                           t[8], t[9], t[10], t[11], t[12], t[13], t[14], vtab};
    }
    RPShared sh{};
    if (!FAST) {
        const BubbleParams &bp = rpl(kp)->bp;
        sh = RPShared{bp.PL0, bp.T0, bp.gam, bp.sig, bp.mu, bp.rho, bp.K0, bp.dt0, bp.pi};
    }
    RPFastConst fk{0, 0, 0, 0, 0, 0, 0, 0};
    // The E longest bubbles (the queue's first entries) run one per workgroup
    // in its first wavefront, alone: a wavefront issues the same instructions
    // whether one lane or 64 are active, so a lone bubble never pays for the
    // paths the other lanes would need, nor waits for their refills, and a
    // pair of lanes evaluates two sub-steps' Omega and Lp in one pass
    // (rp_integrate_pair; the launch is bound by this chain: RP launch 2.69 ->
    // 2.23 ms at 2048^2 with 2^20 bubbles, 2.48 -> 1.79 ms with 30 011, 2.85 ->
    // 2.65 ms at 4096^2 with 2^22, against one lane).  Lane 0 writes back.
    // The wavefront runs at raised issue priority until that bubble is done,
    // then joins the shared queue, which starts after the E dedicated entries.
    int E, nb, X;
    {
        const BubbleArrays &b = rpl(kp)->b;
        nb = b.n;
        X = b.part[(b.n + 255) / 256];
        E = min(min(X, (int)gridDim.x), solo_cap);
        if (!PAIRS) X = E;
    }
    constexpr int quota_x = 32;  // lane pairs of a shared wavefront, for the entries [E, X)
    // The first batch of extreme entries of each shared wavefront is its own by
    // its place, a workgroup after the other, the rest are drawn: the second
    // workgroup of a compute unit holds long chains only when the first of
    // every one does.
    const int waves_x = 4 * (int)gridDim.x - E;  // shared wavefronts
    const int w = (int)(threadIdx.x >> 6);
    int batch_next =
        quota_x * ((int)blockIdx.x * 4 + w - min((int)blockIdx.x + (w > 0), E));  // wave-uniform
    int batch_end = min(batch_next + quota_x, X - E);
    const bool solo_start = w == 0 && (int)blockIdx.x < E;
    if (solo_start || batch_next >= batch_end) batch_next = batch_end = 0;
    RPPhase phase = PAIRS && (batch_end > 0 || X - E > quota_x * waves_x) ? kOnPairs : kOnLanes;
    const bool odd = lane & 1;
    int idx = -1;                  // bubble of this lane, -1 when idle
    bool reuse = false;            // idx keeps its previous iteration's results
    bool pre = false;
    if (threadIdx.x < (FAST ? 2 : 1) && (int)blockIdx.x < E) {
        idx = rpl(kp)->b.order[blockIdx.x];
        pre = true;
    }
    bool solo = solo_start;  // wave-uniform
    if (solo) __builtin_amdgcn_s_setprio(3);
    int head = (int)blockIdx.x & (kQueueHeads - 1);  // wave-uniform
    bool exhausted = false;             // wave-uniform
    RPLane L;              // operation-by-operation path
    RPLaneF<double> LF;    // shortened-chain path
    RPConst k{0.0, 0.0, 0.0, 0.0};
    int sub_max = 0;
    unsigned int sub_sum = 0;  // 2^32 sub-steps of a lane would take half an hour
    unsigned int done = 0;  // bubbles this wavefront wrote back
    unsigned int kept = 0;  // of them, with the previous iteration's results
    bool bad = false, capped_any = false;
    while (true) {
        if (solo && __ballot(idx >= 0) == 0ull) {
            solo = false;
            __builtin_amdgcn_s_setprio(0);
        }
        // ---- refill idle lanes from the wave's batch / the global queue
        if (PAIRS && phase == kOnPairs && !solo && exhausted && __ballot(idx >= 0) == 0ull) {
            phase = kOnLanes;
            exhausted = false;
            batch_next = batch_end = 0;
            head = (int)blockIdx.x & (kQueueHeads - 1);
        }
        const bool pairs = FAST && (phase != kOnLanes || solo);  // wave-uniform
        bool need = idx < 0 && !solo && (pairs ? !odd && (lane >> 1) < quota_x : lane < quota);
        {
        crpl *P = rpl(kp);
        const GridParams &g = P->g;
        const BubbleParams &bp = P->bp;
        const BubbleArrays &b = P->b;
        unsigned long long m = __ballot(need);
        bool fresh = pre;
        pre = false;
        while (m != 0ull && !exhausted) {
            if (batch_next >= batch_end) {
                const int first = pairs ? quota_x * waves_x : 0;  // the first batches went by place
                if (!queue_batch(b.heads + (pairs ? kQueueHeads * kHeadStride : 0), lane,
                                 (pairs ? X - E : nb - X) - first, pairs ? quota_x : quota, head,
                                 batch_next, batch_end)) {
                    exhausted = true;
                    break;
                }
                batch_next += first;
                batch_end += first;
            }
            const int avail = batch_end - batch_next;
            const int rank = __popcll(m & lanemask_lt(lane));
            if (need && rank < avail) {
                idx = b.order[(pairs ? E : X) + batch_next + rank];
                need = false;
                fresh = true;
            }
            batch_next += min(avail, __popcll(m));
            m = __ballot(need);
        }
        if (PAIRS && pairs && !solo) {  // the even lane took it, its partner copies
            idx = __shfl(idx, lane & ~1, 64);
            fresh = __shfl((int)fresh, lane & ~1, 64) != 0;
        }
        if (fresh) {
            const double PL = b.PL[plp][idx];  // gathered by k_queue_keys
            reuse = b.key[idx] < 0;            // the previous iteration's results stand
            const double R0 = b.R0[idx];
            k = RPConst{R0, R0 * R0 * R0, b.PG0[idx], b.calpha[idx]};
            if (FAST) {
                // (g3 from LDS: a register less through the sub-steps)
                ldouble *q = (ldouble *)shc;
                asm volatile("" : "+v"(q));
                RPFastShared f = fsh;
                f.g3 = q[6];
                fk = rp_fast_const(R0, k.PG0, k.calpha, bp.T0, f);
            }
            if (reuse) {
                LF.remain = 0.0;
                LF.counter = 0;
                L.remain = 0.0;
                L.counter = 0;
            } else if (FAST) {
                rp_begin_g(LF, b.R[cur][idx], b.Rn[cur][idx], b.d1R[cur][idx], b.PG[cur][idx],
                           b.bdt[cur][idx], b.re[cur][idx], b.PL[plm][idx], b.PL[pln][idx], PL,
                           g.dt, bp.PL0);
            } else {
                RPState in{b.R[cur][idx], b.Rn[cur][idx], b.d1R[cur][idx],
                           b.PG[cur][idx], b.bdt[cur][idx], b.re[cur][idx]};
                rp_begin(L, in, b.PL[plm][idx], b.PL[pln][idx], PL, g.dt, sh);
            }
        }
        }
        const bool active = idx >= 0;
        if (__ballot(active) == 0ull) {
            if (PAIRS && phase == kOnPairs) continue;
            break;
        }
        // ---- sub-steps until half of the quota's bubbles have reached the
        // sync time (or the sub-step cap), or no active lane is left
        // running; finished lanes idle meanwhile.  The refill and write-back
        // code stays outside this loop, and with it the values only that
        // code needs.  Refilling as soon as one lane finished made every
        // wave with a long chain among short bubbles pay the write-back,
        // scatter, pressure gather and set-up nearly every iteration
        // (measured, as ms per step: 2048^2 16.9 -> 16.0, 4096^2 clustered
        // 46.1 -> 29.2 with a batch of 24 on the full grid).
        bool fin, capped;
        double remain;
        if (FAST && pairs) {
            while (true) {
                const bool run = active && LF.remain > 0.0 && LF.counter < max_substeps;
                const unsigned long long rm = __ballot(run);
                if (rm == 0ull || (!exhausted && !solo && __popcll(rm) <= quota_x)) break;
                if (__popcll(rm) == 2) {  // one bubble: to the end
                    if (run) rp_integrate_pair(LF, fk, fsh, odd, max_substeps);
                } else if (run) {
                    rp_pair_pass<false>(LF, fk, fsh, odd, max_substeps);
                }
            }
            capped = active && LF.counter >= max_substeps;
            remain = active ? LF.remain : 0.0;
            fin = active && (!(remain > 0.0) || capped);
            if (odd && fin) {
                fin = false;  // the even lane writes back
                idx = -1;
            }
        } else
        while (true) {
            capped = false;
            remain = 0.0;
            if (active) {
                capped = (FAST ? LF.counter : L.counter) >= max_substeps;
                remain = FAST ? LF.remain : L.remain;
                if (remain > 0.0 && !capped) {
                    if (FAST)
                        rp_substep_g(LF, fk, fsh);
                    else
                        rp_substep(L, k, sh);
                    remain = FAST ? LF.remain : L.remain;
                }
            }
            fin = active && (!(remain > 0.0) || capped);
            const unsigned long long fm = __ballot(fin);
            if (fm != 0ull && (2 * __popcll(fm) >= quota || __ballot(active && !fin) == 0ull))
                break;
            if (PAIRS && exhausted && __popcll(__ballot(active && !fin)) <= 32) break;
        }
        // ---- write back the bubbles that reached the sync time
        done += (unsigned int)__popcll(__ballot(fin));
        kept += (unsigned int)__popcll(__ballot(fin && reuse));
        if (idx >= 0) {
            crpl *P = rpl(kp);
            const GridParams &g = P->g;
            const BubbleParams &bp = P->bp;
            const BubbleArrays &b = P->b;
            if (fin) {
                double R_t;
                if (reuse) {  // the previous iteration's results are in place
                    R_t = b.R_t[idx];
                } else {
                    RPState out;
                    double Q_B;
                    LF.re_n = b.re[cur][idx];
                    if (FAST)
                        rp_end_g(LF, g.dt, &out, &R_t, &Q_B);
                    else
                        rp_end(L, g.dt, &out, &R_t, &Q_B);
                    const int cnt = FAST ? LF.counter : L.counter;
                    b.R[nxt][idx] = out.Rp;
                    b.Rn[nxt][idx] = out.Rn;
                    b.d1R[nxt][idx] = out.d1R;
                    b.PG[nxt][idx] = out.PG;
                    b.bdt[nxt][idx] = out.dt;
                    b.re[nxt][idx] = out.re;
                    b.R_t[idx] = R_t;
                    b.Q_B[idx] = Q_B;
                    b.sub[idx] = cnt;
                    sub_max = max(sub_max, cnt);
                    sub_sum += (unsigned int)cnt;
                    capped_any |= capped && remain > 0.0;
                }
                bad |= !isfinite(R_t);
                const double x = b.x[idx], y = b.y[idx];
                scatter_bubble_agg(g, bp, x, y, bin_index(x, g.rdx, 0.5), bin_index(y, g.rdy, 0.5),
                                   fg_temp_of(g, bp, b.n_B[idx], R_t, x), agg, fg_target, &bad);
                idx = -1;
                reuse = false;
            }
        }
        if (__builtin_amdgcn_readfirstlane(agg.count) > kAggSlots / 2) agg_flush(agg, lane, fg_target);
        // ---- nothing is left to take and at most 32 bubbles run: onto pairs
        if (PAIRS && phase == kOnLanes && !solo && exhausted) {
            const unsigned long long m = __ballot(idx >= 0);
            if (m != 0ull && __popcll(m) <= 32) {
                phase = kSpread;
                int src = __builtin_amdgcn_ds_permute(
                    (idx >= 0 ? 2 * __popcll(m & lanemask_lt(lane)) : 63) * 4, lane);
                src = __shfl(src, lane & ~1, 64);
                const bool mine = (lane >> 1) < __popcll(m);
                spread_lane(LF, fk, src);
                idx = __shfl(idx, src, 64);
                reuse = __shfl((int)reuse, src, 64) != 0;
                if (!mine) idx = -1;
            }
        }
    }
    agg_flush(agg, lane, fg_target);
    rp_launch_totals(rpl(kp)->b.totals, lane, sub_max, sub_sum, lane ? 0u : done, lane ? 0u : kept, bad,
                     capped_any);
}

// The same launch for a population that the chip can hold at once on lane
// pairs (bubble_step_pairs): every bubble runs on a pair of lanes
// (rp_pair_pass), at most `quota` to a wavefront, so that each sub-step takes
// the pair's time, and the population spreads over all the wavefronts instead
// of filling the lanes of a few.  ORDERED: the queue of launch_order_partition;
// its first bubbles go to wavefronts of their own (at most solo_cap, one per
// workgroup first), the others are taken in order as pairs come free.  Not
// ORDERED: at most one bubble per wavefront, so no queue and no keys are
// needed, and the pressure is gathered here.
template <typename F, bool ORDERED>
__global__ __launch_bounds__(256) void k_bubble_pairs(const RPLaunch *kp, int max_substeps,
                                                      const double *rp_shared, int cur, int plm,
                                                      int pln, int plp, const F *__restrict__ p0,
                                                      int64_t *__restrict__ fg_target,
                                                      StepScalars *sc, int slot, int quota,
                                                      int solo_cap, double p_inf) {
    set_mark(sc, kMarkRP);
    const int lane = threadIdx.x & 63;
    const bool odd = lane & 1;
    const int nxt = cur ^ 1;
    __shared__ WaveAgg agg_all[4];
    __shared__ __align__(16) double vtab[kRpVSize];
    __shared__ double shc[16];
    WaveAgg &agg = agg_all[threadIdx.x >> 6];
    agg_clear(agg, lane);
    const bool needed = ORDERED || picard_needed(sc, p_inf);  // ORDERED: the queue is empty
    rp_vtab_stage(rp_shared, vtab);
    if (threadIdx.x < 15) shc[threadIdx.x] = rp_shared[threadIdx.x];
    __syncthreads();
    if (!needed) return;
    const ldouble *t = (const ldouble *)shc;
    const RPFastShared fsh{t[0], t[1], t[2],  t[3],  t[4],  t[5],  t[6], t[7],
                           t[8], t[9], t[10], t[11], t[12], t[13], t[14], vtab};
    // wavefront slots: the first wavefronts of all workgroups, then the second ...
    const int wslot = (int)(threadIdx.x >> 6) * (int)gridDim.x + (int)blockIdx.x;
    int nb, E;
    {
        const BubbleArrays &b = rpl(kp)->b;
        nb = b.n;
        E = ORDERED ? min(b.part[(b.n + 255) / 256], solo_cap) : nb;
    }
    int idx = -1;
    bool solo = wslot < E;  // wave-uniform
    bool fresh = false;
    if (solo && lane < 2) {
        idx = ORDERED ? rpl(kp)->b.order[wslot] : wslot;
        fresh = true;
    }
    if (solo) __builtin_amdgcn_s_setprio(3);
    int batch_next = 0, batch_end = 0;  // wave-uniform
    int head = (int)blockIdx.x & (kQueueHeads - 1);  // wave-uniform
    bool exhausted = !ORDERED;          // wave-uniform
    bool reuse = false;
    RPLaneF<double> L{};
    RPFastConst fk{0, 0, 0, 0, 0, 0, 0, 0};
    double x = 0.0, y = 0.0;
    int ibnx = 0, ibny = 0;
    int sub_max = 0;
    unsigned long long sub_sum = 0;
    unsigned int done = 0, kept = 0;
    bool bad = false, capped_any = false;
    while (true) {
        if (solo && __ballot(idx >= 0) == 0ull) {
            solo = false;
            __builtin_amdgcn_s_setprio(0);
        }
        {  // ---- refill idle pairs (the even lane takes, its partner copies)
            crpl *P = rpl(kp);
            const GridParams &g = P->g;
            const BubbleParams &bp = P->bp;
            const BubbleArrays &b = P->b;
            bool need = ORDERED && idx < 0 && !solo && !odd && (lane >> 1) < quota;
            unsigned long long m = __ballot(need);
            while (m != 0ull && !exhausted) {
                if (batch_next >= batch_end &&
                    !queue_batch(b.heads, lane, nb - E, quota, head, batch_next, batch_end)) {
                    exhausted = true;
                    break;
                }
                const int avail = batch_end - batch_next;
                const int rank = __popcll(m & lanemask_lt(lane));
                if (need && rank < avail) {
                    idx = b.order[E + batch_next + rank];
                    need = false;
                    fresh = true;
                }
                batch_next += min(avail, __popcll(m));
                m = __ballot(need);
            }
            if (ORDERED && !solo) {
                idx = __shfl(idx, lane & ~1, 64);
                fresh = __shfl((int)fresh, lane & ~1, 64) != 0;
            }
            if (fresh) {
                x = b.x[idx];
                y = b.y[idx];
                ibnx = bin_index(x, g.rdx, 0.5);
                ibny = bin_index(y, g.rdy, 0.5);
                double PL;
                if (ORDERED) {
                    PL = b.PL[plp][idx];  // gathered by k_queue_keys
                    reuse = b.key[idx] < 0;
                } else {  // k_queue_keys' gather and test
                    PL = gather_p0(g, bp, p0, x, y, ibnx, ibny);
                    reuse = slot > 1 && PL == b.PL[plp][idx];
                    if (!odd) b.PL[plp][idx] = PL;
                }
                fk = rp_fast_const(b.R0[idx], b.PG0[idx], b.calpha[idx], bp.T0, fsh);
                rp_begin_g(L, b.R[cur][idx], b.Rn[cur][idx], b.d1R[cur][idx], b.PG[cur][idx],
                           b.bdt[cur][idx], b.re[cur][idx], b.PL[plm][idx], b.PL[pln][idx], PL,
                           g.dt, bp.PL0);
                if (reuse) L.remain = 0.0;
                fresh = false;
            }
        }
        const bool active = idx >= 0;
        if (__ballot(active) == 0ull) break;
        // ---- sub-steps: a bubble of its own to the end; else until half of
        // the wavefront's pairs have finished, or none is running
        if (solo) {
            if (active) rp_integrate_pair(L, fk, fsh, odd, max_substeps);
        } else {
            while (true) {
                const bool run = active && L.remain > 0.0 && L.counter < max_substeps;
                const unsigned long long rm = __ballot(run);
                if (rm == 0ull || (!exhausted && __popcll(rm) <= quota)) break;
                if (run) rp_pair_pass<false>(L, fk, fsh, odd, max_substeps);
            }
        }
        const bool capped = L.counter >= max_substeps;
        const bool fin = active && (!(L.remain > 0.0) || capped);
        if (fin && !odd) {  // ---- write back
            crpl *P = rpl(kp);
            const GridParams &g = P->g;
            const BubbleParams &bp = P->bp;
            const BubbleArrays &b = P->b;
            double R_t;
            if (reuse) {
                R_t = b.R_t[idx];
                kept++;
            } else {
                RPState out;
                double Q_B;
                rp_end_g(L, g.dt, &out, &R_t, &Q_B);
                b.R[nxt][idx] = out.Rp;
                b.Rn[nxt][idx] = out.Rn;
                b.d1R[nxt][idx] = out.d1R;
                b.PG[nxt][idx] = out.PG;
                b.bdt[nxt][idx] = out.dt;
                b.re[nxt][idx] = out.re;
                b.R_t[idx] = R_t;
                b.Q_B[idx] = Q_B;
                b.sub[idx] = L.counter;
                sub_max = max(sub_max, L.counter);
                sub_sum += (unsigned long long)L.counter;
                capped_any |= capped && L.remain > 0.0;
            }
            done++;
            bad |= !isfinite(R_t);
            scatter_bubble_agg(g, bp, x, y, ibnx, ibny, fg_temp_of(g, bp, b.n_B[idx], R_t, x), agg,
                               fg_target, &bad);
        }
        if (fin) idx = -1;
        if (__builtin_amdgcn_readfirstlane(agg.count) > kAggSlots / 2) agg_flush(agg, lane, fg_target);
    }
    agg_flush(agg, lane, fg_target);
    rp_launch_totals(rpl(kp)->b.totals, lane, sub_max, sub_sum, done, kept, bad, capped_any);
}

// ---- frozen schedule (finite differences of the frozen-schedule map) ------
// Record: every bubble's RP integration of this Picard iteration again, from
// the same inputs (the RP start state, the pressure history and the PL_p the
// RP launch gathered), with the same sub-step function, writing each accepted
// step size to dts[off[idx] + k]; the count must equal the launch's, and the
// results the launch left (computed, or kept from the previous iteration)
// must equal these bit for bit (a difference is counted in *mismatch, and a
// count's extra sizes are dropped).
__global__ __launch_bounds__(256) void k_rp_record(const RPLaunch *kp, int cur, int plm, int pln,
                                                    int plp, const int64_t *off, double *dts,
                                                    unsigned int *mismatch) {
    const RPLaunch &P = *kp;
    __shared__ __align__(16) double vtab[kRpVSize];
    rp_vtab_stage(P.bp.rp_shared, vtab);
    __syncthreads();
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const BubbleArrays &b = P.b;
    if (idx >= b.n) return;
    const RPFastShared fs = rp_shared_load(P.bp.rp_shared, vtab);
    const RPFastConst fk = rp_fast_const(b.R0[idx], b.PG0[idx], b.calpha[idx], P.bp.T0, fs);
    RPLaneF<double> L;
    rp_begin_g(L, b.R[cur][idx], b.Rn[cur][idx], b.d1R[cur][idx], b.PG[cur][idx],
               b.bdt[cur][idx], b.re[cur][idx], b.PL[plm][idx], b.PL[pln][idx], b.PL[plp][idx],
               P.g.dt, P.bp.PL0);
    const int64_t o = off[idx], cnt = off[idx + 1] - o;
    while (L.remain > 0.0 && L.counter < P.bp.max_substeps) {
        rp_substep_g(L, fk, fs);
        if (L.counter <= cnt) dts[o + L.counter - 1] = L.dtL;
    }
    RPState out;
    double R_t, Q_B;
    rp_end_g(L, P.g.dt, &out, &R_t, &Q_B);
    const int nxt = cur ^ 1;
    const bool same = R_t == b.R_t[idx] && Q_B == b.Q_B[idx] && out.Rp == b.R[nxt][idx] &&
                      out.Rn == b.Rn[nxt][idx] && out.d1R == b.d1R[nxt][idx] &&
                      out.PG == b.PG[nxt][idx] && out.dt == b.bdt[nxt][idx] &&
                      out.re == b.re[nxt][idx];
    if (L.counter != cnt || !same) atomicAdd(mismatch, 1u);
}

// Replay: one Picard iteration of every bubble with the recorded step sizes
// dts[off[idx] .. off[idx + 1]) instead of the step-size control: the gather,
// the RP integration and the aggregated void-fraction scatter of the
// persistent kernel, one bubble per lane.  A bubble that has not reached the
// sync time when its recorded sizes run out sets the sub-step cap flag.
template <typename F>
__global__ __launch_bounds__(256) void k_rp_replay(const RPLaunch *kp, int cur, int plm, int pln,
                                                    int plp, const F *__restrict__ p0,
                                                    int64_t *__restrict__ fg_target,
                                                    StepScalars *sc, const int64_t *off,
                                                    const double *dts) {
    const unsigned long long began = wall_clock64();
    const RPLaunch &P = *kp;
    const GridParams &g = P.g;
    const BubbleParams &bp = P.bp;
    const BubbleArrays &b = P.b;
    const int lane = threadIdx.x & 63;
    __shared__ WaveAgg agg_all[4];
    __shared__ __align__(16) double vtab[kRpVSize];
    WaveAgg &agg = agg_all[threadIdx.x >> 6];
    agg_clear(agg, lane);
    rp_vtab_stage(bp.rp_shared, vtab);
    __syncthreads();
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int nxt = cur ^ 1;
    bool bad = false, capped = false;
    int cnt = 0;
    unsigned int done = 0;
    if (idx < b.n) {
        const double x = b.x[idx], y = b.y[idx];
        const int ibnx = bin_index(x, g.rdx, 0.5), ibny = bin_index(y, g.rdy, 0.5);
        const double PL = gather_p0(g, bp, p0, x, y, ibnx, ibny);
        b.PL[plp][idx] = PL;
        const RPFastShared fs = rp_shared_load(bp.rp_shared, vtab);
        const RPFastConst fk = rp_fast_const(b.R0[idx], b.PG0[idx], b.calpha[idx], bp.T0, fs);
        RPLaneF<double> L;
        rp_begin_g(L, b.R[cur][idx], b.Rn[cur][idx], b.d1R[cur][idx], b.PG[cur][idx],
                   b.bdt[cur][idx], b.re[cur][idx], b.PL[plm][idx], b.PL[pln][idx], PL, g.dt,
                   bp.PL0);
        const int64_t o = off[idx], n = off[idx + 1] - o;
        for (int64_t k = 0; k < n && L.remain > 0.0; k++)
            rp_substep_g<double, true>(L, fk, fs, dts[o + k]);
        capped = L.remain > 0.0;
        RPState out;
        double R_t, Q_B;
        rp_end_g(L, g.dt, &out, &R_t, &Q_B);
        b.R[nxt][idx] = out.Rp;
        b.Rn[nxt][idx] = out.Rn;
        b.d1R[nxt][idx] = out.d1R;
        b.PG[nxt][idx] = out.PG;
        b.bdt[nxt][idx] = out.dt;
        b.re[nxt][idx] = out.re;
        b.R_t[idx] = R_t;
        b.Q_B[idx] = Q_B;
        b.sub[idx] = L.counter;
        cnt = L.counter;
        done = 1;
        bad |= !isfinite(R_t);
        scatter_bubble_agg(g, bp, x, y, ibnx, ibny, fg_temp_of(g, bp, b.n_B[idx], R_t, x), agg,
                           fg_target, &bad);
    }
    agg_flush(agg, lane, fg_target);
    unsigned long long sum = (unsigned long long)cnt;
    for (int o2 = 32; o2 > 0; o2 >>= 1) {
        cnt = max(cnt, __shfl_xor(cnt, o2, 64));
        sum += __shfl_xor(sum, o2, 64);
        done += __shfl_xor(done, o2, 64);
    }
    if (lane == 0) {
        if (done) atomicAdd(&sc->done, done);
        if (sum) atomicAdd(&sc->sub_sum, sum);
        atomicMax(&sc->sub_max, cnt);
    }
    if (bad) atomicOr(&sc->flags, 2);
    if (capped) atomicOr(&sc->flags, 4);
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->mark[kMarkRP] = began;
}

// The initial void fraction (calculate_void_fraction at set-up,
// bubble_CUDA.cu:180-185): scatter of R_t = R0.
__global__ __launch_bounds__(256) void k_scatter_initial(GridParams g, BubbleParams bp,
                                                          BubbleArrays b, int64_t *fg,
                                                          StepScalars *sc) {
    __shared__ WaveAgg agg_all[4];
    WaveAgg &agg = agg_all[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    agg_clear(agg, lane);
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = false;
    if (idx < b.n) {
        const double x = b.x[idx], y = b.y[idx];
        const int ibnx = bin_index(x, g.rdx, 0.5), ibny = bin_index(y, g.rdy, 0.5);
        scatter_bubble_agg(g, bp, x, y, ibnx, ibny, fg_temp_of(g, bp, b.n_B[idx], b.R_t[idx], x),
                           agg, fg, &bad);
    }
    agg_flush(agg, lane, fg);
    if (bad) atomicOr(&sc->flags, 2);
}

// The scatter of given clamped radii (the persistent kernel's scatter without
// its RP integration): every bubble's B x B stencil at its current position.
__global__ __launch_bounds__(256) void k_scatter_radii(GridParams g, BubbleParams bp,
                                                        BubbleArrays b, const double *Rt,
                                                        int64_t *fg, StepScalars *sc) {
    set_mark(sc, kMarkRP);
    __shared__ WaveAgg agg_all[4];
    WaveAgg &agg = agg_all[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    agg_clear(agg, lane);
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = false;
    if (idx < b.n) {
        const double x = b.x[idx], y = b.y[idx];
        const int ibnx = bin_index(x, g.rdx, 0.5), ibny = bin_index(y, g.rdy, 0.5);
        scatter_bubble_agg(g, bp, x, y, ibnx, ibny, fg_temp_of(g, bp, b.n_B[idx], Rt[idx], x),
                           agg, fg, &bad);
    }
    agg_flush(agg, lane, fg);
    if (bad) atomicOr(&sc->flags, 2);
}

// The scatter of the current clamped radii with another accumulation than
// the int64 fixed point, for comparing accumulation schemes (diagnostic):
//   mode 1: FP64 atomic adds into out (double), the arithmetic of the
//           reference's CAS loop (bubble_CUDA_kernel.cuh:95-114) -- the
//           result depends on the order the adds land in;
//   mode 2: compensated FP32: atomic adds into a float sum; the add returns
//           the old value, so its rounding error is recovered exactly
//           (TwoSum) and added, with the contribution's own rounding to
//           FP32, into a second float array comp; the value is sum + comp;
//   mode 3: plain FP32 atomic adds into the float sum.
// out holds `frame` doubles (mode 1) or 2 * frame floats (modes 2, 3: sum,
// then comp) and must be zero on entry.
template <int MODE>
__global__ __launch_bounds__(256) void k_scatter_variant(GridParams g, BubbleParams bp,
                                                         BubbleArrays b, void *out,
                                                         int64_t frame) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= b.n) return;
    const double x = b.x[idx], y = b.y[idx];
    const int ibnx = bin_index(x, g.rdx, 0.5), ibny = bin_index(y, g.rdy, 0.5);
    const double fg_temp = fg_temp_of(g, bp, b.n_B[idx], b.R_t[idx], x);
    const int nb = bp.mbe - bp.mbs + 1;
    for (int a = 0; a < nb; a++) {
        const int i = ibnx + bp.mbs + a;
        const double wx = delta_w(bp.dcx, bp.dcy, i, g.dx, x);
        for (int c = 0; c < nb; c++) {
            const int j = ibny + bp.mbs + c;
            if (i < 0 || i > g.N + 1 || j < 0 || j > g.M + 1) continue;
            double v;
            {
#pragma clang fp contract(off)
                v = fg_temp * wx * delta_w(bp.dcx, bp.dcz, j, g.dy, y);
            }
            const int64_t o = frame_off(i, j, g.pitch);
            if (MODE == 1) {
                atomicAdd((double *)out + o, v);
            } else {
                float *sum = (float *)out, *comp = (float *)out + frame;
                const float vf = (float)v;
                const float old = atomicAdd(sum + o, vf);
                if (MODE == 2) {
#pragma clang fp contract(off)
                    const float s = old + vf;  // the value the atomic stored
                    const float bv = s - old;
                    const float av = s - bv;
                    const float err = (old - av) + (vf - bv);
                    const float ev = (float)(v - (double)vf);
                    atomicAdd(comp + o, err + ev);
                }
            }
        }
    }
}

// VoidFractionCylinderKernel (bubble_CUDA_kernel.cuh:559-573) for order 2:
// the axis fold f_g(0, j) += f_g(1, j); f_g(1, j) = f_g(0, j), exact in int64.
__global__ void k_cyl_fold(GridParams g, int64_t *fg, StepScalars *sc) {
    if (sc) set_mark(sc, kMarkFold);
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j > g.M + 1) return;
    const int64_t o0 = frame_off(0, j, g.pitch), o1 = frame_off(1, j, g.pitch);
    const int64_t v = fg[o0] + fg[o1];
    fg[o0] = v;
    fg[o1] = v;
}

__global__ void k_copy_d(double *dst, const double *src, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) dst[k] = src[k];
}

// Exports ibm / ibn (which = 0 ibm.x, 1 ibm.y, 2 ibn.x, 3 ibn.y) as doubles.
__global__ void k_bubble_index(GridParams g, BubbleArrays b, double *out, int which) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= b.n) return;
    const double v = (which & 1) ? b.y[idx] : b.x[idx];
    const double r = (which & 1) ? g.rdy : g.rdx;
    out[idx] = (double)bin_index(v, r, which < 2 ? 1.0 : 0.5);
}

}  // namespace

template <typename F>
void launch_motion(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                   const BubbleArrays &b, const F *vx, const F *vy, StepScalars *sc) {
    if (b.n <= 0) return;
    const int nblk = (b.n + 255) / 256;
    if (bp.mbe - bp.mbs == 1)
        hipLaunchKernelGGL((k_motion<F, 2>), dim3(nblk), dim3(256), 0, s, g, bp, b, vx, vy, sc);
    else
        hipLaunchKernelGGL((k_motion<F, 0>), dim3(nblk), dim3(256), 0, s, g, bp, b, vx, vy, sc);
}

// Workgroups of the persistent RP kernel: as many as fit (two per CU) when
// the launch is bound by the work of all bubbles; one per CU ("lean") when a
// few long sub-step chains bound it, so that each wavefront has a SIMD of its
// own.  bubble_step_grid decides from the previous launch, by the sub-steps
// that fall to a lane of the lean grid on average against the longest chain's.
// Collapsing bubbles at 2048^2, steps on the full grid against the lean one,
// by that ratio: 0.03 to 0.05 0.98 to 1.01, 0.09 to 0.13 1.01 to 1.04 (2^20 to 1.4e6
// bubbles), 0.18 to 0.196 1.00 to 1.03 (2^21), 0.24 to 0.26 0.87 (2.8e6; at
// half the amplitude 0.96), 0.27 0.83 (3e6 in clouds), 0.35 to 0.37 0.73
// (2^22): the line at 0.2 lies where they cross.
void rp_grid_query(int device, int *cus, int *per_cu) {
    int c = 0, p = 0;
    (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, device);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&p, k_bubble_persistent<float, true, true>, 256,
                                                       0);
    *cus = std::max(1, c);
    *per_cu = std::max(1, p);
}

// A launch whose longest chain is below 128 sub-steps ends with its work; above,
// a quarter of the longest chain makes a bubble extreme (256 at most): 65 536
// bubbles with chains of 300-700, 11 500 launches 5.75 s with 512 and 256, 4.53
// with these, 4.54 with 256 and a half, 4.66 with an eighth.
int bubble_step_extreme(int sub_max, int extreme_threshold) {
    return std::min(extreme_threshold, std::max(64, sub_max / 4));
}

RPGrid bubble_step_grid(int sub_max, double sub_per_launch, int cus) {
    const double lanes = 256.0 * cus;  // lanes of the lean grid
    if (sub_max < 128) return kRPLight;
    return sub_per_launch < 0.2 * lanes * sub_max ? kRPLean : kRPFull;
}

// A lean launch spreads a small population over all its compute units (30 011
// bubbles: 1.84 ms on 118 workgroups of 256 lanes, 1.75 on 256 with 30 bubbles
// to a wavefront); a full one, whose chains are short, fills its wavefronts,
// since each has the tables to stage and its sums to flush (45 000 bubbles
// with 10 sub-steps: 32 us on 176 workgroups, 42 on 512).
int bubble_step_blocks(int n_bubbles, bool lean, int cus, int per_cu) {
    return std::max(1, lean ? std::min(cus, (n_bubbles + 31) / 32)
                            : std::min(cus * per_cu, (n_bubbles + 255) / 256));
}

// Every bubble on a lane pair while that gives a wavefront at most eight of
// them (one wavefront per SIMD): a pair halves the Omega and Lp work of a
// sub-step but takes two lanes.  RP launch of collapsing bubbles, the queue
// of k_bubble_persistent against pairs: 1024 bubbles 1.62 against 1.11 ms,
// 2500 1.90 against 1.55, 8000 1.43 against 1.40, 30 011 1.76 against 1.79,
// 65 536 1.37 against 1.40.  The cap of one dedicated wavefront per workgroup
// holds here too: two or three of them cost 30 011 bubbles 5 and 7 %, 65 536
// 14 %, and 2500 nothing either way.
bool bubble_step_pairs(const RPLaunch &host, int cus) {
    return !host.bp.rp_exact && host.b.n <= 8 * 4 * cus;
}
bool bubble_step_unordered(const RPLaunch &host, int cus) {
    return bubble_step_pairs(host, cus) && host.b.n <= 4 * cus;
}

template <typename F>
int launch_bubble_step(hipStream_t s, const RPLaunch &host, const RPLaunch *dev, int cur,
                        int plm, int pln, int plp, const F *p0, int64_t *fg_target,
                        StepScalars *sc, int slot, RPGrid shape, int cus, int per_cu,
                        double p_inf) {
    if (host.b.n <= 0) return 0;
    const int cap = host.bp.max_substeps;
    if (bubble_step_pairs(host, cus)) {
        const int n = host.b.n, waves = 4 * cus;
        const int blocks = std::min(cus, n);
        if (n <= waves)
            hipLaunchKernelGGL((k_bubble_pairs<F, false>), dim3(blocks), dim3(256), 0, s,
                               dev, cap, host.bp.rp_shared, cur, plm, pln, plp, p0, fg_target, sc,
                               slot, 1, 0, p_inf);
        else
            hipLaunchKernelGGL((k_bubble_pairs<F, true>), dim3(blocks), dim3(256), 0, s, dev, cap,
                               host.bp.rp_shared, cur, plm, pln, plp, p0, fg_target, sc, slot,
                               (n + waves - 1) / waves, cus, p_inf);
        return 4 * blocks;
    }
    const bool lean = shape == kRPLean;
    const dim3 grid(bubble_step_blocks(host.b.n, lean, cus, per_cu));
    // A wavefront's share of a population too small to fill them all; but with
    // the operation-by-operation sub-step, whose wavefronts at different places
    // of its longer code keep a chain waiting for instructions (20 steps of a
    // collapse, 30 bubbles 88 ms in full wavefronts, 97 spread over four; 100
    // bubbles 154 and 162, 300 and more the same).
    const int waves = 4 * (int)grid.x;
    const int quota =
        host.bp.rp_exact ? 64 : std::max(8, std::min(64, (host.b.n + waves - 1) / waves));
    // Dedicated wavefronts: up to one per workgroup on the lean grid, where
    // the longest chains bound the launch.  On the full grid, bound by the
    // work, every one costs a SIMD of throughput: 2^22 clustered bubbles with
    // 16 / 32 / 64 / 128 / 256 of them 183.9 / 183.4 / 183.4 / 186.7 / 193 ms
    // for 16 steps.
    const int solo_cap = lean ? (int)grid.x : std::max(1, cus / (shape == kRPFull ? 4 : 8));
    const auto k = host.bp.rp_exact    ? k_bubble_persistent<F, false, false>
                   : shape == kRPLight ? k_bubble_persistent<F, true, false>
                                       : k_bubble_persistent<F, true, true>;
    hipLaunchKernelGGL(k, grid, dim3(256), 0, s, dev, cap, host.bp.rp_shared, cur, plm, pln, plp,
                       fg_target, sc, quota, solo_cap);
    return 4 * (int)grid.x;
}

// Work-queue order (longest-first scheduling: long sequential sub-step
// chains start at once and overlap everything else): bubbles whose last RP
// call took >= ext sub-steps ("extreme"), sorted by descending count, then
// those with >= thr ("heavy"), then the rest, the last two in index
// (cell-sorted) order.  Passes: per-block class counts, one-block exclusive
// scans, scatter (the extreme class into a scratch array), then the sort of
// the extreme class.  After a launch without long chains there is hardly an
// extreme class: it is left unsorted, three launches less (300 x 600 with
// 45 000 bubbles 25 -> 14 us).
constexpr int kSortBins = 2048;  // bins of the extreme-class sort

__global__ __launch_bounds__(256) void k_part_count(const int *sub, int n, int ext, int thr,
                                                    int *cntE, int *cntH, int *sort_hist,
                                                    unsigned int *heads, const StepScalars *sc,
                                                    double p_inf) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    // not needed: an empty queue (no classes, and the heads past any end)
    const bool needed = picard_needed(sc, p_inf);
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < kSortBins; k += 256) sort_hist[k] = 0;
        if (threadIdx.x < 2 * kQueueHeads) heads[threadIdx.x * kHeadStride] = needed ? 0u : 0x40000000u;
    }
    const int v = idx < n && needed ? sub[idx] : 0;
    const int ce = __syncthreads_count(idx < n && v >= ext);
    const int ch = __syncthreads_count(idx < n && v >= thr && v < ext);
    if (threadIdx.x == 0) {
        cntE[blockIdx.x] = ce;
        cntH[blockIdx.x] = ch;
    }
}

// Exclusive prefix sums of the per-block class counts, in place, one
// workgroup per class (cntE, then cntH = cntE + nblk + 1): each thread sums a
// run of consecutive blocks, the workgroup scans the runs, each thread
// writes its run's prefixes; cnt[nblk] = the class total.
__global__ __launch_bounds__(1024) void k_part_scan(int *cnt0, int nblk) {
    int *cnt = cnt0 + (size_t)blockIdx.x * (nblk + 1);
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int per = (nblk + 1023) / 1024;
    const int b0 = min(nblk, (int)threadIdx.x * per), b1 = min(nblk, b0 + per);
    int sum = 0;
    for (int k = b0; k < b1; k++) sum += cnt[k];
    int x = sum;  // inclusive wave scan of the runs
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int run = x - sum;
    for (int q = 0; q < w; q++) run += wsum[q];
    for (int k = b0; k < b1; k++) {
        const int v = cnt[k];
        cnt[k] = run;
        run += v;
    }
    if (threadIdx.x == 1023) cnt[nblk] = run;
}

__device__ inline int block_rank(bool f, int *wcnt, int *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long m = __ballot(f);
    __syncthreads();
    if (lane == 0) wcnt[w] = __popcll(m);
    __syncthreads();
    int before = 0, all = 0;
    for (int q = 0; q < 4; q++) {
        if (q < w) before += wcnt[q];
        all += wcnt[q];
    }
    *total = all;
    return before + __popcll(m & lanemask_lt(lane));
}

__global__ __launch_bounds__(256) void k_part_scatter(const int *sub, int n, int ext, int thr,
                                                      const int *offE, const int *offH, int nblk,
                                                      int *order, int *ext_out) {
    __shared__ int wcnt[4];
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const bool valid = idx < n;
    const int v = valid ? sub[idx] : 0;
    const bool e = valid && v >= ext;
    const bool h = valid && v >= thr && v < ext;
    int ne, nh;
    const int re = block_rank(e, wcnt, &ne);
    const int rh = block_rank(h, wcnt, &nh);
    const int totE = offE[nblk], totH = offH[nblk];
    const int bE = offE[blockIdx.x], bH = offH[blockIdx.x];
    if (valid) {
        if (e)
            ext_out[bE + re] = idx;
        else if (h)
            order[totE + bH + rh] = idx;
        else  // light rank = position among the block's light bubbles
            order[totE + totH + (blockIdx.x * 256 - bE - bH) + (threadIdx.x - re - rh)] = idx;
    }
}

// The extreme class, longest first: ext_in[0, E) (E = *totE) scattered into
// order[0, E) by descending sub-step count, in bins of 8 sub-steps (order
// within a bin unspecified; results do not depend on the queue order).  A
// counting sort over many workgroups: bin counts (LDS histograms merged with
// one atomic per non-empty bin and workgroup), one-workgroup exclusive scan,
// then per 256-element chunk a range reserved per non-empty bin and LDS ranks
// within it.  hist (kSortBins ints) is cleared by k_part_count.
__device__ inline int sort_bin(int v) {  // ascending bin = descending count
    return kSortBins - 1 - min(v >> 3, kSortBins - 1);
}

__global__ __launch_bounds__(256) void k_sort_hist(const int *sub, const int *totE,
                                                   const int *ext_in, int *hist) {
    __shared__ int h[kSortBins];
    const int E = *totE;
    if ((int)blockIdx.x * 256 >= E) return;  // workgroup-uniform
    for (int k = threadIdx.x; k < kSortBins; k += 256) h[k] = 0;
    __syncthreads();
    for (int i = blockIdx.x * 256 + threadIdx.x; i < E; i += gridDim.x * 256)
        atomicAdd(&h[sort_bin(sub[ext_in[i]])], 1);
    __syncthreads();
    for (int k = threadIdx.x; k < kSortBins; k += 256)
        if (h[k]) atomicAdd(&hist[k], h[k]);
}

__global__ __launch_bounds__(1024) void k_sort_scan(int *hist) {
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // exclusive scan in place: thread t owns bins 2t and 2t + 1
    const int h0 = hist[2 * threadIdx.x], h1 = hist[2 * threadIdx.x + 1];
    int x = h0 + h1;  // inclusive wave scan of the pair sums
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int before = 0;
    for (int q = 0; q < w; q++) before += wsum[q];
    const int excl = before + x - (h0 + h1);
    hist[2 * threadIdx.x] = excl;
    hist[2 * threadIdx.x + 1] = excl + h0;
}

__global__ __launch_bounds__(256) void k_sort_scatter(const int *sub, const int *totE,
                                                      const int *ext_in, int *off, int *order) {
    __shared__ int cnt[kSortBins];  // chunk counts, then reserved bases
    __shared__ int rank[kSortBins];
    const int E = *totE;
    for (int c0 = blockIdx.x * 256; c0 < E; c0 += gridDim.x * 256) {  // workgroup-uniform
        for (int k = threadIdx.x; k < kSortBins; k += 256) {
            cnt[k] = 0;
            rank[k] = 0;
        }
        __syncthreads();
        const int i = c0 + threadIdx.x;
        int idx = -1, bin = 0;
        if (i < E) {
            idx = ext_in[i];
            bin = sort_bin(sub[idx]);
            atomicAdd(&cnt[bin], 1);
        }
        __syncthreads();
        for (int k = threadIdx.x; k < kSortBins; k += 256)
            if (cnt[k]) cnt[k] = atomicAdd(&off[k], cnt[k]);
        __syncthreads();
        if (idx >= 0) order[cnt[bin] + atomicAdd(&rank[bin], 1)] = idx;
        __syncthreads();
    }
}

// Queue keys of a Picard iteration, with the pressure gather of its bubbles
// (BubbleInterpolationScalarKernel, kernel.cuh:361-395) done here, before
// the queue is ordered; PL_p goes to PL[plp] for k_bubble_persistent.
//  * First iteration of a step: in a cavitating step the longest RP chains
//    belong to bubbles that reach the end of their collapse within the step,
//    and they are other bubbles every step, so the previous step's counts do
//    not find them.  Near its end a collapse goes as (t_c - t)^(2/5), so the
//    time left is 0.4 R / (-dR/dt) and the kinetic energy (dR/dt)^2 R^3 stays:
//    a bubble with less time left than the step (its speed taken half a step
//    on under the pressure around it) gets the key 283 ln((dR/dt)^2 (R / R0)^3)
//    - 1640, an estimate of its sub-steps.  An expanding one (R ~ t^(2/5)
//    after a collapse) takes 100 ln(1 + 2.5 dt (dR/dt) / R), by the 1 % limit
//    on a step's change of radius.  Every other bubble keeps its previous
//    count, capped below the extreme class.  Of 32 400 chains of 256 or more
//    among 2^22 clustered bubbles 31 600 are found so, among 36 000 taken for
//    such, and none missed is longer than half the longest; what is missed
//    starts late and ends the launch.  By 10 (-dR/dt) (R / R0) sqrt(3 um / R0),
//    without regard to the time left, 29 900 were found among 80 900: first RP
//    launch of a step 3.68 -> 2.46 ms, the second 2.29.
//    The two constants of the energy's logarithm are a fit to that population
//    (water, 2 MHz, 3 MPa, steps of 33 ns); surface tension, viscosity and the
//    length of the step do not enter.  The key orders the queue and no more,
//    so a poor estimate costs time.  Elsewhere, first launch before and now /
//    later ones now, ms: 2^20 bubbles, 1 MHz, 1.5 MPa 1.81, 1.54 / 1.54, with
//    steps of 17 ns 1.46, 1.30 / 1.29, of 7 ns 1.28, 1.19 / 1.18, 0.75 MPa 1.37,
//    1.34 / 1.35; 2^18, 3 MPa 2.01, 1.77 / 1.75.
//  * Later iterations: the previous iteration's sub-step count, or -1 where
//    the gathered pressure equals the previous iteration's bit for bit.
//    That iteration integrated the same inputs (start state, pressure
//    history, PL_p), so its results stand: k_bubble_persistent only
//    scatters the bubble, from the light end of the queue.  In mixed
//    precision most cells' FP32 pressure stops changing once the Picard
//    residual is small (4096^2 clustered, a step's fifth iteration: 92-97 %
//    of the bubbles; 2048^2, its fourth: 97 %).
template <typename F>
__global__ __launch_bounds__(256) void k_queue_keys(GridParams g, BubbleParams bp, BubbleArrays b,
                                                    const F *__restrict__ p0, int cur, int plp,
                                                    int slot, int ext, StepScalars *sc,
                                                    double p_inf) {
    if (!picard_needed(sc, p_inf)) return;
    set_mark(sc, kMarkQueue);
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= b.n) return;
    const double x = b.x[idx], y = b.y[idx];
    const double PL =
        gather_p0(g, bp, p0, x, y, bin_index(x, g.rdx, 0.5), bin_index(y, g.rdy, 0.5));
    int k;
    if (slot == 1) {
        const double v = b.d1R[cur][idx];
        k = min(b.sub[idx], ext - 1);
        const double R = b.R[cur][idx];
        if (v > 0.0) {
            const int out = (int)fminf(100.0f * log1pf(2.5f * (float)(v * g.dt / R)), 1.0e6f);
            k = b.sub[idx] >= ext ? out : max(k, out);
        } else {
            // the speed half a step on under the pressure around the bubble
            const double u = v - 0.5 * g.dt * (PL + bp.PL0) / (bp.rho * R);
            const double left = 0.4 * R, in = -u * g.dt;
            if (left < 1.05 * in) {
                const float x = (float)(R / b.R0[idx]);
                const float e = (float)(u * u) * (x * x * x);
                k = max(k, (int)fminf(283.0f * logf(e) - 1640.0f, 1.0e6f));
                if (left < 0.1 * in) k = max(k, ext);
            } else if (left < 1.6 * in) {
                k = max(k, bp.heavy_threshold);
            }
        }
        k = max(k, 0);  // (a negative radius gives negative estimates)
    } else {
        k = PL == b.PL[plp][idx] ? -1 : b.sub[idx];
    }
    b.PL[plp][idx] = PL;
    b.key[idx] = k;
}

template <typename F>
void launch_queue_keys(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                       const BubbleArrays &b, const F *p0, int cur, int plp, int slot, int ext,
                       StepScalars *sc, double p_inf) {
    if (b.n <= 0) return;
    hipLaunchKernelGGL(k_queue_keys<F>, dim3((b.n + 255) / 256), dim3(256), 0, s, g, bp, b, p0,
                       cur, plp, slot, ext, sc, p_inf);
}
template void launch_queue_keys<double>(hipStream_t, const GridParams &, const BubbleParams &,
                                        const BubbleArrays &, const double *, int, int, int, int,
                                        StepScalars *, double);
template void launch_queue_keys<float>(hipStream_t, const GridParams &, const BubbleParams &,
                                       const BubbleArrays &, const float *, int, int, int, int,
                                       StepScalars *, double);

void launch_order_partition(hipStream_t s, const BubbleArrays &b, const int *key, int threshold,
                            int ext, bool sort, const StepScalars *sc, double p_inf) {
    if (b.n <= 0) return;
    const int nblk = (b.n + 255) / 256;
    int *cntE = b.part, *cntH = b.part + (nblk + 1);
    hipLaunchKernelGGL(k_part_count, dim3(nblk), dim3(256), 0, s, key, b.n, ext, threshold,
                       cntE, cntH, b.sort_hist, b.heads, sc, p_inf);
    hipLaunchKernelGGL(k_part_scan, dim3(2), dim3(1024), 0, s, cntE, nblk);
    hipLaunchKernelGGL(k_part_scatter, dim3(nblk), dim3(256), 0, s, key, b.n, ext, threshold,
                       cntE, cntH, nblk, b.order, sort ? b.order_tmp : b.order);
    if (!sort) return;
    const int sblk = std::min(1024, nblk);
    hipLaunchKernelGGL(k_sort_hist, dim3(sblk), dim3(256), 0, s, key, cntE + nblk, b.order_tmp,
                       b.sort_hist);
    hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(1024), 0, s, b.sort_hist);
    hipLaunchKernelGGL(k_sort_scatter, dim3(sblk), dim3(256), 0, s, key, cntE + nblk,
                       b.order_tmp, b.sort_hist, b.order);
}

void launch_scatter_initial(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                            const BubbleArrays &b, int64_t *fg_target, StepScalars *sc) {
    if (b.n <= 0) return;
    hipLaunchKernelGGL(k_scatter_initial, dim3((b.n + 255) / 256), dim3(256), 0, s, g, bp, b,
                       fg_target, sc);
}

void launch_scatter_radii(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                          const BubbleArrays &b, const double *Rt, int64_t *fg, StepScalars *sc) {
    if (b.n <= 0) return;
    hipLaunchKernelGGL(k_scatter_radii, dim3((b.n + 255) / 256), dim3(256), 0, s, g, bp, b, Rt, fg,
                       sc);
}

void launch_scatter_variant(hipStream_t s, const GridParams &g, const BubbleParams &bp,
                            const BubbleArrays &b, int mode, void *out, int64_t frame) {
    if (b.n <= 0) return;
    const dim3 grid((b.n + 255) / 256), blk(256);
    if (mode == 1)
        hipLaunchKernelGGL(k_scatter_variant<1>, grid, blk, 0, s, g, bp, b, out, frame);
    else if (mode == 2)
        hipLaunchKernelGGL(k_scatter_variant<2>, grid, blk, 0, s, g, bp, b, out, frame);
    else
        hipLaunchKernelGGL(k_scatter_variant<3>, grid, blk, 0, s, g, bp, b, out, frame);
}

void launch_rp_record(hipStream_t s, const RPLaunch *dev, int n, int cur, int plm, int pln,
                      int plp, const int64_t *off, double *dts, unsigned int *mismatch) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_rp_record, dim3((n + 255) / 256), dim3(256), 0, s, dev, cur, plm, pln,
                       plp, off, dts, mismatch);
}

template <typename F>
void launch_rp_replay(hipStream_t s, const RPLaunch *dev, int n, int cur, int plm, int pln,
                      int plp, const F *p0, int64_t *fg_target, StepScalars *sc,
                      const int64_t *off, const double *dts) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_rp_replay<F>, dim3((n + 255) / 256), dim3(256), 0, s, dev, cur, plm, pln,
                       plp, p0, fg_target, sc, off, dts);
}
template void launch_rp_replay<double>(hipStream_t, const RPLaunch *, int, int, int, int, int,
                                       const double *, int64_t *, StepScalars *, const int64_t *,
                                       const double *);
template void launch_rp_replay<float>(hipStream_t, const RPLaunch *, int, int, int, int, int,
                                      const float *, int64_t *, StepScalars *, const int64_t *,
                                      const double *);

void launch_cyl_fold(hipStream_t s, const GridParams &g, int64_t *fg, StepScalars *sc) {
    hipLaunchKernelGGL(k_cyl_fold, dim3((g.M + 2 + 255) / 256), dim3(256), 0, s, g, fg, sc);
}

void launch_copy_d(hipStream_t s, double *dst, const double *src, int n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_copy_d, dim3((n + 255) / 256), dim3(256), 0, s, dst, src, n);
}

void launch_bubble_index(hipStream_t s, const GridParams &g, const BubbleArrays &b, double *out,
                         int which) {
    if (b.n <= 0) return;
    hipLaunchKernelGGL(k_bubble_index, dim3((b.n + 255) / 256), dim3(256), 0, s, g, b, out, which);
}

template void launch_motion<double>(hipStream_t, const GridParams &, const BubbleParams &,
                                    const BubbleArrays &, const double *, const double *,
                                    StepScalars *);
template void launch_motion<float>(hipStream_t, const GridParams &, const BubbleParams &,
                                   const BubbleArrays &, const float *, const float *,
                                   StepScalars *);
template int launch_bubble_step<double>(hipStream_t, const RPLaunch &, const RPLaunch *, int, int,
                                         int, int, const double *, int64_t *, StepScalars *, int, RPGrid, int,
                                         int, double);
template int launch_bubble_step<float>(hipStream_t, const RPLaunch &, const RPLaunch *, int, int,
                                         int, int, const float *, int64_t *, StepScalars *, int, RPGrid, int,
                                         int, double);

}  // namespace brp
