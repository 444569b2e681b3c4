// mkde_kernels.hip -- hand-written HIP kernels for gfx950 (CDNA4, wave64).
//
// Hot path of the reference (Guiming/mGPUKDE_tiled) re-designed for MI355X:
//   k_density_tile    per-cell gather density over 64x64-cell blocks
//                     (replaces KernelDesityEstimation_pPoints,
//                     kde_kernel_kdtr.cu:461-574, and the CPU loop tiled:707-733)
//   k_ec              per-point edge-correction integral, O(R) per point
//                     (replaces CalcEdgeCorrectionWeights kde_kernel_kdtr.cu:117-265
//                     and EdgeCorrectionWeightsExact tiled:2694-2807)
//   k_point_sums, k_point_density_f   density at points over the cell-binned
//                     index, pilot and leave-one-out forms (replaces DensityAtPointsKdtr
//                     kde_kernel_kdtr.cu:681-953 and the CPU scatter tiled:3312-3347)
//   k_loo_multi       leave-one-out densities of up to 16 fixed bandwidths in one
//                     pass over point pairs (batched LogLikelihood, tiled:3214-3368)
//   k_boundary, k_dist_boundary   MarkBoundary / CalcDist2Boundary
//                     (kde_kernel_kdtr.cu:1209-1353, tiled:3993-4131)
//   reductions        FP64 sums of logs (replaces ReductionSum kde_kernel_kdtr.cu:1045-1111)
//
// Numerics shared by every kernel (the reference CPU path's rules):
//   cell centre  cx = fl32(xll + (c+0.5)*cs), cy = fl32(yll + (nrows-0.5-r)*cs)
//                evaluated in double (Utilities.h:13-14)
//   cut-off      fl64(dx^2 + dy^2) < 9*h2f with dx = fl32(cx - px), h2f = fl32(h*h)
//                -- evaluated exactly (both squares are exact in double)
//   kernel       K = exp(-d^2/(2 h2f)) / (2*pi*h2f), computed as
//                exp2(fl32(d^2 * a)) with a = -log2(e)/(2 h2f); the density and
//                edge-correction integrands use the separable form
//                exp2(dx^2 a) * exp2(dy^2 a) over raster cells.
//   sums         short FP32 partial sums folded with compensation (Kahan) or
//                into FP64; FP64 prefix sums (edge correction) and FP64
//                log-likelihood sums.
#include <hip/hip_runtime.h>
#include <float.h>
#include <limits.h>
#include <math.h>
#include <algorithm>
#include <mutex>
#include <stdint.h>
#include <stdlib.h>

#include "mkde_device.h"

#define WAVE 64

// ------------------------------------------------------------------ helpers --

__device__ __forceinline__ float cell_x(double xll, double cs, int64_t c)
{
    return (float)__dadd_rn(xll, __dmul_rn((double)c + 0.5, cs));
}

// nrm05 = (double)nrows - 0.5 (ROW_TO_YCOORD evaluates (NROWS - 0.5 - ROW)).
__device__ __forceinline__ float cell_y(double yll, double cs, double nrm05, int64_t r)
{
    return (float)__dadd_rn(yll, __dmul_rn(nrm05 - (double)r, cs));
}

// fl64(a^2 + b^2) for float a, b: both squares are exact in double.
__device__ __forceinline__ double sq2(float a, float b)
{
    double da = a, db = b;
    return __dadd_rn(__dmul_rn(da, da), __dmul_rn(db, db));
}

__device__ __forceinline__ double sqd(float a)
{
    double da = a;
    return __dmul_rn(da, da);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Distance from v to the interval [lo, hi] along one axis as fl32(lo - v) or
// fl32(v - hi); 0 inside.  Because fl32 subtraction is monotone, for every u in
// [lo, hi] |fl32(u - v)| >= this value: it is an exact lower bound of the
// reference's |dx| over the interval.
__device__ __forceinline__ float gap1(float v, float lo, float hi)
{
    return v < lo ? (lo - v) : (v > hi ? (v - hi) : 0.0f);
}

// Largest |fl32(u - v)| over u in [lo, hi]: attained at an end point.
__device__ __forceinline__ float far1(float v, float lo, float hi)
{
    float a = fabsf(lo - v), b = fabsf(hi - v);
    return a > b ? a : b;
}

// Launch-wide counters spread over MKDE_CNT_SLOTS cache lines: atomics of
// many workgroups to one address serialise (measured: 400k one-per-workgroup
// adds to a single counter cost ~2.6 ms), so workgroup b adds to slot
// b % MKDE_CNT_SLOTS and k_fold_slots sums the slots into the word after them.
#define MKDE_CNT_SLOTS 512
#define MKDE_CNT_STRIDE 16   // 64-bit words between slots (128 B)
__device__ __forceinline__ void slot_add(unsigned long long *slots, unsigned long long v)
{
    if (v) atomicAdd(&slots[(blockIdx.x % MKDE_CNT_SLOTS) * MKDE_CNT_STRIDE], v);
}

// Kahan fold of a short FP32 partial sum into (sum, comp).
__device__ __forceinline__ void kahan_fold(float part, float &sum, float &comp)
{
    float y = part - comp;
    float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
}

// Order-preserving compaction across a workgroup of NW waves.  Returns this
// thread's slot among the flagged threads; *total gets the flagged count.
template <int NW>
__device__ __forceinline__ int block_compact(bool flag, int *s_wcnt, int *total)
{
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    uint64_t m = __ballot(flag);
    int rank = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) s_wcnt[wave] = __popcll(m);
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        off += (w < wave) ? s_wcnt[w] : 0;
        tot += s_wcnt[w];
    }
    *total = tot;
    __syncthreads();
    return off + rank;
}
__device__ __forceinline__ int block_compact256(bool flag, int *s_wcnt, int *total)
{
    return block_compact<4>(flag, s_wcnt, total);
}

__device__ __forceinline__ unsigned wave_incl_scan(unsigned v, int lane)
{
    for (int d = 1; d < WAVE; d <<= 1) {
        const unsigned o = __shfl_up(v, d, WAVE);
        if (lane >= d) v += o;
    }
    return v;
}

__device__ __forceinline__ int clampi(int64_t v, int64_t lo, int64_t hi)
{
    return (int)(v < lo ? lo : (v > hi ? hi : v));
}

// Candidate-bin range of a query rectangle [qx0,qx1]x[qy0,qy1] grown by reach.
__device__ __forceinline__ void bin_range(const BinGrid &bg, double qx0, double qx1, double qy0, double qy1,
                                          double reach, int &bxa, int &bxb, int &bya, int &byb)
{
    bxa = clampi((int64_t)floor((qx0 - reach - bg.x0) / bg.size), 0, bg.nbx - 1);
    bxb = clampi((int64_t)floor((qx1 + reach - bg.x0) / bg.size), 0, bg.nbx - 1);
    bya = clampi((int64_t)floor((qy0 - reach - bg.y0) / bg.size), 0, bg.nby - 1);
    byb = clampi((int64_t)floor((qy1 + reach - bg.y0) / bg.size), 0, bg.nby - 1);
}

// Exact lower bound of the cut-off distance between any point of bin box B and
// any position in rectangle Q (both in float coordinates).
__device__ __forceinline__ double box_gap2(const BinInfo &B, float qx0, float qx1, float qy0, float qy1)
{
    float gx = B.x1 < qx0 ? (qx0 - B.x1) : (B.x0 > qx1 ? (B.x0 - qx1) : 0.0f);
    float gy = B.y1 < qy0 ? (qy0 - B.y1) : (B.y0 > qy1 ? (B.y0 - qy1) : 0.0f);
    return sq2(gx, gy);
}

// ============================================================ point index ====

// Per-job point records in bin order: gather h and ew through the permutation
// and derive the kernel constants.
__global__ void k_prep_points(int64_t n, const int *perm, const float *xs, const float *ys, const float *w_orig,
                              const float *h_orig, const float *ew_orig, float h_fixed, PtRec *out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int o = perm[i];
    float h = h_fixed > 0.0f ? h_fixed : (h_orig ? h_orig[o] : 0.0f);
    float w = w_orig[o];
    float ew = ew_orig[o];
    double h2 = (double)(float)(h * h);
    PtRec r;
    r.x = xs[i];
    r.y = ys[i];
    r.pad = 0.0f;
    if (h2 > 0.0 && h2 < 1e300) {
        r.coef = (float)((double)w * (double)ew / (h2 * (double)MKDE_TWO_PI_F));
        r.a = -MKDE_LOG2E / (2.0 * h2);
        r.thr = 9.0 * h2;
    } else {
        r.coef = 0.0f;
        r.a = 0.0;
        r.thr = -1.0;
    }
    out[i] = r;
}

// Whether a source may enter a sum whose weights have both signs (moments of a
// group, nodes of a block): an infinite coefficient, or one whose float sums may
// overflow, would cancel to NaN there, while its kernels add up to +inf.
__device__ __forceinline__ bool coef_signed_ok(float coef) { return fabsf(coef) < 1e30f; }

// A float squared distance below lo is inside the cut-off thr, one above hi is
// not.  fl32(dx^2 + dy^2) is within 2^-22 relative where it neither overflows nor
// becomes subnormal; elsewhere nothing is taken as decided (lo = -1, a hi that
// holds for every distance in doubt).  thr < 0: nothing is inside.
__device__ __forceinline__ void thr_bracket(double thr, float &lo, float &hi)
{
    const bool plain = thr > 1e-30 && thr < 1e37;
    lo = plain ? (float)(thr * (1.0 - 1.0 / 1048576.0)) : -1.0f;
    hi = plain ? (float)(thr * (1.0 + 1.0 / 1048576.0)) : thr > 1.0 ? INFINITY : thr < 0.0 ? -1.0f : 1e-29f;
}

// The same in fine order (SrcRec, one wave per group of 64), with each group's
// box and thresholds.  A group with a coefficient that must not enter the moments
// gets a smallest threshold that no pair is inside.
__global__ __launch_bounds__(256) void k_prep_fine(int64_t n, const int *perm, const float *xs, const float *ys,
                                                   const float *w_orig, const float *h_orig, const float *ew_orig,
                                                   float h_fixed, SrcRec *out, GroupInfo *grp)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool on = i < n;
    SrcRec r;
    if (on) {
        const int o = perm[i];
        const float h = h_fixed > 0.0f ? h_fixed : (h_orig ? h_orig[o] : 0.0f);
        const double h2 = (double)(float)(h * h);
        r.x = xs[i];
        r.y = ys[i];
        r.coef = r.af = 0.0f;
        r.thr = -1.0;
        r.lo = r.hi = -1.0f;
        if (h2 > 0.0 && h2 < 1e300) {
            r.coef = (float)((double)w_orig[o] * (double)ew_orig[o] / (h2 * (double)MKDE_TWO_PI_F));
            r.af = (float)(-MKDE_LOG2E / (2.0 * h2));
            r.thr = 9.0 * h2;
            thr_bracket(r.thr, r.lo, r.hi);
        }
        out[i] = r;
    }
    float x0 = on ? r.x : FLT_MAX, y0 = on ? r.y : FLT_MAX, x1 = on ? r.x : -FLT_MAX, y1 = on ? r.y : -FLT_MAX;
    double lo = on ? (coef_signed_ok(r.coef) ? r.thr : -1.0) : DBL_MAX, hi = on ? r.thr : -DBL_MAX;
    for (int d = 32; d >= 1; d >>= 1) {
        x0 = fminf(x0, __shfl_xor(x0, d, WAVE));
        x1 = fmaxf(x1, __shfl_xor(x1, d, WAVE));
        y0 = fminf(y0, __shfl_xor(y0, d, WAVE));
        y1 = fmaxf(y1, __shfl_xor(y1, d, WAVE));
        lo = fmin(lo, __shfl_xor(lo, d, WAVE));
        hi = fmax(hi, __shfl_xor(hi, d, WAVE));
    }
    if (on && (threadIdx.x & 63) == 0) grp[i >> 6] = GroupInfo{x0, y0, x1, y1, lo, hi};
}

// Per-bin bounding box of the points and largest threshold.
// One wave per bin (bins in dense clusters hold thousands of points):
// lanes stride over the bin's points, then wave min / max reductions.
__global__ __launch_bounds__(256) void k_bin_stats(int nbins, const int *bin_start, const PtRec *pts, BinInfo *box,
                                                   double *thr)
{
    const int lane = threadIdx.x & 63;
    const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= nbins) return;
    const int s = bin_start[b], e = bin_start[b + 1];
    float x0 = FLT_MAX, y0 = FLT_MAX, x1 = -FLT_MAX, y1 = -FLT_MAX;
    double t = -1.0;
    for (int i = s + lane; i < e; i += 64) {
        const PtRec p = pts[i];
        x0 = fminf(x0, p.x);
        x1 = fmaxf(x1, p.x);
        y0 = fminf(y0, p.y);
        y1 = fmaxf(y1, p.y);
        t = fmax(t, p.thr);
    }
    for (int d = 32; d >= 1; d >>= 1) {
        x0 = fminf(x0, __shfl_xor(x0, d, WAVE));
        x1 = fmaxf(x1, __shfl_xor(x1, d, WAVE));
        y0 = fminf(y0, __shfl_xor(y0, d, WAVE));
        y1 = fmaxf(y1, __shfl_xor(y1, d, WAVE));
        t = fmax(t, __shfl_xor(t, d, WAVE));
    }
    if (lane == 0) {
        box[b] = BinInfo{x0, y0, x1, y1};
        thr[b] = t;
    }
}

// Wait states between the matrix cores and the inline-assembly FMAs on the
// same accumulators.  The compiler inserts them between its own instructions
// but not around inline assembly, so both directions are pinned here: the
// asm statements name the accumulators as operands, which keeps them between
// the producer and the consumer.  A VALU write of a VGPR needs 2 wait states
// before an MFMA reads it as SrcC (5 here); a 16-pass MFMA result needs 18
// before a VALU instruction reads it (24 here).
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define MKDE_ACC16(a)                                                                                                 \
    "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(a[8]),     \
        "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15])
__device__ __forceinline__ void wait_valu_to_mfma(float (&a)[16]) { asm volatile("s_nop 4" : MKDE_ACC16(a)); }
__device__ __forceinline__ void wait_mfma_to_valu(float (&a)[16]) { asm volatile("s_nop 15\ns_nop 7" : MKDE_ACC16(a)); }

// Reach of one raster row for one point: the smallest float f >= 0 with
// fl64(f^2 + dy2) >= thr.  f^2 is exact in FP64 and the sum is monotone in f,
// so a cell of the row is inside the cut-off fl64(dx2 + dy2) < thr exactly
// when |fl32(cx - px)| < f; f = 0 when no cell of the row is inside.  The
// hardware FP64 square root (within about one FP32 ulp) only seeds the search.
// The answer is almost always the seed or the float after it, which two
// evaluations of the exact predicate settle without a loop: inside(seed)
// says which of the two it can be, and the predicate at the neighbour on the
// other side confirms it.  Anything else walks by single ulps.  v^2 is exact
// in FP64 for a float v, so fma(v, v, dy2) rounds once, like fl64(v^2 + dy2).
__device__ __forceinline__ float row_reach(double dy2, double thr)
{
    auto inside = [&](float v) { return __fma_rn((double)v, (double)v, dy2) < thr; };
    auto up = [](float v) { return __uint_as_float(__float_as_uint(v) + 1u); };
    auto down = [](float v) { return __uint_as_float(__float_as_uint(v) - 1u); };
    const bool any = dy2 < thr;
    float f = (float)__builtin_amdgcn_sqrt(fmax(thr - dy2, 0.0));
    // c0: the answer is above f; then f' = up(f) must be outside, else
    // f' = f must have down(f) inside (f > 0: inside(0) holds when any)
    const bool c0 = inside(f);
    const float t = c0 ? up(f) : down(f);
    const bool ok = f > 0.0f && (inside(t) != c0);
    if (__builtin_expect(!any || ok, 1)) return any ? (c0 ? t : f) : 0.0f;
    for (int k = 0; k < 4096 && inside(f); ++k) f = up(f);
    for (int k = 0; k < 4096 && f > 0.0f && !inside(down(f)); ++k) f = down(f);
    return f;
}

// Accumulators R..R+3 of a PARTIAL sub-block: m_i = |dx| < reach_i ? ex : 0
// (the exact cut-off, row_reach), then acc[R+i] += Ey[R+i] * m_i.  Ey of a
// wave's 16 accumulator rows lives in one VGPR (lane l holds the row of
// accumulator l & 15, the same 16 rows in every 16-lane row of the wave), and
// DPP row_newbcast:j hands accumulator j's value to the lanes as the FMA's
// first operand instead of a 64-lane LDS broadcast read per value.  The four
// lane masks go to four SGPR pairs and the four m_i are formed before the
// four DPP FMAs, so each m_i is at least 2 VALU instructions old when it is
// read (the wait states a DPP read needs after a VALU write).
#define MKDE_XCMP(I) "v_cmp_gt_f32_e64 %[s" #I "], %[x" #I "], |%[dx]|\n"
#define MKDE_XSEL(I) "v_cndmask_b32_e64 %[m" #I "], 0, %[ex], %[s" #I "]\n"
#define MKDE_XFMA(I, J) "v_fmac_f32_dpp %[a" #I "], %[ey], %[m" #I "] row_newbcast:" #J " row_mask:0xf bank_mask:0xf\n"
#define MKDE_PART4(R0, R1, R2, R3)                                                                                    \
    __device__ __forceinline__ void part4_##R0(float &a0, float &a1, float &a2, float &a3, float4 x, float ex,         \
                                               float eyv, float dx)                                                   \
    {                                                                                                                 \
        float m0, m1, m2, m3;                                                                                         \
        uint64_t s0, s1, s2, s3;                                                                                      \
        asm(MKDE_XCMP(0) MKDE_XCMP(1) MKDE_XCMP(2) MKDE_XCMP(3) MKDE_XSEL(0) MKDE_XSEL(1) MKDE_XSEL(2) MKDE_XSEL(3)   \
                MKDE_XFMA(0, R0) MKDE_XFMA(1, R1) MKDE_XFMA(2, R2) MKDE_XFMA(3, R3)                                   \
            : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [m0] "=&v"(m0), [m1] "=&v"(m1),             \
              [m2] "=&v"(m2), [m3] "=&v"(m3), [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2), [s3] "=&s"(s3)          \
            : [x0] "v"(x.x), [x1] "v"(x.y), [x2] "v"(x.z), [x3] "v"(x.w), [ex] "v"(ex), [ey] "v"(eyv), [dx] "v"(dx));   \
    }
MKDE_PART4(0, 1, 2, 3)
MKDE_PART4(4, 5, 6, 7)
MKDE_PART4(8, 9, 10, 11)
MKDE_PART4(12, 13, 14, 15)

// ======================================================== density raster ====
//
// One workgroup computes a block of 64 x MKDE_DT_BW cells of a tile (64 x 64,
// 256 threads).  Each wave owns a 32x32 quadrant (lane layout below), each
// lane one column of it and 16 of its rows (16 accumulators).
// Blocks without a valid cell only copy the mask's nodata values.
// The workgroup walks the candidate bins, classifies every point of those
// bins against the block exactly (EMPTY: no cell inside the cut-off; FULL:
// every cell inside; PARTIAL), queues the non-empty ones in bin order, and
// consumes them in sub-batches of DT_SB points:
//   1. cooperatively, in LDS: Ex[p][col] = exp2(dx2 a_p) for the 64 columns,
//      Ey[p][row] = coef_p exp2(dy2 a_p) for the 64 rows, and for PARTIAL
//      points the exact reach of each row (row_reach) and the class of each
//      wave's sub-block (the same exact EMPTY / FULL test on the
//      smaller rectangle);
//   2. each wave adds Ex * Ey[p][row] to its 16 cells with one FMA each
//      (FULL), or with Ex replaced by 0 on the lanes with |dx| >= reach[p][row]
//      (PARTIAL: the exact cut-off fl64(dx2 + dy2) < thr), and skips EMPTY
//      sub-blocks;
//   3. the FP32 partial sums are added to FP64 cell sums after every DT_FOLD
//      sub-batches.
// The order of points is fixed (bins in row-major order, points in bin order)
// so results are deterministic.

#define DT_SB 32
#define DT_EYP 68   // floats per point row of the Ey and reach tables (64 + pad)
#define DT_Q (DT_SB + DT_NT)
// Sub-batches summed in FP32 before the fold into FP64: at most 64 positive
// terms, a relative error below 64 * 2^-24 = 3.8e-6 per fold
#define DT_FOLD 2

// stats[0] candidate points classified, [1] FULL blocks, [2] PARTIAL blocks,
// [3] FULL / [4] PARTIAL / [5] EMPTY wave sub-blocks of PARTIAL points,
// [6] blocks skipped (no valid cell)
#define DT_NSTATS 8

// Lane -> cells of a wave: the block's 64 x MKDE_DT_BW cells are DT_QX x 2
// quadrants of 32 x 32, wave w covering the one at column 32 (w % DT_QX), row
// 32 (w / DT_QX); lane l holds column 32 (w % DT_QX) + (l & 31) and, in
// accumulator j < 16, row 32 (w / DT_QX) + 8 (j >> 2) + 4 (l >> 5) + (j & 3):
// the accumulator layout of v_mfma_f32_32x32x2_f32.  Accumulators 4g .. 4g+3
// of a lane are four consecutive rows, and the lanes of one 16-lane DPP row
// all hold the same 16 rows.
#define DT_QX (MKDE_DT_BW / 32)
#define DT_NW (2 * DT_QX)   // waves per workgroup
#define DT_NT (64 * DT_NW)  // threads per workgroup
#define DT_WX0(w) (32 * ((w) % DT_QX))
#define DT_WY0(w) (32 * ((w) / DT_QX))
#define DT_WC(w, l) (DT_WX0(w) + ((l) & 31))
#define DT_ROW(w, l, j) (DT_WY0(w) + 8 * ((j) >> 2) + 4 * ((l) >> 5) + ((j) & 3))
#define DT_WNX 32
#define DT_WNY 32

// Raster of one or more tiles.  Single tile: g holds the tile geometry.
// Tiled (tl.tw > 0): g.ncols / g.nrows are the raster size and each tile takes
// its origin from the raster geotransform as AsciiRasterFromGeoTIFFTile does
// for a GeoTIFF tile (tiled:2218-2220, GeoTIFF.cpp:190-195):
//   xll = fl32(gt0 + gt1*xoff), yll = fl32((gt3 + gt5*yoff) + rows*gt5), cs = fl32(gt1).
// A work item is one part of a 64x64 block: {block, part j, parts K, partial
// slot (K > 1) or -1}.  A block whose candidate count exceeds the split
// threshold is cut into K parts by candidate ordinal (the position of a point
// in the block's bin-order candidate sequence): part j takes ordinals
// [C j / K, C (j+1) / K) of the C candidates and writes FP64 partial sums to
// its slot; k_density_merge adds the K partials in part order.  Items are
// visited heaviest first (order[]).
struct TileArgs {
    GridDesc g;
    const float *mask;   // raster values (nullable: all valid)
    float *out;
    PointIndex idx;
    unsigned long long *stats;   // nullable
    const int *order;            // nullable: items in raster order, one per block
    const int4 *items;           // with order: work items
    const unsigned *cost;        // with order: candidate count of each block
    double *partials;            // MKDE_DT_CELLS per slot
    int nbx;                     // density blocks per raster row
    Tiling tl;
    double *nodes;               // per item DN_N x DN_N sums of wide kernels
    int *node_on;                // per item: whether it has them
};

// Geometry of one 64x64 block: global cell range [c0,c1]x[r0,r1], and the
// origin of the tile it belongs to (block-local cell index = global - off).
struct BlockGeom {
    int64_t c0, r0, c1, r1, xoff, yoff;
    double xll, yll, cs, nrm05;
};

__device__ __forceinline__ BlockGeom block_geom(const GridDesc &g, const Tiling &tl, int nbx, int blk)
{
    BlockGeom b;
    if (tl.tw > 0) {
        const int t = blk / tl.bpt, lb = blk - t * tl.bpt;
        b.xoff = (int64_t)(t % tl.ntx) * tl.tw;
        b.yoff = (int64_t)(t / tl.ntx) * tl.th;
        const int64_t tcols = (tl.tw < g.ncols - b.xoff) ? tl.tw : g.ncols - b.xoff;
        const int64_t trows = (tl.th < g.nrows - b.yoff) ? tl.th : g.nrows - b.yoff;
        b.c0 = b.xoff + (int64_t)(lb % tl.bpx) * MKDE_DT_BW;
        b.r0 = b.yoff + (int64_t)(lb / tl.bpx) * 64;
        b.c1 = (b.c0 + MKDE_DT_BW - 1 < b.xoff + tcols - 1) ? b.c0 + MKDE_DT_BW - 1 : b.xoff + tcols - 1;
        b.r1 = (b.r0 + 63 < b.yoff + trows - 1) ? b.r0 + 63 : b.yoff + trows - 1;
        const double g0 = tl.gt0 + tl.gt1 * (double)b.xoff;
        const double g3 = tl.gt3 + tl.gt5 * (double)b.yoff;
        b.xll = (double)(float)g0;
        b.yll = (double)(float)(g3 + (double)trows * tl.gt5);
        b.cs = (double)(float)tl.gt1;
        b.nrm05 = (double)trows - 0.5;
    } else {
        b.c0 = (int64_t)(blk % nbx) * MKDE_DT_BW;
        b.r0 = (int64_t)(blk / nbx) * 64;
        b.c1 = (b.c0 + MKDE_DT_BW - 1 < g.ncols - 1) ? b.c0 + MKDE_DT_BW - 1 : g.ncols - 1;
        b.r1 = (b.r0 + 63 < g.nrows - 1) ? b.r0 + 63 : g.nrows - 1;
        b.xoff = b.yoff = 0;
        b.xll = g.xll;
        b.yll = g.yll;
        b.cs = g.cs;
        b.nrm05 = (double)g.nrows - 0.5;
    }
    return b;
}

// Wide kernels at nodes.  A block-FULL point whose bandwidth is not small against
// the block is smooth over it: the sum of all such points is formed at 16 x 16
// Chebyshev nodes of the block instead of its 64 x 64 cells, one 16 x 16 x 4 MFMA
// for four points, and interpolated to the cells once at the end (FP64).  For h >=
// half extent / (2 DN_KAPPA) (24 cells) the interpolant of a point is within
// 4.4e-9 of its value anywhere in the block.  A cell's weights have a root sum of
// squares of 1 on average, 1.39 at most in each direction (1.94 in a corner), by
// which rounding at the nodes can grow; the nodes fold into FP64 every 16 points,
// and the error against 64 bits came out no larger than at the cells.  Per point and
// block: 0.25 MFMA of 8 passes, 10 VALU instructions and 1.3 lane permutations,
// where the cells take 2 MFMA of 16 passes and 30 instructions.  Every wave walks
// the candidate bins by itself, without barriers, and takes every fourth 64 points.
// Bound by instruction issue.  A kernel of its own: inside k_density_tile, whose
// registers and scalars it then shares, everything else took 10% longer.
// 1M points, adaptive bandwidths, 8192^2 cells: 23.6 ms with all points at the
// cells, 1.6 + 15.7 ms now.  Rasters of few candidates an item (MKDE_DN_SPLIT)
// keep to the cells: 50,000 points on 2048^2 took 405 us there and 464 us here.
#define DN_N 16
#define DN_KAPPA 0.65
// Candidates of an item from which on its bins are searched for such points, and
// points from which on the interpolation (about 1200 instructions a wave) pays.
#define DN_CAND 2048
#define DN_MIN 192
// Smallest cut-off threshold 9 h^2 of a point that goes to the nodes
// (MKDE_DN_REACH: its root for a whole block, in cells).
__device__ __forceinline__ double dn_thr_min(double L) { return L * L * (9.0 / (4.0 * DN_KAPPA * DN_KAPPA)) * 0.999999; }

__device__ __forceinline__ double dn_node(int j)
{
    const int i = j < 8 ? j : 15 - j;
    const double c = i == 0   ? 0.99518472667219692873
                     : i == 1 ? 0.95694033573220882438
                     : i == 2 ? 0.88192126434835504956
                     : i == 3 ? 0.77301045336273699338
                     : i == 4 ? 0.63439328416364548779
                     : i == 5 ? 0.47139673682599780857
                     : i == 6 ? 0.29028467725446233105
                              : 0.09801714032956077016;   // cos((2i + 1) pi / 32)
    return j < 8 ? c : -c;
}

// Centre and half extent of a block's node grid.
struct BlockNodes {
    double mx, my, L;
};
__device__ __forceinline__ BlockNodes block_nodes(float bx0, float bx1, float by0, float by1, double cs)
{
    return BlockNodes{0.5 * ((double)bx0 + (double)bx1), 0.5 * ((double)by0 + (double)by1),
                      0.5 * fmax(fmax((double)bx1 - (double)bx0, (double)by1 - (double)by0), 0.5 * cs)};
}

// Whether a point that is FULL for a block of half extent L goes to the nodes:
// L <= 2 DN_KAPPA h, a = -log2(e) / (2 h^2).
__device__ __forceinline__ bool dn_wide(const PtRec &p, double L)
{
    return L * L * -p.a <= 2.0 * DN_KAPPA * DN_KAPPA * MKDE_LOG2E && coef_signed_ok(p.coef);
}

// Interpolation weights of a cell at v (centre mid, half extent L) to w[64 j],
// barycentric: w_j = b_j / (x - x_j) / sum, b_j = (-1)^j sin((2j + 1) pi / 32).
__device__ __forceinline__ void dn_weights(double v, double mid, double L, double *w)
{
    const double x = (v - mid) / L;
    double t[DN_N], sum = 0.0;
    int hit = -1;
#pragma unroll
    for (int j = 0; j < DN_N; ++j) {
        const double d = x - dn_node(j);
        if (d == 0.0) hit = j;
        const double b = dn_node(j < 8 ? 7 - j : j - 8);   // the sine
        t[j] = ((j & 1) ? -b : b) / d;
        sum += t[j];
    }
    const double r = 1.0 / sum;
#pragma unroll
    for (int j = 0; j < DN_N; ++j) w[64 * j] = hit < 0 ? t[j] * r : hit == j ? 1.0 : 0.0;
}

// This wave's share of the node sums of an item: lane l, entry v of s is row node
// 4 (l >> 4) + v, column node l & 15 (the accumulator layout of
// v_mfma_f32_16x16x4_f32).  Returns the points summed.  win0 .. win1 - 1: the
// item's candidate ordinals (split: there are others).
__device__ __forceinline__ int dn_sums(const PointIndex &I, int bxa, int bxb, int bya, int byb, bool split, int64_t win0,
                                       int64_t win1, float bx0, float bx1, float by0, float by1, double mx, double my,
                                       double L, double (&s)[4])
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double nx = mx + L * dn_node(lane & 15), ny = my + L * dn_node(lane & 15);
    const int nbx_r = bxb - bxa + 1, nb_total = nbx_r * (byb - bya + 1);
    // no point of a bin is wide enough when its largest threshold is not
    const double thr_min = dn_thr_min(L);
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] = 0.0;
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
    int terms = 0, total = 0, turn = 0;   // turn: 64s of points seen, of all waves
    int64_t ord = 0;
    for (int base = 0; base < nb_total; base += 64) {
        const int k = base + lane;
        const int kc = k < nb_total ? k : nb_total - 1;
        const int b = (bya + kc / nbx_r) * I.bg.nbx + (bxa + kc % nbx_r);
        int p0 = I.bin_start[b], p1 = I.bin_start[b + 1];
        const double lim = I.bin_thr[b];
        bool on = k < nb_total && p1 > p0 && box_gap2(I.bin_box[b], bx0, bx1, by0, by1) < lim;
        if (split) {
            const int cnt = on ? p1 - p0 : 0;
            const unsigned incl = wave_incl_scan((unsigned)cnt, lane);
            const int64_t o1 = ord + incl, o0 = o1 - cnt;
            ord += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
            on = on && o1 > win0 && o0 < win1;
            if (win1 < o1) p1 -= (int)(o1 - win1);
            if (win0 > o0) p0 += (int)(win0 - o0);
        }
        uint64_t m = __ballot(on && lim >= thr_min);
        while (m) {
            const int l = __builtin_ctzll(m);
            m &= m - 1ull;
            const int a = __builtin_amdgcn_readlane(p0, l), e = __builtin_amdgcn_readlane(p1, l);
            for (int st = a; st < e; st += 64) {
                if ((turn++ & 3) != wave) continue;
                const int i = st + lane;
                PtRec p{};
                bool take = false;
                if (i < e) {
                    p = I.pts[i];
                    take = p.thr > 0.0 && dn_wide(p, L) && sq2(far1(p.x, bx0, bx1), far1(p.y, by0, by1)) < p.thr;
                }
                const uint64_t tm = __ballot(take);
                if (!tm) continue;
                const int cnt = __popcll(tm);
                total += cnt;
                // taken points to the front lanes, the others behind them
                const uint64_t below = ((uint64_t)1 << lane) - 1;
                const int to = 4 * (take ? __popcll(tm & below) : cnt + __popcll(~tm & below));
                const double pa = p.a;
                const int alo = __builtin_amdgcn_ds_permute(to, __double2loint(pa));
                const int ahi = __builtin_amdgcn_ds_permute(to, __double2hiint(pa));
                const int px = __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, p.x));
                const int py = __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, p.y));
                const int pc = __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, take ? p.coef : 0.0f));
                for (int g = 0; g < cnt; g += 4) {
                    // lane l: point g + l / 16 (past the end: one without a weight)
                    const int from = 4 * (g + (lane >> 4));
                    const double qa = __hiloint2double(__builtin_amdgcn_ds_bpermute(from, ahi),
                                                       __builtin_amdgcn_ds_bpermute(from, alo));
                    const float qx = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, px));
                    const float qy = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, py));
                    const float qc = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, pc));
                    const bool in = g + (lane >> 4) < cnt;
                    const double dx = nx - (double)qx, dy = ny - (double)qy;
                    const float ex = fast_exp2((float)(dx * dx * qa)), ey = fast_exp2((float)(dy * dy * qa)) * qc;
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? ey : 0.0f, in ? ex : 0.0f, c, 0, 0, 0);
                    if (++terms == 4) {   // 16 terms in FP32
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            s[v] += (double)c[v];
                            c[v] = 0.0f;
                        }
                        terms = 0;
                    }
                }
            }
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] += (double)c[v];
    return total;
}

// Node sums of every item that has enough candidates and such points.
__global__ __launch_bounds__(DT_NT) void k_density_nodes(TileArgs A)
{
    static_assert(DT_NW == 4 && DN_N * DN_N == DT_NT, "a node per thread");
    __shared__ double s_part[DT_NW * DN_N * DN_N];
    __shared__ int s_cnt[DT_NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int at = A.order[blockIdx.x];
    const int4 item = A.items[at];
    const int64_t C = A.cost[item.x];
    const BlockGeom B = block_geom(A.g, A.tl, A.nbx, item.x);
    const int64_t lc0 = B.c0 - B.xoff, lr0 = B.r0 - B.yoff, lc1 = B.c1 - B.xoff, lr1 = B.r1 - B.yoff;
    const float bx0 = cell_x(B.xll, B.cs, lc0), bx1 = cell_x(B.xll, B.cs, lc1);
    const float by1 = cell_y(B.yll, B.cs, B.nrm05, lr0), by0 = cell_y(B.yll, B.cs, B.nrm05, lr1);
    const BlockNodes bn = block_nodes(bx0, bx1, by0, by1, B.cs);
    const double reach = *A.idx.reach_p;
    if (C / item.z < DN_CAND || reach * reach < dn_thr_min(bn.L)) {
        if (tid == 0) A.node_on[at] = 0;
        return;
    }
    int64_t win0 = 0, win1 = INT64_MAX;
    if (item.y > 0) win0 = C * item.y / item.z;
    if (item.y < item.z - 1) win1 = C * (item.y + 1) / item.z;
    int bxa, bxb, bya, byb;
    bin_range(A.idx.bg, bx0, bx1, by0, by1, reach, bxa, bxb, bya, byb);
    double s[4];
    const int got = dn_sums(A.idx, bxa, bxb, bya, byb, item.z > 1, win0, win1, bx0, bx1, by0, by1, bn.mx, bn.my, bn.L, s);
#pragma unroll
    for (int v = 0; v < 4; ++v) s_part[wave * 256 + (4 * (lane >> 4) + v) * DN_N + (lane & 15)] = s[v];
    if (lane == 0) s_cnt[wave] = got;
    __syncthreads();
    const bool on = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3] >= DN_MIN;
    if (tid == 0) A.node_on[at] = on;
    if (on) A.nodes[(int64_t)at * (DN_N * DN_N) + tid] = ((s_part[tid] + s_part[256 + tid]) + s_part[512 + tid]) + s_part[768 + tid];
}

// 4 waves per SIMD: at most 128 VGPRs (no spills).  64 x 64 blocks: 37.7 KB
// of LDS per workgroup, 4 workgroups per CU, so each SIMD's 4 waves belong to
// 4 workgroups and a barrier wait in one leaves 3 to issue.  (64 x 128
// blocks share Ey and the reach over twice the columns, but at 55 KB and 8
// waves only 2 workgroups fit per CU: measured 31.6 ms against 24.3 ms on
// the adaptive 1M job.)
template <bool STATS, bool NODES>
__global__ __launch_bounds__(DT_NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_density_tile(TileArgs A)
{
    __shared__ int s_bins[DT_NT];
    __shared__ int s_wcnt[DT_NW];
    __shared__ unsigned s_queue[DT_Q];   // point index | 0x80000000 for block-PARTIAL
    // records of the queued points, stored when they are classified, so a
    // sub-batch reads its parameters from LDS instead of global memory
    __shared__ float s_qx[DT_Q], s_qy[DT_Q], s_qc[DT_Q];
    __shared__ double s_qa[DT_Q], s_qt[DT_Q];
    __shared__ float s_px[DT_SB];
    __shared__ float s_py[DT_SB];
    __shared__ float s_coef[DT_SB];
    __shared__ double s_a[DT_SB];
    __shared__ double s_thr[DT_SB];
    __shared__ int s_wcls[DT_SB];   // 2 bits per wave: 0 skip, 1 full, 2 partial
    __shared__ int s_nfull;         // block-FULL points at the front of the sub-batch
    __shared__ __attribute__((aligned(16))) float s_ex[DT_SB * MKDE_DT_BW];
    __shared__ __attribute__((aligned(16))) float s_ey[DT_SB * DT_EYP];
    __shared__ __attribute__((aligned(16))) float s_xr[DT_SB * DT_EYP];   // row reach, PARTIAL points
    __shared__ float s_ccx[MKDE_DT_BW], s_ccy[64];   // cell-centre x of the block's columns, y of its rows
    __shared__ float s_wyb[2 * DT_NW];               // y of the first / last row of each wave's sub-block
    __shared__ float s_wxb[2 * DT_NW];               // x of the first / last column of each wave's sub-block

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const GridDesc g = A.g;
    int4 item = make_int4((int)blockIdx.x, 0, 1, -1);
    if (A.order) {
        const int at = A.order[blockIdx.x];
        if (A.node_on && (A.node_on[at] != 0) != NODES) return;   // the other form's
        item = A.items[at];
    }
    const int blk = item.x;
    // candidate-ordinal window of this part
    int64_t win0 = 0, win1 = INT64_MAX;
    if (item.z > 1) {
        // the first and last parts are open-ended, so the parts always cover
        // the whole candidate sequence
        const int64_t C = A.cost[blk];
        if (item.y > 0) win0 = C * item.y / item.z;
        if (item.y < item.z - 1) win1 = C * (item.y + 1) / item.z;
    }
    const BlockGeom B = block_geom(g, A.tl, A.nbx, blk);
    const double xll = B.xll, yll = B.yll, cs = B.cs, nrm05 = B.nrm05;
    const int64_t c0 = B.c0, r0 = B.r0, c1 = B.c1, r1 = B.r1;
    // tile-local indices for cell centres
    const int64_t lc0 = c0 - B.xoff, lr0 = r0 - B.yoff, lc1 = c1 - B.xoff, lr1 = r1 - B.yoff;
    const int wc = DT_WC(wave, lane);   // this lane's column
    const int64_t col = c0 + wc;

    // validity of this thread's cells; blocks without a valid cell are skipped
    unsigned vbits = 0;
    if (col <= c1) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int64_t row = r0 + DT_ROW(wave, lane, j);
            if (row <= r1) {
                bool v = true;
                if (A.mask) v = A.mask[row * g.ncols + col] != g.nodata;
                vbits |= (v ? 1u : 0u) << j;
            }
        }
    }
    if (!__syncthreads_or(vbits != 0)) {
        if (col <= c1) {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int64_t row = r0 + DT_ROW(wave, lane, j);
                if (row <= r1) A.out[row * g.ncols + col] = A.mask[row * g.ncols + col];
            }
        }
        if (STATS && tid == 0) atomicAdd(&A.stats[6], 1ull);
        return;
    }

    // Block extent in cell-centre coordinates (exact N2 floats).
    const float bx0 = cell_x(xll, cs, lc0), bx1 = cell_x(xll, cs, lc1);
    const float by1 = cell_y(yll, cs, nrm05, lr0), by0 = cell_y(yll, cs, nrm05, lr1);
    const float cx = cell_x(xll, cs, lc0 + wc);
    {
        // thread ranges (even starts): columns, rows, then per wave [0] first /
        // [1] last row and [0] first / [1] last column of its quadrant
        constexpr int T1 = MKDE_DT_BW, T2 = T1 + 64, T3 = T2 + 2 * DT_NW, T4 = T3 + 2 * DT_NW;
        static_assert(T4 <= DT_NT, "too few threads for the block tables");
        if (tid < T1) s_ccx[tid] = cell_x(xll, cs, lc0 + tid);
        else if (tid < T2) s_ccy[tid - T1] = cell_y(yll, cs, nrm05, lr0 + (tid - T1));
        else if (tid < T3) {
            const int w = (tid - T2) >> 1;
            const int64_t wr0 = lr0 + DT_WY0(w);
            const int64_t wr1 = (wr0 + DT_WNY - 1 < lr1) ? wr0 + DT_WNY - 1 : lr1;
            s_wyb[tid - T2] = (tid & 1) ? cell_y(yll, cs, nrm05, wr1) : cell_y(yll, cs, nrm05, wr0);
        } else if (tid < T4) {
            const int w = (tid - T3) >> 1;
            const int64_t wc0 = lc0 + DT_WX0(w);
            const int64_t wc1 = (wc0 + DT_WNX - 1 < lc1) ? wc0 + DT_WNX - 1 : lc1;
            s_wxb[tid - T3] = (tid & 1) ? cell_x(xll, cs, wc1) : cell_x(xll, cs, wc0);
        }
    }

    // FP32 partial sums (at most DT_FOLD sub-batches of terms) folded into
    // FP64 cell sums
    float acc[16];
    double sum[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) { acc[j] = 0.0f; sum[j] = 0.0; }
    unsigned st_cand = 0, st_full = 0, st_part = 0, st_wf = 0, st_wp = 0, st_we = 0;

    const PointIndex &I = A.idx;
    int bxa, bxb, bya, byb;
    bin_range(I.bg, bx0, bx1, by0, by1, *I.reach_p, bxa, bxb, bya, byb);
    const int nbx_r = bxb - bxa + 1;
    const int nb_total = nbx_r * (byb - bya + 1);

    // wide kernels at the nodes (k_density_nodes)
    const BlockNodes bn = block_nodes(bx0, bx1, by0, by1, cs);
    int qn = 0;       // queue length (uniform)
    int npend = 0;    // sub-batches in acc since the last fold (uniform)
    auto fold = [&]() {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            sum[j] += (double)acc[j];
            acc[j] = 0.0f;
        }
        npend = 0;
    };
    int64_t ord = 0;  // candidate ordinal at the start of the next candidate bin (uniform)

    auto process = [&](int cnt, int head) {
        // 1a. point parameters of queue entries [head, head + cnt), block-FULL
        //     points first (stable partition, so the order stays
        //     deterministic); cnt <= DT_SB <= 64: one wave
        if (tid < 64) {
            const int e = head + tid;
            const unsigned q = tid < cnt ? s_queue[e] : 0u;
            const bool isfull = tid < cnt && !(q >> 31);
            const uint64_t fm = __ballot(isfull);
            const uint64_t below = (1ull << tid) - 1ull;
            const int nf = __popcll(fm);
            const int slot = isfull ? __popcll(fm & below) : nf + (tid - __popcll(fm & below));
            if (tid == 0) s_nfull = nf;
            if (tid < cnt) {
                const float px = s_qx[e], py = s_qy[e];
                const double thr = s_qt[e];
                const int t = slot;
                s_px[t] = px;
                s_py[t] = py;
                s_coef[t] = s_qc[e];
                s_a[t] = s_qa[e];
                s_thr[t] = thr;
                // wave sub-block classes
                // 2 bits per wave: 0 skip, 1 full, 2 partial
                int cl4 = (int)(0x55555555u >> (32 - 2 * DT_NW));
                if (q >> 31) {
                    cl4 = 0;
#pragma unroll
                    for (int w = 0; w < DT_NW; ++w) {
                        int cw = 0;
                        if (lr0 + DT_WY0(w) <= lr1 && lc0 + DT_WX0(w) <= lc1) {
                            const float wy1 = s_wyb[2 * w], wy0 = s_wyb[2 * w + 1];
                            const float wx0 = s_wxb[2 * w], wx1 = s_wxb[2 * w + 1];
                            const float fx = far1(px, wx0, wx1), nx = gap1(px, wx0, wx1);
                            if (sq2(nx, gap1(py, wy0, wy1)) < thr) cw = sq2(fx, far1(py, wy0, wy1)) < thr ? 1 : 2;
                        }
                        cl4 |= cw << (2 * w);
                    }
                }
                s_wcls[t] = cl4;
            }
        }
        __syncthreads();
        // 1b. tables: lane -> row / column slot, wave -> DT_SB / DT_NW points;
        //     consecutive lanes write consecutive LDS words (no bank
        //     conflicts).  Ey and the reach of a row serve every column of
        //     the block, so a wider block shares them.
        const int nfull = s_nfull;
        {
            const float cyr = s_ccy[lane];
            float cxr[MKDE_DT_BW / 64];
#pragma unroll
            for (int cb = 0; cb < MKDE_DT_BW / 64; ++cb) cxr[cb] = s_ccx[lane + 64 * cb];
            // the point index is wave-uniform: made explicit (scalar index
            // and bound test, fewer VALU address operations)
            const int pw = __builtin_amdgcn_readfirstlane(wave) * (DT_SB / DT_NW);
#pragma unroll 2
            for (int q = 0; q < DT_SB / DT_NW; ++q) {
                const int p = pw + q;
                if (p < cnt) {
                    const float py = s_py[p], px = s_px[p], coef = s_coef[p];
                    const double a = s_a[p];
                    const double dy2 = sqd(cyr - py);
                    s_ey[p * DT_EYP + lane] = fast_exp2((float)(dy2 * a)) * coef;
#pragma unroll
                    for (int cb = 0; cb < MKDE_DT_BW / 64; ++cb)
                        s_ex[p * MKDE_DT_BW + lane + 64 * cb] = fast_exp2((float)(sqd(cxr[cb] - px) * a));
                    if (p >= nfull) s_xr[p * DT_EYP + lane] = row_reach(dy2, s_thr[p]);
                }
            }
        }
        __syncthreads();
        // 2a. this wave's FULL points on the matrix cores: the quadrant's
        //     cells += Ey (32 rows x 2 points) * Ex (2 points x 32 columns),
        //     one v_mfma_f32_32x32x2_f32 per two points, lane l feeding row /
        //     column l & 31 of the pair's point l >> 5 (0 for a missing
        //     second point).  FULL are the block-FULL points [0, nfull) and
        //     the block-PARTIAL points whose class for this wave is FULL;
        //     the classes come as two wave-uniform bit masks over the
        //     sub-batch's PARTIAL points.
        const int np = cnt - nfull;   // <= DT_SB
        const int wcl = lane < np ? (s_wcls[nfull + lane] >> (2 * wave)) & 3 : 0;
        const uint64_t mf = __ballot(wcl == 1);
        uint64_t mp = __ballot(wcl == 2);
        if (STATS && lane == 0) {
            st_wf += nfull + __popcll(mf);
            st_wp += __popcll(mp);
            st_we += np - __popcll(mf) - __popcll(mp);
        }
        if (nfull > 0 || mf) {
            wait_valu_to_mfma(acc);
            f32x16 c;
#pragma unroll
            for (int j = 0; j < 16; ++j) c[j] = acc[j];
            const int k = lane >> 5, li = lane & 31;
            const float *eyp = s_ey + DT_WY0(wave) + li, *exp = s_ex + DT_WX0(wave) + li;
            // block-FULL points eight, then four per step (the later pairs'
            // operands arrive while the first pair's MFMA runs), then the
            // rest in pairs
            int p = 0;
            for (; p + 8 <= nfull; p += 8) {
                const float ey0 = eyp[(p + k) * DT_EYP], ex0 = exp[(p + k) * MKDE_DT_BW];
                const float ey1 = eyp[(p + 2 + k) * DT_EYP], ex1 = exp[(p + 2 + k) * MKDE_DT_BW];
                const float ey2 = eyp[(p + 4 + k) * DT_EYP], ex2 = exp[(p + 4 + k) * MKDE_DT_BW];
                const float ey3 = eyp[(p + 6 + k) * DT_EYP], ex3 = exp[(p + 6 + k) * MKDE_DT_BW];
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey0, ex0, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey1, ex1, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey2, ex2, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey3, ex3, c, 0, 0, 0);
            }
            for (; p + 4 <= nfull; p += 4) {
                const float ey0 = eyp[(p + k) * DT_EYP], ex0 = exp[(p + k) * MKDE_DT_BW];
                const float ey1 = eyp[(p + 2 + k) * DT_EYP], ex1 = exp[(p + 2 + k) * MKDE_DT_BW];
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey0, ex0, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(ey1, ex1, c, 0, 0, 0);
            }
            uint64_t rest = (((1ull << (nfull - p)) - 1ull) << p) | (mf << nfull);
            while (rest) {
                const int p0 = __builtin_ctzll(rest);
                rest &= rest - 1ull;
                const int p1 = rest ? __builtin_ctzll(rest) : -1;
                rest &= rest - 1ull;
                const int q = k ? p1 : p0, qs = q < 0 ? 0 : q;
                const float ey = eyp[qs * DT_EYP], ex = exp[qs * MKDE_DT_BW];
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(q >= 0 ? ey : 0.0f, q >= 0 ? ex : 0.0f, c, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[j] = c[j];
            wait_mfma_to_valu(acc);
        }
        // 2b. this wave's PARTIAL points: Ey of the wave's rows as one VGPR
        //     (lane l holds the row of accumulator l & 15, broadcast to its
        //     16-lane DPP row), the FMAs masked by the row reach
        const int eyo = DT_ROW(wave, lane, lane & 15);
        while (mp) {
            const int p = nfull + __builtin_ctzll(mp);
            mp &= mp - 1ull;
            const float ex = s_ex[p * MKDE_DT_BW + wc];
            const float eyv = s_ey[p * DT_EYP + eyo];
            const float dx = cx - s_px[p];
            // rows of accumulators 4g .. 4g+3: a float4 every 8 rows
            const float4 *xr = (const float4 *)&s_xr[p * DT_EYP + DT_ROW(wave, lane, 0)];
            part4_0(acc[0], acc[1], acc[2], acc[3], xr[0], ex, eyv, dx);
            part4_4(acc[4], acc[5], acc[6], acc[7], xr[2], ex, eyv, dx);
            part4_8(acc[8], acc[9], acc[10], acc[11], xr[4], ex, eyv, dx);
            part4_12(acc[12], acc[13], acc[14], acc[15], xr[6], ex, eyv, dx);
        }
        // (with node sums: every sub-batch, so that no raster loses precision)
        if (NODES || ++npend == DT_FOLD) fold();
        __syncthreads();
    };

    for (int base = 0; base < nb_total; base += DT_NT) {
        // candidate bins of this chunk
        const int k = base + tid;
        bool cand = false;
        int b = 0;
        if (k < nb_total) {
            b = (bya + k / nbx_r) * I.bg.nbx + (bxa + k % nbx_r);
            if (I.bin_start[b + 1] > I.bin_start[b]) {
                double g2 = box_gap2(I.bin_box[b], bx0, bx1, by0, by1);
                cand = g2 < I.bin_thr[b];
            }
        }
        int nb;
        int slot = block_compact<DT_NW>(cand, s_wcnt, &nb);
        if (cand) s_bins[slot] = b;
        __syncthreads();
        for (int kb = 0; kb < nb; ++kb) {
            const int bb = s_bins[kb];
            const int bst = I.bin_start[bb], ben = I.bin_start[bb + 1];
            // clip the bin's points to this part's ordinal window
            const int64_t o0 = ord, o1 = ord + (ben - bst);
            ord = o1;
            if (o1 <= win0 || o0 >= win1) continue;
            const int st = bst + (int)(win0 > o0 ? win0 - o0 : 0);
            const int en = ben - (int)(o1 > win1 ? o1 - win1 : 0);
            for (int off = st; off < en; off += DT_NT) {
                const int i = off + tid;
                int cls = 0;   // 0 empty, 1 full, 2 partial
                PtRec p;
                if (i < en) {
                    p = I.pts[i];
                    if (STATS) ++st_cand;
                    if (p.thr > 0.0) {
                        double near2 = sq2(gap1(p.x, bx0, bx1), gap1(p.y, by0, by1));
                        if (near2 < p.thr) {
                            double far2 = sq2(far1(p.x, bx0, bx1), far1(p.y, by0, by1));
                            cls = far2 < p.thr ? 1 : 2;
                        }
                    }
                    if (STATS && cls == 1) ++st_full;
                    if (STATS && cls == 2) ++st_part;
                    if (NODES && cls == 1 && dn_wide(p, bn.L)) {   // summed at the nodes
                        cls = 0;
                        if (STATS) st_wf += DT_NW;
                    }
                }
                int na;
                int pos = block_compact<DT_NW>(cls != 0, s_wcnt, &na);
                if (cls != 0) {
                    const int e = qn + pos;
                    s_queue[e] = (unsigned)i | (cls == 2 ? 0x80000000u : 0u);
                    s_qx[e] = p.x;
                    s_qy[e] = p.y;
                    s_qc[e] = p.coef;
                    s_qa[e] = p.a;
                    s_qt[e] = p.thr;
                }
                __syncthreads();
                qn += na;
                if (qn >= DT_SB) {
                    int head = 0;
                    while (qn - head >= DT_SB) {
                        process(DT_SB, head);
                        head += DT_SB;
                    }
                    // keep the remainder at the front
                    const int rem = qn - head;
                    unsigned v = 0;
                    float vx = 0.0f, vy = 0.0f, vc = 0.0f;
                    double va = 0.0, vt = 0.0;
                    if (tid < rem) {
                        const int e = head + tid;
                        v = s_queue[e];
                        vx = s_qx[e];
                        vy = s_qy[e];
                        vc = s_qc[e];
                        va = s_qa[e];
                        vt = s_qt[e];
                    }
                    __syncthreads();
                    if (tid < rem) {
                        s_queue[tid] = v;
                        s_qx[tid] = vx;
                        s_qy[tid] = vy;
                        s_qc[tid] = vc;
                        s_qa[tid] = va;
                        s_qt[tid] = vt;
                    }
                    __syncthreads();
                    qn = rem;
                }
            }
        }
        __syncthreads();
    }
    if (qn > 0) process(qn, 0);
    if (npend > 0) fold();
    if (NODES) {
        // cell (row, column) += sum_i Wy[i][row] sum_j N[i][j] Wx[j][column]
        static_assert(sizeof(s_ex) >= 64 * DN_N * sizeof(double) && sizeof(s_ey) >= 64 * DN_N * sizeof(double) &&
                          MKDE_DT_BW == 64, "weights of the cells");
        double *wx = (double *)s_ex, *wy = (double *)s_ey;
        const double *N = A.nodes + (int64_t)__builtin_amdgcn_readfirstlane(A.order[blockIdx.x]) * (DN_N * DN_N);
        __syncthreads();
        if (tid < 64) dn_weights((double)s_ccx[tid], bn.mx, bn.L, wx + tid);
        else if (tid < 128) dn_weights((double)s_ccy[tid - 64], bn.my, bn.L, wy + (tid - 64));
        __syncthreads();
#pragma unroll 1
        for (int i = 0; i < DN_N; ++i) {
            double t = 0.0;
#pragma unroll
            for (int j = 0; j < DN_N; ++j) t = __builtin_fma(N[i * DN_N + j], wx[64 * j + wc], t);
#pragma unroll
            for (int j = 0; j < 16; ++j) sum[j] = __builtin_fma(wy[64 * i + DT_ROW(wave, lane, j)], t, sum[j]);
        }
    }

    // write back: nodata cells keep the mask value; parts of a split block
    // leave FP64 partial sums for k_density_merge
    if (item.z > 1) {
        double *pp = A.partials + (int64_t)item.w * MKDE_DT_CELLS;
#pragma unroll
        for (int j = 0; j < 16; ++j) pp[DT_ROW(wave, lane, j) * MKDE_DT_BW + wc] = sum[j];
    } else if (col <= c1) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int64_t row = r0 + DT_ROW(wave, lane, j);
            if (row <= r1) {
                const int64_t ix = row * g.ncols + col;
                A.out[ix] = ((vbits >> j) & 1u) ? (float)sum[j] : A.mask[ix];
            }
        }
    }
    if (STATS) {
        auto put = [&](int slot, unsigned v) {
            unsigned long long t = v;
            for (int d = 32; d >= 1; d >>= 1) t += __shfl_xor(t, d, WAVE);
            if (lane == 0 && t) atomicAdd(&A.stats[slot], t);
        };
        put(0, st_cand);
        put(1, st_full);
        put(2, st_part);
        put(3, st_wf);
        put(4, st_wp);
        put(5, st_we);
    }
}

// Work estimate of each density block: points in the candidate bins (0 for
// blocks without a valid cell), then a heaviest-first visiting order by
// log2 buckets, so the long blocks start early and the launch drains evenly.
__global__ __launch_bounds__(256) void k_block_cost(GridDesc g, const float *mask, PointIndex I, int nbx,
                                                    Tiling tl, unsigned *cost)
{
    __shared__ unsigned s_sum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int blk = blockIdx.x;
    const BlockGeom B = block_geom(g, tl, nbx, blk);
    bool v = false;
    if (mask) {
        // each thread stops at its first valid cell (most blocks are valid
        // from their first row on)
        for (int k = tid; k < MKDE_DT_CELLS && !v; k += 256) {
            const int64_t r = B.r0 + k / MKDE_DT_BW, c = B.c0 + k % MKDE_DT_BW;
            if (r <= B.r1 && c <= B.c1 && mask[r * g.ncols + c] != g.nodata) v = true;
        }
    } else {
        v = B.c0 <= B.c1 && B.r0 <= B.r1;   // edge tiles leave some blocks empty
    }
    const int any = __syncthreads_or(v);
    const float bx0 = cell_x(B.xll, B.cs, B.c0 - B.xoff), bx1 = cell_x(B.xll, B.cs, B.c1 - B.xoff);
    const float by1 = cell_y(B.yll, B.cs, B.nrm05, B.r0 - B.yoff), by0 = cell_y(B.yll, B.cs, B.nrm05, B.r1 - B.yoff);
    unsigned acc = 0;
    if (any) {
        int bxa, bxb, bya, byb;
        bin_range(I.bg, bx0, bx1, by0, by1, *I.reach_p, bxa, bxb, bya, byb);
        const int nbx_r = bxb - bxa + 1;
        const int nb_total = nbx_r * (byb - bya + 1);
        for (int k = tid; k < nb_total; k += 256) {
            const int b = (bya + k / nbx_r) * I.bg.nbx + (bxa + k % nbx_r);
            const int cntb = I.bin_start[b + 1] - I.bin_start[b];
            if (cntb > 0 && box_gap2(I.bin_box[b], bx0, bx1, by0, by1) < I.bin_thr[b]) acc += (unsigned)cntb;
        }
    }
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
    if (lane == 0) s_sum[wave] = acc;
    __syncthreads();
    if (tid == 0) cost[blk] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

__device__ __forceinline__ int cost_bucket(unsigned c)
{
    // 32 buckets, heaviest first: bucket 0 holds the largest costs
    return c == 0 ? 31 : (__clz(c) < 31 ? __clz(c) : 30);
}

// Sum of the K partials of each split block in part order (FP64), rounded once to
// FP32; nodata cells keep the mask value.  splits[k] = {block, slot0, K}.  Bound by
// the partials' bytes: a thread has eight 16-byte loads in flight (cell by cell it
// waited for each part's load: the 8192^2 raster at h = 16, 448 us, now 93 us).
__global__ __launch_bounds__(256) void k_density_merge(GridDesc g, Tiling tl, int nbx, const float *mask,
                                                       const int4 *splits, const double *partials, float *out)
{
    const int4 sp = splits[blockIdx.x];
    const BlockGeom B = block_geom(g, tl, nbx, sp.x);
    constexpr int U = 4;   // pairs of cells of a thread at a time
    for (int k0 = 2 * (int)threadIdx.x; k0 < MKDE_DT_CELLS; k0 += 512 * U) {
        const double *pp = partials + (int64_t)sp.y * MKDE_DT_CELLS + k0;
        double2 t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = make_double2(0.0, 0.0);
#pragma unroll 2
        for (int q = 0; q < sp.z; ++q)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double2 v = *(const double2 *)(pp + (int64_t)q * MKDE_DT_CELLS + 512 * u);
                t[u].x += v.x;
                t[u].y += v.y;
            }
        // row-major cells of the block, two per pair
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int k = k0 + 512 * u + e;
                const int64_t row = B.r0 + k / MKDE_DT_BW, col = B.c0 + k % MKDE_DT_BW;
                if (row > B.r1 || col > B.c1) continue;
                const int64_t ix = row * g.ncols + col;
                const bool valid = !mask || mask[ix] != g.nodata;
                out[ix] = valid ? (float)(e ? t[u].y : t[u].x) : mask[ix];
            }
    }
    static_assert(MKDE_DT_CELLS % (512 * U) == 0, "whole steps");
}

// ---- work lists
//
// cost[b] of every unit (candidates of a density block or of a 64-query wave)
// -> split threshold T, parts[b] = cost > T ? ceil(cost / T) : 1, exclusive
// scans for item and slot offsets, items[], splits[], and a heaviest-first
// order of the items by cost / parts.  Two launches after the costs: one
// workgroup forms total, threshold, scans and the bucket sizes (k_work_scan),
// then every unit writes its items and takes their places in the order
// (k_work_items).  With each of those in a launch of its own a list took 16
// launches, ~70 us of a small job; one workgroup needs 4 us at 1,000 units and
// 31 us at 16,384 (66 us with the buckets counted by ballots).  Longer lists than
// MKDE_WS_ONE are scanned by a workgroup per 4096 units, in three launches (totals,
// counts, scan): rasters of few points, 16,384 / 65,536 / 262,144 / 1,048,576 blocks,
// 225 / 744 / 2813 / 11080 us by one workgroup, 220 / 667 / 2430 / 9446 us by many
// (16 launches: 259 / 708 / 2480 / 9496 us); 4,096 blocks 97 and 108 us,
// and between 6,000 and 16,000 units both are within 13 us.
#define DT_TMIN 2048u
#define DT_TARGET 4096ull

__device__ __forceinline__ unsigned split_threshold(unsigned long long total, const SplitRule &r)
{
    const unsigned long long t = (total + r.target - 1) / r.target;
    unsigned low = r.tmin;
    if (r.few > 0) {
        const unsigned long long f = (total + r.few - 1) / r.few;
        if (f < low) low = f > r.few_tmin ? (unsigned)f : r.few_tmin;
    }
    return t > low ? (unsigned)(t < 0xffffffffull ? t : 0xffffffffull) : low;
}

__device__ __forceinline__ unsigned split_parts(unsigned c, unsigned T)
{
    return c > T ? (unsigned)(((unsigned long long)c + T - 1) / T) : 1u;
}

#define WS_UNITS MKDE_WS_UNITS   // units of a step: four per thread

// Sum over the 1024 threads of a workgroup, in all of them (s_t: 16 words).
__device__ __forceinline__ unsigned long long sum1024(unsigned long long v, unsigned long long *s_t)
{
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, WAVE);
    __syncthreads();   // s_t of the sum before has been read
    if ((threadIdx.x & 63) == 0) s_t[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long total = 0;
    for (int w = 0; w < 16; ++w) total += s_t[w];
    return total;
}

// Costs and parts of this thread's four units, and the number of items, slots and
// split units among them.
struct StepUnits {
    unsigned c[4], k[4], ni, np, ns;
};
__device__ __forceinline__ StepUnits step_units(const unsigned *cost, int b0, int n, unsigned T)
{
    StepUnits u;
    u.ni = u.np = u.ns = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        u.c[j] = b0 + j < n ? cost[b0 + j] : 0u;
        u.k[j] = b0 + j < n ? split_parts(u.c[j], T) : 0u;
        u.ni += u.k[j];
        u.np += u.k[j] > 1 ? u.k[j] : 0u;
        u.ns += u.k[j] > 1 ? 1u : 0u;
    }
    return u;
}

// Total of the chunks' costs -> split threshold.
__device__ __forceinline__ unsigned chunks_threshold(const WorkList &W, int nchunks, const SplitRule &rule,
                                                     unsigned long long *s_t)
{
    unsigned long long acc = 0;
    for (int i = threadIdx.x; i < nchunks; i += 1024) acc += W.chunks[i].cost;
    return split_threshold(sum1024(acc, s_t), rule);
}

// Long lists, first launch: each chunk's total cost.
__global__ __launch_bounds__(1024) void k_work_totals(int n, WorkList W)
{
    __shared__ unsigned long long s_t[16];
    const int b0 = (int)blockIdx.x * WS_UNITS + 4 * (int)threadIdx.x;
    unsigned long long acc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc += b0 + j < n ? W.cost[b0 + j] : 0u;
    acc = sum1024(acc, s_t);
    if (threadIdx.x == 0) W.chunks[blockIdx.x].cost = acc;
}

// Second launch: each chunk's items, slots, split units and bucket sizes.
__global__ __launch_bounds__(1024) void k_work_counts(int n, SplitRule rule, WorkList W)
{
    __shared__ unsigned long long s_t[16];
    __shared__ unsigned s_h[16][32];
    const int tid = threadIdx.x, wave = tid >> 6;
    if (tid < 512) s_h[tid >> 5][tid & 31] = 0;
    const unsigned T = chunks_threshold(W, (int)gridDim.x, rule, s_t);
    const StepUnits u = step_units(W.cost, (int)blockIdx.x * WS_UNITS + 4 * tid, n, T);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (u.k[j]) atomicAdd(&s_h[wave][cost_bucket(u.c[j] / u.k[j])], u.k[j]);
    const unsigned long long ni = sum1024(u.ni, s_t), np = sum1024(u.np, s_t), ns = sum1024(u.ns, s_t);
    WorkChunk &ch = W.chunks[blockIdx.x];
    if (tid == 0) {
        ch.n[0] = (unsigned)ni;
        ch.n[1] = (unsigned)np;
        ch.n[2] = (unsigned)ns;
    }
    if (tid < 32) {
        unsigned h = 0;
        for (int w = 0; w < 16; ++w) h += s_h[w][tid];
        ch.hist[tid] = h;
    }
}

// One workgroup of 1024 threads, four units per thread and step; MANY: the last
// launch of a long list, a workgroup per step.  host (nullable, pinned): also
// receives the counts.
template <bool MANY>
__global__ __launch_bounds__(1024) void k_work_scan(int n, SplitRule rule, WorkList W, unsigned *host, const double *extra)
{
    __shared__ unsigned long long s_t[16];
    __shared__ unsigned s_w[16][3];
    __shared__ unsigned s_h[16][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < 512) s_h[tid >> 5][tid & 31] = 0;
    unsigned T;
    unsigned run_i = 0, run_p = 0, run_s = 0;   // items, slots, splits before this step
    unsigned all[3] = {0, 0, 0};                // MANY, first workgroup: of the list
    if (MANY) {
        T = chunks_threshold(W, (int)gridDim.x, rule, s_t);
        const int lim = blockIdx.x ? (int)blockIdx.x : (int)gridDim.x;
        unsigned long long a[3] = {0, 0, 0};
        for (int i = tid; i < lim; i += 1024)
            for (int q = 0; q < 3; ++q) a[q] += W.chunks[i].n[q];
        for (int q = 0; q < 3; ++q) all[q] = (unsigned)sum1024(a[q], s_t);
        if (blockIdx.x) {
            run_i = all[0];
            run_p = all[1];
            run_s = all[2];
        } else {
            for (int i = tid >> 5; i < (int)gridDim.x; i += 32) atomicAdd(&s_h[wave][tid & 31], W.chunks[i].hist[tid & 31]);
        }
    } else {
        unsigned long long acc = 0;
        for (int i = tid; i < n; i += 1024) acc += W.cost[i];
        T = split_threshold(sum1024(acc, s_t), rule);
    }
    const int first = MANY ? (int)blockIdx.x * WS_UNITS : 0, end = MANY ? first + 1 : n;
    for (int base = first; base < end; base += WS_UNITS) {
        const int b0 = base + 4 * tid;
        const StepUnits u = step_units(W.cost, b0, n, T);
        const unsigned ii = wave_incl_scan(u.ni, lane), ip = wave_incl_scan(u.np, lane), is = wave_incl_scan(u.ns, lane);
        if (lane == WAVE - 1) {
            s_w[wave][0] = ii;
            s_w[wave][1] = ip;
            s_w[wave][2] = is;
        }
        __syncthreads();
        unsigned oi = run_i + ii - u.ni, op = run_p + ip - u.np, os = run_s + is - u.ns;
        for (int w = 0; w < 16; ++w) {
            const unsigned a0 = s_w[w][0], a1 = s_w[w][1], a2 = s_w[w][2];
            if (w < wave) {
                oi += a0;
                op += a1;
                os += a2;
            }
            run_i += a0;
            run_p += a1;
            run_s += a2;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (b0 + j >= n) break;
            W.item0[b0 + j] = oi;
            oi += u.k[j];
            if (u.k[j] > 1) {
                W.slot0[b0 + j] = op;
                W.sidx[b0 + j] = os++;
                op += u.k[j];
            }
        }
        // bucket sizes, a copy per wave
        if (!MANY)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (u.k[j]) atomicAdd(&s_h[wave][cost_bucket(u.c[j] / u.k[j])], u.k[j]);
        __syncthreads();
    }
    if (tid == 0 && (!MANY || blockIdx.x == 0)) {
        const unsigned out[4] = {MANY ? all[0] : run_i, MANY ? all[1] : run_p, MANY ? all[2] : run_s, T};
        for (int j = 0; j < 4; ++j) {
            W.counts[j] = out[j];
            if (host) host[j] = out[j];
        }
        if (host && extra) *(double *)(host + 4) = *extra;
        unsigned run = 0;
        for (int b = 0; b < 32; ++b) {
            W.hist[b] = run;
            for (int w = 0; w < 16; ++w) run += s_h[w][b];
        }
    }
}

// Items, split list and visiting order.  Places in a bucket are reserved once
// per workgroup (LDS counters, one global atomic per bucket), so the few large
// buckets do not serialise every item on one address.
__global__ __launch_bounds__(256) void k_work_items(int n, WorkList W, int4 *items, int4 *splits, int *order)
{
    __shared__ unsigned s_h[32], s_base[32];
    if (threadIdx.x < 32) s_h[threadIdx.x] = 0;
    __syncthreads();
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    int bk = 0;
    unsigned k = 0, r = 0, i0 = 0;
    if (b < n) {
        const unsigned c = W.cost[b];
        k = split_parts(c, W.counts[3]);
        i0 = W.item0[b];
        bk = cost_bucket(c / k);
        r = atomicAdd(&s_h[bk], k);
    }
    __syncthreads();
    if (threadIdx.x < 32 && s_h[threadIdx.x]) s_base[threadIdx.x] = atomicAdd(&W.hist[threadIdx.x], s_h[threadIdx.x]);
    __syncthreads();
    if (b >= n) return;
    const int slot0 = k > 1 ? (int)W.slot0[b] : -1;
    for (unsigned j = 0; j < k; ++j) {
        items[i0 + j] = make_int4(b, (int)j, (int)k, k > 1 ? slot0 + (int)j : -1);
        order[s_base[bk] + r + j] = (int)(i0 + j);
    }
    if (k > 1) splits[W.sidx[b]] = make_int4(b, slot0, (int)k, 0);
}

// ---- exclusive scan of unsigned values (1024 per workgroup, two levels)
__global__ __launch_bounds__(256) void k_scan_local(int n, const unsigned *in, unsigned *out, unsigned *chunk_sums)
{
    __shared__ unsigned s_w[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * 1024 + tid * 4;
    unsigned v[4], t = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        t += v[k];
    }
    unsigned x = t;   // inclusive wave scan of thread totals
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned y = __shfl_up(x, d, WAVE);
        if (lane >= d) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    unsigned woff = 0;
    for (int w = 0; w < wave; ++w) woff += s_w[w];
    unsigned run = woff + x - t;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (tid == 255) chunk_sums[blockIdx.x] = woff + x;
}

__global__ __launch_bounds__(256) void k_scan_chunks(int nchunks, unsigned *chunk_sums, unsigned *total)
{
    __shared__ unsigned s_w[4];
    __shared__ unsigned s_carry;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) s_carry = 0;
    __syncthreads();
    for (int base = 0; base < nchunks; base += 256) {
        const unsigned t = base + tid < nchunks ? chunk_sums[base + tid] : 0u;
        unsigned x = t;
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned y = __shfl_up(x, d, WAVE);
            if (lane >= d) x += y;
        }
        if (lane == 63) s_w[wave] = x;
        __syncthreads();
        unsigned woff = s_carry;
        for (int w = 0; w < wave; ++w) woff += s_w[w];
        if (base + tid < nchunks) chunk_sums[base + tid] = woff + x - t;
        __syncthreads();
        if (tid == 255) s_carry = woff + x;
        __syncthreads();
    }
    if (tid == 0) *total = s_carry;
}

__global__ void k_scan_add(int n, unsigned *out, const unsigned *chunk_sums)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += chunk_sums[i / 1024];
}

// ==================================================== density at points ====
//
// One wave owns consecutive query points (lane = query) and walks the candidate
// bins of its bounding box; every source is taken up by the whole wave at once.
//   k_point_sums, k_loo_multi   bin order: pilot densities, and the leave-one-out
//                      densities whose logarithms are summed
//   k_point_density_f  fine order: the densities that are an output (a bandwidth
//                      per source, leave-one-out), with sums over whole groups
// Duplicates at distance 0 are kept.  Waves run heaviest first
// (k_wave_cost).
//
// Cut-off test: d2f = fl32(dx*dx + dy*dy) decides unless it lies within a
// relative 2^-20 band around the threshold (its error is below 2^-22
// relative); where any lane is in the band the exact FP64 test
// fl64(dx^2 + dy^2) < thr is evaluated instead, so the result is exact.

struct PtsArgs {
    PointIndex idx;
    float *den;   // output, the index's order
    float *res;   // n floats of scratch (fine order)
    // work items (nullable order: one item per wave): {wave, part j, parts K,
    // partial slot}; part j of a wave takes candidate ordinals
    // [C j / K, C (j+1) / K) of its C candidate sources (cost[wave])
    const int *order;
    const int4 *items;
    const unsigned *cost;
    double *partials;            // 64 per slot
    int n_items;
    const unsigned *n_items_dev;   // non-null: the item count on the device (n_items: grid bound)
};

// Orders LDS accesses of the lanes of one wave (its LDS operations complete in
// order, so only the compiler has to keep them).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float wave_min(float v)
{
    for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, WAVE));
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, WAVE));
    return v;
}
__device__ __forceinline__ float uni(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v))); }
__device__ __forceinline__ int4 uniform_item(int4 v)
{
    return make_int4(__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y),
                     __builtin_amdgcn_readfirstlane(v.z), __builtin_amdgcn_readfirstlane(v.w));
}

// Work estimate of each 64-query wave of the point kernels: the points in
// its candidate bins (same culling as the kernels: bins within the reach of
// the wave's bounding box whose box gap is below the threshold -- lim_fixed
// when > 0, else lim_dev[0] when given, else each bin's own threshold).
// Waves then run heaviest first.
__global__ __launch_bounds__(256) void k_wave_cost(PointIndex I, double lim_fixed, const double *lim_dev,
                                                   unsigned *cost)
{
    const int lane = threadIdx.x & 63;
    const int64_t nw = (I.n + 63) / 64;
    const int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wv >= nw) return;
    const int64_t q = wv * 64 + lane;
    const bool qv = q < I.n;
    float qx = 0.0f, qy = 0.0f;
    if (qv) {
        const PtRec p = I.pts[q];
        qx = p.x;
        qy = p.y;
    }
    const float mnx = wave_min(qv ? qx : FLT_MAX), mxx = wave_max(qv ? qx : -FLT_MAX);
    const float mny = wave_min(qv ? qy : FLT_MAX), mxy = wave_max(qv ? qy : -FLT_MAX);
    const bool uni_lim = lim_fixed > 0.0 || lim_dev;
    const double lim = lim_fixed > 0.0 ? lim_fixed : (lim_dev ? *lim_dev : 0.0);
    const double reach = uni_lim ? sqrt(fmax(lim, 0.0)) * 1.000001 + 1e-6 : *I.reach_p;
    int bxa, bxb, bya, byb;
    bin_range(I.bg, mnx, mxx, mny, mxy, reach, bxa, bxb, bya, byb);
    const int nbx_r = bxb - bxa + 1;
    const int nb_total = nbx_r * (byb - bya + 1);
    unsigned acc = 0;
    for (int k = lane; k < nb_total; k += 64) {
        const int b = (bya + k / nbx_r) * I.bg.nbx + (bxa + k % nbx_r);
        const int c = I.bin_start[b + 1] - I.bin_start[b];
        if (c > 0 && box_gap2(I.bin_box[b], mnx, mxx, mny, mxy) < (uni_lim ? lim : I.bin_thr[b])) acc += (unsigned)c;
    }
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
    if (lane == 0) cost[wv] = acc;
}

// Whole groups of sources.  For a group of 64 sources whose every pair with the
// wave is inside the cut-off, and a wave whose points lie close together
// compared with the sources' bandwidths, the 64 kernels are expanded about the
// centre c of the wave's box: with d = s - c, t = q - c, b = 1 / (2 h^2)
//   exp(-b |t - d|^2) = exp(-b d^2) sum_ij m_i(dx) m_j(dy) tx^i ty^j / (i! j!),
//   m_0 = 1, m_1 = 2 b d, m_(k+1) = 2 b d m_k - 2 b k m_(k-1)
// (the Hermite generating function), so a source adds coef exp(-b d^2) m_i m_j
// to 36 moments (i + j < PF_P), one source per lane, and the polynomial is
// evaluated once per query at the end of the walk.  About 100 instructions a
// group instead of 64 times 8.  Moments are FP64 (its rate is that of FP32
// here).  What is left out is below 0.025 tau^8 of a source's kernel, tau =
// |t| / h <= PF_TAU: 1.1e-8, under the rounding of the FP32 exponentials.
#define PF_P 8
#define PF_NM (PF_P * (PF_P + 1) / 2)
#define PF_TAU 0.16

__device__ __forceinline__ void group_moments(const SrcRec &p, bool on, double cx, double cy, double (&M)[PF_NM])
{
    const double dx = (double)p.x - cx, dy = (double)p.y - cy;
    const double d2 = __builtin_fma(dy, dy, dx * dx);
    const double af = p.af;
    const double b2 = af * (-2.0 * 0.69314718055994530942);   // 1 / h^2
    const double ux = b2 * dx, uy = b2 * dy;
    double gx[PF_P], gy[PF_P];
    gx[0] = on ? (double)p.coef * (double)fast_exp2((float)(d2 * af)) : 0.0;
    gx[1] = ux * gx[0];
    gy[0] = 1.0;
    gy[1] = uy;
#pragma unroll
    for (int k = 1; k + 1 < PF_P; ++k) {
        const double v = b2 * (double)k;
        gx[k + 1] = __builtin_fma(ux, gx[k], -v * gx[k - 1]);
        gy[k + 1] = __builtin_fma(uy, gy[k], -v * gy[k - 1]);
    }
    int o = 0;
#pragma unroll
    for (int i = 0; i < PF_P; ++i)
#pragma unroll
        for (int j = 0; j < PF_P - i; ++j, ++o) M[o] = __builtin_fma(gx[i], gy[j], M[o]);
}

// A work item of the fine-order kernels and its wave's box.
struct FineItem {
    int4 item;
    int win0, win1;     // candidate ordinals of this part
    int q;              // this lane's query
    GroupInfo W;
    int bxa, bxb, bya, byb;
    double cx, cy;      // centre of the box
    double wide;        // groups are taken whole from this smallest 9 h^2 on
};

// false: the grid is larger than the list (whole wave).
__device__ __forceinline__ bool fine_item(const PtsArgs &A, FineItem &F)
{
    const PointIndex &I = A.idx;
    // the wave index and the work item are wave-uniform: made explicit so that
    // item and box are read with scalar loads and the walk's limits are scalars
    const int64_t g = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t units = A.n_items_dev ? (int64_t)*A.n_items_dev : A.order ? (int64_t)A.n_items : (I.n + 63) / 64;
    if (g >= units) return false;
    F.item = uniform_item(A.order ? A.items[A.order[g]] : make_int4((int)g, 0, 1, -1));
    F.win0 = 0;
    F.win1 = INT_MAX;   // candidate counts are below 2^31
    if (F.item.z > 1) {
        const int64_t C = A.cost[F.item.x];
        if (F.item.y > 0) F.win0 = (int)(C * F.item.y / F.item.z);
        if (F.item.y < F.item.z - 1) F.win1 = (int)(C * (F.item.y + 1) / F.item.z);
    }
    F.q = F.item.x * 64 + (int)(threadIdx.x & 63);   // below 2^30
    F.W = I.grp[F.item.x];
    const GroupInfo &W = F.W;
    bin_range(I.bg, W.x0, W.x1, W.y0, W.y1, *I.reach_p, F.bxa, F.bxb, F.bya, F.byb);
    F.bxa = __builtin_amdgcn_readfirstlane(F.bxa);
    F.bxb = __builtin_amdgcn_readfirstlane(F.bxb);
    F.bya = __builtin_amdgcn_readfirstlane(F.bya);
    F.byb = __builtin_amdgcn_readfirstlane(F.byb);
    F.cx = 0.5 * ((double)W.x0 + (double)W.x1);
    F.cy = 0.5 * ((double)W.y0 + (double)W.y1);
    const double hx = (double)W.x1 - F.cx, hy = (double)W.y1 - F.cy;
    F.wide = fmax((hx * hx + hy * hy) * (9.0 / (PF_TAU * PF_TAU)), 1e-30);
    return true;
}

// What lane l sees of group gb + l of a row of bins, whose sources s0 .. s1 - 1
// are consecutive: its share c0 .. c1 - 1 of them and cls 0: no pair with the
// wave's box W is inside the cut-off, 1: some may be, 2: all are (the largest
// fl32 offsets are, and sq2 is monotone), 3: all are and the group is taken
// whole.  own: the wave's group (LOO) or -1; wide: FineItem::wide.
__device__ __forceinline__ int group_class(const PointIndex &I, const GroupInfo &W, int gb, int s0, int s1, int own,
                                           double wide, int &c0, int &c1)
{
    const int g = gb + (int)(threadIdx.x & 63);
    const bool on = g <= (s1 - 1) >> 6;
    const GroupInfo G = I.grp[on ? g : gb];
    c0 = s0 > g * 64 ? s0 : g * 64;
    c1 = s1 < g * 64 + 64 ? s1 : g * 64 + 64;
    const float fx = fmaxf(G.x1 - W.x0, W.x1 - G.x0), fy = fmaxf(G.y1 - W.y0, W.y1 - G.y0);
    const bool near = on && box_gap2(BinInfo{G.x0, G.y0, G.x1, G.y1}, W.x0, W.x1, W.y0, W.y1) < G.tmax;
    const bool full = sq2(fx, fy) < G.tmin && g != own;
    const bool whole = full && G.tmin >= wide && G.tmin < 1e37;
    return near ? 1 + (int)full + (int)whole : 0;
}

// Walks an item's candidate groups, 64 at a time (one per lane), and calls
// fn(c0, c1, all) for those taken whole (WHOLE) or for the others; all: every
// pair is inside.  (Group by group with wave-uniform tests the walks took a
// third of the kernels' instructions.)
template <bool LOO, bool WHOLE, class F>
__device__ __forceinline__ void fine_walk(const PointIndex &I, const FineItem &T, F fn)
{
    const int lane = threadIdx.x & 63;
    int ord = 0;   // candidate ordinal of the next group
    for (int by = T.bya; by <= T.byb; ++by) {
        const int row = by * I.bg.nbx;
        const int s0 = I.bin_start[row + T.bxa], s1 = I.bin_start[row + T.bxb + 1];
        for (int gb = s0 >> 6; gb * 64 < s1; gb += 64) {
            int c0, c1;
            int cls = group_class(I, T.W, gb, s0, s1, LOO ? T.item.x : -1, T.wide, c0, c1);
            if (T.item.z > 1) {
                // this part's share of the candidate sequence
                const int cnt = cls ? c1 - c0 : 0;
                const int o1 = ord + (int)wave_incl_scan((unsigned)cnt, lane), o0 = o1 - cnt;
                ord = __builtin_amdgcn_readlane(o1, 63);
                if (o1 <= T.win0 || o0 >= T.win1) cls = 0;
                if (T.win0 > o0) c0 += T.win0 - o0;
                if (T.win1 < o1) c1 -= o1 - T.win1;
            }
            if (cls == 3 && c1 - c0 < 12) cls = 2;   // cheaper source by source
            uint64_t m = __ballot(WHOLE ? cls == 3 : cls == 1 || cls == 2);
            const uint64_t all = __ballot(cls >= 2);
            while (m) {
                const int l = __builtin_ctzll(m);
                m &= m - 1ull;
                fn(__builtin_amdgcn_readlane(c0, l), __builtin_amdgcn_readlane(c1, l), (bool)((all >> l) & 1ull));
            }
        }
    }
}

// Work estimate of each fine-order wave: the sources of its candidate groups.
__global__ __launch_bounds__(256) void k_fine_cost(PointIndex I, unsigned *cost)
{
    const int lane = threadIdx.x & 63;
    const int wv = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int64_t)wv * 64 >= I.n) return;
    const GroupInfo W = I.grp[wv];
    int bxa, bxb, bya, byb;
    bin_range(I.bg, W.x0, W.x1, W.y0, W.y1, *I.reach_p, bxa, bxb, bya, byb);
    unsigned acc = 0;
    for (int by = bya; by <= byb; ++by) {
        const int row = by * I.bg.nbx;
        const int s0 = I.bin_start[row + bxa], s1 = I.bin_start[row + bxb + 1];
        for (int gb = s0 >> 6; gb * 64 < s1; gb += 64) {
            int c0, c1;
            if (group_class(I, W, gb, s0, s1, -1, 1e300, c0, c1)) acc += (unsigned)(c1 - c0);
        }
    }
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
    if (lane == 0) cost[wv] = acc;
}

// The sources taken in whole groups.  Runs before k_point_density_f and
// leaves an unsplit wave's sum as a pair of floats in den and res, a part's in
// its slot of the partials.  A kernel of its own: its moments take 128 registers
// (4 waves per SIMD), in one kernel they took 164 or spilled.
// 1M clustered points, adaptive bandwidths, leave-one-out: 8.8 ms pair by pair
// with an FP64 test each, 0.64 + 2.71 ms now (12.0 ms with both in one kernel).
template <bool LOO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_group_density_f(PtsArgs A)
{
    const PointIndex &I = A.idx;
    const SrcRec *src = (const SrcRec *)I.pts;
    const int lane = threadIdx.x & 63;
    FineItem T;
    if (!fine_item(A, T)) return;
    double v = 0.0;
    // no source is wide enough when the largest cut-off radius is not
    if ((*I.reach_p) * (*I.reach_p) >= T.wide) {
        double M[PF_NM];
#pragma unroll
        for (int k = 0; k < PF_NM; ++k) M[k] = 0.0;
        // a group's records are loaded while the one before is summed
        SrcRec next;
        bool next_on = false, any = false;
        fine_walk<LOO, true>(I, T, [&](int c0, int c1, bool) {
            const bool on = c0 + lane < c1;
            const SrcRec p = next;
            next = src[on ? c0 + lane : c0];
            if (any) group_moments(p, next_on, T.cx, T.cy, M);
            next_on = on;
            any = true;
        });
        if (any) {
            group_moments(next, next_on, T.cx, T.cy, M);
            // moments over the lanes, then this query's polynomial (Horner in
            // both variables, with the factorials)
            const bool qv = T.q < I.n;
            const double tx = (qv ? (double)src[T.q].x : T.cx) - T.cx, ty = (qv ? (double)src[T.q].y : T.cy) - T.cy;
            int o = PF_NM;
#pragma unroll
            for (int i = PF_P - 1; i >= 0; --i) {
                double row = 0.0;
#pragma unroll
                for (int j = PF_P - 1 - i; j >= 0; --j) {
                    double m = M[--o];
                    for (int d = 32; d >= 1; d >>= 1) m += __shfl_xor(m, d, WAVE);
                    row = __builtin_fma(row, ty * (1.0 / (double)(j + 1)), m);
                    __builtin_amdgcn_sched_barrier(0);   // one moment after the other, few registers
                }
                v = __builtin_fma(v, tx * (1.0 / (double)(i + 1)), row);
            }
        }
    }
    if (T.item.z > 1) {
        A.partials[(int64_t)T.item.w * 64 + lane] = v;
    } else if (T.q < I.n) {
        const float hi = (float)v;
        A.den[T.q] = hi;
        A.res[T.q] = (float)(v - (double)hi);
    }
}

// The other sources, pair by pair, and the total.  (The select is on the
// coefficient: an infinite one adds nothing outside its cut-off.)  A group's records come in one
// per lane and are handed round through LDS.  Bound by instruction issue, 8 or 12
// a pair.  (Scalar loads, four records at a time: 3.66 ms on 1M clustered points, 2.71 ms now.)
template <bool LOO>
__global__ __launch_bounds__(256) void k_point_density_f(PtsArgs A)
{
    __shared__ float4 s_a[4][64];   // x, y, coef, af
    __shared__ float2 s_b[4][64];   // lo, hi
    const PointIndex &I = A.idx;
    const SrcRec *src = (const SrcRec *)I.pts;
    const int lane = threadIdx.x & 63;
    FineItem T;
    if (!fine_item(A, T)) return;
    float4 *pa = s_a[threadIdx.x >> 6];
    float2 *pb = s_b[threadIdx.x >> 6];
    const int q = T.q;
    const bool qv = q < I.n;
    const float qx = qv ? src[q].x : T.W.x0, qy = qv ? src[q].y : T.W.y0;
    float sum = 0.0f, comp = 0.0f;
    fine_walk<LOO, false>(I, T, [&](int c0, int c1, bool all) {
        // the query itself is left out of its own group's sums
        const bool self = LOO && (c0 >> 6) == T.item.x;
        wave_sync();
        if (c0 + lane < c1) {
            const SrcRec p = src[c0 + lane];
            pa[lane] = make_float4(p.x, p.y, p.coef, p.af);
            pb[lane] = make_float2(p.lo, p.hi);
        }
        wave_sync();
        for (int s0 = 0; s0 < c1 - c0; s0 += 32) {
            const int s1 = s0 + 32 < c1 - c0 ? s0 + 32 : c1 - c0;
            float acc = 0.0f;
            bool band = self;
            if (all) {
#pragma unroll 4
                for (int j = s0; j < s1; ++j) {
                    const float4 p = pa[j];
                    const float dx = p.x - qx, dy = p.y - qy;
                    const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                    acc = __builtin_fmaf(fast_exp2(d2f * p.w), p.z, acc);
                }
            } else if (!self) {
#pragma unroll 4
                for (int j = s0; j < s1; ++j) {
                    const float4 p = pa[j];
                    const float2 t = pb[j];
                    const float dx = p.x - qx, dy = p.y - qy;
                    const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                    const bool in = d2f < t.x;
                    band |= !(d2f > t.y) != in;
                    const float e = fast_exp2(d2f * p.w);
                    acc = __builtin_fmaf(e, in ? p.z : 0.0f, acc);
                }
            }
            if (__any(band)) {   // rare, and the wave's own group: exact FP64 test
                acc = 0.0f;
                for (int j = s0; j < s1; ++j) {
                    const float4 p = pa[j];
                    const float dx = p.x - qx, dy = p.y - qy;
                    const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                    bool in = sq2(dx, dy) < src[c0 + j].thr;
                    if (LOO && c0 + j == q) in = false;
                    const float e = fast_exp2(d2f * p.w);
                    acc = __builtin_fmaf(e, in ? p.z : 0.0f, acc);
                }
            }
            kahan_fold(acc, sum, comp);
            if (!(fabsf(sum) < INFINITY)) comp = 0.0f;   // an infinite sum stays one
        }
    });
    const double den = (double)sum - (double)comp;
    if (T.item.z > 1) A.partials[(int64_t)T.item.w * 64 + lane] += den;
    else if (qv) A.den[q] = (float)(den + ((double)A.den[q] + (double)A.res[q]));
}

// Exclusive scan of one int per thread across a 256-thread block.
__device__ __forceinline__ int block_exscan256(int v, int *s_w, int *total)
{
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x >> 6;
    int inc = v;
    for (int d = 1; d < WAVE; d <<= 1) {
        int o = __shfl_up(inc, d, WAVE);
        if (lane >= d) inc += o;
    }
    if (lane == WAVE - 1) s_w[wave] = inc;
    __syncthreads();
    int off = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) off += (w < wave) ? s_w[w] : 0;
    *total = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    __syncthreads();
    return off + inc - v;
}



// =================================================== point sums in bin order ==
//
// Sums at the points that are more than an output: pilot densities, from which
// the adaptive bandwidths and so the cut-offs follow, and the leave-one-out
// densities whose logarithms are summed (bandwidth search).  With weights of very
// different sizes a float sum of 32 terms depends on the order of the sources, and
// alike for all queries around, so the order is part of the result: bins row by
// row, the caller's order within a bin, 32 sources at a time in FP32 from the
// bin's first one (or from where a wave of many candidates is cut), these sums in
// Kahan pairs.  What is outside the cut-off adds nothing and is left out by bins.
// A short list fills the device by candidates and by queries, fewer per wave, not
// by cuts.

#define LM_K MKDE_LM_K

struct SumArgs {
    PointIndex idx;          // bin order; thr of the largest candidate (K bandwidths)
    const float *coefk;      // [K][n] bin order
    const double *a_k;       // [K]
    const double *thr_k;     // [K] ascending
    int K, kw;               // candidates, and how many a wave takes (blockIdx.y picks them)
    double thr_fixed, a_fixed;   // pilot
    float *den1;             // [K][n] bin order
    // work items (nullable order: one item per wave), as for the fine-order kernels
    const int *order;
    const int4 *items;
    const unsigned *cost;
    double *partials;        // 64 * LM_K per slot (64, one density)
    int n_items;
    const unsigned *n_items_dev;   // non-null: the item count on the device (n_items: grid bound)
};

// A work item: its candidate ordinals, and its 64 queries' box.
struct SumItem {
    int4 item;
    int win0, win1;
    int q;              // this lane's query of the 64
    bool qv;
    float qx, qy, mnx, mxx, mny, mxy;
};

// Item g of the list; false: the grid is larger than the list (whole wave).
__device__ __forceinline__ bool sum_item(const SumArgs &A, int64_t g, SumItem &T)
{
    const PointIndex &I = A.idx;
    const int64_t units = A.n_items_dev ? (int64_t)*A.n_items_dev : A.order ? (int64_t)A.n_items : (I.n + 63) / 64;
    if (g >= units) return false;
    T.item = uniform_item(A.order ? A.items[A.order[g]] : make_int4((int)g, 0, 1, -1));
    T.win0 = 0;
    T.win1 = INT_MAX;   // candidate counts are below 2^31
    if (T.item.z > 1) {
        const int64_t C = A.cost[T.item.x];
        if (T.item.y > 0) T.win0 = (int)(C * T.item.y / T.item.z);
        if (T.item.y < T.item.z - 1) T.win1 = (int)(C * (T.item.y + 1) / T.item.z);
    }
    T.q = T.item.x * 64 + (int)(threadIdx.x & 63);   // below 2^30
    T.qv = T.q < I.n;
    T.qx = T.qy = 0.0f;
    if (T.qv) {
        T.qx = I.pts[T.q].x;
        T.qy = I.pts[T.q].y;
    }
    T.mnx = uni(wave_min(T.qv ? T.qx : FLT_MAX));
    T.mxx = uni(wave_max(T.qv ? T.qx : -FLT_MAX));
    T.mny = uni(wave_min(T.qv ? T.qy : FLT_MAX));
    T.mxy = uni(wave_max(T.qv ? T.qy : -FLT_MAX));
    return true;
}

// Walks an item's candidate bins, 64 of a row at a time (one per lane): the whole
// wave calls fn(m, p0, p1, B, lm) with the mask m of the lanes whose bin, box B and
// cut-off lm = lim(b), has sources p0 .. p1 - 1 of this part.
template <class L, class F>
__device__ __forceinline__ void sum_walk(const PointIndex &I, const SumItem &T, double reach, L lim, F fn)
{
    const int lane = threadIdx.x & 63;
    int bxa, bxb, bya, byb;
    bin_range(I.bg, T.mnx, T.mxx, T.mny, T.mxy, reach, bxa, bxb, bya, byb);
    bxa = __builtin_amdgcn_readfirstlane(bxa);
    bxb = __builtin_amdgcn_readfirstlane(bxb);
    bya = __builtin_amdgcn_readfirstlane(bya);
    byb = __builtin_amdgcn_readfirstlane(byb);
    int ord = 0;   // candidate ordinal of the next candidate bin
    for (int by = bya; by <= byb; ++by) {
        for (int bx = bxa; bx <= bxb; bx += 64) {
            const bool on = bx + lane <= bxb;
            const int b = by * I.bg.nbx + (on ? bx + lane : bxb);
            int p0 = I.bin_start[b], p1 = I.bin_start[b + 1];
            const BinInfo B = I.bin_box[b];
            const double lm = lim(b);
            bool mine = on && p0 < p1 && box_gap2(B, T.mnx, T.mxx, T.mny, T.mxy) < lm;
            if (T.item.z > 1) {
                const int cnt = mine ? p1 - p0 : 0;
                const int o1 = ord + (int)wave_incl_scan((unsigned)cnt, lane), o0 = o1 - cnt;
                ord = __builtin_amdgcn_readlane(o1, 63);
                mine = mine && o1 > T.win0 && o0 < T.win1;
                if (T.win1 < o1) p1 -= o1 - T.win1;
                if (T.win0 > o0) p0 += T.win0 - o0;
            }
            const uint64_t m = __ballot(mine);
            if (m) fn(m, p0, p1, B, lm);
        }
    }
}

// Bounds of the squared distances between a bin's box and the box x0 .. y1.
__device__ __forceinline__ double box_far2(const BinInfo &B, float x0, float x1, float y0, float y1)
{
    return sq2(fmaxf(B.x1 - x0, x1 - B.x0), fmaxf(B.y1 - y0, y1 - B.y0));
}

// One bandwidth, or one per source.  A wave takes 64 / P of an item's queries and
// P of the sums of 32 at a time, one per 64 / P lanes, which are then folded in
// their order: as many waves more, each that much shorter, and the same sums.
// The sources come in one per lane and are handed round through LDS.  The cut-off
// is decided in FP32 where the distance is clear of the threshold (thr_bracket),
// else by the exact FP64 test, and not at all for bins that are inside as a whole.
// Bound by instruction issue: 8 a pair of an inside bin, 12 else.  (Scalar loads
// of each source, one wave an item: two steps of the adaptive search on 100,000
// clustered points 1.63 ms, now 0.81 ms; two candidates 0.84 -> 0.34 ms.)
enum { SUM_PILOT, SUM_LOO, SUM_LOO_EACH };   // one bandwidth, one of K without the query, one per source without it
template <int KIND, int P>
__global__ __launch_bounds__(256) void k_point_sums(SumArgs A)
{
    constexpr int Q = 64 / P;
    constexpr bool EACH = KIND == SUM_LOO_EACH, SELF = KIND == SUM_PILOT;
    __shared__ float4 s_a[4][P][33];                // x, y, coef, af (33: the P records read together are in different banks)
    __shared__ float2 s_b[EACH ? 4 : 1][P][33];     // lo, hi
    const PointIndex &I = A.idx;
    const int lane = threadIdx.x & 63, r = lane % Q, ph = lane / Q;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t gw = (int64_t)blockIdx.x * 4 + wid;
    const int u = (int)(gw % P), k = blockIdx.y;
    SumItem T;
    if (!sum_item(A, gw / P, T)) return;
    const int q0 = T.item.x * 64, q = q0 + u * Q + r;
    const bool qv = q < I.n;
    const float qx = __shfl(T.qx, u * Q + r, WAVE), qy = __shfl(T.qy, u * Q + r, WAVE);
    const float x0 = uni(wave_min(qv ? qx : FLT_MAX)), x1 = uni(wave_max(qv ? qx : -FLT_MAX));
    const float y0 = uni(wave_min(qv ? qy : FLT_MAX)), y1 = uni(wave_max(qv ? qy : -FLT_MAX));
    const double thr = EACH ? 0.0 : SELF ? A.thr_fixed : A.thr_k[k];
    const double lim_all = EACH ? 0.0 : SELF ? A.thr_fixed : A.thr_k[A.K - 1];   // of the work list
    const float f_a = EACH ? 0.0f : uni((float)(SELF ? A.a_fixed : A.a_k[k]));
    float f_lo = 0.0f, f_hi = 0.0f;
    if (!EACH) thr_bracket(thr, f_lo, f_hi);
    float sum = 0.0f, comp = 0.0f;
    int pos = 0, cnt = 0, np = 0;   // this lane's chunk, chunks taken up
    bool all = true, own = false;

    auto flush = [&]() __attribute__((always_inline)) {
        wave_sync();
#pragma unroll
        for (int i = r; i < 32; i += Q) {
            if (P == 1 && i >= 32) break;
            // past the chunk's end: too far to count, without a weight
            float4 v = make_float4(1e19f, 1e19f, 0.0f, -1.0f);
            float2 t = make_float2(-1.0f, -1.0f);
            if (i < cnt) {
                const PtRec p = I.pts[pos + i];
                v = make_float4(p.x, p.y, KIND == SUM_LOO ? A.coefk[(int64_t)k * I.n + pos + i] : p.coef, (float)p.a);
                if (EACH) thr_bracket(p.thr, t.x, t.y);
            }
            s_a[wid][ph][i] = v;
            if (EACH) s_b[EACH ? wid : 0][ph][i] = t;
        }
        wave_sync();
        int jn = __builtin_amdgcn_readlane(cnt, 0);
#pragma unroll
        for (int i = 1; i < P; ++i) {
            const int c = __builtin_amdgcn_readlane(cnt, i * Q);
            jn = jn > c ? jn : c;
        }
        float acc = 0.0f;
        bool band = !SELF && own;
        if (!EACH && all && !band) {
#pragma unroll 4
            for (int j = 0; j < jn; ++j) {
                const float4 p = s_a[wid][ph][j];
                const float dx = p.x - qx, dy = p.y - qy;
                const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                acc = __builtin_fmaf(fast_exp2(d2f * f_a), p.z, acc);
            }
        } else if (!band) {
#pragma unroll 4
            for (int j = 0; j < jn; ++j) {
                const float4 p = s_a[wid][ph][j];
                const float2 t = EACH ? s_b[EACH ? wid : 0][ph][j] : make_float2(f_lo, f_hi);
                const float dx = p.x - qx, dy = p.y - qy;
                const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                const bool in = d2f < t.x;
                band |= !(d2f > t.y) != in;
                const float e = fast_exp2(d2f * (EACH ? p.w : f_a));
                acc = __builtin_fmaf(in ? e : 0.0f, p.z, acc);
            }
        }
        if (__any(band)) {   // rare, and the bins of the queries themselves
            acc = 0.0f;
            for (int j = 0; j < jn; ++j) {
                const float4 p = s_a[wid][ph][j];
                const float dx = p.x - qx, dy = p.y - qy;
                const float d2f = __builtin_fmaf(dy, dy, dx * dx);
                bool in = sq2(dx, dy) < (EACH ? (j < cnt ? I.pts[pos + j].thr : -1.0) : thr);
                if (!SELF && pos + j == q) in = false;
                const float e = fast_exp2(d2f * (EACH ? p.w : f_a));
                acc = __builtin_fmaf(in ? e : 0.0f, p.z, acc);
            }
        }
        if (P == 1) {
            kahan_fold(acc, sum, comp);
        } else {
            // the P sums in their order, in all of a query's lanes
#pragma unroll
            for (int i = 0; i < P; ++i) {
                const float v = __shfl(acc, i * Q + r, WAVE);
                if (i < np) kahan_fold(v, sum, comp);
            }
        }
        np = 0;
        cnt = 0;
        all = true;
        own = false;
    };

    const double reach = EACH ? *I.reach_p : sqrt(fmax(lim_all, 0.0)) * 1.000001 + 1e-6;
    sum_walk(I, T, reach, [&](int b) { return EACH ? I.bin_thr[b] : lim_all; },
             [&](uint64_t m, int p0, int p1, const BinInfo &B, double lm) __attribute__((always_inline)) {
                 // of this wave's queries
                 const int bin_all = !EACH && box_far2(B, x0, x1, y0, y1) < thr;
                 m &= __ballot(box_gap2(B, x0, x1, y0, y1) < (EACH ? lm : thr));
                 const uint64_t inside = __ballot(bin_all);
                 while (m) {
                     const int l = __builtin_ctzll(m);
                     m &= m - 1ull;
                     const int a = __builtin_amdgcn_readlane(p0, l), b = __builtin_amdgcn_readlane(p1, l);
                     const bool is_own = b > q0 && a < q0 + 64, is_all = (inside >> l) & 1ull;
                     for (int c = a; c < b; c += 32) {
                         if (P == 1 || ph == np) {
                             pos = c;
                             cnt = b - c < 32 ? b - c : 32;
                         }
                         all = all && is_all;
                         own = own || is_own;
                         if (++np == P) flush();
                     }
                 }
             });
    if (P > 1 && np) flush();
    if (ph != 0) return;
    if (T.item.z > 1) {
        const int64_t at = KIND == SUM_LOO ? (int64_t)T.item.w * LM_K + k : (int64_t)T.item.w;
        A.partials[at * 64 + u * Q + r] = (double)sum - (double)comp;
    } else if (qv) {
        A.den1[(int64_t)k * I.n + q] = sum;
    }
}

// Sources c0 .. c1 - 1 for candidates k .. k + N - 1: candidate k's term is
// exp2(d2f a_k) coef_k if the exact cut-off fl64(dx^2 + dy^2) < thr_k holds (ALL:
// every pair is inside), else 0, d2f = fl32(dx^2 + dy^2).  FP64 compares run at
// the FP32 rate on gfx950, so exactness costs one instruction per candidate and
// no re-check.  32 sources at a time: their positions and these N coefficients
// come in one per lane and are handed round through LDS (s_src).  (With scalar
// loads of each source the kernel waited for them two thirds of its time.)
// s_sum: this lane's Kahan pairs from candidate k on, 64 apart.  The query itself is left out.
#define LM_REC 12   // floats of a source's record for 8 candidates: x, y, coefficients
template <int N, bool ALL>
__device__ __forceinline__ void loo_run(const SumArgs &A, const SumItem &T, int k, int c0, int c1, float2 *s_sum,
                                        float *s_src)
{
    constexpr int R = (N + 2 + 3) / 4 * 4;
    const int lane = threadIdx.x & 63;
    const int64_t n = A.idx.n;
    double thr[N];
    float af[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        thr[i] = A.thr_k[k + i];
        af[i] = uni((float)A.a_k[k + i]);
    }
    const bool own = !ALL && c1 > T.item.x * 64 && c0 < T.item.x * 64 + 64;
    for (int b0 = c0; b0 < c1; b0 += 32) {
        const int cnt = c1 - b0 < 32 ? c1 - b0 : 32;
        wave_sync();
        if (lane < cnt) {
            const int p = b0 + lane;
            float rec[R] = {A.idx.pts[p].x, A.idx.pts[p].y};
#pragma unroll
            for (int i = 0; i < N; ++i) rec[2 + i] = A.coefk[(int64_t)(k + i) * n + p];
#pragma unroll
            for (int i = 0; i < R; i += 4)
                *(float4 *)(s_src + lane * R + i) = make_float4(rec[i], rec[i + 1], rec[i + 2], rec[i + 3]);
        }
        wave_sync();
        float acc[N];
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] = 0.0f;
#pragma unroll 2
        for (int j = 0; j < cnt; ++j) {
            float rec[R];
#pragma unroll
            for (int i = 0; i < R; i += 4) {
                const float4 v = *(const float4 *)(s_src + j * R + i);
                rec[i] = v.x;
                rec[i + 1] = v.y;
                rec[i + 2] = v.z;
                rec[i + 3] = v.w;
            }
            const float dx = rec[0] - T.qx, dy = rec[1] - T.qy;
            const float d2f = __builtin_fmaf(dy, dy, dx * dx);
            if (ALL) {
#pragma unroll
                for (int i = 0; i < N; ++i) acc[i] = __builtin_fmaf(fast_exp2(d2f * af[i]), rec[2 + i], acc[i]);
            } else {
                double d2 = sq2(dx, dy);
                if (own) d2 = b0 + j == T.q ? (double)INFINITY : d2;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const float e = fast_exp2(d2f * af[i]);
                    acc[i] = __builtin_fmaf(d2 < thr[i] ? e : 0.0f, rec[2 + i], acc[i]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float2 v = s_sum[i * 64];
            kahan_fold(acc[i], v.x, v.y);
            s_sum[i * 64] = v;
        }
    }
}

// Candidates ka .. kb - 1, up to 8 at a time (s_sum: from candidate k0 on).
template <bool ALL>
__device__ __forceinline__ void loo_runs(const SumArgs &A, const SumItem &T, int k0, int ka, int kb, int c0, int c1,
                                         float2 *s_sum, float *s_src)
{
    for (int k = ka; k < kb;) {
        const int left = kb - k, m = left <= 8 ? left : left < 16 ? (left + 1) / 2 : 8;
        switch (m) {
#define MKDE_LR(N) case N: loo_run<N, ALL>(A, T, k, c0, c1, s_sum + (k - k0) * 64, s_src); break;
            MKDE_LR(1) MKDE_LR(2) MKDE_LR(3) MKDE_LR(4) MKDE_LR(5) MKDE_LR(6) MKDE_LR(7) MKDE_LR(8)
#undef MKDE_LR
        }
        k += m;
    }
}

// Up to LM_K fixed bandwidths, ascending.  Each wave owns 64 queries (lane =
// query).  A bin is summed only for the candidates that reach it, without tests
// for those that hold every pair of it.  Bound by instruction issue: 9 a pair and
// 6 a candidate's term, 4 and 4 where all pairs are inside.  The 16 largest of 64
// candidates on 200,000 points: 42.7 ms with every source tested for the
// candidates four at a time and scalar loads, 30.6 ms now.
__global__ __launch_bounds__(256) void k_loo_multi(SumArgs A)
{
    extern __shared__ float2 s_loo[];   // [4][kw][64]
    __shared__ float4 s_rec[4][32 * LM_REC / 4];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ka = blockIdx.y * A.kw, kb = ka + A.kw < A.K ? ka + A.kw : A.K;
    SumItem T;
    if (!sum_item(A, (int64_t)blockIdx.x * 4 + wid, T)) return;
    float2 *s_sum = s_loo + wid * A.kw * 64 + lane;
    float *s_src = (float *)s_rec[wid];
    for (int k = 0; k < kb - ka; ++k) s_sum[k * 64] = make_float2(0.0f, 0.0f);
    const int q0 = T.item.x * 64;
    // all candidates' ordinals: the work list counts them for the largest
    const double tmax = A.thr_k[A.K - 1];
    sum_walk(A.idx, T, sqrt(tmax) * 1.000001 + 1e-6, [&](int) { return tmax; },
             [&](uint64_t m, int p0, int p1, const BinInfo &B, double) {
                 const double near = box_gap2(B, T.mnx, T.mxx, T.mny, T.mxy);
                 const double far = p1 > q0 && p0 < q0 + 64 ? (double)INFINITY
                                                            : box_far2(B, T.mnx, T.mxx, T.mny, T.mxy);
                 int k0 = ka, kf = ka;   // candidates below k0 reach no pair, those from kf on hold all
                 for (int k = ka; k < kb; ++k) {
                     const double t = A.thr_k[k];
                     k0 += t <= near ? 1 : 0;
                     kf += t <= far ? 1 : 0;
                 }
                 m &= __ballot(k0 < kb);
                 while (m) {
                     const int l = __builtin_ctzll(m);
                     m &= m - 1ull;
                     const int a = __builtin_amdgcn_readlane(p0, l), b = __builtin_amdgcn_readlane(p1, l);
                     const int f = __builtin_amdgcn_readlane(kf, l);
                     loo_runs<false>(A, T, ka, __builtin_amdgcn_readlane(k0, l), f, a, b, s_sum, s_src);
                     loo_runs<true>(A, T, ka, f, kb, a, b, s_sum, s_src);
                 }
             });
    if (T.item.z > 1) {
        double *pp = A.partials + ((int64_t)T.item.w * LM_K + ka) * 64 + lane;
        for (int k = 0; k < kb - ka; ++k) pp[k * 64] = (double)s_sum[k * 64].x - (double)s_sum[k * 64].y;
    } else if (T.qv) {
        for (int k = 0; k < kb - ka; ++k) A.den1[(int64_t)(ka + k) * A.idx.n + T.q] = s_sum[k * 64].x;
    }
}

// Parts of split waves: FP64 partials added in part order, rounded once.
// splits[k] = {wave, slot0, parts}; m = values per query (1, or MKDE_LM_K).
__global__ void k_point_merge(int64_t n, int m, int K, const unsigned *n_split_dev, const int4 *splits,
                              const double *partials, float *den)
{
    if (n_split_dev && blockIdx.x >= *n_split_dev) return;   // grid sized for the most splits
    const int4 sp = splits[blockIdx.x];
    const int lane = threadIdx.x & 63, kk = threadIdx.x >> 6;   // 64 x 4 threads
    const int64_t q = (int64_t)sp.x * 64 + lane;
    if (q >= n) return;
    for (int k = kk; k < K; k += 4) {
        double t = 0.0;
        for (int j = 0; j < sp.z; ++j) t += partials[((int64_t)(sp.y + j) * m + k) * 64 + lane];
        den[(int64_t)k * n + q] = (float)t;
    }
}


// ==================================================== range candidates ====
// Candidate sets of N1 with the QUERY's own threshold (tests only).  Pass 1
// counts (out_idx == nullptr), pass 2 fills at offsets (bin-order indexes).

struct RangeArgs {
    PointIndex idx;       // the query threshold is the point's own pts[q].thr
    int64_t *counts;      // bin order
    const int64_t *offsets;
    int32_t *out_idx;
};

__global__ __launch_bounds__(256) void k_range(RangeArgs A)
{
    __shared__ int s_bins[256];
    __shared__ int s_wcnt[4];
    __shared__ float s_sx[256];
    __shared__ float s_sy[256];
    __shared__ float s_red[4][4];

    const PointIndex &I = A.idx;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t q = (int64_t)blockIdx.x * 256 + tid;
    const bool qv = q < I.n;
    float qx = 0.0f, qy = 0.0f;
    double qt = -1.0;
    if (qv) {
        PtRec p = I.pts[q];
        qx = p.x;
        qy = p.y;
        qt = p.thr;
    }
    float mnx = qv ? qx : FLT_MAX, mxx = qv ? qx : -FLT_MAX, mny = qv ? qy : FLT_MAX, mxy = qv ? qy : -FLT_MAX;
    for (int d = 32; d >= 1; d >>= 1) {
        mnx = fminf(mnx, __shfl_xor(mnx, d, WAVE));
        mxx = fmaxf(mxx, __shfl_xor(mxx, d, WAVE));
        mny = fminf(mny, __shfl_xor(mny, d, WAVE));
        mxy = fmaxf(mxy, __shfl_xor(mxy, d, WAVE));
    }
    if (lane == 0) {
        s_red[wave][0] = mnx;
        s_red[wave][1] = mxx;
        s_red[wave][2] = mny;
        s_red[wave][3] = mxy;
    }
    __syncthreads();
    mnx = fminf(fminf(s_red[0][0], s_red[1][0]), fminf(s_red[2][0], s_red[3][0]));
    mxx = fmaxf(fmaxf(s_red[0][1], s_red[1][1]), fmaxf(s_red[2][1], s_red[3][1]));
    mny = fminf(fminf(s_red[0][2], s_red[1][2]), fminf(s_red[2][2], s_red[3][2]));
    mxy = fmaxf(fmaxf(s_red[0][3], s_red[1][3]), fmaxf(s_red[2][3], s_red[3][3]));

    int bxa, bxb, bya, byb;
    const double reach = *I.reach_p;
    const double qthr_max = reach * reach;
    bin_range(I.bg, mnx, mxx, mny, mxy, reach, bxa, bxb, bya, byb);
    const int nbx_r = bxb - bxa + 1;
    const int nb_total = nbx_r * (byb - bya + 1);
    int64_t cnt_q = 0;
    int64_t wpos = (A.out_idx && qv) ? A.offsets[q] : 0;
    for (int base = 0; base < nb_total; base += 256) {
        const int kk = base + tid;
        bool cand = false;
        int b = 0;
        if (kk < nb_total) {
            b = (bya + kk / nbx_r) * I.bg.nbx + (bxa + kk % nbx_r);
            if (I.bin_start[b + 1] > I.bin_start[b])
                cand = box_gap2(I.bin_box[b], mnx, mxx, mny, mxy) < qthr_max;
        }
        int nb;
        int slot = block_compact256(cand, s_wcnt, &nb);
        if (cand) s_bins[slot] = b;
        __syncthreads();
        for (int kb = 0; kb < nb; ++kb) {
            const int bb = s_bins[kb];
            const int st = I.bin_start[bb], en = I.bin_start[bb + 1];
            for (int off = st; off < en; off += 256) {
                const int cnt = (en - off) < 256 ? (en - off) : 256;
                if (tid < cnt) {
                    PtRec p = I.pts[off + tid];
                    s_sx[tid] = p.x;
                    s_sy[tid] = p.y;
                }
                __syncthreads();
                if (qv) {
                    for (int s = 0; s < cnt; ++s) {
                        const double d2 = sq2(qx - s_sx[s], qy - s_sy[s]);
                        if (d2 < qt) {
                            if (A.out_idx) A.out_idx[wpos++] = off + s;
                            cnt_q++;
                        }
                    }
                }
                __syncthreads();
            }
        }
        __syncthreads();
    }
    if (qv && !A.out_idx) A.counts[q] = cnt_q;
}

// ============================================================ boundary ====

__global__ void k_valid(int64_t ncells, const float *mask, float nodata, uint8_t *valid)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ncells) valid[i] = mask[i] != nodata ? 1 : 0;
}

// Valid-cell runs of the mask rows, one wave per row, columns 64 at a time:
// a run starts at a valid cell whose left neighbour is not valid (or at
// column 0) and ends at a valid cell whose right neighbour is not valid (or
// at the last column).  k_run_count counts each row's runs; k_run_fill
// writes them, in column order, from the row's first index (the exclusive
// scan of the counts): a start is run number (starts before it in the row),
// an end belongs to the last start at or before it.
__device__ __forceinline__ void run_flags(const uint8_t *row, int64_t ncols, int64_t c, bool &start, bool &end)
{
    const bool v = c < ncols && row[c];
    start = v && (c == 0 || !row[c - 1]);
    end = v && (c == ncols - 1 || !row[c + 1]);
}

__global__ __launch_bounds__(256) void k_run_count(int64_t ncols, int64_t nrows, const uint8_t *valid, unsigned *cnt)
{
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= nrows) return;   // whole wave
    const uint8_t *row = valid + r * ncols;
    unsigned n = 0;
    for (int64_t c0 = 0; c0 < ncols; c0 += WAVE) {
        bool s, e;
        run_flags(row, ncols, c0 + lane, s, e);
        n += (unsigned)__popcll(__ballot(s));
    }
    if (lane == 0) cnt[r] = n;
}

__global__ __launch_bounds__(256) void k_run_fill(int64_t ncols, int64_t nrows, const uint8_t *valid,
                                                  const unsigned *first, int2 *se, int2 *row_run)
{
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= nrows) return;   // whole wave
    const uint8_t *row = valid + r * ncols;
    const uint64_t le = ~0ull >> (63 - lane);   // lanes 0 .. lane
    int64_t k = first[r];
    int s0 = 0, e1 = 0;   // first start and last end of the row
    const int64_t k0 = k;
    for (int64_t c0 = 0; c0 < ncols; c0 += WAVE) {
        const int64_t c = c0 + lane;
        bool s, e;
        run_flags(row, ncols, c, s, e);
        const uint64_t ms = __ballot(s);
        const int64_t upto = k + __popcll(ms & le);   // starts at columns <= c
        if (s) se[upto - 1].x = (int)c;
        if (e) se[upto - 1].y = (int)c;
        const uint64_t me = __ballot(e);
        if (ms && k == k0) s0 = (int)c0 + __builtin_ctzll(ms);
        if (me) e1 = (int)c0 + 63 - __builtin_clzll(me);
        k += __popcll(ms);
    }
    if (lane == 0) row_run[r] = k - k0 == 1 ? make_int2(s0, e1) : make_int2(k == k0 ? 1 : -1, 0);
}

// run_ptr[r] = first index of row r's runs, run_ptr[nrows] = the total.
__global__ void k_run_ptr(int64_t nrows, const unsigned *first, const unsigned *total, int64_t *ptr)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrows) ptr[r] = first[r];
    else if (r == nrows) ptr[r] = *total;
}

// MarkBoundary: a valid cell is a boundary cell iff it is on the outer rows /
// columns or one of its 8 neighbours is nodata (tiled:3993-4059).  Boundary
// cell centres are appended to blist (order irrelevant: only minima are taken),
// counted in bcount.  Row r = blockIdx.y (+ gridDim.y strides), column from
// blockIdx.x: no 64-bit division per cell.  For rasters whose distances are
// taken by brute force; the others use k_boundary_leaf.
__global__ __launch_bounds__(256) void k_boundary(GridDesc g, const uint8_t *valid, uint8_t *flags, float2 *blist,
                                                  unsigned long long *bcount)
{
    const int64_t nc = g.ncols, nr = g.nrows;
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    for (int64_t r = blockIdx.y; r < nr; r += gridDim.y) {
        const int64_t i = r * nc + c;
        uint8_t f = 0;
        if (valid[i]) {
            if (r == 0 || r == nr - 1 || c == 0 || c == nc - 1) {
                f = 1;
            } else {
                const uint8_t *up = valid + (r - 1) * nc + c, *mid = valid + r * nc + c, *dn = valid + (r + 1) * nc + c;
                f = !(up[-1] & up[0] & up[1] & mid[-1] & mid[1] & dn[-1] & dn[0] & dn[1]);
            }
        }
        flags[i] = f;
        if (f) {
            const unsigned long long k = atomicAdd(bcount, 1ull);
            const double nrm05 = (double)nr - 0.5;
            blist[k] = make_float2(cell_x(g.xll, g.cs, c), cell_y(g.yll, g.cs, nrm05, r));
        }
    }
}

// CalcDist2Boundary (CPU semantics, tiled:4091-4131): min over boundary cells
// of fl64(dx^2 + dy^2), DBL_MAX if none.  Boundary centres streamed via LDS.
// A float screen skips a cell when fl32(dx*dx + dy*dy) exceeds the running
// minimum by more than a relative 2^-20 (its error is below 2^-22 relative),
// so only cells that can lower the minimum take the exact FP64 path.
__global__ __launch_bounds__(256) void k_dist_boundary(int64_t n, const float *x, const float *y, const float2 *blist,
                                                       int64_t nb, double *dist)
{
    __shared__ float2 s_b[1024];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float px = i < n ? x[i] : 0.0f, py = i < n ? y[i] : 0.0f;
    double m = DBL_MAX;
    float mf = FLT_MAX;   // screen: cells with d2f > mf cannot lower m
    for (int64_t base = 0; base < nb; base += 1024) {
        const int cnt = (nb - base) < 1024 ? (int)(nb - base) : 1024;
        for (int t = threadIdx.x; t < cnt; t += blockDim.x) s_b[t] = blist[base + t];
        __syncthreads();
        for (int t = 0; t < cnt; ++t) {
            const float2 b = s_b[t];
            const float dx = b.x - px, dy = b.y - py;
            const float d2f = __builtin_fmaf(dy, dy, dx * dx);
            if (d2f <= mf) {
                const double d2 = sq2(dx, dy);
                if (d2 < m) {
                    m = d2;
                    mf = (float)(m * (1.0 + 1.0 / 1048576.0));
                    if (!(mf < FLT_MAX)) mf = FLT_MAX;
                }
            }
        }
        __syncthreads();
    }
    if (i < n) dist[i] = m;
}

// ---- boundary flags, hierarchy and nearest-boundary search
//
// k_boundary_leaf: flags (as k_boundary) and leaves in one pass over the valid
// cells.  One wave takes 64 columns x 16 rows, four leaves side by side: a row's
// valid cells are one ballot, its boundary cells a few 64-bit scalar operations
// on three neighbouring rows' ballots, and a leaf's 16 bits of a row a slice of
// the result.  Cells outside the raster count as nodata, which makes the outer
// rows and columns boundary cells.  The box of a leaf spans its extreme columns
// and rows (cell_x is non-decreasing in the column, cell_y non-increasing in
// the row).  Against a flags pass and one thread per leaf reading them back:
// 54 -> 13 us at 1500 x 1200 cells, 282 -> 142 us at 8192^2.
__global__ __launch_bounds__(256) void k_boundary_leaf(GridDesc g, const uint8_t *valid, uint8_t *flags, int nx, int ny,
                                                       int pnx, int wnx, int64_t nwaves, uint4 *bits, float4 *box,
                                                       unsigned long long *bcount)
{
    const int lane = threadIdx.x & 63;
    const int64_t wv = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wv >= nwaves) return;   // whole wave
    const int by = (int)(wv / wnx), bx0 = (int)(wv % wnx) * 4;
    const int64_t nc = g.ncols, nr = g.nrows;
    const int64_t c0 = (int64_t)bx0 * MKDE_BT_S, c = c0 + lane, r0 = (int64_t)by * MKDE_BT_S;
    // valid cells of rows r0 - 1 .. r0 + 16, and whether a cell's left and
    // right neighbours are valid too
    const int64_t ch = lane == 0 ? c0 - 1 : c0 + 64;   // halo column of lanes 0 and 63
    const bool halo = (lane == 0 || lane == 63) && ch >= 0 && ch < nc;
    uint8_t v[MKDE_BT_S + 2], e[MKDE_BT_S + 2];
#pragma unroll
    for (int k = 0; k < MKDE_BT_S + 2; ++k) {
        const int64_t r = r0 + k - 1;
        const bool in = r >= 0 && r < nr;
        v[k] = in && c < nc ? valid[r * nc + c] : 0;
        e[k] = in && halo ? valid[r * nc + ch] : 0;
    }
    uint64_t V[MKDE_BT_S + 2], H[MKDE_BT_S + 2];
#pragma unroll
    for (int k = 0; k < MKDE_BT_S + 2; ++k) {
        V[k] = __ballot(v[k] != 0);
        const uint64_t E = __ballot(e[k] != 0);
        H[k] = V[k] & ((V[k] << 1) | (E & 1ull)) & ((V[k] >> 1) | (E & (1ull << 63)));
    }
    unsigned mine = 0;   // row (lane & 15) of leaf lane >> 4: its 16 bits
    int count = 0;
#pragma unroll
    for (int k = 1; k <= MKDE_BT_S; ++k) {
        const uint64_t b = V[k] & ~(H[k - 1] & H[k] & H[k + 1]);
        const int64_t r = r0 + k - 1;
        if (r < nr && c < nc) flags[r * nc + c] = (uint8_t)((b >> lane) & 1ull);
        count += __popcll(b);
        const unsigned sl = (unsigned)(b >> (lane & 48)) & 0xffffu;
        mine = (lane & 15) == k - 1 ? sl : mine;
    }
    if (lane == 0 && count) atomicAdd(&bcount[(wv % MKDE_CNT_SLOTS) * MKDE_CNT_STRIDE], (unsigned long long)count);
    unsigned cols = mine;   // columns of the leaf with a boundary cell
    for (int d = 1; d < 16; d <<= 1) cols |= __shfl_xor(cols, d, WAVE);
    const unsigned rows = (unsigned)(__ballot(mine != 0) >> (lane & 48)) & 0xffffu;
    const int bx = bx0 + (lane >> 4);
    // missing children of the level above are written as empty nodes
    if (bx >= 2 * pnx) return;
    const int64_t t = bt_node(bx, by, pnx);
    ((uint16_t *)bits)[t * 16 + (lane & 15)] = (uint16_t)mine;
    if (lane & 15) return;
    float4 b = make_float4(FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX);
    if (cols && bx < nx && by < ny) {
        const double nrm05 = (double)nr - 0.5;
        const int64_t cb = (int64_t)bx * MKDE_BT_S;
        b.x = cell_x(g.xll, g.cs, cb + __builtin_ctz(cols));
        b.z = cell_x(g.xll, g.cs, cb + 31 - __builtin_clz(cols));
        b.y = cell_y(g.yll, g.cs, nrm05, r0 + 31 - __builtin_clz(rows));
        b.w = cell_y(g.yll, g.cs, nrm05, r0 + __builtin_ctz(rows));
    }
    box[t] = b;
}

__device__ __forceinline__ float4 box_union(float4 a, float4 b)
{
    return make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fmaxf(a.z, b.z), fmaxf(a.w, b.w));
}

// Boxes of up to four levels above level l: a workgroup covers 16 x 16 nodes of
// level l + 1 and hands their boxes up through LDS (seven levels: 28 us in a
// launch each, 7 us in two).  Empty boxes are neutral in the union.
__global__ __launch_bounds__(256) void k_bt_up(BndTree T, int l, float4 *box)
{
    __shared__ float4 s_b[256];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    for (int k = 1; k <= 4 && l + k < T.nlev; ++k) {
        const int m = l + k, w = 16 >> (k - 1);   // w x w nodes of level m in this workgroup
        const bool on = tx < w && ty < w;
        const int X = (int)blockIdx.x * w + tx, Y = (int)blockIdx.y * w + ty;
        float4 b = make_float4(FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX);
        if (k == 1) {
            if (X < T.nx[m] && Y < T.ny[m]) {
                const float4 *ch = box + T.off[l] + (((int64_t)Y * T.nx[m] + X) << 2);
                b = box_union(box_union(ch[0], ch[1]), box_union(ch[2], ch[3]));
            }
        } else if (on) {
            const int i = 2 * ty * 16 + 2 * tx;
            b = box_union(box_union(s_b[i], s_b[i + 1]), box_union(s_b[i + 16], s_b[i + 17]));
        }
        __syncthreads();   // the level below has been read
        if (on) {
            s_b[ty * 16 + tx] = b;
            const int pnx = T.nx[m + 1], pny = T.ny[m + 1];
            if (X < 2 * pnx && Y < 2 * pny) box[T.off[m] + bt_node(X, Y, pnx)] = b;
        }
        __syncthreads();
    }
}

// Lower bound of fl64(dx^2 + dy^2) over the cells of a node (gap1 is an exact
// lower bound of |fl32(u - v)| over an interval; both squares are exact).
__device__ __forceinline__ double node_lb(float4 b, float px, float py)
{
    return b.x > b.z ? DBL_MAX : sq2(gap1(px, b.x, b.z), gap1(py, b.y, b.w));
}

// CalcDist2Boundary as a search of the hierarchy that prunes nodes whose lower
// bound is not below the best squared distance so far: the result is the
// brute-force minimum over all boundary cells, exactly.  One wave searches for
// 64 neighbouring points (bin order).
//   1. Every lane searches by itself, nearest child first, down to a leaf.
//   2. The points that are still open go on together where they lie close
//      together compared with their distances (BT_WAVE_AREA): the wave keeps one
//      stack of nodes (LDS).  Up to 64 nodes are popped at a time, one per lane,
//      with their loads in flight together; children within the largest distance
//      of the open points' box are pushed.  Leaves are then taken one by one for
//      all of them, where any needs them: the leaf's cells are listed in LDS, four
//      at a time are taken without waiting on each other.
//   3. What is left, where the wave did not search or gave up, every lane finishes
//      by itself.  The wave gives up when too few points need the leaves it
//      visits: one that none needs costs it BT_COST, the others pay one a point.
// What bounds a search is its longest one: points near the centre of a round study
// area find hundreds of leaves nearly equidistant, and node by node each costs a
// memory latency, so there the wave takes nodes 64 at a time.  Near a ragged
// boundary every point needs a few leaves of its own and the wave would look at
// all leaves around: 64 points on 8192^2 cells with 2% nodata cells 119 us with a
// stack per lane, 33.9 ms by the wave alone, 72 us now; half the raster like that
// and half without, 200,000 points 305 / 1878 / 292 us; a coast, 1M points 889 /
// 1662 / 337 us; a disk with 20 holes, 1M points 1270 / 333 / 355 us; a plain disk
// on 4096^2, 200,000 points 6.2 / 0.77 / 0.77 ms (times with the flags and the
// hierarchy, 60 to 150 us).

#define BT_STACK 1024
// Nodes popped at a time are limited so that their children fit below this; at
// the limit nodes go one by one, which needs at most 3 more per level.
#define BT_STACK_SOFT (BT_STACK - 64)
// The wave looks at the leaves within far of the open points' box, a lane at those
// within far of its point.  Area of the first in far^2 up to which the wave starts,
// its cost of a leaf that no point needs, and what it may lose before it gives up.
// (Area 10: 50,000 points in a disk with 5 holes 89 instead of 68 us, 64 points on 2048^2
// cells without holes 97 instead of 172.  Credit 512 / 1024 / 2048 at that cost: a disk
// with 20 holes, 1M points 491 / 355 / 355 us, a coast 294 / 337 / 420.)
#define BT_WAVE_AREA 20.0
#define BT_COST 2
#define BT_CREDIT 1024

// A lane's search, depth first: at node (ix, iy) of level lev, with the children
// that are left at the nodes above in 4 bits a level (level l in bits 4 l - 4 ..
// 4 l - 1; none below lev), so it needs no stack.
struct LaneSearch {
    int lev, ix, iy;
    uint64_t todo;
};

__device__ __forceinline__ void leaf_best(const GridDesc &g, const BndTree &T, int ix, int iy, double nrm05, float px,
                                          float py, double &best)
{
    const int64_t at = bt_node(ix, iy, T.nx[1]);
    const uint4 m0 = T.bits[2 * at], m1 = T.bits[2 * at + 1];
    const unsigned m[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        unsigned v = m[w];
        while (v) {
            const int k = w * 32 + __builtin_ctz(v);
            v &= v - 1u;
            const float cx = cell_x(g.xll, g.cs, (int64_t)ix * MKDE_BT_S + (k & (MKDE_BT_S - 1)));
            const float cy = cell_y(g.yll, g.cs, nrm05, (int64_t)iy * MKDE_BT_S + (k >> 4));
            best = fmin(best, sq2(cx - px, cy - py));
        }
    }
}

// Of the four children ch of a node, those of `left` that may hold a cell nearer than
// best: all of them in rest, the nearest in k (-1: none).
__device__ __forceinline__ void nearest_child(const float4 *ch, unsigned left, float px, float py, double best,
                                              unsigned &rest, int &k)
{
    double lb = best;
    rest = 0;
    k = -1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double l = (left >> j) & 1u ? node_lb(ch[j], px, py) : DBL_MAX;
        rest |= l < best ? 1u << j : 0u;
        k = l < lb ? j : k;
        lb = l < lb ? l : lb;
    }
}

// One step (todo != 0): back to the lowest node with children left, and to the
// nearest of them; a leaf's cells are taken.
__device__ __forceinline__ void lane_step(const GridDesc &g, const BndTree &T, double nrm05, float px, float py,
                                          LaneSearch &L, double &best)
{
    const int at = __builtin_ctzll(L.todo) & ~3, up = (at >> 2) + 1 - L.lev;
    L.lev += up;
    L.ix >>= up;
    L.iy >>= up;
    const float4 *ch = T.box + T.off[L.lev - 1] + (((int64_t)L.iy * T.nx[L.lev] + L.ix) << 2);
    unsigned rest;
    int k;
    nearest_child(ch, (unsigned)(L.todo >> at) & 15u, px, py, best, rest, k);
    L.todo &= ~((uint64_t)15 << at);
    if (k < 0) return;
    L.todo |= (uint64_t)(rest & ~(1u << k)) << at;
    L.ix = 2 * L.ix + (k & 1);
    L.iy = 2 * L.iy + (k >> 1);
    --L.lev;
    if (L.lev > 0) L.todo |= (uint64_t)15 << (at - 4);
    else leaf_best(g, T, L.ix, L.iy, nrm05, px, py, best);
}

__global__ __launch_bounds__(64) void k_dist_tree(int64_t n, const float *xs, const float *ys, const int *perm,
                                                  GridDesc g, BndTree T, double *dist)
{
    __shared__ unsigned s_node[BT_STACK];
    __shared__ float2 s_cell[MKDE_BT_S * MKDE_BT_S + 4];   // cell centres of a leaf
    const int lane = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * 64 + lane;
    const bool on = i < n;
    const float px = xs[on ? i : n - 1], py = ys[on ? i : n - 1];
    const double nrm05 = (double)g.nrows - 0.5;
    const int top = T.nlev - 1;
    double best = DBL_MAX;

    // 1. down to a leaf, all lanes level by level
    LaneSearch L{0, 0, 0, 0};
    bool down = on;
    for (int lev = top; lev > 0; --lev) {
        unsigned rest;
        int k;
        nearest_child(T.box + T.off[lev - 1] + (((int64_t)L.iy * T.nx[lev] + L.ix) << 2), 15u, px, py, best, rest, k);
        down = down && k >= 0;
        if (!down) continue;
        L.todo |= (uint64_t)(rest & ~(1u << k)) << (4 * lev - 4);
        L.ix = 2 * L.ix + (k & 1);
        L.iy = 2 * L.iy + (k >> 1);
    }
    if (down) leaf_best(g, T, L.ix, L.iy, nrm05, px, py, best);
    float wx0 = 0.0f, wx1 = 0.0f, wy0 = 0.0f, wy1 = 0.0f;   // box of the open points
    double far = 0.0;   // no node beyond this is needed
    auto wave_far = [&]() {
        double v = best;
        for (int d = 32; d >= 1; d >>= 1) v = fmax(v, __shfl_xor(v, d, WAVE));
        return v;
    };

    // 2. the open ones together
    const bool open = L.todo != 0;
    const double closed = best;
    if (!open) best = -1.0;   // nothing is nearer
    int sp = 0, credit = BT_CREDIT;
    if (__ballot(open)) {
        wx0 = uni(wave_min(open ? px : FLT_MAX));
        wx1 = uni(wave_max(open ? px : -FLT_MAX));
        wy0 = uni(wave_min(open ? py : FLT_MAX));
        wy1 = uni(wave_max(open ? py : -FLT_MAX));
        far = wave_far();
        const double f = sqrt(far), w = (double)wx1 - (double)wx0 + 2.0 * f, h = (double)wy1 - (double)wy0 + 2.0 * f;
        if (w * h <= BT_WAVE_AREA * far) sp = 1;
        if (lane == 0) s_node[0] = (unsigned)top << 28;
    }
    const bool together = sp > 0;
    while (sp > 0 && credit >= 0) {
        wave_sync();
        const int room = (BT_STACK_SOFT - sp) / 3;
        int take = sp < 64 ? sp : 64;
        take = take < room ? take : (room > 1 ? room : 1);
        sp -= take;
        const bool mine = lane < take;
        const unsigned e = s_node[sp + (mine ? lane : 0)];
        wave_sync();
        const int lev = (int)(e >> 28), iy = (int)((e >> 14) & 0x3fff), ix = (int)(e & 0x3fff);
        const int64_t at = bt_node(ix, iy, T.nx[lev + 1]);
        const float4 own = T.box[T.off[lev] + at];
        const bool need = mine && box_gap2(BinInfo{own.x, own.y, own.z, own.w}, wx0, wx1, wy0, wy1) < far;
        float4 cb[4];
        uint4 m0 = make_uint4(0, 0, 0, 0), m1 = m0;
        if (need && lev > 0) {
            const float4 *ch = T.box + T.off[lev - 1] + (((int64_t)iy * T.nx[lev] + ix) << 2);
#pragma unroll
            for (int k = 0; k < 4; ++k) cb[k] = ch[k];
        }
        if (need && lev == 0) {
            m0 = T.bits[2 * at];
            m1 = T.bits[2 * at + 1];
        }
        // leaves, one after the other for all points
        uint64_t leaves = __ballot(need && lev == 0);
        if (leaves) {
            do {
                const int l = __builtin_ctzll(leaves);
                leaves &= leaves - 1ull;
                auto get = [&](unsigned v) { return (unsigned)__builtin_amdgcn_readlane((int)v, l); };
                auto getf = [&](float v) { return __uint_as_float(get(__float_as_uint(v))); };
                const float4 lb = make_float4(getf(own.x), getf(own.y), getf(own.z), getf(own.w));
                const uint64_t who = __ballot(node_lb(lb, px, py) < best);
                credit += who ? __popcll(who) : -BT_COST;
                if (!who) continue;
                const uint64_t m[4] = {get(m0.x) | (uint64_t)get(m0.y) << 32, get(m0.z) | (uint64_t)get(m0.w) << 32,
                                       get(m1.x) | (uint64_t)get(m1.y) << 32, get(m1.z) | (uint64_t)get(m1.w) << 32};
                const int64_t c0 = (int64_t)get((unsigned)ix) * MKDE_BT_S, r0 = (int64_t)get((unsigned)iy) * MKDE_BT_S;
                // this lane's column and its rows 4 j + (lane >> 4)
                const float cx = cell_x(g.xll, g.cs, c0 + (lane & 15));
                int cnt = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (!m[j]) continue;
                    const float cy = cell_y(g.yll, g.cs, nrm05, r0 + 4 * j + (lane >> 4));
                    if ((m[j] >> lane) & 1ull)
                        s_cell[cnt + __popcll(m[j] & ((1ull << lane) - 1ull))] = make_float2(cx, cy);
                    cnt += __popcll(m[j]);
                }
                wave_sync();
                // up to a multiple of four: the last cell again
                const float2 last = s_cell[cnt - 1];
                if (lane < 3) s_cell[cnt + lane] = last;
                wave_sync();
                for (int k = 0; k < cnt; k += 4) {
                    const float2 q0 = s_cell[k], q1 = s_cell[k + 1], q2 = s_cell[k + 2], q3 = s_cell[k + 3];
                    const double d0 = sq2(q0.x - px, q0.y - py), d1 = sq2(q1.x - px, q1.y - py);
                    const double d2 = sq2(q2.x - px, q2.y - py), d3 = sq2(q3.x - px, q3.y - py);
                    best = fmin(best, fmin(fmin(d0, d1), fmin(d2, d3)));
                }
                wave_sync();
            } while (leaves);
            far = wave_far();
        }
        // children of the other nodes
        if (__ballot(need && lev > 0)) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                bool push = false;
                if (need && lev > 0)
                    push = cb[k].x <= cb[k].z &&
                           box_gap2(BinInfo{cb[k].x, cb[k].y, cb[k].z, cb[k].w}, wx0, wx1, wy0, wy1) < far;
                const uint64_t pm = __ballot(push);
                if (push)
                    s_node[sp + __popcll(pm & ((1ull << lane) - 1ull))] =
                        ((unsigned)(lev - 1) << 28) | ((unsigned)(2 * iy + (k >> 1)) << 14) | (unsigned)(2 * ix + (k & 1));
                sp += __popcll(pm);
            }
        }
    }
    // 3. all has been seen, or each lane goes on where it was
    if (!open) best = closed;
    if (together && sp == 0) L.todo = 0;
    while (__ballot(L.todo != 0))
        if (L.todo) lane_step(g, T, nrm05, px, py, L, best);
    if (on) dist[perm[i]] = best;
}

// ===================================================== edge correction ====
//
// EdgeCorrectionWeightsExact with O(R) work per point instead of O(R^2).
// The integrand is separable on the mask grid:
//   K(c, r) = exp2(dx2_c a) * exp2(dy2_r a) / (2 pi h2f)
// and for a fixed row the cells inside the cut-off form one interval of
// columns (the reference's test is monotone in |dx|).  One wave handles one
// point: columns of the NARROW box (tiled:2716-2727) are processed in chunks
// of EC_CW (1024), with an FP64 prefix sum of exp2(dx2 a) in LDS; lanes then
// take rows, find each row's exact column interval, intersect it with the
// row's valid-cell runs and add exp2(dy2 a) * (prefix differences).
// Output ew = 1/(cellArea * sum / (2 pi h2f)); points whose boundary distance
// is >= 9 h2f were given weight 1 by k_ec_active.


struct EcArgs {
    GridDesc g;
    MaskRuns runs;
    const float *colx, *rowy;   // cell-centre tables of the mask grid
    const float *x, *y;     // original order
    const float *h;         // original order (nullable when h_fixed > 0 or h_dev)
    float h_fixed;
    const float *h_dev;     // non-null: every point's bandwidth is *h_dev (a device value)
    const int *count;       // non-null: {narrow, wide} list lengths on the device
    const int *list;        // active points
    float *ew;              // original order
    unsigned long long *n_eval;
    int cx32;               // cell centres of the mask's columns are exact in FP32 (host-checked)
    double inv_cs;          // 1 / cell size
    int cs_exact;           // the cell size is a power of two: x / cs == x * inv_cs exactly
};

__device__ __forceinline__ float ec_bandwidth(const EcArgs &A, int p)
{
    return A.h_dev ? *A.h_dev : (A.h_fixed > 0.0f ? A.h_fixed : A.h[p]);
}

// NARROW box with the reference's macro semantics (Utilities.h:16-17,30-31;
// tiled:2716-2727): size_t arithmetic for row_upper / col_upper.
struct DivCs {   // division by the cell size
    double cs;
    __device__ __forceinline__ double operator()(double v) const { return v / cs; }
};
struct MulInvCs {   // the same for a cell size that is a power of two
    double inv;
    __device__ __forceinline__ double operator()(double v) const { return v * inv; }
};
template <class D>
__device__ __forceinline__ void narrow_box_d(const GridDesc &g, const D &div, float px, float py, float h, int &rl,
                                             int &ru, int &cl, int &cu)
{
    const uint64_t nR = (uint64_t)g.nrows, nC = (uint64_t)g.ncols;
    const double yll = g.yll, xll = g.xll, hh = h;
    const int k_top = (int)div((double)py + 3.0 * hh - yll);
    const int r = (int)(int32_t)(uint32_t)(nR - 1 - (uint64_t)(int64_t)k_top);
    rl = 0 < r ? r : 0;
    const int k_bot = (int)div((double)py - 3.0 * hh - yll);
    const uint64_t yu = nR - 1 - (uint64_t)(int64_t)k_bot;
    ru = (int)(int32_t)(uint32_t)((nR - 1 < yu) ? nR - 1 : yu);
    const int k_left = (int)div((double)px - 3.0 * hh - xll);
    cl = 0 < k_left ? k_left : 0;
    const int k_right = (int)div((double)px + 3.0 * hh - xll);
    const uint64_t kr = (uint64_t)(int64_t)k_right;
    cu = (int)(int32_t)(uint32_t)((nC - 1 < kr) ? nC - 1 : kr);
}

__device__ __forceinline__ void narrow_box(const GridDesc &g, float px, float py, float h, int &rl, int &ru, int &cl,
                                           int &cu)
{
    narrow_box_d(g, DivCs{(double)g.cs}, px, py, h, rl, ru, cl, cu);
}
// Four FP64 divisions a point are a sixth of a small box's instructions.
__device__ __forceinline__ void narrow_box(const EcArgs &A, float px, float py, float h, int &rl, int &ru, int &cl,
                                           int &cu)
{
    if (A.cs_exact) narrow_box_d(A.g, MulInvCs{A.inv_cs}, px, py, h, rl, ru, cl, cu);
    else narrow_box_d(A.g, DivCs{(double)A.g.cs}, px, py, h, rl, ru, cl, cu);
}

// Column centres of the mask grid (ColCompute) and dx = fl32(cell_x(c) - px) of a
// point (DxCompute).
struct ColCompute {
    double xll, cs;
    // columns of one raster row fit in 32 bits (one-instruction conversion)
    __device__ __forceinline__ float operator()(int64_t c) const { return cell_x(xll, cs, (int64_t)(int)c); }
};
// CX32: the grid's centres fl32(xll + (c + 0.5) cs) (FP64 arithmetic) equal
// fl32(fma(c + 0.5, cs, xll)) in FP32 for every column (checked on the host
// column by column: then the FP32 form, three instructions instead of five,
// gives the same centres).
template <bool CX32>
struct DxCompute {
    double xll, cs;
    float px;
    __device__ __forceinline__ float operator()(int64_t c) const
    {
        if constexpr (CX32) return __builtin_fmaf((float)(int)c + 0.5f, (float)cs, (float)xll) - px;
        else return ColCompute{xll, cs}(c) - px;
    }
};
template <class DX>
__device__ __forceinline__ bool pred_col(const DX &dxf, int64_t c, float px, double dy2, double thr)
{
    const float dx = dxf(c);
    return __dadd_rn(sqd(dx), dy2) < thr;
}

// Exact column interval [lo, hi] within [cl, cu] of the cells of one row that
// are inside the cut-off; lo > hi when empty.  cn is the column of [cl, cu]
// nearest to px (|dx| is smallest there, and the predicate is monotone in the
// distance from cn on either side).  The first guess (FP32 square root,
// multiplication by 1/cs) only seeds the search: the four predicates that
// confirm it (both ends, one step beyond each end) are evaluated together, so
// table loads of their centres are in flight at once; when the seed is off,
// the row is empty unless cn is inside, and the ends are moved by the exact
// predicate until they are the last columns inside.
template <class DX>
__device__ __forceinline__ void row_interval(const DX &colx, double xll, double inv_cs, int cl, int cu, int cn,
                                             float px, double dy2, double thr, int &lo, int &hi)
{
    const double rem = thr - dy2;
    const double w = rem > 0.0 ? (double)sqrtf((float)rem) : 0.0;
    const double fh = floor(((double)px + w - xll) * inv_cs - 0.5);
    const double fl = ceil(((double)px - w - xll) * inv_cs - 0.5);
    int h_e = (int)fmin(fmax(fh, (double)cn), (double)cu);
    int l_e = (int)fmin(fmax(fl, (double)cl), (double)cn);
    const int h1 = h_e < cu ? h_e + 1 : h_e, l1 = l_e > cl ? l_e - 1 : l_e;
    const bool p_h = pred_col(colx, h_e, px, dy2, thr);
    const bool p_h1 = pred_col(colx, h1, px, dy2, thr) & (h_e < cu);
    const bool p_l = pred_col(colx, l_e, px, dy2, thr);
    const bool p_l1 = pred_col(colx, l1, px, dy2, thr) & (l_e > cl);
    if (!(p_h & !p_h1 & p_l & !p_l1)) {
        // cn is inside whenever any column is (p_h implies it)
        if (!pred_col(colx, cn, px, dy2, thr)) {
            lo = 1;
            hi = 0;
            return;
        }
#pragma unroll 1
        while (h_e < cu && pred_col(colx, h_e + 1, px, dy2, thr)) ++h_e;
#pragma unroll 1
        while (h_e > cn && !pred_col(colx, h_e, px, dy2, thr)) --h_e;
#pragma unroll 1
        while (l_e > cl && pred_col(colx, l_e - 1, px, dy2, thr)) --l_e;
#pragma unroll 1
        while (l_e < cn && !pred_col(colx, l_e, px, dy2, thr)) ++l_e;
    }
    lo = l_e;
    hi = h_e;
}

// Points whose boundary distance is below the cut-off get a work-list entry:
// count[0] narrow points from the front of list (box at most cw_narrow
// columns wide: k_ec, one wave per point, column chunks of cw_narrow),
// count[1] wide points from the back (wider boxes up to cw_wide columns:
// k_ec_wide, the whole box in LDS), count[2] the widest wide box.
//
// List slots are reserved per workgroup (LDS adds per wave, then one global
// atomic per list): atomics on one address serialise at some 18 ns each, which
// at one workgroup per 256 points was the whole of the 71 us a pass over 1M
// points took; at one per 2048 it takes 16 us.
#define EC_ACT_T 512
#define EC_ACT_K 4   // points per thread

__global__ __launch_bounds__(EC_ACT_T) void k_ec_active(int64_t n, GridDesc g, double inv_cs, int cs_exact,
                                                        const float *x, const float *y, const double *dist,
                                                        const float *h, float h_fixed, const float *h_dev, float *ew,
                                                        int *list, int *count, int cw_narrow, int cw_wide)
{
    __shared__ int s_n[2], s_base[2], s_wmax;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid == 0) {
        s_n[0] = s_n[1] = 0;
        s_wmax = 0;
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
    int kind[EC_ACT_K], slot[EC_ACT_K];   // 0 narrow, 1 wide
    const int64_t i0 = (int64_t)blockIdx.x * (EC_ACT_T * EC_ACT_K) + tid;
#pragma unroll
    for (int k = 0; k < EC_ACT_K; ++k) {
        const int64_t i = i0 + (int64_t)k * EC_ACT_T;
        int w = 0;
        kind[k] = -1;
        if (i < n) {
            const float hh = h_dev ? *h_dev : (h_fixed > 0.0f ? h_fixed : h[i]);
            const double h2 = (double)(float)(hh * hh);
            if (dist[i] >= 9.0 * h2) {
                ew[i] = 1.0f;
            } else {
                int rl, ru, cl, cu;
                if (cs_exact) narrow_box_d(g, MulInvCs{inv_cs}, x[i], y[i], hh, rl, ru, cl, cu);
                else narrow_box(g, x[i], y[i], hh, rl, ru, cl, cu);
                w = cu - cl + 1;
                kind[k] = (rl <= ru && w > cw_narrow && w <= cw_wide) ? 1 : 0;
            }
        }
        const uint64_t m0 = __ballot(kind[k] == 0), m1 = __ballot(kind[k] == 1);
        int b0 = 0, b1 = 0;
        if (lane == 0 && m0) b0 = atomicAdd(&s_n[0], __popcll(m0));
        if (m1) {
            int wm = kind[k] == 1 ? w : 0;
            for (int d = 32; d >= 1; d >>= 1) wm = max(wm, __shfl_xor(wm, d, WAVE));
            if (lane == 0) {
                b1 = atomicAdd(&s_n[1], __popcll(m1));
                atomicMax(&s_wmax, wm);
            }
        }
        b0 = __builtin_amdgcn_readfirstlane(b0);
        b1 = __builtin_amdgcn_readfirstlane(b1);
        slot[k] = kind[k] == 0 ? b0 + __popcll(m0 & below) : b1 + __popcll(m1 & below);
    }
    __syncthreads();
    if (tid < 2 && s_n[tid]) s_base[tid] = atomicAdd(&count[tid], s_n[tid]);
    if (tid == 2 && s_wmax) atomicMax(&count[2], s_wmax);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EC_ACT_K; ++k) {
        const int i = (int)(i0 + (int64_t)k * EC_ACT_T);
        if (kind[k] == 0) list[s_base[0] + slot[k]] = i;
        else if (kind[k] == 1) list[n - 1 - (s_base[1] + slot[k])] = i;
    }
}

// Cell-centre tables of a grid: colx[c] = cell_x(c), rowy[r] = cell_y(r).
__global__ void k_centres(GridDesc g, float *colx, float *rowy)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < g.ncols) colx[i] = cell_x(g.xll, g.cs, i);
    if (i < g.nrows) rowy[i] = cell_y(g.yll, g.cs, (double)g.nrows - 0.5, i);
}

// First run index in [rs, re) whose end >= c (binary search).
__device__ __forceinline__ int64_t first_run_ending_at_or_after(const int2 *runs, int64_t rs, int64_t re, int c)
{
    int64_t lo = rs, hi = re;
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (runs[mid].y < c) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// A point's integral: what every row needs.
struct EcPoint {
    float px, py;
    double thr, a;
    double inv_cs, pxc;     // columns per unit, and px in columns (centre of column c: c)
    double slack;           // 0.5 - tol, or negative: no row is plain
    double rem_min;
    int cl, cu;
};

// tol, in columns: how far the end of a row's chord, computed below, can lie
// from the place where the exact predicate fl64(fl32(cx - px)^2 + dy^2) < thr
// changes: half an ulp of a column centre, half an ulp of dx, and the float
// square root (1.5 ulp of at most 3h with the rounding of its argument), with a
// quarter in hand.  Rows whose chord is too short for the FP64 sum's own
// rounding to vanish in that (rem_min) are left to the search.
__device__ __forceinline__ EcPoint ec_setup(const GridDesc &g, double inv_cs, float px, float py, float h, double h2,
                                            int cl, int cu)
{
    EcPoint P;
    P.px = px;
    P.py = py;
    P.thr = 9.0 * h2;
    P.a = -MKDE_LOG2E / (2.0 * h2);
    const double xll = g.xll, cs = g.cs;
    P.inv_cs = inv_cs;
    P.pxc = ((double)px - xll) * P.inv_cs - 0.5;
    const double far = fmax(fabs(xll), fabs(xll + (double)g.ncols * cs));
    const double reach = 3.0 * (double)h;
    const double tol = 1.25 * P.inv_cs * (far + (1.0 + 3.0) * reach) * (1.0 / 16777216.0) + 1e-9;
    P.slack = tol < 0.25 && P.thr > 1e-20 && P.thr < 1e30 ? 0.5 - tol : -1.0;
    P.rem_min = P.thr * 1e-9;
    P.cl = cl;
    P.cu = cu;
    return P;
}

// Rows r, r + step, ... <= ru of a point's integral: the exact column interval
// of the row clipped to the columns [ca, cb] whose prefix sums of Ex are in s_pd
// (s_pd[k] = sum of the first k), intersected with the row's valid runs;
// acc += exp2(dy2 a) * (sum of Ex over those cells), cnt += their number.
//
// The ends of a row's chord are computed as real column positions.  Where both
// are further than tol from every centre, the interval follows without any
// predicate; the others (a row in a few hundred) are searched with the exact
// predicate (row_interval).  The next row's run is loaded at the top of an
// iteration.  About 45 instructions a row instead of 90 with four predicates
// each; a row's run is one 8-byte load instead of 24 bytes.  64 candidates on
// 200,000 points and 4096^2 cells: wide boxes 30.0 -> 20.3 ms, narrow ones 5.1 ->
// 3.5 ms; adaptive bandwidths of 1M points (both passes of a job) 2.41 -> 1.93 ms.
// VALU-bound (two thirds busy).
template <bool CX32>
__device__ __forceinline__ void ec_rows(const EcArgs &A, const EcPoint &P, const double *s_pd, int ca, int cb, int r,
                                        int ru, int step, double &acc, unsigned &cnt)
{
    const GridDesc &g = A.g;
    const double yll = g.yll, cs = g.cs, nrm05 = (double)g.nrows - 0.5;
    const DxCompute<CX32> dxf{(double)g.xll, cs, P.px};
    const int c0 = P.cl > ca ? P.cl : ca, c1 = P.cu < cb ? P.cu : cb;
    const double *pd = s_pd - ca;
    int2 run = make_int2(1, 0);
    if (r <= ru) run = A.runs.row_run[r];
    for (; r <= ru; r += step) {
        const int2 rr = run;
        const int next = r + step <= ru ? r + step : ru;
        run = A.runs.row_run[next];
        const float cy = cell_y(yll, cs, nrm05, r);
        const double dy2 = sqd(cy - P.py);
        const double rem = P.thr - dy2;
        const double w = (double)__builtin_amdgcn_sqrtf((float)rem);
        const double vh = __builtin_fma(w, P.inv_cs, P.pxc), vl = __builtin_fma(-w, P.inv_cs, P.pxc);
        int hi = (int)floor(vh), lo = (int)floor(vl) + 1;
        // (rem <= 0 makes w a NaN and the row one to be searched)
        const bool plain = (fabs(__builtin_amdgcn_fract(vh) - 0.5) <= P.slack) &
                           (fabs(__builtin_amdgcn_fract(vl) - 0.5) <= P.slack) & (rem > P.rem_min);
        if (__builtin_expect(!plain, 0)) {
            lo = 1;
            hi = 0;
            if (dy2 < P.thr) {
                const int cn = clampi((int64_t)floor(((double)P.px - (double)g.xll) / cs), P.cl, P.cu);
                row_interval(dxf, (double)g.xll, P.inv_cs, P.cl, P.cu, cn, P.px, dy2, P.thr, lo, hi);
            }
        }
        lo = lo > c0 ? lo : c0;
        hi = hi < c1 ? hi : c1;
        double seg = 0.0;
        if (__builtin_expect(rr.x >= 0, 1)) {
            const int s = rr.x > lo ? rr.x : lo;
            const int e = rr.y < hi ? rr.y : hi;
            if (s <= e) {
                seg = pd[e + 1] - pd[s];
                cnt += (unsigned)(e - s + 1);
            }
        } else if (lo <= hi) {
            const int64_t re = A.runs.run_ptr[r + 1];
#pragma unroll 1
            for (int64_t k = first_run_ending_at_or_after(A.runs.run_se, A.runs.run_ptr[r], re, lo); k < re; ++k) {
                const int2 q = A.runs.run_se[k];
                if (q.x > hi) break;
                const int s = q.x > lo ? q.x : lo;
                const int e = q.y < hi ? q.y : hi;
                seg += pd[e + 1] - pd[s];
                cnt += (unsigned)(e - s + 1);
            }
        }
        const float ey = fast_exp2((float)(dy2 * P.a));
        acc = __builtin_fma(seg, (double)ey, acc);
    }
}

// Ex over `per` columns from column c on, their running sums to s_pd[k0 + 1 ..]
// (below w); returns the last one.
template <bool CX32>
__device__ __forceinline__ double ec_columns(const GridDesc &g, const EcPoint &P, double *s_pd, int c, int k0, int per,
                                             int w)
{
    const DxCompute<CX32> dxf{(double)g.xll, (double)g.cs, P.px};
    // FP64 prefix (53-bit significand, more than the 48 of a float-float pair;
    // FP64 adds cost one VALU instruction each)
    double run = 0.0;
#pragma unroll 4
    for (int t = 0; t < per; ++t) {
        const int k = k0 + t;
        if (k < w) {
            run += (double)fast_exp2((float)(sqd(dxf(c + t)) * P.a));
            s_pd[k + 1] = run;
        }
    }
    return run;
}

// The weight 1 / (cell area * sum / (2 pi h2f)), in one division.
__device__ __forceinline__ void ec_store(const EcArgs &A, int p, double acc, double h2)
{
    A.ew[p] = (float)((h2 * (double)MKDE_TWO_PI_F) / (acc * (double)(float)(A.g.cs * A.g.cs)));
}

// EC weight of point p by one wave: column chunks of EC_CW with the FP64
// prefix sums of Ex in s_pd, rows on lanes.
template <int EC_CW, bool CX32>
__device__ __forceinline__ void ec_point_t(const EcArgs &A, double *s_pd, int p)
{
    const int lane = threadIdx.x;
    const GridDesc g = A.g;
    const float px = A.x[p], py = A.y[p];
    const float hh = ec_bandwidth(A, p);
    const double h2 = (double)(float)(hh * hh);

    int rl, ru, cl, cu;
    narrow_box(A, px, py, hh, rl, ru, cl, cu);
    double acc = 0.0;
    unsigned cnt = 0;   // a box of at most 2^31 columns per row is cut into chunks: below 2^32 a lane and chunk
    unsigned long long total = 0;
    if (rl <= ru && cl <= cu) {
        const EcPoint P = ec_setup(g, A.inv_cs, px, py, hh, h2, cl, cu);
        if (lane == 0) s_pd[0] = 0.0;
        for (int ca = cl; ca <= cu; ca += EC_CW) {
            const int cb = (ca + EC_CW - 1 < cu) ? ca + EC_CW - 1 : cu;
            const int w = cb - ca + 1;
            // lane owns columns [ca + lane*per, ...); an odd per puts the
            // lanes' FP64 prefix entries in distinct LDS banks
            const int per = ((w + WAVE - 1) / WAVE) | 1;
            const int my0 = lane * per;
            const double run = ec_columns<CX32>(g, P, s_pd, ca + my0, my0, per, w);
            // exclusive wave scan of the lane totals
            double inc = run;
            for (int d = 1; d < WAVE; d <<= 1) {
                const double o = __shfl_up(inc, d, WAVE);
                if (lane >= d) inc += o;
            }
            const double offv = inc - run;
            for (int t = 0; t < per; ++t) {
                const int k = my0 + t;
                if (k < w) s_pd[k + 1] += offv;
            }
            __syncthreads();
            cnt = 0;
            ec_rows<CX32>(A, P, s_pd, ca, cb, rl + lane, ru, WAVE, acc, cnt);
            total += cnt;
            __syncthreads();
        }
    }
    // wave reduction
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
    if (lane == 0) ec_store(A, p, acc, h2);
    if (A.n_eval) {
        for (int d = 32; d >= 1; d >>= 1) total += __shfl_xor(total, d, WAVE);
        if (lane == 0) slot_add(A.n_eval, total);
    }
}

// One wave per point of the narrow part of the list: a workgroup takes list
// items blockIdx.x, blockIdx.x + gridDim.x, ... below the narrow count (the
// device count when given, else one item per workgroup).
template <int EC_CW, bool CX32>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_ec(EcArgs A)
{
    __shared__ double s_pd[EC_CW + 1];   // 0, then the prefix sums of Ex over the chunk's columns
    const int lim = A.count ? A.count[0] : (int)gridDim.x;
    for (int it = blockIdx.x; it < lim; it += gridDim.x) ec_point_t<EC_CW, CX32>(A, s_pd, A.list[it]);
}

// Wide points (NARROW box wider than the column chunk of k_ec): one
// 256-thread workgroup per point and the whole box's prefix sums in dynamic
// LDS, so every row is visited once instead of once per chunk.  Same row
// arithmetic as k_ec.  The prefix is scanned across the workgroup (four waves).
template <bool CX32>
__device__ __forceinline__ void ec_point_wide(const EcArgs &A, double *s_pd, double *s_wt, double *s_acc,
                                              unsigned long long *s_cnt, int p)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const GridDesc g = A.g;
    const float px = A.x[p], py = A.y[p];
    const float hh = ec_bandwidth(A, p);
    const double h2 = (double)(float)(hh * hh);

    int rl, ru, cl, cu;
    narrow_box(A, px, py, hh, rl, ru, cl, cu);   // non-empty: k_ec_active checked
    const EcPoint P = ec_setup(g, A.inv_cs, px, py, hh, h2, cl, cu);
    const int w = cu - cl + 1;
    // thread owns columns [cl + tid*per, ...); an odd per puts the threads'
    // FP64 prefix entries in distinct LDS banks
    const int per = ((w + 255) / 256) | 1;
    const int my0 = tid * per;
    if (tid == 0) s_pd[0] = 0.0;
    const double run = ec_columns<CX32>(g, P, s_pd, cl + my0, my0, per, w);
    // exclusive scan of the thread totals: within each wave, then the waves
    double inc = run;
    for (int d = 1; d < WAVE; d <<= 1) {
        const double o = __shfl_up(inc, d, WAVE);
        if (lane >= d) inc += o;
    }
    if (lane == WAVE - 1) s_wt[wave] = inc;
    __syncthreads();
    double woff = 0.0;
    for (int v = 0; v < wave; ++v) woff += s_wt[v];
    const double offv = woff + (inc - run);
    for (int t = 0; t < per; ++t) {
        const int k = my0 + t;
        if (k < w) s_pd[k + 1] += offv;
    }
    __syncthreads();
    double acc = 0.0;
    unsigned cnt = 0;
    ec_rows<CX32>(A, P, s_pd, cl, cu, rl + tid, ru, 256, acc, cnt);
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, WAVE);
    if (lane == 0) s_acc[wave] = acc;
    if (A.n_eval) {
        unsigned long long total = cnt;
        for (int d = 32; d >= 1; d >>= 1) total += __shfl_xor(total, d, WAVE);
        if (lane == 0) s_cnt[wave] = total;
    }
    __syncthreads();
    if (tid == 0) {
        ec_store(A, p, ((s_acc[0] + s_acc[1]) + s_acc[2]) + s_acc[3], h2);
        if (A.n_eval) slot_add(A.n_eval, s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3]);
    }
}

// One workgroup per point of the wide part of the list (stored from the back
// of the list), items blockIdx.x, blockIdx.x + gridDim.x, ... below the wide
// count (the device count when given, else one item per workgroup).
template <bool CX32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_ec_wide(EcArgs A, int64_t n)
{
    extern __shared__ double s_pd[];   // 0, then the widest box's prefix sums
    __shared__ double s_wt[4];
    __shared__ double s_acc[4];
    __shared__ unsigned long long s_cnt[4];
    const int lim = A.count ? A.count[1] : (int)gridDim.x;
    for (int it = blockIdx.x; it < lim; it += gridDim.x) {
        ec_point_wide<CX32>(A, s_pd, s_wt, s_acc, s_cnt, A.list[n - 1 - it]);
        __syncthreads();   // the next point rewrites the LDS this one read
    }
}

// Exact count of (point, valid cell) pairs inside the cut-off on a tile (the
// density kernel's algorithmic work), one wave per point, rows on lanes.
struct CountArgs {
    GridDesc g;
    MaskRuns runs;      // valid runs of the tile (all-valid tiles have one run per row)
    PointIndex idx;
    unsigned long long *total;
};

__global__ __launch_bounds__(64) void k_count_pairs(CountArgs A)
{
    const int lane = threadIdx.x;
    const int64_t i = blockIdx.x;
    const PtRec P = A.idx.pts[i];
    const GridDesc g = A.g;
    unsigned long long cnt = 0;
    if (P.thr > 0.0) {
        const double xll = g.xll, yll = g.yll, cs = g.cs, nrm05 = (double)g.nrows - 0.5;
        const double h = sqrt(P.thr / 9.0);
        int rl, ru, cl, cu;
        narrow_box(g, P.x, P.y, (float)(h * 1.000001) + 1e-6f, rl, ru, cl, cu);
        if (rl <= ru && cl <= cu) {
            const int cn = clampi((int64_t)floor(((double)P.x - xll) / cs), cl, cu);
            for (int r = rl + lane; r <= ru; r += WAVE) {
                const float cy = cell_y(yll, cs, nrm05, r);
                const double dy2 = sqd(cy - P.y);
                if (!(dy2 < P.thr)) continue;
                int lo, hi;
                row_interval(DxCompute<false>{xll, cs, P.x}, xll, 1.0 / cs, cl, cu, cn, P.x, dy2, P.thr, lo, hi);
                if (lo > hi) continue;
                const int64_t rs = A.runs.run_ptr[r], re = A.runs.run_ptr[r + 1];
                for (int64_t k = first_run_ending_at_or_after(A.runs.run_se, rs, re, lo); k < re; ++k) {
                    const int2 rr = A.runs.run_se[k];
                    if (rr.x > hi) break;
                    const int s = rr.x > lo ? rr.x : lo;
                    const int e = rr.y < hi ? rr.y : hi;
                    cnt += (unsigned long long)(e - s + 1);
                }
            }
        }
    }
    for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d, WAVE);
    if (lane == 0) slot_add(A.total, cnt);
}

// reach = sqrt(max bin threshold) (world units), slightly enlarged so that the
// bin range computed from it is a superset.
__global__ __launch_bounds__(256) void k_reach(int nbins, const double *bin_thr, double *reach)
{
    __shared__ double s[4];
    double m = 0.0;
    for (int b = threadIdx.x; b < nbins; b += 256) m = fmax(m, bin_thr[b]);
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, WAVE));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(s[0], s[1]), fmax(s[2], s[3]));
        reach[0] = m > 0.0 ? sqrt(m) * 1.000001 + 1e-6 : 0.0;
    }
}

// g = exp(S / n): the geometric mean of the pilot densities (compGML, tiled:3807-3814).
__global__ void k_gml(const double *S, int64_t n, double *g)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) g[0] = exp(S[0] / (double)n);
}

// ============================================================ reductions ====

// partial[k * nblk + b] = sum over the block's points of log(max(den, 1e-14f))
// (or of log(den) when clamp == 0), in FP64.  Sequential second pass.
__global__ __launch_bounds__(256) void k_sumlog_partial(int64_t n, const float *den, int clamp, double *partial)
{
    __shared__ double s[4];
    const int k = blockIdx.y;
    const float *d = den + (int64_t)k * n;
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float v = d[i];
        if (clamp) v = v < MKDE_EPS_DEN ? MKDE_EPS_DEN : v;
        acc += log((double)v);
    }
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, WAVE);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[(int64_t)k * gridDim.x + blockIdx.x] = ((s[0] + s[1]) + s[2]) + s[3];
}

// One workgroup per candidate: thread t adds partials t, t + 256, ... in
// order, then a fixed-shape tree over the 256 thread sums (deterministic).
__global__ __launch_bounds__(256) void k_sum_final(int nblk, int K, const double *partial, double *out)
{
    __shared__ double s_w[256];
    const int k = blockIdx.x;
    const double *pk = partial + (int64_t)k * nblk;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 256) s += pk[b];
    s_w[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) s_w[threadIdx.x] += s_w[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = s_w[0];
}

// Abramson update h_i = h0 * powf(den0_i / g, alpha) (tiled:571, kde_kernel_kdtr.cu:1007-1037),
// den0 in bin order, h written in original order.
__global__ void k_abramson(int64_t n, const int *perm, const float *den0_sorted, const double *g, float h0,
                           float alpha, float *h_orig)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float ratio = (float)((double)den0_sorted[i] / g[0]);
    h_orig[perm[i]] = h0 * powf(ratio, alpha);
}

// scatter a bin-order array back to original order
__global__ void k_unsort_f32(int64_t n, const int *perm, const float *src, float *dst)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[perm[i]] = src[i];
}

// gather an original-order array into bin order
__global__ void k_sort_f32(int64_t n, const int *perm, const float *src, float *dst)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[perm[i]];
}

// coefk[k*n + i] = w * ew_k / (2 pi h2_k), bin order
// coef_out[i]: one candidate's coefficient of every point (bin order)
__global__ void k_coef_k(int64_t n, const int *perm, const float *w_orig, const float *ew_k_orig, double h2k,
                         float *coef_out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int o = perm[i];
    coef_out[i] = (float)((double)w_orig[o] * (double)ew_k_orig[o] / (h2k * (double)MKDE_TWO_PI_F));
}

// k_coef_k with the bandwidth read from the device: h2k = fl32(h*h).
__global__ void k_coef_k_dev(int64_t n, const int *perm, const float *w_orig, const float *ew_k_orig, const float *h_dev,
                             float *coef_out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float h = *h_dev;
    const double h2k = (double)(float)(h * h);
    const int o = perm[i];
    coef_out[i] = (float)((double)w_orig[o] * (double)ew_k_orig[o] / (h2k * (double)MKDE_TWO_PI_F));
}

__global__ void k_fill_f32(int64_t n, float v, float *dst)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = v;
}

// ====================================================== host launchers ====

extern "C++" {
namespace mkde_dev {

// ------------------------------------------------------------- scratch --
// Device memory of the allocation-free entry point
// (mkde_density_at_points_noalloc): the point kernels' work list, their FP64
// partial sums and the bin-order densities are carved from this file-scope
// array instead of buffers the library allocates.  Every device the library
// runs on holds one copy of it until the process ends; all calls on a device
// share it.  Host code never passes the array's name to a kernel (on the host
// it is a stand-in, not a device address): scratch_address() resolves the
// device address once per device, with that device current, and callers use
// that pointer.
static __device__ __align__(256) unsigned char scratch[MKDE_SCRATCH_BYTES];

hipError_t scratch_address(int device, void **out)
{
    static std::mutex mu;
    static void *addr[MKDE_MAX_DEVICES] = {};
    if (!out || device < 0 || device >= MKDE_MAX_DEVICES) return hipErrorInvalidValue;
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[device]) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != device) return hipErrorInvalidDevice;   // the caller makes the device current
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        addr[device] = p;
    }
    *out = addr[device];
    return hipSuccess;
}

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
static inline unsigned nblk_(int64_t n) { return nblk(n, 256); }

hipError_t prep_points(hipStream_t s, int64_t n, const int *perm, const float *xs, const float *ys,
                       const float *w, const float *h, const float *ew, float h_fixed, PtRec *out)
{
    if (n > 0) hipLaunchKernelGGL(k_prep_points, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, xs, ys, w, h, ew,
                                  h_fixed, out);
    return hipGetLastError();
}

hipError_t prep_fine(hipStream_t s, int64_t n, const int *perm, const float *xs, const float *ys, const float *w,
                     const float *h, const float *ew, float h_fixed, PtRec *out, GroupInfo *grp)
{
    if (n > 0) hipLaunchKernelGGL(k_prep_fine, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, xs, ys, w, h, ew, h_fixed,
                                  (SrcRec *)out, grp);
    return hipGetLastError();
}

hipError_t bin_stats(hipStream_t s, int nbins, const int *bin_start, const PtRec *pts, BinInfo *box, double *thr)
{
    hipLaunchKernelGGL(k_bin_stats, dim3(nblk(nbins, 4)), dim3(256), 0, s, nbins, bin_start, pts, box, thr);
    return hipGetLastError();
}

// Density blocks of a single tile or of a tiled raster (tile-major numbering)
int64_t raster_blocks(const GridDesc &g, const Tiling &tl)
{
    if (tl.tw > 0) {
        const int64_t nty = (g.nrows + tl.th - 1) / tl.th;
        return (int64_t)tl.ntx * nty * tl.bpt;
    }
    return ((g.ncols + MKDE_DT_BW - 1) / MKDE_DT_BW) * ((g.nrows + 63) / 64);
}

static void scan_u32(hipStream_t s, int n, const unsigned *in, unsigned *out, unsigned *chunks, unsigned *total)
{
    const int nchunks = (n + 1023) / 1024;
    hipLaunchKernelGGL(k_scan_local, dim3((unsigned)nchunks), dim3(256), 0, s, n, in, out, chunks);
    hipLaunchKernelGGL(k_scan_chunks, dim3(1), dim3(256), 0, s, nchunks, chunks, total);
    hipLaunchKernelGGL(k_scan_add, dim3(nblk_(n)), dim3(256), 0, s, n, out, chunks);
}

// Scans of n units' costs.
static void work_scan(hipStream_t s, int n, const SplitRule &rule, const WorkList &W, unsigned *host, const double *extra)
{
    const unsigned nchunks = (unsigned)work_chunks(n);
    if (nchunks == 0) {
        hipLaunchKernelGGL(k_work_scan<false>, dim3(1), dim3(1024), 0, s, n, rule, W, host, extra);
        return;
    }
    hipLaunchKernelGGL(k_work_totals, dim3(nchunks), dim3(1024), 0, s, n, W);
    hipLaunchKernelGGL(k_work_counts, dim3(nchunks), dim3(1024), 0, s, n, rule, W);
    hipLaunchKernelGGL(k_work_scan<true>, dim3(nchunks), dim3(1024), 0, s, n, rule, W, host, extra);
}

// Costs and scans of the density work list; W.counts and, when given, the
// pinned host words receive {items, slots, splits, T} and, in the next two, the
// points' reach.
hipError_t density_plan(hipStream_t s, const GridDesc &g, const float *mask, const PointIndex &idx, const Tiling &tl,
                        const WorkList &W, const Tuning &T, unsigned *host)
{
    const int nbx = (int)((g.ncols + MKDE_DT_BW - 1) / MKDE_DT_BW);
    const int nblk = (int)raster_blocks(g, tl);
    hipLaunchKernelGGL(k_block_cost, dim3((unsigned)nblk), dim3(256), 0, s, g, mask, idx, nbx, tl, W.cost);
    const SplitRule rule{DT_TMIN, T.dt_target, 0u, 0ull};
    work_scan(s, nblk, rule, W, host, idx.reach_p);
    return hipGetLastError();
}

// Items, splits and order of n units after their plan; the buffers hold the
// planned counts (or the bounds of point_work_bounds).
hipError_t work_items(hipStream_t s, int n, const WorkList &W, int4 *items, int4 *splits, int *order)
{
    hipLaunchKernelGGL(k_work_items, dim3(nblk_(n)), dim3(256), 0, s, n, W, items, splits, order);
    return hipGetLastError();
}

// order == nullptr: one item per block in raster order; else n_items items.
// nodes, node_on: non-null where wide kernels are summed at nodes (with order);
// items without such sums run in the form without them, which is 10% faster.
hipError_t density_tile(hipStream_t s, const GridDesc &g, const float *mask, float *out, const PointIndex &idx,
                        unsigned long long *stats, const int *order, const int4 *items, const unsigned *cost,
                        double *partials, int n_items, const Tiling &tl, double *nodes, int *node_on)
{
    const int nbx = (int)((g.ncols + MKDE_DT_BW - 1) / MKDE_DT_BW);
    const bool dn = order && nodes;
    TileArgs A{g, mask, out, idx, stats, order, items, cost, partials, nbx, tl, nodes, dn ? node_on : nullptr};
    dim3 grid((unsigned)(order ? n_items : raster_blocks(g, tl)));
    if (dn) {
        hipLaunchKernelGGL(k_density_nodes, grid, dim3(DT_NT), 0, s, A);
        if (stats) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_density_tile<true, true>), grid, dim3(DT_NT), 0, s, A);
        else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_density_tile<false, true>), grid, dim3(DT_NT), 0, s, A);
    }
    if (stats) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_density_tile<true, false>), grid, dim3(DT_NT), 0, s, A);
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_density_tile<false, false>), grid, dim3(DT_NT), 0, s, A);
    return hipGetLastError();
}

hipError_t density_merge(hipStream_t s, const GridDesc &g, const Tiling &tl, const float *mask, int n_split,
                         const int4 *splits, const double *partials, float *out)
{
    if (n_split <= 0) return hipSuccess;
    const int nbx = (int)((g.ncols + MKDE_DT_BW - 1) / MKDE_DT_BW);
    hipLaunchKernelGGL(k_density_merge, dim3((unsigned)n_split), dim3(256), 0, s, g, tl, nbx, mask, splits, partials,
                       out);
    return hipGetLastError();
}

// Split rule of the point work lists.  kind 0: density at points, 1: the
// leave-one-out sums (density at points without the query, or batched); binned:
// in bin order, whose sums depend a little on where a wave is cut and keep to the
// larger parts.
SplitRule point_rule(int kind, const Tuning &T, bool batched, bool binned)
{
    SplitRule r{MKDE_PTS_TMIN, batched ? T.loo_target : T.pts_target, 0u, 0ull};
    if (kind == 1 && !binned) {
        r.few_tmin = MKDE_LOO_FEW_TMIN;
        r.few = MKDE_LOO_FEW;
    }
    return r;
}

// Work list of the point kernels (64-query waves): costs and scans; W.counts
// and, when given, the pinned host words receive {items, slots, splits, T}.
// thr_k non-null: batched leave-one-out with thresholds thr_k[0..K-1]
// ascending, else density at points (h_fixed > 0: one bandwidth), in the
// index's order.
hipError_t point_plan(hipStream_t s, const PointIndex &idx, float h_fixed, const double *thr_k, int K,
                      const SplitRule &rule, const WorkList &W, unsigned *host)
{
    const int nw = (int)((idx.n + 63) / 64);
    const double *lim_dev = thr_k ? thr_k + (K - 1) : nullptr;
    const double lim_fixed = !thr_k && h_fixed > 0.0f ? 9.0 * (double)(float)(h_fixed * h_fixed) : 0.0;
    if (idx.grp) hipLaunchKernelGGL(k_fine_cost, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0, s, idx, W.cost);
    else hipLaunchKernelGGL(k_wave_cost, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0, s, idx, lim_fixed, lim_dev, W.cost);
    work_scan(s, nw, rule, W, host, nullptr);
    return hipGetLastError();
}

// Four waves an item while the list is short (1563 waves: two pilots 720 us with
// one wave an item, 287 us with four; 15625 waves: 3.43 and 3.58 ms).
template <int KIND>
static void launch_sums(hipStream_t s, const SumArgs &A)
{
    const int64_t nw = (A.idx.n + 63) / 64, items = A.order ? A.n_items : nw;
    const int P = nw * A.K <= MKDE_SUM_SHORT ? 4 : 1;
    const dim3 grid((unsigned)((items * P + 3) / 4), (unsigned)A.K);
    if (P == 4) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_point_sums<KIND, 4>), grid, dim3(256), 0, s, A);
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_point_sums<KIND, 1>), grid, dim3(256), 0, s, A);
}

// n_items_dev non-null (here and in loo_multi): the item count is read on the
// device and n_items is only the grid bound.
// fine: the index is in fine order and res is scratch for n floats; else one
// bandwidth h_fixed > 0, the query itself included.
hipError_t point_density(hipStream_t s, const PointIndex &idx, bool fine, int loo, float *den_sorted, float *res,
                         float h_fixed, const int *order, const int4 *items, const unsigned *cost,
                         double *partials, int n_items, const unsigned *n_items_dev)
{
    PtsArgs A{idx, den_sorted, res, order, items, cost, partials, n_items, n_items_dev};
    if (idx.n <= 0) return hipSuccess;
    const int64_t units = order ? n_items : (idx.n + 63) / 64;
    const unsigned grid = (unsigned)((units + 3) / 4);
    if (fine) {
        if (loo) {
            hipLaunchKernelGGL(k_group_density_f<true>, dim3(grid), dim3(256), 0, s, A);
            hipLaunchKernelGGL(k_point_density_f<true>, dim3(grid), dim3(256), 0, s, A);
        } else {
            hipLaunchKernelGGL(k_group_density_f<false>, dim3(grid), dim3(256), 0, s, A);
            hipLaunchKernelGGL(k_point_density_f<false>, dim3(grid), dim3(256), 0, s, A);
        }
    } else {
        if (loo || !(h_fixed > 0.0f)) return hipErrorInvalidValue;
        const double h2 = (double)(float)(h_fixed * h_fixed);
        SumArgs S{};
        S.idx = idx;
        S.K = S.kw = 1;
        S.thr_fixed = 9.0 * h2;
        S.a_fixed = -MKDE_LOG2E / (2.0 * h2);
        S.den1 = den_sorted;
        S.order = order;
        S.items = items;
        S.cost = cost;
        S.partials = partials;
        S.n_items = n_items;
        S.n_items_dev = n_items_dev;
        launch_sums<SUM_PILOT>(s, S);
    }
    return hipGetLastError();
}

hipError_t loo_multi(hipStream_t s, const PointIndex &idx, const float *coefk, const double *a_k,
                     const double *thr_k, int K, float *den1, const int *order, const int4 *items,
                     const unsigned *cost, double *partials, int n_items, const unsigned *n_items_dev)
{
    if (idx.n <= 0) return hipSuccess;
    if (idx.grp) return hipErrorInvalidValue;   // fine order
    const int64_t nw = (idx.n + 63) / 64;
    SumArgs A{idx, coefk, a_k, thr_k, K, 1, 0.0, 0.0, den1, order, items, cost, partials, n_items, n_items_dev};
    // a distance shared by few candidates saves nothing, and a short list is
    // better filled by a wave per candidate
    if (K <= 2 || nw * K <= MKDE_LOO_WAVES) {
        launch_sums<SUM_LOO>(s, A);
        return hipGetLastError();
    }
    int ky = (int)((MKDE_LOO_WAVES + nw - 1) / nw);
    ky = ky < K ? ky : K;
    A.kw = (K + ky - 1) / ky;
    hipLaunchKernelGGL(k_loo_multi, dim3((unsigned)((n_items + 3) / 4), (unsigned)((K + A.kw - 1) / A.kw)), dim3(256),
                       4 * 64 * A.kw * sizeof(float2), s, A);
    return hipGetLastError();
}

// Leave-one-out densities in bin order with the index's bandwidths.
hipError_t loo_density(hipStream_t s, const PointIndex &idx, float *den, const int *order, const int4 *items,
                       const unsigned *cost, double *partials, int n_items, const unsigned *n_items_dev)
{
    if (idx.n <= 0) return hipSuccess;
    if (idx.grp) return hipErrorInvalidValue;   // fine order
    SumArgs A{idx, nullptr, nullptr, nullptr, 1, 1, 0.0, 0.0, den, order, items, cost, partials, n_items, n_items_dev};
    launch_sums<SUM_LOO_EACH>(s, A);
    return hipGetLastError();
}

// n_split_dev non-null: the split count is read on the device and n_split is
// only the grid bound.
hipError_t point_merge(hipStream_t s, int64_t n, int m, int K, int n_split, const int4 *splits, const double *partials,
                       float *den, const unsigned *n_split_dev)
{
    if (n_split > 0)
        hipLaunchKernelGGL(k_point_merge, dim3((unsigned)n_split), dim3(256), 0, s, n, m, K, n_split_dev, splits,
                           partials, den);
    return hipGetLastError();
}

hipError_t range_count(hipStream_t s, const PointIndex &idx, int64_t *counts)
{
    RangeArgs A{idx, counts, nullptr, nullptr};
    if (idx.n > 0) hipLaunchKernelGGL(k_range, dim3(nblk(idx.n, 256)), dim3(256), 0, s, A);
    return hipGetLastError();
}

hipError_t range_fill(hipStream_t s, const PointIndex &idx, const int64_t *offsets, int32_t *out_idx)
{
    RangeArgs A{idx, nullptr, offsets, out_idx};
    if (idx.n > 0) hipLaunchKernelGGL(k_range, dim3(nblk(idx.n, 256)), dim3(256), 0, s, A);
    return hipGetLastError();
}

hipError_t valid_cells(hipStream_t s, int64_t ncells, const float *mask, float nodata, uint8_t *valid)
{
    hipLaunchKernelGGL(k_valid, dim3(nblk(ncells, 256)), dim3(256), 0, s, ncells, mask, nodata, valid);
    return hipGetLastError();
}

// Valid-cell runs of every row of a mask: per-row counts, their exclusive scan
// (first[r]) and run_ptr; the total is left in *total for the caller to size
// the run list before runs_fill.  first, cnt: nrows each; chunks:
// (nrows + 1023) / 1024.
hipError_t runs_count(hipStream_t s, const GridDesc &g, const uint8_t *valid, unsigned *cnt, unsigned *first,
                      unsigned *chunks, unsigned *total, int64_t *ptr)
{
    hipLaunchKernelGGL(k_run_count, dim3(nblk(g.nrows, 4)), dim3(256), 0, s, g.ncols, g.nrows, valid, cnt);
    scan_u32(s, (int)g.nrows, cnt, first, chunks, total);
    hipLaunchKernelGGL(k_run_ptr, dim3(nblk_(g.nrows + 1)), dim3(256), 0, s, g.nrows, first, total, ptr);
    return hipGetLastError();
}

hipError_t runs_fill(hipStream_t s, const GridDesc &g, const uint8_t *valid, const unsigned *first, int2 *se,
                     int2 *row_run)
{
    hipLaunchKernelGGL(k_run_fill, dim3(nblk(g.nrows, 4)), dim3(256), 0, s, g.ncols, g.nrows, valid, first, se,
                       row_run);
    return hipGetLastError();
}

hipError_t boundary(hipStream_t s, const GridDesc &g, const uint8_t *valid, uint8_t *flags, float2 *blist,
                    unsigned long long *bcount)
{
    if (g.ncols <= 0 || g.nrows <= 0) return hipSuccess;
    const unsigned gy = (unsigned)std::min<int64_t>(g.nrows, 65535);
    hipLaunchKernelGGL(k_boundary, dim3(nblk(g.ncols, 256), gy), dim3(256), 0, s, g, valid, flags, blist, bcount);
    return hipGetLastError();
}

// Entries of a level's box array (and, for level 0, of the bits): four per node
// of the level above.
int64_t bt_level_size(const BndTree &T, int l) { return 4 * (int64_t)T.nx[l + 1] * T.ny[l + 1]; }

// Boundary flags, their count (counter slots) and the hierarchy's leaves.
hipError_t boundary_leaf(hipStream_t s, const GridDesc &g, const uint8_t *valid, uint8_t *flags, const BndTree &T,
                         uint4 *bits, float4 *box, unsigned long long *bcount)
{
    const int wnx = (2 * T.nx[1] + 3) / 4;
    const int64_t nw = (int64_t)wnx * (2 * T.ny[1]);
    hipLaunchKernelGGL(k_boundary_leaf, dim3(nblk(nw, 4)), dim3(256), 0, s, g, valid, flags, T.nx[0], T.ny[0], T.nx[1],
                       wnx, nw, bits, box, bcount);
    return hipGetLastError();
}

hipError_t bt_build(hipStream_t s, const BndTree &T, float4 *box)
{
    for (int l = 0; l + 1 < T.nlev; l += 4)
        hipLaunchKernelGGL(k_bt_up, dim3(nblk(2 * T.nx[l + 2], 16), nblk(2 * T.ny[l + 2], 16)), dim3(256), 0, s, T, l,
                           box);
    return hipGetLastError();
}

hipError_t dist_tree(hipStream_t s, int64_t n, const float *xs, const float *ys, const int *perm, const GridDesc &g,
                     const BndTree &T, double *dist)
{
    if (n > 0) hipLaunchKernelGGL(k_dist_tree, dim3(nblk(n, 64)), dim3(64), 0, s, n, xs, ys, perm, g, T, dist);
    return hipGetLastError();
}

hipError_t dist_boundary(hipStream_t s, int64_t n, const float *x, const float *y, const float2 *blist, int64_t nb,
                         double *dist)
{
    if (n > 0) hipLaunchKernelGGL(k_dist_boundary, dim3(nblk(n, 256)), dim3(256), 0, s, n, x, y, blist, nb, dist);
    return hipGetLastError();
}

// A cell size is a power of two when its mantissa is: x / cs and x * (1 / cs) are
// then the same double (away from the subnormals, where none of the sizes lie).
static void ec_cell_size(EcArgs &A)
{
    int e = 0;
    A.inv_cs = 1.0 / (double)A.g.cs;
    A.cs_exact = frexp((double)A.g.cs, &e) == 0.5 ? 1 : 0;
}

// h_dev non-null: every point's bandwidth is the device value *h_dev.
hipError_t ec_active(hipStream_t s, int64_t n, const GridDesc &g, const float *x, const float *y, const double *dist,
                     const float *h, float h_fixed, const float *h_dev, float *ew, int *list, int *count,
                     int cw_narrow, int cw_wide)
{
    EcArgs A{};
    A.g = g;
    ec_cell_size(A);
    if (n > 0)
        hipLaunchKernelGGL(k_ec_active, dim3(nblk(n, EC_ACT_T * EC_ACT_K)), dim3(EC_ACT_T), 0, s, n, g, A.inv_cs,
                           A.cs_exact, x, y, dist, h, h_fixed, h_dev, ew, list, count, cw_narrow, cw_wide);
    return hipGetLastError();
}

hipError_t centres(hipStream_t s, const GridDesc &g, float *colx, float *rowy)
{
    const int64_t m = g.ncols > g.nrows ? g.ncols : g.nrows;
    hipLaunchKernelGGL(k_centres, dim3(nblk(m, 256)), dim3(256), 0, s, g, colx, rowy);
    return hipGetLastError();
}

// Widest box k_ec_wide takes, and its LDS: an FP64 prefix sum per column, at
// most 64,008 B.
int ec_wide_max() { return 8000; }
static size_t ec_wide_lds(int w) { return (size_t)(w + 1) * sizeof(double); }
static void launch_ec_wide(hipStream_t s, unsigned grid, int w, const EcArgs &A, int64_t n)
{
    if (A.cx32) hipLaunchKernelGGL(k_ec_wide<true>, dim3(grid), dim3(256), ec_wide_lds(w), s, A, n);
    else hipLaunchKernelGGL(k_ec_wide<false>, dim3(grid), dim3(256), ec_wide_lds(w), s, A, n);
}

template <int CW>
static void launch_ec_cw(hipStream_t s, unsigned grid, const EcArgs &A)
{
    if (A.cx32) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ec<CW, true>), dim3(grid), dim3(64), 0, s, A);
    else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ec<CW, false>), dim3(grid), dim3(64), 0, s, A);
}
static void launch_ec(hipStream_t s, unsigned grid, int cw, const EcArgs &A)
{
    if (cw == 512) launch_ec_cw<512>(s, grid, A);
    else if (cw == 1024) launch_ec_cw<1024>(s, grid, A);
    else launch_ec_cw<2048>(s, grid, A);
}

// Most columns of the NARROW box of a point at the fixed bandwidth h on grid
// g, for every point within 3h of a valid cell (narrow_box: the box spans
// 6h / cs columns between two truncations, so at most floor(6h / cs) + 2;
// one more for the rounding of the double expressions).  A point whose box is
// wider (only one lying more than 3h left of the raster, whose box the size_t
// arithmetic stretches to the whole row) goes to the chunked k_ec.
int ec_box_cols(const GridDesc &g, float h)
{
    const double w = std::floor(6.0 * (double)h / g.cs + 1e-6) + 3.0;
    return (int)std::min<double>((double)g.ncols, std::max(w, 1.0));
}

static long long env_ll(const char *name, long long dflt)
{
    const char *e = getenv(name);
    const long long v = e ? atoll(e) : 0;
    return v > 0 ? v : dflt;
}

// Default launch shapes (measured on one MI355X), each overridable from the
// environment:
//   ec_chunk 1024 (MKDE_EC_CHUNK; 512 / 1024 / 2048: the adaptive job's EC
//     within 1%, the 64-candidate search 314 / 296 / 307 ms);
//   ec_wide_min = ec_chunk (MKDE_EC_WIDE_MIN): every box k_ec would cut into
//     two or more chunks runs in k_ec_wide;
//   loo_target 32768 (MKDE_LOO_TARGET; 2048 / 8192 / 32768 / 65536 / 131072:
//     search 237 / 200 / 187 / 191 / 194 ms);
//   pts_target 16384 (MKDE_PTS_TARGET; 4096 / 16384 / 65536: bandwidth phase
//     of the adaptive 1M job 8.2 / 7.5 / 8.0 ms);
//   dt_target 4096 (MKDE_DENSITY_TARGET; adaptive 1M job / 10M-point tiles,
//     density ms: 1024: 30.9 / 32.7, 2048: 30.9 / 27.5, 4096: 31.0 / 27.8,
//     16384: 31.7 / 27.9, 65536: 33.3 / 29.2).
Tuning default_tuning()
{
    Tuning t;
    const long long cw = env_ll("MKDE_EC_CHUNK", 1024);
    t.ec_chunk = (cw == 512 || cw == 2048) ? (int)cw : 1024;
    t.ec_wide_min = (int)env_ll("MKDE_EC_WIDE_MIN", t.ec_chunk);
    t.loo_target = (unsigned long long)env_ll("MKDE_LOO_TARGET", 32768);
    t.pts_target = (unsigned long long)env_ll("MKDE_PTS_TARGET", 16384);
    t.dt_target = (unsigned long long)env_ll("MKDE_DENSITY_TARGET", (long long)DT_TARGET);
    return t;
}

// The n_narrow points at the front of list run in k_ec (one wave each, column
// chunks), the n_wide points at the back in k_ec_wide (one workgroup each,
// max_w columns of LDS).
hipError_t ec(hipStream_t s, int64_t n, int n_narrow, int n_wide, int max_w, const GridDesc &g, const MaskRuns &runs,
              const float *colx, const float *rowy, const float *x, const float *y, const float *h, float h_fixed,
              const int *list, float *ew, unsigned long long *n_eval, int cw, int cx32)
{
    EcArgs A{g, runs, colx, rowy, x, y, h, h_fixed, nullptr, nullptr, list, ew, n_eval, cx32, 0.0, 0};
    ec_cell_size(A);
    if (n_narrow > 0) launch_ec(s, (unsigned)n_narrow, cw, A);
    if (n_wide > 0) {
        if (max_w < 1 || max_w > ec_wide_max()) return hipErrorInvalidValue;
        launch_ec_wide(s, (unsigned)n_wide, max_w, A, n);
    }
    return hipGetLastError();
}

// The same EC pass with every size on the device (no host read-back, so the
// launches can be captured in a graph): the bandwidth is *h_dev, the list
// lengths count[0] (narrow) and count[1] (wide) as k_ec_active left them.
// Fixed grids loop over the list.  w_wide is the cw_wide k_ec_active was given
// (the widest wide box): the wide kernel takes that much LDS, as many
// workgroups as fit on 256 CUs, and is left out when no box can be wide
// (w_wide <= cw_narrow).
hipError_t ec_dev(hipStream_t s, int64_t n, const GridDesc &g, const MaskRuns &runs, const float *colx,
                  const float *rowy, const float *x, const float *y, const float *h_dev, const int *count,
                  const int *list, float *ew, int cw, int cw_narrow, int w_wide, int cx32)
{
    if (n <= 0) return hipSuccess;
    if (w_wide > ec_wide_max()) return hipErrorInvalidValue;
    EcArgs A{g, runs, colx, rowy, x, y, nullptr, 0.0f, h_dev, count, list, ew, nullptr, cx32, 0.0, 0};
    ec_cell_size(A);
    const unsigned gn = (unsigned)std::min<int64_t>(n, 256 * 32);   // 8 waves per SIMD
    launch_ec(s, gn, cw, A);
    if (w_wide > cw_narrow) {
        const size_t lds = ec_wide_lds(w_wide);
        const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(8, (160u << 10) / (lds + 256)));
        const unsigned gw = (unsigned)std::min<int64_t>(n, 256 * per_cu);
        launch_ec_wide(s, gw, w_wide, A, n);
    }
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fold_slots(unsigned long long *slots)
{
    __shared__ unsigned long long s_w[4];
    unsigned long long v = 0;
    for (int k = threadIdx.x; k < MKDE_CNT_SLOTS; k += 256) v += slots[k * MKDE_CNT_STRIDE];
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, WAVE);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) slots[MKDE_CNT_SLOTS * MKDE_CNT_STRIDE] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Words of a slot counter (slots, then the folded total).
int64_t slot_words() { return (int64_t)MKDE_CNT_SLOTS * MKDE_CNT_STRIDE + 1; }

// slots[slot_words() - 1] = sum of the slots.
hipError_t fold_slots(hipStream_t s, unsigned long long *slots)
{
    hipLaunchKernelGGL(k_fold_slots, dim3(1), dim3(256), 0, s, slots);
    return hipGetLastError();
}

hipError_t count_pairs(hipStream_t s, const GridDesc &g, const MaskRuns &runs, const PointIndex &idx,
                       unsigned long long *total)
{
    CountArgs A{g, runs, idx, total};
    if (idx.n > 0) hipLaunchKernelGGL(k_count_pairs, dim3((unsigned)idx.n), dim3(64), 0, s, A);
    return hipGetLastError();
}

hipError_t reach(hipStream_t s, int nbins, const double *bin_thr, double *reach_out)
{
    hipLaunchKernelGGL(k_reach, dim3(1), dim3(256), 0, s, nbins, bin_thr, reach_out);
    return hipGetLastError();
}

hipError_t gml(hipStream_t s, const double *S, int64_t n, double *g)
{
    hipLaunchKernelGGL(k_gml, dim3(1), dim3(64), 0, s, S, n, g);
    return hipGetLastError();
}

hipError_t sumlog(hipStream_t s, int64_t n, int K, const float *den, int clamp, double *partial, int nb, double *out)
{
    hipLaunchKernelGGL(k_sumlog_partial, dim3((unsigned)nb, (unsigned)K), dim3(256), 0, s, n, den, clamp, partial);
    hipLaunchKernelGGL(k_sum_final, dim3((unsigned)K), dim3(256), 0, s, nb, K, partial, out);
    return hipGetLastError();
}

hipError_t abramson(hipStream_t s, int64_t n, const int *perm, const float *den0_sorted, const double *g, float h0,
                    float alpha, float *h_orig)
{
    if (n > 0) hipLaunchKernelGGL(k_abramson, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, den0_sorted, g, h0,
                                  alpha, h_orig);
    return hipGetLastError();
}

hipError_t unsort_f32(hipStream_t s, int64_t n, const int *perm, const float *src, float *dst)
{
    if (n > 0) hipLaunchKernelGGL(k_unsort_f32, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, src, dst);
    return hipGetLastError();
}

hipError_t sort_f32(hipStream_t s, int64_t n, const int *perm, const float *src, float *dst)
{
    if (n > 0) hipLaunchKernelGGL(k_sort_f32, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, src, dst);
    return hipGetLastError();
}

hipError_t coef_k(hipStream_t s, int64_t n, const int *perm, const float *w, const float *ew_k, double h2k,
                  float *coef_out)
{
    if (n > 0)
        hipLaunchKernelGGL(k_coef_k, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, w, ew_k, h2k, coef_out);
    return hipGetLastError();
}

hipError_t coef_k_dev(hipStream_t s, int64_t n, const int *perm, const float *w, const float *ew_k, const float *h_dev,
                      float *coef_out)
{
    if (n > 0)
        hipLaunchKernelGGL(k_coef_k_dev, dim3(nblk(n, 256)), dim3(256), 0, s, n, perm, w, ew_k, h_dev, coef_out);
    return hipGetLastError();
}

hipError_t fill_f32(hipStream_t s, int64_t n, float v, float *dst)
{
    if (n > 0) hipLaunchKernelGGL(k_fill_f32, dim3(nblk(n, 256)), dim3(256), 0, s, n, v, dst);
    return hipGetLastError();
}

}  // namespace mkde_dev
}
