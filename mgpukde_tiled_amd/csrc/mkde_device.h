// mkde_device.h -- types shared by the HIP kernels (mkde_kernels.hip) and the
// host library (mkde_capi.cpp, mkde_serve.cpp).  Plain structs only: no torch, no STL.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// Utilities.h:8 -- the reference's TWO_PI is a float literal.
#define MKDE_TWO_PI_F 6.2831853071795862f
#define MKDE_LOG2E 1.4426950408889634073599
// Utilities.h:19 -- EPSILONDENSITY (a float literal).
#define MKDE_EPS_DEN 0.00000000000001f
// candidate bandwidths per batched leave-one-out pass
#define MKDE_LM_K 16
// static device scratch of the allocation-free entry point (bytes per device)
// and the device ordinals it is resolved for
#define MKDE_SCRATCH_BYTES (32u << 20)
#define MKDE_MAX_DEVICES 64

// Launch-shape settings of one context: defaults from the environment
// (default_tuning), changed by mkde_set_option or the autotuner.  They set how
// work is cut into pieces, so a change can move FP32 rounding (never the
// cut-off sets or the error bound).
struct Tuning {
    int ec_chunk;                    // 512, 1024 or 2048: columns per prefix chunk of k_ec
    int ec_wide_min;                 // boxes wider than this run in k_ec_wide
    unsigned long long loo_target;   // split target of the batched leave-one-out work list
    unsigned long long pts_target;   // split target of the point-density work list
    unsigned long long dt_target;    // split target of the density-raster work list
};

// A work list cuts units (64-query waves, density blocks) whose cost exceeds a
// threshold T into ceil(cost / T) parts.  T = max(ceil(total / target),
// min(tmin, max(few_tmin, ceil(total / few)))): about `target` parts when there
// is much work, none below tmin sources a part, but with little work in all
// (few > 0) up to `few` smaller parts, down to few_tmin sources each, so that a
// short list still fills the device.
struct SplitRule {
    unsigned tmin;
    unsigned long long target;
    unsigned few_tmin;
    unsigned long long few;   // 0: no smaller parts
};

// Smallest split threshold of the point work lists (candidate sources per part).
#define MKDE_PTS_TMIN 4096u
// Leave-one-out lists in fine order: smaller parts while they are at most 4096.
#define MKDE_LOO_FEW_TMIN 256u
#define MKDE_LOO_FEW 4096ull
// The batched pass gives each wave fewer candidates until it has this many waves.
#define MKDE_LOO_WAVES 4096
// Lists of at most so many waves (times candidates) run with 16 queries a wave.
#define MKDE_SUM_SHORT 8192

// Most items and split parts a point work list of nw 64-query waves can have:
// each wave's cost is at most n sources, so split parts <= min(target, total /
// T) + the number of split waves.
inline void point_work_bounds(int64_t n, const SplitRule &r, int64_t *items_max, int64_t *slots_max)
{
    const int64_t nw = (n + 63) / 64;
    const double tot = (double)nw * (double)n;
    const int64_t by_t = (int64_t)((tot + r.tmin - 1) / (double)r.tmin);
    int64_t parts = by_t < (int64_t)r.target ? by_t : (int64_t)r.target;
    int64_t split_waves = by_t < nw ? by_t : nw;
    if (r.few > 0) {
        const int64_t by_f = (int64_t)((tot + r.few_tmin - 1) / (double)r.few_tmin);
        const int64_t few = by_f < (int64_t)r.few ? by_f : (int64_t)r.few;
        parts = parts > few ? parts : few;
        const int64_t fw = few < nw ? few : nw;
        split_waves = split_waves > fw ? split_waves : fw;
    }
    *items_max = nw + parts + 1;
    *slots_max = parts + split_waves + 1;
}

// Raster geometry (AsciiRaster.h:9-33 geometry fields).
struct GridDesc {
    int64_t ncols, nrows;
    float xll, yll, cs, nodata;
};

// Uniform world-space bin grid over the points' bounding box.  Bin (bx, by)
// covers [x0 + bx*size, x0 + (bx+1)*size) x [y0 + by*size, ...).
struct BinGrid {
    double x0, y0, size;
    int nbx, nby;
};

// One sample point in bin order, with the per-job derived constants of the
// Gaussian kernel: coef = w*ew / (2*pi*h2f), a = -log2(e) / (2*h2f),
// thr = 9*h2f, where h2f = (double)fl32(h*h).  A point with h <= 0 has
// thr = -1 (it can never be inside the cut-off) and coef = 0.
struct __attribute__((aligned(32))) PtRec {
    float x, y, coef, pad;
    double a, thr;
};

// One source of the point densities in fine order (PtRec's places for x, y,
// coef and thr): af = (float)a, and lo / hi bracket thr so that a float squared
// distance below lo is inside the cut-off and one above hi is not.
struct __attribute__((aligned(32))) SrcRec {
    float x, y, coef, af, lo, hi;
    double thr;
};

// 64 consecutive points in fine order: their bounding box and the smallest and
// largest cut-off threshold.
struct GroupInfo {
    float x0, y0, x1, y1;
    double tmin, tmax;
};

// Per-bin summary used for culling: bounding box of the bin's points and the
// largest cut-off threshold 9*h2f among them.
struct BinInfo {
    float x0, y0, x1, y1;
};

// Two orders share the bins.  In bin order a bin's points keep the caller's
// order; in fine order they follow a Hilbert curve through the bin, so that 64
// consecutive points are close together.  The pilot densities, whose rounding
// every adaptive bandwidth inherits, are summed in bin order.
struct PointIndex {
    const PtRec *pts;       // n, bin order; fine order: SrcRec
    const GroupInfo *grp;   // fine order: (n + 63) / 64
    const int *bin_start;   // nbins + 1
    const BinInfo *bin_box; // nbins
    const double *bin_thr;  // nbins
    BinGrid bg;
    const double *reach_p;  // device scalar: max over bins of sqrt(bin_thr), world units
    int64_t n;
};

// Density blocks: 64 rows x MKDE_DT_BW columns (64 or 128), one workgroup
// each, one 32 x 32 quadrant per wave (MKDE_DT_BW / 16 waves).
#define MKDE_DT_BW 64
#define MKDE_DT_CELLS (64 * MKDE_DT_BW)
// Sums of an item at the nodes of its block, for rasters whose split threshold
// (candidates of an item) is at least this.
#define MKDE_DN_CELLS 256
#define MKDE_DN_SPLIT 4096
// Cells that some point's cut-off radius must reach: 3 * 31.5 / (2 * 0.65).
#define MKDE_DN_REACH 72.7

// A raster processed as tiles of tw x th cells, each tile with its own origin
// from the raster geotransform (GDAL order gt0, gt1, gt3, gt5).  Density
// blocks are numbered tile-major: bpx blocks per tile row, bpt per tile, ntx
// tiles per raster row (edge tiles leave some blocks empty).
// tw == 0 means one tile described by its GridDesc.
struct Tiling {
    int64_t tw, th;
    int ntx, bpx, bpt;
    double gt0, gt1, gt3, gt5;
};

// Lists of more units than MKDE_WS_ONE are scanned by several workgroups, in chunks
// of MKDE_WS_UNITS: a chunk's cost, {items, slots, split units} and items of each
// cost bucket.
#define MKDE_WS_ONE 16384
#define MKDE_WS_UNITS 4096
struct WorkChunk {
    unsigned long long cost;
    unsigned n[3];
    unsigned hist[32];
};
inline int64_t work_chunks(int64_t units)
{
    return units > MKDE_WS_ONE ? (units + MKDE_WS_UNITS - 1) / MKDE_WS_UNITS : 0;
}

// Device buffers of a work list (per unit unless noted): costs, the exclusive
// scan of the parts, and for split units the first partial slot and the place
// in the split list; the counts {items, slots, splits, T} and the places of the
// 32 cost buckets in the visiting order.
struct WorkList {
    unsigned *cost, *item0, *slot0, *sidx;
    unsigned *counts;              // 4
    unsigned *hist;                // 32
    WorkChunk *chunks;             // work_chunks(units); unused when that is 0
};

// Boundary-cell hierarchy for exact nearest-boundary distances: leaves of
// 16 x 16 cells hold a 256-bit mask of their boundary cells; every level keeps
// the bounding box {x0, y0, x1, y1} of the boundary cell centres below a node
// (x0 > x1: empty); level l has nx[l] x ny[l] nodes starting at off[l], the four
// children of a node next to each other (bt_node), missing ones empty, so that
// a node's expansion reads one 64-byte line.
#define MKDE_BT_S 16
#define MKDE_BT_MAXL 15
struct BndTree {
    const uint4 *bits;     // 2 per leaf (256 bits, row-major within the leaf)
    const float4 *box;     // all levels
    int nlev;
    int nx[MKDE_BT_MAXL + 1], ny[MKDE_BT_MAXL + 1];   // one level above the root: 1 x 1
    int64_t off[MKDE_BT_MAXL];
};

// Place of node (ix, iy) in its level, pnx = nx of the level above.
__host__ __device__ inline int64_t bt_node(int ix, int iy, int pnx)
{
    return (((int64_t)(iy >> 1) * pnx + (ix >> 1)) << 2) | ((iy & 1) << 1) | (ix & 1);
}

// Per-row runs of valid cells of a mask (CSR): runs of row r are
// run_se[run_ptr[r] .. run_ptr[r+1]), each (start, end) inclusive, ascending.
// row_run[r] is the run of a row with one, (1, 0) for a row without, and
// (-1, 0) for a row with more.
struct MaskRuns {
    const int64_t *run_ptr;
    const int2 *run_se;
    const int2 *row_run;
};
