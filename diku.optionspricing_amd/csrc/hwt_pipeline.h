// hwt_pipeline.h -- what the host side of the pricer and the pricing-kernel
// translation units share: the device views of the batch, the task classes
// and bucket layout, the counter slots, and the pricing kernels' signatures.
// The kernels are defined in hwt_pricers.h and instantiated one per
// translation unit (hwt_k_*.hip), so the library's slowest code compiles in
// parallel.
#pragma once

#include "../../include/hwtree.h"
#include "hwt_flat.h"
#include "hwt_rows.h"
#include "hwt_wave.h"

namespace hwt {

struct DevOpts {
    int32_t n;  // options, or the capacity bound when `count` is set
    const double *strike, *maturity, *length;
    const uint16_t *term_unit, *term_steps;
    const double *a, *sigma;
    const int8_t *type;
    const int32_t *count;  // device-side option count (<= n), or null
    // per-option tree constants given by the caller instead of the fields
    // above (which are then null), or null
    const hwt_option_constants_f64 *consts;
    // with consts: the constants are a float caller's, widened; the exercise
    // step is then (int)(t / dt) in float arithmetic
    int32_t consts_f32;
};

struct DevYield {
    int32_t n;
    const double *rate;
    const int32_t *day;
};

// Task classes of mixed mode and form 1, in task-list order:
//   wide  (w > 64*KSMALL)           k_price_wide, one option per wave, LPT queue
//   mid   (ROW_MAX_WIDTH < w <= 64*KSMALL)  k_price_narrow, one option per wave
//   row   (w <= ROW_MAX_WIDTH)      k_price_narrow, four options per wave
//   flat  (w <= FLAT_MAX_WIDTH)     k_price_narrow, 64 / w options per wave, one
//                                   node per lane (hwt_flat.h)
// Bucket ranges: wide [B_WIDE, NBUCKET) and mid [B_MID, B_WIDE), log-spaced
// by the sort key (work unless a width/height order is asked for); row
// [B_ROW, B_MID), by (nodes per lane, height) so the four rows of a wave share
// their step count; flat [0, B_ROW), by (width, height).  The scan walks each
// class from its largest key down.
constexpr int NBUCKET = 2048;
constexpr int B_ROW = 640, B_MID = 1280, B_WIDE = 1536;
constexpr int ROW_HBUCKETS = 160;   // height buckets per row part (nodes per lane 1..4)
constexpr int FLAT_HBUCKETS = 64;   // height buckets per flat part (one width each)
constexpr int MAX_PADS = 640;       // idle task slots padding the parts of one task list, at most
constexpr int KSMALL = 2;  // trees up to 64*KSMALL nodes wide go to the narrow-tree kernel
#ifndef WIDE_WINDOW_STEP
#define WIDE_WINDOW_STEP 4  // nodes per lane a wide tree's light-cone window grows or shrinks by
#endif
#ifndef REACH_WINDOW_STEP
#define REACH_WINDOW_STEP 1  // ... and its FP64 window along the reach
#endif

// FP64 (hwt_tri.h) has its own classes, in task-list order:
//   big     trees the tridiagonal form cannot hold (tri_ok, more than
//           TRI_MAX_NODES nodes of weight): k_price_wide, LPT queue
//   window  one tree per wave, LPT queue
//   parts   64 / L trees per wave, L lanes of K nodes each: one part per (L, K),
//           L the least power of two that holds the tree at K <= 11.  Of two
//           splits that hold a tree the one with fewer lanes spends fewer
//           instructions per tree (27 of a wave for 32 trees at L = 2, K = 11,
//           against 8 for 4 at L = 16, K = 2), but a batch too small to fill the
//           chip waits for its longest wave: up to TRI_SPREAD options trees up to 64
//           nodes take 16 lanes each, wider ones a wave.  (K <= 13 or 15 saves 3%
//           of the instructions and loses more: spills, fewer and longer groups.)
// Buckets: parts [0, B_TRI_WIN) by (part, height), window and big above by the
// sort key.  The scan takes them from the highest down, so the groups of few
// lanes, which hold the most trees and take longest, come first.
constexpr int TRI_EDGE = 10;     // doubles per edge record (TriEdge)
constexpr int TRI_MAXK = 11;     // nodes per lane
constexpr int TRI_MAX_NODES = WAVE * TRI_MAXK;
constexpr int TRI_SPREAD = 16384;
constexpr int TRI_GROUP_WIDTH = 16 * TRI_MAXK, TRI_SPREAD_WIDTH = 64;
// parts: L = 16 with K = 2, 3, 4 (spread); L = 16, 8, 4 with K = 6 .. 11 each; L = 2
// with K = 7 .. 11; L = 1 with K = 3, 5 .. 11
constexpr int TRI_PARTS = 31;
constexpr HWT_HD int tri_lanes(int part) { return part < 9 ? 16 : part < 15 ? 8 : part < 21 ? 4 : part < 26 ? 2 : 1; }
constexpr HWT_HD int tri_nodes(int part)  // K
{
    return part < 3 ? 2 + part : part < 21 ? 6 + (part - 3) % 6 : part < 26 ? part - 14 : 2 * part - 49;
}
constexpr HWT_HD int tri_part(int w, bool spread)  // w up to TRI_GROUP_WIDTH, odd
{
    return spread ? (w <= 32 ? 0 : (w + 15) / 16 - 2)
           : w <= 11 ? 26 + (w - 3) / 2
           : w <= 22 ? 14 + (w + 1) / 2
           : w <= 44 ? 9 + (w + 3) / 4
           : w <= 88 ? 3 + (w + 7) / 8
                     : (w + 15) / 16 - 3;
}
constexpr int SMALL_MAX = 2048;  // options of a batch that k_price_small takes, a wave each
constexpr int SMALL_YMAX = 512;  // ... and points of its curve
// Wave b takes tasks b % TRI_QUEUES + i * TRI_QUEUES, claimed from its own queue
// head.  With one head for all, 4,096 waves' claims of 1,000 to 10,000 tasks
// serialise at 9 ns each (60k skewed batch 486 us).
constexpr int TRI_QUEUES = 32;
constexpr int TRI_HBUCKETS = 72;  // heights below 24, then 8 per octave
constexpr int B_TRI_WIN = TRI_PARTS * TRI_HBUCKETS, B_TRI_BIG = B_TRI_WIN + 256, NBUCKET_TRI = 2560;
constexpr int NBUCKET_MAX = NBUCKET > NBUCKET_TRI ? NBUCKET : NBUCKET_TRI;

// k_setup's class switches
constexpr int CLASS_ROWS = 1, CLASS_FLAT = 2;
enum Tally {
    T_QUEUE = 0,    // next task of the wide-tree kernel (tasks [0, T_NLARGE))
    T_QUEUE_S = 1,  // next mid-class task (fused kernel; the narrow-tree kernel strides statically)
    T_NTASK = 2,
    T_NLARGE = 3,
    T_INVALID = 4,
    T_UNSUP = 5,
    T_WORK = 6,     // int64
    T_SEQWORK = 8,  // int64
    T_WORKW = 10,   // int64, wide trees only
    T_NMID = 12,    // end of the mid-class tasks
    T_NPAD = 13,    // idle slots padding the row class
    T_NCOUNT = 14,  // end of the execution counts (slots 16-23 are k_setup's accumulators)
    T_QUEUE_R = 15, // next chunk of row groups (fused kernel)
    // accumulated by k_setup's blocks, then moved into the slots above and
    // cleared by k_order's writer block
    A_WORK = 16,    // int64
    A_SEQWORK = 18, // int64
    A_WORKW = 20,   // int64
    A_INVALID = 22,
    A_UNSUP = 23,
    T_NREDO = 24,   // mixed mode: options handed to the FP64 re-pricing (host-visible)
    T_QUEUE_X = 25, // next task of the FP64 re-pricing kernel
    T_NROW = 26,    // end of the row-class tasks (start of the flat class)
    T_QUEUE_F = 27, // next chunk of flat groups (fused kernel)
    T_NFLATG = 28,  // flat groups in all
    // first task and first group of each flat part (one width each, widest
    // first, as the scan lays them out), then the end of the last part
    T_FLAT_START = 32,  // FLAT_PARTS + 1 entries
    // int64, device wall clock (constant rate) of the last execution at
    // k_setup's start (its first block)
    T_T0 = 44,
    T_FLAT_GROUP = 48,  // FLAT_PARTS + 1 entries
    // int64: what the windowed kernels' stencil steps executed (StepCount):
    // operations, unit-form node slots, plain-form node slots
    T_XFLOP = 64,
    T_XUNIT = 66,
    T_XPLAIN = 68,
    // int64 x N_END: the latest end of a pricing wavefront, wavefront w in
    // slot w % N_END (one address for all of them serialised 4,096 atomics
    // into 37 us); cleared by k_order's writer block, the maximum taken at sync
    T_END = 72,
    T_HOST = T_END + 2 * 256,  // [0, T_HOST) is copied to the host by hwt_plan_sync
    // FP64: ends of the big and the window tasks, groups in all, first task and
    // first group of each part (in scan order, highest part first)
    T_TBIG = T_HOST,
    T_TWIN = T_HOST + 1,
    T_TNGROUP = T_HOST + 2,
    T_SMALL = T_HOST + 3,   // options of the last execution if k_price_small ran it and no sync has counted it, else 0
    T_TSTART = T_HOST + 8,  // TRI_PARTS entries
    T_TGROUP = T_HOST + 56, // TRI_PARTS entries
    A_NWIDE = T_HOST + 104,  // accumulated by k_setup: wide trees
    // the bucket histogram (k_setup's atomics), cleared by the first pricing
    // kernel of each execution
    T_HIST = T_HOST + 128,
    // FP64: queue heads of the window tasks and of the groups (the big tasks use
    // T_QUEUE), TRI_QUEUES of each, a 128-byte line apart
    T_TQWIN = (T_HIST + NBUCKET_MAX + 31) / 32 * 32,
    T_TQGROUP = T_TQWIN + 32 * TRI_QUEUES,
    T_ALLOC = T_TQGROUP + 32 * TRI_QUEUES
};
constexpr int N_END = (T_HOST - T_END) / 2;

// The bucket histogram (in the tally) back to zero for the next execution:
// its last readers, k_order's blocks, are done once a pricing kernel runs (mixed
// mode's first one, FP64's k_price_tri).
__device__ __forceinline__ void clear_bucket_counts(int32_t *tally)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < NBUCKET_MAX; i += gridDim.x * blockDim.x)
        tally[T_HIST + i] = 0;
}

// The execution's latest pricing-wavefront end so far, for
// hwt_stats.total_ms: one 64-bit atomic per wavefront, as it exits, into the
// wavefront's end slot.
__device__ __forceinline__ void stamp_wave_end(int32_t *tally)
{
    const int w = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (threadIdx.x % WAVE == 0)
        atomicMax(reinterpret_cast<unsigned long long *>(tally + T_END) + w % N_END,
                  (unsigned long long)__builtin_amdgcn_s_memrealtime());
}

// Pricing kernels (hwt_pricers.h).  All are persistent: one single-wave
// workgroup per resident slot, tasks from the ordered task list.
template <class T>
__global__ void k_price_wide(const OptConst *__restrict__ cst, const double *__restrict__ edge,
                             const int32_t *__restrict__ order, int32_t *__restrict__ tally,
                             double *__restrict__ out, double *__restrict__ scratch, int32_t *__restrict__ redo);
template <class T>
__global__ void k_price_narrow(const OptConst *__restrict__ cst, const double *__restrict__ edge,
                               const int32_t *__restrict__ order, int32_t *__restrict__ tally,
                               double *__restrict__ out, int32_t *__restrict__ redo);
template <class T>
__global__ void k_price_fused(const OptConst *__restrict__ cst, const double *__restrict__ edge,
                              const int32_t *__restrict__ order, int32_t *__restrict__ tally,
                              double *__restrict__ out, double *__restrict__ scratch, int32_t *__restrict__ redo);
__global__ void k_price_tri(const OptConst *__restrict__ cst, const double *__restrict__ edge,
                            const int32_t *__restrict__ order, int32_t *__restrict__ tally, double *__restrict__ out,
                            double *__restrict__ scratch);
__global__ void k_price_small(DevOpts o, DevYield y, int32_t maxWidth, double unit_dmin, OptConst *__restrict__ cst,
                              int32_t *__restrict__ tally, double *__restrict__ out, double *__restrict__ scratch);
__global__ void k_price_redo(const OptConst *__restrict__ cst, const double *__restrict__ edge,
                             const int32_t *__restrict__ redo, int32_t *__restrict__ tally,
                             double *__restrict__ out, double *__restrict__ scratch);

} // namespace hwt
