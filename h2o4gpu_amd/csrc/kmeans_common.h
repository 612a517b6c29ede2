// Shared declarations of the gfx950 k-means engine: status codes, logging,
// launch-parameter structs and the kernel launchers each .hip file provides.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/h2o4gpu_kmeans.h"
#include "row_bounds.h"

namespace kmhip {

// Logger levels as the reference defines them (src/common/logger.h:10-25):
// a message of level L is printed when 0 < L <= verbose.
enum LogLevel {
  LOG_NOTHING = 0,
  LOG_FATAL = 100,
  LOG_ERROR = 200,
  LOG_INFO = 300,
  LOG_WARN = 400,
  LOG_DEBUG = 500,
  LOG_VERBOSE = 600
};
void log_msg(int verbose, int level, const char *fmt, ...)
    __attribute__((format(printf, 3, 4)));

#define KM_HIP_TRY(expr)                                                     \
  do {                                                                       \
    hipError_t _e = (expr);                                                  \
    if (_e != hipSuccess) {                                                  \
      ::kmhip::log_msg(LOG_ERROR, LOG_ERROR, "%s:%d %s failed: %s", __FILE__, \
                       __LINE__, #expr, hipGetErrorString(_e));              \
      return (_e == hipErrorOutOfMemory) ? H2O4GPU_KMEANS_EALLOC              \
                                         : H2O4GPU_KMEANS_EDEVICE;           \
    }                                                                        \
  } while (0)

#define KM_TRY(expr)            \
  do {                          \
    int _rc = (expr);           \
    if (_rc != 0) return _rc;   \
  } while (0)

// Kernels that use more than 64 KB of dynamic LDS need their limit raised first. That is
// done once per kernel instance, device and size (the largest size granted so far is
// remembered) instead of on every launch; forget_dynamic_lds drops what is remembered for
// a device whose context was reset.
int ensure_dynamic_lds(const void *kernel, size_t bytes);
// How many workgroups of `block` threads with `lds` bytes of dynamic LDS one CU holds at once
// (registers, LDS and wave slots all counted; asked of the runtime once per kernel instance,
// device and size): the grid of a persistent kernel must not exceed this times the CUs, or its
// last workgroups start only when the first ones have finished.
int resident_blocks_per_cu(const void *kernel, int block, size_t lds);
void forget_dynamic_lds(int dev);

// Assign-kernel variants (value of the "assign" option).
enum AssignVariant {
  ASSIGN_AUTO = 0,
  ASSIGN_VALU = 1,     // one thread per row, centroids broadcast from LDS
  ASSIGN_ROWSTAT = 2,  // MFMA, row tile stationary in registers, all centroids in LDS
  ASSIGN_TILED = 3,    // MFMA, both operands staged through LDS over a d-loop
  ASSIGN_LONGROW = 4   // no MFMA: a wavefront along the features of four rows (k <= 16, rows beyond 64 features)
};

// Rows the centroid buffer C (zeros) and entries the norm buffer cnorm (+inf) must
// be padded to: launch_assign / launch_transform may read that far.
static const int CENTROID_PAD = 256;

// Several independent centroid sets (restarts of one fit) laid end to end as one model:
// `sets` sets, each padded to kps rows (a multiple of 32; padding rows are zero) of which
// the first kset are centroids. Labels and minimum distances then hold one [n] block per
// set, the labels counting from the set's own first centroid; partial sums and counts are
// those of the whole stacked model. sets <= 1: an ordinary model. Only the row-stationary
// kernels with the whole model in LDS take a stacked model.
struct StackShape {
  int sets = 1;
  int kps = 0;
  int kset = 0;
};

// The number of bfloat16 products per feature pair (0: the float32 instructions) a launch runs
// with when nobody asked for a number, for each of the three uses of the distance kernels.
static const int SPLIT_DEFAULT = -1;
enum SplitUse { SPLIT_ASSIGN, SPLIT_FUSED, SPLIT_TRANSFORM };
template <typename T>
int default_split(SplitUse use, int64_t n, int d, int k);

// Rows a split launch of the tiled kernel has found within rounding of a tie (near_ties_kernel). A launch
// on the float32 instructions that is given one runs only if more rows were counted than it holds, or
// if a split launch counted 2^31 for rows or norms that are not its.
struct NearTies {
  unsigned *count = nullptr;  // null: nothing is counted (float32: the launch always runs)
  int *rows = nullptr;  // null: none are listed
  unsigned long long *keys = nullptr;
  unsigned cap = 0;
  float margin = 0;  // relative to xx + cc
  unsigned mask = ~0u;  // bits of a distance that are compared (keys: 16 ulp)
};

// Device memory a launch with the bfloat16-parts option may write the centroids' parts to
// (tiled kernel only; tiled_split_scratch_bytes() says how much a launch needs). A launch that
// is given less runs the float32 instructions.
struct SplitScratch {
  void *ptr = nullptr;
  size_t bytes = 0;
  // assignments: settle near ties as the float32 instructions do
  bool near_ties = false;
  // every value of X was a bfloat16 when its norms were made (row_norms' check): the products with its
  // other parts are zeros
  bool rows_bf16 = false;
  // tiled kernels: stage the operands through registers also where the direct-to-LDS form
  // applies (handle option "tiled_direct" = 0)
  bool through_registers = false;
};

// Fused distance + argmin. labels[i] = argmin_c |(xx_i + cc_c) - 2 x_i.c_c|,
// strict '<', lowest index wins, -1 when no distance is below FLT_MAX.
// mindist (nullable) receives the minimum. Returns the variant actually used
// through *used (nullable).
// exact (float32 MFMA kernels only): compare the float distances themselves instead of
// 16-ulp integer keys; slower, for measuring what the key resolution costs in parity.
template <typename T>
int launch_assign(hipStream_t s, int variant, const T *X, const T *xnorm,
                  const T *C, const T *cnorm, int *labels, T *mindist,
                  int64_t n, int d, int k, int num_cu, int *used, bool exact = false,
                  StackShape st = StackShape(), int split = 0, SplitScratch split_scratch = SplitScratch());
// The assignment pass of a loop that keeps bounds (row_bounds.h): the rows rb names get their label and
// their limit (where the next step will look at it), and rb.ctl->changed is set where a label is not the one before. No minimum distances.
// Tiled shapes: float32 with six products (and their scratch, near ties settled), float64.
template <typename T>
bool bounded_assign_applies(int64_t n, int d, int k, int split, const SplitScratch &scratch);
template <typename T>
int launch_bounded_assign(hipStream_t s, const T *X, const T *xnorm, const T *C, const T *cnorm, int *labels,
                          int64_t n, int d, int k, SplitScratch scratch, const RowBounds &rb);
// The fused step of such a loop (float32: row-stationary shapes with six products, long rows with a
// handful of centroids): labels and limits as above; partial sums and counts of all rows where the control block says that all are measured, of
// what the new labels change otherwise, for launch_finalize with RunningSums.
template <typename T>
bool bounded_accumulate_applies(int64_t n, int d, int k, int split, int num_cu);
template <typename T>
int launch_bounded_accumulate(hipStream_t s, const T *X, const T *xnorm, const T *C, int *labels, int64_t n, int d,
                              int k, int num_cu, double *psums, int *pcounts, int *slots, int *tile_rows,
                              const RowBounds &rb);
// The launches before such a pass: how far the centroids have moved, the drift that leaves (drift_old ->
// drift_new), the rows whose limit it has passed, those of them that the centroids' neighbours do not decide,
// and the control block. BOUNDS_FIRST: zeros, and every row is measured. BOUNDS_FRESH: that, for a step that
// leaves no limits; the next one's rows are all looked at. news_host (nullable, pinned) receives the step's news.
// grain: see RowBounds.
struct StepNews {
  unsigned still;    // 1: no centroid has moved
  unsigned failing;  // 1: most rows had to be measured at BOUND_FAILS looks in a row (or see SumsLimit)
  unsigned listed;   // the rows whose limit the drift had passed, where it was looked at
};
static const unsigned BOUND_FAILS = 3;
static const int MAX_BOUND_CENTROIDS = 8192;
enum BoundStart { BOUNDS_GO, BOUNDS_FIRST, BOUNDS_FRESH };
int bound_counts(int64_t n);
bool neighbours_apply(int64_t n, int d, int k);
template <typename T>
int launch_bounds(hipStream_t s, const BoundBuffers &b, BoundStart start, const T *X, const T *xnorm, const T *c_old,
                  const T *c_new, int *labels, int64_t n, int d, int k, const double *drift_old, double *drift_new,
                  const BoundControl *ctl_old, BoundControl *ctl_new, StepNews *news_host, float grain);
// The squared distance of every row to the centroid it is labelled with, from the differences.
bool own_distances_apply(int d);
template <typename T>
int launch_own_distances(hipStream_t s, const T *X, const T *C, const int *labels, T *mindist, int64_t n, int d, int k,
                         int num_cu);
// The resolution distances are compared at by the two passes above.
template <typename T>
float bound_grain(int64_t n, int d, int k, bool fused);
// What launch_assign (variant ASSIGN_AUTO) needs beside the rows and the k centroids for a shape:
enum AssignInputs {
  ASSIGN_FROM_ROWS,       // nothing: xnorm and cnorm may be null, C need not be padded
  ASSIGN_FROM_ROW_NORMS,  // xnorm; cnorm may be null, C need not be padded
  ASSIGN_FROM_MODEL       // both norms, and the padding described at CENTROID_PAD
};
template <typename T>
AssignInputs assign_inputs(int64_t n, int d, int k);
template <typename T>
int pick_assign_variant(int requested, int64_t n, int d, int k);
// The one-pass kernel for long rows and at most 16 centroids (longrow_kernels.hip): whether a
// shape is its (rows of whole 16-byte vectors, centroids and double-precision sums within one
// CU's LDS), the largest number of partial-sum slots its fused form writes, and the launch
// (SUMS false: labels and minimum distances only; cnorm may be null as for the fused kernels).
template <typename T>
bool longrow_applies(int d, int k);
template <typename T>
int longrow_max_slots(int d, int k, int num_cu);
// LIST (float32, SUMS): the rows rb names. longrow_tile_rows: rows a workgroup takes at a time.
template <typename T, bool SUMS, bool LIST = false>
int launch_longrow(hipStream_t s, const T *X, const T *xnorm, const T *C, const T *cnorm, int *labels,
                   T *mindist, int64_t n, int d, int k, int num_cu, double *psums, int *pcounts,
                   int *slots, const RowBounds &rb = RowBounds());
template <typename T>
int longrow_tile_rows(int d);
// The kernel for rows of three to eight float32 features and more than 16 centroids
// (shortrow_kernels.hip): whether a shape is its, and the launch. It makes both norms itself and
// reads the k centroids only; fused: partial sums and counts per workgroup, at most 2 * num_cu slots.
bool shortrow_applies(int d, int k, bool fused);
int launch_shortrow(hipStream_t s, const float *X, const float *C, int *labels, float *mindist, int64_t n, int d,
                    int k, int num_cu, bool fused, double *psums, int *pcounts, int *slots, bool settle);
// Lloyd steps over such rows (three features) once they have been ordered in space and cut into
// blocks of 64 (cell_kernels.hip). ids: a number below CELL_IDS per row, whose order (launch_bucket_rows) the
// windows then refine; range: [cell_range_values()], Xs: [n][d], blocks: [cell_blocks(n)]. The step leaves
// partial sums and counts of at most 2 * num_cu slots and no labels; measured (nullable, zero before): receives
// how many centroids the blocks' rows were measured against, added up over the blocks; stopped: see StopRule.
struct CellBlock {
  float lo[4], hi[4];
  double sum[4];
};
static const int CELL_IDS = 4096;
bool cells_apply(int64_t n, int d, int k);
int64_t cell_blocks(int64_t n);
int cell_range_values();
int launch_cell_ids(hipStream_t s, const float *X, int64_t n, int d, float *range, int *ids);
int launch_cell_windows(hipStream_t s, const float *X, int64_t n, int d, const float *range, const int *order,
                        float *Xs, CellBlock *blocks);
int launch_cell_step(hipStream_t s, const float *Xs, const CellBlock *blocks, int64_t n, const float *C, int d, int k,
                     int num_cu, double *psums, int *pcounts, int *slots, unsigned long long *measured,
                     const unsigned *stopped = nullptr);
const char *assign_variant_name(int variant);
// split (float32 matrix-core kernels; 0, 6 or 9): run the dot products on the bfloat16
// matrix pipe as that many products of bfloat16 parts per feature pair (9: every product
// exact, 6: the three below 2^-24 of |x||c| left out). assign_split_products() returns the
// number a launch of this shape uses: 0 where the option does not apply (float64, the
// vector-ALU kernels, rows of fewer than 4 features; row-stationary kernel: rows padded to
// fewer than 16 or more than 64 features, fused step whose staged parts exceed the LDS
// budget; tiled kernel: 64 centroids or fewer), and such launches run the float32 matrix
// instructions.
template <typename T>
int assign_split_products(int variant, int split, int64_t n, int d, int k, bool fused);
// The tiled kernel keeps the centroids' parts in device scratch of this many bytes
// (split_scratch of launch_assign / launch_transform), written anew by every launch; without
// the scratch (or with 0 bytes needed) it runs the float32 instructions. ties: the rows of an
// assignment whose near ties are settled (0: none are), whose list lies behind the parts.
template <typename T>
size_t tiled_split_scratch_bytes(int split, int d, int k, int64_t ties);

// Fused assign + accumulate (row-stationary MFMA shapes and the small VALU shapes): labels/mindist as
// launch_assign, plus per-workgroup partial sums psums[slot][k][d] and counts
// pcounts[slot][k]; *slots receives the number of slots written. fused_slots()
// returns the largest slot count the launch can use, or 0 when the shape (or a
// forced assign variant) rules the fused kernel out. cnorm may be null: the kernel then
// computes the centroid norms from C itself (same values, j ascending). settle: labels found
// with six products are made the float32 instructions' (near ties settled).
template <typename T>
int fused_slots(int requested_variant, int64_t n, int d, int k, int num_cu);
template <typename T>
int launch_assign_accumulate(hipStream_t s, int variant, const T *X, const T *xnorm, const T *C,
                             const T *cnorm, int *labels, T *mindist, int64_t n, int d,
                             int k, int num_cu, double *psums, int *pcounts, int *slots,
                             int *used, StackShape st = StackShape(), int split = 0, bool settle = false);

// Full squared-distance matrix, centroid-major: D[c * ldn + i], i < n.
template <typename T>
int launch_transform(hipStream_t s, const T *X, const T *xnorm, const T *C,
                     const T *cnorm, T *D, int64_t n, int64_t ldn, int d, int k,
                     int num_cu, int split = 0, SplitScratch split_scratch = SplitScratch());

// out[0 .. n-1] = value
template <typename T>
int launch_fill(hipStream_t s, T *out, T value, int64_t n);

// out[i] = sum_j X[i][j]^2, j ascending, no contraction.
// inexact (nullable, device, zero before the call): receives 1 when some value of X is not a
// bfloat16. Only the pass over many long float32 rows looks (row_norms_check tells); others leave it.
template <typename T>
int launch_row_norms(hipStream_t s, const T *X, T *out, int64_t n, int d, int *inexact = nullptr);
template <typename T>
bool row_norms_check(int64_t n, int d);

// Centroid update, pass 1: per-row-block partial sums (always double) and counts.
struct UpdatePlan {
  int row_blocks;   // partial slots along rows
  int kc;           // centroids per LDS chunk
  int k_chunks;     // ceil(k / kc)
  int vec;          // elements per load (1, 2 or 4)
  int sd;           // LDS row stride of the sums, in elements
  int threads;      // workgroup size of the accumulate kernel (256, 512 or 1024)
  size_t lds_bytes;
};
template <typename T>
UpdatePlan plan_update(int64_t n, int d, int k, int num_cu);
template <typename T>
int launch_accumulate(hipStream_t s, const UpdatePlan &p, const T *X,
                      const int *labels, double *psums, int *pcounts, int64_t n,
                      int d, int k, const unsigned *changed = nullptr);
// Pass 1 for shapes whose sums need many LDS chunks: the rows are ordered by label with a
// stable counting sort (order / order_label: [n] int32 each, offsets: [k] int32,
// block_hist: [bucket_blocks(n, k)][k] int32, seg_hist: [32][k] int32) and summed in fixed
// windows of the ordered rows (partials: [bucket_partial_slots(n, k)][d] double) into
// gsum [k][d] double; counts receives the bucket sizes. Run-to-run reproducible for
// both precisions. The result is consumed by launch_finalize with slots = 1. changed (nullable, device): 0
// says that the labels are those of the pass before, whose gsum and counts are then left as they are.
bool bucketed_update_applies(int k_chunks, int64_t n, int k, int d, size_t elem);
int bucket_blocks(int64_t n, int k);
size_t bucket_partial_slots(int64_t n, int k);
// (the sort alone: order, order_label, counts and offsets, *total rows in all)
int launch_bucket_rows(hipStream_t s, const int *labels, int *order, int *order_label, int *offsets, int *block_hist,
                       int *seg_hist, int *total, int *counts, int64_t n, int k, const unsigned *changed = nullptr);
template <typename T>
int launch_bucketed_accumulate(hipStream_t s, const T *X, const int *labels, int *order,
                               int *order_label, int *offsets, int *block_hist, int *seg_hist,
                               int *total, double *partials, double *gsum, int *counts, int64_t n,
                               int d, int k, const unsigned *changed = nullptr);

// Pass 2: fixed-order reduction of the partials, empty clusters keep the old
// centroid, mean = sum * (1/count), per-block partial of sum((old-new)^2).
// shift_partials must hold max_shift_partials(d, k) entries. frozen (nullable, device,
// [k / kps] flags): centroids of a set of a stacked model whose flag is set stay as they
// are; each block of 32 coordinates then lies inside one set (kps is a multiple of 32), so
// a set's squared shift is the sum of its own partials.
// done (nullable): a counter that is zero between launches; the launch then also leaves the sum of
// its shift partials in *shift2 and, where given, in *shift_host (pinned host memory).
static const int64_t FINALIZE_NARROW_KD = 4096;
static inline int max_shift_partials(int d, int k) {
  const int64_t kd = (int64_t)k * d;
  return (int)(kd <= FINALIZE_NARROW_KD ? (kd + 3) / 4 : (kd + 31) / 32);
}
// run (launch_bounded_accumulate): the partials are changes to sums kept here, unless its control block
// says that all rows were measured; slots is what a launch over all rows writes.
//
// A value that leaves a sum leaves its rounding behind, up to the last bit of the largest sum it has been part of. That
// is of no account to a float32 mean unless the sum is a 2^-28th of what it may have been, rows times the largest value:
// such a sum is made anew, from the rows. (One value that leaves some rows has left 2^-53 of it, and a few times that
// where it met many of them in one workgroup: 2^-25 of a sum at this line. At 2^-24 one fit in fifty of 10M x 32, k = 256, had a
// sum that was small by chance, at 4 ms for each.) No value is larger than the largest row's norm, which is
// enough for most data; where the first sums have smaller ones (features of sizes of their own, features that are zero
// throughout a cluster) the features' values are looked at (launch_least_sums).
struct SumsLimit {
  unsigned anew;       // workgroups that made sums anew since the bounds were begun
  unsigned look;       // 1: the features are to be looked at
  unsigned norm_bits;  // the largest finite norm of a row
};
struct RunningSums {
  double *sums = nullptr;           // [k][d], updated
  const int *counts_old = nullptr;  // [k]
  int *counts_new = nullptr;        // [k], another buffer
  const BoundControl *ctl = nullptr;
  int tile_rows = 0;  // listed rows a workgroup takes at a time: fewer tiles, fewer slots written
  const double *least = nullptr;    // [d]
  const float *X = nullptr;         // [n][d], with the labels the new centroids are made from
  const int *labels = nullptr;
  int64_t n = 0;
  SumsLimit *limit = nullptr;
  StepNews *news_host = nullptr;    // (pinned) `failing` is set when `anew` comes to SUMS_ANEW
};
static const unsigned SUMS_ANEW = 4;
// Before the step that begins the bounds, and behind it.
int launch_sums_limit(hipStream_t s, const float *xnorm, int64_t n, SumsLimit *limit);
// least[f]: a sum of m rows is made anew below m * |least[f]|; 0: never (the sums of the feature are exact in whatever
// order they are made). Negative: also where the partials say that it is what it was.
// scratch: [least_sums_values(n, d)].
size_t least_sums_values(int64_t n, int d);
int launch_least_sums(hipStream_t s, const float *X, const float *xnorm, int64_t n, int d, float *scratch, double *least,
                      const SumsLimit *limit);
// A loop that is queued ahead of its convergence test: the update whose shift is below the threshold says so, and
// the launches behind it that are given the flag do nothing.
struct StopRule {
  unsigned *stopped = nullptr;    // device, 0 at first; null: no such test
  unsigned *step_host = nullptr;  // pinned: receives `step`
  double threshold = 0;
  unsigned step = 0;
};
template <typename T>
int launch_finalize(hipStream_t s, int slots, const double *psums,
                    const int *pcounts, const T *c_old, T *c_new, int *counts,
                    T *shift_partials, int *n_shift_partials, int d, int k,
                    const int *frozen = nullptr, int kps = 1, unsigned *done = nullptr,
                    T *shift2 = nullptr, T *shift_host = nullptr, RunningSums run = RunningSums(),
                    StopRule stop = StopRule());
// Pass 3: cnorm of the new centroids and the fixed-order sum of the shift
// partials into *shift2.
template <typename T>
int launch_post_update(hipStream_t s, const T *c_new, T *cnorm,
                       const T *shift_partials, int n_shift_partials, T *shift2,
                       int d, int k);

// Deterministic sum of n values (two fixed-order stages), result in double.
template <typename T>
int launch_sum(hipStream_t s, const T *v, int64_t n, double *partials,
               int n_partials, double *out);
int sum_partials_needed();

// k-means++ seeding, round t (t = 0 first): mind[i] = min(mind[i], |xx_i + cc - 2 x_i.c|)
// against the t-th chosen centre (row `centre_row` of X; t == 0 overwrites), then
// bsums[b] = sum of mind over rows [b*KPP_BLOCK, (b+1)*KPP_BLOCK) in double with a fixed
// tree. nearest [n] keeps the index of the closest chosen centre so far, rows [k] the
// chosen rows and dcc [k] the distances from the newest centre to the earlier ones: rows
// that the triangle inequality rules out are not read.
static const int KPP_BLOCK = 1024;
template <typename T>
int launch_min_dist_update(hipStream_t s, const T *X, const T *xnorm, int64_t centre_row,
                           T *mind, int *nearest, int *rows, T *dcc, int t, double *bsums,
                           int64_t n, int d);

// k-means|| building blocks (kmeans_h2o4gpu.cu:331-563): a padded model of candidate rows
// for the assign kernels; running minimum cost + its fixed-order block sums
// (bsums: [ceil(n / KPP_BLOCK)]); the reference's per-row acceptance test, rows taken
// appended to list (arrival order, *count may exceed cap); rows per nearest candidate;
// one distance step of the host k-means++ over the candidates.
template <typename T>
int launch_gather_model(hipStream_t s, const T *X, const T *xnorm, const int *idx, int m, int mpad,
                        T *Cc, T *ccn, int d);
template <typename T>
int launch_fold_min(hipStream_t s, const T *cur, T *cost, double *bsums, int64_t n, int init,
                    const int *cur_label = nullptr, int *near = nullptr, int label_off = 0);
template <typename T>
int launch_select_rows(hipStream_t s, const T *cost, T total, uint32_t state0, int k, int *list,
                       int *count, int cap, int64_t n);
int launch_label_histogram(hipStream_t s, const int *labels, int *counts, int64_t n, int m);
// CcT: column-major copy of the m candidate rows Cc (launch_transpose_candidates): the dot
// products are then summed over the features in ascending order, as a scalar loop sums them.
// CcT null: several lanes share a candidate (strided partial sums and a tree; much faster,
// another summation order).
template <typename T>
int launch_transpose_candidates(hipStream_t s, const T *Cc, T *CcT, int m, int d);
template <typename T>
int launch_candidate_dists(hipStream_t s, const T *Cc, const T *CcT, const T *ccn, int centre, T *best,
                           T *mirror, int m, int d, int first);

// The draws of a random permutation that its first k entries depend on. positions draws of
// minstd_rand0 follow state x; draw q serves step first_step + q of the permutation, less the
// draws turned down before it, of which there are at most shuffle_slack(first_step + q) (the
// caller checks). Those that could be turned down (at or past the largest multiple of step + 1) or land in
// [0, k) go to list as (q, value), a block's draws together and in order, table[block] saying where
// they start and how many there are; *total, zero at the start, counts them all (beyond cap they are
// counted and not written).
static const int64_t SHUFFLE_MAX_ROWS = (int64_t)1 << 27;  // beyond, more draws are turned down than the slack
static const int SHUFFLE_BLOCK_DRAWS = 8192;
__host__ __device__ static inline int64_t shuffle_slack(int64_t step) { return step / 32 + 64; }
static inline int shuffle_draw_blocks(int64_t positions) {
  return (int)((positions + SHUFFLE_BLOCK_DRAWS - 1) / SHUFFLE_BLOCK_DRAWS);
}
static inline size_t shuffle_draw_capacity(int64_t n) { return (size_t)n / 16 + 16384; }
int launch_shuffle_draws(hipStream_t s, uint32_t x, int64_t first_step, int64_t positions, int k, uint2 *table,
                         uint2 *list, unsigned cap, unsigned *total);

// Copy rows idx[0..k-1] of X into C ([k][d]).
template <typename T>
int launch_gather_rows(hipStream_t s, const T *X, const int *idx, T *C, int k,
                       int d);

}  // namespace kmhip
