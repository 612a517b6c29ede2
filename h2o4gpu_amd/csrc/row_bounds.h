// What a Lloyd loop keeps per row so that it need not measure every row against every centroid again.
//
// A row at a distance of at most u from its centroid a, and of at least l from every other one, keeps its
// label until the centroids have moved by l - u in all: a by its own move, the others by the largest
// move among them (triangle inequality). An assignment pass that measures a row leaves l - u, less what
// the rounding of any later pass could make of it, in `limit`, plus the drift its centroid has
// gathered so far; the row is measured again once the drift has caught up with the limit. A pass
// over all rows would give the rows in between the labels they have, so labels, sums and centroids are
// those of a loop that measures every row every time.
//
// 10M x 32, k = 256 blobs from random rows: the third step measures all rows (1.05 ms, 0.88 without limits),
// the fifth 30 %, the ninth 10, the thirtieth 5 (0.10 ms, a third of it looking for them); thirty steps
// 30.3 -> 11.4 ms. 261k x 298, k = 1000, a hundred steps 93 -> 12.2 ms, 2M x 256, k = 1024 float64, twenty
// 350 -> 81, 500k x 784, k = 10, twenty 9.8 -> 3.9. Data without clusters (normal noise) keeps all rows on the list and
// pays for the limits: 0 to 5 % of twenty steps, 8 where a step is no more than reading long rows.
#pragma once
#include <hip/hip_runtime.h>

namespace kmhip {

// Written by the kernel that gathers the rows to measure, for the assignment pass behind it. (The next
// step's is written from it, so the two alternate.)
struct BoundControl {
  unsigned count;    // rows listed
  unsigned full;     // 1: every row is measured, whatever is listed
  unsigned wait;     // steps to come that measure every row without looking at the limits
  unsigned fails;    // steps in a row whose list held most rows
  unsigned changed;  // 1: some row has a new label
  unsigned still;    // 1: no centroid has moved, and no row is measured
  unsigned fresh;    // 1: no row has a limit yet
  unsigned look;     // 1: decide_rows_kernel goes through the rows
  unsigned listed;   // rows whose limit the drift had passed
};

// The nearest centroids of each centroid (bound_kernels.hip). matrix null: none are kept.
// A pass over fewer listed rows than DECIDE_ROWS leaves CUs idle and takes as long whatever is taken from the list
// (128 rows a workgroup; 261k x 298, k = 1000: 117 us, looking for neighbours 35 and through the list 50). What a
// step needs the neighbours for is known when they have been found, so the list before it is asked as well.
static const int NEAREST = 8;
static const unsigned DECIDE_ROWS = 32768;
struct Neighbours {
  float *matrix = nullptr;  // [k][k] squared distances
  float *dist = nullptr;    // [k][NEAREST + 1] ascending, rounded down; the last is that of the next one
  int *at = nullptr;        // [k][NEAREST + 1]
};

// What a loop keeps beside the drift and the control blocks.
struct BoundBuffers {
  float *limit = nullptr;        // [n]
  int *found = nullptr;          // [n]
  int *listed = nullptr;         // [n]
  int *found_counts = nullptr;   // [bound_counts(n)]
  float *moves = nullptr;        // [k]
  float *drift_float = nullptr;  // [k] the drift, for the pass
  Neighbours near;
  BoundControl *mid = nullptr;   // between the two packings of a step
};

struct RowBounds {
  const int *rows = nullptr;  // rows to measure, ascending
  BoundControl *ctl = nullptr;
  float *limit = nullptr;          // [n]
  const float *drift = nullptr;    // [k] of the centroids the rows are measured against
  float noise = 0;  // a computed squared distance is off by at most noise * (xx + cc)
  float grain = 0;  // and compared at this relative resolution
};

// The rows of a launch: all of them, or (LIST) those a RowBounds names.
template <bool LIST>
struct ListedRows {
  int64_t count;
  __device__ __forceinline__ ListedRows(const RowBounds &, int64_t n) : count(n) {}
  __device__ __forceinline__ int64_t row(int64_t i) const { return i; }
  __device__ __forceinline__ bool all() const { return true; }
  __device__ __forceinline__ void label(int *labels, int64_t row, int c) const { labels[row] = c; }
};
template <>
struct ListedRows<true> {
  int64_t count;
  const int *rows;  // null: all
  unsigned *changed;
  bool limits;  // the next step looks at them
  __device__ __forceinline__ ListedRows(const RowBounds &rb, int64_t n)
      : count(rb.ctl->full ? n : (int64_t)rb.ctl->count), rows(rb.ctl->full ? nullptr : rb.rows),
        changed(&rb.ctl->changed), limits(rb.ctl->wait == 0) {}
  __device__ __forceinline__ int64_t row(int64_t i) const { return rows ? (int64_t)rows[i] : i; }
  __device__ __forceinline__ bool all() const { return rows == nullptr; }
  __device__ __forceinline__ void label(int *labels, int64_t row, int c) const {
    if (rows && labels[row] == c) return;
    labels[row] = c;
    if (rows) *changed = 1;  // (set already where all rows are measured)
  }
};

// The limit of a row whose nearest centroid (with this drift) is at the squared distance `best`, the
// next one at `second`. A centroid at a squared distance D has a norm of at most 2 xx + 2 D, so D is known
// to noise * (3 xx + 2 D). What a later pass needs to order the two as they are is e2 between their squares,
// i.e. e2 / (l + u) between the distances, and l + u is at least u + sqrt(u^2 + e2) while it holds.
// -infinity (the row is measured every time) where there is no such gap, and where anything is not finite.
__device__ __forceinline__ float row_limit(float best, float second, float xx, float drift, float noise,
                                           float grain) {
  // (one-instruction square roots and reciprocal, good to an ulp: every row of a full pass comes through here)
  const float hi = best * (1.0f + grain + 2e-7f) + noise * (3.0f * xx + 2.0f * best);
  const float lo = second * (1.0f - 2e-7f) - noise * (3.0f * xx + 2.0f * second);
  const float e2 = 6.0f * noise * xx + (4.0f * noise + 2.0f * grain) * lo;
#if defined(__HIP_DEVICE_COMPILE__)
  const float u = __builtin_amdgcn_sqrtf(hi), l = __builtin_amdgcn_sqrtf(lo);
  const float s = e2 * __builtin_amdgcn_rcpf(u + __builtin_amdgcn_sqrtf(hi + e2));
#else
  const float u = sqrtf(hi), l = sqrtf(lo), s = e2 / (u + sqrtf(hi + e2));
#endif
  // (1e-6 l: the roundings of this function; 4e-19: square roots of what is too small for the instruction)
  const float gap = l - u - s - (1e-6f * l + 4e-19f);
  const float at = (drift + gap) * (1.0f - 2.4e-7f);
  return gap > 0.0f && at < 3e38f ? at : -__builtin_huge_valf();
}

// What a squared distance can be off by at most, relative to xx + cc, by whichever kernel measures it (u = half an eps
// is a rounding). Norms are sums of d rounded squares one after the other: d u, and as much for any data whose
// roundings all go the same way, equal features for one. Then the dot product, on a scale where no partial sum is
// above xx + cc and each rounding counts twice: d of them on the float32 instructions, and fewer on the bfloat16 parts (six
// instructions per 16 features, one truncation each). Long rows (a lane adds up to 16 products, a tree of six levels the
// lanes) have 23 instead. Of 1200 eps at 784 features equal ones show 213, random ones some 4; a multiple of the random
// error, 2 sqrt(d) eps, left rows of equal features with limits that rounding can pass. 10M x 32, k = 256, and 261k x 298,
// k = 1000, take the same time with either, 500k x 784, k = 10, twenty steps 3.29 and 3.34 ms.
template <typename T>
static inline float bound_noise(int d, bool long_rows = false) {
  if (sizeof(T) == 4) return (long_rows ? 16.0f + 0.5f * (float)d : 24.0f + 1.5f * (float)d) * 1.1920929e-7f;
  return (2.0f * (float)d + 16.0f) * 2.3e-16f;
}

}  // namespace kmhip
