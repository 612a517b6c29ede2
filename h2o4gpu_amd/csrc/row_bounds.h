// What a Lloyd loop keeps per row so that it need not measure every row against every centroid again.
//
// A row at a distance of at most u from its centroid a, and of at least l from every other one, keeps its
// label until the centroids have moved by l - u in all: a by its own move, the others by the largest
// move among them (triangle inequality). An assignment pass that measures a row leaves l - u, less what
// the rounding of any later pass could make of it, in `limit`, plus the drift its centroid has
// gathered so far; the row is measured again once the drift has caught up with the limit. A pass
// over all rows would give the rows in between the labels they have, so labels and counts are those of a loop
// that measures every row every time, from the same centroids. Sums: the tiled kernels' are made from all rows in
// every step, in the same order. The fused step carries its sums; they are the same bits where sums of the values are exact
// in double (whole numbers, a feature spanning less than some 14 binades in a cluster), and else within what SumsLimit
// (kmeans_common.h) allows, which may be the last bit of a float32 mean.
//
// 10M x 32, k = 256 blobs from random rows: the third and fourth step measure all rows (1.13 and 1.23 ms, 0.91 without
// limits), the fifth takes 0.49, the ninth 0.13, the thirtieth 0.06, and finding the rows 0.04; a fit of thirty steps
// 31.5 -> 11.7 ms. 261k x 298, k = 1000, a hundred steps 96 -> 10.5 to 14.9 ms (by the rows), 2M x 256, k = 1024 float64, twenty
// 350 -> 82 to 84, 500k x 784, k = 10, twenty 9.8 -> 2.7 to 4.8. Data without clusters (normal noise) keeps all rows on the list
// and pays for the limits: 0 to 5 % of twenty steps, 8 where a step is no more than reading long rows.
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

// What a computed squared distance is off by at most: products * (xx + cc) by the dot product and the sum,
// norms * xx and norms * cc by the two norms.
struct Rounding {
  float products = 0, norms = 0;
};

struct RowBounds {
  const int *rows = nullptr;  // rows to measure, ascending
  BoundControl *ctl = nullptr;
  float *limit = nullptr;          // [n]
  const float *drift = nullptr;    // [k] of the centroids the rows are measured against
  Rounding noise;
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
// next one at `second`. A centroid at a squared distance D has a norm of at most (sqrt(xx) + sqrt(D))^2, so D is known
// to `own` and to what xx is off by; the latter is the same for all centroids and all passes, and so moves l^2 and u^2 the
// same way: l - u is smallest where both are largest. What a later pass needs to order the two as they are is e2 between
// their squares, i.e. e2 / (l + u) between the distances, and l + u is at least u + sqrt(u^2 + e2) while it holds. Passes
// compare magnitudes: the error of xx is the same for both only where neither distance can come out negative. While
// the limit holds l is at least u / 2, so a u^2 of 8 times what a square may be off by keeps that away; nearer ones have
// it counted against both. -infinity (the row is measured every time) where there is no such gap, and where
// anything is not finite.
// (500k x 784, k = 10, twenty steps, sixteen sets of rows on average: 4.05 ms with all of it counted
// against both, 3.93 so.)
__host__ __device__ __forceinline__ float row_limit(float best, float second, float xx, float drift,
                                                    const Rounding &noise, float grain) {
  // (one-instruction square roots and reciprocal, good to an ulp: every row of a full pass comes through here)
#if defined(__HIP_DEVICE_COMPILE__)
#define KM_SQRT(x) __builtin_amdgcn_sqrtf(x)
#else
#define KM_SQRT(x) sqrtf(x)
#endif
  const float common = noise.norms * xx;
  const float top = second * (1.0f + grain + 2e-7f) + common;
  const float reach = top + 2.0f * KM_SQRT(xx) * KM_SQRT(top);  // (cc - xx, at most)
  const float own = noise.products * (2.0f * xx + reach) + noise.norms * (xx + reach);
  const float step = 2.0f * grain * top;  // of the comparison
  const float hi = best * (1.0f + grain + 2e-7f) + common + own;
  const bool apart = hi > 8.0f * (common + own) + 4.0f * step;
  const float lo = second * (1.0f - 2e-7f) - own + (apart ? common : -common);
  const float e2 = 2.0f * own + step + (apart ? 0.0f : 2.0f * common);
  const float u = KM_SQRT(hi), l = KM_SQRT(lo);
#if defined(__HIP_DEVICE_COMPILE__)
  const float s = e2 * __builtin_amdgcn_rcpf(u + KM_SQRT(hi + e2));
#else
  const float s = e2 / (u + KM_SQRT(hi + e2));
#endif
#undef KM_SQRT
  // (1e-6 l: the roundings of this function; 4e-19: square roots of what is too small for the instruction)
  const float gap = l - u - s - (1e-6f * l + 4e-19f);
  const float at = (drift + gap) * (1.0f - 2.4e-7f);
  return gap > 0.0f && at < 3e38f ? at : -__builtin_huge_valf();
}

// The worst case of whichever kernel measures a distance (u = half an eps is a rounding). Norms are sums of d
// rounded squares one after the other: d u, and as much for any data whose roundings all go the same way, equal
// features for one. Then the dot product, on a scale where no partial sum is above xx + cc and each rounding counts
// twice: d of them on the float32 instructions, and fewer on the bfloat16 parts (six instructions per 16 features, one
// truncation each). Long rows (a lane adds up to 16 products, a tree of six levels the lanes) have 23 instead. Of 1200 eps
// at 784 features equal ones show 213, random ones some 4; a multiple of the random error, 2 sqrt(d) eps, left rows of
// equal features with limits that rounding can pass.
template <typename T>
static inline Rounding bound_noise(int d, bool long_rows = false) {
  const float eps = sizeof(T) == 4 ? 1.1920929e-7f : 2.3e-16f;
  Rounding r;
  r.norms = 0.5f * (float)d * eps;
  if (sizeof(T) == 4) r.products = (long_rows ? 16.0f : 24.0f + (float)d) * eps;
  else r.products = (1.5f * (float)d + 16.0f) * eps;
  return r;
}

}  // namespace kmhip
