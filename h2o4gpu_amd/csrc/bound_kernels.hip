// The rows an assignment pass of a Lloyd loop has to measure (row_bounds.h).
//
// Three launches before the pass: how far each centroid has moved, the rows whose limit the drift
// has passed (every wavefront a stretch of rows of its own, its finds written in row order to the same
// stretch of a list), and the stretches packed into one list. No counter is shared: one atomic
// addition per workgroup to a single address costs some 40 ns behind the others of the chip. Bound by
// the reads of labels and limits: 10M rows, 5 to 30 % found, 20 to 30 us, packing them 8 to 16, moves 5.
#include <algorithm>

#include "kmeans_common.h"

namespace kmhip {

namespace {

constexpr int WG = 256;
constexpr int BOUND_SEGMENTS = 4096;  // stretches of rows at most, one per wavefront

// rows of a stretch: whole rounds of 256
int64_t segment_rows(int64_t n) {
  const int64_t per = (n + BOUND_SEGMENTS - 1) / BOUND_SEGMENTS;
  return (per + 255) / 256 * 256;
}

// moves[c] = |c_new - c_old|, rounded up. A wavefront per centroid.
template <typename T>
__global__ __launch_bounds__(WG) void centroid_moves_kernel(const T *__restrict__ c_old, const T *__restrict__ c_new,
                                                           float *__restrict__ moves, int d, int k) {
  const int c = blockIdx.x * (WG / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (c >= k) return;
  const T *a = c_old + (size_t)c * d, *b = c_new + (size_t)c * d;
  double s = 0;
  bool moved = false;
  for (int j = lane; j < d; j += 64) {
    const double v = (double)b[j] - (double)a[j];
    s += v * v;
    moved |= v != 0;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) s += __shfl_xor(s, off, 64);
  moved = __ballot(moved) != 0;
  // (a move too small for its square or for a float is a move all the same)
  const float m = (float)sqrt(s) * (1.0f + 1e-6f);
  if (lane == 0) moves[c] = moved && m < 1.2e-38f ? 1.2e-38f : m;
}

__global__ __launch_bounds__(WG) void rows_to_measure_kernel(
    const int *__restrict__ labels, const float *__restrict__ limit, int64_t n, int k, int64_t seg_rows,
    const float *__restrict__ moves, const double *__restrict__ drift_old, double *__restrict__ drift_new,
    float *__restrict__ drift_float, int *__restrict__ found, int *__restrict__ found_counts, const BoundControl *__restrict__ ctl,
    BoundControl *__restrict__ ctl_new) {
  extern __shared__ float drift[];  // [k]
  __shared__ float red1[WG / 64], red2[WG / 64];
  __shared__ int red_at[WG / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const bool idle = ctl->wait > 0;  // (nothing is looked for in this step, but the drift goes on)
  if (idle && blockIdx.x > 0) return;
  // the largest move, whose it is, and the largest of the others
  float m1 = -1.0f, m2 = -1.0f;
  int at = -1;
  for (int c = tid; c < k; c += WG) {
    const float m = moves[c];
    if (!(m <= m1)) {  // (a NaN is the largest of all, and no row is then left alone)
      m2 = m1;
      m1 = m;
      at = c;
    } else if (!(m <= m2)) {
      m2 = m;
    }
  }
  auto join = [&](float o1, float o2, int oat) {
    if (!(o1 <= m1)) {
      m2 = !(m1 <= o2) ? m1 : o2;
      m1 = o1;
      at = oat;
    } else if (!(o1 <= m2)) {
      m2 = o1;
    }
  };
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float o1 = __shfl_xor(m1, off, 64), o2 = __shfl_xor(m2, off, 64);
    const int oat = __shfl_xor(at, off, 64);
    join(o1, o2, oat);
  }
  if (lane == 0) {
    red1[tid >> 6] = m1;
    red2[tid >> 6] = m2;
    red_at[tid >> 6] = at;
  }
  __syncthreads();
  m1 = red1[0];
  m2 = red2[0];
  at = red_at[0];
#pragma unroll
  for (int w = 1; w < WG / 64; w++) join(red1[w], red2[w], red_at[w]);
  for (int c = tid; c < k; c += WG) {
    const double s = drift_old[c] + ((double)moves[c] + (double)(c == at ? (m2 > 0 ? m2 : 0.0f) : m1));
    drift[c] = (float)s * (1.0f + 2.4e-7f);
    if (blockIdx.x == 0) {
      drift_new[c] = s;
      drift_float[c] = (float)s;
    }
  }
  // (Centroids that stand still give every row the label it has, near ties and rows without a limit too.)
  if (blockIdx.x == 0 && tid == 0) ctl_new->still = m1 == 0.0f;
  if (idle || m1 == 0.0f) return;
  __syncthreads();
  const int64_t seg = (int64_t)blockIdx.x * (WG / 64) + (tid >> 6);
  const int64_t r0 = seg * seg_rows, r1 = r0 + seg_rows < n ? r0 + seg_rows : n;
  if (r0 >= n) return;
  int *const mine = found + r0;
  int cnt = 0;
  for (int64_t i0 = r0; i0 < r1; i0 += 256) {
    const int64_t i = i0 + lane * 4;
    bool hit[4];
    if (i0 + 256 <= r1) {
      const int4 lab = *reinterpret_cast<const int4 *>(labels + i);
      const float4 lim = *reinterpret_cast<const float4 *>(limit + i);
      const int l[4] = {lab.x, lab.y, lab.z, lab.w};
      const float t[4] = {lim.x, lim.y, lim.z, lim.w};
#pragma unroll
      for (int e = 0; e < 4; e++) hit[e] = (unsigned)l[e] >= (unsigned)k || !(t[e] > drift[l[e]]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        hit[e] = false;
        if (i + e < r1) {
          const int l = labels[i + e];
          hit[e] = (unsigned)l >= (unsigned)k || !(limit[i + e] > drift[l]);
        }
      }
    }
    const unsigned long long below = (1ull << lane) - 1;
    int before = 0, all = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const unsigned long long m = __ballot(hit[e]);
      before += __popcll(m & below);
      all += __popcll(m);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (hit[e]) mine[cnt + before++] = (int)(i + e);
    }
    cnt += all;
  }
  if (lane == 0) found_counts[seg] = cnt;
}

// A workgroup copies the finds of its four stretches behind those of the stretches before.
__global__ __launch_bounds__(WG) void pack_rows_kernel(const int *__restrict__ found,
                                                      const int *__restrict__ found_counts, int segments,
                                                      int64_t seg_rows, int64_t n, int *__restrict__ listed,
                                                      const BoundControl *__restrict__ ctl_old,
                                                      BoundControl *__restrict__ ctl_new, unsigned *news_host) {
  __shared__ unsigned before_s[WG / 64], all_s[WG / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const BoundControl was = *ctl_old;
  const unsigned still = ctl_new->still;
  if (still || was.wait > 0) {
    if (blockIdx.x == 0 && tid == 0) {
      if (still && news_host) __hip_atomic_store(news_host + BOUND_STILL, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      *ctl_new = BoundControl{0u, still ? 0u : 1u, was.wait > 0 ? was.wait - 1 : 0u, was.fails, still ? 0u : 1u, still};
    }
    return;
  }
  const int s0 = blockIdx.x * (WG / 64);
  unsigned before = 0, all = 0;
  for (int s = tid; s < segments; s += WG) {
    const unsigned c = (unsigned)found_counts[s];
    all += c;
    if (s < s0) before += c;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    before += __shfl_xor(before, off, 64);
    all += __shfl_xor(all, off, 64);
  }
  if (lane == 0) {
    before_s[tid >> 6] = before;
    all_s[tid >> 6] = all;
  }
  __syncthreads();
  before = all = 0;
#pragma unroll
  for (int w = 0; w < WG / 64; w++) {
    before += before_s[w];
    all += all_s[w];
  }
  // Most rows: all of them, in order, are cheaper than a list. And while that goes on, the limits are not
  // looked at every time (0, 1, 3, then 7 steps in between).
  const bool full = (int64_t)all * 8 > n * 5;
  if (blockIdx.x == 0 && tid == 0) {
    const unsigned fails = full ? was.fails + 1 : 0;
    if (fails == BOUND_FAILS && news_host)
      __hip_atomic_store(news_host + BOUND_FAILING, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *ctl_new = BoundControl{all, full ? 1u : 0u, full ? (1u << (fails < 4 ? fails - 1 : 3)) - 1 : 0u, fails, full ? 1u : 0u, 0u};
  }
  if (full) return;
  const int wave = tid >> 6;
  for (int w = 0; w < wave; w++)
    if (s0 + w < segments) before += (unsigned)found_counts[s0 + w];
  const int s = s0 + wave;
  if (s >= segments) return;
  const int cnt = found_counts[s];
  const int *const src = found + (int64_t)s * seg_rows;
  for (int e = lane; e < cnt; e += 64) listed[before + e] = src[e];
}

__global__ void first_bounds_kernel(double *__restrict__ drift, float *__restrict__ drift_float, int k,
                                    BoundControl *__restrict__ ctl) {
  for (int c = threadIdx.x; c < k; c += blockDim.x) drift[c] = drift_float[c] = 0.0f;
  if (threadIdx.x == 0) *ctl = BoundControl{0u, 1u, 0u, 0u, 1u, 0u};
}

}  // namespace

int bound_segments(int64_t n) {
  const int64_t per = segment_rows(n);
  return (int)((n + per - 1) / per);
}

template <typename T>
int launch_bounds(hipStream_t s, const T *c_old, const T *c_new, const int *labels, const float *limit, int64_t n,
                  int d, int k, float *moves, const double *drift_old, double *drift_new, float *drift_float, int *found,
                  int *found_counts, int *listed, const BoundControl *ctl_old, BoundControl *ctl_new, unsigned *news_host) {
  if (n < 1 || n > 2147483647 || k < 1 || k > MAX_BOUND_CENTROIDS) return H2O4GPU_KMEANS_EARG;
  if (drift_old == nullptr) {
    hipLaunchKernelGGL(first_bounds_kernel, dim3(1), dim3(WG), 0, s, drift_new, drift_float, k, ctl_new);
    KM_HIP_TRY(hipGetLastError());
    return 0;
  }
  const int segments = bound_segments(n);
  const unsigned groups = (unsigned)((segments + WG / 64 - 1) / (WG / 64));
  hipLaunchKernelGGL((centroid_moves_kernel<T>), dim3((unsigned)((k + WG / 64 - 1) / (WG / 64))), dim3(WG), 0, s,
                     c_old, c_new, moves, d, k);
  hipLaunchKernelGGL(rows_to_measure_kernel, dim3(groups), dim3(WG), (size_t)k * sizeof(float), s, labels, limit, n, k,
                     segment_rows(n), moves, drift_old, drift_new, drift_float, found, found_counts,
                     ctl_old, ctl_new);
  hipLaunchKernelGGL(pack_rows_kernel, dim3(groups), dim3(WG), 0, s, found, found_counts, segments, segment_rows(n), n,
                     listed, ctl_old, ctl_new, news_host);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}
template int launch_bounds<float>(hipStream_t, const float *, const float *, const int *, const float *, int64_t, int,
                                  int, float *, const double *, double *, float *, int *, int *, int *, const BoundControl *,
                                  BoundControl *, unsigned *);
template int launch_bounds<double>(hipStream_t, const double *, const double *, const int *, const float *, int64_t,
                                   int, int, float *, const double *, double *, float *, int *, int *, int *,
                                   const BoundControl *, BoundControl *, unsigned *);

}  // namespace kmhip
