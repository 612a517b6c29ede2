// The rows an assignment pass of a Lloyd loop has to measure (row_bounds.h).
//
// Three launches before the pass: how far each centroid has moved, the rows whose limit the drift
// has passed (every wavefront a stretch of rows of its own, its finds written in row order to the same
// stretch of a list), and the stretches packed into one list. Then, where the centroids' neighbours are kept,
// two more: the listed rows that their neighbours decide, and the others packed again. No counter is shared: one atomic
// addition per workgroup to a single address costs some 40 ns behind the others of the chip. Bound by
// the reads of labels and limits: 10M rows, 5 to 30 % found, 20 to 30 us, packing them 8 to 16, moves 5.
#include <algorithm>

#include "kmeans_common.h"
#include "mfma_traits.h"

namespace kmhip {

namespace {

constexpr int WG = 256;
constexpr int BOUND_SEGMENTS = 4096;  // stretches of rows at most, one per wavefront
constexpr int DECIDE_SEGMENTS = 4096;  // stretches of listed rows (decide_rows_kernel)
constexpr int CT = 32, CT_STEP = 32;  // centroids per tile of the matrix of centroids, features staged at a time

// rows of a stretch: whole rounds of 256
int64_t segment_rows(int64_t n) {
  const int64_t per = (n + BOUND_SEGMENTS - 1) / BOUND_SEGMENTS;
  return (per + 255) / 256 * 256;
}

// |c_new - c_old|, rounded up, by a wavefront.
template <typename T>
__device__ __forceinline__ void centroid_move(const T *__restrict__ a, const T *__restrict__ b, int d, int lane,
                                              float *__restrict__ move) {
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
  if (lane == 0) *move = moved && m < 1.2e-38f ? 1.2e-38f : m;
}

// Squared distances between centroids (float, both triangles), and how far each has moved.
template <typename T>
__global__ __launch_bounds__(WG) void centre_matrix_kernel(const T *__restrict__ c_old, const T *__restrict__ c_new,
                                                          float *__restrict__ moves, float *__restrict__ M, int d, int k,
                                                          int tiles, const BoundControl *__restrict__ ctl) {
  const int tid = threadIdx.x;
  const int pairs = tiles * (tiles + 1) / 2;
  if ((int)blockIdx.x >= pairs) {
    const int c = ((int)blockIdx.x - pairs) * (WG / 64) + (tid >> 6), lane = tid & 63;
    if (c < k) centroid_move(c_old + (size_t)c * d, c_new + (size_t)c * d, d, lane, moves + c);
    return;
  }
  if (ctl->wait > 0 || ctl->listed < DECIDE_ROWS) return;  // (see pack_rows_kernel)
  __shared__ T as[CT_STEP][CT + 1], bs[CT_STEP][CT + 1];
  int ti = 0, rest = blockIdx.x;
  while (rest >= tiles - ti) {
    rest -= tiles - ti;
    ti++;
  }
  const int i0 = ti * CT, j0 = (ti + rest) * CT;
  const int tx = tid & 15, ty = tid >> 4;
  float acc[CT / 16][CT / 16];
#pragma unroll
  for (int p = 0; p < CT / 16; p++)
#pragma unroll
    for (int q = 0; q < CT / 16; q++) acc[p][q] = 0;
  for (int f0 = 0; f0 < d; f0 += CT_STEP) {
    __syncthreads();
    for (int e = tid; e < CT * CT_STEP; e += WG) {
      const int c = e / CT_STEP, f = e % CT_STEP;
      const bool in = f0 + f < d;
      as[f][c] = in && i0 + c < k ? c_new[(size_t)(i0 + c) * d + f0 + f] : (T)0;
      bs[f][c] = in && j0 + c < k ? c_new[(size_t)(j0 + c) * d + f0 + f] : (T)0;
    }
    __syncthreads();
    const int steps = min(CT_STEP, d - f0);
    for (int f = 0; f < steps; f++) {
      T a[CT / 16], b[CT / 16];
#pragma unroll
      for (int p = 0; p < CT / 16; p++) {
        a[p] = as[f][ty + 16 * p];
        b[p] = bs[f][tx + 16 * p];
      }
#pragma unroll
      for (int p = 0; p < CT / 16; p++)
#pragma unroll
        for (int q = 0; q < CT / 16; q++) {
          const float e = (float)(a[p] - b[q]);
          acc[p][q] = fmaf(e, e, acc[p][q]);
        }
    }
  }
#pragma unroll
  for (int p = 0; p < CT / 16; p++)
#pragma unroll
    for (int q = 0; q < CT / 16; q++) {
      const int i = i0 + ty + 16 * p, j = j0 + tx + 16 * q;
      if (i < k && j < k) {
        M[(size_t)i * k + j] = acc[p][q];
        M[(size_t)j * k + i] = acc[p][q];
      }
    }
}

// The nearest centroids of centroid a, by a wavefront: their distances, rounded down, ascending, then that of the
// next one; infinite where there are no more.
__device__ __forceinline__ void nearest_centroids(const float *__restrict__ row, int a, int k, int d, int lane,
                                                  float *__restrict__ dist, int *__restrict__ at) {
  constexpr int HELD = 16;  // (models of up to 1024 centroids are read once)
  unsigned v[HELD];
  const bool hold = k <= HELD * 64;
#pragma unroll
  for (int e = 0; e < HELD; e++) v[e] = hold && e * 64 + lane < k ? __float_as_uint(row[e * 64 + lane]) : ~0u;
  unsigned long long last = 0;  // (distance, centroid) + 1 of the one before
  for (int b = 0; b <= NEAREST; b++) {
    unsigned long long best = ~0ull;
    auto look = [&](unsigned bits, int c) {
      // (a NaN is a distance that rules nothing out; centroid a has none to itself)
      const unsigned long long key = (unsigned long long)(bits > 0x7F800000u ? 0u : bits) << 32 | (unsigned)c;
      if (c < k && c != a && key >= last && key < best) best = key;
    };
    if (hold) {
#pragma unroll
      for (int e = 0; e < HELD; e++)
        if (e * 64 < k) look(v[e], e * 64 + lane);
    } else {
      for (int c = lane; c < k; c += 64) look(__float_as_uint(row[c]), c);
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned long long o = __shfl_xor(best, off, 64);
      best = o < best ? o : best;
    }
    last = best + 1;
    if (lane == 0) {
      // (d + 16 roundings of a sum of squares, and what is too small to square)
      const float r = sqrtf(__uint_as_float((unsigned)(best >> 32))) * (1.0f - 3.1e-8f * (float)(d + 32)) - 4e-19f;
      dist[b] = best == ~0ull ? pos_inf<float>() : r;
      at[b] = best == ~0ull ? a : (int)(best & 0xFFFFFFFFu);
    }
    if (best == ~0ull) last = ~0ull;
  }
}

__global__ __launch_bounds__(WG) void rows_to_measure_kernel(
    const int *__restrict__ labels, const float *__restrict__ limit, int64_t n, int k, int64_t seg_rows,
    const float *__restrict__ moves, const double *__restrict__ drift_old, double *__restrict__ drift_new,
    float *__restrict__ drift_float, int *__restrict__ found, int *__restrict__ found_counts, const BoundControl *__restrict__ ctl,
    BoundControl *__restrict__ ctl_new, int groups, int d, Neighbours near) {
  if ((int)blockIdx.x >= groups) {  // (these look at the centroids, and at no rows)
    const int c = ((int)blockIdx.x - groups) * (WG / 64) + (threadIdx.x >> 6);
    if (c < k && ctl->wait == 0 && ctl->listed >= DECIDE_ROWS)
      nearest_centroids(near.matrix + (size_t)c * k, c, k, d, threadIdx.x & 63, near.dist + (size_t)c * (NEAREST + 1),
                        near.at + (size_t)c * (NEAREST + 1));
    return;
  }
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
  if (idle || m1 == 0.0f || ctl->fresh) return;
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

// Where stretch `seg` of `count` listed rows begins, of DECIDE_SEGMENTS at most.
__device__ __forceinline__ int64_t decide_stretch(int64_t count, int64_t seg) {
  const int64_t per = ((count + DECIDE_SEGMENTS - 1) / DECIDE_SEGMENTS + 7) / 8 * 8;
  const int64_t at = seg * per;
  return at < count ? at : count;
}

// A workgroup copies the finds of its four stretches behind those of the stretches before. AGAIN: the rows that
// decide_rows_kernel has left (ctl_old: the step's control block so far, of the first packing; decides: that
// kernel is to come).
template <bool AGAIN>
__global__ __launch_bounds__(WG) void pack_rows_kernel(const int *__restrict__ found,
                                                      const int *__restrict__ found_counts, int segments,
                                                      int64_t seg_rows, int64_t n, int *__restrict__ listed,
                                                      const BoundControl *__restrict__ ctl_old,
                                                      BoundControl *__restrict__ ctl_new, StepNews *news_host,
                                                      bool decides) {
  __shared__ unsigned before_s[WG / 64], all_s[WG / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const bool one = blockIdx.x == 0 && tid == 0;
  const BoundControl was = *ctl_old;
  if constexpr (AGAIN) {
    if (was.look == 0) {
      if (one) *ctl_new = was;
      return;
    }
  } else {
    const unsigned still = ctl_new->still;
    if (still || was.wait > 0) {
      if (one) {
        if (still && news_host)
          __hip_atomic_store(&news_host->still, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        BoundControl c = {};
        c.full = c.changed = still ? 0u : 1u;
        c.wait = was.wait > 0 ? was.wait - 1 : 0u;
        c.fails = was.fails;
        c.still = still;
        c.listed = still ? 0u : (unsigned)n;
        *ctl_new = c;
      }
      return;
    }
    if (was.fresh) {  // (no row has a limit yet)
      if (one) {
        BoundControl c = {};
        c.full = c.look = 1;
        c.listed = (unsigned)n;
        *ctl_new = c;
      }
      return;
    }
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
  const bool look = !AGAIN && decides && all >= DECIDE_ROWS && was.listed >= DECIDE_ROWS;
  if (one) {
    BoundControl c = {};
    const unsigned fails = full ? was.fails + 1 : 0;
    if (fails == BOUND_FAILS && !look && news_host)
      __hip_atomic_store(&news_host->failing, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    c.count = all;
    c.full = full;
    c.fails = look ? was.fails : fails;
    c.wait = full && !look ? (1u << (fails < 4 ? fails - 1 : 3)) - 1 : 0u;
    c.changed = full || (AGAIN && was.changed);
    c.look = look;
    c.listed = AGAIN ? was.listed : all;
    if (!AGAIN && news_host)
      __hip_atomic_store(&news_host->listed, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *ctl_new = c;
  }
  if (full) return;
  const int wave = tid >> 6;
  for (int w = 0; w < wave; w++)
    if (s0 + w < segments) before += (unsigned)found_counts[s0 + w];
  const int s = s0 + wave;
  if (s >= segments) return;
  const int cnt = found_counts[s];
  const int *const src = found + (AGAIN ? decide_stretch(was.full ? n : (int64_t)was.count, s) : (int64_t)s * seg_rows);
  for (int e = lane; e < cnt; e += 64) listed[before + e] = src[e];
}

// Listed rows whose label the distances between centroids decide.
//
// A row at a distance u from its centroid a is at least |a - b| - u from centroid b (triangle inequality), so only
// centroids within 2 u of a can be nearer: on clustered data the few that share a cluster with a. A listed row is
// measured against its own centroid and against at most NEAREST neighbours of it, and where that decides the
// label beyond any rounding of the pass to come (row_limit) the row has its label and its limit from here.
// Bound by chains of loads, the rows' reads where the list is long: 2M x 256 float64, k = 1024 0.23 ms for the 12 %
// of the rows a late step lists, and the pass behind it 1.86 -> 0.29 ms; 1.4 ms for all rows. A fit of twenty steps
// 142 -> 97 ms, 1M x 256, k = 300 float32 on noise 31.2 -> 31.3 ms (a stretch of rows none of which it decides is given up).
// Rows of LPR lanes each, NV pieces of VW values a lane; U rounds of 64 / LPR rows under way at a time, so that
// their loads overlap. LOCAL: centroids and neighbours are staged in LDS by workgroups as large as a CU takes.
template <bool LOCAL>
constexpr int decide_threads() { return LOCAL ? 1024 : 256; }
template <typename T>
__host__ __device__ inline int decide_row_stride(int d) { return d + 16 / (int)sizeof(T); }  // (LOCAL; other banks)

template <typename T, int VW, int LPR, int NV, bool LOCAL>
__global__ __launch_bounds__(decide_threads<LOCAL>()) void decide_rows_kernel(
    const T *__restrict__ X, const T *__restrict__ xnorm, const T *__restrict__ C, int *__restrict__ labels,
    float *__restrict__ limit, int64_t n, int d, int k, const int *__restrict__ listed, const float *__restrict__ near_dist,
    const int *__restrict__ near_at, const float *__restrict__ drift, int *__restrict__ found,
    int *__restrict__ found_counts, BoundControl *ctl, Rounding noise, float grain) {
  constexpr int TPB = decide_threads<LOCAL>();
  constexpr int RPW = 64 / LPR;
  constexpr int PIECES = VW * NV * (int)sizeof(T) / 4;  // registers of a row's part
  constexpr int U = PIECES <= 4 && sizeof(T) == 4 ? 4 : (PIECES <= 8 ? 2 : 1);
  static_assert(NEAREST == 8 && LPR >= 8, "a lane of a row holds a neighbour");
  typedef T vec_t __attribute__((ext_vector_type(VW), aligned(sizeof(T))));
  const int lane = threadIdx.x & 63, sub = lane % LPR, base = lane - sub;
  const int seg = blockIdx.x * (TPB / 64) + (threadIdx.x >> 6);
  if (ctl->look == 0) return;
  const bool all = ctl->full != 0;
  const int64_t count = all ? n : (int64_t)ctl->count;
  const int64_t lo = decide_stretch(count, seg), hi = decide_stretch(count, seg + 1);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *const cs = reinterpret_cast<T *>(smem_raw);  // (LOCAL) [k][stride], 16-byte rows
  const int stride = LOCAL ? decide_row_stride<T>(d) : d;
  float *const ds = reinterpret_cast<float *>(cs + (size_t)k * stride);  // [k][NEAREST + 1]
  int *const as = reinterpret_cast<int *>(ds + k * (NEAREST + 1));       // [k][NEAREST + 1]
  if constexpr (LOCAL) {
    if (decide_stretch(count, blockIdx.x * (TPB / 64)) >= count) {
      if (lane == 0) found_counts[seg] = 0;
      return;
    }
    for (int e = threadIdx.x; e < k * d; e += TPB) cs[(size_t)(e / d) * stride + e % d] = C[e];
    for (int e = threadIdx.x; e < k * (NEAREST + 1); e += TPB) {
      ds[e] = near_dist[e];
      as[e] = near_at[e];
    }
    __syncthreads();
  }
  const T *const centres = LOCAL ? cs : C;
  const float *const dist_of = LOCAL ? ds : near_dist;
  const int *const at_of = LOCAL ? as : near_at;
  int *const mine = found + lo;
  int cnt = 0, seen = 0;
  const int pieces = (d + VW - 1) / VW;  // (vectors: whole)
  auto distance = [&](const vec_t (&xr)[NV], int c) -> T {  // this lane's part of |x - c|^2
    const T *src = centres + (size_t)c * stride;
    T s = 0;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      if (v * LPR + sub < pieces) {
        const vec_t cv = *reinterpret_cast<const vec_t *>(src + (size_t)(v * LPR + sub) * VW);
#pragma unroll
        for (int q = 0; q < VW; q++) {
          const T e = xr[v][q] - cv[q];
          s = fma(e, e, s);
        }
      }
    }
    return s;
  };
  auto row_sum = [&](T s) -> T {
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) s += __shfl_xor(s, off, 64);
    return s;
  };
  for (int64_t i0 = lo; i0 < hi; i0 += RPW * U) {
    // Data that nothing decides this way (noise): the rest of the stretch is not tried.
    if (seen >= 16 && cnt * 8 > seen * 7) {
      for (int64_t i = i0 + lane; i < hi; i += 64) mine[cnt + (int)(i - i0)] = all ? (int)i : listed[i];
      cnt += (int)(hi - i0);
      break;
    }
    int row[U], own[U], bidx[U], at[U];
    bool valid[U], out[U], open[U];
    vec_t x[U][NV];
    T best[U], second[U];
    float reach[U], rest[U], away[U], xx[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = i0 + u * RPW + lane / LPR;
      valid[u] = i < hi;
      row[u] = all ? (int)min(i, hi - 1) : listed[min(i, hi - 1)];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      own[u] = labels[row[u]];
      xx[u] = (float)xnorm[row[u]];
      const T *src = X + (int64_t)row[u] * d;
#pragma unroll
      for (int v = 0; v < NV; v++)
        x[u][v] = *reinterpret_cast<const vec_t *>(src + (size_t)min(v * LPR + sub, pieces - 1) * VW);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      out[u] = (unsigned)own[u] >= (unsigned)k;
      bidx[u] = out[u] ? 0 : own[u];
      best[u] = distance(x[u], bidx[u]);
      // (lane b of the row holds its b-th neighbour)
      away[u] = dist_of[bidx[u] * (NEAREST + 1) + sub % NEAREST];
      at[u] = at_of[bidx[u] * (NEAREST + 1) + sub % NEAREST];
      rest[u] = dist_of[bidx[u] * (NEAREST + 1) + NEAREST];
    }
    bool any = false;
#pragma unroll
    for (int u = 0; u < U; u++) {
      best[u] = row_sum(best[u]);
      second[u] = pos_inf<T>();
      reach[u] = sqrtf((float)best[u]) * (1.0f + 2e-6f) + 1e-30f;
      // more than the listed neighbours may be nearer, or anything (a NaN): not decided here
      out[u] = out[u] || !valid[u] || !(rest[u] > 2.0f * reach[u]);
      open[u] = !out[u];
      rest[u] -= reach[u];
      any |= open[u];
    }
#pragma unroll 1
    for (int b = 0; b < NEAREST && __ballot(any) != 0; b++) {
      int c[U];
      T dist[U];
      any = false;
#pragma unroll
      for (int u = 0; u < U; u++) {
        const float gap = __shfl(away[u], base + b, 64) - reach[u];
        c[u] = __shfl(at[u], base + b, 64);
        // (a little more than needed: what is measured and not just ruled out leaves the better limit)
        const bool go = open[u] && !(gap >= 1.1f * sqrtf((float)best[u]));
        if (open[u] && !go) rest[u] = gap;
        open[u] = go;
        any |= go;
      }
      if (__ballot(any) == 0) break;
#pragma unroll
      for (int u = 0; u < U; u++) dist[u] = distance(x[u], open[u] ? c[u] : bidx[u]);
#pragma unroll
      for (int u = 0; u < U; u++) {
        dist[u] = row_sum(dist[u]);
        if (open[u]) {
          if (dist[u] < best[u]) {
            second[u] = best[u];
            best[u] = dist[u];
            bidx[u] = c[u];
          } else if (dist[u] < second[u]) {
            second[u] = dist[u];
          }
          out[u] = out[u] || !(dist[u] == dist[u]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      rest[u] = rest[u] > 0 ? rest[u] * (1.0f - 1e-6f) : 0.0f;
      const float others = fminf((float)second[u], rest[u] * rest[u]);
      const float lim = out[u] ? -pos_inf<float>()
                               : row_limit((float)best[u], others, xx[u], drift[bidx[u]], noise, grain);
      const bool left = !(lim > -3e38f);
      if (valid[u] && !left && sub == 0) {
        limit[row[u]] = lim;
        if (bidx[u] != own[u]) {
          labels[row[u]] = bidx[u];
          ctl->changed = 1;
        }
      }
      const unsigned long long m = __ballot(valid[u] && left && sub == 0);
      if (valid[u] && left && sub == 0) mine[cnt + __popcll(m & ((1ull << lane) - 1))] = row[u];
      cnt += __popcll(m);
    }
    seen += (int)min((int64_t)(RPW * U), hi - i0);
  }
  if (lane == 0) found_counts[seg] = cnt;
}

// mindist[i] = |x - c|^2 of each row and the centroid it is labelled with, from the differences (a row without
// a label: the start value of the passes). Rows of LPR lanes, NV pieces of VW values a lane. Bound by reading the
// rows.
template <typename T, int VW, int LPR, int NV>
__global__ __launch_bounds__(WG) void own_distances_kernel(const T *__restrict__ X, const T *__restrict__ C,
                                                          const int *__restrict__ labels, T *__restrict__ mindist,
                                                          int64_t n, int d, int k) {
  constexpr int RPW = 64 / LPR, U = VW * NV * (int)sizeof(T) <= 16 ? 4 : 2;
  typedef T vec_t __attribute__((ext_vector_type(VW), aligned(sizeof(T))));
  const int lane = threadIdx.x & 63, sub = lane % LPR, pieces = (d + VW - 1) / VW;
  const int64_t waves = (int64_t)gridDim.x * (WG / 64);
  for (int64_t i0 = ((int64_t)blockIdx.x * (WG / 64) + (threadIdx.x >> 6)) * (RPW * U); i0 < n; i0 += waves * (RPW * U)) {
    int own[U];
    T s[U];
    vec_t x[U][NV];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t row = min(i0 + u * RPW + lane / LPR, n - 1);
      own[u] = labels[row];
#pragma unroll
      for (int v = 0; v < NV; v++)
        x[u][v] = *reinterpret_cast<const vec_t *>(X + row * d + (size_t)min(v * LPR + sub, pieces - 1) * VW);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const T *src = C + (size_t)((unsigned)own[u] < (unsigned)k ? own[u] : 0) * d;
      s[u] = 0;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        if (v * LPR + sub < pieces) {
          const vec_t cv = *reinterpret_cast<const vec_t *>(src + (size_t)(v * LPR + sub) * VW);
#pragma unroll
          for (int q = 0; q < VW; q++) {
            const T e = x[u][v][q] - cv[q];
            s[u] = fma(e, e, s[u]);
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
#pragma unroll
      for (int off = 1; off < LPR; off <<= 1) s[u] += __shfl_xor(s[u], off, 64);
      const int64_t row = i0 + u * RPW + lane / LPR;
      if (sub == 0 && row < n) mindist[row] = (unsigned)own[u] < (unsigned)k ? s[u] : argmin_start<T>();
    }
  }
}

__global__ void first_bounds_kernel(double *__restrict__ drift, float *__restrict__ drift_float, int k,
                                    BoundControl *__restrict__ ctl, bool fresh) {
  for (int c = threadIdx.x; c < k; c += blockDim.x) drift[c] = drift_float[c] = 0.0f;
  if (threadIdx.x == 0) {
    BoundControl first = {};
    first.full = first.changed = 1;
    first.fresh = fresh;
    first.listed = ~0u;
    *ctl = first;
  }
}

template <typename T>
int launch_decide(hipStream_t s, const BoundBuffers &b, const T *X, const T *xnorm, const T *C, int *labels, int64_t n,
                  int d, int k, float grain) {
  const Rounding noise = bound_noise<T>(d);
  constexpr int VW = Mfma<T>::VW;
  // a model within half a CU's LDS is staged there
  const size_t lds = (size_t)k * (decide_row_stride<T>(d) * sizeof(T) + (NEAREST + 1) * 8);
  const bool local = lds <= 80 * 1024;
#define KM_DECIDE_L(VW, LPR, NV, LOCAL)                                                                            \
  do {                                                                                                             \
    auto kern = decide_rows_kernel<T, VW, LPR, NV, LOCAL>;                                                         \
    constexpr int TPB = decide_threads<LOCAL>();                                                                   \
    KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(kern), LOCAL ? lds : 0));                             \
    hipLaunchKernelGGL(kern, dim3(DECIDE_SEGMENTS / (TPB / 64)), dim3(TPB), LOCAL ? lds : 0, s, X, xnorm, C, labels, \
                       b.limit, n, d, k, b.listed, b.near.dist, b.near.at, b.drift_float, b.found, b.found_counts, \
                       b.mid, noise, grain);                                                     \
  } while (0)
#define KM_DECIDE(VW, LPR, NV)                       \
  do {                                               \
    if (local) KM_DECIDE_L(VW, LPR, NV, true);       \
    else KM_DECIDE_L(VW, LPR, NV, false);            \
  } while (0)
  if (d % VW == 0) {
    const int v = d / VW;
    if (v <= 8) KM_DECIDE(VW, 8, 1);
    else if (v <= 16) KM_DECIDE(VW, 16, 1);
    else if (v <= 32) KM_DECIDE(VW, 32, 1);
    else if (v <= 64) KM_DECIDE(VW, 64, 1);
    else if (v <= 128) KM_DECIDE(VW, 64, 2);
    else if (v <= 256) KM_DECIDE(VW, 64, 4);
    else KM_DECIDE(VW, 64, 8);
  } else {
    // (A piece beyond the row is loaded all the same. 261k x 298, k = 1000, five lists 1199 us with eight pieces, 1115 with six;
    // 150k rows of 601 and 701, 4.94 ms with sixteen, 4.82 with twelve.)
    if (d <= 64) KM_DECIDE(1, 16, 4);
    else if (d <= 256) KM_DECIDE(1, 64, 4);
    else if (d <= 384) KM_DECIDE(1, 64, 6);
    else if (d <= 512) KM_DECIDE(1, 64, 8);
    else if (d <= 768) KM_DECIDE(1, 64, 12);
    else KM_DECIDE(1, 64, 16);
  }
#undef KM_DECIDE
#undef KM_DECIDE_L
  return 0;
}

}  // namespace

template <typename T>
int launch_own_distances(hipStream_t s, const T *X, const T *C, const int *labels, T *mindist, int64_t n, int d, int k,
                         int num_cu) {
  if (n < 1 || k < 1 || !own_distances_apply(d)) return H2O4GPU_KMEANS_EARG;
  constexpr int VW = Mfma<T>::VW;
#define KM_OWN(VW, LPR, NV)                                                                                         \
  hipLaunchKernelGGL((own_distances_kernel<T, VW, LPR, NV>), dim3((unsigned)std::min<int64_t>(                      \
                         (int64_t)num_cu * 8, (n + WG / LPR - 1) / (WG / LPR))), dim3(WG), 0, s, X, C, labels, mindist, n, d, k)
  if (d % VW == 0) {
    const int v = d / VW;
    if (v <= 8) KM_OWN(VW, 8, 1);
    else if (v <= 16) KM_OWN(VW, 16, 1);
    else if (v <= 32) KM_OWN(VW, 32, 1);
    else if (v <= 64) KM_OWN(VW, 64, 1);
    else if (v <= 128) KM_OWN(VW, 64, 2);
    else if (v <= 256) KM_OWN(VW, 64, 4);
    else KM_OWN(VW, 64, 8);
  } else {
    if (d <= 64) KM_OWN(1, 16, 4);
    else if (d <= 256) KM_OWN(1, 64, 4);
    else if (d <= 512) KM_OWN(1, 64, 8);
    else KM_OWN(1, 64, 16);
  }
#undef KM_OWN
  KM_HIP_TRY(hipGetLastError());
  return 0;
}
bool own_distances_apply(int d) { return d >= 1 && d <= 1024; }
template int launch_own_distances<float>(hipStream_t, const float *, const float *, const int *, float *, int64_t, int, int, int);
template int launch_own_distances<double>(hipStream_t, const double *, const double *, const int *, double *, int64_t, int, int,
                                          int);

int bound_segments(int64_t n) {
  const int64_t per = segment_rows(n);
  return (int)((n + per - 1) / per);
}
int bound_counts(int64_t n) { return std::max(bound_segments(n), DECIDE_SEGMENTS); }

// The matrix of centroids costs k^2 d / 2 on the vector ALU: small beside a pass over 64 k rows.
bool neighbours_apply(int64_t n, int d, int k) { return k >= 2 && k <= 4096 && d <= 1024 && n / 64 >= k; }

template <typename T>
int launch_bounds(hipStream_t s, const BoundBuffers &b, BoundStart start, const T *X, const T *xnorm, const T *c_old,
                  const T *c_new, int *labels, int64_t n, int d, int k, const double *drift_old, double *drift_new,
                  const BoundControl *ctl_old, BoundControl *ctl_new, StepNews *news_host, float grain) {
  if (n < 1 || n > 2147483647 || k < 1 || k > MAX_BOUND_CENTROIDS) return H2O4GPU_KMEANS_EARG;
  if (start != BOUNDS_GO) {
    hipLaunchKernelGGL(first_bounds_kernel, dim3(1), dim3(WG), 0, s, drift_new, b.drift_float, k, ctl_new,
                       start == BOUNDS_FRESH);
    KM_HIP_TRY(hipGetLastError());
    return 0;
  }
  const bool decides = b.near.matrix != nullptr;
  if (decides && !neighbours_apply(n, d, k)) return H2O4GPU_KMEANS_EARG;
  const int segments = bound_segments(n);
  const unsigned groups = (unsigned)((segments + WG / 64 - 1) / (WG / 64));
  const unsigned waves = (unsigned)((k + WG / 64 - 1) / (WG / 64));  // a wavefront per centroid
  const int tiles = decides ? (k + CT - 1) / CT : 0;
  hipLaunchKernelGGL((centre_matrix_kernel<T>), dim3((unsigned)(tiles * (tiles + 1) / 2) + waves), dim3(WG), 0, s,
                     c_old, c_new, b.moves, b.near.matrix, d, k, tiles, ctl_old);
  BoundControl *const packed = decides ? b.mid : ctl_new;
  hipLaunchKernelGGL(rows_to_measure_kernel, dim3(groups + (decides ? waves : 0u)), dim3(WG), (size_t)k * sizeof(float), s,
                     labels, b.limit, n, k, segment_rows(n), b.moves, drift_old, drift_new, b.drift_float, b.found,
                     b.found_counts, ctl_old, packed, (int)groups, d, b.near);
  hipLaunchKernelGGL(pack_rows_kernel<false>, dim3(groups), dim3(WG), 0, s, b.found, b.found_counts, segments,
                     segment_rows(n), n, b.listed, ctl_old, packed, news_host, decides);
  if (decides) {
    KM_TRY(launch_decide<T>(s, b, X, xnorm, c_new, labels, n, d, k, grain));
    hipLaunchKernelGGL(pack_rows_kernel<true>, dim3(DECIDE_SEGMENTS / (WG / 64)), dim3(WG), 0, s, b.found,
                       b.found_counts, DECIDE_SEGMENTS, (int64_t)0, n, b.listed, b.mid, ctl_new, news_host, false);
  }
  KM_HIP_TRY(hipGetLastError());
  return 0;
}
#define KM_INST(T)                                                                                                  \
  template int launch_bounds<T>(hipStream_t, const BoundBuffers &, BoundStart, const T *, const T *, const T *, const T *, \
                                int *, int64_t, int, int, const double *, double *, const BoundControl *, BoundControl *,  \
                                StepNews *, float)
KM_INST(float);
KM_INST(double);
#undef KM_INST

}  // namespace kmhip
