// Row norms, centroid update and reductions.
//
// The centroid update replaces the reference's find_centroids
// (src/gpu/kmeans/kmeans_centroids.h:108-189: copy old centroids, sort (label,
// index) pairs, zero, 30-block run-length accumulate with global atomics,
// revert empties, scale) by
//   pass 1  accumulate : every workgroup owns a contiguous block of rows and a
//           chunk of centroids, keeps that chunk's sums and counts in LDS and
//           writes them to its own slot of a partials buffer (no global
//           atomics, no sort);
//   pass 2  finalize   : sums the slots in slot order, applies the reference's
//           rules (count < 1 keeps the old centroid; mean = sum * (1/count)),
//           and emits per-block partials of sum((old-new)^2), which its last
//           workgroup adds up in order when there are few;
//   pass 3  post_update: the ordered sum of the shift partials when there are
//           many, or of each set of a stacked model, with that set's centroid
//           norms. (Norms of an ordinary model are made by whoever needs them.)
#include <algorithm>

#include "kmeans_common.h"

namespace kmhip {

static constexpr int WG = 256;

// Sums are kept in double in LDS for both precisions and added with ds_add_f64:
// measured on gfx950, ds_add_f32 retires about 0.33 lane-operations per clock
// per CU whatever the address pattern, ds_add_f64 about 8. As a side effect a
// float32 column whose values span fewer than ~14 binades is summed exactly, so
// the result does not depend on the order in which wavefronts arrive.
__device__ __forceinline__ void lds_add(double *p, double v) { unsafeAtomicAdd(p, v); }

// 2 or 4 consecutive row values as one load. The types are aligned to their elements
// only: a row of d values starts wherever it starts, and gfx950 serves such a load with
// one instruction.
template <typename T, int VEC>
struct VecOf;
template <> struct VecOf<float, 4> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct VecOf<float, 2> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct VecOf<double, 2> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };

template <typename T, int VEC>
struct RowVec {
  typedef typename VecOf<T, VEC>::type type;
};
template <typename T>
struct RowVec<T, 1> {
  typedef T type;
};
template <typename T, int VEC>
__device__ __forceinline__ typename RowVec<T, VEC>::type load_vec(const T *p) {
  return *reinterpret_cast<const typename RowVec<T, VEC>::type *>(p);
}
// ---------------------------------------------------------------------------
// out[i] = sum_j X[i][j]^2, j ascending, multiply and add rounded separately
// (what self_dots does, kmeans_labels.h:187-199). One thread per row; used once
// per fit on the data and on k rows per iteration.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(WG) void row_norms_kernel(const T *__restrict__ X,
                                                      T *__restrict__ out,
                                                      int64_t n, int d) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x;
  if (i >= n) return;
  const T *x = X + i * (int64_t)d;
  T acc = 0;
  for (int j = 0; j < d; j++) {
    const T v = x[j];
    acc = acc + v * v;
  }
  out[i] = acc;
}

// Same result, but a group of LPR lanes cooperates on a row so that global
// loads are coalesced; the partial products are exchanged and then added in j
// order by one lane, which keeps the sum bit-identical to the scalar loop.
// Used for the large one-off pass over the data (d <= 64 * VEC).
template <typename T, int LPR>
__global__ __launch_bounds__(WG) void row_norms_coalesced_kernel(
    const T *__restrict__ X, T *__restrict__ out, int64_t n, int d) {
#pragma clang fp contract(off)
  constexpr int ROWS = WG / LPR;
  __shared__ T sq[ROWS][LPR + 1];
  const int sub = threadIdx.x / LPR, col = threadIdx.x % LPR;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int64_t row = row0 + sub;
  T acc = 0;
  for (int j0 = 0; j0 < d; j0 += LPR) {
    const int j = j0 + col;
    T v = (row < n && j < d) ? X[row * (int64_t)d + j] : (T)0;
    sq[sub][col] = v * v;
    __syncthreads();
    if (col == 0) {
      const int lim = min(LPR, d - j0);
      for (int e = 0; e < lim; e++) acc = acc + sq[sub][e];
    }
    __syncthreads();
  }
  if (col == 0 && row < n) out[row] = acc;
}

// Same result for short rows (d <= 64) of a large matrix: a block of 256 rows is one
// contiguous run of 256*d values, fetched as a flat array of 16-byte vectors (the block
// starts on a 16-byte boundary whatever d is; VEC = 1 for data that is not 16-byte aligned)
// into LDS with an odd row stride, and every thread then sums its own row in j order.
template <typename T, int VEC>
__global__ __launch_bounds__(WG) void row_norms_staged_kernel(const T *__restrict__ X,
                                                             T *__restrict__ out, int64_t n, int d) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *Xs = reinterpret_cast<T *>(smem_raw);  // [WG][sx]
  typedef typename RowVec<T, VEC>::type ld_t;
  int sx = d | 1;
  if (((sx + 1) & sx) == 0) sx += 2;  // never 2^m - 1 (measured slow as an LDS row stride)
  const int pad = sx - d;
  const int tid = threadIdx.x;
  const unsigned dinv = d > 1 ? 0xFFFFFFFFu / (unsigned)d + 1u : 0u;  // el / d by multiply-high
  auto row_of = [&](int el) -> int { return d > 1 ? (int)__umulhi((unsigned)el, dinv) : el; };
  for (int64_t base = (int64_t)blockIdx.x * WG; base < n; base += (int64_t)gridDim.x * WG) {
    const int rows = (int)min<int64_t>(WG, n - base);
    const T *xb = X + base * (int64_t)d;
    const int total = rows * d;     // values of this block
    const int nvec = total / VEC;   // complete vectors
    __syncthreads();                // the previous block has been consumed
    for (int e = tid; e < nvec; e += WG) {
      const ld_t v = *reinterpret_cast<const ld_t *>(xb + (size_t)e * VEC);
      const int el = e * VEC;
      if constexpr (VEC == 1) {
        Xs[el + row_of(el) * pad] = v;
      } else {
#pragma unroll
        for (int q = 0; q < VEC; q++) Xs[el + q + row_of(el + q) * pad] = v[q];
      }
    }
    if (tid < total - nvec * VEC) {  // values behind the last complete vector of the data set
      const int el = nvec * VEC + tid;
      Xs[el + row_of(el) * pad] = xb[el];
    }
    __syncthreads();
    if (tid < rows) {
      const T *x = Xs + tid * sx;
      T acc = 0;
      for (int j = 0; j < d; j++) {
        const T v = x[j];
        acc = acc + v * v;
      }
      out[base + tid] = acc;
    }
  }
}

// Same result for many long rows (d > 64): a workgroup owns 256 rows, one per thread, and walks
// along them in pieces of 128 bytes. A piece of all 256 rows is fetched with coalesced 16-byte
// loads (eight lanes per row, eight loads in flight per thread while the piece before is being
// summed), staged in LDS with an odd row stride, and every thread then adds its own row's
// values in j order: all 256 lanes carry a chain of their own, where the cooperative kernel
// above has one lane in 64 adding and two barriers per 64 features.
// Bound by the read of X: 500k x 784 1.40 -> 0.314 ms (5.0 TB/s), 261k x 298 0.078 ms.
template <typename T>
__global__ __launch_bounds__(WG) void row_norms_long_kernel(const T *__restrict__ X, T *__restrict__ out,
                                                           int64_t n, int d, int *__restrict__ inexact) {
#pragma clang fp contract(off)
  constexpr int VW = 16 / sizeof(T);
  constexpr int PIECE = 128 / sizeof(T);  // features per step
  constexpr int VPP = PIECE / VW;         // vectors per row and step: 8
  constexpr int NLD = VPP;                // loads per thread and step (WG rows / (WG / VPP) rows per load)
  constexpr int SX = PIECE + 1;
  typedef typename RowVec<T, VW>::type ld_t;  // aligned to its elements only
  __shared__ T xs[WG * SX];
  const int tid = threadIdx.x;
  const int64_t row0 = (int64_t)blockIdx.x * WG;
  const int lr = tid / VPP, lj = (tid % VPP) * VW;  // this thread's row (of 32 per load) and first feature
  const T *src[NLD];
#pragma unroll
  for (int i = 0; i < NLD; i++) src[i] = X + min(row0 + lr + i * (WG / VPP), n - 1) * (int64_t)d;
  ld_t pre[NLD];
  // a vector that would reach past the end of its row is taken from the row's last VW values;
  // `skip` of its elements then belong to the vector before it
  auto fetch = [&](int j0) {
    const int j = min(j0 + lj, d - VW);
#pragma unroll
    for (int i = 0; i < NLD; i++) pre[i] = load_vec<T, VW>(src[i] + j);
  };
  fetch(0);
  T acc = 0;
  unsigned low = 0;  // bits of the row values below a bfloat16's
  for (int j0 = 0; j0 < d; j0 += PIECE) {
    const int skip = j0 + lj - min(j0 + lj, d - VW);
    __syncthreads();  // the piece before has been consumed
#pragma unroll
    for (int i = 0; i < NLD; i++) {
      T *dst = xs + (lr + i * (WG / VPP)) * SX + lj - skip;
#pragma unroll
      for (int e = 0; e < VW; e++)
        if (e >= skip) dst[e] = pre[i][e];
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int e = 0; e < VW; e++) low |= __float_as_uint(pre[i][e]);
      }
    }
    __syncthreads();
    if (j0 + PIECE < d) fetch(j0 + PIECE);
    const T *x = xs + tid * SX;
    const int lim = min(PIECE, d - j0);
    if (lim == PIECE) {
#pragma unroll
      for (int e = 0; e < PIECE; e++) acc = acc + x[e] * x[e];
    } else {
      for (int e = 0; e < lim; e++) acc = acc + x[e] * x[e];
    }
  }
  if (row0 + tid < n) out[row0 + tid] = acc;
  // (every writer writes the same value; one per wavefront at most)
  if (inexact && __ballot((low & 0xFFFFu) != 0) != 0 && (tid & 63) == 0) *inexact = 1;
}

template <typename T>
__global__ __launch_bounds__(WG) void fill_kernel(T *__restrict__ out, T value, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x;
  if (i < n) out[i] = value;
}
template <typename T>
int launch_fill(hipStream_t s, T *out, T value, int64_t n) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL((fill_kernel<T>), dim3((unsigned)((n + WG - 1) / WG)), dim3(WG), 0, s, out, value, n);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}
template int launch_fill<float>(hipStream_t, float *, float, int64_t);
template int launch_fill<int>(hipStream_t, int *, int, int64_t);
template int launch_fill<double>(hipStream_t, double *, double, int64_t);

static bool row_norms_long(int64_t n, int d) { return d > 64 && n >= 256 * 192; }
template <typename T>
bool row_norms_check(int64_t n, int d) { return sizeof(T) == 4 && row_norms_long(n, d); }
template bool row_norms_check<float>(int64_t, int);
template bool row_norms_check<double>(int64_t, int);

template <typename T>
int launch_row_norms(hipStream_t s, const T *X, T *out, int64_t n, int d, int *inexact) {
  if (n <= 0) return 0;
  if (d >= 4 && d <= 64 && n * (int64_t)d >= (1 << 22)) {
    int sx = d | 1;
    if (((sx + 1) & sx) == 0) sx += 2;
    const size_t lds = (size_t)WG * sx * sizeof(T);
    int64_t grid = (n + WG - 1) / WG;
    if (grid > 256 * 8) grid = 256 * 8;
    constexpr int VW = 16 / sizeof(T);
    if ((reinterpret_cast<uintptr_t>(X) & 15) == 0)
      hipLaunchKernelGGL((row_norms_staged_kernel<T, VW>), dim3((unsigned)grid), dim3(WG), lds, s, X, out,
                         n, d);
    else
      hipLaunchKernelGGL((row_norms_staged_kernel<T, 1>), dim3((unsigned)grid), dim3(WG), lds, s, X, out,
                         n, d);
    KM_HIP_TRY(hipGetLastError());
    return 0;
  }
  // Many long rows: enough workgroups of 256 rows to give most CUs one. Below that (the
  // centroids of a model, a short batch) a row per wavefront spreads further over the chip.
  if (row_norms_long(n, d)) {
    hipLaunchKernelGGL((row_norms_long_kernel<T>), dim3((unsigned)((n + WG - 1) / WG)), dim3(WG), 0, s, X, out, n,
                       d, inexact);
    KM_HIP_TRY(hipGetLastError());
    return 0;
  }
  // (a thread per row is enough for a handful of short rows; long rows always go
  // through the cooperative kernel, a single thread would walk them serially)
  if (d >= 8 && (n * (int64_t)d >= 65536 || d >= 64)) {
    if (d <= 16) {
      constexpr int LPR = 16;
      hipLaunchKernelGGL((row_norms_coalesced_kernel<T, LPR>),
                         dim3((unsigned)((n + WG / LPR - 1) / (WG / LPR))), dim3(WG), 0,
                         s, X, out, n, d);
    } else if (d <= 32) {
      constexpr int LPR = 32;
      hipLaunchKernelGGL((row_norms_coalesced_kernel<T, LPR>),
                         dim3((unsigned)((n + WG / LPR - 1) / (WG / LPR))), dim3(WG), 0,
                         s, X, out, n, d);
    } else {
      constexpr int LPR = 64;
      hipLaunchKernelGGL((row_norms_coalesced_kernel<T, LPR>),
                         dim3((unsigned)((n + WG / LPR - 1) / (WG / LPR))), dim3(WG), 0,
                         s, X, out, n, d);
    }
  } else {
    hipLaunchKernelGGL((row_norms_kernel<T>), dim3((unsigned)((n + WG - 1) / WG)),
                       dim3(WG), 0, s, X, out, n, d);
  }
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// pass 1: accumulate
// grid (row_blocks, k_chunks). LDS: sums[kc][d] + counts[kc].
// A wavefront reads 64 labels at a time, then serves the matching rows one
// group at a time: LPR lanes (each VEC consecutive features per step) per row,
// 64/LPR rows in flight. With a single centroid chunk every row matches and
// the ballot is skipped.
// ---------------------------------------------------------------------------
// adds elements first .. VEC-1 of v to dst[first .. VEC-1]
template <typename T, int VEC, bool RAGGED>
__device__ __forceinline__ void lds_add_vec(double *dst, typename RowVec<T, VEC>::type v, int first) {
  if constexpr (VEC == 1) {
    lds_add(dst, (double)v);
  } else {
#pragma unroll
    for (int e = 0; e < VEC; e++)
      if (!RAGGED || e >= first) lds_add(dst + e, (double)v[e]);
  }
}

// RAGGED: d is not a multiple of VEC (d >= VEC). The vector that would reach past the end
// of the row is fetched from the row's last VEC values instead, and only the elements the
// lane is responsible for (from `first` on) are added.
template <typename T, int VEC, bool RAGGED>
__device__ __forceinline__ void add_row_slice(double *srow, const T *xrow, int col,
                                              int lpr, int d) {
  // lanes col, col+lpr, ... each take VEC consecutive features; four loads are issued
  // before the first add (a load past the end of the row is clamped into it and unused;
  // eight in flight measured slower: short rows then mostly fetch clamped duplicates)
  constexpr int U = 4;
  const int step = lpr * VEC;
  for (int j0 = col * VEC; j0 < d; j0 += U * step) {
    typename RowVec<T, VEC>::type v[U];
    int jc[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      jc[u] = VEC > 1 ? min(j0 + u * step, d - VEC) : min(j0 + u * step, d - 1);
      v[u] = load_vec<T, VEC>(xrow + jc[u]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int j = j0 + u * step;
      if (j < d) lds_add_vec<T, VEC, RAGGED>(srow + jc[u], v[u], j - jc[u]);
    }
  }
}

// sd = LDS row stride of the sums (>= d): chosen odd-ish by the host so that
// rows of different centroids do not all start on the same bank.
template <typename T, int VEC, bool RAGGED, int TPB>
__global__ __launch_bounds__(TPB) void accumulate_kernel(
    const T *__restrict__ X, const int *__restrict__ labels,
    double *__restrict__ psums, int *__restrict__ pcounts, int64_t n, int d, int k,
    int kc, int64_t rows_per_block, int lpr, int sd, const unsigned *changed) {
  if (changed && *changed == 0) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *sums = reinterpret_cast<double *>(smem_raw);         // [kc][sd]
  int *cnt = reinterpret_cast<int *>(sums + (size_t)kc * sd);  // [kc]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int k0 = blockIdx.y * kc;
  const int nk = min(kc, k - k0);
  for (int e = tid; e < nk * sd; e += TPB) sums[e] = 0.0;
  for (int c = tid; c < nk; c += TPB) cnt[c] = 0;
  __syncthreads();

  const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  const int rps = 64 / lpr;  // rows served per wavefront step
  const int sub = lane / lpr, col = lane % lpr;
  const bool single_chunk = gridDim.y == 1;
  const bool narrow = d <= lpr * VEC;  // one vector per lane covers a row
  constexpr int U = 8;

  for (int64_t g0 = r0 + (int64_t)wave * 64; g0 < r1; g0 += (TPB / 64) * 64) {
    const int64_t myrow = g0 + lane;
    int lab = -1;
    if (myrow < r1) lab = labels[myrow] - k0;
    const bool match = lab >= 0 && lab < nk;
    if (match) atomicAdd(&cnt[lab], 1);
    if (single_chunk && narrow) {
      // all loads of U row groups are issued before the first LDS add
      const bool has = col * VEC < d;
      const int jc = RAGGED ? min(col * VEC, d - VEC) : col * VEC;  // see add_row_slice
      const int first = col * VEC - jc;
      for (int b = 0; b < 64; b += rps * U) {
        typename RowVec<T, VEC>::type v[U];
        int l[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int src = b + u * rps + sub;
          l[u] = src < 64 ? __shfl(lab, src & 63, 64) : -1;
          const int64_t row = g0 + src;
          if (!(l[u] >= 0 && l[u] < nk && row < r1 && has)) l[u] = -1;
          v[u] = load_vec<T, VEC>(X + (l[u] >= 0 ? row : r0) * (int64_t)d + (has ? jc : 0));
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          if (l[u] >= 0) lds_add_vec<T, VEC, RAGGED>(sums + (size_t)l[u] * sd + jc, v[u], first);
      }
    } else if (single_chunk) {
      for (int b = 0; b < 64; b += rps) {
        const int src = b + sub;
        const int l = __shfl(lab, src, 64);
        const int64_t row = g0 + src;
        if (l >= 0 && l < nk && row < r1)
          add_row_slice<T, VEC, RAGGED>(sums + (size_t)l * sd, X + row * (int64_t)d, col, lpr, d);
      }
    } else {
      unsigned long long mask = __ballot(match);
      while (mask) {
        // take up to rps set bits; sub-group `sub` serves the sub-th of them
        int src = -1;
        unsigned long long m = mask;
        for (int q = 0; q < rps; q++) {
          if (!m) break;
          const int b = __ffsll((long long)m) - 1;
          if (q == sub) src = b;
          m &= m - 1;
        }
        mask = m;
        const int l = __shfl(lab, src < 0 ? 0 : src, 64);
        if (src >= 0) {
          const int64_t row = g0 + src;
          add_row_slice<T, VEC, RAGGED>(sums + (size_t)l * sd, X + row * (int64_t)d, col, lpr, d);
        }
      }
    }
  }
  __syncthreads();
  double *dst = psums + ((size_t)blockIdx.x * k + k0) * d;
  for (int e = tid; e < nk * d; e += TPB) {
    const int c = e / d, j = e - c * d;
    dst[e] = sums[(size_t)c * sd + j];
  }
  int *cdst = pcounts + (size_t)blockIdx.x * k + k0;
  for (int c = tid; c < nk; c += TPB) cdst[c] = cnt[c];
}

// LDS row stride of the sums (in doubles): odd, so that the rows of different
// centroids start on different banks.
static int update_lds_stride(int d) { return d | 1; }
static constexpr size_t UPDATE_LDS_MAX = 150 * 1024;
static constexpr int KM_MAX_LDS_CHUNKS = 8;

template <typename T>
UpdatePlan plan_update(int64_t n, int d, int k, int num_cu) {
  UpdatePlan p;
  p.sd = update_lds_stride(d);
  const size_t per_centroid = (size_t)p.sd * sizeof(double) + sizeof(int);
  // As few balanced chunks of centroids as a CU's LDS allows (one 1024-thread workgroup
  // per CU when a chunk is large). Every chunk scans all labels and reads the rows that
  // fall into it, so X is read once in total.
  int kc = (int)(UPDATE_LDS_MAX / per_centroid);
  if (kc < 1) kc = 1;
  if (kc > k) kc = k;
  p.k_chunks = (k + kc - 1) / kc;
  kc = (k + p.k_chunks - 1) / p.k_chunks;  // balanced chunks
  p.kc = kc;
  p.lds_bytes = (size_t)kc * per_centroid;
  p.vec = sizeof(T) == 4 ? (d >= 4 ? 4 : (d >= 2 ? 2 : 1)) : (d >= 2 ? 2 : 1);  // see launch_accumulate
  // enough workgroups to cover the machine a few times, but bounded so the
  // partials buffer (row_blocks * k * d) stays small next to the data
  // (fewer when a workgroup's LDS image leaves room for only one or two per CU)
  // An LDS image above 40 KB leaves room for at most three 4-wave workgroups per CU: one
  // 16-wave workgroup per CU then keeps more loads in flight (500k x 784, k = 10, 63 KB:
  // 0.48 -> 0.43 ms); below that, four 4-wave workgroups per CU.
  const bool wide = p.lds_bytes > 40 * 1024;
  p.threads = wide ? 1024 : 256;
  const int per_cu = wide ? 1 : 4;
  int64_t want = (int64_t)num_cu * per_cu / p.k_chunks;
  if (want < 1) want = 1;
  int64_t max_by_rows = (n + 1023) / 1024;  // at least 1024 rows per block
  if (max_by_rows < 1) max_by_rows = 1;
  if (want > max_by_rows) want = max_by_rows;
  // partials traffic 2*rb*k*d should stay below ~1/8 of the data n*d
  int64_t max_by_bytes = n / ((int64_t)16 * k);
  if (max_by_bytes < 1) max_by_bytes = 1;
  if (want > max_by_bytes) want = max_by_bytes;
  p.row_blocks = (int)want;
  return p;
}

template <typename T, int VEC, bool RAGGED>
static int launch_accumulate_vec(hipStream_t s, const UpdatePlan &p, const T *X,
                                 const int *labels, double *psums, int *pcounts,
                                 int64_t n, int d, int k, const unsigned *changed) {
  const int64_t rows_per_block = ((n + p.row_blocks - 1) / p.row_blocks + 63) / 64 * 64;
  int groups = (d + VEC - 1) / VEC;  // lanes wanted per row
  int lpr = 1;
  while (lpr < groups && lpr < 64) lpr <<= 1;
  // workgroup size from the plan: 16 wavefronts when only one workgroup fits a CU
#define KM_ACC_LAUNCH(TPB)                                                                      \
  do {                                                                                          \
    auto kern = accumulate_kernel<T, VEC, RAGGED, TPB>;                                         \
    KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(kern), p.lds_bytes));              \
    hipLaunchKernelGGL(kern, dim3(p.row_blocks, p.k_chunks), dim3(TPB), p.lds_bytes, s, X,      \
                       labels, psums, pcounts, n, d, k, p.kc, rows_per_block, lpr, p.sd, changed);       \
  } while (0)
  if (p.threads == 1024) KM_ACC_LAUNCH(1024);
  else KM_ACC_LAUNCH(256);
#undef KM_ACC_LAUNCH
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

// Lanes take 16 bytes of a row each wherever a row holds that much (8 bytes for float rows
// of 2 or 3 values); the rows need element alignment only.
template <>
int launch_accumulate<float>(hipStream_t s, const UpdatePlan &p, const float *X,
                             const int *labels, double *psums, int *pcounts,
                             int64_t n, int d, int k, const unsigned *changed) {
  if (d >= 4 && d % 4 == 0) return launch_accumulate_vec<float, 4, false>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  if (d >= 4) return launch_accumulate_vec<float, 4, true>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  if (d == 2) return launch_accumulate_vec<float, 2, false>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  if (d == 3) return launch_accumulate_vec<float, 2, true>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  return launch_accumulate_vec<float, 1, false>(s, p, X, labels, psums, pcounts, n, d, k, changed);
}
template <>
int launch_accumulate<double>(hipStream_t s, const UpdatePlan &p, const double *X,
                              const int *labels, double *psums, int *pcounts,
                              int64_t n, int d, int k, const unsigned *changed) {
  if (d >= 2 && d % 2 == 0) return launch_accumulate_vec<double, 2, false>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  if (d >= 2) return launch_accumulate_vec<double, 2, true>(s, p, X, labels, psums, pcounts, n, d, k, changed);
  return launch_accumulate_vec<double, 1, false>(s, p, X, labels, psums, pcounts, n, d, k, changed);
}

// ---------------------------------------------------------------------------
// pass 1, large k*d: bucket rows by label, then sum each bucket.
//
// When the per-centroid sums do not fit in LDS the chunked kernel above has to
// scan all labels once per centroid chunk. Instead the rows are ordered by label
// with a stable counting sort and the ordered rows are summed in fixed windows.
// Nothing in it depends on the order in which workgroups or wavefronts run, so the
// sums are the same bit for bit from run to run, in float64 too:
//   histogram : rows per label of every block of rows               [blocks][k]
//   scan      : per label, exclusive sum over the blocks (two levels), bucket
//               sizes, and the exclusive sum of those over the labels
//   scatter   : position of a row = start of its label's bucket + rows of that
//               label in earlier blocks + rows of that label earlier in its own
//               block (each wavefront walks a contiguous quarter of the block in
//               row order and ranks 64 rows at a time with ballots)
//   window sum: a wavefront sums WPOS consecutive positions of the ordered rows in
//               registers, lanes across features, and stores the sum of every run
//               of equal labels to a slot of its own (window + label: the index
//               grows by at least one from each run to the next, so no two runs
//               share a slot and nothing is added atomically)
//   bucket sum: per label, the slots of its windows are added in window order by
//               four strands with a fixed tree.
// Replaces the reference's sort_by_key + calculate_centroids
// (kmeans_centroids.h:40-75, 131), whose atomic adds arrive in no fixed order.
// ---------------------------------------------------------------------------
// Rows per block of the histogram / scatter: few, so that the blocks fill the chip (261k rows, 64 blocks
// of 4096 rows: a quarter of the CUs), but at least half as many as there are labels, so that a
// block's [k] counters stay small beside its rows.
static constexpr int BUCKET_ROWS_MIN = 1024, BUCKET_ROWS_MAX_MIN = 4096;
static constexpr int BUCKET_MAX_BLOCKS = 2048;
static constexpr int BUCKET_SEGS = 32;        // block segments of the two-level scan

int64_t bucket_rows_per_block(int64_t n, int k) {
  int64_t rpb = (n + BUCKET_MAX_BLOCKS - 1) / BUCKET_MAX_BLOCKS;
  rpb = (rpb + 255) / 256 * 256;
  const int64_t least = std::min<int64_t>(std::max<int64_t>(BUCKET_ROWS_MIN, ((int64_t)k / 2 + 255) / 256 * 256),
                                          BUCKET_ROWS_MAX_MIN);
  return rpb < least ? least : rpb;
}
int bucket_blocks(int64_t n, int k) {
  const int64_t rpb = bucket_rows_per_block(n, k);
  return (int)((n + rpb - 1) / rpb);
}
// wavefronts per scatter workgroup: each keeps its own [k] counters in LDS
static int bucket_waves(int k) {
  if ((size_t)4 * k * sizeof(int) <= 128 * 1024) return 4;
  if ((size_t)2 * k * sizeof(int) <= 128 * 1024) return 2;
  return 1;
}
// positions per window of the window sum: 128 once there are enough windows to fill the GPU
int bucket_window(int64_t n) { return n >= (int64_t)1 << 20 ? 128 : 64; }
size_t bucket_partial_slots(int64_t n, int k) { return (size_t)(n / bucket_window(n) + 2) + k; }

__global__ __launch_bounds__(WG) void bucket_hist_kernel(const int *__restrict__ labels,
                                                        int *__restrict__ bh, int64_t n, int k,
                                                        int64_t rpb, const unsigned *changed) {
  if (changed && *changed == 0) return;
  extern __shared__ int hist[];  // [k]
  const int tid = threadIdx.x;
  for (int c = tid; c < k; c += WG) hist[c] = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * rpb;
  const int64_t r1 = min(n, r0 + rpb);
  for (int64_t i = r0 + tid; i < r1; i += WG) {
    const int l = labels[i];
    if (l >= 0 && l < k) atomicAdd(&hist[l], 1);  // integer counts: order-independent
  }
  __syncthreads();
  int *dst = bh + (size_t)blockIdx.x * k;
  for (int c = tid; c < k; c += WG) dst[c] = hist[c];
}

// Level 1 of the scan over blocks: seg[s][c] = rows of label c in the blocks of segment s.
__global__ __launch_bounds__(WG) void bucket_seg_kernel(const int *__restrict__ bh,
                                                       int *__restrict__ seg, int nb, int k,
                                                       int per_seg, const unsigned *changed) {
  if (changed && *changed == 0) return;
  const int c = blockIdx.x * WG + threadIdx.x;
  if (c >= k) return;
  const int b0 = blockIdx.y * per_seg, b1 = min(nb, b0 + per_seg);
  int sum = 0;
  int b = b0;
  for (; b + 4 <= b1; b += 4) {
    const int v0 = bh[(size_t)b * k + c], v1 = bh[(size_t)(b + 1) * k + c];
    const int v2 = bh[(size_t)(b + 2) * k + c], v3 = bh[(size_t)(b + 3) * k + c];
    sum += v0 + v1 + v2 + v3;
  }
  for (; b < b1; b++) sum += bh[(size_t)b * k + c];
  seg[(size_t)blockIdx.y * k + c] = sum;
}
// Level 2: bh[b][c] <- rows of label c in blocks before b; the last segment also leaves the
// bucket size in counts[c].
__global__ __launch_bounds__(WG) void bucket_block_scan_kernel(int *__restrict__ bh,
                                                              const int *__restrict__ seg,
                                                              int *__restrict__ counts, int nb,
                                                              int k, int per_seg, const unsigned *changed) {
  if (changed && *changed == 0) return;
  const int c = blockIdx.x * WG + threadIdx.x;
  if (c >= k) return;
  int run = 0;
  for (int s = 0; s < (int)blockIdx.y; s++) run += seg[(size_t)s * k + c];
  const int b0 = blockIdx.y * per_seg, b1 = min(nb, b0 + per_seg);
  int b = b0;
  for (; b + 4 <= b1; b += 4) {
    const int v0 = bh[(size_t)b * k + c], v1 = bh[(size_t)(b + 1) * k + c];
    const int v2 = bh[(size_t)(b + 2) * k + c], v3 = bh[(size_t)(b + 3) * k + c];
    bh[(size_t)b * k + c] = run;
    bh[(size_t)(b + 1) * k + c] = run + v0;
    bh[(size_t)(b + 2) * k + c] = run + v0 + v1;
    bh[(size_t)(b + 3) * k + c] = run + v0 + v1 + v2;
    run += v0 + v1 + v2 + v3;
  }
  for (; b < b1; b++) {
    const int v = bh[(size_t)b * k + c];
    bh[(size_t)b * k + c] = run;
    run += v;
  }
  if (blockIdx.y == gridDim.y - 1) counts[c] = run;
}

// offsets[c] = sum of counts[0..c), *total = sum of all; single workgroup.
__global__ __launch_bounds__(WG) void bucket_scan_kernel(const int *__restrict__ counts,
                                                        int *__restrict__ offsets,
                                                        int *__restrict__ total, int k, const unsigned *changed) {
  if (changed && *changed == 0) return;
  __shared__ int part[WG];
  const int tid = threadIdx.x;
  const int per = (k + WG - 1) / WG;
  const int lo = tid * per, hi = min(k, lo + per);
  int s = 0;
  for (int c = lo; c < hi; c++) s += counts[c];
  part[tid] = s;
  __syncthreads();
  if (tid == 0) {
    int run = 0;
    for (int t = 0; t < WG; t++) {
      const int v = part[t];
      part[t] = run;
      run += v;
    }
    *total = run;  // rows that carry a label in [0, k)
  }
  __syncthreads();
  int run = part[tid];
  for (int c = lo; c < hi; c++) {
    offsets[c] = run;
    run += counts[c];
  }
}

// Stable scatter. The workgroup has NWB wavefronts; wavefront w owns rows
// [r0 + w*q, r0 + (w+1)*q) of the block, q = rpb / NWB, and its own counters wh[w][k].
__global__ void bucket_scatter_kernel(const int *__restrict__ labels, const int *__restrict__ bh,
                                      const int *__restrict__ offsets, int *__restrict__ order,
                                      int *__restrict__ order_label, int64_t n, int k, int64_t rpb, const unsigned *changed) {
  if (changed && *changed == 0) return;
  extern __shared__ int wh[];  // [NWB][k]
  const int tid = threadIdx.x, tpb = blockDim.x;
  const int nwb = tpb >> 6, wave = tid >> 6, lane = tid & 63;
  for (int e = tid; e < nwb * k; e += tpb) wh[e] = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * rpb;
  const int64_t q = rpb / nwb;  // rpb is a multiple of 256
  const int64_t w0 = min(n, r0 + wave * q), w1 = min(n, w0 + q);
  int *mine = wh + (size_t)wave * k;
  for (int64_t i = w0 + lane; i < w1; i += 64) {
    const int l = labels[i];
    if (l >= 0 && l < k) atomicAdd(&mine[l], 1);
  }
  __syncthreads();
  // counters -> first position of (this wavefront, label): bucket start + earlier blocks +
  // earlier wavefronts of this block
  const int *bbase = bh + (size_t)blockIdx.x * k;
  for (int c = tid; c < k; c += tpb) {
    int run = offsets[c] + bbase[c];
    for (int w = 0; w < nwb; w++) {
      const int v = wh[(size_t)w * k + c];
      wh[(size_t)w * k + c] = run;
      run += v;
    }
  }
  __syncthreads();
  // 64 rows at a time, in row order: every lane reads its label's counter, lanes with the
  // same label rank themselves by lane number, the first of them advances the counter. The
  // lanes with a lane's own label: one ballot per bit of the label, each narrowing the set to
  // the lanes that agree in it (some 60 instructions for a thousand labels; a loop over the
  // distinct labels of the 64 rows takes ten dependent instructions and two cross-lane reads
  // for each: 261k rows, k = 1000, whole kernel 119 -> 10.6 us, blocks of 1024 instead of 4096 rows included).
  const int bits = 32 - __builtin_clz((unsigned)k);  // labels 0 .. k-1, and k for a row without one
  int l_next = w0 + lane < w1 ? labels[w0 + lane] : -1;
  for (int64_t i0 = w0; i0 < w1; i0 += 64) {
    const int64_t i = i0 + lane;
    const int l = l_next;
    l_next = i + 64 < w1 ? labels[i + 64] : -1;  // travels while this round is ranked
    const bool valid = l >= 0 && l < k;
    const int cur = valid ? mine[l] : 0;
    const unsigned key = valid ? (unsigned)l : (unsigned)k;
    unsigned long long same = ~0ull;
    for (int b = 0; b < bits; b++) {
      const bool set = (key >> b) & 1u;
      const unsigned long long m = __ballot(set);
      same &= set ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    if (valid) {
      order[cur + rank] = (int)i;
      order_label[cur + rank] = l;
      // (one lane per label; read again only in the next round)
      if (rank == 0) mine[l] = cur + __popcll(same);
    }
  }
}

// One wavefront per window of WM*64 consecutive ordered positions; lanes across features
// (VEC each, NVEC vectors per lane cover up to 64*VEC*NVEC features per pass over the rows).
// The sum of every run of equal labels goes to slot (window + label) of P, [slots][d].
template <typename T, int VEC, int NVEC>
__global__ __launch_bounds__(WG) void window_sum_kernel(
    const T *__restrict__ X, const int *__restrict__ order,
    const int *__restrict__ order_label, double *__restrict__ P,
    const int *__restrict__ total, int d, int wm, const unsigned *changed) {
  if (changed && *changed == 0) return;
  const int64_t m = *total;
  const int lane = threadIdx.x & 63;
  const int64_t win = (int64_t)blockIdx.x * (WG / 64) + (threadIdx.x >> 6);
  const int64_t wpos0 = win * wm * 64;
  if (wpos0 >= m) return;
  constexpr int SPAN = 64 * VEC * NVEC;
  for (int d0 = 0; d0 < d; d0 += SPAN) {
    double acc[NVEC][VEC];
#pragma unroll
    for (int q = 0; q < NVEC; q++)
#pragma unroll
      for (int e = 0; e < VEC; e++) acc[q][e] = 0.0;
    // Lane slot q covers features [j, j + VEC). When d is not a multiple of VEC the last
    // such vector would reach past the row: it is fetched from the row's last VEC values
    // instead (offset jc) and only its elements from `first` on belong to this lane.
    int jc[NVEC], first[NVEC];
    bool active[NVEC];
#pragma unroll
    for (int q = 0; q < NVEC; q++) {
      const int j = d0 + (q * 64 + lane) * VEC;
      active[q] = j < d;
      jc[q] = active[q] ? min(j, d - VEC) : 0;
      first[q] = active[q] ? j - jc[q] : 0;
    }
    auto flush = [&](int label) {
      double *dst = P + (size_t)(win + label) * d;
#pragma unroll
      for (int q = 0; q < NVEC; q++) {
#pragma unroll
        for (int e = 0; e < VEC; e++) {
          if (active[q] && e >= first[q]) dst[jc[q] + e] = acc[q][e];
          acc[q][e] = 0.0;
        }
      }
    };
    int cur = -1;
    for (int sub = 0; sub < wm; sub++) {
      const int64_t pos0 = wpos0 + (int64_t)sub * 64;
      if (pos0 >= m) break;
      const int cnt = (int)min<int64_t>(64, m - pos0);
      const int my_row = lane < cnt ? order[pos0 + lane] : 0;
      const int my_lab = lane < cnt ? order_label[pos0 + lane] : -1;
      if (sub == 0) cur = __shfl(my_lab, 0, 64);
      constexpr int U = 4;
      for (int i0 = 0; i0 < cnt; i0 += U) {
        typename RowVec<T, VEC>::type v[U][NVEC];
        int lab[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int i = min(i0 + u, cnt - 1);
          const int row = __shfl(my_row, i, 64);
          lab[u] = __shfl(my_lab, i, 64);
          const T *x = X + (int64_t)row * d;
#pragma unroll
          for (int q = 0; q < NVEC; q++) v[u][q] = load_vec<T, VEC>(x + jc[q]);  // inactive: masked below
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (i0 + u >= cnt) break;
          if (lab[u] != cur) {
            flush(cur);
            cur = lab[u];
          }
#pragma unroll
          for (int q = 0; q < NVEC; q++) {
            if (active[q]) {
              if constexpr (VEC == 1) {
                acc[q][0] += (double)v[u][q];
              } else {
#pragma unroll
                for (int e = 0; e < VEC; e++) acc[q][e] += (double)v[u][q][e];
              }
            }
          }
        }
      }
    }
    flush(cur);
  }
}

// gsum[c][j] = sum over the windows of label c's bucket of P[window + c][j], windows in
// ascending order dealt to 4 strands (window w: strand (w - first) % 4), the four strand
// sums then added as ((s0 + s1) + s2) + s3. grid (k, ceil(d / 64)).
__global__ __launch_bounds__(WG) void bucket_sum_kernel(const double *__restrict__ P,
                                                       const int *__restrict__ offsets,
                                                       const int *__restrict__ counts,
                                                       double *__restrict__ gsum, int d, int wpos, const unsigned *changed) {
  if (changed && *changed == 0) return;
  __shared__ double part[4][64];
  const int c = blockIdx.x;
  const int f = threadIdx.x & 63, strand = threadIdx.x >> 6;
  const int j = blockIdx.y * 64 + f;
  const int cnt = counts[c], off = offsets[c];
  double s = 0.0;
  if (cnt > 0 && j < d) {
    const int w_first = off / wpos, w_last = (off + cnt - 1) / wpos;
    const double *src = P + (size_t)c * d + j;
    int w = w_first + strand;
    for (; w + 12 <= w_last; w += 16) {
      const double a0 = src[(size_t)w * d], a1 = src[(size_t)(w + 4) * d];
      const double a2 = src[(size_t)(w + 8) * d], a3 = src[(size_t)(w + 12) * d];
      s = s + a0;
      s = s + a1;
      s = s + a2;
      s = s + a3;
    }
    for (; w <= w_last; w += 4) s = s + src[(size_t)w * d];
  }
  part[strand][f] = s;
  __syncthreads();
  if (strand == 0 && j < d) gsum[(size_t)c * d + j] = ((part[0][f] + part[1][f]) + part[2][f]) + part[3][f];
}

size_t bucket_lds_bytes(int k) { return (size_t)bucket_waves(k) * k * sizeof(int); }
bool bucketed_update_applies(int k_chunks, int64_t n, int k, int d, size_t elem) {
  if ((size_t)k * sizeof(int) > 128 * 1024) return false;
  // Short rows: up to 8 chunks of centroids the LDS kernel is ahead (2M x 32, k = 4096: 0.15 vs
  // 0.21 ms, 2M x 64, k = 1000: 0.19 vs 0.22).
  if (k_chunks > KM_MAX_LDS_CHUNKS) return true;
  // From rows of about 100 features on, a gathered row is a few whole cache lines and bucketing
  // is ahead as soon as there is more than one chunk (2M x 101, k = 256: 0.30 vs 0.27 ms, 2M x 256,
  // k = 100: 0.57 vs 0.45, 640k x 784, k = 100: 0.54 vs 0.45). With a single chunk (298 features, k = 48
  // 0.59 vs 0.47; 256, k = 48 0.47 vs 0.45) it would need counts that a handful of centroids, whose
  // buckets span thousands of windows each, does not have.
  if (d < 96 || k_chunks <= 1) return false;
  // Float64 rows beyond 256 features: the chunks read whole pages in a row, and on a table that is read
  // from memory that is ahead of gathering (1M x 300, k = 100: 0.51 ordered, 0.47 in chunks; 300k x 784, k = 60
  // 0.40 and 0.37, 200k x 2500, k = 8 0.89 and 0.74; but 300k x 300, k = 100 0.168 and 0.173, 100k x 784, k = 60
  // 0.155 and 0.169, 1M x 256, k = 80 0.432 and 0.433, 1M x 160, k = 120 0.29 and 0.39).
  return !(elem == 8 && d > 256 && (size_t)n * d * elem > ((size_t)1 << 30));
}

int launch_bucket_rows(hipStream_t s, const int *labels, int *order, int *order_label, int *offsets, int *block_hist,
                       int *seg_hist, int *total, int *counts, int64_t n, int k, const unsigned *changed) {
  const int64_t rpb = bucket_rows_per_block(n, k);
  const int nb = bucket_blocks(n, k);
  const int per_seg = (nb + BUCKET_SEGS - 1) / BUCKET_SEGS;
  const int segs = (nb + per_seg - 1) / per_seg;
  const size_t lds1 = (size_t)k * sizeof(int), lds2 = bucket_lds_bytes(k);
  KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(bucket_hist_kernel), lds1));
  KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(bucket_scatter_kernel), lds2));
  const unsigned kblocks = (unsigned)((k + WG - 1) / WG);
  hipLaunchKernelGGL(bucket_hist_kernel, dim3(nb), dim3(WG), lds1, s, labels, block_hist, n, k, rpb, changed);
  hipLaunchKernelGGL(bucket_seg_kernel, dim3(kblocks, segs), dim3(WG), 0, s, block_hist, seg_hist, nb, k,
                     per_seg, changed);
  hipLaunchKernelGGL(bucket_block_scan_kernel, dim3(kblocks, segs), dim3(WG), 0, s, block_hist, seg_hist,
                     counts, nb, k, per_seg, changed);
  hipLaunchKernelGGL(bucket_scan_kernel, dim3(1), dim3(WG), 0, s, counts, offsets, total, k, changed);
  hipLaunchKernelGGL(bucket_scatter_kernel, dim3(nb), dim3(bucket_waves(k) * 64), lds2, s, labels,
                     block_hist, offsets, order, order_label, n, k, rpb, changed);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

template <typename T>
int launch_bucketed_accumulate(hipStream_t s, const T *X, const int *labels, int *order,
                               int *order_label, int *offsets, int *block_hist, int *seg_hist,
                               int *total, double *partials, double *gsum, int *counts, int64_t n,
                               int d, int k, const unsigned *changed) {
  KM_TRY(launch_bucket_rows(s, labels, order, order_label, offsets, block_hist, seg_hist, total, counts, n, k, changed));
  // rows with a label outside [0, k) are not bucketed, so the ordered rows may be fewer
  // than n: the grid covers n positions and every wavefront bounds itself by the
  // device-side total
  const int wm = bucket_window(n) / 64;
  const int64_t windows = (n + (int64_t)wm * 64 - 1) / ((int64_t)wm * 64);
  const unsigned sblocks = (unsigned)((windows + WG / 64 - 1) / (WG / 64));
  // 16-byte loads for any d that holds a whole vector (rows need element alignment only)
#define KM_SEG(VEC, NVEC)                                                                  \
  hipLaunchKernelGGL((window_sum_kernel<T, VEC, NVEC>), dim3(sblocks), dim3(WG), 0, s, X, \
                     order, order_label, partials, total, d, wm, changed)
  if constexpr (sizeof(T) == 4) {
    if (d >= 4) {
      if (d <= 256) KM_SEG(4, 1);
      else if (d <= 512) KM_SEG(4, 2);
      else KM_SEG(4, 4);
    } else {
      KM_SEG(1, 4);
    }
  } else {
    if (d >= 2) {
      if (d <= 128) KM_SEG(2, 1);
      else if (d <= 256) KM_SEG(2, 2);
      else KM_SEG(2, 4);
    } else {
      KM_SEG(1, 4);
    }
  }
#undef KM_SEG
  hipLaunchKernelGGL(bucket_sum_kernel, dim3((unsigned)k, (unsigned)((d + 63) / 64)), dim3(WG), 0, s,
                     partials, offsets, counts, gsum, d, wm * 64, changed);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// pass 2: finalize. One thread per centroid coordinate.
// ---------------------------------------------------------------------------
// A workgroup takes EPW consecutive coordinates; RS = 256 / EPW thread groups
// each sum a contiguous range of the row-block slots for those coordinates (slot
// order), then group 0 adds the RS range sums in range order. EPW is 32, or 4
// for a small model with many slots, where 32 would leave a handful of
// workgroups walking thousands of slots one after the other.
// Fixed-order sum of n partials by the whole workgroup, valid in thread 0.
template <typename T>
__device__ __forceinline__ T sum_shift_partials(const T *shift_partials, int n) {
#pragma clang fp contract(off)
  __shared__ T red[WG];
  const int tid = threadIdx.x;
  // eight loads in flight per thread, added in index order
  T acc = 0;
  int i = tid;
  for (; i + 7 * WG < n; i += 8 * WG) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = shift_partials[i + u * WG];
#pragma unroll
    for (int u = 0; u < 8; u++) acc = acc + v[u];
  }
  for (; i < n; i += WG) acc = acc + shift_partials[i];
  red[tid] = acc;
  __syncthreads();
  for (int off = WG / 2; off > 0; off >>= 1) {
    if (tid < off) red[tid] = red[tid] + red[tid + off];
    __syncthreads();
  }
  return red[0];
}

// What a launch of an update takes beside the sums. Most take nothing, and then the kernel has neither the
// arguments nor the tests: it is a few microseconds long and each step of a fit waits for it (100k x 16, k = 8, two
// hundred steps 2.14 to 2.32 -> 2.01 ms).
struct UpdateAlone {
  static constexpr bool RUN = false, STOP = false;
};
struct UpdateRunning {
  static constexpr bool RUN = true, STOP = false;
  RunningSums run;
};
struct UpdateStopping {
  static constexpr bool RUN = false, STOP = true;
  StopRule stop;
};

template <typename T>
__device__ __forceinline__ void leave_shift(T sum, T *shift2, T *shift_host) {
  *shift2 = sum;
  if (shift_host) __hip_atomic_store(shift_host, sum, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <typename T>
__device__ __forceinline__ void test_shift(T sum, const StopRule &stop) {
  if ((double)sum < stop.threshold) {
    *stop.stopped = 1;
    __hip_atomic_store(stop.step_host, stop.step, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__device__ __forceinline__ double least_by_norm(const SumsLimit &limit) {
  return 3.8e-9 * sqrt((double)__uint_as_float(limit.norm_bits));  // (2^-28, and more than a norm can be off by)
}

// The sums of a workgroup's EPW coordinates (e, of centroid c, of thread tid % EPW) from the rows that are labelled with their
// centroids: valid in the first EPW threads. A wavefront goes through 1024 labels at a time, keeps a queue of the rows that
// are wanted and takes 64 of them at once, its groups of EPW lanes some each, with eight loads under way. Bound by
// one workgroup's loads: 4.2 ms for 10M rows, d = 32, k = 256, whichever number of workgroups it is.
template <int EPW>
__device__ double sums_from_rows(const RunningSums &run, int d, int64_t e, int c, bool valid) {
  constexpr int NW = WG / 64, GROUPS = 64 / EPW, BATCH = 64, U = BATCH / GROUPS < 8 ? BATCH / GROUPS : 8, LOADS = 4;
  __shared__ double red[NW * GROUPS][EPW];
  __shared__ int2 queue[NW][BATCH + 256 * LOADS];  // (row, label)
  const int tid = threadIdx.x, lane = tid & 63, group = lane / EPW;
  const int f = (int)(e - (int64_t)c * d);
  // (a workgroup's coordinates ascend)
  const int first = __shfl(c, 0, 64);
  int last = valid ? c : first;
#pragma unroll
  for (int off = 1; off < EPW; off <<= 1) last = max(last, __shfl_xor(last, off, 64));
  if (tid == 0 && atomicAdd(&run.limit->anew, 1u) + 1 == SUMS_ANEW && run.news_host)
    __hip_atomic_store(&run.news_host->failing, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  double acc = 0;
  int2 *const mine = queue[tid >> 6];
  int waiting = 0;
  auto take = [&](const int2 *from, int count) {
    for (int q0 = 0; q0 < count; q0 += GROUPS * U) {
      float x[U];
      bool is[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int q = q0 + u * GROUPS + group;
        const int2 row = from[min(q, count - 1)];
        is[u] = valid && q < count && row.y == c;
        x[u] = is[u] ? run.X[(int64_t)row.x * d + f] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (is[u]) acc = acc + (double)x[u];
    }
  };
  for (int64_t i0 = (int64_t)(tid >> 6) * (256 * LOADS); i0 < run.n; i0 += (int64_t)NW * 256 * LOADS) {
    int4 label[LOADS];
#pragma unroll
    for (int v = 0; v < LOADS; v++) {
      const int64_t i = i0 + v * 256 + lane * 4;
      if (i + 3 < run.n) {
        label[v] = *reinterpret_cast<const int4 *>(run.labels + i);
      } else {
        label[v].x = i < run.n ? run.labels[i] : -1;
        label[v].y = i + 1 < run.n ? run.labels[i + 1] : -1;
        label[v].z = i + 2 < run.n ? run.labels[i + 2] : -1;
        label[v].w = -1;
      }
    }
    unsigned wanted = 0;  // of this lane's labels
#pragma unroll
    for (int v = 0; v < LOADS; v++) {
      const int its[4] = {label[v].x, label[v].y, label[v].z, label[v].w};
#pragma unroll
      for (int q = 0; q < 4; q++) wanted |= (its[q] >= first && its[q] <= last ? 1u : 0u) << (v * 4 + q);
    }
    if (__ballot(wanted != 0) == 0) continue;
    int before = __popc(wanted);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(before, off, 64);
      if (lane >= off) before += o;
    }
    const int all = __shfl(before, 63, 64);
    before += waiting - __popc(wanted);
#pragma unroll
    for (int v = 0; v < LOADS; v++) {
      const int its[4] = {label[v].x, label[v].y, label[v].z, label[v].w};
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (wanted >> (v * 4 + q) & 1) mine[before++] = make_int2((int)(i0 + v * 256 + lane * 4 + q), its[q]);
    }
    waiting += all;
    int taken = 0;
    for (; waiting - taken >= BATCH; taken += BATCH) take(mine + taken, BATCH);
    waiting -= taken;
    if (taken > 0 && waiting > 0) {
      const int2 rest = mine[taken + min(lane, waiting - 1)];
      if (lane < waiting) mine[lane] = rest;
    }
  }
  if (waiting > 0) take(mine, waiting);
  red[(tid >> 6) * GROUPS + group][lane % EPW] = acc;
  __syncthreads();
  double sum = 0;
  if (tid < EPW)
    for (int q = 0; q < NW * GROUPS; q++) sum = sum + red[q][tid];
  return sum;
}

template <typename T, int EPW, typename With>
__global__ __launch_bounds__(WG) void finalize_kernel(
    const double *__restrict__ psums, const int *__restrict__ pcounts, int row_blocks,
    const T *__restrict__ c_old, T *__restrict__ c_new, int *__restrict__ counts,
    T *__restrict__ shift_partials, int d, int k, const int *__restrict__ frozen, int kps,
    unsigned *__restrict__ done, T *__restrict__ shift2, T *__restrict__ shift_host, With with) {
#pragma clang fp contract(off)
  if constexpr (With::STOP)
    if (*with.stop.stopped != 0) return;
  constexpr int RS = WG / EPW;
  bool changes = false;
  if constexpr (With::RUN) {
    changes = with.run.ctl->full == 0;
    if (changes)
      row_blocks = min(row_blocks, (int)((with.run.ctl->count + with.run.tile_rows - 1) / with.run.tile_rows));
  }
  __shared__ double part[RS][EPW];
  __shared__ int cpart[RS][EPW];
  __shared__ T red[EPW];
  const int tid = threadIdx.x;
  const int slice = tid / EPW, el = tid % EPW;
  const int64_t kd = (int64_t)k * d;
  const int64_t e = (int64_t)blockIdx.x * EPW + el;
  const bool valid = e < kd;
  const int c = valid ? (int)(e / d) : 0;
  const int per = (row_blocks + RS - 1) / RS;
  const int lo = slice * per, hi = min(row_blocks, lo + per);
  double s = 0;
  int cnt = 0;
  if (valid) {
    int rb = lo;
    for (; rb + 4 <= hi; rb += 4) {
      const double a0 = psums[(size_t)rb * kd + e], a1 = psums[(size_t)(rb + 1) * kd + e];
      const double a2 = psums[(size_t)(rb + 2) * kd + e], a3 = psums[(size_t)(rb + 3) * kd + e];
      const int b0 = pcounts[(size_t)rb * k + c], b1 = pcounts[(size_t)(rb + 1) * k + c];
      const int b2 = pcounts[(size_t)(rb + 2) * k + c], b3 = pcounts[(size_t)(rb + 3) * k + c];
      s = s + a0;
      s = s + a1;
      s = s + a2;
      s = s + a3;
      cnt += b0 + b1 + b2 + b3;
    }
    for (; rb < hi; rb++) {
      s = s + psums[(size_t)rb * kd + e];
      cnt += pcounts[(size_t)rb * k + c];
    }
  }
  part[slice][el] = s;
  cpart[slice][el] = cnt;
  __syncthreads();
  bool remade = false;
  double remade_sum = 0;
  if constexpr (With::RUN && sizeof(T) == 4) {
    if (changes && with.run.ctl->count > 0) {
      bool small = false;
      if (slice == 0 && valid) {
        double change = 0;
        int rows = 0;
#pragma unroll
        for (int q = 0; q < RS; q++) {
          change = change + part[q][el];
          rows += cpart[q][el];
        }
        const double least = with.run.least[e - (int64_t)c * d];
        const int old = with.run.counts_old[c];
        rows += old;
        small = least != 0 && rows > 0 && !(least > 0 && change == 0) &&
                !(fabs(with.run.sums[e] + change) >= fabs(least) * (double)max(rows, old));
      }
      remade = __syncthreads_or(small) != 0;
      if (remade) remade_sum = sums_from_rows<EPW>(with.run, d, e, c, valid);
    }
  }
  T diff2 = 0;
  if (slice == 0 && valid) {
    double tot = part[0][el];
    int ctot = cpart[0][el];
#pragma unroll
    for (int q = 1; q < RS; q++) {
      tot = tot + part[q][el];
      ctot += cpart[q][el];
    }
    if constexpr (With::RUN) {
      if (remade) {
        tot = remade_sum;
        ctot += with.run.counts_old[c];
      } else if (changes) {
        tot = with.run.sums[e] + tot;
        ctot += with.run.counts_old[c];
        if (ctot == 0) tot = 0;
      } else if (ctot > 0 && !(fabs(tot) >= 2 * (double)ctot * least_by_norm(*with.run.limit))) {
        with.run.limit->look = 1;
      }
      with.run.sums[e] = tot;
      if (e - (int64_t)c * d == 0) with.run.counts_new[c] = ctot;
    }
    const T oldv = c_old[e];
    T newv;
    // (frozen: a stacked model's set that has met its convergence test keeps its centroids)
    if (ctot < 1 || (frozen != nullptr && frozen[c / kps] != 0)) {
      newv = oldv;  // revert_zeroed_centroids, kmeans_centroids.h:77-88
    } else {
      const T scale = (T)1.0 / (T)ctot;  // scale_centroids, kmeans_centroids.h:90-105
      newv = (T)tot * scale;
    }
    c_new[e] = newv;
    if (e - (int64_t)c * d == 0) counts[c] = ctot;
    const T df = oldv - newv;
    diff2 = df * df;
  }
  if (slice == 0) red[el] = diff2;
  __syncthreads();
  if (tid == 0) {
    T acc = 0;
    for (int q = 0; q < EPW; q++) acc = acc + red[q];
    shift_partials[blockIdx.x] = acc;
  }
  if (done == nullptr) return;
  // The workgroup that finishes last adds the blocks' partials up, in the order of
  // sum_shift_partials whichever it is, and leaves the scalar on the device and, where the host
  // waits for it, in pinned memory: a loop with a convergence test ran a kernel and a copy command
  // for that, some 12 us of an iteration that may have 60.
  __shared__ bool last;
  if (tid == 0)
    last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  const T sum = sum_shift_partials<T>(shift_partials, (int)gridDim.x);
  if (tid == 0) {
    leave_shift(sum, shift2, shift_host);
    if constexpr (With::STOP) test_shift(sum, with.stop);
    *done = 0;  // for the next launch
  }
}

// ---------------------------------------------------------------------------
// pass 3: centroid norms + ordered sum of shift partials.
// Blocks 0 .. ceil(k/WG)-1 compute norms; the last block sums the partials
// with one wavefront in a fixed order.
// ---------------------------------------------------------------------------
template <typename T, typename With>
__global__ __launch_bounds__(WG) void post_update_kernel(
    const T *__restrict__ c_new, T *__restrict__ cnorm,
    const T *__restrict__ shift_partials, int n_partials, T *__restrict__ shift2,
    T *__restrict__ shift_host, int d, int k, With with) {
#pragma clang fp contract(off)
  if constexpr (With::STOP)
    if (*with.stop.stopped != 0) return;
  const int tid = threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {
    const T sum = sum_shift_partials<T>(shift_partials, n_partials);
    if (tid == 0) {
      leave_shift(sum, shift2, shift_host);
      if constexpr (With::STOP) test_shift(sum, with.stop);
    }
    return;
  }
  const int c = blockIdx.x * WG + tid;
  if (c >= k || cnorm == nullptr) return;
  const T *x = c_new + (size_t)c * d;
  T acc = 0;
  for (int j = 0; j < d; j++) {
    const T v = x[j];
    acc = acc + v * v;
  }
  cnorm[c] = acc;
}

template <typename T, typename With>
static int launch_finalize_with(hipStream_t s, int slots, const double *psums, const int *pcounts, const T *c_old,
                                T *c_new, int *counts, T *shift_partials, int *n_shift_partials, int d, int k,
                                const int *frozen, int kps, unsigned *done, T *shift2, T *shift_host, const With &with) {
  const int64_t kd = (int64_t)k * d;
  // (a stacked model always takes the wide form: its sets' partials must not share a block)
  const bool narrow = kd <= FINALIZE_NARROW_KD && slots >= 256 && frozen == nullptr;
  const int blocks = narrow ? (int)((kd + 3) / 4) : (int)((kd + 31) / 32);
  // the last workgroup adds up the shift only while there are few: every one releases its writes and
  // adds to one counter on the way (1024 workgroups: 32 us instead of 8; 48: 6 instead of 4 + 2)
  T *const sum_to = done && blocks > 64 ? shift2 : nullptr;
  if (sum_to) done = nullptr;
  if (narrow)
    hipLaunchKernelGGL((finalize_kernel<T, 4, With>), dim3(blocks), dim3(WG), 0, s, psums, pcounts, slots, c_old,
                       c_new, counts, shift_partials, d, k, frozen, kps, done, shift2, shift_host, with);
  else
    hipLaunchKernelGGL((finalize_kernel<T, 32, With>), dim3(blocks), dim3(WG), 0, s, psums, pcounts, slots, c_old,
                       c_new, counts, shift_partials, d, k, frozen, kps, done, shift2, shift_host, with);
  if (sum_to)
    hipLaunchKernelGGL((post_update_kernel<T, With>), dim3(1), dim3(WG), 0, s, c_new, (T *)nullptr, shift_partials,
                       blocks, sum_to, shift_host, d, k, with);
  KM_HIP_TRY(hipGetLastError());
  *n_shift_partials = blocks;
  return 0;
}

template <typename T>
int launch_finalize(hipStream_t s, int slots, const double *psums,
                    const int *pcounts, const T *c_old, T *c_new, int *counts,
                    T *shift_partials, int *n_shift_partials, int d, int k, const int *frozen,
                    int kps, unsigned *done, T *shift2, T *shift_host, RunningSums run, StopRule stop) {
#define KM_FINALIZE(with)                                                                                          \
  launch_finalize_with<T>(s, slots, psums, pcounts, c_old, c_new, counts, shift_partials, n_shift_partials, d, k,  \
                          frozen, kps, done, shift2, shift_host, with)
  if (run.sums != nullptr && stop.stopped != nullptr) return H2O4GPU_KMEANS_EARG;  // (no loop has both)
  if (run.sums != nullptr) {
    UpdateRunning with;
    with.run = run;
    return KM_FINALIZE(with);
  }
  if (stop.stopped != nullptr) {
    UpdateStopping with;
    with.stop = stop;
    return KM_FINALIZE(with);
  }
  return KM_FINALIZE(UpdateAlone());
#undef KM_FINALIZE
}

// Largest and smallest magnitude of each feature other than zero, and the smallest last bit that is set, over the rows
// whose norm is finite (others have no label). A thread has VEC features of its own; rows beyond the end are the last
// one again. Bound by reading the rows: 500k x 784 0.30 ms (5.2 TB/s), 10M x 32 0.27.
template <int VEC>
__global__ __launch_bounds__(WG) void feature_range_kernel(const float *__restrict__ X, const float *__restrict__ xnorm,
                                                          int64_t n, int d, float *__restrict__ part,
                                                          const SumsLimit *__restrict__ limit) {
  if (limit->look == 0) return;
  constexpr int U = 8;
  extern __shared__ float red[];  // [3][rows of a pass][d]
  const int dv = d / VEC, at_once = WG / dv, tid = threadIdx.x;
  const int r = tid / dv, v = tid - r * dv;
  const bool active = r < at_once;
  float big[VEC], small[VEC], last[VEC];
#pragma unroll
  for (int q = 0; q < VEC; q++) {
    big[q] = 0;
    small[q] = last[q] = __builtin_huge_valf();
  }
  const int64_t step = (int64_t)gridDim.x * at_once;
  for (int64_t i0 = (int64_t)blockIdx.x * at_once + (active ? r : 0); i0 < n; i0 += step * U) {
    typename RowVec<float, VEC>::type x[U];
    float norm[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = min(i0 + u * step, n - 1);
      x[u] = load_vec<float, VEC>(X + i * d + (size_t)v * VEC);
      norm[u] = xnorm[i];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
#pragma unroll
      for (int q = 0; q < VEC; q++) {
        float a;
        if constexpr (VEC == 1) a = fabsf(x[u]);
        else a = fabsf(x[u][q]);
        if (!(norm[u] <= 3.4028234e38f)) a = 0;
        const unsigned bits = __float_as_uint(a);
        const float rest = (bits & 0x7FFFFFu) != 0 ? __uint_as_float(bits & (bits - 1)) : 0.0f;
        big[q] = fmaxf(big[q], a);
        small[q] = fminf(small[q], a > 0 ? a : __builtin_huge_valf());
        last[q] = fminf(last[q], a > 0 ? a - rest : __builtin_huge_valf());
      }
    }
  }
  if (active) {
#pragma unroll
    for (int q = 0; q < VEC; q++) {
      red[(0 * at_once + r) * d + v * VEC + q] = big[q];
      red[(1 * at_once + r) * d + v * VEC + q] = small[q];
      red[(2 * at_once + r) * d + v * VEC + q] = last[q];
    }
  }
  __syncthreads();
  for (int e = tid; e < 3 * d; e += WG) {
    const int what = e / d, f = e - what * d;
    float m = red[what * at_once * d + f];
    for (int q = 1; q < at_once; q++) {
      const float o = red[(what * at_once + q) * d + f];
      m = what == 0 ? fmaxf(m, o) : fminf(m, o);
    }
    part[((size_t)what * gridDim.x + blockIdx.x) * d + f] = m;
  }
}

// A feature's values are multiples of its smallest last bit; sums below 2^53 of that are exact. And where the
// smallest value is no smaller than a 2^-40th of the largest, partials that add up to nothing have lost nothing.
__global__ __launch_bounds__(WG) void least_sums_kernel(const float *__restrict__ part, int parts, int64_t n, int d,
                                                       double *__restrict__ least,
                                                       const SumsLimit *__restrict__ limit) {
  __shared__ float red[3][WG];
  const int tid = threadIdx.x, f = blockIdx.x;
  if (limit->look == 0) {
    if (tid == 0) least[f] = -least_by_norm(*limit);
    return;
  }
#pragma unroll
  for (int what = 0; what < 3; what++) {
    float m = what == 0 ? 0.0f : __builtin_huge_valf();
    for (int b = tid; b < parts; b += WG) {
      const float o = part[((size_t)what * parts + b) * d + f];
      m = what == 0 ? fmaxf(m, o) : fminf(m, o);
    }
    red[what][tid] = m;
  }
  __syncthreads();
  for (int off = WG / 2; off > 0; off >>= 1) {
    if (tid < off) {
      red[0][tid] = fmaxf(red[0][tid], red[0][tid + off]);
      red[1][tid] = fminf(red[1][tid], red[1][tid + off]);
      red[2][tid] = fminf(red[2][tid], red[2][tid + off]);
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double big = red[0][0], small = red[1][0], last = red[2][0];
    const bool exact = big == 0 || (double)n * big <= 4503599627370496.0 * last;  // (2^52)
    const double below = big * 3.7252902984619140625e-9;                         // (2^-28)
    least[f] = exact ? 0.0 : (small * 1099511627776.0 >= big ? below : -below);
  }
}

static int range_blocks(int64_t n) { return (int)std::min<int64_t>((n + 63) / 64, 1024); }
size_t least_sums_values(int64_t n, int d) { return (size_t)3 * range_blocks(n) * d; }

int launch_least_sums(hipStream_t s, const float *X, const float *xnorm, int64_t n, int d, float *scratch, double *least,
                      const SumsLimit *limit) {
  const int vec = d % 4 == 0 ? 4 : 1;
  if (n < 1 || d < 1 || d / vec > WG) return H2O4GPU_KMEANS_EARG;
  const int parts = range_blocks(n);
  const size_t lds = (size_t)3 * (WG / (d / vec)) * d * sizeof(float);  // (12 KB at most)
  if (vec == 4)
    hipLaunchKernelGGL(feature_range_kernel<4>, dim3(parts), dim3(WG), lds, s, X, xnorm, n, d, scratch, limit);
  else
    hipLaunchKernelGGL(feature_range_kernel<1>, dim3(parts), dim3(WG), lds, s, X, xnorm, n, d, scratch, limit);
  hipLaunchKernelGGL(least_sums_kernel, dim3(d), dim3(WG), 0, s, scratch, parts, n, d, least, limit);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

__global__ __launch_bounds__(WG) void largest_norm_kernel(const float *__restrict__ xnorm, int64_t n,
                                                         SumsLimit *__restrict__ limit) {
  constexpr int U = 8;
  unsigned big = 0;
  const int64_t step = (int64_t)gridDim.x * WG;
  for (int64_t i0 = (int64_t)blockIdx.x * WG + threadIdx.x; i0 < n; i0 += step * U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned bits = __float_as_uint(xnorm[min(i0 + u * step, n - 1)]);  // (not negative: ordered as its bits are)
      if (bits < 0x7F800000u) big = max(big, bits);
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) big = max(big, (unsigned)__shfl_xor((int)big, off, 64));
  __shared__ unsigned red[WG / 64];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = big;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < WG / 64; w++) big = max(big, red[w]);
    atomicMax(&limit->norm_bits, big);
  }
}
int launch_sums_limit(hipStream_t s, const float *xnorm, int64_t n, SumsLimit *limit) {
  if (n < 1) return H2O4GPU_KMEANS_EARG;
  KM_TRY(launch_fill<int>(s, reinterpret_cast<int *>(limit), 0, sizeof(SumsLimit) / sizeof(int)));
  const int grid = (int)std::min<int64_t>((n + 8 * WG - 1) / (8 * WG), 512);
  hipLaunchKernelGGL(largest_norm_kernel, dim3(grid), dim3(WG), 0, s, xnorm, n, limit);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

template <typename T>
int launch_post_update(hipStream_t s, const T *c_new, T *cnorm,
                       const T *shift_partials, int n_shift_partials, T *shift2,
                       int d, int k) {
  // large centroid sets: norms by the coalesced row-norm kernel (same summation order),
  // this kernel then only adds up the shift partials
  const bool separate_norms = d >= 8 && ((int64_t)k * d >= 65536 || d >= 64);
  const int blocks = separate_norms ? 1 : (k + WG - 1) / WG + 1;
  hipLaunchKernelGGL((post_update_kernel<T, UpdateAlone>), dim3(blocks), dim3(WG), 0, s, c_new,
                     separate_norms ? (T *)nullptr : cnorm, shift_partials, n_shift_partials,
                     shift2, (T *)nullptr, d, k, UpdateAlone());
  KM_HIP_TRY(hipGetLastError());
  if (separate_norms) return launch_row_norms<T>(s, c_new, cnorm, k, d);
  return 0;
}

// ---------------------------------------------------------------------------
// Deterministic sum of n values in double: stage 1 gives every block a fixed
// contiguous range and a fixed tree, stage 2 adds the block results in order.
// ---------------------------------------------------------------------------
static const int SUM_BLOCKS = 1024;
int sum_partials_needed() { return SUM_BLOCKS; }

template <typename T>
__global__ __launch_bounds__(WG) void sum_stage1_kernel(const T *__restrict__ v,
                                                       int64_t n,
                                                       double *__restrict__ partials) {
  __shared__ double red[WG];
  const int tid = threadIdx.x;
  const int64_t per = (n + gridDim.x - 1) / gridDim.x;
  const int64_t lo = (int64_t)blockIdx.x * per;
  const int64_t hi = min(n, lo + per);
  double acc = 0;
  for (int64_t i = lo + tid; i < hi; i += WG) acc += (double)v[i];
  red[tid] = acc;
  __syncthreads();
  for (int off = WG / 2; off > 0; off >>= 1) {
    if (tid < off) red[tid] += red[tid + off];
    __syncthreads();
  }
  if (tid == 0) partials[blockIdx.x] = red[0];
}
__global__ __launch_bounds__(WG) void sum_stage2_kernel(const double *__restrict__ partials,
                                                       int np, double *__restrict__ out) {
  __shared__ double red[WG];
  const int tid = threadIdx.x;
  double acc = 0;
  for (int i = tid; i < np; i += WG) acc += partials[i];
  red[tid] = acc;
  __syncthreads();
  for (int off = WG / 2; off > 0; off >>= 1) {
    if (tid < off) red[tid] += red[tid + off];
    __syncthreads();
  }
  if (tid == 0) *out = red[0];
}

template <typename T>
int launch_sum(hipStream_t s, const T *v, int64_t n, double *partials,
               int n_partials, double *out) {
  int blocks = n_partials < SUM_BLOCKS ? n_partials : SUM_BLOCKS;
  if (blocks < 1) return H2O4GPU_KMEANS_EARG;
  hipLaunchKernelGGL((sum_stage1_kernel<T>), dim3(blocks), dim3(WG), 0, s, v, n, partials);
  hipLaunchKernelGGL(sum_stage2_kernel, dim3(1), dim3(WG), 0, s, partials, blocks, out);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

template <typename T>
__global__ void gather_rows_kernel(const T *__restrict__ X, const int *__restrict__ idx,
                                   T *__restrict__ C, int k, int d) {
  const int64_t e = (int64_t)blockIdx.x * WG + threadIdx.x;
  if (e >= (int64_t)k * d) return;
  const int c = (int)(e / d), j = (int)(e - (int64_t)c * d);
  C[e] = X[(int64_t)idx[c] * d + j];
}
template <typename T>
int launch_gather_rows(hipStream_t s, const T *X, const int *idx, T *C, int k, int d) {
  const int64_t kd = (int64_t)k * d;
  hipLaunchKernelGGL((gather_rows_kernel<T>), dim3((unsigned)((kd + WG - 1) / WG)),
                     dim3(WG), 0, s, X, idx, C, k, d);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

template int launch_bucketed_accumulate<float>(hipStream_t, const float *, const int *, int *, int *,
                                               int *, int *, int *, int *, double *, double *, int *,
                                               int64_t, int, int, const unsigned *);
template int launch_bucketed_accumulate<double>(hipStream_t, const double *, const int *, int *, int *,
                                                int *, int *, int *, int *, double *, double *, int *,
                                                int64_t, int, int, const unsigned *);

#define KM_INSTANTIATE(T)                                                            \
  template int launch_row_norms<T>(hipStream_t, const T *, T *, int64_t, int, int *);       \
  template UpdatePlan plan_update<T>(int64_t, int, int, int);                        \
  template int launch_finalize<T>(hipStream_t, int, const double *,                  \
                                  const int *, const T *, T *, int *, T *, int *,    \
                                  int, int, const int *, int, unsigned *, T *, T *, RunningSums, StopRule);                       \
  template int launch_post_update<T>(hipStream_t, const T *, T *, const T *, int,    \
                                     T *, int, int);                                 \
  template int launch_sum<T>(hipStream_t, const T *, int64_t, double *, int,         \
                             double *);                                              \
  template int launch_gather_rows<T>(hipStream_t, const T *, const int *, T *, int,  \
                                     int);
KM_INSTANTIATE(float)
KM_INSTANTIATE(double)

}  // namespace kmhip
