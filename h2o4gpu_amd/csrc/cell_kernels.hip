// Lloyd steps over rows of three float32 features that have been ordered in space once.
//
// A step over such rows (pixels, coordinates) is a few instructions per row and centroid, and a fit that
// runs until its centroids stand still makes hundreds of steps over the same rows. After the first steps
// the rows are therefore copied in the order of a space-filling curve (Morton order of a 64^3 grid
// over their range; empty space costs nothing, what is cut is the ordered rows) and cut into blocks of 64, of
// which the box and the sums are kept. A step then asks per block which centroids can be the nearest of a
// row in its box: |x - a|^2 - |x - b|^2 is linear in x, so its largest value over a box is at a corner. Where
// a single centroid is left the block's sums are added at once; otherwise its rows are measured
// against those left only. Labels are not stored: the pass over all rows that ends a fit makes them.
//
// Centroids are those of steps that measure every row, bit for bit: a row's label is that of the chain of
// multiply-adds the float32 instructions make (compared at 16 ulp, lowest index first), a centroid is
// ruled out only where it is further by more than any rounding of that chain, and sums of float32 values in
// double do not depend on their order where they are exact (colours, coordinates of less than some 14 binades; others
// differ by some 2^-50 of the largest value, as two orders do. Each step makes its sums from the blocks'.)
//
// Bound by latency and by the additions in LDS: a block's test reads 64 bytes and takes some 20 instructions per
// centroid, an undecided block's rows (a third of them with k = 27) are measured against two to four centroids.
// A step, 10M rows: k = 27 84 -> 18 us on pixels, k = 60 110 -> 38 on blobs; putting the rows in order 0.65 ms, of which
// 0.28 each for the sort and for the windows. (Rows of four features had fewer blocks decided: 1.3 to 1.7 times as
// fast on blobs, 0.6 to 1.1 on noise; models of 300 centroids 1.1 and 0.8. Rows
// of two features and float64 rows have not been tried.)
#include <algorithm>

#include "bf16_parts.h"
#include "kmeans_common.h"
#include "mfma_traits.h"

namespace kmhip {

namespace {

constexpr int CELL_WG = 1024;
constexpr int CELL_NW = CELL_WG / 64;
constexpr int CELL_WINDOW = 4096;      // rows put in order by one workgroup
constexpr int CELL_RANGE_GROUPS = 256;
constexpr int CELL_CAND = 14;          // centroids a block's rows are measured against; more: against all
constexpr int CELL_MAX_K = 128;

constexpr int CELL_BITS = 6;           // per feature of the finest grid; the two lowest are left to the windows

// [group][2][4]: smallest and largest finite values of the features
template <int D>
__global__ __launch_bounds__(256) void cell_range_kernel(const float *__restrict__ X, int64_t n,
                                                        float *__restrict__ range) {
  __shared__ float red[2][4][4];
  float lo[D], hi[D];
#pragma unroll
  for (int f = 0; f < D; f++) {
    lo[f] = pos_inf<float>();
    hi[f] = -pos_inf<float>();
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
#pragma unroll
    for (int f = 0; f < D; f++) {
      const float v = X[i * D + f];
      if (fabsf(v) <= argmin_start<float>()) {
        lo[f] = fminf(lo[f], v);
        hi[f] = fmaxf(hi[f], v);
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int f = 0; f < D; f++) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      lo[f] = fminf(lo[f], __shfl_xor(lo[f], off, 64));
      hi[f] = fmaxf(hi[f], __shfl_xor(hi[f], off, 64));
    }
    if (lane == 0) {
      red[0][f][wave] = lo[f];
      red[1][f][wave] = hi[f];
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int f = threadIdx.x;
    float l = red[0][f][0], h = red[1][f][0];
    for (int w = 1; w < 4; w++) {
      l = fminf(l, red[0][f][w]);
      h = fmaxf(h, red[1][f][w]);
    }
    range[blockIdx.x * 8 + f] = l;
    range[blockIdx.x * 8 + 4 + f] = h;
  }
}

// The whole range from the groups' (all threads of a workgroup of 256 or more): first values and steps per unit.
template <int D>
__device__ __forceinline__ void cell_grid(const float *__restrict__ range, float (&first)[D], float (&per_unit)[D]) {
  __shared__ float red[2][4][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  static_assert(CELL_RANGE_GROUPS == 256, "a group per thread of the first four wavefronts");
  if (tid < CELL_RANGE_GROUPS) {
#pragma unroll
    for (int f = 0; f < D; f++) {
      float l = range[tid * 8 + f], h = range[tid * 8 + 4 + f];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        l = fminf(l, __shfl_xor(l, off, 64));
        h = fmaxf(h, __shfl_xor(h, off, 64));
      }
      if (lane == 0) {
        red[0][f][wave] = l;
        red[1][f][wave] = h;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int f = 0; f < D; f++) {
    const float l = fminf(fminf(red[0][f][0], red[0][f][1]), fminf(red[0][f][2], red[0][f][3]));
    const float h = fmaxf(fmaxf(red[1][f][0], red[1][f][1]), fmaxf(red[1][f][2], red[1][f][3]));
    first[f] = l;
    // (an empty or endless range has one cell)
    per_unit[f] = h > l && h - l < 3e38f ? (float)(1 << CELL_BITS) / (h - l) : 0.0f;
  }
}

// The cell's place on the curve. (A NaN is in the first cell of its feature.)
template <int D>
__device__ __forceinline__ unsigned cell_code(const float (&x)[D], const float (&first)[D], const float (&per_unit)[D]) {
  constexpr int B = CELL_BITS;
  unsigned code = 0;
#pragma unroll
  for (int f = 0; f < D; f++) {
    const unsigned q = (unsigned)fminf(fmaxf((x[f] - first[f]) * per_unit[f], 0.0f), (float)((1 << B) - 1));
#pragma unroll
    for (int b = 0; b < B; b++) code |= ((q >> b) & 1u) << (b * D + f);
  }
  return code;
}

template <int D>
__global__ __launch_bounds__(256) void cell_ids_kernel(const float *__restrict__ X, int64_t n,
                                                      const float *__restrict__ range, int *__restrict__ ids) {
  float first[D], per_unit[D];
  cell_grid<D>(range, first, per_unit);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    float x[D];
#pragma unroll
    for (int f = 0; f < D; f++) x[f] = X[i * D + f];
    ids[i] = (int)(cell_code<D>(x, first, per_unit) >> (2 * D));
  }
}

// A workgroup puts CELL_WINDOW rows of neighbouring cells in order of their finest cells (a counting sort in
// LDS; rows of one cell come in any order) and leaves their blocks' boxes and sums.
template <int D>
__global__ __launch_bounds__(CELL_WG) void cell_windows_kernel(const float *__restrict__ X, int64_t n,
                                                              const float *__restrict__ range,
                                                              const int *__restrict__ order, float *__restrict__ Xs,
                                                              CellBlock *__restrict__ blocks) {
  constexpr int SUB = 1 << (2 * D), BINS = CELL_WINDOW, PER = CELL_WINDOW / CELL_WG;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned *bin = reinterpret_cast<unsigned *>(smem_raw);  // [BINS]
  float *rows = reinterpret_cast<float *>(bin + BINS);     // [CELL_WINDOW][D]
  __shared__ unsigned first_cell, last_cell, wave_sum[CELL_NW];
  float first[D], per_unit[D];
  cell_grid<D>(range, first, per_unit);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t p0 = (int64_t)blockIdx.x * CELL_WINDOW;
  const int cnt = (int)min((int64_t)CELL_WINDOW, n - p0);
  float x[PER][D];
  unsigned code[PER], rank[PER];
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const int i = e * CELL_WG + tid;
    const float *src = X + (int64_t)order[p0 + min(i, cnt - 1)] * D;
#pragma unroll
    for (int f = 0; f < D; f++) x[e][f] = src[f];
    code[e] = cell_code<D>(x[e], first, per_unit);
    bin[i] = 0;
    // (the rows come in order of their coarse cells)
    if (i == 0) first_cell = code[e] / SUB;
    if (i == cnt - 1) last_cell = code[e] / SUB;
  }
  __syncthreads();
  int shift = 0;  // (a window of many thinly filled cells: neighbouring ones share bins)
  while (((last_cell - first_cell) >> shift) >= (unsigned)(BINS / SUB)) shift++;
#pragma unroll
  for (int e = 0; e < PER; e++) {
    code[e] = ((code[e] / SUB - first_cell) >> shift) * SUB + code[e] % SUB;
    if (e * CELL_WG + tid < cnt) rank[e] = atomicAdd(&bin[code[e]], 1u);
  }
  __syncthreads();
  // bins -> their first places
  unsigned mine[PER], sum = 0;
#pragma unroll
  for (int e = 0; e < PER; e++) {
    mine[e] = bin[tid * PER + e];
    sum += mine[e];
  }
  unsigned before = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned o = __shfl_up(before, off, 64);
    if (lane >= off) before += o;
  }
  if (lane == 63) wave_sum[wave] = before;
  before -= sum;
  __syncthreads();
  for (int w = 0; w < wave; w++) before += wave_sum[w];
#pragma unroll
  for (int e = 0; e < PER; e++) {
    bin[tid * PER + e] = before;
    before += mine[e];
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < PER; e++) {
    if (e * CELL_WG + tid < cnt) {
      const unsigned at = bin[code[e]] + rank[e];
#pragma unroll
      for (int f = 0; f < D; f++) rows[at * D + f] = x[e][f];
    }
  }
  __syncthreads();
  for (int i = tid; i < cnt * D; i += CELL_WG) Xs[p0 * D + i] = rows[i];
  for (int b = wave; b * 64 < cnt; b += CELL_NW) {
    const int i = b * 64 + lane;
    const bool valid = i < cnt;
    const int at = valid ? i : 0;
    float lo[D], hi[D];
    double sum[D];
    bool finite = true;
#pragma unroll
    for (int f = 0; f < D; f++) {
      const float v = rows[at * D + f];
      lo[f] = valid ? v : pos_inf<float>();
      hi[f] = valid ? v : -pos_inf<float>();
      sum[f] = valid ? (double)v : 0.0;
      finite &= !valid || fabsf(v) <= argmin_start<float>();
    }
    const bool all_finite = __ballot(finite) == ~0ull;
#pragma unroll
    for (int f = 0; f < D; f++) {
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        lo[f] = fminf(lo[f], __shfl_xor(lo[f], off, 64));
        hi[f] = fmaxf(hi[f], __shfl_xor(hi[f], off, 64));
        sum[f] += __shfl_xor(sum[f], off, 64);
      }
    }
    if (lane == 0) {
      CellBlock out;
#pragma unroll
      for (int f = 0; f < 4; f++) {
        // (a row that is not finite: a box that rules nothing out)
        out.lo[f] = f < D ? (all_finite ? lo[f < D ? f : 0] : -pos_inf<float>()) : 0.0f;
        out.hi[f] = f < D ? (all_finite ? hi[f < D ? f : 0] : pos_inf<float>()) : 0.0f;
        out.sum[f] = f < D ? sum[f < D ? f : 0] : 0.0;
      }
      blocks[p0 / 64 + b] = out;
    }
  }
}

// Doubles from one copy of the sums to the next: odd, so that the copies of a sum lie in different banks (10M x 3,
// k = 60, with 240: 85 -> 38 us).
__host__ __device__ inline int cell_copy_stride(int d, int k) { return (k * (d + 1)) | 1; }

size_t cell_step_lds(int d, int k, int ncopy) {
  return (size_t)k * 5 * sizeof(float) + 8 + (size_t)ncopy * cell_copy_stride(d, k) * sizeof(double) +
         (size_t)CELL_WG * (CELL_CAND + 2) * sizeof(uint16_t);
}

template <int D>
__global__ __launch_bounds__(CELL_WG) void cell_step_kernel(const float *__restrict__ Xs,
                                                           const CellBlock *__restrict__ blocks, int64_t n,
                                                           const float *__restrict__ C, int k,
                                                           double *__restrict__ psums, int *__restrict__ pcounts,
                                                           int ncopy, unsigned long long *__restrict__ measured,
                                                           const unsigned *__restrict__ stopped) {
  if (stopped != nullptr && *stopped != 0) return;
  constexpr int SD = D + 1;
  const int stride = cell_copy_stride(D, k);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  floatx4 *cen = reinterpret_cast<floatx4 *>(smem_raw);                      // [k]
  double *sums = reinterpret_cast<double *>(cen + k);                        // [ncopy][k][SD], the count last
  uint16_t(*cand)[CELL_CAND + 2] = reinterpret_cast<uint16_t(*)[CELL_CAND + 2]>(sums + (size_t)ncopy * stride);  // [CELL_WG]
  float *cc = reinterpret_cast<float *>(cand + CELL_WG);                     // [k]
  __shared__ int listed;
  __shared__ unsigned long long work;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < ncopy * stride; e += CELL_WG) sums[e] = 0.0;
  for (int c = tid; c < k; c += CELL_WG) {
    floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int f = 0; f < D; f++) v[f] = C[(size_t)c * D + f];
    cen[c] = v;
    cc[c] = row_sqnorm<float>(C + (size_t)c * D, D);
  }
  double *const my_sums = sums + (size_t)(lane & (ncopy - 1)) * stride;
  const int64_t nblocks = (n + 63) / 64;
  if (tid == 0) work = 0;
  // (neighbouring blocks go to different workgroups: undecided ones lie side by side)
  for (int64_t b0 = blockIdx.x; b0 < nblocks; b0 += (int64_t)gridDim.x * CELL_WG) {
    if (tid == 0) listed = 0;
    __syncthreads();
    const int64_t blk = b0 + (int64_t)tid * gridDim.x;
    if (blk < nblocks) {
      const CellBlock box = blocks[blk];
      float m[D], h[D], r2 = 0;
#pragma unroll
      for (int f = 0; f < D; f++) {
        m[f] = 0.5f * box.lo[f] + 0.5f * box.hi[f];
        h[f] = fmaxf(box.hi[f] - m[f], m[f] - box.lo[f]) * 2.000001f;
        r2 += fmaxf(box.lo[f] * box.lo[f], box.hi[f] * box.hi[f]);
      }
      int a = 0;
      float near = pos_inf<float>();
      for (int c = 0; c < k; c++) {
        const floatx4 v = cen[c];
        float t = cc[c];
#pragma unroll
        for (int f = 0; f < D; f++) t -= 2.0f * m[f] * v[f];
        if (t < near) {
          near = t;
          a = c;
        }
      }
      const floatx4 va = cen[a];
      const float cca = cc[a];
      // A row's distance to a centroid is rounded by less than (D + 4) 2^-24 (xx + cc) and compared at
      // 1.9e-6 of it, and is at most 2 (xx + cc): 1.2e-5 (xx + cc_a + cc_b) is twice what two of them, their
      // comparison and this test can be off by.
      int others = 0;
      for (int c = 0; c < k; c++) {
        const floatx4 v = cen[c];
        const float ccc = cc[c];
        float t = cca - ccc;
#pragma unroll
        for (int f = 0; f < D; f++) {
          const float e = va[f] - v[f];
          t += h[f] * fabsf(e) - 2.0f * m[f] * e;
        }
        if (!(t < -1.2e-5f * (r2 + cca + ccc)) && c != a) {
          if (others < CELL_CAND - 1) cand[tid][3 + others] = (uint16_t)c;
          others++;
        }
      }
      if (others == 0) {
        double *s = my_sums + (size_t)a * SD;
#pragma unroll
        for (int f = 0; f < D; f++) unsafeAtomicAdd(s + f, box.sum[f]);
        unsafeAtomicAdd(s + D, (double)min((int64_t)64, n - blk * 64));
      } else {
        cand[tid][1] = (uint16_t)(others < CELL_CAND ? others + 1 : 0);  // (0: all)
        cand[tid][2] = (uint16_t)a;
        cand[atomicAdd(&listed, 1)][0] = (uint16_t)tid;
      }
    }
    __syncthreads();
    const int cnt = listed;
    float ahead[D];  // the next block's row is on its way while one is worked on
    auto fetch = [&](int e) {
      const int t = __builtin_amdgcn_readfirstlane((int)cand[min(e, cnt - 1)][0]);
      const float *src = Xs + min((b0 + (int64_t)t * gridDim.x) * 64 + lane, n - 1) * D;
#pragma unroll
      for (int f = 0; f < D; f++) ahead[f] = src[f];
    };
    if (wave < cnt) fetch(wave);
    for (int e = wave; e < cnt; e += CELL_NW) {
      const int t = __builtin_amdgcn_readfirstlane((int)cand[e][0]);
      const int nc = __builtin_amdgcn_readfirstlane((int)cand[t][1]);
      const int64_t row = (b0 + (int64_t)t * gridDim.x) * 64 + lane;
      float x[D], xx = 0;
#pragma unroll
      for (int f = 0; f < D; f++) x[f] = ahead[f];
      fetch(e + CELL_NW);
      {
#pragma clang fp contract(off)
#pragma unroll
        for (int f = 0; f < D; f++) xx = xx + x[f] * x[f];
      }
      unsigned best = 0x7F7FFFF0u;  // FLT_MAX with the compared bits only
      int bidx = -1;
      auto measure = [&](int c) {
        const floatx4 v = cen[c];
        float acc = xx + cc[c];
#pragma unroll
        for (int f = 0; f < D; f++) acc = fmaf(-2.0f * v[f], x[f], acc);
        const unsigned key = __float_as_uint(acc) & 0x7FFFFFF0u;
        if (key < best || (key == best && (unsigned)c < (unsigned)bidx && bidx >= 0)) {
          best = key;
          bidx = c;
        }
      };
      if (nc > 0) {
        for (int q = 0; q < nc; q++) measure(cand[t][2 + q]);
      } else {
        for (int c = 0; c < k; c++) measure(c);
      }
      if (measured != nullptr && lane == 0) atomicAdd(&work, (unsigned long long)(nc > 0 ? nc : k));
      if (row < n && bidx >= 0) {
        double *s = my_sums + (size_t)bidx * SD;
#pragma unroll
        for (int f = 0; f < D; f++) unsafeAtomicAdd(s + f, (double)x[f]);
        unsafeAtomicAdd(s + D, 1.0);
      }
    }
    __syncthreads();
  }
  if (measured != nullptr && tid == 0 && work > 0) atomicAdd(measured, work);  // (past the loop's last barrier)
  double *dst = psums + (size_t)blockIdx.x * k * D;
  for (int e = tid; e < k * SD; e += CELL_WG) {
    const int c = e / SD, f = e - c * SD;
    double v = 0;
    for (int cp = 0; cp < ncopy; cp++) v += sums[(size_t)cp * stride + e];  // copy order
    if (f < D) dst[(size_t)c * D + f] = v;
    else pcounts[(size_t)blockIdx.x * k + c] = (int)v;
  }
}

}  // namespace

bool cells_apply(int64_t n, int d, int k) {
  return d == 3 && k >= 2 && k <= CELL_MAX_K && n >= 1 && n <= 2147483647 && shortrow_applies(d, k, true);
}
int64_t cell_blocks(int64_t n) { return (n + 63) / 64; }
int cell_range_values() { return CELL_RANGE_GROUPS * 8; }

int launch_cell_ids(hipStream_t s, const float *X, int64_t n, int d, float *range, int *ids) {
  if (n < 1 || d != 3) return H2O4GPU_KMEANS_EARG;
  const int grid = (int)std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(cell_range_kernel<3>, dim3(CELL_RANGE_GROUPS), dim3(256), 0, s, X, n, range);
  hipLaunchKernelGGL(cell_ids_kernel<3>, dim3(grid), dim3(256), 0, s, X, n, range, ids);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

int launch_cell_windows(hipStream_t s, const float *X, int64_t n, int d, const float *range, const int *order,
                        float *Xs, CellBlock *blocks) {
  if (n < 1 || d != 3) return H2O4GPU_KMEANS_EARG;
  const unsigned grid = (unsigned)((n + CELL_WINDOW - 1) / CELL_WINDOW);
  const size_t lds = (size_t)CELL_WINDOW * (sizeof(unsigned) + d * sizeof(float));
  KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(cell_windows_kernel<3>), lds));
  hipLaunchKernelGGL(cell_windows_kernel<3>, dim3(grid), dim3(CELL_WG), lds, s, X, n, range, order, Xs, blocks);
  KM_HIP_TRY(hipGetLastError());
  return 0;
}

int launch_cell_step(hipStream_t s, const float *Xs, const CellBlock *blocks, int64_t n, const float *C, int d, int k,
                     int num_cu, double *psums, int *pcounts, int *slots, unsigned long long *measured,
                     const unsigned *stopped) {
  if (!cells_apply(n, d, k)) return H2O4GPU_KMEANS_EARG;
  // copies of the sums: what fits beside a second workgroup's
  int ncopy = 1;
  while (ncopy < 16 && cell_step_lds(d, k, 2 * ncopy) <= 72 * 1024) ncopy *= 2;
  const size_t lds = cell_step_lds(d, k, ncopy);
  const int grid = (int)std::min<int64_t>(2 * num_cu, cell_blocks(n));
  KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(cell_step_kernel<3>), lds));
  hipLaunchKernelGGL(cell_step_kernel<3>, dim3(grid), dim3(CELL_WG), lds, s, Xs, blocks, n, C, k, psums, pcounts, ncopy,
                     measured, stopped);
  KM_HIP_TRY(hipGetLastError());
  *slots = grid;
  return 0;
}

}  // namespace kmhip
