// Rows of three to eight float32 features against more than 16 centroids (pixels, coordinates).
//
// The row-stationary kernel of assign_kernels.hip pads such rows to eight features and spends
// four 64-cycle matrix instructions and 16 vector additions on a 32 x 32 tile of distances. Here
// the tile comes from three (up to four features) or four 32-cycle bfloat16 instructions: a float
// is the exact sum of three bfloat16 parts (bf16_parts.h), six products of parts make a product of
// floats to float32 accuracy, and with so few features the six products of all of them lie side by
// side in the 16-wide k-steps. A lane group holds NP pairs of features, group 0 the features
// 0 .. 2NP-1, group 1 the rest. A pair (a, b) packs into one register per part, and the k-steps are
//     one for each pair, its small products    m m  l l  h h  m m    (h, m, l: the parts of a and of b)
//                                       with   H H  H H  M M  M M    (parts of -2c)
//     lane group 0 h h of all pairs with L L, lane group 1 the parts of xx and cc against ones
//     lane group 0 h h of all pairs with H H, lane group 1 zeros
// The instruction adds the eight products of lane group 0, then those of group 1, and rounds after
// either at the size of the largest term (bf16_parts.h). The small products are thus summed at their own
// size, and a distance is rounded twice at the size of xx + cc, where the float32 instructions round
// once per feature and once for xx + cc. (Rms error of the minimum distances over the float32
// instructions': 0.73 to 0.93 in the mean, 1.06 at worst over forty sets of columns with scales and
// offsets of their own; 0.70 to 0.96 and 1.19 with the accumulators starting at cc and large and small
// products side by side. The small products last: 0.86 to 1.02.)
// Labels (16-ulp integer keys, lowest index on ties; near ties settled by the float32 instructions),
// minimum distances, -1 where nothing is below FLT_MAX: as in the row-stationary kernel. xx is summed from the row in feature order with
// separate multiply and add, the value row_norms stores, so the norm buffer is not read.
//
// FUSE: sums in LDS in double, [copy][centroid][4 NP + 1]: every lane adds the 2NP features it
// holds, lane group 0 counts the row in the last slot (a double counts exactly); lane l adds into
// copy l % ncopy, so that rows of one wavefront that share a centroid meet less often.
// Bound by the vector instructions per row (splitting, keys), not by memory. 10.1M rows, a fused step,
// against the row-stationary kernel on the float32 instructions: 3 features, k = 27 124 -> 98 us; 10M
// rows: 4, k = 100 285 -> 200; 5, k = 60 188 -> 151; 8, k = 100 293 -> 235 (85, 160, 136 and 206 without
// the second minimum that near ties are found by).
#include <algorithm>

#include "bf16_parts.h"
#include "kmeans_common.h"
#include "mfma_traits.h"

namespace kmhip {

namespace {

constexpr int SR_TPB = 1024;
constexpr int SR_NW = SR_TPB / 64;
constexpr int SR_MAX_D = 8;
constexpr size_t SR_LDS_MAX = 150 * 1024;
__host__ __device__ constexpr int sr_pairs(int d) { return d <= 4 ? 1 : 2; }
__host__ __device__ constexpr int sr_steps(int d) { return sr_pairs(d) + 1; }  // k-steps before the last

// row tiles a wavefront keeps in flight: as many as its 128 registers hold beside the work
__host__ __device__ constexpr int sr_ahead(int d) { return d <= 3 ? 8 : d == 4 ? 6 : d == 5 ? 4 : 2; }

size_t sr_model_lds(int d, int k) { return (size_t)((k + 31) / 32) * (sr_steps(d) * 64 + 32) * 16 + 16; }
size_t sr_sums_lds(int d, int k) { return (size_t)k * (4 * sr_pairs(d) + 1) * sizeof(double); }

template <int D, bool FUSE>
__global__ __launch_bounds__(SR_TPB) void assign_shortrow_kernel(
    const float *__restrict__ X, const float *__restrict__ C, int *__restrict__ labels,
    float *__restrict__ mindist, int64_t n, int k, double *__restrict__ psums, int *__restrict__ pcounts,
    int ncopy, TieBound bound) {
  constexpr int NP = sr_pairs(D), NM = sr_steps(D), NV = 2 * NP;
  constexpr int SD = 2 * NV + 1;  // doubles per centroid of the sums, the count last
  constexpr int MT = 32, NACC = 16, ROWT = 2;
  static_assert(D >= 1 && D <= 2 * NV && 2 * NP <= 4, "a lane group holds the leading parts of all pairs");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int KT = (k + MT - 1) / MT;
  uintx4 *cs = reinterpret_cast<uintx4 *>(smem_raw);                     // [KT][NM][64]
  uintx4 *lead = cs + (size_t)KT * NM * 64;                              // [KT][32] the last step, then zeros
  double *sums = reinterpret_cast<double *>(lead + (size_t)KT * 32 + 1);  // (FUSE) [ncopy][k][SD]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane % MT, g = lane / MT;
  if (FUSE)
    for (int e = tid; e < ncopy * k * SD; e += SR_TPB) sums[e] = 0.0;
  // the centroid side, one (tile, lane) per thread and turn
  for (int e = tid; e < KT * 64; e += SR_TPB) {
    const int t = e >> 6, l = e & 63, c = t * MT + l % MT, gg = l / MT;
    Bf16x3Pair s[2 * NP];
#pragma unroll
    for (int p = 0; p < 2 * NP; p++) {
      float v[2];
#pragma unroll
      for (int q = 0; q < 2; q++) v[q] = (c < k && 2 * p + q < D) ? -2.0f * C[(size_t)c * D + 2 * p + q] : 0.0f;
      s[p] = split_pair_bf16x3(v[0], v[1]);
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const unsigned h = gg == 0 ? s[p].h : s[NP + p].h, m = gg == 0 ? s[p].m : s[NP + p].m;
      const uintx4 q = {h, h, m, m};
      cs[(size_t)(t * NM + p) * 64 + l] = q;
    }
    uintx4 q = {0u, 0u, 0u, 0u}, last = q;
    if (gg == 0) {
#pragma unroll
      for (int p = 0; p < 2 * NP; p++) {
        q[p] = s[p].l;
        last[p] = s[p].h;
      }
      lead[c] = last;
    } else {  // (a padding centroid is infinitely far)
      const Bf16x3 n = split_norm_bf16x3(c < k ? row_sqnorm<float>(C + (size_t)c * D, D) : pos_inf<float>());
      q[0] = n.h | (n.m << 16);
      q[1] = n.l | (0x3F80u << 16);
      q[2] = 0x3F803F80u;
    }
    cs[(size_t)(t * NM + NP) * 64 + l] = q;
  }
  if (tid == 0) {
    const uintx4 zero = {0u, 0u, 0u, 0u};
    lead[KT * 32] = zero;
  }
  __syncthreads();

  double *const my_sums = sums + (size_t)(lane & (ncopy - 1)) * k * SD;
  // PF row tiles are under way while two are worked on: with two in flight per wavefront the
  // kernel waited for memory (three features: 1.6 TB/s).
  constexpr int PF = sr_ahead(D);
  float xn[PF][D];
  // rows past the end re-read the last one; their results are never stored
  auto fetch = [&](float (&x)[D], int64_t row0) {
    const float *src = X + min(row0 + r, n - 1) * D;
#pragma unroll
    for (int j = 0; j < D; j++) x[j] = src[j];
  };
  const uintx4 *const my_lead = g == 0 ? lead + r : lead + KT * 32;
  const int lead_step = g == 0 ? 32 : 0;
  auto work = [&](const float (&xr)[ROWT][D], int64_t row0) {
    float val[ROWT][NV];  // what this lane group holds of the row
    float nrm[ROWT];
    uintx4 b[ROWT][NM];  // (the last step has the row side of the one before)
#pragma unroll
    for (int rt = 0; rt < ROWT; rt++) {
      float x[4 * NP];
#pragma unroll
      for (int j = 0; j < 4 * NP; j++) x[j] = j < D ? xr[rt][j] : 0.0f;
      float xx;
      {
#pragma clang fp contract(off)
        xx = 0;
#pragma unroll
        for (int j = 0; j < D; j++) xx = xx + x[j] * x[j];
      }
      nrm[rt] = xx;
#pragma unroll
      for (int q = 0; q < NV; q++) val[rt][q] = g == 0 ? x[q] : x[NV + q];
      uintx4 lastq = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int p = 0; p < NP; p++) {
        const Bf16x3Pair s = split_pair_bf16x3(val[rt][2 * p], val[rt][2 * p + 1]);
        const uintx4 q = {s.m, s.l, s.h, s.m};
        b[rt][p] = q;
        lastq[p] = s.h;
        lastq[NP + p] = cvt_pk_bf16(x[NV + 2 * p], x[NV + 2 * p + 1]);
      }
      const Bf16x3 xp = split_norm_bf16x3(xx);
      lastq[0] = g == 0 ? lastq[0] : 0x3F803F80u;
      lastq[1] = g == 0 ? lastq[1] : 0x3F80u | (xp.h << 16);
      lastq[2] = g == 0 ? lastq[2] : xp.m | (xp.l << 16);
      lastq[3] = g == 0 ? lastq[3] : 0u;
      b[rt][NP] = lastq;
    }
    unsigned bkey[ROWT], skey[ROWT];
    int btile[ROWT];
#pragma unroll
    for (int rt = 0; rt < ROWT; rt++) {
      bkey[rt] = skey[rt] = 0x7F7FFFF0u;  // FLT_MAX with the index bits cleared
      btile[rt] = -1;
    }
    for (int t = 0; t < KT; t++) {
      uintx4 a[NM];
#pragma unroll
      for (int m = 0; m < NM; m++) a[m] = cs[(size_t)(t * NM + m) * 64 + lane];
      const uintx4 al = my_lead[t * lead_step];
#pragma unroll
      for (int rt = 0; rt < ROWT; rt++) {
        floatx16 acc;
#pragma unroll
        for (int v = 0; v < NACC; v++) acc[v] = 0;
#pragma unroll
        for (int m = 0; m < NM; m++) acc = mma_bf16(a[m], b[rt][m], acc);
        acc = mma_bf16(al, b[rt][NP], acc);
        unsigned key[NACC];
#pragma unroll
        for (int v = 0; v < NACC; v++) key[v] = (__float_as_uint(acc[v]) & 0x7FFFFFF0u) | (unsigned)v;
        const unsigned m = two_smallest_keys(key, bkey[rt], skey[rt]);
        if ((m | 15u) < bkey[rt]) {
          bkey[rt] = m;
          btile[rt] = t;
        }
      }
    }
#pragma unroll
    for (int rt = 0; rt < ROWT; rt++) {
      float best = __uint_as_float(bkey[rt] & 0xFFFFFFF0u);
      int bidx = btile[rt] < 0 ? -1 : btile[rt] * MT + key_row(bkey[rt] & 15u, g);
      const float ob = __shfl_xor(best, MT, 64);
      const float second = fminf(fmaxf(best, ob), __uint_as_float(skey[rt] & 0xFFFFFFF0u));
      argmin_merge(best, bidx, ob, __shfl_xor(bidx, MT, 64));
      // Near ties, settled as the float32 instructions settle them (assign_rowstat_kernel): a tile with
      // such a row is swept again by them, with the operands the row-stationary kernel gives them
      // (lane group 0 the features 0 to 3, group 1 the rest).
      unsigned long long ties = __ballot(near_tie(best, second, nrm[rt], bound));
      if (ties != 0) ties &= __ballot(nrm[rt] <= argmin_start<float>());  // (no distance to settle)
      if (__builtin_expect(ties != 0, 0)) {
        const bool tie = (((ties | ties >> 32) >> r) & 1) != 0;
        unsigned fkey = 0x7F7FFFF0u;
        int ftile = -1;
#pragma unroll 1
        for (int t = 0; t < KT; t++) {
          floatx16 acc;
#pragma unroll
          for (int v = 0; v < NACC; v++) {
            const uintx4 p = cs[(size_t)(t * NM + NP) * 64 + MT + Mfma<float>::acc_row(v, g)];
            acc[v] = nrm[rt] + ((bf16_low(p[0]) + bf16_high(p[0])) + bf16_low(p[1]));
          }
#pragma unroll
          for (int e = 0; e < 4; e++) {
            // feature 4 g + e of this lane's centroid, from the words of its three parts
            auto word = [&](int step, int at, int w) {
              const unsigned u = reinterpret_cast<const unsigned *>(cs + (size_t)(t * NM + step) * 64 + at)[w];
              return e % 2 ? bf16_high(u) : bf16_low(u);
            };
            const int own = NP == 2 ? lane : r + e / 2 * MT, step = NP == 2 ? e / 2 : 0;
            float a = (word(step, own, 0) + word(step, own, 2)) + word(NP, r, NP == 2 ? 2 * g + e / 2 : e / 2);
            float b = NP == 2 ? val[rt][e % NV] : (e < D ? xr[rt][e < D ? e : 0] : 0.0f);
            if (NP == 1 && g == 1) a = b = 0.0f;
            acc = Mfma<float>::mma(a, b, acc);
          }
          unsigned key[NACC];
#pragma unroll
          for (int v = 0; v < NACC; v++) key[v] = (__float_as_uint(acc[v]) & 0x7FFFFFF0u) | (unsigned)v;
          unsigned m = umin3(key[0], key[1], key[2]);
#pragma unroll
          for (int v = 3; v + 1 < NACC; v += 2) m = umin3(m, key[v], key[v + 1]);
          m = min(m, key[NACC - 1]);
          if ((m | 15u) < fkey) {
            fkey = m;
            ftile = t;
          }
        }
        float fbest = __uint_as_float(fkey & 0xFFFFFFF0u);
        int fidx = ftile < 0 ? -1 : ftile * MT + key_row(fkey & 15u, g);
        argmin_merge(fbest, fidx, __shfl_xor(fbest, MT, 64), __shfl_xor(fidx, MT, 64));
        if (tie) {
          best = fbest;
          bidx = fidx;
        }
      }
      const int64_t row = row0 + rt * MT + r;
      if (g == 0 && row < n) {
        labels[row] = bidx;
        if (mindist) mindist[row] = best;
      }
      if (FUSE && row < n && bidx >= 0) {
        double *srow = my_sums + (size_t)bidx * SD;
#pragma unroll
        for (int q = 0; q < NV; q++) {
          // (a slot that no feature fills in either lane group is left out)
          if (q < D) unsafeAtomicAdd(srow + g * NV + q, (double)val[rt][q]);
        }
        if (g == 0) unsafeAtomicAdd(srow + SD - 1, 1.0);
      }
    }
  };
  constexpr int ROWS = PF * MT;
  const int64_t stride = (int64_t)gridDim.x * SR_NW * ROWS;
  const int64_t first = ((int64_t)wave * gridDim.x + blockIdx.x) * ROWS;
  if (first < n) {
#pragma unroll
    for (int rt = 0; rt < PF; rt++) fetch(xn[rt], first + rt * MT);
  }
  for (int64_t row0 = first; row0 < n; row0 += stride) {
#pragma unroll
    for (int p = 0; p < PF; p += ROWT) {
      float x[ROWT][D];
#pragma unroll
      for (int rt = 0; rt < ROWT; rt++) {
#pragma unroll
        for (int j = 0; j < D; j++) x[rt][j] = xn[p + rt][j];
        fetch(xn[p + rt], row0 + stride + (p + rt) * MT);
      }
      if (row0 + p * MT < n) work(x, row0 + p * MT);
    }
  }
  if (!FUSE) return;
  __syncthreads();
  double *dst = psums + (size_t)blockIdx.x * k * D;
  for (int e = tid; e < k * SD; e += SR_TPB) {
    const int c = e / SD, f = e - c * SD;
    double v = 0;
    for (int cp = 0; cp < ncopy; cp++) v += sums[(size_t)cp * k * SD + e];  // copy order
    if (f < D) dst[(size_t)c * D + f] = v;
    else if (f == SD - 1) pcounts[(size_t)blockIdx.x * k + c] = (int)v;
  }
}

}  // namespace

// One or two features stay with the float32 instructions, whose two or three roundings per
// distance are hard to beat. Up to four features every model of more
// than 16 centroids is ahead (2M x 4, k = 17: 32.9 -> 29.8 us a fused step, k = 100: 66 -> 44); five to eight from
// about 48 (2M x 8, k = 40: 42.5 -> 43.3, k = 65: 54 -> 47, k = 100: 66 -> 53).
bool shortrow_applies(int d, int k, bool fused) {
  return d >= 3 && d <= SR_MAX_D && k > (d <= 4 ? 16 : 48) &&
         sr_model_lds(d, k) + (fused ? sr_sums_lds(d, k) : 0) <= SR_LDS_MAX;
}

int launch_shortrow(hipStream_t s, const float *X, const float *C, int *labels, float *mindist, int64_t n, int d,
                    int k, int num_cu, bool fused, double *psums, int *pcounts, int *slots, bool settle) {
  const TieBound bound = settle_margin(d, settle);
  if (!shortrow_applies(d, k, fused)) return H2O4GPU_KMEANS_EARG;
  // copies of the sums: what fits beside the model in half a CU's LDS, eight at most (one is
  // always there)
  int ncopy = 1;
  const size_t model = sr_model_lds(d, k), sums = sr_sums_lds(d, k);
  while (fused && ncopy < 8 && model + 2 * ncopy * sums <= 72 * 1024) ncopy *= 2;
  const size_t lds = model + (fused ? ncopy * sums : 0);
  const int rows_per_wave = sr_ahead(d) * 32;
  const int64_t tiles = (n + rows_per_wave - 1) / rows_per_wave;
  int grid = 1;
#define KM_SR_X(D, FUSE)                                                                                   \
  do {                                                                                                     \
    auto kern = assign_shortrow_kernel<D, FUSE>;                                                           \
    KM_TRY(ensure_dynamic_lds(reinterpret_cast<const void *>(kern), lds));                                 \
    const int per_cu = std::min(2, resident_blocks_per_cu(reinterpret_cast<const void *>(kern), SR_TPB, lds)); \
    grid = (int)std::min<int64_t>((int64_t)num_cu * per_cu, tiles);                                        \
    hipLaunchKernelGGL(kern, dim3(grid), dim3(SR_TPB), lds, s, X, C, labels, mindist, n, k, psums, pcounts, ncopy, \
                       bound);                                                                             \
  } while (0)
#define KM_SR(D)                    \
  case D:                           \
    if (fused) KM_SR_X(D, true);    \
    else KM_SR_X(D, false);         \
    break
  switch (d) {
    KM_SR(3);
    KM_SR(4);
    KM_SR(5);
    KM_SR(6);
    KM_SR(7);
    KM_SR(8);
  }
#undef KM_SR
#undef KM_SR_X
  KM_HIP_TRY(hipGetLastError());
  if (slots) *slots = grid;
  return 0;
}

}  // namespace kmhip
