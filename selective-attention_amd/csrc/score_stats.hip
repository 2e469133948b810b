// Per-head statistics of the valid attention scores, for SelectiveMHA's
// training forward: the count, sum and sum of squares of
//   s_ij = scale * q_i . k_j
// over the valid (query i, key j) pairs of every batch row -- i inside the
// row's query length, j inside its key length and, for causal attention,
// j <= i.  The score matrix is never written: each tile of scores is reduced
// where the MFMA leaves it.
//
// Replaces the dense reductions of modules/selective_attention.py:234-246
// (self attention: query and key lengths both the row's length) and
// modules/cross_selective_attention.py:129-146 (cross attention: every
// query, keys inside the context length): valid mask, masked_fill,
// sum / square().sum() over batch, queries and keys.  The std and the
// running average stay with the caller.
//
// score_stats_kernel: one block per (batch row, head, 64-query block); wave
// w owns queries 16 w .. 16 w + 15 of the block.  Per 16-key tile, the K rows
// are the MFMA A operand and the wave's queries (kept in registers) the B
// operand, so a lane holds 4 keys of its own query.  fp32 inputs are split
// into bf16 hi + lo (products hi*hi + lo*hi + hi*lo).  Per-lane tile sums
// are fp32, running sums fp64; each block writes (count, sum, sum^2) and
// score_stats_reduce sums those in a fixed order (deterministic).
//
// The moments without the pairs (sa_score_moments, sa_score_std_bwd).  The
// scores are bilinear, so over a set of keys with M = sum k k^T and
// kappa = sum k the sum of a query's scores is scale q . kappa and the sum of
// their squares scale^2 q . M q; the gradient of the std,
//   g_ij = coef (s_ij - mean),   dq_i = scale sum_j g_ij k_j,
// is scale coef (scale M q_i - mean kappa), and dk_j the same over the queries.
// Causal attention needs M over the keys before each query: Gram matrices
// of 256-row chunks (score_gram_kernel), their exclusive prefix (suffix for
// dk) over the chunks (score_gram_scan_kernel), and in score_apply_kernel
// the chunk's own pairs as 64x64 score tiles.  Work per row: 4 D^2 FLOP for
// the Gram matrix and its product and 160 pairs on average, against L / 2
// pairs.
// Precision.  q . M q and scale M q - mean kappa cancel where rows share a
// component, as sum^2 / n - mean^2 does, so everything that stands for a sum over
// pairs is fp64: the Gram matrices (exact products of fp32 values on
// v_mfma_f64_16x16x4_f64), their scan, the products with them, and the sums over
// the scores and over a chunk's tiles.  fp32 is the score of one pair and a
// gradient's sum over one 64-row tile.  The std's error is that of its rounding
// (at most 5e-8, also with common parts of 100 standard deviations), the
// gradients' at most 6e-8 without a common part and below the dense fp32 form's
// with one (q and k offset by 10: 5e-8 for 3e-7; k by 100, across q: 6e-7 for
// 1.2e-6).  With fp32 Gram matrices the std was off by 1.5e-5 and a gradient by
// 5e-5 there, for 17 us and 40 us less:
// at b 4, H 8, L 2048, D 64, fp32: statistics 69 us (Gram 16, scan 5, apply 43,
// reduction 5; the pass over every pair 202), gradient 163 us (the same in torch
// ops by query chunks of the dense scores 2.7 ms).
// Memory: b H ceil(L / 256) (D^2 + D) doubles of workspace, about the size of k
// itself in fp32 at D 128 and half of it at D 64 (b 8, H 16, L 32768, D 128:
// 2.2 GB).  sa_score_stats keeps the pass over every pair for callers that size
// its workspace without the key length and head_dim.
#include "common.h"
#include "fp32_tile.h"
#include "prof.h"

namespace sa {

// 8 consecutive elements of a row as bf16 (hi) and the rounding remainder (lo)
__device__ __forceinline__ void load8_split(const bf16* p, bool ok, v8bf& hi, v8bf& lo) {
  hi = ok ? load_v8bf(p) : zero_v8bf();
  lo = zero_v8bf();
}
__device__ __forceinline__ void load8_split(const float* p, bool ok, v8bf& hi, v8bf& lo) {
  if (!ok) {
    hi = lo = zero_v8bf();
    return;
  }
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  split_p(v4f{a.x, a.y, a.z, a.w}, v4f{b.x, b.y, b.z, b.w}, hi, lo);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void score_stats_kernel(const T* __restrict__ q,
                                                          const T* __restrict__ k,
                                                          const int64_t* __restrict__ q_length,
                                                          const int64_t* __restrict__ k_length,
                                                          int H, int Lq, int Lk, int causal,
                                                          float scale, double* __restrict__ part) {
  constexpr int KS = D / 32;
  constexpr bool SPLIT = sizeof(T) == 4;
  constexpr int TU = 4;   // 16-key tiles per step (loads issued together)
  __shared__ double red[4][3];
  const int nqb = (Lq + 63) / 64;
  const int qb = blockIdx.x % nqb;
  const int bh = blockIdx.x / nqb;
  const int b = bh / H;
  const int qlen = q_length ? static_cast<int>(min(max(q_length[b], int64_t{0}), int64_t{Lq})) : Lq;
  const int klen = k_length ? static_cast<int>(min(max(k_length[b], int64_t{0}), int64_t{Lk})) : Lk;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const T* qh = q + static_cast<long>(bh) * Lq * D;
  const T* kh = k + static_cast<long>(bh) * Lk * D;
  const int qi = 64 * qb + 16 * w + li;   // this lane's query
  const bool qv = qi < qlen;

  v8bf qf[KS], ql[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    load8_split(qh + static_cast<long>(min(qi, Lq - 1)) * D + 32 * ks + 8 * lg, qv, qf[ks], ql[ks]);

  double s1 = 0.0, s2 = 0.0;
  int cnt = 0;
  // keys [0, kend): the row's key length, and for causal attention up to this block's last query
  const int kend = causal ? min(klen, 64 * qb + 64) : klen;
  for (int k0 = 0; k0 < kend; k0 += 16 * TU) {
    v8bf kf[TU][KS], kl[TU][KS];
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      const int kr = k0 + 16 * u + li;   // the key row this lane supplies
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        load8_split(kh + static_cast<long>(min(kr, Lk - 1)) * D + 32 * ks + 8 * lg, kr < kend,
                    kf[u][ks], kl[u][ks]);
    }
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        acc = mfma_bf16(kf[u][ks], qf[ks], acc);
        if constexpr (SPLIT) {
          acc = mfma_bf16(kl[u][ks], qf[ks], acc);
          acc = mfma_bf16(kf[u][ks], ql[ks], acc);
        }
      }
      // acc[r]: key k0 + 16 u + 4 lg + r, query qi
      float t1 = 0.f, t2 = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = k0 + 16 * u + 4 * lg + r;
        const bool ok = qv && key < klen && (!causal || key <= qi);
        const float s = acc[r] * scale;
        t1 += ok ? s : 0.f;
        t2 += ok ? s * s : 0.f;
        cnt += ok ? 1 : 0;
      }
      s1 += t1;
      s2 += t2;
    }
  }
  double c = static_cast<double>(cnt);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s1 += __shfl_xor(s1, o, 64);
    s2 += __shfl_xor(s2, o, 64);
    c += __shfl_xor(c, o, 64);
  }
  if (lane == 0) {
    red[w][0] = c;
    red[w][1] = s1;
    red[w][2] = s2;
  }
  __syncthreads();
  if (tid < 3) {
    double* out = part + (static_cast<long>(bh) * nqb + qb) * 3;
    out[tid] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
  }
}

// out[h] = (count, sum, sum^2) over batch rows and query blocks of head h, and
// (when std is given) the population std sqrt(max(sum^2 / n - (sum / n)^2, 0))
__global__ __launch_bounds__(256) void score_stats_reduce_kernel(const double* __restrict__ part,
                                                                 int batch, int H, int nqb,
                                                                 double* __restrict__ out,
                                                                 float* __restrict__ std) {
  __shared__ double red[256][3];
  const int h = blockIdx.x, tid = threadIdx.x;
  double a[3] = {0.0, 0.0, 0.0};
  const int items = batch * nqb;
  for (int it = tid; it < items; it += 256) {
    const int b = it / nqb, qb = it % nqb;
    const double* p = part + ((static_cast<long>(b) * H + h) * nqb + qb) * 3;
    a[0] += p[0];
    a[1] += p[1];
    a[2] += p[2];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) red[tid][i] = a[i];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s)
#pragma unroll
      for (int i = 0; i < 3; ++i) red[tid][i] += red[tid + s][i];
    __syncthreads();
  }
  if (tid < 3) out[h * 3 + tid] = red[0][tid];
  if (std && tid == 0) {
    const double n = fmax(red[0][0], 1.0), mean = red[0][1] / n;
    const double var = red[0][2] / n - mean * mean;
    std[h] = static_cast<float>(sqrt(var < 0.0 ? 0.0 : var));   // a NaN stays one
  }
}

// ---------------------------------------------------------------------------
// moments through Gram matrices
// ---------------------------------------------------------------------------
constexpr int kChunk = 256;   // rows of a Gram matrix

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
// 16x16 += 16x4 . 4x16: lane l supplies A row l % 16 and B column l % 16 at
// k = l / 16 and holds result rows l / 16 + 4 i (not 4 (l / 16) + i as in fp32)
__device__ __forceinline__ v4d mfma_f64(double a, double b, const v4d& c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
enum class Pairs { kBefore, kAfter, kAll };   // keys y <= x, y >= x, every y

__device__ __forceinline__ int row_count(const int64_t* length, int b, int L) {
  return length ? static_cast<int>(min(max(length[b], int64_t{0}), int64_t{L})) : L;
}

// one chunk's sum y y^T (D x D) followed by sum y (D); rows past the length
// count as zero.  The 16x16 result tiles go round the four waves.
template <typename T, int D>
__global__ __launch_bounds__(256) void score_gram_kernel(const T* __restrict__ y,
                                                         const int64_t* __restrict__ length, int H,
                                                         int L, int nc, double* __restrict__ gram) {
  constexpr int NT = D / 16, NP = NT * NT / 4;
  __shared__ __align__(16) float yt[kRows * (D + 4)];
  const int bh = blockIdx.x / nc, c = blockIdx.x % nc;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int len = row_count(length, bh / H, L);
  const T* yh = y + static_cast<long>(bh) * L * D;
  double* out = gram + static_cast<long>(blockIdx.x) * (D * D + D);
  v4d acc[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) acc[j] = v4d{0.0, 0.0, 0.0, 0.0};
  double sum = 0.0;
  TileRegs<D> yr;
  const int r1 = min(kChunk * (c + 1), len);   // (may lie before the chunk: zeros are written)
  tile_load<D>(yr, yh, D, kChunk * c, r1, tid);
  for (int r0 = kChunk * c; r0 < r1; r0 += kRows) {
    __syncthreads();
    tile_store<D>(yr, yt, tid);
    __syncthreads();
    if (r0 + kRows < r1) tile_load<D>(yr, yh, D, r0 + kRows, r1, tid);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* row = yt + (16 * t + 4 * lg + i) * (D + 4) + li;
        // tile pair p = w + 4 j, (row tile p / NT, column tile p % NT)
        if constexpr (NT % 4 == 0) {
          double a[NT], z[NT / 4];
#pragma unroll
          for (int n = 0; n < NT; ++n) a[n] = row[16 * n];
#pragma unroll
          for (int n = 0; n < NT / 4; ++n) z[n] = row[16 * (4 * n + w)];
#pragma unroll
          for (int j = 0; j < NP; ++j) acc[j] = mfma_f64(a[4 * j / NT], z[j % (NT / 4)], acc[j]);
        } else {
#pragma unroll
          for (int j = 0; j < NP; ++j) {
            const int p = w + 4 * j;
            acc[j] = mfma_f64(row[16 * (p / NT)], row[16 * (p % NT)], acc[j]);
          }
        }
      }
    if (tid < D)
      for (int r = 0; r < kRows; ++r) sum += yt[r * (D + 4) + tid];
  }
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int p = w + 4 * j;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[(16 * (p / NT) + lg + 4 * i) * D + 16 * (p % NT) + li] = acc[j][i];
  }
  if (tid < D) out[D * D + tid] = sum;
}

// over the chunks of one (batch row, head), in place: each slot becomes the sum
// of the slots before it (kBefore), after it (kAfter); kAll: slot 0 the total
template <Pairs PAIRS>
__global__ __launch_bounds__(256) void score_gram_scan_kernel(double* __restrict__ gram, int nc,
                                                              int size) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= size) return;
  double* g = gram + static_cast<long>(blockIdx.y) * nc * size + i;
  double run = 0.0;
  for (int c0 = 0; c0 < nc; c0 += 8) {
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = min(c0 + u, nc - 1);
      t[u] = g[static_cast<long>(PAIRS == Pairs::kAfter ? nc - 1 - c : c) * size];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + u;
      if (c < nc) {
        if (PAIRS != Pairs::kAll) g[static_cast<long>(PAIRS == Pairs::kAfter ? nc - 1 - c : c) * size] = run;
        run += t[u];
      }
    }
  }
  if (PAIRS == Pairs::kAll) g[0] = run;
}

// 64 rows x against the rows y they pair with.  STATS: (count, sum, sum^2) of
// the scores.  Otherwise the gradient of the std:
//   dx_i = scale sum_j coef (s_ij - mean) y_j
template <typename T, int D, Pairs PAIRS, bool STATS>
__global__ __launch_bounds__(256, D <= 64 ? 3 : 1) void score_apply_kernel(
    const T* __restrict__ x, const T* __restrict__ y, const int64_t* __restrict__ x_length,
    const int64_t* __restrict__ y_length, int H, int Lx, int Ly, int nc, float scale,
    const double* __restrict__ gram, const double* __restrict__ stats, const float* __restrict__ g,
    double* __restrict__ part, T* __restrict__ dx) {
  constexpr int NT = D / 16;
  __shared__ __align__(16) float yt[kRows * (D + 4)];
  __shared__ double red[4][3];
  const int nxb = (Lx + kRows - 1) / kRows;
  const int xb = blockIdx.x % nxb, bh = blockIdx.x / nxb, b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int xlen = row_count(x_length, b, Lx), ylen = row_count(y_length, b, Ly);
  const T* yh = y + static_cast<long>(bh) * Ly * D;
  const int xi = kRows * xb + 16 * w + li;
  const long row = static_cast<long>(bh) * Lx + min(xi, Lx - 1);
  v4f xf[NT];
  v4d mx[NT];   // M x, then the row's gradient
  row_frag<D>(xf, x + row * D, lg, xi < xlen);
#pragma unroll
  for (int n = 0; n < NT; ++n) mx[n] = v4d{0.0, 0.0, 0.0, 0.0};

  double coef = 0.0, mean = 0.0;
  if (!STATS) {
    const double n = fmax(stats[3 * h], 1.0), mu = stats[3 * h + 1] / n;
    const double var = stats[3 * h + 2] / n - mu * mu, sd = sqrt(var < 0.0 ? 0.0 : var);
    coef = sd > 0.0 ? static_cast<double>(g[h]) / (n * sd) : 0.0;
    mean = mu;
  }

  // rows y outside the chunk, through their Gram matrix
  const int c = PAIRS == Pairs::kAll ? 0 : kRows * xb / kChunk;
  const bool outside =
      PAIRS == Pairs::kAfter ? kChunk * (c + 1) < ylen : ylen > 0 && (PAIRS == Pairs::kAll || c > 0);
  double s1 = 0.0, s2 = 0.0;
  if (outside) {
    const double* gm = gram + (static_cast<long>(bh) * nc + c) * (D * D + D);
    // row 4 (li % 4) + li / 4 of a 16-row tile as A row li: result element i of
    // lane group lg is then row 4 lg + i of the tile, as in xf
    const double* gr = gm + (4 * (li & 3) + (li >> 2)) * D + 4 * lg;
#pragma unroll
    for (int s = 0; s < NT; ++s) {
      v2d a[NT][2];
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          a[n][i] = *reinterpret_cast<const v2d*>(gr + 16 * n * D + 16 * s + 2 * i);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) mx[n] = mfma_f64(a[n][i >> 1][i & 1], xf[s][i], mx[n]);
    }
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double kap = gm[D * D + 16 * s + 4 * lg + i], xv = xf[s][i];
        if (STATS) {
          s1 = fma(xv, kap, s1);
          s2 = fma(xv, mx[s][i], s2);
        } else {
          mx[s][i] = coef * (scale * mx[s][i] - mean * kap);
        }
      }
    s1 = xi < xlen ? s1 * scale : 0.0;   // (a zero row times an infinite sum is no number)
    s2 = xi < xlen ? s2 * scale * scale : 0.0;
  }

  // the chunk's own pairs: tiles of 64 rows y
  if (PAIRS != Pairs::kAll) {
    const int first = PAIRS == Pairs::kBefore ? c * (kChunk / kRows) : xb;
    const int last = PAIRS == Pairs::kBefore ? xb : min((c + 1) * (kChunk / kRows), nxb) - 1;
    TileRegs<D> yr;
    tile_load<D>(yr, yh, D, kRows * first, ylen, tid);
    for (int t0 = first; t0 <= last; ++t0) {
      __syncthreads();
      tile_store<D>(yr, yt, tid);
      __syncthreads();
      if (t0 < last) tile_load<D>(yr, yh, D, kRows * (t0 + 1), ylen, tid);
      v4f s[4];
      score_tile<D>(s, yt, xf, li, lg);
      // the pair order matters in the diagonal tile, lengths in the last ones
      const bool edge = t0 == xb || kRows * (t0 + 1) > ylen || kRows * (xb + 1) > xlen;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int yi = kRows * t0 + 16 * t + 4 * lg + i;
          bool ok = true;
          if (edge)
            ok = xi < xlen && yi < ylen &&
                 (t0 != xb || (PAIRS == Pairs::kBefore ? yi <= xi : yi >= xi));
          const double v = static_cast<double>(s[t][i]) * scale;
          if (STATS) {
            s1 += ok ? v : 0.0;
            s2 += ok ? v * v : 0.0;
          } else {
            s[t][i] = ok ? static_cast<float>(coef * (v - mean)) : 0.f;
          }
        }
      if (!STATS) {
        v4f tile[NT];   // fp32 over a tile, fp64 from there on
        zero_frag(tile);
        weigh_tile<D>(tile, yt, s, li, lg);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx[n][i] += tile[n][i];
      }
    }
  }
  if (!STATS) {
    if (xi >= Lx) return;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      v4f v = {0.f, 0.f, 0.f, 0.f};
      if (xi < xlen)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = static_cast<float>(mx[n][i] * scale);
      store4(dx + row * D + 16 * n + 4 * lg, v);
    }
    return;
  }
  double n = xi < xlen && lg == 0 ? (PAIRS == Pairs::kAll ? ylen : min(xi + 1, ylen)) : 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s1 += __shfl_xor(s1, o, 64);
    s2 += __shfl_xor(s2, o, 64);
    n += __shfl_xor(n, o, 64);
  }
  if (lane == 0) {
    red[w][0] = n;
    red[w][1] = s1;
    red[w][2] = s2;
  }
  __syncthreads();
  if (tid < 3)
    part[static_cast<long>(blockIdx.x) * 3 + tid] =
        ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
}

// Gram matrices of y and their scan; nothing to do for causal rows of one chunk
template <typename T, int D, Pairs PAIRS>
int launch_gram(const T* y, const int64_t* length, int batch, int H, int L, double* gram,
                hipStream_t s) {
  const int nc = (L + kChunk - 1) / kChunk, size = D * D + D;
  if (PAIRS != Pairs::kAll && nc == 1) return 0;
  {
    ProfScope prof_("score_gram", s);
    hipLaunchKernelGGL((score_gram_kernel<T, D>), dim3(static_cast<unsigned>(batch) * H * nc),
                       dim3(256), 0, s, y, length, H, L, nc, gram);
    SA_CHECK_LAUNCH("score_gram");
  }
  if (nc == 1) return 0;
  // (batch row, head) in y, at most 65535 of them a launch
  const int rows = batch * H;
  for (int r0 = 0; r0 < rows; r0 += 65535) {
    ProfScope prof_("score_gram_scan", s);
    hipLaunchKernelGGL((score_gram_scan_kernel<PAIRS>),
                       dim3((size + 255) / 256, min(rows - r0, 65535)), dim3(256), 0, s,
                       gram + static_cast<long>(r0) * nc * size, nc, size);
    SA_CHECK_LAUNCH("score_gram_scan");
  }
  return 0;
}

template <typename T, int D, Pairs PAIRS, bool STATS>
int launch_apply(const T* x, const T* y, const int64_t* x_length, const int64_t* y_length,
                 int batch, int H, int Lx, int Ly, float scale, double* gram, const double* stats,
                 const float* g, double* part, T* dx, hipStream_t s) {
  const int rc = launch_gram<T, D, PAIRS>(y, y_length, batch, H, Ly, gram, s);
  if (rc) return rc;
  const int nc = (Ly + kChunk - 1) / kChunk;
  const unsigned blocks = static_cast<unsigned>(batch) * H * ((Lx + kRows - 1) / kRows);
  ProfScope prof_(STATS ? "score_moments" : "score_std_bwd", s);
  hipLaunchKernelGGL((score_apply_kernel<T, D, PAIRS, STATS>), dim3(blocks), dim3(256), 0, s, x, y,
                     x_length, y_length, H, Lx, Ly, nc, scale, gram, stats, g, part, dx);
  SA_CHECK_LAUNCH(STATS ? "score_moments" : "score_std_bwd");
  return 0;
}

template <typename T, int D>
int launch_moments(const void* q, const void* k, const int64_t* ql, const int64_t* kl, int batch,
                   int H, int Lq, int Lk, int causal, float scale, double* part, double* gram,
                   double* out, float* std, hipStream_t s) {
  const T *qt = static_cast<const T*>(q), *kt = static_cast<const T*>(k);
  const int rc =
      causal ? launch_apply<T, D, Pairs::kBefore, true>(qt, kt, ql, kl, batch, H, Lq, Lk, scale,
                                                        gram, nullptr, nullptr, part, nullptr, s)
             : launch_apply<T, D, Pairs::kAll, true>(qt, kt, ql, kl, batch, H, Lq, Lk, scale, gram,
                                                     nullptr, nullptr, part, nullptr, s);
  if (rc) return rc;
  ProfScope prof_("score_stats_reduce", s);
  hipLaunchKernelGGL(score_stats_reduce_kernel, dim3(H), dim3(256), 0, s, part, batch, H,
                     (Lq + kRows - 1) / kRows, out, std);
  SA_CHECK_LAUNCH("score_stats_reduce");
  return 0;
}

template <typename T, int D>
int launch_std_bwd(const void* q, const void* k, const int64_t* ql, const int64_t* kl, int batch,
                   int H, int Lq, int Lk, int causal, float scale, const double* stats,
                   const float* g, double* gram, void* dq, void* dk, hipStream_t s) {
  const T *qt = static_cast<const T*>(q), *kt = static_cast<const T*>(k);
  T *dqt = static_cast<T*>(dq), *dkt = static_cast<T*>(dk);
  if (causal) {
    const int rc = launch_apply<T, D, Pairs::kBefore, false>(
        qt, kt, ql, kl, batch, H, Lq, Lk, scale, gram, stats, g, nullptr, dqt, s);
    return rc ? rc : launch_apply<T, D, Pairs::kAfter, false>(kt, qt, kl, ql, batch, H, Lk, Lq,
                                                              scale, gram, stats, g, nullptr, dkt, s);
  }
  const int rc = launch_apply<T, D, Pairs::kAll, false>(qt, kt, ql, kl, batch, H, Lq, Lk, scale,
                                                        gram, stats, g, nullptr, dqt, s);
  return rc ? rc : launch_apply<T, D, Pairs::kAll, false>(kt, qt, kl, ql, batch, H, Lk, Lq, scale,
                                                          gram, stats, g, nullptr, dkt, s);
}

template <typename T, int D>
int launch_score_stats(const void* q, const void* k, const int64_t* q_length, const int64_t* k_length,
                       int batch, int H, int Lq, int Lk, int causal, float scale, double* part,
                       double* out, hipStream_t s) {
  const int nqb = (Lq + 63) / 64;
  const long blocks = static_cast<long>(batch) * H * nqb;
  {
    ProfScope prof_("score_stats", s);
    hipLaunchKernelGGL((score_stats_kernel<T, D>), dim3(static_cast<unsigned>(blocks)), dim3(256),
                       0, s, static_cast<const T*>(q), static_cast<const T*>(k), q_length,
                       k_length, H, Lq, Lk, causal, scale, part);
    SA_CHECK_LAUNCH("score_stats");
  }
  ProfScope prof_("score_stats_reduce", s);
  hipLaunchKernelGGL(score_stats_reduce_kernel, dim3(H), dim3(256), 0, s, part, batch, H, nqb, out,
                     nullptr);
  SA_CHECK_LAUNCH("score_stats_reduce");
  return 0;
}

template <typename T>
int dispatch_score_stats(int D, const void* q, const void* k, const int64_t* q_length,
                         const int64_t* k_length, int batch, int H, int Lq, int Lk, int causal,
                         float scale, double* part, double* out, hipStream_t s) {
#define SA_SS(DD) \
  launch_score_stats<T, DD>(q, k, q_length, k_length, batch, H, Lq, Lk, causal, scale, part, out, s)
  switch (D) {
    case 32: return SA_SS(32);
    case 64: return SA_SS(64);
    case 96: return SA_SS(96);
    case 128: return SA_SS(128);
    default: break;
  }
#undef SA_SS
  sa_set_error("sa_score_stats: head_dim %d not supported (32, 64, 96, 128)", D);
  return 1;
}

}  // namespace sa

extern "C" size_t sa_score_stats_workspace_size(int batch, int heads, int q_len) {
  if (batch <= 0 || heads <= 0 || q_len <= 0) return 0;
  return static_cast<size_t>(batch) * heads * ((q_len + 63) / 64) * 3 * sizeof(double);
}

extern "C" int sa_score_stats(int dtype, const void* q, const void* k, const int64_t* q_length,
                              const int64_t* k_length, int batch, int heads, int q_len, int k_len,
                              int head_dim, int causal, float scale, void* workspace,
                              size_t workspace_bytes, double* out, void* stream) {
  SA_CHECK_ARG(batch >= 0 && heads > 0 && q_len >= 0 && k_len >= 0 && head_dim > 0,
               "sa_score_stats: bad sizes b=%d H=%d Lq=%d Lk=%d D=%d", batch, heads, q_len, k_len,
               head_dim);
  SA_CHECK_ARG(!causal || q_len == k_len, "sa_score_stats: causal needs q_len == k_len");
  SA_CHECK_ARG(q && k && out, "sa_score_stats: null tensor pointer");
  // the same checks for empty and non-empty calls: dtype and head_dim first
  SA_CHECK_ARG(dtype == sa::kBF16 || dtype == sa::kF32, "sa_score_stats: unsupported dtype %d",
               dtype);
  SA_CHECK_ARG(head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128,
               "sa_score_stats: head_dim %d not supported (32, 64, 96, 128)", head_dim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (batch == 0 || q_len == 0 || k_len == 0) {   // no pairs: the reduction writes zeros
    hipLaunchKernelGGL(sa::score_stats_reduce_kernel, dim3(heads), dim3(256), 0, s, nullptr, 0,
                       heads, 0, out, nullptr);
    SA_CHECK_LAUNCH("score_stats_reduce");
    return 0;
  }
  const size_t need = sa_score_stats_workspace_size(batch, heads, q_len);
  SA_CHECK_ARG(workspace && workspace_bytes >= need,
               "sa_score_stats: workspace of %zu B, %zu B needed", workspace_bytes, need);
  SA_CHECK_ARG(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15) == 0,
               "sa_score_stats: q and k must be 16-byte aligned");
  double* part = static_cast<double*>(workspace);
  if (dtype == sa::kBF16)
    return sa::dispatch_score_stats<sa::bf16>(head_dim, q, k, q_length, k_length, batch, heads,
                                              q_len, k_len, causal, scale, part, out, s);
  if (dtype == sa::kF32)
    return sa::dispatch_score_stats<float>(head_dim, q, k, q_length, k_length, batch, heads, q_len,
                                           k_len, causal, scale, part, out, s);
  sa_set_error("sa_score_stats: unsupported dtype %d", dtype);
  return 1;
}

namespace {
// doubles of the block partials, rounded up so that the Gram matrices behind
// them stay 16-byte aligned
size_t moments_part(int batch, int heads, int q_len) {
  return (static_cast<size_t>(batch) * heads * ((q_len + sa::kRows - 1) / sa::kRows) * 3 + 1) &
         ~static_cast<size_t>(1);
}
int check_moments(const char* what, int dtype, const void* q, const void* k, int batch, int heads,
                  int q_len, int k_len, int head_dim, int causal) {
  SA_CHECK_ARG(batch > 0 && heads > 0 && q_len > 0 && k_len > 0, "%s: bad sizes b=%d H=%d Lq=%d Lk=%d",
               what, batch, heads, q_len, k_len);
  SA_CHECK_ARG(!causal || q_len == k_len, "%s: causal needs q_len == k_len", what);
  SA_CHECK_ARG(dtype == sa::kBF16 || dtype == sa::kF32, "%s: unsupported dtype %d", what, dtype);
  SA_CHECK_ARG(head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128,
               "%s: head_dim %d not supported (32, 64, 96, 128)", what, head_dim);
  SA_CHECK_ARG(q && k && ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15) == 0,
               "%s: q and k must be non-null and 16-byte aligned", what);
  SA_CHECK_ARG(static_cast<int64_t>(batch) * heads * ((max(q_len, k_len) + sa::kRows - 1) / sa::kRows) <
                   (1LL << 31), "%s: too many blocks", what);
  return 0;
}
}  // namespace

extern "C" size_t sa_score_moments_workspace_size(int batch, int heads, int q_len, int k_len,
                                                  int head_dim) {
  if (batch <= 0 || heads <= 0 || q_len <= 0 || k_len <= 0 || head_dim <= 0) return 0;
  const size_t nc = (static_cast<size_t>(max(q_len, k_len)) + sa::kChunk - 1) / sa::kChunk;
  return moments_part(batch, heads, q_len) * sizeof(double) +
         static_cast<size_t>(batch) * heads * nc * (head_dim * head_dim + head_dim) * sizeof(double);
}

#define SA_MOMENTS_CASE(DD, FN, ...) \
  case DD:                           \
    return dtype == sa::kBF16 ? sa::FN<sa::bf16, DD>(__VA_ARGS__) : sa::FN<float, DD>(__VA_ARGS__)
#define SA_MOMENTS_DISPATCH(FN, ...)       \
  switch (head_dim) {                      \
    SA_MOMENTS_CASE(32, FN, __VA_ARGS__);  \
    SA_MOMENTS_CASE(64, FN, __VA_ARGS__);  \
    SA_MOMENTS_CASE(96, FN, __VA_ARGS__);  \
    SA_MOMENTS_CASE(128, FN, __VA_ARGS__); \
    default: return 1;                     \
  }

extern "C" int sa_score_moments(int dtype, const void* q, const void* k, const int64_t* q_length,
                                const int64_t* k_length, int batch, int heads, int q_len, int k_len,
                                int head_dim, int causal, float scale, void* workspace,
                                size_t workspace_bytes, double* out, float* std, void* stream) {
  if (check_moments("sa_score_moments", dtype, q, k, batch, heads, q_len, k_len, head_dim, causal))
    return 1;
  SA_CHECK_ARG(out, "sa_score_moments: null tensor pointer");
  const size_t need = sa_score_moments_workspace_size(batch, heads, q_len, k_len, head_dim);
  SA_CHECK_ARG(workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace_bytes >= need,
               "sa_score_moments: 16-byte aligned workspace of %zu B needed, %zu B given", need,
               workspace_bytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  double* part = static_cast<double*>(workspace);
  double* gram = part + moments_part(batch, heads, q_len);
  SA_MOMENTS_DISPATCH(launch_moments, q, k, q_length, k_length, batch, heads, q_len, k_len, causal,
                      scale, part, gram, out, std, s)
}

extern "C" int sa_score_std_bwd(int dtype, const void* q, const void* k, const int64_t* q_length,
                                const int64_t* k_length, int batch, int heads, int q_len, int k_len,
                                int head_dim, int causal, float scale, const double* stats,
                                const float* std_grad, void* dq, void* dk, void* workspace,
                                size_t workspace_bytes, void* stream) {
  if (check_moments("sa_score_std_bwd", dtype, q, k, batch, heads, q_len, k_len, head_dim, causal))
    return 1;
  SA_CHECK_ARG(stats && std_grad && dq && dk &&
                   ((reinterpret_cast<uintptr_t>(dq) | reinterpret_cast<uintptr_t>(dk)) & 15) == 0,
               "sa_score_std_bwd: tensor pointers must be non-null, dq and dk 16-byte aligned");
  const size_t need = sa_score_moments_workspace_size(batch, heads, q_len, k_len, head_dim);
  SA_CHECK_ARG(workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace_bytes >= need,
               "sa_score_std_bwd: 16-byte aligned workspace of %zu B needed, %zu B given", need,
               workspace_bytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  double* gram = static_cast<double*>(workspace) + moments_part(batch, heads, q_len);
  SA_MOMENTS_DISPATCH(launch_std_bwd, q, k, q_length, k_length, batch, heads, q_len, k_len, causal,
                      scale, stats, std_grad, gram, dq, dk, s)
}
