// SelectiveMHA's training attention in fp32, forward and backward, without
// the score matrix (modules/selective_attention.py:86-95, 125-144):
//   s_ij = scale q_i . k_j + [j != i] log_gate_j,  j <= i when causal,
//   out_i = softmax_j(s_ij) v_j,
// and for an upstream gradient dO, with P the softmax and
// delta_i = dO_i . out_i = sum_j P_ij dO_i . v_j,
//   dS_ij = P_ij (dO_i . v_j - delta_i)
//   dq_i = scale sum_j dS_ij k_j      dk_j = scale sum_i dS_ij q_i
//   dv_j = sum_i P_ij dO_i            dlog_gate_j = sum_{i != j} dS_ij.
//
// Every product is a v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 sums, as
// the dense fp32 form), so the matrix cores' fp32 rate (157 TFLOP/s) bounds
// all three kernels: 4, 6 and 8 D FLOP per (query, key) pair.  Operands need
// no transposes.  A score tile is computed with the contraction that follows
// it in the MFMA's row index (keys for out and dq, queries for dk and dv),
// so accumulator element i of a lane is the B operand of that product's i-th
// issue, and the A operand is a column of the row-major LDS tile, read as
// dwords (conflict-free at a row length of D + 4).  The score products
// themselves take four issues per 16-byte LDS read, both operands with the
// same (lane group, element) -> d assignment.
//
// A 256-thread block owns 64 queries (64 keys in the dk / dv kernel), 16 per
// wave, and streams 64-row tiles of the other side through one LDS stage;
// the next tile's loads are in flight during a tile's products.  Registers set
// how many blocks share a CU and cover each other's barriers and softmax (35 KB
// of LDS would let four): at D 64, causal, 166 VGPRs in the forward, 198 for dq,
// 232 for dk / dv, so three, two and two.  Causal blocks do unequal work; they are issued longest first
// with every other 256 reversed, so that the blocks of a CU add up to about
// the same.
//
// Measured at b 4, H 8, L 2048, D 64, causal (67 M pairs): forward 185 us,
// dq 266 us, dk / dv 359 us, 93 to 97 TFLOP/s of fp32 MFMA each, 60 % of the
// 155 TFLOP/s that a large fp32 GEMM reaches here.  The dense form took 3.9 ms
// for the same (elementwise passes over 0.5 GB score matrices, and products
// over the masked half).
#include "common.h"
#include "fp32_tile.h"
#include "prof.h"

namespace sa {
namespace {

struct TrainDims {
  int batch, H, L;
  float scale;
  long q[3], k[3], v[3], d[3];   // element strides of batch, head, row
};

// block -> (batch * H + head, tile index): the tile index runs from the
// longest walk to the shortest over the whole launch, every other run of
// 256 blocks reversed
__device__ __forceinline__ void block_tile(int bid, int nblocks, int nbh, bool last_longest,
                                           int ntiles, int& bh, int& tile) {
  const int run = bid >> 8;
  if (run & 1) {
    const int lo = run << 8, hi = min(lo + 256, nblocks) - 1;
    bid = hi - (bid - lo);
  }
  bh = bid % nbh;
  tile = bid / nbh;
  if (last_longest) tile = ntiles - 1 - tile;
}

__device__ __forceinline__ float expf_fast(float x) { return fast_exp2(x * kLog2e); }

// ---------------------------------------------------------------------------
// forward: out, and per query the softmax's maximum and 1 / sum
// ---------------------------------------------------------------------------
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, D <= 64 ? (CAUSAL ? 3 : 2) : 1) void attn_train_fwd_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ log_gate, TrainDims dm, float* __restrict__ out,
    float* __restrict__ smax, float* __restrict__ srcp) {
  __shared__ __align__(16) float kt[kRows * (D + 4)];
  __shared__ __align__(16) float vt[kRows * (D + 4)];
  __shared__ __align__(16) float bt[kRows];
  const int L = dm.L, nt = (L + kRows - 1) / kRows;
  int bh, qb;
  block_tile(blockIdx.x, gridDim.x, dm.batch * dm.H, CAUSAL, nt, bh, qb);
  const int b = bh / dm.H, h = bh % dm.H;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const float* kh = k + b * dm.k[0] + h * dm.k[1];
  const float* vh = v + b * dm.v[0] + h * dm.v[1];
  const float* gate = log_gate + static_cast<long>(bh) * L;
  const int qi = kRows * qb + 16 * w + li;
  v4f qf[D / 16], o[D / 16];
  row_frag<D>(qf, q + b * dm.q[0] + h * dm.q[1] + min(qi, L - 1) * dm.q[2], lg, true);
#pragma unroll
  for (int i = 0; i < D / 16; ++i) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const int ntiles = CAUSAL ? qb + 1 : nt;
  TileRegs<D> kr, vr;
  float br = 0.f;
  tile_load<D>(kr, kh, dm.k[2], 0, L, tid);
  tile_load<D>(vr, vh, dm.v[2], 0, L, tid);
  if (tid < kRows) br = tid < L ? gate[tid] : 0.f;
  for (int t0 = 0; t0 < ntiles; ++t0) {
    __syncthreads();   // every wave is done with the tile before
    tile_store<D>(kr, kt, tid);
    tile_store<D>(vr, vt, tid);
    if (tid < kRows) bt[tid] = br;
    __syncthreads();
    const int k0 = kRows * t0, kn = k0 + kRows;
    if (t0 + 1 < ntiles) {
      tile_load<D>(kr, kh, dm.k[2], kn, L, tid);
      tile_load<D>(vr, vh, dm.v[2], kn, L, tid);
      if (tid < kRows) br = kn + tid < L ? gate[kn + tid] : 0.f;
    }
    v4f s[4];
    score_tile<D>(s, kt, qf, li, lg);
    // a tile that holds a block row's own key or keys past the row is masked
    const bool edge = t0 == qb || kn > L;
    float tmax = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const v4f bias = *reinterpret_cast<const v4f*>(bt + 16 * t + 4 * lg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 16 * t + 4 * lg + i;
        float x = fmaf(s[t][i], dm.scale, bias[i]);
        if (edge) {
          if (key == qi) x = s[t][i] * dm.scale;
          if (key >= L || (CAUSAL && key > qi)) x = -INFINITY;
        }
        s[t][i] = x;
        tmax = fmaxf(tmax, x);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float mn = fmaxf(m, tmax);
    const float mu = mn == -INFINITY ? 0.f : mn;   // no key so far: every weight 0
    const float alpha = expf_fast(m - mu);
    m = mn;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[t][i] = expf_fast(s[t][i] - mu);
        sum += s[t][i];
      }
    l = fmaf(l, alpha, sum);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) o[i] *= alpha;
    weigh_tile<D>(o, vt, s, li, lg);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (qi >= L) return;
  const float r = 1.0f / l;
  const long row = static_cast<long>(bh) * L + qi;
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    *reinterpret_cast<v4f*>(out + row * D + 16 * i + 4 * lg) = o[i] * r;
  if (lg == 0) {
    smax[row] = m;
    srcp[row] = r;
  }
}

// ---------------------------------------------------------------------------
// backward over queries: dq, and delta_i = dO_i . out_i for the key kernel
// ---------------------------------------------------------------------------
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attn_train_dq_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ log_gate, const float* __restrict__ out,
    const float* __restrict__ dout, const float* __restrict__ smax,
    const float* __restrict__ srcp, TrainDims dm, float* __restrict__ dq,
    float* __restrict__ delta) {
  __shared__ __align__(16) float kt[kRows * (D + 4)];
  __shared__ __align__(16) float vt[kRows * (D + 4)];
  __shared__ __align__(16) float bt[kRows];
  const int L = dm.L, nt = (L + kRows - 1) / kRows;
  int bh, qb;
  block_tile(blockIdx.x, gridDim.x, dm.batch * dm.H, CAUSAL, nt, bh, qb);
  const int b = bh / dm.H, h = bh % dm.H;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const float* kh = k + b * dm.k[0] + h * dm.k[1];
  const float* vh = v + b * dm.v[0] + h * dm.v[1];
  const float* gate = log_gate + static_cast<long>(bh) * L;
  const int qi = kRows * qb + 16 * w + li, qc = min(qi, L - 1);
  const long row = static_cast<long>(bh) * L + qc;
  v4f qf[D / 16], df[D / 16], acc[D / 16];
  row_frag<D>(qf, q + b * dm.q[0] + h * dm.q[1] + qc * dm.q[2], lg, true);
  row_frag<D>(df, dout + b * dm.d[0] + h * dm.d[1] + qc * dm.d[2], lg, true);
  const float m = smax[row], r = srcp[row];
  float dl = 0.f;
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const v4f of = *reinterpret_cast<const v4f*>(out + row * D + 16 * s + 4 * lg);
#pragma unroll
    for (int i = 0; i < 4; ++i) dl = fmaf(df[s][i], of[i], dl);
    acc[s] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  dl += __shfl_xor(dl, 16, 64);
  dl += __shfl_xor(dl, 32, 64);

  const int ntiles = CAUSAL ? qb + 1 : nt;
  TileRegs<D> kr, vr;
  float br = 0.f;
  tile_load<D>(kr, kh, dm.k[2], 0, L, tid);
  tile_load<D>(vr, vh, dm.v[2], 0, L, tid);
  if (tid < kRows) br = tid < L ? gate[tid] : 0.f;
  for (int t0 = 0; t0 < ntiles; ++t0) {
    __syncthreads();
    tile_store<D>(kr, kt, tid);
    tile_store<D>(vr, vt, tid);
    if (tid < kRows) bt[tid] = br;
    __syncthreads();
    const int k0 = kRows * t0, kn = k0 + kRows;
    if (t0 + 1 < ntiles) {
      tile_load<D>(kr, kh, dm.k[2], kn, L, tid);
      tile_load<D>(vr, vh, dm.v[2], kn, L, tid);
      if (tid < kRows) br = kn + tid < L ? gate[kn + tid] : 0.f;
    }
    v4f s[4], dp[4];
    score_tile<D>(s, kt, qf, li, lg);
    score_tile<D>(dp, vt, df, li, lg);
    const bool edge = t0 == qb || kn > L;
    // sum of P dO.v over the tile: a row that ends in its only tile takes it as
    // its delta.  There one weight is often near 1 and dO.v - delta cancels, to 0
    // in a row of one key; dO.out, summed in another order, leaves a rounding
    // (dq off by 4.0e-7 instead of 4.3e-7 at L 500, D 128, as in the dense form)
    float own = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const v4f bias = *reinterpret_cast<const v4f*>(bt + 16 * t + 4 * lg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 16 * t + 4 * lg + i;
        float x = fmaf(s[t][i], dm.scale, bias[i]);
        if (edge && key == qi) x = s[t][i] * dm.scale;
        float p = expf_fast(x - m) * r;
        if (edge && (key >= L || (CAUSAL && key > qi))) p = dp[t][i] = 0.f;
        s[t][i] = p;
        own = fmaf(p, dp[t][i], own);
      }
    }
    if (ntiles == 1) {
      own += __shfl_xor(own, 16, 64);
      dl = own + __shfl_xor(own, 32, 64);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[t][i] *= dp[t][i] - dl;
    weigh_tile<D>(acc, kt, s, li, lg);
  }
  if (qi >= L) return;
  if (lg == 0) delta[row] = dl;
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    *reinterpret_cast<v4f*>(dq + row * D + 16 * i + 4 * lg) = acc[i] * dm.scale;
}

// ---------------------------------------------------------------------------
// backward over keys: dk, dv and dlog_gate
// ---------------------------------------------------------------------------
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) void attn_train_dkv_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ log_gate, const float* __restrict__ dout,
    const float* __restrict__ smax, const float* __restrict__ srcp,
    const float* __restrict__ delta, TrainDims dm, float* __restrict__ dk, float* __restrict__ dv,
    float* __restrict__ dgate) {
  __shared__ __align__(16) float qt[kRows * (D + 4)];
  __shared__ __align__(16) float dt[kRows * (D + 4)];
  __shared__ __align__(16) float st[3][kRows];   // max, 1 / sum, delta of the tile's queries
  const int L = dm.L, nt = (L + kRows - 1) / kRows;
  int bh, kb;
  block_tile(blockIdx.x, gridDim.x, dm.batch * dm.H, false, nt, bh, kb);
  const int b = bh / dm.H, h = bh % dm.H;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const float* qh = q + b * dm.q[0] + h * dm.q[1];
  const float* dh = dout + b * dm.d[0] + h * dm.d[1];
  const long rows = static_cast<long>(bh) * L;
  const int key = kRows * kb + 16 * w + li, kc = min(key, L - 1);
  v4f kf[D / 16], vf[D / 16], ak[D / 16], av[D / 16];
  row_frag<D>(kf, k + b * dm.k[0] + h * dm.k[1] + kc * dm.k[2], lg, true);
  row_frag<D>(vf, v + b * dm.v[0] + h * dm.v[1] + kc * dm.v[2], lg, true);
  const float bias = log_gate[rows + kc];
  // fp32 over a tile's 16 values, fp64 over the tiles: a chain of fp32 sums over
  // every query is off by 6.5e-7 at L 2048 and 7.9e-7 at 4096 (here and in torch's
  // own sum 3.5e-7)
  double dg = 0.0;
#pragma unroll
  for (int i = 0; i < D / 16; ++i) ak[i] = av[i] = v4f{0.f, 0.f, 0.f, 0.f};

  const int first = CAUSAL ? kb : 0;
  TileRegs<D> qr, dr;
  float sr = 0.f;
  const float* stat = tid < 64 ? smax : tid < 128 ? srcp : delta;
  const int sx = tid & 63;
  tile_load<D>(qr, qh, dm.q[2], kRows * first, L, tid);
  tile_load<D>(dr, dh, dm.d[2], kRows * first, L, tid);
  if (tid < 192) sr = kRows * first + sx < L ? stat[rows + kRows * first + sx] : 0.f;
  for (int t0 = first; t0 < nt; ++t0) {
    __syncthreads();
    tile_store<D>(qr, qt, tid);
    tile_store<D>(dr, dt, tid);
    if (tid < 192) st[tid >> 6][sx] = sr;
    __syncthreads();
    const int q0 = kRows * t0, qn = q0 + kRows;
    if (t0 + 1 < nt) {
      tile_load<D>(qr, qh, dm.q[2], qn, L, tid);
      tile_load<D>(dr, dh, dm.d[2], qn, L, tid);
      if (tid < 192) sr = qn + sx < L ? stat[rows + qn + sx] : 0.f;
    }
    v4f s[4], dp[4];
    score_tile<D>(s, qt, kf, li, lg);
    score_tile<D>(dp, dt, vf, li, lg);
    const bool edge = t0 == kb || qn > L;
    float dgt = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const v4f mx = *reinterpret_cast<const v4f*>(st[0] + 16 * t + 4 * lg);
      const v4f rc = *reinterpret_cast<const v4f*>(st[1] + 16 * t + 4 * lg);
      const v4f dl = *reinterpret_cast<const v4f*>(st[2] + 16 * t + 4 * lg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int qi = q0 + 16 * t + 4 * lg + i;
        float x = fmaf(s[t][i], dm.scale, bias);
        if (edge && key == qi) x = s[t][i] * dm.scale;
        float p = expf_fast(x - mx[i]) * rc[i];
        float ds = p * (dp[t][i] - dl[i]);
        if (edge && (qi >= L || (CAUSAL && key > qi))) p = ds = 0.f;
        dgt += edge && key == qi ? 0.f : ds;
        s[t][i] = p;
        dp[t][i] = ds;
      }
    }
    dg += dgt;
    weigh_tile<D>(av, dt, s, li, lg);
    weigh_tile<D>(ak, qt, dp, li, lg);
  }
  dg += __shfl_xor(dg, 16, 64);
  dg += __shfl_xor(dg, 32, 64);
  if (key >= L) return;
  const long row = rows + key;
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    *reinterpret_cast<v4f*>(dk + row * D + 16 * i + 4 * lg) = ak[i] * dm.scale;
    *reinterpret_cast<v4f*>(dv + row * D + 16 * i + 4 * lg) = av[i];
  }
  if (lg == 0) dgate[row] = static_cast<float>(dg);
}

template <int D, bool CAUSAL>
int launch_fwd(const float* q, const float* k, const float* v, const float* log_gate,
               const TrainDims& dm, float* out, float* smax, float* srcp, hipStream_t s) {
  const unsigned blocks = static_cast<unsigned>(dm.batch) * dm.H * ((dm.L + kRows - 1) / kRows);
  ProfScope prof_("attn_train_fwd", s);
  hipLaunchKernelGGL((attn_train_fwd_kernel<D, CAUSAL>), dim3(blocks), dim3(256), 0, s, q, k, v,
                     log_gate, dm, out, smax, srcp);
  SA_CHECK_LAUNCH("attn_train_fwd");
  return 0;
}

template <int D, bool CAUSAL>
int launch_bwd(const float* q, const float* k, const float* v, const float* log_gate,
               const float* out, const float* dout, const float* smax, const float* srcp,
               const TrainDims& dm, float* dq, float* dk, float* dv, float* dgate, float* delta,
               hipStream_t s) {
  const unsigned blocks = static_cast<unsigned>(dm.batch) * dm.H * ((dm.L + kRows - 1) / kRows);
  {
    ProfScope prof_("attn_train_dq", s);
    hipLaunchKernelGGL((attn_train_dq_kernel<D, CAUSAL>), dim3(blocks), dim3(256), 0, s, q, k, v,
                       log_gate, out, dout, smax, srcp, dm, dq, delta);
    SA_CHECK_LAUNCH("attn_train_dq");
  }
  ProfScope prof_("attn_train_dkv", s);
  hipLaunchKernelGGL((attn_train_dkv_kernel<D, CAUSAL>), dim3(blocks), dim3(256), 0, s, q, k, v,
                     log_gate, dout, smax, srcp, delta, dm, dk, dv, dgate);
  SA_CHECK_LAUNCH("attn_train_dkv");
  return 0;
}

// sizes, strides and alignment every launch assumes; 0 when they hold
int check_train(const char* what, int batch, int heads, int len, int head_dim, const void* const* p,
                int np, const int64_t* strides, int ns) {
  SA_CHECK_ARG(batch > 0 && heads > 0 && len > 0, "%s: bad sizes b=%d H=%d L=%d", what, batch,
               heads, len);
  SA_CHECK_ARG(head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128,
               "%s: head_dim %d not supported (32, 64, 96, 128)", what, head_dim);
  SA_CHECK_ARG(static_cast<int64_t>(batch) * heads * ((len + kRows - 1) / kRows) < (1LL << 31),
               "%s: too many blocks", what);
  SA_CHECK_ARG(strides, "%s: null strides", what);
  for (int i = 0; i < ns; ++i)
    SA_CHECK_ARG(strides[i] >= 0 && strides[i] % 4 == 0, "%s: stride %lld not a multiple of 4", what,
                 static_cast<long long>(strides[i]));
  for (int i = 0; i < np; ++i)
    SA_CHECK_ARG(p[i] && (reinterpret_cast<uintptr_t>(p[i]) & 15) == 0,
                 "%s: tensor pointers must be non-null and 16-byte aligned", what);
  return 0;
}

TrainDims train_dims(int batch, int heads, int len, float scale, const int64_t* st, int n) {
  TrainDims dm{};
  dm.batch = batch;
  dm.H = heads;
  dm.L = len;
  dm.scale = scale;
  for (int i = 0; i < 3; ++i) {
    dm.q[i] = st[i];
    dm.k[i] = st[3 + i];
    dm.v[i] = st[6 + i];
    dm.d[i] = n == 12 ? st[9 + i] : 0;
  }
  return dm;
}

}  // namespace
}  // namespace sa

#define SA_TRAIN_CASE(DD, FN, ...) \
  case DD: return causal ? sa::FN<DD, true>(__VA_ARGS__) : sa::FN<DD, false>(__VA_ARGS__)
#define SA_TRAIN_DISPATCH(FN, ...)       \
  switch (head_dim) {                    \
    SA_TRAIN_CASE(32, FN, __VA_ARGS__);  \
    SA_TRAIN_CASE(64, FN, __VA_ARGS__);  \
    SA_TRAIN_CASE(96, FN, __VA_ARGS__);  \
    SA_TRAIN_CASE(128, FN, __VA_ARGS__); \
    default: return 1;                   \
  }

extern "C" int sa_gated_attn_train_fwd(const float* q, const float* k, const float* v,
                                       const float* log_gate, const int64_t* strides, int batch,
                                       int heads, int len, int head_dim, int causal, float scale,
                                       float* out, float* row_max, float* row_rcp, void* stream) {
  const void* p[] = {q, k, v, out};
  if (sa::check_train("sa_gated_attn_train_fwd", batch, heads, len, head_dim, p, 4, strides, 9))
    return 1;
  SA_CHECK_ARG(log_gate && row_max && row_rcp, "sa_gated_attn_train_fwd: null tensor pointer");
  const sa::TrainDims dm = sa::train_dims(batch, heads, len, scale, strides, 9);
  hipStream_t s = static_cast<hipStream_t>(stream);
  SA_TRAIN_DISPATCH(launch_fwd, q, k, v, log_gate, dm, out, row_max, row_rcp, s)
}

extern "C" int sa_gated_attn_train_bwd(const float* q, const float* k, const float* v,
                                       const float* log_gate, const float* out, const float* dout,
                                       const float* row_max, const float* row_rcp,
                                       const int64_t* strides, int batch, int heads, int len,
                                       int head_dim, int causal, float scale, float* dq, float* dk,
                                       float* dv, float* dlog_gate, float* delta, void* stream) {
  const void* p[] = {q, k, v, out, dout, dq, dk, dv};
  if (sa::check_train("sa_gated_attn_train_bwd", batch, heads, len, head_dim, p, 8, strides, 12))
    return 1;
  SA_CHECK_ARG(log_gate && row_max && row_rcp && dlog_gate && delta,
               "sa_gated_attn_train_bwd: null tensor pointer");
  const sa::TrainDims dm = sa::train_dims(batch, heads, len, scale, strides, 12);
  hipStream_t s = static_cast<hipStream_t>(stream);
  SA_TRAIN_DISPATCH(launch_bwd, q, k, v, log_gate, out, dout, row_max, row_rcp, dm, dq, dk, dv,
                    dlog_gate, delta, s)
}
