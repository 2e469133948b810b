// SSD chunked scan in fp32, forward and backward, for head_dim 32 or a
// multiple of 64, state_dim 32, 64 or 128 and chunks of whole 64-row tiles
// (the models' sizes); other fp32 sizes run the general kernels of ssd_fwd.hip
// and ssd_bwd.hip.  Same formulas and the same saved tensors.
//
// All products are v_mfma_f32_16x16x4_f32 on the tiles of fp32_tile.h.  The
// scan is gated linear attention: per head, the weight of row sigma for row
// tau is CB[tau,sigma] exp(min(dc_tau - dc_sigma, 0)) (times dt_sigma), and
// because a score tile's accumulator is the next product's B operand as it
// stands, weighted tiles never go through LDS or a transpose.  What the
// general kernels spend on fp32 (one 64x64 tile per block, both operands
// transposed into LDS, four barriers and no loads in flight per product, and
// for dCB one block per 64 rows walking every head and tile in turn) bounds
// them at 14 TFLOP/s; here a tile's loads are in flight during the products
// of the one before, a barrier pair covers 64 to 192 MFMAs per wave, and
// launches with too few blocks are split over the heads of a group.
//
// Measured at b 4, L 2000, H 16, P 64, N 64, one group, chunk 256 (general
// kernel before -> here): scan 148 -> 63 us, chunk states 53 -> 17, their
// gradient 51 -> 17, dCB 348 -> 93, du 160 -> 50, dB / dC 122 -> 59 + 5; the
// forward and backward 934 -> 328 us.
#include "fp32_tile.h"
#include "prof.h"
#include "ssd_common.h"

namespace sa {
namespace {

// exp(min(x, 0))
__device__ __forceinline__ float decay(float x) { return fast_exp2(fminf(x, 0.0f) * kLog2e); }

__device__ __forceinline__ float sum_groups(float v) {   // over the four lane groups
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

struct Tok {   // where a block's (batch row, chunk) starts
  int b, c, qlim, lim;
  long tok0;
};
__device__ __forceinline__ Tok tok_of(int bc, const SsdDims& d, const int64_t* length) {
  Tok k;
  k.b = bc / d.nc;
  k.c = bc % d.nc;
  k.qlim = min(d.Lc, d.L - k.c * d.Lc);
  k.lim = max(0, chunk_limit(seq_limit(length, k.b, d.L), k.c, d.Lc));
  k.tok0 = static_cast<long>(k.b) * d.L + static_cast<long>(k.c) * d.Lc;
  return k;
}
__device__ __forceinline__ long chunk_row(const Tok& k, int h, const SsdDims& d) {
  return ((static_cast<long>(k.b) * d.H + h) * d.nc + k.c) * d.Lc;
}
__device__ __forceinline__ long state_row(const Tok& k, int h, int p0, const SsdDims& d) {
  return (((static_cast<long>(k.b) * d.nc + k.c) * d.H + h) * d.P + p0) * static_cast<long>(d.N);
}

// ---------------------------------------------------------------------------
// chunk states (MODE 0): S = sum_t e^{min(dc_last - dc_t, 0)} dt_t u_t B_t^T;
// their gradient (MODE 1): sum_t e^{dc_t} dy_t C_t^T.  One block per (b, c,
// head, PT rows p): wave w owns 16 of the p and its share of the n tiles.
// ---------------------------------------------------------------------------
template <int N, int PT, int MODE>
__global__ __launch_bounds__(256) void f32_outer_kernel(
    const float* __restrict__ a, const float* __restrict__ x, const float* __restrict__ dt,
    const float* __restrict__ dc, const int64_t* __restrict__ length, float* __restrict__ out,
    SsdDims d) {
  constexpr int PW = PT / 16, NW = N / 16 * PW / 4;   // p tiles; n tiles of a wave
  __shared__ __align__(16) float at[kRows * (PT + 4)];
  __shared__ __align__(16) float xt[kRows * (N + 4)];
  __shared__ float scl[1024];
  const int pts = d.P / PT;
  const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
  const int p0 = bid % pts * PT, h = bid / pts % d.H;
  const Tok k = tok_of(bid / pts / d.H, d, length);
  const int g = h / (d.H / d.G);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int klim = MODE == 0 ? k.qlim : k.lim;
  const long crow = chunk_row(k, h, d);
  const long a_rs = static_cast<long>(d.H) * d.P, x_rs = static_cast<long>(d.G) * d.N;
  const float* ab = a + k.tok0 * a_rs + static_cast<long>(h) * d.P + p0;
  const float* xb = x + k.tok0 * x_rs + static_cast<long>(g) * d.N;
  TileRegs<PT> ar;
  TileRegs<N> xr;
  tile_load(ar, ab, a_rs, 0, klim, tid);
  tile_load(xr, xb, x_rs, 0, klim, tid);
  const float last = dc[crow + d.Lc - 1];
  for (int t = tid; t < d.Lc; t += 256)
    scl[t] = t >= klim ? 0.f
             : MODE == 0 ? expf(fminf(last - dc[crow + t], 0.0f)) * dt[crow + t]
                         : expf(dc[crow + t]);
  v4f acc[NW];
  zero_frag(acc);
  const int pw = w % PW, n0 = w / PW * NW;
  for (int r0 = 0; r0 < klim; r0 += kRows) {
    __syncthreads();
    tile_store(ar, at, tid);
    tile_store(xr, xt, tid);
    __syncthreads();
    if (r0 + kRows < klim) {
      tile_load(ar, ab, a_rs, r0 + kRows, klim, tid);
      tile_load(xr, xb, x_rs, r0 + kRows, klim, tid);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const v4f sc = *reinterpret_cast<const v4f*>(scl + r0 + 16 * t + 4 * lg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * t + 4 * lg + i;
        const float av = at[r * (PT + 4) + 16 * pw + li] * sc[i];
#pragma unroll
        for (int n = 0; n < NW; ++n)
          acc[n] = mfma_f32(av, xt[r * (N + 4) + 16 * (n0 + n) + li], acc[n]);
      }
    }
  }
  float* o = out + state_row(k, h, p0, d);
#pragma unroll
  for (int n = 0; n < NW; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[(16 * pw + 4 * lg + i) * N + 16 * (n0 + n) + li] = acc[n][i];
}

// ---------------------------------------------------------------------------
// chunk scan: y_t = e^{dc_t} H_in C_t + sum_{s <= t} (C_t . B_s) decay dt_s u_s.
// One block per (b, c, HC heads of a group, 64 rows t, PT of p); the score
// tile C B^T is shared by the heads.  Longest tiles first.
// ---------------------------------------------------------------------------
template <int N, int PT, int HC>
__global__ __launch_bounds__(256) void f32_scan_kernel(
    const float* __restrict__ u, const float* __restrict__ Bm, const float* __restrict__ Cm,
    const float* __restrict__ dt, const float* __restrict__ dc, const float* __restrict__ states,
    float* __restrict__ y, SsdDims d) {
  __shared__ __align__(16) float bt[kRows * (N + 4)];
  __shared__ __align__(16) float ut[HC][kRows * (PT + 4)];
  __shared__ __align__(16) float dct[HC][kRows], dtt[HC][kRows];
  const int tts = d.Lc / kRows, pts = d.P / PT, hgs = d.H / HC;
  const int per = gridDim.x / tts;
  const int ti = tts - 1 - static_cast<int>(blockIdx.x) / per;
  const int bid = xcd_swizzle(blockIdx.x % per, per);
  const int p0 = bid % pts * PT, h0 = bid / pts % hgs * HC;
  const Tok k = tok_of(bid / pts / hgs, d, nullptr);
  const int t0 = ti * kRows;
  if (t0 >= k.qlim) return;
  const int g = h0 / (d.H / d.G);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const long u_rs = static_cast<long>(d.H) * d.P, x_rs = static_cast<long>(d.G) * d.N;
  const float* bb = Bm + k.tok0 * x_rs + static_cast<long>(g) * d.N;
  const float* ub = u + k.tok0 * u_rs + static_cast<long>(h0) * d.P + p0;
  const int t = t0 + 16 * w + li;   // this lane's row
  v4f cf[N / 16];
  row_frag<N>(cf, Cm + (k.tok0 + min(t, k.qlim - 1)) * x_rs + static_cast<long>(g) * d.N, lg, true);
  const long crow = chunk_row(k, h0, d), hstep = static_cast<long>(d.nc) * d.Lc;
  float dct_own[HC];
  v4f o[HC][PT / 16];
  TileRegs<N, PT> hr[HC];
#pragma unroll
  for (int j = 0; j < HC; ++j) tile_load(hr[j], states + state_row(k, h0 + j, p0, d), N, 0, PT, tid);
#pragma unroll
  for (int j = 0; j < HC; ++j) {
    dct_own[j] = dc[crow + j * hstep + min(t, d.Lc - 1)];
    const float e = fast_exp2(dct_own[j] * kLog2e);
    if (j) __syncthreads();
    tile_store(hr[j], bt, tid);
    __syncthreads();
    score_tile<N>(o[j], bt, cf, li, lg);
#pragma unroll
    for (int i = 0; i < PT / 16; ++i) o[j][i] *= e;
  }
  TileRegs<N> br;
  TileRegs<PT> ur[HC];
  float tc = 0.f, td = 0.f;
  const auto fetch = [&](int s0) {
    tile_load(br, bb, x_rs, s0, k.qlim, tid);
#pragma unroll
    for (int j = 0; j < HC; ++j) tile_load(ur[j], ub + j * d.P, u_rs, s0, k.qlim, tid);
    if (tid < HC * kRows) {
      const long at = crow + (tid >> 6) * hstep + s0 + (tid & 63);
      tc = dc[at];
      td = dt[at];
    }
  };
  fetch(0);
  for (int s0 = 0; s0 <= t0; s0 += kRows) {
    __syncthreads();
    tile_store(br, bt, tid);
#pragma unroll
    for (int j = 0; j < HC; ++j) tile_store(ur[j], ut[j], tid);
    if (tid < HC * kRows) {
      dct[tid >> 6][tid & 63] = tc;
      dtt[tid >> 6][tid & 63] = td;
    }
    __syncthreads();
    if (s0 < t0) fetch(s0 + kRows);
    v4f cb[4];
    score_tile<N>(cb, bt, cf, li, lg);
#pragma unroll
    for (int j = 0; j < HC; ++j) {
      v4f wt[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v4f dcs = *reinterpret_cast<const v4f*>(dct[j] + 16 * q + 4 * lg);
        const v4f dts = *reinterpret_cast<const v4f*>(dtt[j] + 16 * q + 4 * lg);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = cb[q][i] * decay(dct_own[j] - dcs[i]) * dts[i];
          wt[q][i] = s0 < t0 || 16 * q + 4 * lg + i <= 16 * w + li ? v : 0.f;
        }
      }
      weigh_tile<PT>(o[j], ut[j], wt, li, lg);
    }
  }
  if (t >= k.qlim) return;
#pragma unroll
  for (int j = 0; j < HC; ++j)
#pragma unroll
    for (int i = 0; i < PT / 16; ++i)
      store4(y + (k.tok0 + t) * u_rs + static_cast<long>(h0 + j) * d.P + p0 + 16 * i + 4 * lg,
             o[j][i]);
}

// 16 values a lane, summed over the 16 lanes of its group: lane li gets the sum
// of value li (a reduce-scatter, 15 shuffles)
__device__ __forceinline__ float reduce_scatter16(const v4f (&m)[4], int li) {
  float v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = m[j >> 2][j & 3];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1)
#pragma unroll
    for (int j = 0; j < o; ++j) {
      const bool up = li & o;
      const float keep = up ? v[j + o] : v[j], send = up ? v[j] : v[j + o];
      v[j] = keep + __shfl_xor(send, o, 64);
    }
  return v[0];
}

// ---------------------------------------------------------------------------
// dCB and the intra-chunk decay sums.  One block per (b, c, group, tile pair
// I >= J, share of the group's heads): W^T tiles (rows sigma of J, columns
// tau of I) = u dy^T, weighted and summed over the heads.  The first share
// also stores C B^T for the du kernel.
// ---------------------------------------------------------------------------
template <int N, int PT>
__global__ __launch_bounds__(256) void f32_dcb_kernel(
    const float* __restrict__ u, const float* __restrict__ Bm, const float* __restrict__ Cm,
    const float* __restrict__ dy, const float* __restrict__ dt, const float* __restrict__ dc,
    const int64_t* __restrict__ length, float* __restrict__ cbm, float* __restrict__ dCB,
    float* __restrict__ rpart, float* __restrict__ qpart, SsdDims d, int shares, int per_share) {
  constexpr int LD = (N > PT ? N : PT) + 4;
  __shared__ __align__(16) float lds[kRows * LD];   // B rows, then u rows
  __shared__ float red[4][kRows];
  const int tts = d.Lc / kRows, pairs = tts * (tts + 1) / 2, hpg = d.H / d.G;
  const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
  const int share = bid % shares, pair = bid / shares % pairs;
  const int bcg = bid / shares / pairs, g = bcg % d.G;
  const Tok k = tok_of(bcg / d.G, d, length);
  int I = 0;
  while ((I + 1) * (I + 2) / 2 <= pair) ++I;
  const int J = pair - I * (I + 1) / 2;
  const int t0 = I * kRows, s0 = J * kRows;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int t = t0 + 16 * w + li;   // tau of this lane
  const int k0 = share * per_share, k1 = min(hpg, k0 + per_share);
  const long bhc0 = (static_cast<long>(k.b) * d.H + g * hpg) * d.nc + k.c;

  if (t0 >= k.lim) {   // past the length: zero sums
    for (int j = k0; j < k1; ++j) {
      const long bhc = bhc0 + static_cast<long>(j) * d.nc;
      if (tid < kRows) rpart[(bhc * tts + J) * d.Lc + t0 + tid] = 0.f;
      if (tid < kRows) qpart[(bhc * tts + I) * d.Lc + s0 + tid] = 0.f;
    }
    return;
  }
  const long u_rs = static_cast<long>(d.H) * d.P, x_rs = static_cast<long>(d.G) * d.N;
  v4f cb[4];
  {
    TileRegs<N> br;
    tile_load(br, Bm + k.tok0 * x_rs + static_cast<long>(g) * d.N, x_rs, s0, k.lim, tid);
    v4f cf[N / 16];
    row_frag<N>(cf, Cm + (k.tok0 + min(t, k.lim - 1)) * x_rs + static_cast<long>(g) * d.N, lg,
                t < k.lim);
    tile_store(br, lds, tid);
    __syncthreads();
    score_tile<N>(cb, lds, cf, li, lg);
  }
  const long tile = (static_cast<long>(bcg) * d.Lc + t) * d.Lc + s0;
  if (share == 0)
#pragma unroll
    for (int q = 0; q < 4; ++q) store4(cbm + tile + 16 * q + 4 * lg, cb[q]);

  v4f sum[4];
  zero_frag(sum);
  const int pts = d.P / PT;
  const float* ub = u + k.tok0 * u_rs + static_cast<long>(g * hpg) * d.P;
  const float* yb = dy + (k.tok0 + min(t, k.lim - 1)) * u_rs + static_cast<long>(g * hpg) * d.P;
  TileRegs<PT> ur;
  v4f yn[PT / 16];
  tile_load(ur, ub + static_cast<long>(k0) * d.P, u_rs, s0, k.lim, tid);
  row_frag<PT>(yn, yb + static_cast<long>(k0) * d.P, lg, t < k.lim);
  for (int j = k0; j < k1; ++j) {
    const long bhc = bhc0 + static_cast<long>(j) * d.nc;
    v4f wv[4];
    zero_frag(wv);
    const float dct = dc[bhc * d.Lc + t];
    v4f dcs[4], dts[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      dcs[q] = *reinterpret_cast<const v4f*>(dc + bhc * d.Lc + s0 + 16 * q + 4 * lg);
      dts[q] = *reinterpret_cast<const v4f*>(dt + bhc * d.Lc + s0 + 16 * q + 4 * lg);
    }
    for (int pt = 0; pt < pts; ++pt) {
      v4f yf[PT / 16];
#pragma unroll
      for (int i = 0; i < PT / 16; ++i) yf[i] = yn[i];
      __syncthreads();   // the tile before, and the column sums, are read
      tile_store(ur, lds, tid);
      __syncthreads();
      const long nxt = static_cast<long>(j) * d.P + (pt + 1) * PT;
      if (nxt < static_cast<long>(k1) * d.P) {
        tile_load(ur, ub + nxt, u_rs, s0, k.lim, tid);
        row_frag<PT>(yn, yb + nxt, lg, t < k.lim);
      }
      score_add<PT>(wv, lds, yf, li, lg);
    }
    v4f m[4];
    float rs = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = s0 + 16 * q + 4 * lg + i;
        const float v = wv[q][i] * dts[q][i] * decay(dct - dcs[q][i]);
        sum[q][i] += I > J || s <= t ? v : 0.f;
        m[q][i] = I > J || s < t ? v * cb[q][i] : 0.f;
        rs += m[q][i];
      }
    rs = sum_groups(rs);
    if (lg == 0) rpart[(bhc * tts + J) * d.Lc + t] = rs;
    const float cs = reduce_scatter16(m, li);
    red[w][16 * (li >> 2) + 4 * lg + (li & 3)] = cs;
    __syncthreads();
    if (tid < kRows)
      qpart[(bhc * tts + I) * d.Lc + s0 + tid] =
          ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
  }
  float* out = dCB + static_cast<long>(share) * d.b * d.nc * d.G * d.Lc * d.Lc + tile;
#pragma unroll
  for (int q = 0; q < 4; ++q) store4(out + 16 * q + 4 * lg, sum[q]);
}

// ---------------------------------------------------------------------------
// du and its part of ddt: acc = e^{min(dc_last - dc_s, 0)} dS B_s
//   + sum_{t >= s} CB[t,s] decay dy_t;  du = acc dt, ddt_direct = acc . u.
// One block per (b, c, head, 64 rows s, PT of p).  Longest tiles first.
// ---------------------------------------------------------------------------
template <int N, int PT>
__global__ __launch_bounds__(256) void f32_du_kernel(
    const float* __restrict__ u, const float* __restrict__ Bm, const float* __restrict__ dy,
    const float* __restrict__ dt, const float* __restrict__ dc, const float* __restrict__ dS,
    const float* __restrict__ cbm, const int64_t* __restrict__ length, float* __restrict__ du,
    float* __restrict__ ddt_part, SsdDims d) {
  constexpr int SZ = PT * (N + 4) > kRows * (PT + 4) ? PT * (N + 4) : kRows * (PT + 4);
  __shared__ __align__(16) float lds[SZ];   // dS rows, then dy rows
  __shared__ __align__(16) float dct[kRows];
  const int tts = d.Lc / kRows, pts = d.P / PT;
  const int per = gridDim.x / tts;
  const int si = static_cast<int>(blockIdx.x) / per;
  const int bid = xcd_swizzle(blockIdx.x % per, per);
  const int pt = bid % pts, p0 = pt * PT, h = bid / pts % d.H;
  const int bc = bid / pts / d.H;
  const Tok k = tok_of(bc, d, length);
  const int g = h / (d.H / d.G), s0 = si * kRows;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int s = s0 + 16 * w + li;   // sigma of this lane
  const long u_rs = static_cast<long>(d.H) * d.P, x_rs = static_cast<long>(d.G) * d.N;
  const long crow = chunk_row(k, h, d);
  const long own = (k.tok0 + s) * u_rs + static_cast<long>(h) * d.P + p0;
  float* dpart = ddt_part + (crow / d.Lc * pts + pt) * d.Lc;
  if (s0 >= k.lim) {   // past the length
    if (s < k.qlim)
#pragma unroll
      for (int i = 0; i < PT / 16; ++i) store4(du + own + 16 * i + 4 * lg, v4f{0.f, 0.f, 0.f, 0.f});
    if (lg == 0) dpart[s] = 0.f;
    return;
  }
  v4f o[PT / 16], bf[N / 16];
  TileRegs<N, PT> hr;
  tile_load(hr, dS + state_row(k, h, p0, d), N, 0, PT, tid);
  row_frag<N>(bf, Bm + (k.tok0 + min(s, k.lim - 1)) * x_rs + static_cast<long>(g) * d.N, lg, true);
  const float dcs = dc[crow + s], last = dc[crow + d.Lc - 1];
  const float* yb = dy + k.tok0 * u_rs + static_cast<long>(h) * d.P + p0;
  const float* cb = cbm + (static_cast<long>(bc) * d.G + g) * d.Lc * d.Lc + s;
  TileRegs<PT> yr;
  float tc = 0.f;
  v4f cn[4];
  const auto fetch = [&](int t0) {
    tile_load(yr, yb, u_rs, t0, k.lim, tid);
    if (tid < kRows) tc = dc[crow + t0 + tid];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) cn[q][i] = cb[static_cast<long>(t0 + 16 * q + 4 * lg + i) * d.Lc];
  };
  fetch(s0);
  tile_store(hr, lds, tid);
  __syncthreads();
  score_tile<N>(o, lds, bf, li, lg);
  const float e = decay(last - dcs);
#pragma unroll
  for (int i = 0; i < PT / 16; ++i) o[i] *= e;
  for (int t0 = s0; t0 < k.lim; t0 += kRows) {
    __syncthreads();
    tile_store(yr, lds, tid);
    if (tid < kRows) dct[tid] = tc;
    v4f wt[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) wt[q] = cn[q];
    __syncthreads();
    if (t0 + kRows < k.lim) fetch(t0 + kRows);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const v4f dtau = *reinterpret_cast<const v4f*>(dct + 16 * q + 4 * lg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = wt[q][i] * decay(dtau[i] - dcs);
        wt[q][i] = t0 > s0 || 16 * q + 4 * lg + i >= 16 * w + li ? v : 0.f;
      }
    }
    weigh_tile<PT>(o, lds, wt, li, lg);   // rows past the length are zero in the tile
  }
  const bool in = s < k.lim;
  const float dts = dt[crow + s];
  float dd = 0.f;
#pragma unroll
  for (int i = 0; i < PT / 16; ++i) {
    const float4 uv = in ? load4_f32(u + own + 16 * i + 4 * lg) : float4{0.f, 0.f, 0.f, 0.f};
    dd += o[i][0] * uv.x + o[i][1] * uv.y + o[i][2] * uv.z + o[i][3] * uv.w;
    if (s < k.qlim)
      store4(du + own + 16 * i + 4 * lg, in ? o[i] * dts : v4f{0.f, 0.f, 0.f, 0.f});
  }
  dd = sum_groups(dd);
  if (lg == 0) dpart[s] = in ? dd : 0.f;
}

// ---------------------------------------------------------------------------
// dB and dC with their decay terms x_B, x_C.  One block per (dC or dB, b, c,
// group, 64 rows, share of the group's heads): per head the state part,
// summed; the first share adds the intra-chunk part through dCB.  With more
// than one share the sums go to `part` and f32_sum_kernel adds them.
// ---------------------------------------------------------------------------
template <int N, int PT>
__global__ __launch_bounds__(256) void f32_dbdc_kernel(
    const float* __restrict__ u, const float* __restrict__ Bm, const float* __restrict__ Cm,
    const float* __restrict__ dy, const float* __restrict__ dt, const float* __restrict__ dc,
    const float* __restrict__ states, const float* __restrict__ dS, const float* __restrict__ dCB,
    const int64_t* __restrict__ length, float* __restrict__ dB, float* __restrict__ dC,
    float* __restrict__ part, float* __restrict__ xB, float* __restrict__ xC, SsdDims d, int shares,
    int per_share, int cb_shares) {
  __shared__ __align__(16) float lds[kRows * (N + 4)];   // state rows, then C or B rows
  const int tts = d.Lc / kRows, hpg = d.H / d.G, pts = d.P / PT;
  const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
  const int which = bid % 2, share = bid / 2 % shares, ti = bid / 2 / shares % tts;
  const int bcg = bid / 2 / shares / tts, g = bcg % d.G;
  const Tok k = tok_of(bcg / d.G, d, length);
  const int r0 = ti * kRows;
  if (r0 >= k.qlim) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int r = r0 + 16 * w + li, rc = max(0, min(r, k.lim - 1));
  const bool in = r < k.lim;
  const long u_rs = static_cast<long>(d.H) * d.P, x_rs = static_cast<long>(d.G) * d.N;
  const int k0 = share * per_share, k1 = min(hpg, k0 + per_share);
  v4f acc[N / 16], act[N / 16];
  zero_frag(acc);
  row_frag<N>(act, (which ? Cm : Bm) + (k.tok0 + rc) * x_rs + static_cast<long>(g) * d.N, lg, in);
  if (r0 < k.lim) {
    const float* ab = (which ? dy : u) + (k.tok0 + rc) * u_rs + static_cast<long>(g * hpg) * d.P;
    const float* sb = (which ? states : dS) + state_row(k, g * hpg, 0, d);
    TileRegs<N, PT> sr;
    v4f an[PT / 16];
    tile_load(sr, sb + static_cast<long>(k0) * d.P * N, N, 0, PT, tid);
    row_frag<PT>(an, ab + static_cast<long>(k0) * d.P, lg, in);
    for (int j = k0; j < k1; ++j) {
      const long bhc = (static_cast<long>(k.b) * d.H + g * hpg + j) * d.nc + k.c;
      const float* dch = dc + bhc * d.Lc;
      float sc = which ? dch[r] : dch[d.Lc - 1] - dch[r];
      const float dtr = which ? 1.f : dt[bhc * d.Lc + r];
      v4f tmp[N / 16];
      zero_frag(tmp);
      for (int pt = 0; pt < pts; ++pt) {
        v4f af[PT / 16];
#pragma unroll
        for (int i = 0; i < PT / 16; ++i) af[i] = an[i];
        __syncthreads();
        tile_store(sr, lds, tid);
        __syncthreads();
        const long nxt = static_cast<long>(j) * d.P + (pt + 1) * PT;
        if (nxt < static_cast<long>(k1) * d.P) {
          tile_load(sr, sb + nxt * N, N, 0, PT, tid);
          row_frag<PT>(an, ab + nxt, lg, in);
        }
        weigh_tile<N>(tmp, lds, af, li, lg);
      }
      sc = in ? expf(which ? sc : fminf(sc, 0.0f)) * dtr : 0.f;
      float x = 0.f;
#pragma unroll
      for (int i = 0; i < N / 16; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float v = tmp[i][q] * sc;
          acc[i][q] += v;
          x = fmaf(v, act[i][q], x);
        }
      x = sum_groups(x);
      if (lg == 0) (which ? xC : xB)[bhc * d.Lc + r] = x;
    }
    if (share == 0) {
      const float* cb = dCB + static_cast<long>(bcg) * d.Lc * d.Lc;
      const long cb_step = static_cast<long>(d.b) * d.nc * d.G * d.Lc * d.Lc;
      const float* xs = (which ? Bm : Cm) + k.tok0 * x_rs + static_cast<long>(g) * d.N;
      const int first = which ? 0 : r0, last = which ? r0 : (k.lim - 1) / kRows * kRows;
      TileRegs<N> xr;
      tile_load(xr, xs, x_rs, first, k.lim, tid);
      for (int q0 = first; q0 <= last; q0 += kRows) {
        v4f wt[4];
        zero_frag(wt);
        for (int e = 0; e < cb_shares; ++e) {
          const float* ce = cb + e * cb_step;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (which) {   // dC[r] += sum_s dCB[r,s] B_s
              wt[q] += *reinterpret_cast<const v4f*>(ce + static_cast<long>(r) * d.Lc + q0 + 16 * q + 4 * lg);
            } else {       // dB[r] += sum_t dCB[t,r] C_t
#pragma unroll
              for (int i = 0; i < 4; ++i)
                wt[q][i] += ce[static_cast<long>(q0 + 16 * q + 4 * lg + i) * d.Lc + r];
            }
          }
        }
        __syncthreads();
        tile_store(xr, lds, tid);
        __syncthreads();
        if (q0 < last) tile_load(xr, xs, x_rs, q0 + kRows, k.lim, tid);
        weigh_tile<N>(acc, lds, wt, li, lg);
      }
    }
  }
  if (r >= k.qlim) return;
  const long at = (k.tok0 + r) * x_rs + static_cast<long>(g) * d.N;
  float* out = shares == 1 ? (which ? dC : dB)
                           : part + (static_cast<long>(share) * 2 + which) * d.b * d.L * x_rs;
#pragma unroll
  for (int i = 0; i < N / 16; ++i)
    store4(out + at + 16 * i + 4 * lg, in ? acc[i] : v4f{0.f, 0.f, 0.f, 0.f});
}

// dB and dC (n4 float4 each) = their shares' sums, in order
__global__ __launch_bounds__(256) void f32_sum_kernel(const float4* __restrict__ part, long n4,
                                                      int shares, float4* __restrict__ dB,
                                                      float4* __restrict__ dC) {
  const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= 2 * n4) return;
  float4 a = part[i];
  for (int e = 1; e < shares; ++e) {
    const float4 v = part[e * 2 * n4 + i];
    a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
  }
  if (i < n4) dB[i] = a;
  else dC[i - n4] = a;
}

// shares of a group's heads that bring `blocks` to about four per CU (one for
// an empty scan, which launches nothing)
int head_shares(long blocks, int hpg) {
  if (blocks <= 0) return 1;
  long want = (1024 + blocks - 1) / blocks;
  if (want > hpg) want = hpg;
  const int per = (hpg + static_cast<int>(want) - 1) / static_cast<int>(want);
  return (hpg + per - 1) / per;
}

}  // namespace

bool ssd_f32_shape_ok(const SsdDims& d) {
  return (d.N == 32 || d.N == 64 || d.N == 128) && (d.P == 32 || d.P % 64 == 0) && d.Lc % kRows == 0;
}
int ssd_f32_dcb_shares(const SsdDims& d) {
  const int tts = d.Lc / kRows;
  return head_shares(static_cast<long>(d.b) * d.nc * d.G * tts * (tts + 1) / 2, d.H / d.G);
}
int ssd_f32_dbdc_shares(const SsdDims& d) {
  return head_shares(2L * d.b * d.nc * d.G * (d.Lc / kRows), d.H / d.G);
}

#define SA_F32_N(PT, FN, ...)                  \
  switch (d.N) {                               \
    case 32: return FN<32, PT>(__VA_ARGS__);   \
    case 64: return FN<64, PT>(__VA_ARGS__);   \
    default: return FN<128, PT>(__VA_ARGS__);  \
  }
#define SA_F32_DISPATCH(FN, ...)      \
  if (d.P == 32) {                    \
    SA_F32_N(32, FN, __VA_ARGS__)     \
  } else {                            \
    SA_F32_N(64, FN, __VA_ARGS__)     \
  }

namespace {

template <int N, int PT>
int outer_np(const float* a, const float* x, const float* dt, const float* dc, const int64_t* length,
             float* out, const SsdDims& d, int mode, hipStream_t s) {
  const long blocks = static_cast<long>(d.P / PT) * d.H * d.b * d.nc;
  ProfScope prof_(mode == 0 ? "chunk_state_fwd" : "chunk_dstate_bwd", s);
  auto kernel = mode == 0 ? f32_outer_kernel<N, PT, 0> : f32_outer_kernel<N, PT, 1>;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, s, a, x, dt, dc, length, out, d);
  SA_CHECK_LAUNCH("f32_outer");
  return 0;
}

template <int N, int PT>
int scan_np(const float* u, const float* B, const float* C, const float* dt, const float* dc,
            const float* states, float* y, const SsdDims& d, hipStream_t s) {
  const long tiles = static_cast<long>(d.Lc / kRows) * (d.P / PT) * d.b * d.nc;
  // two heads a block share the score tile; one where that leaves the chip short of blocks
  const bool two = (d.H / d.G) % 2 == 0 && tiles * d.H >= 2048;
  ProfScope prof_("chunk_scan_fwd", s);
  hipLaunchKernelGGL((two ? f32_scan_kernel<N, PT, 2> : f32_scan_kernel<N, PT, 1>),
                     dim3(tiles * (d.H / (two ? 2 : 1))), dim3(256), 0, s, u, B, C, dt, dc, states, y,
                     d);
  SA_CHECK_LAUNCH("f32_scan");
  return 0;
}

template <int N, int PT>
int bwd_np(const float* u, const float* B, const float* C, const float* dy, const float* dt,
           const float* dc, const float* states, const float* dS, const int64_t* length, float* du,
           float* dB, float* dC, const SsdF32Ws& w, const SsdDims& d, hipStream_t s) {
  const int tts = d.Lc / kRows, hpg = d.H / d.G;
  const long bnc = static_cast<long>(d.b) * d.nc;
  const int cs = ssd_f32_dcb_shares(d), bs = ssd_f32_dbdc_shares(d);
  {
    ProfScope prof_("chunk_dcb_bwd", s);
    hipLaunchKernelGGL((f32_dcb_kernel<N, PT>), dim3(bnc * d.G * (tts * (tts + 1) / 2) * cs), dim3(256),
                       0, s, u, B, C, dy, dt, dc, length, w.cb, w.dCB, w.rpart, w.qpart, d, cs,
                       (hpg + cs - 1) / cs);
    SA_CHECK_LAUNCH("f32_dcb");
  }
  {
    ProfScope prof_("chunk_du_bwd", s);
    hipLaunchKernelGGL((f32_du_kernel<N, PT>), dim3(bnc * d.H * (d.P / PT) * tts), dim3(256), 0, s, u,
                       B, dy, dt, dc, dS, w.cb, length, du, w.ddt_part, d);
    SA_CHECK_LAUNCH("f32_du");
  }
  {
    ProfScope prof_("chunk_dbdc_bwd", s);
    hipLaunchKernelGGL((f32_dbdc_kernel<N, PT>), dim3(2 * bnc * d.G * tts * bs), dim3(256), 0, s, u, B,
                       C, dy, dt, dc, states, dS, w.dCB, length, dB, dC, w.part, w.xB, w.xC, d, bs,
                       (hpg + bs - 1) / bs, cs);
    SA_CHECK_LAUNCH("f32_dbdc");
  }
  if (bs > 1) {
    const long n4 = static_cast<long>(d.b) * d.L * d.G * d.N / 4;
    ProfScope prof_("dbdc_sum", s);
    hipLaunchKernelGGL(f32_sum_kernel, dim3((2 * n4 + 255) / 256), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(w.part), n4, bs,
                       reinterpret_cast<float4*>(dB), reinterpret_cast<float4*>(dC));
    SA_CHECK_LAUNCH("f32_sum");
  }
  return 0;
}

}  // namespace

int launch_f32_outer(const float* a, const float* x, const float* dt, const float* dc,
                     const int64_t* length, float* out, const SsdDims& d, int mode, hipStream_t s) {
  SA_F32_DISPATCH(outer_np, a, x, dt, dc, length, out, d, mode, s)
}
int launch_f32_scan(const float* u, const float* B, const float* C, const float* dt, const float* dc,
                    const float* states, float* y, const SsdDims& d, hipStream_t s) {
  SA_F32_DISPATCH(scan_np, u, B, C, dt, dc, states, y, d, s)
}
int launch_f32_bwd(const float* u, const float* B, const float* C, const float* dy, const float* dt,
                   const float* dc, const float* states, const float* dS, const int64_t* length,
                   float* du, float* dB, float* dC, const SsdF32Ws& w, const SsdDims& d,
                   hipStream_t s) {
  SA_F32_DISPATCH(bwd_np, u, B, C, dy, dt, dc, states, dS, length, du, dB, dC, w, d, s)
}

}  // namespace sa
