// fp32 tiles on v_mfma_f32_16x16x4_f32, shared by the training attention, the
// score statistics and the fp32 SSD scan: a row-major LDS tile of row length
// D + 4 floats serves both as the row operand of a score product (16-byte
// reads) and, transposed, as the weighted sum of its rows (dword reads); both
// are free of bank conflicts at that row length.
#pragma once

#include "common.h"

namespace sa {

constexpr int kRows = 64;   // rows of a tile

// 4 consecutive elements as fp32
__device__ __forceinline__ float4 load4_f32(const float* p) {
  return *reinterpret_cast<const float4*>(p);
}
__device__ __forceinline__ float4 load4_f32(const bf16* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return float4{bf16lo_to_f32(u.x), bf16hi_to_f32(u.x), bf16lo_to_f32(u.y), bf16hi_to_f32(u.y)};
}
__device__ __forceinline__ void store4(float* p, const v4f& v) { *reinterpret_cast<v4f*>(p) = v; }
__device__ __forceinline__ void store4(bf16* p, const v4f& v) {
  *reinterpret_cast<uint2*>(p) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// tile rows r0 .. r0 + R - 1 of x (row stride ld elements), zero at and past
// row L, as R D / 1024 float4 per thread of a 256-thread block
template <int D, int R = kRows>
struct TileRegs {
  float4 r[R * D / 1024];
};
template <int D, int R, typename T>
__device__ __forceinline__ void tile_load(TileRegs<D, R>& t, const T* x, long ld, int r0, int L,
                                          int tid) {
#pragma unroll
  for (int p = 0; p < R * D / 1024; ++p) {
    const int idx = tid + 256 * p, row = idx / (D / 4), c = 4 * (idx % (D / 4));
    const int g = r0 + row;
    t.r[p] = g < L ? load4_f32(x + g * ld + c) : float4{0.f, 0.f, 0.f, 0.f};
  }
}
template <int D, int R>
__device__ __forceinline__ void tile_store(const TileRegs<D, R>& t, float* lds, int tid) {
#pragma unroll
  for (int p = 0; p < R * D / 1024; ++p) {
    const int idx = tid + 256 * p, row = idx / (D / 4), c = 4 * (idx % (D / 4));
    *reinterpret_cast<float4*>(lds + row * (D + 4) + c) = t.r[p];
  }
}

// one row of D floats as a score operand: lane group g holds elements
// 16 s + 4 g + i
template <int D, typename T>
__device__ __forceinline__ void row_frag(v4f (&f)[D / 16], const T* row, int lg, bool ok) {
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const float4 x = ok ? load4_f32(row + 16 * s + 4 * lg) : float4{0.f, 0.f, 0.f, 0.f};
    f[s] = v4f{x.x, x.y, x.z, x.w};
  }
}

__device__ __forceinline__ v4f mfma_f32(float a, float b, const v4f& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void zero_frag(v4f (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) f[i] = v4f{0.f, 0.f, 0.f, 0.f};
}

// acc[t] (rows 16 t + 4 g + i of the LDS tile, column li) += tile . f^T over
// the first 16 NT rows
template <int D, int NT>
__device__ __forceinline__ void score_add(v4f (&acc)[NT], const float* lds, const v4f (&f)[D / 16],
                                          int li, int lg) {
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    v4f a[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
      a[t] = *reinterpret_cast<const v4f*>(lds + (16 * t + li) * (D + 4) + 16 * s + 4 * lg);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma_f32(a[t][i], f[s][i], acc[t]);
  }
}
template <int D, int NT>
__device__ __forceinline__ void score_tile(v4f (&acc)[NT], const float* lds, const v4f (&f)[D / 16],
                                           int li, int lg) {
  zero_frag(acc);
  score_add<D>(acc, lds, f, li, lg);
}

// out[dt] (d = 16 dt + 4 g + i, column li) += tile^T . w, w[t][i] the weight
// of tile row 16 t + 4 g + i
template <int D, int NT>
__device__ __forceinline__ void weigh_tile(v4f (&out)[D / 16], const float* lds, const v4f (&w)[NT],
                                           int li, int lg) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* row = lds + (16 * t + 4 * lg + i) * (D + 4) + li;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) out[dt] = mfma_f32(row[16 * dt], w[t][i], out[dt]);
    }
}

}  // namespace sa
