// Pieces shared by the prefill attention kernels (attention.hip: block-sparse
// and small dense launches; attention_dense.hip: dense modes).
#pragma once

#include "common.h"

namespace sa {

constexpr float kNegInf = -__builtin_huge_valf();

// MODE (which keys a query sees, and which key is exempt from the bias):
//   kCausalSelf  keys j <= i of the query's own sequence; j = i exempt
//   kFullSelf    every key of the query's own sequence;  j = i exempt
//   kCross       every key of the sequence's key range cu_k[s]..cu_k[s+1]
//                (k, v, key_bias indexed by key token); key 0 exempt
constexpr int kCausalSelf = 0, kFullSelf = 1, kCross = 2;

// chunk permutations of row r (16-byte chunks; D = 128: 16 per row, D = 64:
// 8).  The K tile is read as MFMA A fragments (16 rows key_of_row(kt, 0..15),
// one chunk per 16-lane group), the V tile by ds_read_b64_tr_b16 (rows
// 8g + 0..3 and + 4, one chunk pair per group), so each gets its own
// permutation; both were chosen with the LDS bank-conflict counter
// (SQ_LDS_BANK_CONFLICT = 0 for these read sets on gfx950).  The V
// permutation never uses bit 2 of r, so rows r and r + 4 (the two halves of
// one transpose read) share it.
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  if constexpr (D == 128) return (r & 3) | (((r >> 3) & 3) << 2);
  else return (((r >> 1) & 1) << 2) | (((r >> 3) & 1) << 1) | ((r >> 4) & 1);
}
template <int D>
__device__ __forceinline__ int v_swz(int r) {
  if constexpr (D == 128) return ((r & 3) << 2) | (((r >> 3) & 1) << 1) | ((r >> 4) & 1);
  else return (((r >> 1) & 1) << 2) | (((r >> 3) & 1) << 1) | ((r >> 4) & 1);
}

// Online softmax of the block-sparse kernel, with a lazy reference.  s[kt][i]
// holds log2-domain scores of this lane's keys for query column lane & 15 (-inf
// where masked).  The running reference m of a column (log2 domain, shared by
// its four lane groups) is raised, and O and the partial sums rescaled, only when
// some score exceeds it by more than 2^8: the common block needs no cross-lane
// reduction at all, and probabilities stay <= 256.  l is this lane's partial
// row sum (its own keys); the four lane groups' parts are added at the end.
// The scores may come unscaled: the log2-domain score is s * sc (sc > 0), and
// the scale is folded into the exponent's argument.
// (softmax_col's sum test computes a row's first block twice; a block-sparse
// row has 16 blocks at most: rows of 214 to 1284 tokens, H 16, took 350 us
// with it and take 337 so at D = 128, 198 and 186 at D = 64, against 683 and
// 687 us at 512 to 8192 tokens, D = 128.)
template <int KT, int DT>
__device__ __forceinline__ void softmax_lazy(v4f (&s)[KT], v4f (&o)[DT], float& m, float& l,
                                             float sc = 1.0f) {
  float mx = kNegInf;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kt][i]);
  mx *= sc;
  if (__ballot(mx > m + 8.0f)) {
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (mx > m + 8.0f) {   // the column's new reference
      if (m != kNegInf) {   // (while m = -inf, every p so far was 0: l and o are 0)
        const float alpha = fast_exp2(m - mx);
        l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= alpha;
      }
      m = mx;
    }
  }
  // masked scores are -inf; a column without any admissible key yet keeps
  // m = -inf and only -inf scores, so a zero reference gives p = 0 there
  const float mref = m == kNegInf ? 0.0f : m;
  float sum = 0.0f;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = fast_exp2(fmaf(s[kt][i], sc, -mref));
      s[kt][i] = p;
      sum += p;
    }
  l += sum;
}

// Online softmax of one query column of the dense kernel (rows of many blocks),
// with a lazy reference (log2 domain): p =
// 2^(score - reference), the reference raised, and O and the lane's partial
// row sum rescaled, only when needed.  A p above 2^8 shows in the sum of the
// lane's eight p, which the row sum needs anyway: no maximum is taken in the
// common block.  (The sum passes 2^8 without a single p above it at times;
// the reference is then raised early, to the same effect.)  A test that sends
// the first block straight to the maximum costs the others more: 405 -> 435 us
// (causal rows, b 4, H 16, L 8192).
struct SoftmaxCol {
  float limit;   // sums above this raise the reference: 2^8, or -1 while there is none
  float neg;     // minus the reference; 0 while there is none
  float l;       // the lane's sum of p
};
__device__ __forceinline__ float exp_sum(const v4f (&s)[2], v4f (&p)[2], float sc, float neg) {
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) p[u][i] = fast_exp2(fmaf(s[u][i], sc, neg));
  return ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) + ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
}
template <int DT>
__device__ __forceinline__ v8bf softmax_col(const v4f (&s)[2], v4f (&o)[DT], SoftmaxCol& c, float sc) {
  v4f p[2];
  float sum = exp_sum(s, p, sc, c.neg);
  const uint64_t vote = __ballot(sum > c.limit);
  if (vote) {
    // a column's four lane groups share the reference and decide by their own
    // sums alone: a row's bits do not depend on the rows beside it
    const uint32_t half = static_cast<uint32_t>(vote) | static_cast<uint32_t>(vote >> 32);
    const bool mine = ((half | half >> 16) >> (threadIdx.x & 15)) & 1;
    float mx = kNegInf;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[u][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float ref = mx * sc;
    const bool up = mine && (c.limit < 0.f ? mx > kNegInf : ref > -c.neg);
    if (up) {
      if (c.limit > 0.f) {
        const float alpha = fast_exp2(-c.neg - ref);
        c.l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= alpha;
      }
      c.neg = -ref;
      c.limit = 256.0f;
    }
    // (a column without a reference has met masked keys, whose p are 0, and
    // scores that are no numbers, whose p have to stay)
    sum = exp_sum(s, p, sc, c.neg);
  }
  c.l += sum;
  return pack_p(p[0], p[1]);
}

// dense attention on 128-query blocks (attention_dense.hip).  Packed sequences
// (cu, and cu_k for kCross) of the modes above:
bool dense_attn_ok(int num_heads, int total_q);
int launch_dense_varlen(int mode, int D, const void* q, const void* k, const void* v,
                        const int32_t* cu, const int32_t* cu_k, int nseq, const float* key_bias,
                        void* o, int T, int Tk, int H, float scale_log2, hipStream_t s);

}  // namespace sa
