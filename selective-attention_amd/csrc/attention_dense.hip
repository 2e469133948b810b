// Dense prefill attention (gfx950, bf16): the causal, bidirectional and cross
// modes of attn_varlen at sizes that fill the chip, and SelectiveMHA's prefill
// over (batch, seq_len) rows.  Same formula and masks as the block-sparse
// kernel (attention.hip); what differs is the split of the work.
//
// A block owns 64 JT queries, 16 JT per wave, and every wave takes all 64 keys
// of a tile (two halves of 32), where the block-sparse kernel has 64 queries
// and two waves per query half that share the keys out and merge at the end.
// With JT = 2 a K / V tile in LDS serves twice the queries: half the L2 -> LDS
// traffic, barriers and per-tile overhead per score, and no merge.  The key
// bias enters as the MFMA's initial accumulator (bias / softmax_scale, one value
// per key row of the transposed score tile), which costs no instruction per
// score; the scale is folded into the exponent's argument as before.  Wave 0
// turns a tile's biases into raw score units on their way to its stage, once.
// What is left per score is an FMA, an exponential (half rate), an add and
// half a conversion: VALU busy 47 % of the cycles and the matrix cores 37 %,
// 13 % both; the rest is waits on LDS, barriers and, for launches of one to
// two resident rounds, the last round.
//
// JT = 1 (64 queries) takes SelectiveMHA launches that would leave the chip
// short of 128-query blocks.  Small packed launches keep the block-sparse
// kernel's dense form.
// Measured, block-sparse kernel -> here: causal rows b 4, H 16, L 8192 (ragged),
// D 64, the whole op: 574 -> 412 us; bidirectional, 4 sequences of 1500 to 4096,
// H 16, D 64, biased: 253 -> 219 us (2 us of either are the columns that raise
// their reference one by one).  Before that, 214 us, with a maximum per block
// instead of the sum test 234, the biases scaled by every wave 224, 168 instead
// of 128 VGPRs 226 us.
#include "attn_tile.h"
#include "prof.h"

namespace sa {
namespace {

constexpr int kKeys = 64;   // keys of a tile

template <int D>
constexpr int kStage = 2 * kKeys * D + 128;   // bf16: K tile, V tile, 64 fp32 biases

struct DenseArgs {
  const bf16 *q, *k, *v;
  const int32_t *cu, *cu_k;    // packed sequences (null: rows of L tokens)
  const int64_t* lengths;      // valid tokens of each row (null: all)
  const float* key_bias;       // packed: (H, Tk); rows: (rows, H, L)
  bf16* o;
  int nseq, grid_q, T, Tk, H, L;
  float scale_log2, inv_scale;   // softmax_scale log2(e), 1 / softmax_scale
};

// D = 64: 33 KB of LDS and a 128-VGPR budget (no spills), four blocks per CU;
// D = 128 (66 KB): two.
template <int D, bool BIAS, int MODE, bool ROWS, int JT>
__global__ __launch_bounds__(256, D == 64 ? 4 : 2) void dense_attn_kernel(DenseArgs a) {
  constexpr int BQ = 64 * JT, QW = 16 * JT;
  constexpr int DT = D / 16, KS = D / 32, IPW = D / 32;
  __shared__ __align__(16) bf16 stage0[kStage<D>];
  __shared__ __align__(16) bf16 stage1[kStage<D>];
  const int lid = xcd_swizzle(blockIdx.x, gridDim.x);
  const int h = lid / a.grid_q;
  const int gq = a.grid_q - 1 - (lid - h * a.grid_q);   // longest causal walks first
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const long rs = static_cast<long>(a.H) * D;

  // the block's sequence: [start, start + n), query block jq
  int start = 0, n = 0, jq = -1, seq = 0;
  if constexpr (ROWS) {
    const int nb = (a.L + BQ - 1) / BQ;
    seq = gq / nb;
    jq = gq - seq * nb;
    start = seq * a.L;
    n = a.lengths ? static_cast<int>(min(max(a.lengths[seq], int64_t{0}), int64_t{a.L})) : a.L;
    n = __builtin_amdgcn_readfirstlane(n);
    if (jq * BQ + BQ > n) {   // rows past the length are zeros
      for (int e = tid; e < BQ * (D / 8); e += 256) {
        const int r = jq * BQ + e / (D / 8);
        if (r >= n && r < a.L)
          *reinterpret_cast<uint4*>(a.o + (start + static_cast<long>(r)) * rs +
                                    static_cast<long>(h) * D + 8 * (e % (D / 8))) = uint4{0, 0, 0, 0};
      }
      if (jq * BQ >= n) return;
    }
  } else {
    for (int s0 = 0, first = 0; s0 < a.nseq && jq < 0; s0 += 64) {
      const int si = s0 + lane;
      int at = 0, nb = 0, len = 0;
      if (si < a.nseq) {
        at = min(max(a.cu[si], 0), a.T);
        len = min(max(a.cu[si + 1], at), a.T) - at;
        nb = (len + BQ - 1) / BQ;
      }
      int incl = nb;
#pragma unroll
      for (int o2 = 1; o2 < 64; o2 <<= 1) {
        const int t = __shfl_up(incl, o2, 64);
        if (lane >= o2) incl += t;
      }
      const int excl = first + incl - nb;
      const uint64_t hit = __ballot(si < a.nseq && gq >= excl && gq < excl + nb);
      if (hit) {
        const int l0 = __builtin_ctzll(hit);
        start = __builtin_amdgcn_readlane(at, l0);
        n = __builtin_amdgcn_readlane(len, l0);
        jq = gq - __builtin_amdgcn_readlane(excl, l0);
        seq = s0 + l0;
      }
      first += __builtin_amdgcn_readlane(incl, 63);
    }
    if (jq < 0) return;   // more query blocks than the packing holds
  }
  int kstart = start, nks = n;
  if constexpr (MODE == kCross) {
    kstart = min(max(a.cu_k[seq], 0), a.Tk);
    nks = min(max(a.cu_k[seq + 1], kstart), a.Tk) - kstart;
  }
  const bf16* kbase = a.k + static_cast<long>(kstart) * rs + static_cast<long>(h) * D;
  const bf16* vbase = a.v + static_cast<long>(kstart) * rs + static_cast<long>(h) * D;
  const float* bias = nullptr;
  if constexpr (BIAS)
    bias = ROWS ? a.key_bias + (static_cast<long>(seq) * a.H + h) * a.L
                : a.key_bias + static_cast<long>(h) * a.Tk + kstart;

  // this wave's queries qw0 .. qw0 + QW - 1; a lane holds column c of each 16
  const int qw0 = jq * BQ + QW * w;
  int qloc[JT];
  v8bf qf[JT][KS];
#pragma unroll
  for (int jt = 0; jt < JT; ++jt) {
    qloc[jt] = qw0 + 16 * jt + c;
    const bf16* qrow = a.q + (start + static_cast<long>(min(qloc[jt], n - 1))) * rs + static_cast<long>(h) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[jt][ks] = load_v8bf(qrow + 32 * ks + 8 * g);
  }
  // key tiles of the block, and of this wave
  const int nkb = (nks + kKeys - 1) / kKeys;
  const int nt = MODE == kCausalSelf ? min(nkb, (min(n, (jq + 1) * BQ) + kKeys - 1) / kKeys) : nkb;
  const int wt = qw0 >= n ? 0 : MODE == kCausalSelf ? min(nt, (qw0 + QW - 1) / kKeys + 1) : nt;

  // DMA: lane l of instruction i fills tile bytes 1024 (IPW w + i) + 16 l, i.e.
  // row `row`, stored chunk `ch` (holding chunk ch ^ swizzle(row)); rows past the
  // key range repeat its last key (masked)
  int dma_k[IPW], dma_v[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int pos = ((w * IPW + i) << 10) + (lane << 4);
    const int row = pos / (2 * D), ch = (pos % (2 * D)) >> 4;
    dma_k[i] = row * static_cast<int>(rs) + 8 * (ch ^ k_swz<D>(row));
    dma_v[i] = row * static_cast<int>(rs) + 8 * (ch ^ v_swz<D>(row));
  }
  const uint32_t lds_st0 = lds_addr(stage0), lds_st1 = lds_addr(stage1);
  const uint32_t lds_wave = static_cast<uint32_t>(w * IPW) << 10;
  auto issue = [&](int kb, uint32_t st) __attribute__((always_inline)) {
    const int k0 = kb * kKeys, nk = min(kKeys, nks - k0);
    const uint32_t kt = st + lds_wave, vt = kt + 2 * kKeys * D;
    const bf16* kb0 = kbase + static_cast<long>(k0) * rs;
    const bf16* vb0 = vbase + static_cast<long>(k0) * rs;
    if (nk == kKeys) {
#pragma unroll
      for (int i = 0; i < IPW; ++i) {
        dma_lds16(kb0, 2u * dma_k[i], kt + (i << 10));
        dma_lds16(vb0, 2u * dma_v[i], vt + (i << 10));
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int pos = ((w * IPW + i) << 10) + (lane << 4);
      const int row = pos / (2 * D), rr = min(row, nk - 1), ch = (pos % (2 * D)) >> 4;
      dma_lds16(kb0, 2u * (rr * static_cast<int>(rs) + 8 * (ch ^ k_swz<D>(row))), kt + (i << 10));
      dma_lds16(vb0, 2u * (rr * static_cast<int>(rs) + 8 * (ch ^ v_swz<D>(row))), vt + (i << 10));
    }
  };

  SoftmaxCol col[JT];
  v4f acc[JT][DT];
#pragma unroll
  for (int jt = 0; jt < JT; ++jt) {
    col[jt] = SoftmaxCol{-1.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[jt][t] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  // the next tile's biases, one per lane of wave 0, on their way to its stage in raw score units
  float bnext = 0.f;
  auto load_bias = [&](int kb) __attribute__((always_inline)) {
    if constexpr (BIAS) {
      if (w == 0) bnext = bias[min(kb * kKeys + lane, nks - 1)];
    }
  };
  auto store_bias = [&](bf16* st) __attribute__((always_inline)) {
    if constexpr (BIAS) {
      if (w == 0) reinterpret_cast<float*>(st + 2 * kKeys * D)[lane] = bnext * a.inv_scale;
    }
  };
  // per-lane pieces of the swizzled LDS addresses (rows 32 apart share them)
  int krow_off[2], kswz[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = key_of_row(u, c);
    krow_off[u] = r * D;
    kswz[u] = k_swz<D>(r);
  }
  const int vr = 8 * g + (c >> 2), vswz = v_swz<D>(vr);
  const int vhalf = 4 * (c & 1), vchunk = (c & 3) >> 1;

  auto step = [&](int e, const bf16* Ks, bf16* nst, uint32_t nxt) __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vm_wait<0>());
    __builtin_amdgcn_s_barrier();   // tile e has landed; every wave is done with tile e - 1
    asm volatile("" ::: "memory");
    if (e + 1 < nt) {
      store_bias(nst);   // (loaded a step ago)
      issue(e + 1, nxt);
      if (e + 2 < nt) load_bias(e + 2);
    }
    if (e < wt) {
      const bf16* Vs = Ks + kKeys * D;
      const int k0 = e * kKeys;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int kh0 = k0 + 32 * hh;   // the half's first key
        if (MODE == kCausalSelf ? kh0 > qw0 + QW - 1 : kh0 >= nks) break;
        // masks or an exempt key in this half: causal, from the wave's diagonal
        // on; otherwise past the key range, or the exempt key itself
        const bool edge = MODE == kCausalSelf ? kh0 + 31 >= qw0
                          : kh0 + 32 > nks ||
                                (BIAS && (MODE == kCross ? kh0 == 0
                                                         : kh0 < qw0 + QW && kh0 + 32 > qw0));
        v4f b0 = v4f{0.f, 0.f, 0.f, 0.f}, b1 = b0;   // biases of keys 8g .. 8g + 7, in raw score units
        if constexpr (BIAS) {
          const float* bs = reinterpret_cast<const float*>(Vs + kKeys * D) + 32 * hh + 8 * g;
          b0 = *reinterpret_cast<const v4f*>(bs);
          b1 = *reinterpret_cast<const v4f*>(bs + 4);
        }
        v8bf kfr[2][KS];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            kfr[u][ks] = load_v8bf(Ks + 32 * hh * D + krow_off[u] + 8 * ((4 * ks + g) ^ kswz[u]));
        v4f sc[JT][2];
        if (!edge) {
#pragma unroll
          for (int jt = 0; jt < JT; ++jt) {
            sc[jt][0] = mfma_bf16(kfr[0][0], qf[jt][0], b0);
            sc[jt][1] = mfma_bf16(kfr[1][0], qf[jt][0], b1);
          }
        } else {
          const v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int jt = 0; jt < JT; ++jt) {
            sc[jt][0] = mfma_bf16(kfr[0][0], qf[jt][0], z);
            sc[jt][1] = mfma_bf16(kfr[1][0], qf[jt][0], z);
          }
        }
#pragma unroll
        for (int ks = 1; ks < KS; ++ks)
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int jt = 0; jt < JT; ++jt) sc[jt][u] = mfma_bf16(kfr[u][ks], qf[jt][ks], sc[jt][u]);
        if (edge) {
#pragma unroll
          for (int jt = 0; jt < JT; ++jt)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int key = kh0 + 8 * g + 4 * u + i;
                float val = sc[jt][u][i];
                if constexpr (BIAS) {
                  const bool exempt = MODE == kCross ? key == 0 : key == qloc[jt];
                  val += exempt ? 0.f : (u ? b1[i] : b0[i]);
                }
                const bool ok = MODE == kCausalSelf ? key <= qloc[jt] : key < nks;
                sc[jt][u][i] = ok ? val : kNegInf;
              }
        }
        v8bf vfr[DT];   // read before the softmax: their latency passes under it
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
          const bf16* p = Vs + (32 * hh + vr) * D + 8 * ((2 * t + vchunk) ^ vswz) + vhalf;
          const v4i16 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p));
          const v4i16 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + 4 * D));
          vfr[t] = __builtin_bit_cast(v8bf, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
        }
        __builtin_amdgcn_sched_barrier(0);
        v8bf pb[JT];
#pragma unroll
        for (int jt = 0; jt < JT; ++jt) {
          pb[jt] = softmax_col<DT>(sc[jt], acc[jt], col[jt], a.scale_log2);
        }
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int jt = 0; jt < JT; ++jt) acc[jt][t] = mfma_bf16(vfr[t], pb[jt], acc[jt][t]);
      }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kLgkmWait0);
  };
  // the query fragments have arrived before the loop: nothing the compiler
  // tracks is in flight inside it
  __builtin_amdgcn_s_waitcnt(vm_wait<0>());
  if (nt > 0) {
    load_bias(0);
    store_bias(stage0);
    // complete before the first barrier, as a step's own stores are by the wait
    // that ends it: neither the barrier nor the wait on the DMA covers them
    __builtin_amdgcn_s_waitcnt(kLgkmWait0);
    issue(0, lds_st0);
    if (nt > 1) load_bias(1);
  }
  for (int e = 0; e < nt; e += 2) {
    step(e, stage0, stage1, lds_st1);
    if (e + 1 >= nt) break;
    step(e + 1, stage1, stage0, lds_st0);
  }
  __builtin_amdgcn_s_barrier();   // every wave is done with the tiles
  asm volatile("" ::: "memory");
  if (qw0 >= n) return;
  // normalised rows go out through LDS as whole rows: [QW rows][D] bf16 per
  // wave, 16-byte chunk ch of row r at ch ^ (r % chunks)
  constexpr int RCH = D / 8;
  static_assert(4 * QW * D <= kStage<D>, "output rows fit a stage");
  bf16* ot = stage0 + w * QW * D;
#pragma unroll
  for (int jt = 0; jt < JT; ++jt) {
    float lt = col[jt].l;
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    const int r = 16 * jt + c;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int ch = 2 * t + (g >> 1);
      *reinterpret_cast<uint2*>(ot + r * D + 8 * (ch ^ (r & (RCH - 1))) + 4 * (g & 1)) =
          uint2{pack_bf16x2(acc[jt][t][0] * inv, acc[jt][t][1] * inv),
                pack_bf16x2(acc[jt][t][2] * inv, acc[jt][t][3] * inv)};
    }
  }
  asm volatile("" ::: "memory");
  bf16* obase = a.o + (start + static_cast<long>(qw0)) * rs + static_cast<long>(h) * D;
#pragma unroll
  for (int i = 0; i < QW * RCH / 64; ++i) {
    const int e = lane + 64 * i, r = e / RCH, ch = e % RCH;
    if (qw0 + r < n)
      *reinterpret_cast<uint4*>(obase + r * rs + 8 * ch) =
          *reinterpret_cast<const uint4*>(ot + r * D + 8 * (ch ^ (r & (RCH - 1))));
  }
}

template <int D, int MODE, bool ROWS, int JT>
int launch_dense(const DenseArgs& a, hipStream_t s) {
  const long blocks = static_cast<long>(a.H) * a.grid_q;
  ProfScope prof_(MODE == kCausalSelf ? "dense_attn_fwd" : MODE == kFullSelf ? "attn_full_fwd" : "attn_cross_fwd", s);
  auto kernel = dense_attn_kernel<D, true, MODE, ROWS, JT>;
  if constexpr (!ROWS) {   // (rows always come with their log-gates)
    if (!a.key_bias) kernel = dense_attn_kernel<D, false, MODE, ROWS, JT>;
  }
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, s, a);
  SA_CHECK_LAUNCH("dense_attn");
  return 0;
}

}  // namespace

// 128-query blocks: two and more of them for every CU.  The tokens are counted,
// not the sequences: a pack of short ones leaves waves without queries and
// empty blocks behind, and is still the faster here, since a tile's 64-query
// blocks (four waves that share its keys) and their merge cost more.  Packs past
// this line, block-sparse kernel -> here, H 16, D 64, causal with biases: 256
// sequences of 16 tokens 25.4 -> 21.5 us, 32: 31 -> 25, 64: 42 -> 38, 100: 66 ->
// 50, 200: 168 -> 106; 1024 of 32: 195 -> 158, of 100: 428 -> 302 us.  Over 4 and
// 16 heads, both head_dims, all modes, 64 to 1024 sequences of 16 to 1000
// tokens: 0.93 to 2.1 times as fast, 1.3 in the middle (below 1 at 4 heads and
// 256 sequences of 80 to 128 tokens alone).
bool dense_attn_ok(int num_heads, int total_q) {
  return static_cast<long>(num_heads) * (total_q / 128) >= 512;
}

int launch_dense_varlen(int mode, int D, const void* q, const void* k, const void* v,
                        const int32_t* cu, const int32_t* cu_k, int nseq, const float* key_bias,
                        void* o, int T, int Tk, int H, float scale_log2, hipStream_t s) {
  DenseArgs a{};
  a.q = static_cast<const bf16*>(q);
  a.k = static_cast<const bf16*>(k);
  a.v = static_cast<const bf16*>(v);
  a.cu = cu;
  a.cu_k = cu_k;
  a.key_bias = key_bias;
  a.o = static_cast<bf16*>(o);
  a.nseq = nseq;
  a.grid_q = T / 128 + nseq;   // at least the packing's query blocks
  a.T = T;
  a.Tk = Tk;
  a.H = H;
  a.scale_log2 = scale_log2;
  a.inv_scale = kLog2e / scale_log2;
  if (D == 128) {
    if (mode == kCausalSelf) return launch_dense<128, kCausalSelf, false, 2>(a, s);
    if (mode == kFullSelf) return launch_dense<128, kFullSelf, false, 2>(a, s);
    return launch_dense<128, kCross, false, 2>(a, s);
  }
  if (mode == kCausalSelf) return launch_dense<64, kCausalSelf, false, 2>(a, s);
  if (mode == kFullSelf) return launch_dense<64, kFullSelf, false, 2>(a, s);
  return launch_dense<64, kCross, false, 2>(a, s);
}

}  // namespace sa

extern "C" int sa_mha_prefill_fwd(int dtype, const void* q, const void* k, const void* v,
                                  const float* log_gate, const int64_t* lengths, int batch,
                                  int seq_len, int num_heads, int head_dim, float softmax_scale,
                                  void* o, void* stream) {
  SA_CHECK_ARG(dtype == sa::kBF16, "sa_mha_prefill_fwd: only bfloat16 is supported");
  SA_CHECK_ARG(head_dim == 64 || head_dim == 128, "sa_mha_prefill_fwd: head_dim %d not in {64,128}",
               head_dim);
  SA_CHECK_ARG(batch >= 0 && seq_len >= 0 && num_heads > 0 &&
                   static_cast<int64_t>(batch) * seq_len < (1LL << 31),
               "sa_mha_prefill_fwd: bad sizes");
  SA_CHECK_ARG(q && k && v && log_gate && o, "sa_mha_prefill_fwd: null pointer");
  SA_CHECK_ARG(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                 reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(o)) & 15) == 0,
               "sa_mha_prefill_fwd: q, k, v and o must be 16-byte aligned");
  if (batch == 0 || seq_len == 0) return 0;
  const float scale = softmax_scale > 0.f ? softmax_scale : 1.0f / sqrtf(static_cast<float>(head_dim));
  sa::DenseArgs a{};
  a.q = static_cast<const sa::bf16*>(q);
  a.k = static_cast<const sa::bf16*>(k);
  a.v = static_cast<const sa::bf16*>(v);
  a.lengths = lengths;
  a.key_bias = log_gate;
  a.o = static_cast<sa::bf16*>(o);
  a.nseq = batch;
  a.H = num_heads;
  a.L = seq_len;
  a.T = a.Tk = batch * seq_len;
  a.scale_log2 = scale * sa::kLog2e;
  a.inv_scale = 1.0f / scale;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool wide = sa::dense_attn_ok(num_heads, a.T);
  a.grid_q = batch * ((seq_len + (wide ? 127 : 63)) / (wide ? 128 : 64));
  if (head_dim == 128)
    return wide ? sa::launch_dense<128, sa::kCausalSelf, true, 2>(a, s)
                : sa::launch_dense<128, sa::kCausalSelf, true, 1>(a, s);
  return wide ? sa::launch_dense<64, sa::kCausalSelf, true, 2>(a, s)
              : sa::launch_dense<64, sa::kCausalSelf, true, 1>(a, s);
}
