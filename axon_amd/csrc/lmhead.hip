// (a) Fused LM head: per-token log-prob and entropy, and its backward, without
// materialising the [tokens x vocab] logits.
//
// Forward    logits^T tile = W[vocab tile] . hidden[token tile]^T on MFMA; the
//            epilogue folds each tile into per-token (max, sum exp, sum logit*exp)
//            partials; a small kernel merges partials and adds the label logit.
// Backward   per vocab chunk:
//   B1  recompute the logits tile (or decode the forward's stash), form dlogit in
//       registers, write it as bf16 dl[token][vocab];
//   B2  dHidden[token][h] (+)= sum_v dl[token][v]  * W[v][h]
//   B3  dWeight[v][h]      =  sum_t dl[t][v]       * hiddenT[h][t]
// hiddenT is a bf16 transpose made once per call.  B2 reads the weight and B3 reads
// dl as they lie, K-major for these products (gemm_nt.h).  Small hidden sizes and
// vocabularies that are no multiple of 8 get a second, vocab-major copy
// dlT[vocab][token] from B1 for B3.
#include "common.h"
#include "dweight_rows.h"
#include "gemm_nt.h"
#include <vector>

namespace axon {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ----------------------------------------------------------------------------
// Forward: tile epilogue -> partial statistics
// ----------------------------------------------------------------------------
struct FwdParams {
  // [parts][n_tokens][3]: running max in log2 units of the scaled logit, sum 2^(x*c - max), sum (x*c - max) * 2^(x*c - max);
  // side by side, so that sixteen tokens of a part are 192 contiguous bytes for the kernel that folds them
  float* stats;
  float* pm;   // [parts][n_tokens]: the max once more, where the backward reads it (null: it does not)
  int n_tokens, vocab;
  float c;     // inv_temperature * log2(e)
  float cap, inv_cap;  // logit soft-capping cap * tanh(logit / cap) (SOFTCAP kernels only)
  uint4* stash;        // kernels that keep something for the backward: the stash or the logits, see below
  int halved;          // the walk's last tiles that are computed in two halves of 128 vocabulary rows
};
// What a forward leaves for its backward beside the statistics.
enum Keep { kKeepNone, kKeepStash, kKeepLogits };

// What a stashing forward leaves for the backward: for every logit, w = 2^(y - M) as fp16, where
// y is the scaled logit in log2 units and M the maximum of y over the 128 vocabulary rows of the
// same token that one wavefront holds (the `pm` partial of that (token, 128-row part)), so that
// 0 <= w <= 1 and softmax = w * 2^(M - logsumexp).  fp16 keeps eleven bits of w whatever the size
// of the logit; entries below 2^-24 of their part's maximum read back as 0 and contribute no
// gradient.  Each wavefront's 128 x 128 sub-tile is stored in accumulator order, 16 bytes per lane
// and store (two 16-row blocks), every store one contiguous kilobyte:
//   uint4 index = ((tile * 4 + wave) * 32 + j * 4 + i / 2) * 64 + lane,   tile = tm * tiles_n + tn.
// Vocabulary rows beyond the matrix are stored as 0.
constexpr int64_t kStashTileBytes = 131072;
constexpr int kStashWaveVecs = 2048;  // uint4 per wavefront sub-tile

// kKeepLogits: the accumulators themselves (fp32, before temperature and soft-capping), so that the backward forms
// the very dlogits that it would form from recomputed logits, without the product.  Accumulator order again, one
// contiguous kilobyte per store:  uint4 index = ((tile * 4 + wave) * 64 + j * 8 + i) * 64 + lane.
constexpr int64_t kLogitsTileBytes = 262144;
constexpr int kLogitsWaveVecs = 4096;  // uint4 per wavefront sub-tile

__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  const f16x2 r = __builtin_convertvector(v, f16x2);  // round to nearest even
  return *reinterpret_cast<const uint32_t*>(&r);
}
__device__ __forceinline__ void unpack_f16(uint32_t w, float& lo, float& hi) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  const f16x2 r = *reinterpret_cast<const f16x2*>(&w);
  lo = (float)r[0];
  hi = (float)r[1];
}

// tanh(u) = 1 - 2 / (e^(2u) + 1): saturates cleanly at +-1 (2^x -> inf gives rcp 0, 2^x -> 0 gives -1)
__device__ __forceinline__ float fast_tanh(float u) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(fast_exp2(u * (2.f * kLog2e)) + 1.f);
}

constexpr float kEmptyMax = -3.0e38f;  // running max of a partial that saw no vocabulary row

// Partial statistics of a set of scaled logits y = logit * c (log2 units):
//   M = reference (the set's max), s = sum 2^(y-M), e = sum 2^(y-M) * (y-M).
// Merge (M2,s2,e2) into (M,s,e) under the common reference Mn >= M, M2.
__device__ __forceinline__ void merge_stats(float M, float& s, float& e, float M2, float s2,
                                            float e2, float Mn) {
  const float d1 = M - Mn, d2 = M2 - Mn;
  const float f1 = fast_exp2(d1), f2 = fast_exp2(d2);
  e = fmaf(f1, fmaf(s, d1, e), f2 * fmaf(s2, d2, e2));  // written out: the same roundings wherever this is inlined
  s = fmaf(s, f1, s2 * f2);
}

// Exchange of 16-lane rows between two registers: row 1 of a with row 0 of b and row 3 of a with row 2 of b
// (swap_rows16), rows 2 and 3 of a with rows 0 and 1 of b (swap_rows32); one vector instruction each, where a shuffle
// would take a trip through the LDS crossbar with a wait behind it.
// Written as instructions: through the builtins the compiler takes the two results of a swap for one
// value and folds op(a, b) to op(a, a).  The s_nop covers the wait states the swaps need after a
// vector instruction has written their operands.
__device__ __forceinline__ void swap_rows16(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void swap_rows32(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}

// Four values reduced over the four rows of the wavefront (lanes l, l^16, l^32, l^48: the four lanes that hold the same
// token) at once: row r of the result has the reduction of v[r].  The halves of a swap carry two values, so that four
// take three swaps; an all-reduce of each by itself took eight, and a store of sixteen lanes each behind it.  The same
// pairs in the same order as the xor-16, xor-32 butterfly, so sums come out bit for bit the same.
template <class Op>
__device__ __forceinline__ float rows_reduce4(const float (&v)[4], Op op) {
  float a = v[0], b = v[1], c = v[2], d = v[3];
  swap_rows16(a, b);  // a: a0 b0 a2 b2, b: a1 b1 a3 b3
  swap_rows16(c, d);
  float x = op(a, b), y = op(c, d);
  swap_rows32(x, y);  // x: a01 b01 c01 d01, y: a23 b23 c23 d23
  return op(x, y);
}
// The way back: row r of x in every row of o[r].
__device__ __forceinline__ void rows_spread4(float x, float (&o)[4]) {
  float y = x;
  swap_rows32(x, y);  // x: x0 x1 x0 x1, y: x2 x3 x2 x3
  o[0] = o[1] = x;
  o[2] = o[3] = y;
  swap_rows16(o[0], o[1]);
  swap_rows16(o[2], o[3]);
}

// Fold a logits tile of 32 * BM vocabulary rows x 256 tokens into per-token partials, one per 128 rows.  BM 8: a
// whole tile, whose wavefronts have a part each; BM 4: the half `half` of one, whose part the wavefronts 0 and 2 (1
// and 3) share: its maximum and its sums go through LDS, in the order in which one wavefront of a whole tile adds
// them up (a lane adds the first four and the last four 16-row blocks apart), so that the results do not depend on
// how a tile was computed. MASKED: some rows of the tile lie beyond the vocabulary; they are excluded by predicate —
// their accumulators hold finite values.  STASH: also store every 2^(y - M) for the backward (`kept_tile`: the part's
// share of the tile, its two sub-tiles one behind the other, already offset by the lane).  BN: columns of 16 tokens per
// wavefront, fewer than 8 where the call has no more (narrow tiles).
//
// Bound by the issue of vector instructions, one wavefront to a SIMD and the matrix pipes idle: five per logit (maximum
// for two, read of the accumulator, fma, exponential, sum, product sum), of which the exponential takes four times as
// long.  The exponentials of a block run between the sums of the block before it, so that none of its users waits for
// one, and the reductions over lanes are done for four columns at a time: 1600 instructions where there were 2030 and 330
// wait states.  8192 x 896 x 151936 forward 1866 -> 1818 us, 187 tokens 88.8 -> 85.5 (one card each).
template <bool MASKED, bool SOFTCAP, Keep KEEP, int BM, int BN>
__device__ __forceinline__ void fwd_epilogue(AccTileOf<BM, BN>& acc, const FwdParams& p, const LanePos& lp,
                                             const TilePos& t, int part, uint4* kept_tile, float* lds) {
  constexpr bool STASH = KEEP == kKeepStash;
  constexpr bool kHalf = BM < kBlocks;
  constexpr int kRun = kBlocks / 2;  // blocks that a lane adds up in one go
  constexpr int kGroups = (BN + 3) / 4;
  auto cols = [](int g) { return BN - 4 * g < 4 ? BN - 4 * g : 4; };  // of group g
  auto add = [](float a, float b) { return a + b; };
  auto row_ok = [&](int i, int r) { return !MASKED || t.m0 + lp.m<BM>(i, r) < p.vocab; };
  // where column j of this wavefront is kept: the sub-tiles there are those of the whole tile, 128 columns each
  auto kept_col = [&](int j) {
    constexpr int kCol = (STASH ? kStashWaveVecs : kLogitsWaveVecs) / kBlocks;
    const int at = BN == kBlocks ? j : lp.wn * BN + j;
    return kept_tile + (int64_t)((BN == kBlocks ? lp.wn * kBlocks : 0) + at) * kCol;
  };
  // logits for the backward: written once, read once, long after: past the caches
  auto keep_logits = [&](int i, int j, const float (&z)[4]) {
    const acc4 v = {z[0], z[1], z[2], z[3]};
    __builtin_nontemporal_store(v, reinterpret_cast<acc4*>(kept_col(j) + (kHalf ? lp.wm * BM + i : i) * 64));
  };
  // columns 4 g .. 4 g + 3, read from the accumulators where they are needed (SOFTCAP: through cap * tanh(. / cap))
  float x[kHalf ? kGroups : 1][BM][4][4];
  auto take = [&](int g) {
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q >= cols(g)) continue;
        float(&z)[4] = x[kHalf ? g : 0][i][q];
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = read_acc(acc[i][4 * g + q], r);
        if (SOFTCAP) {
          if (KEEP == kKeepLogits) keep_logits(i, 4 * g + q, z);  // what is kept is not capped
#pragma unroll
          for (int r = 0; r < 4; ++r) z[r] = p.cap * fast_tanh(z[r] * p.inv_cap);
        }
      }
  };
  // the part's maxima over this wavefront's rows of columns 4 g .. 4 g + 3, row r of the lanes that of column 4 g + r;
  // the four lanes that hold the same token (lane ^ 16, lane ^ 32) share one reference
  auto max_of = [&](int g) {
    float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (q < cols(g)) mx[q] = row_ok(i, r) ? fmaxf(mx[q], x[kHalf ? g : 0][i][q][r]) : mx[q];
    return rows_reduce4(mx, [](float a, float b) { return fmaxf(a, b); });
  };
  // columns 4 g .. 4 g + 3 are 64 consecutive tokens, one per lane (the last group of six columns has 32)
  auto write = [&](int g, float M, const float (&s)[4], const float (&e)[4]) {
    const float sum = rows_reduce4(s, add), prod = rows_reduce4(e, add);
    const int n = t.n0 + lp.wn * BN * kBlk + g * 64 + lp.lane;
    if (n < p.n_tokens && (cols(g) == 4 || lp.lane < cols(g) * kBlk)) {
      const int64_t at = (int64_t)part * p.n_tokens + n;
      float* const o = p.stats + at * 3;
      o[0] = M;
      o[1] = sum;
      o[2] = prod;
      if (STASH) p.pm[at] = M;
    }
  };
  float* const mine = lds + lp.wave * 1024 + lp.lane;  // per wavefront: 8 x 64 of each of the two sums
  const float* const other = lds + (lp.wave ^ 2) * 1024 + lp.lane;
  float mxs[kGroups];
  if (kHalf) {
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      take(g);
      mine[g * 64] = mxs[g] = max_of(g);
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < kGroups; ++g) mxs[g] = fmaxf(mxs[g], other[g * 64]);
    __syncthreads();
  }
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    if (!kHalf) take(g);
    const float mx = kHalf ? mxs[g] : max_of(g);
    mxs[g] = (MASKED && mx == -INFINITY) ? kEmptyMax : mx * p.c;
    float M[4], s4[4] = {}, e4[4] = {};
    rows_spread4(mxs[g], M);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q >= cols(g)) continue;
      const int j = 4 * g + q;
      float s[2] = {0.f, 0.f}, e[2] = {0.f, 0.f};
      uint32_t hw[BM][2];
      float y[3][4], w[2][4];  // blocks i + 1, i, i - 1; i, i - 1
      auto rel = [&](int i, int r) { return fmaf(x[kHalf ? g : 0][i][q][r], p.c, -M[q]); };  // scaled logit relative to the max, <= 0
#pragma unroll
      for (int r = 0; r < 4; ++r) y[0][r] = rel(0, r);
#pragma unroll
      for (int i = 0; i <= BM; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // one store under the arithmetic of a block: all of them at the epilogue's head make it wait for their way out
          // (GSPO step of 6007 x 896 x 151936 5443 -> 5362 us)
          if (KEEP == kKeepLogits && !SOFTCAP && i < BM && r == 0) keep_logits(i, j, x[kHalf ? g : 0][i][q]);
          if (i < BM) w[i % 2][r] = row_ok(i, r) ? fast_exp2(y[i % 3][r]) : 0.f;
          if (i > 0) {
            const int b = i - 1;
            s[b / kRun] += w[b % 2][r];
            e[b / kRun] = fmaf(w[b % 2][r], y[b % 3][r], e[b / kRun]);
          }
          if (i + 1 < BM) y[(i + 1) % 3][r] = rel(i + 1, r);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (STASH && i < BM) {
          hw[i][0] = pack_f16(w[i % 2][0], w[i % 2][1]);
          hw[i][1] = pack_f16(w[i % 2][2], w[i % 2][3]);
        }
      }
      if (STASH) {
#pragma unroll
        for (int ip = 0; ip < BM / 2; ++ip)
        {  // written once, read once by the backward: kept out of the way of the operand slices in L2
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
          const u32x4 x = {hw[2 * ip][0], hw[2 * ip][1], hw[2 * ip + 1][0], hw[2 * ip + 1][1]};
          const int at = kHalf ? lp.wm * (BM / 2) + ip : ip;
          __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(kept_col(j) + at * 64));
        }
      }
      s4[q] = kHalf ? s[0] : s[0] + s[1];
      e4[q] = kHalf ? e[0] : e[0] + e[1];
      if (kHalf) {
        mine[j * 64] = s4[q];
        mine[(kBlocks + j) * 64] = e4[q];
      }
    }
    if (!kHalf) write(g, mxs[g], s4, e4);
  }
  if (kHalf) {
    __syncthreads();
    if (lp.wm == 0) {
#pragma unroll
      for (int g = 0; g < kGroups; ++g) {
        float s4[4] = {}, e4[4] = {};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (q >= cols(g)) continue;
          s4[q] = mine[(4 * g + q) * 64] + other[(4 * g + q) * 64];
          e4[q] = mine[(kBlocks + 4 * g + q) * 64] + other[(kBlocks + 4 * g + q) * 64];
        }
        write(g, mxs[g], s4, e4);
      }
    }
  }
}

// One tile (BM 8), or the half `half` of one (BM 4: t.m0 is its first row).  SOFTCAP: the logits go through
// cap * tanh(. / cap) before the statistics (fused_linear.py:19-23).
template <class Loop, int BM, bool SOFTCAP, Keep KEEP>
__device__ __forceinline__ void fwd_tile(const GemmOperands& g, const FwdParams& p, const TilePos& t, int tile, int part0,
                                         int half, char* smem) {
  constexpr bool kHalf = BM < kBlocks;
  constexpr int BN = Loop::kBN;
  AccTileOf<BM, BN> acc;
  Loop::run(g, t, acc, smem);
  const LanePos lp;
  const int wm = kHalf ? half : lp.wm;  // the 128-row part of the tile, and with it the place of what is kept
  uint4* const kept_tile = KEEP == kKeepNone ? nullptr
                                             : p.stash + ((int64_t)tile * 4 + wm * 2) *
                                                             (KEEP == kKeepStash ? kStashWaveVecs : kLogitsWaveVecs) + lp.lane;
  float* const lds = reinterpret_cast<float*>(smem);
  if (t.m0 + 2 * BM * kBlk > p.vocab)
    fwd_epilogue<true, SOFTCAP, KEEP, BM, BN>(acc, p, lp, t, part0 + wm, kept_tile, lds);
  else
    fwd_epilogue<false, SOFTCAP, KEEP, BM, BN>(acc, p, lp, t, part0 + wm, kept_tile, lds);
}

template <class Loop, bool SOFTCAP, Keep KEEP>
__device__ __forceinline__ void fwd_body(const GemmOperands& g, const FwdParams& p, int tiles_m,
                                         int tiles_n) {
  extern __shared__ __align__(16) char smem[];
  const int whole = tiles_m * tiles_n - p.halved;
  int tm, tn;
  if constexpr (!std::is_void_v<typename Loop::Half>) {
    if ((int)blockIdx.x >= whole) {
      const int h = blockIdx.x - whole;
      tile_coords<8>(whole + (h >> 1), tiles_m, tiles_n, tm, tn);
      TilePos t = Loop::place(tm, tn);
      t.m0 += (h & 1) * (kTile / 2);
      fwd_tile<typename Loop::Half, kBlocks / 2, SOFTCAP, KEEP>(g, p, t, tm * tiles_n + tn, tm * 2, h & 1, smem);
      return;
    }
  }
  tile_coords<8>(xcd_order(whole), tiles_m, tiles_n, tm, tn);
  fwd_tile<Loop, kBlocks, SOFTCAP, KEEP>(g, p, Loop::place(tm, tn), tm * tiles_n + tn, tm * 2, 0, smem);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_kernel(GemmOperands g, FwdParams p,
                                                                  int tiles_m, int tiles_n) {
  fwd_body<Loop, false, kKeepNone>(g, p, tiles_m, tiles_n);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_softcap_kernel(GemmOperands g,
                                                                          FwdParams p, int tiles_m,
                                                                          int tiles_n) {
  fwd_body<Loop, true, kKeepNone>(g, p, tiles_m, tiles_n);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_stash_kernel(GemmOperands g, FwdParams p,
                                                                        int tiles_m, int tiles_n) {
  fwd_body<Loop, false, kKeepStash>(g, p, tiles_m, tiles_n);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_softcap_stash_kernel(GemmOperands g,
                                                                                FwdParams p,
                                                                                int tiles_m,
                                                                                int tiles_n) {
  fwd_body<Loop, true, kKeepStash>(g, p, tiles_m, tiles_n);
}

template <bool SOFTCAP>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_logits_kernel(GemmOperands g, FwdParams p,
                                                                         int tiles_m, int tiles_n) {
  fwd_body<DmaLoop, SOFTCAP, kKeepLogits>(g, p, tiles_m, tiles_n);
}

// Token-aligned packed layout.  With `is_start` (one byte per packed position, 1 where a sequence
// begins) the head works on a packed stream of token ids directly: hidden position n predicts the
// token at position n + 1, so its label is ids[n + 1] and its outputs land at position n + 1; a
// sequence's first position receives 0 (there is no prediction for it) and its upstream gradient
// is ignored.  This is roll(ids, -1) before and the shift-right after the head
// (axon/utils/fsdp/forward_utils.py:131,180-182) without the extra passes.  The position after the
// last one is `last_dst`: 0 for a whole packed stream (it wraps to the first position, which is always
// a sequence start).  A call that covers a block of consecutive positions of a longer stream hands
// over its arrays offset to the block's first position and names where its last row's output goes:
// n_tokens (the stream goes on: the first position of the next block) or minus the block's first
// position (the block ends the stream: position 0 of the stream).
__device__ __forceinline__ int aligned_pos(int n, int n_tokens, const uint8_t* is_start, int last_dst) {
  if (is_start == nullptr) return n;
  return (n + 1 == n_tokens) ? last_dst : n + 1;
}

typedef uint32_t AnyWord __attribute__((aligned(1)));  // the caller's array of flags begins anywhere
// Four positions per thread (the array is padded to that): one search for the sequence of the first, and from there a
// gallop per position, so that offsets padded with empty sequences to a fixed number cost a thread a few steps more
// (one sequence after the other 20000 of them took 2245 us for 5.1).  In one launch; a fill followed by a store per
// sequence took two, 4.8 us each.
__global__ __launch_bounds__(256) void seq_start_kernel(const int32_t* __restrict__ cu, int n_seqs,
                                                        int n_tokens, AnyWord* __restrict__ is_start) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x, p0 = v * 4;
  if (p0 >= n_tokens) return;
  int lo = 0, hi = n_seqs;  // the number of sequences that begin before p0
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int64_t)cu[mid] < p0) lo = mid + 1; else hi = mid;
  }
  uint32_t bits = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t p = p0 + u;
    if (p >= n_tokens) break;
    // lo: the number of sequences that begin at p or before it; the last of them is the one that owns p, those before it
    // with the same offset are empty
    int top = lo;
    for (int step = 1; top < n_seqs && (int64_t)cu[top] <= p; step *= 2) {
      lo = top + 1;
      top = min(lo + step - 1, n_seqs);
    }
    hi = top;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if ((int64_t)cu[mid] <= p) lo = mid + 1; else hi = mid;
    }
    if (lo > 0 && (int64_t)cu[lo - 1] == p && (int64_t)cu[lo] > p) bits |= 1u << (8 * u);
  }
  is_start[v] = bits;
}

// The last kernel of the forward: folds a token's partials into lse, entropy_b and entropy, forms the label's logit
// and with it logprob[n] = softcap(hidden[n] . W[label[n]]) / T - lse[n].
// A token's partials are folded in 256 groups, group c taking c, c + 256, ... (a chain of five for 151936 vocabulary
// rows); sixteen neighbouring groups are folded as a tree, the sixteen results one after the other.  That order is
// the same whatever T and PER, hence whatever the number of tokens.  A workgroup of 1024 threads owns T * PER
// consecutive tokens, a thread 256 * T / 1024 groups of PER tokens (T apart) with eight partials requested before the
// first is folded: T = 4 up to 1024 tokens, to put a short call on as many compute units as there are; T = 16 beyond,
// PER = 2 once a workgroup per 16 tokens would be more than one per CU.  The label dots (one wavefront per token) run
// before the barrier, beside the folds of the other wavefronts. 187 tokens x 896 x 151936 5.9 us (11.0 with three
// arrays of partials, 64 groups and 16 tokens per workgroup), 700 x 4096 11.9 (19.0), 1500 x 896 9.8 (12.8), 3001 x
// 2880 x 201088 22.5 (31.4), 8192 x 4096 41.4 (49.0).
template <int T, int PER, typename LabelT>
__global__ __launch_bounds__(1024) void lmhead_finish_kernel(
    const float* __restrict__ stats, int parts, const __bf16* __restrict__ hidden, const __bf16* __restrict__ weight,
    const LabelT* __restrict__ labels, int n_tokens, int hidden_sz, int vocab, float inv_temp, float cap,
    float* __restrict__ lse, float* __restrict__ entropy_b, float* __restrict__ entropy,
    float* __restrict__ logprobs, const uint8_t* __restrict__ is_start, int last_dst) {
  constexpr int TOK = T * PER, kWaves = 16, kGroups = 256, SUB = kGroups * T / 1024;
  constexpr int kDeep = 8 / (SUB * PER) < 1 ? 1 : 8 / (SUB * PER);
  __shared__ float red[3][kWaves][TOK];
  __shared__ float dots[TOK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int grp = threadIdx.x / T * SUB;  // this thread's groups: grp .. grp + SUB - 1
  int nc[PER];
#pragma unroll
  for (int t = 0; t < PER; ++t)  // a valid token; the results of those beyond the last are dropped below
    nc[t] = min(blockIdx.x * TOK + t * T + (int)(threadIdx.x % T), n_tokens - 1);
  // the first token's label is on its way while the partials are folded
  int64_t lab = 0;
  const int n_dot = blockIdx.x * TOK + wave;
  if (wave < TOK && n_dot < n_tokens) lab = (int64_t)labels[aligned_pos(n_dot, n_tokens, is_start, last_dst)];
  // a group beyond the number of partials holds an empty set (s = 0 below any reference)
  float M[SUB][PER], s[SUB][PER], e[SUB][PER];
#pragma unroll
  for (int g = 0; g < SUB; ++g)
#pragma unroll
    for (int t = 0; t < PER; ++t) { M[g][t] = kEmptyMax; s[g][t] = 0.f; e[g][t] = 0.f; }
  auto fold = [](float& M1, float& s1, float& e1, float M2, float s2, float e2) {
    const float Mn = fmaxf(M1, M2);
    merge_stats(M1, s1, e1, M2, s2, e2, Mn);
    M1 = Mn;
  };
  for (int q0 = grp; q0 < parts; q0 += kDeep * kGroups) {
    float x[kDeep][SUB][PER][3];
#pragma unroll
    for (int u = 0; u < kDeep; ++u)
#pragma unroll
      for (int g = 0; g < SUB; ++g)
#pragma unroll
        for (int t = 0; t < PER; ++t) {
          const float* o = stats + ((int64_t)min(q0 + u * kGroups + g, parts - 1) * n_tokens + nc[t]) * 3;
          x[u][g][t][0] = o[0]; x[u][g][t][1] = o[1]; x[u][g][t][2] = o[2];
        }
#pragma unroll
    for (int u = 0; u < kDeep; ++u)
#pragma unroll
      for (int g = 0; g < SUB; ++g) {
        if (q0 + u * kGroups + g >= parts) continue;
#pragma unroll
        for (int t = 0; t < PER; ++t)
          fold(M[g][t], s[g][t], e[g][t], x[u][g][t][0], x[u][g][t][1], x[u][g][t][2]);
      }
  }
#pragma unroll
  for (int t = 0; t < PER; ++t) {
#pragma unroll
    for (int off = 1; off < SUB; off <<= 1)
#pragma unroll
      for (int g = 0; g < SUB; g += 2 * off)
        fold(M[g][t], s[g][t], e[g][t], M[g + off][t], s[g + off][t], e[g + off][t]);
#pragma unroll
    for (int off = T; off < 64; off <<= 1)
      fold(M[0][t], s[0][t], e[0][t], __shfl_xor(M[0][t], off), __shfl_xor(s[0][t], off), __shfl_xor(e[0][t], off));
    if (lane < T) {
      const int tok = t * T + lane;
      red[0][wave][tok] = M[0][t]; red[1][wave][tok] = s[0][t]; red[2][wave][tok] = e[0][t];
    }
  }

  for (int k = wave; k < TOK; k += kWaves) {  // label dots
    const int nk = blockIdx.x * TOK + k;
    if (nk >= n_tokens) break;
    if (k != wave) lab = (int64_t)labels[aligned_pos(nk, n_tokens, is_start, last_dst)];
    float dot = 0.f;
    if (lab >= 0 && lab < vocab) {
      const uint4* h = reinterpret_cast<const uint4*>(hidden + (int64_t)nk * hidden_sz);
      const uint4* w = reinterpret_cast<const uint4*>(weight + lab * hidden_sz);
#pragma unroll 4
      for (int c = lane; c < hidden_sz / 8; c += 64) {
        const uint4 hv = h[c], wv = w[c];
        const uint32_t hs[4] = {hv.x, hv.y, hv.z, hv.w}, ws[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dot = fmaf(__uint_as_float(hs[i] << 16), __uint_as_float(ws[i] << 16), dot);
          dot = fmaf(__uint_as_float(hs[i] & 0xffff0000u), __uint_as_float(ws[i] & 0xffff0000u), dot);
        }
      }
    }
    dot = wave_sum(dot);
    if (cap != 0.f) dot = cap * fast_tanh(dot / cap);
    if (lane == 0) dots[k] = dot;
  }
  __syncthreads();
  const int tok = threadIdx.x, n = blockIdx.x * TOK + tok;
  if (tok >= TOK || n >= n_tokens) return;
  float Mt = red[0][0][tok], st = red[1][0][tok], et = red[2][0][tok];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) fold(Mt, st, et, red[0][w][tok], red[1][w][tok], red[2][w][tok]);
  // log2 units: logsumexp = M + L, sum softmax*logit = M + e/s; differences are taken
  // before adding M so that large logits do not cancel
  const float L = __log2f(st);
  const float d = et / st;
  lse[n] = (Mt + L) * kLn2;
  entropy_b[n] = (Mt + d) * kLn2;
  const int dst = aligned_pos(n, n_tokens, is_start, last_dst);
  const bool start = is_start && is_start[dst];
  entropy[dst] = start ? 0.f : (L - d) * kLn2;
  // (logit*c - M) is formed in one rounding, then log2(sum) is subtracted: no cancellation
  logprobs[dst] = start ? 0.f : (fmaf(dots[tok], inv_temp * kLog2e, -Mt) - L) * kLn2;
}

// ----------------------------------------------------------------------------
// Backward B1: recompute logits, write dlogit (bf16) in both orientations
// ----------------------------------------------------------------------------
struct DlogitParams {
  const float* lse;
  const float* entropy_b;
  const float* dlogprobs;
  const float* dentropy;  // may be null
  const void* labels;
  int labels_i64;
  __bf16* dl;    // [n_pad][chunk_cols]   token-major
  __bf16* dlT;   // [chunk_cols][n_pad]   vocab-major; null: not wanted (the dWeight GEMM reads dl as a K-major operand)
  int64_t ld_dl, ld_dlT;
  int n_tokens, vocab, v_begin;  // v_begin: first vocab row of this chunk
  // Rows of dl from here on (a multiple of 64, at least n_tokens) are read by nobody and need not be written:
  // sixty-four or a hundred and twenty-eight of them are left out together.  The zeros between n_tokens and n_end are
  // k of the weight gradient.
  int n_end;
  float inv_temp;
  float cap, inv_cap;  // soft-capping (SOFTCAP kernels only)
  const uint8_t* is_start;  // token-aligned packed layout (see aligned_pos), or null
  int last_dst;             // where the last row's label and gradients live (see aligned_pos)
};

// Four rows of four bf16 (rws[f] = row f) -> their transpose (o[e] = column e).
__device__ __forceinline__ void transpose_4x4_bf16(const uint2 (&rws)[4], uint2 (&o)[4]) {
  o[0].x = (rws[0].x & 0xffffu) | (rws[1].x << 16);
  o[0].y = (rws[2].x & 0xffffu) | (rws[3].x << 16);
  o[1].x = (rws[0].x >> 16) | (rws[1].x & 0xffff0000u);
  o[1].y = (rws[2].x >> 16) | (rws[3].x & 0xffff0000u);
  o[2].x = (rws[0].y & 0xffffu) | (rws[1].y << 16);
  o[2].y = (rws[2].y & 0xffffu) | (rws[3].y << 16);
  o[3].x = (rws[0].y >> 16) | (rws[1].y & 0xffff0000u);
  o[3].y = (rws[2].y >> 16) | (rws[3].y & 0xffff0000u);
}

// Per-wave staging of the wave's 128(n) x 128(m) bf16 sub-tile in its own 32 KB of LDS:
// row nw (256 bytes = 32 units of 4 bf16), unit u stored at slot perm(u) ^ swz(nw),
// swz(nw) = (nw & 31) ^ (nw >> 5), perm(u) = u rotated right by two bits (unit = 4 * block + lane
// quarter: the quarter's low bit becomes the slot's high bit).  The three access patterns
// (accumulator write: sixteen rows x two quarters per 32 lanes; row read; 4x4-block read) then each
// touch 32 distinct slots per 32 lanes.
__device__ __forceinline__ int stage_off(int nw, int unit) {
  const int pu = ((unit & 1) << 4) | ((unit & 2) << 2) | (unit >> 2);
  return nw * 256 + ((pu ^ ((nw & 31) ^ (nw >> 5))) << 3);
}

// The same where the row's lane part and the unit's are apart: accumulator block (i, j) of a wavefront (row 16 j + l16,
// unit 4 i + lq), and the row 16 j + 2 u + lane / 32 that half a wavefront reads (unit lane % 32).  Per lane, then
// constants: an exclusive or and an offset per access, where the compiler spent four instructions.
__device__ __forceinline__ int stage_block_base(const LanePos& lp) {
  return lp.l16 * 256 + (((((lp.lq & 1) << 4) | ((lp.lq & 2) << 2)) ^ lp.l16) << 3);
}
__device__ __forceinline__ int stage_block(int base, int i, int j) {
  return (base ^ ((i ^ (j >> 1) ^ ((j & 1) << 4)) << 3)) + j * kBlk * 256;
}
__device__ __forceinline__ int stage_row_base(const LanePos& lp) { return stage_off(lp.lane >> 5, lp.lane & 31); }
__device__ __forceinline__ int stage_row(int base, int j, int u) {
  return (base ^ (((2 * u) ^ (j >> 1) ^ ((j & 1) << 4)) << 3)) + (j * kBlk + 2 * u) * 256;
}

// Per-token factors of dlogit = softmax * (ca + cb * logit) + onehot * gl for tile-relative token
// row nr; lab_rel is the label's row inside the tile whose first vocabulary row is m0_abs (-1: not
// in this tile).
struct TokenCoef {
  float ca, cb, gl, lse2;
  int lab_rel, nn;
  bool n_ok;
  TokenCoef() = default;
  __device__ __forceinline__ TokenCoef(const DlogitParams& p, int n, int64_t m0_abs) {
    n_ok = n < p.n_tokens;
    nn = n_ok ? n : 0;
    const int src = aligned_pos(nn, p.n_tokens, p.is_start, p.last_dst);  // where the label and the gradients live
    const bool g_ok = n_ok && !(p.is_start && p.is_start[src]);
    const float g_lp = g_ok ? p.dlogprobs[src] : 0.f;
    const float g_en = (g_ok && p.dentropy) ? p.dentropy[src] : 0.f;
    lse2 = p.lse[nn] * kLog2e;
    const float eb = p.entropy_b[nn];
    ca = (-g_lp + g_en * eb) * p.inv_temp;
    cb = -g_en * p.inv_temp * p.inv_temp;
    gl = g_lp * p.inv_temp;
    const int64_t lab = p.labels_i64 ? static_cast<const int64_t*>(p.labels)[src]
                                     : (int64_t) static_cast<const int32_t*>(p.labels)[src];
    const int64_t lab_rel64 = lab - m0_abs;
    lab_rel = (lab_rel64 >= 0 && lab_rel64 < kTile) ? (int)lab_rel64 : -1;
  }
};

// The dlogit of one logit (the accumulator, before temperature and soft-capping), row mrel of the tile.  SOFTCAP:
// the logit goes through cap * tanh(. / cap) and the gradient is multiplied by the derivative 1 - tanh^2
// (fused_linear.py:80-83).
template <bool SOFTCAP, bool LABEL = true>
__device__ __forceinline__ float dlogit_of(float raw, int mrel, const TokenCoef& k, const DlogitParams& p, float c) {
  float dcap = 1.f;
  if (SOFTCAP) {
    const float th = fast_tanh(raw * p.inv_cap);
    raw = p.cap * th;
    dcap = fmaf(-th, th, 1.f);
  }
  const float pr = fast_exp2(fmaf(raw, c, -k.lse2));
  float v = pr * fmaf(k.cb, raw, k.ca);
  if (LABEL && mrel == k.lab_rel) v += k.gl;
  if (SOFTCAP) v *= dcap;
  return v;
}

// f(true_type) where one of the lanes' sixteen tokens has its label among the wavefront's 128 vocabulary rows (2048 / V of
// the cases: one in 74 at 151936, one in 16 at 32768); else f(false_type), without the label's two instructions per logit.  Decode of a stash
// or of kept logits, us, before / after: 300 x 896 x 151936 59.2 / 55.3, 1000 x 4096 x 151936 with an entropy gradient
// 137.6 / 130.4, 333 x 2880 x 201088 102.3 / 97.5, 6007 x 896 x 151936 (memory-bound) 1056 / 1048.
template <class F>
__device__ __forceinline__ void with_label_or_not(const TokenCoef& k, const LanePos& lp, F&& f) {
  const unsigned at = (unsigned)(k.lab_rel - lp.wm * kWaveTile);
  if (__builtin_amdgcn_ballot_w64(at < (unsigned)kWaveTile) != 0) f(std::true_type{});
  else f(std::false_type{});
}

// Accumulators -> bf16 dlogits, token-major to dl through the wave's staging area, where they stay for the
// vocab-major copy.  MASKED: the tile reaches past the last token or the last vocabulary row; those entries are
// written as zeros.  Sixteen tokens at a time, and all tokens' scalars requested before the first: the main loop ends for
// all workgroups of the chip at about the same time, so that this is a burst of 33 MB of stores, which the arithmetic
// of the next sixteen tokens now runs under (whole sub-tile first, then its copy: 6007 x 896 x 151936 1.98 ms for
// 1.79, 3001 x 1024 x 50257 0.408 for 0.380, 8192 x 4096 x 151936 7.43 for 7.27).  Bound by the issue of vector
// instructions: 1900 where no label is among the wavefront's logits, 3470 with the label's two per logit and the staging
// addresses formed anew for each access (us, before / after: 6007 x 896 x 151936 1791 / 1686, 3001 x 2880 x 201088 2645 / 2583,
// 2048 x 3072 x 128264 1206 / 1176, 333 x 896 x 151936 164 / 158).
template <bool SOFTCAP, bool MASKED>
__device__ __forceinline__ void dlogit_store(AccTile& acc, const DlogitParams& p, const LanePos& lp,
                                             const TilePos& t, char* stage) {
  const float c = p.inv_temp * kLog2e;
  const int l32 = lp.lane & 31, lhi = lp.lane >> 5;
  const int n_wave = t.n0 + lp.wn * kWaveTile;
  // token-major: 32 lanes cover one 256-byte row of the sub-tile, two rows per store
  char* d = reinterpret_cast<char*>(p.dl + (int64_t)(n_wave + lhi) * p.ld_dl + t.m0 + lp.wm * kWaveTile + l32 * 4);
  const int64_t dstep = p.ld_dl * 4;  // two rows of bf16
  TokenCoef k[kBlocks];
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) k[j] = TokenCoef(p, n_wave + j * kBlk + lp.l16, (int64_t)p.v_begin + t.m0);
  const int block = stage_block_base(lp), row = stage_row_base(lp);
  uint2 o[kBlocks];  // sixteen complete tokens on their way from LDS to memory, under the arithmetic of the next sixteen
  auto put = [&]() {
#pragma unroll
    for (int u = 0; u < kBlocks; ++u) {
      *reinterpret_cast<uint2*>(d) = o[u];
      d += dstep;
    }
  };
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) {
    const int m_end = MASKED ? (k[j].n_ok ? p.vocab - p.v_begin - t.m0 : 0) : kTile;  // rows that count
    auto compute = [&](auto label) {
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mrel = lp.m(i, r);
          const float x = dlogit_of<SOFTCAP, decltype(label)::value>(read_acc(acc[i][j], r), mrel, k[j], p, c);
          v[r] = (!MASKED || mrel < m_end) ? x : 0.f;
        }
        uint2 w;
        w.x = pack_bf16(v[0], v[1]);
        w.y = pack_bf16(v[2], v[3]);
        *reinterpret_cast<uint2*>(stage + stage_block(block, i, j)) = w;
      }
    };
    with_label_or_not(k[j], lp, compute);
    if (j > 0) put();
#pragma unroll
    for (int u = 0; u < kBlocks; ++u) o[u] = *reinterpret_cast<const uint2*>(stage + stage_row(row, j, u));
  }
  put();
}

// The same from a forward's stash (see StashLayout above FwdParams): softmax = w * 2^(M - lse), scaled logit =
// log2(w) + M.  One call covers 64 tokens (four 16-token blocks, j0 .. j0 + 3) x 128 vocabulary rows of a wavefront's
// sub-tile; staged row = token - 16 * j0.  SOFTCAP: the stash describes the capped logit, whose derivative factor is
// 1 - (capped / cap)^2.  EDGE: entries beyond the last token or the last vocabulary row are staged as zeros.
// ENT: the entropies have a gradient.  Without one (and without soft-capping) the logit itself is not needed, and the
// logarithm that recovers it is half of the vector work: 333 tokens x 1024 x 50257 36.8 us for 42.7, 300 x 896 x
// 151936 58.7 for 66.9 (rows beyond n_end left out as well), 700 x 4096 83 for 94; from some thousand tokens on
// memory bounds both.
constexpr int kStashHalfBlocks = kBlocks / 2;
template <bool SOFTCAP, bool ENT, bool EDGE>
__device__ __forceinline__ void dlogit_stage_stash(const uint4 (&st)[4 * kStashHalfBlocks], int j0,
                                                   const float* __restrict__ pm, int part,
                                                   const DlogitParams& p, const LanePos& lp,
                                                   const TilePos& t, char* stage) {
  const float inv_c = 1.f / (p.inv_temp * kLog2e);
  const int block = stage_block_base(lp);
#pragma unroll
  for (int jl = 0; jl < kStashHalfBlocks; ++jl) {
    const TokenCoef k(p, t.n0 + lp.wn * kWaveTile + (j0 + jl) * kBlk + lp.l16, (int64_t)p.v_begin + t.m0);
    const float Mp = pm[(int64_t)part * p.n_tokens + k.nn];
    const float scale = fast_exp2(Mp - k.lse2);
    const bool n_counts = !EDGE || k.n_ok;
    with_label_or_not(k, lp, [&](auto label) {
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        const uint4 q = st[jl * 4 + (i >> 1)];
        float wv[4];
        unpack_f16((i & 1) ? q.z : q.x, wv[0], wv[1]);
        unpack_f16((i & 1) ? q.w : q.y, wv[2], wv[3]);
        float d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mrel = lp.m(i, r);
          const float pr = wv[r] * scale;
          float raw = 0.f;
          if (SOFTCAP || ENT) raw = (__builtin_amdgcn_logf(fmaxf(wv[r], 1e-30f)) + Mp) * inv_c;
          float v = pr * (ENT ? fmaf(k.cb, raw, k.ca) : k.ca);
          if (decltype(label)::value && mrel == k.lab_rel) v += k.gl;
          if (SOFTCAP) {
            const float th = raw * p.inv_cap;
            v *= fmaf(-th, th, 1.f);
          }
          const bool ok = !EDGE || (n_counts && p.v_begin + t.m0 + mrel < p.vocab);
          d[r] = ok ? v : 0.f;
        }
        uint2 w;
        w.x = pack_bf16(d[0], d[1]);
        w.y = pack_bf16(d[2], d[3]);
        *reinterpret_cast<uint2*>(stage + stage_block(block, i, jl)) = w;
      }
    });
  }
}

// The same from the logits that a forward kept (kKeepLogits): the arithmetic of dlogit_store on what the
// accumulators held.
template <bool SOFTCAP, bool EDGE>
__device__ __forceinline__ void dlogit_stage_logits(const float4 (&x)[kStashHalfBlocks * kBlocks], int j0,
                                                    const DlogitParams& p, const LanePos& lp, const TilePos& t,
                                                    char* stage) {
  const float c = p.inv_temp * kLog2e;
  const int block = stage_block_base(lp);
#pragma unroll
  for (int jl = 0; jl < kStashHalfBlocks; ++jl) {
    const TokenCoef k(p, t.n0 + lp.wn * kWaveTile + (j0 + jl) * kBlk + lp.l16, (int64_t)p.v_begin + t.m0);
    const int m_end = EDGE ? (k.n_ok ? p.vocab - p.v_begin - t.m0 : 0) : kTile;  // rows that count
    with_label_or_not(k, lp, [&](auto label) {
#pragma unroll
      for (int i = 0; i < kBlocks; ++i) {
        const float4 q = x[jl * kBlocks + i];
        const float raw[4] = {q.x, q.y, q.z, q.w};
        float d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mrel = lp.m(i, r);
          const float v = dlogit_of<SOFTCAP, decltype(label)::value>(raw[r], mrel, k, p, c);
          d[r] = (!EDGE || mrel < m_end) ? v : 0.f;
        }
        uint2 w;
        w.x = pack_bf16(d[0], d[1]);
        w.y = pack_bf16(d[2], d[3]);
        *reinterpret_cast<uint2*>(stage + stage_block(block, i, jl)) = w;
      }
    });
  }
}

// A staged 64 x 128 half sub-tile (tokens 16 * j0 .. of the wavefront's sub-tile) -> dl and dlT.  Token-major 32
// lanes cover one 256-byte row, eight rows per trip (reads before writes); vocab-major: sixteen lanes cover the 64
// tokens of one vocabulary row (one 128-byte line), the four lane groups take units u, u + 8, u + 16, u + 24, whose
// permuted slots differ in a bit that the rows' swizzles (a set with that bit fixed) cannot cancel.
__device__ __forceinline__ void dlogit_copy_out_half(const char* stage, int j0, const DlogitParams& p,
                                                     const LanePos& lp, const TilePos& t) {
  const int l32 = lp.lane & 31, lhi = lp.lane >> 5;
  const int m_base = t.m0 + lp.wm * kWaveTile;
  const int n_base = t.n0 + lp.wn * kWaveTile + j0 * kBlk;
  {
    const int unit = l32;
    char* d = reinterpret_cast<char*>(p.dl + (int64_t)(n_base + lhi) * p.ld_dl + m_base + unit * 4);
    const int64_t dstep = p.ld_dl * 4;  // two rows of bf16
#pragma unroll 1
    for (int nw0 = lhi; nw0 < kStashHalfBlocks * kBlk; nw0 += 16) {
      uint2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const uint2*>(stage + stage_off(nw0 + 2 * u, unit));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        *reinterpret_cast<uint2*>(d) = v[u];
        d += dstep;
      }
    }
  }
  if (p.dlT) {
    const int nq = lp.lane & 15, grp = lp.lane >> 4;
    const int64_t rstep = p.ld_dlT * 2;  // one row of bf16
    char* d = reinterpret_cast<char*>(p.dlT + (int64_t)(m_base + grp * 32) * p.ld_dlT + n_base + nq * 4);
#pragma unroll 2
    for (int u8 = 0; u8 < 8; ++u8) {
      const int unit = grp * 8 + u8;
      uint2 rws[4];
#pragma unroll
      for (int f = 0; f < 4; ++f)
        rws[f] = *reinterpret_cast<const uint2*>(stage + stage_off(nq * 4 + f, unit));
      uint2 o[4];
      transpose_4x4_bf16(rws, o);
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<uint2*>(d + e * rstep) = o[e];
      d += 4 * rstep;
    }
  }
}

// The wave's staged 128 x 128 bf16 sub-tile -> dlT (vocab-major), where it is wanted.  The wave
// reads back only what it wrote itself; LDS operations of one wave complete in order.
__device__ __forceinline__ void dlogit_copy_out_vocab(const char* stage, const DlogitParams& p,
                                                      const LanePos& lp, const TilePos& t) {
  const int l32 = lp.lane & 31, lhi = lp.lane >> 5;
  const int m_base = t.m0 + lp.wm * kWaveTile;  // chunk-relative column of the sub-tile
  const int n_base = t.n0 + lp.wn * kWaveTile;
  // vocab-major copy: 4x4 blocks transposed in registers; 32 lanes cover 128 tokens of one vocab row
  if (p.dlT) {
    const int nq = l32;  // token quad
    const int64_t rstep = p.ld_dlT * 2;  // one row of bf16
    char* d = reinterpret_cast<char*>(p.dlT + (int64_t)(m_base + lhi * 4) * p.ld_dlT + n_base + nq * 4);
#pragma unroll 2
    for (int unit = lhi; unit < 32; unit += 2) {
      uint2 rws[4];
#pragma unroll
      for (int f = 0; f < 4; ++f)
        rws[f] = *reinterpret_cast<const uint2*>(stage + stage_off(nq * 4 + f, unit));
      uint2 o[4];
      transpose_4x4_bf16(rws, o);
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<uint2*>(d + e * rstep) = o[e];
      d += 8 * rstep;
    }
  }
}

template <class Loop, bool SOFTCAP>
__device__ __forceinline__ void dlogit_body(const GemmOperands& g, const DlogitParams& p,
                                            int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) char smem[];
  int tm, tn;
  tile_coords(xcd_order(tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
  const TilePos t = Loop::place(tm, tn);  // t.m0 is relative to the chunk
  AccTile acc;
  Loop::run(g, t, acc, smem);
  __syncthreads();  // every wave is past its last main-loop LDS access

  const LanePos lp;
  if (t.n0 + lp.wn * kWaveTile >= p.n_end) return;
  char* const stage = smem + lp.wave * 32768;
  if (t.n0 + kTile > p.n_tokens || p.v_begin + t.m0 + kTile > p.vocab)
    dlogit_store<SOFTCAP, true>(acc, p, lp, t, stage);
  else
    dlogit_store<SOFTCAP, false>(acc, p, lp, t, stage);
  dlogit_copy_out_vocab(stage, p, lp, t);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_dlogit_kernel(GemmOperands g, DlogitParams p,
                                                                     int tiles_m, int tiles_n) {
  dlogit_body<Loop, false>(g, p, tiles_m, tiles_n);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void lmhead_dlogit_softcap_kernel(GemmOperands g,
                                                                             DlogitParams p,
                                                                             int tiles_m,
                                                                             int tiles_n) {
  dlogit_body<Loop, true>(g, p, tiles_m, tiles_n);
}

// Backward B1 without the recompute: one wavefront per workgroup turns half (64 tokens x 128 rows) of a sub-tile that
// a stashing forward stored into bf16 dlogits in both orientations (16 KB of LDS and few registers: ten wavefronts
// per CU hide the latency of the loads and of the per-token operands).  A streaming kernel: 2 bytes read and 4
// written per logit.  Tiles are the forward's: `tm0` is the forward tile row of the chunk's first vocabulary row, and
// t.m0 is made chunk-relative after the edge tests.
struct StashSource {
  const uint4* stash;
  const float* pm;
  int tiles_n, tm0;
};

template <bool SOFTCAP, bool ENT>
__global__ __launch_bounds__(64) void lmhead_dlogit_stash_kernel(DlogitParams p, StashSource src) {
  __shared__ __align__(16) char stage[kStashHalfBlocks * kBlk * 256];  // 64 tokens x 128 bf16
  const int half = blockIdx.x & 1, wave = (blockIdx.x >> 1) & 3, tile = blockIdx.x >> 3;
  const int tm = src.tm0 + tile / src.tiles_n, tn = tile % src.tiles_n;
  TilePos t{tm * kTile, tn * kTile};
  LanePos lp;
  lp.wave = wave;
  lp.wm = wave >> 1;
  lp.wn = wave & 1;
  const int j0 = half * kStashHalfBlocks;
  if (t.n0 + lp.wn * kWaveTile + j0 * kBlk >= p.n_end) return;
  const uint4* sv = src.stash + ((int64_t)(tm * src.tiles_n + tn) * 4 + wave) * kStashWaveVecs +
                    j0 * 4 * 64 + lp.lane;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  uint4 st[4 * kStashHalfBlocks];
#pragma unroll
  for (int q = 0; q < 4 * kStashHalfBlocks; ++q) {  // read once: keep it out of the way of the GEMMs' operands in L2
    const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(sv + q * 64));
    st[q] = make_uint4(x[0], x[1], x[2], x[3]);
  }
  const bool edge = t.m0 + kTile > p.vocab || t.n0 + kTile > p.n_tokens;
  t.m0 -= p.v_begin;
  const int part = tm * 2 + lp.wm;
  if (edge) {
    dlogit_stage_stash<SOFTCAP, ENT, true>(st, j0, src.pm, part, p, lp, t, stage);
  } else {
    dlogit_stage_stash<SOFTCAP, ENT, false>(st, j0, src.pm, part, p, lp, t, stage);
  }
  dlogit_copy_out_half(stage, j0, p, lp, t);
}

// The same from kept logits: 4 bytes read and 2 written per logit.
template <bool SOFTCAP>
__global__ __launch_bounds__(64) void lmhead_dlogit_logits_kernel(DlogitParams p, StashSource src) {
  __shared__ __align__(16) char stage[kStashHalfBlocks * kBlk * 256];  // 64 tokens x 128 bf16
  const int half = blockIdx.x & 1, wave = (blockIdx.x >> 1) & 3, tile = blockIdx.x >> 3;
  const int tm = src.tm0 + tile / src.tiles_n, tn = tile % src.tiles_n;
  TilePos t{tm * kTile, tn * kTile};
  LanePos lp;
  lp.wave = wave;
  lp.wm = wave >> 1;
  lp.wn = wave & 1;
  const int j0 = half * kStashHalfBlocks;
  if (t.n0 + lp.wn * kWaveTile + j0 * kBlk >= p.n_end) return;
  const uint4* sv = src.stash + ((int64_t)(tm * src.tiles_n + tn) * 4 + wave) * kLogitsWaveVecs +
                    j0 * kBlocks * 64 + lp.lane;
  float4 x[kStashHalfBlocks * kBlocks];
#pragma unroll
  for (int q = 0; q < kStashHalfBlocks * kBlocks; ++q) {  // read once
    const acc4 v = __builtin_nontemporal_load(reinterpret_cast<const acc4*>(sv + q * 64));
    x[q] = make_float4(v[0], v[1], v[2], v[3]);
  }
  const bool edge = t.m0 + kTile > p.vocab || t.n0 + kTile > p.n_tokens;
  t.m0 -= p.v_begin;
  if (edge)
    dlogit_stage_logits<SOFTCAP, true>(x, j0, p, lp, t, stage);
  else
    dlogit_stage_logits<SOFTCAP, false>(x, j0, p, lp, t, stage);
  dlogit_copy_out_half(stage, j0, p, lp, t);
}

// ----------------------------------------------------------------------------
// Backward B2/B3 and the plain GEMM: store the tile as out[n][m]
// ----------------------------------------------------------------------------
struct StoreParams {
  float* out_f32 = nullptr;    // [n][ld_f32] fp32 output (may be null)
  __bf16* out_bf16 = nullptr;  // [n][ld_bf16] (may be null)
  int64_t ld_f32 = 0, ld_bf16 = 0;
  int m_valid = 0, n_valid = 0;
  int accumulate = 0;  // add the previous contents of tile_acc first
  int keep_f32 = 0;    // write the sum back to tile_acc (0: it is only read, the sum leaves as bf16)
  // fp32 partial sums (the weight gradient carried from one token block to the next, dHidden carried from one
  // vocabulary chunk to the next or formed in parts): kept per tile in the order the accumulators lie in the
  // registers, so that every wavefront load and store is one contiguous kilobyte.  float4 index = ((tile * 4 + wave)
  // * 64 + i * 8 + j) * 64 + lane, tile = tm * tiles_n + tn.  Null: not used.
  float4* tile_acc = nullptr;
  // Split reduction: `splits` workgroups per tile, each over `k_split` (a multiple of 64) of the k; they leave their
  // partial sums in tile_acc, one array of tiles after the other, for split_sum_kernel.
  int splits = 1, k_split = 0;
  // The last tile of an m that fills at most half of it is computed as half a tile (DmaLoopT's BM).  Its rows lie in
  // tile_acc where a whole tile leaves them, the other half of the tile is left as it was.
  int half_edge = 0;
};
constexpr int64_t kTileAccVecs = 4 * kBlocks * kBlocks * 64;  // float4 per tile (256 KB)

// U rows of staged bf16 values, kStep apart, to out_bf16: 16 bytes per lane and row.
template <int U, int kStep>
__device__ __forceinline__ void store_rows(const StoreParams& p, const char* stage, int row, int unit, int n, int m) {
  uint2 v[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int q = 0; q < 2; ++q)
      v[u][q] = *reinterpret_cast<const uint2*>(stage + stage_off(row + kStep * u, unit + q));
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (n + kStep * u >= p.n_valid) continue;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 x = {v[u][0].x, v[u][0].y, v[u][1].x, v[u][1].y};  // read by nobody soon
    __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(p.out_bf16 + (int64_t)(n + kStep * u) * p.ld_bf16 + m));
  }
}

template <class Loop, int BM>
__device__ __forceinline__ void store_tile(const GemmOperands& g, const StoreParams& p, const TilePos& t, int64_t tile,
                                           char* smem) {
  constexpr bool kHalf = BM < kBlocks;
  AccTileOf<BM> acc;
  Loop::run(g, t, acc, smem);
  const LanePos lp;
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  auto value = [&](int i, int j) {
    return f32x4{read_acc(acc[i][j], 0), read_acc(acc[i][j], 1), read_acc(acc[i][j], 2), read_acc(acc[i][j], 3)};
  };
  if (p.out_f32) {  // the plain product
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
      const int n = t.n0 + lp.n(j);
      if (n >= p.n_valid) continue;
#pragma unroll
      for (int i = 0; i < BM; ++i) {
        const int m = t.m0 + lp.m<BM>(i, 0);
        if (m >= p.m_valid) continue;  // m_valid % 4 == 0: a quad is all in or all out
        *reinterpret_cast<f32x4*>(p.out_f32 + (int64_t)n * p.ld_f32 + m) = value(i, j);
      }
    }
    return;
  }
  // bf16 rows leave through the wavefront's own 32 KB of LDS, so that a store instruction writes four rows of 256
  // contiguous bytes (whole cache lines) instead of sixteen pieces of 32: the main loop has ended with a barrier, and
  // LDS operations of one wave complete in order.  Two half-waves' reads touch 32 distinct slots each (rows 16
  // apart, see stage_off).  dWeight of 700 tokens in these tiles (11 k-tiles; 151936 x 4096 written, inside a step) 979 us
  // before, 832 with the staging, 809 with the non-temporal hint on top; long reductions do not notice.  Accumulators are
  // read on their way out (read_acc): read at the head and written back around the branches below they cost 600
  // instructions more (us between events, medians of three processes of each, before / after: dHidden 1201 x 1024 x 50257
  // 138 / 132, 1500 x 2048 x 32768 168 / 164, 6007 x 896 x 151936 1207 / 1193; the dWeight of the same calls 146 / 143, 168 / 166,
  // 1223 / 1229, within what processes differ).
  char* const stage = smem + lp.wave * 32768;
  const int block = stage_block_base(lp);
  auto to_stage = [&](int i, int j, const f32x4& v) {
    uint2 w;
    w.x = pack_bf16(v[0], v[1]);
    w.y = pack_bf16(v[2], v[3]);
    *reinterpret_cast<uint2*>(stage + stage_block(block, i, j)) = w;
  };
  if (p.tile_acc) {
    f32x4* ta = reinterpret_cast<f32x4*>(p.tile_acc) +
                (tile * 4 + (kHalf ? lp.wn : lp.wave)) * (kBlocks * kBlocks * 64) +
                (kHalf ? lp.wm * BM * kBlocks * 64 : 0) + lp.lane;
#pragma unroll
    for (int i = 0; i < BM; ++i) {
      f32x4 v[kBlocks];
      if (p.accumulate) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) v[j] = __builtin_nontemporal_load(ta + (i * kBlocks + j) * 64);
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) v[j] = value(i, j) + v[j];
      } else {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) v[j] = value(i, j);
      }
      if (p.keep_f32) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) __builtin_nontemporal_store(v[j], ta + (i * kBlocks + j) * 64);
      }
      if (p.out_bf16) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) to_stage(i, j, v[j]);
      }
    }
    if (!p.out_bf16) return;
  } else {
#pragma unroll
    for (int j = 0; j < kBlocks; ++j)
#pragma unroll
      for (int i = 0; i < BM; ++i) to_stage(i, j, value(i, j));
  }
  if (kHalf) {  // 64 values of m per wavefront: eight rows of 128 contiguous bytes per store instruction
    const int row0 = lp.lane >> 3, col = lp.lane & 7, m = t.m0 + lp.wm * BM * kBlk + col * 8;
    if (m >= p.m_valid) return;
#pragma unroll 1
    for (int r64 = 0; r64 < kWaveTile; r64 += 64)
      store_rows<8, 8>(p, stage, r64 + row0, 2 * col, t.n0 + lp.wn * kWaveTile + r64 + row0, m);
    return;
  }
  const int m = t.m0 + lp.wm * kWaveTile + lp.l16 * 8;
  if (m >= p.m_valid) return;  // m_valid % 8 == 0: a vector of eight is all in or all out
  const int row0 = (lp.lane >> 5) + 16 * (lp.lq & 1);
#pragma unroll 1
  for (int r32 = 0; r32 < kWaveTile; r32 += 32)
    store_rows<8, 2>(p, stage, r32 + row0, 2 * lp.l16, t.n0 + lp.wn * kWaveTile + r32 + row0, m);
}

template <class Loop>
__global__ __launch_bounds__(kGemmThreads) void gemm_store_kernel(GemmOperands g, StoreParams p,
                                                                  int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) char smem[];
  int tm, tn;
  const int tiles = tiles_m * tiles_n;
  const int pid = xcd_order(tiles * p.splits);
  const int split = pid / tiles;  // the tiles of one part of k side by side: they share operand slices
  tile_coords(pid - split * tiles, tiles_m, tiles_n, tm, tn);
  const int64_t k0 = (int64_t)split * p.k_split;
  g.a += Loop::kAMajor ? k0 * g.lda : k0;
  g.b += Loop::kBMajor ? k0 * g.ldb : k0;
  g.k = min(g.k - (int)k0, p.k_split);
  const TilePos t = Loop::place(tm, tn);
  const int64_t tile = (int64_t)split * tiles + tm * tiles_n + tn;
  if constexpr (!std::is_void_v<typename Loop::HalfEdge>) {
    if (p.half_edge && t.m0 + kTile / 2 >= p.m_valid) {
      store_tile<typename Loop::HalfEdge, kBlocks / 2>(g, p, t, tile, smem);
      return;
    }
  }
  store_tile<Loop, kBlocks>(g, p, t, tile, smem);
}

// out[n][m] = the sum over the parts of a split reduction, rounded to bf16: a streaming kernel, one thread per
// four accumulators (read as whole kilobytes per wavefront, in the order of the parts).
__global__ __launch_bounds__(256) void split_sum_kernel(const float4* __restrict__ parts, int splits, int tiles_m,
                                                        int tiles_n, int m_valid, int n_valid,
                                                        __bf16* __restrict__ out, int64_t ld) {
  const int64_t stride = (int64_t)tiles_m * tiles_n * kTileAccVecs;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;  // lane, then block (i, j), wavefront, tile
  const int lane = (int)(q & 63), ij = (int)(q >> 6) & 63, wave = (int)(q >> 12) & 3, tile = (int)(q >> 14);
  const int m = (tile / tiles_n) * kTile + (wave >> 1) * kWaveTile + (ij >> 3) * kBlk + 4 * (lane >> 4);
  const int n = (tile % tiles_n) * kTile + (wave & 1) * kWaveTile + (ij & 7) * kBlk + (lane & 15);
  if (m >= m_valid || n >= n_valid) return;
  const float4* src = parts + q;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  int s = 0;
  for (; s + 4 <= splits; s += 4) {
    float4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = src[(s + u) * stride];
#pragma unroll
    for (int u = 0; u < 4; ++u) { v.x += x[u].x; v.y += x[u].y; v.z += x[u].z; v.w += x[u].w; }
  }
  for (; s < splits; ++s) {
    const float4 x = src[s * stride];
    v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
  }
  uint2 w;
  w.x = pack_bf16(v.x, v.y);
  w.y = pack_bf16(v.z, v.w);
  *reinterpret_cast<uint2*>(out + (int64_t)n * ld + m) = w;
}

// out[c][r] = in[r][c] for r < rows, c < cols; zero for r in [rows, rows_pad).
// 64x64 tiles through LDS; both sides move 16 bytes per thread and access (two per thread each
// way) where the tile is whole, element by element at the ragged edges.  ld_in and ld_out are
// multiples of 8 elements and both bases 16-byte aligned (checked by the launcher).
__global__ __launch_bounds__(256) void transpose_bf16_kernel(const uint16_t* __restrict__ in,
                                                             int64_t ld_in, int rows, int cols,
                                                             uint16_t* __restrict__ out,
                                                             int64_t ld_out, int rows_pad) {
  __shared__ uint16_t t[64][66 + 6];  // 144-byte rows: 16-byte row writes stay aligned
  const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
#pragma unroll
  for (int q = threadIdx.x; q < 512; q += 256) {
    const int r = q >> 3, c = (q & 7) * 8;
    union { uint4 v; uint16_t h[8]; } u;
    u.v = make_uint4(0, 0, 0, 0);
    if (r0 + r < rows) {
      const uint16_t* src = in + (int64_t)(r0 + r) * ld_in + c0 + c;
      if (c0 + c + 8 <= cols) {
        u.v = *reinterpret_cast<const uint4*>(src);
      } else {
        for (int e = 0; e < 8; ++e)
          if (c0 + c + e < cols) u.h[e] = src[e];
      }
    }
    *reinterpret_cast<uint4*>(&t[r][c]) = u.v;
  }
  __syncthreads();
#pragma unroll
  for (int q = threadIdx.x; q < 512; q += 256) {
    const int c = q >> 3, r = (q & 7) * 8;
    if (c0 + c >= cols || r0 + r >= rows_pad) continue;
    union { uint4 v; uint16_t h[8]; } u;
#pragma unroll
    for (int e = 0; e < 8; ++e) u.h[e] = t[r + e][c];
    uint16_t* dst = out + (int64_t)(c0 + c) * ld_out + r0 + r;
    if (r0 + r + 8 <= rows_pad) {
      *reinterpret_cast<uint4*>(dst) = u.v;
    } else {
      for (int e = 0; e < 8; ++e)
        if (r0 + r + e < rows_pad) dst[e] = u.h[e];
    }
  }
}

// ----------------------------------------------------------------------------
// Rows without an upstream gradient (prompt positions, masked or clipped tokens)
// ----------------------------------------------------------------------------
// One workgroup walks the rows in blocks of 4096 (four consecutive rows per thread) and numbers the
// active ones in ascending order (ballots + popcounts inside a wave, wave totals through LDS): the
// list is the same on every run.
__global__ __launch_bounds__(1024) void active_rows_kernel(
    const float* __restrict__ dlogprobs, const float* __restrict__ dentropy,
    const uint8_t* __restrict__ is_start, int n_tokens, int32_t* __restrict__ row_index,
    int32_t* __restrict__ row_rank, int32_t* __restrict__ count) {
  __shared__ int wave_total[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  int base = 0;
  for (int n0 = 0; n0 < n_tokens; n0 += 4096) {
    const int first = n0 + (int)threadIdx.x * 4;
    bool act[4];
    int before = 0, mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = first + j;
      act[j] = false;
      if (n < n_tokens) {
        const int src = aligned_pos(n, n_tokens, is_start, 0);
        if (!(is_start && is_start[src]))
          act[j] = dlogprobs[src] != 0.f || (dentropy && dentropy[src] != 0.f);  // NaN counts as active
      }
      const unsigned long long b = __ballot(act[j]);
      before += __popcll(b & below);  // active rows of the lanes below, this j
      mine += __popcll(b);
    }
    if (lane == 0) wave_total[wave] = mine;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before += wave_total[w];
      total += wave_total[w];
    }
    int r = base + before;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = first + j;
      if (n < n_tokens) {
        if (act[j]) row_index[r] = n;
        row_rank[n] = act[j] ? r : -1;
        r += act[j] ? 1 : 0;
      }
    }
    base += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) count[0] = base;
}

// One workgroup per active row: its hidden vector (16-byte accesses) and its scalars, the label and the
// gradients taken from the aligned position.
template <typename LabelT>
__global__ __launch_bounds__(256) void gather_rows_kernel(
    const uint4* __restrict__ hidden, int row_vec, const LabelT* __restrict__ labels,
    const float* __restrict__ lse, const float* __restrict__ entropy_b,
    const float* __restrict__ dlogprobs, const float* __restrict__ dentropy,
    const uint8_t* __restrict__ is_start, int n_tokens, const int32_t* __restrict__ row_index,
    uint4* __restrict__ hidden_c, LabelT* __restrict__ labels_c, float* __restrict__ lse_c,
    float* __restrict__ entropy_b_c, float* __restrict__ dlogprobs_c, float* __restrict__ dentropy_c) {
  const int r = blockIdx.x;
  const int n = row_index[r];
  const uint4* src_row = hidden + (int64_t)n * row_vec;
  uint4* dst_row = hidden_c + (int64_t)r * row_vec;
  for (int c = threadIdx.x; c < row_vec; c += 256) dst_row[c] = src_row[c];
  if (threadIdx.x == 0) {
    const int src = aligned_pos(n, n_tokens, is_start, 0);
    labels_c[r] = labels[src];
    lse_c[r] = lse[n];
    entropy_b_c[r] = entropy_b[n];
    dlogprobs_c[r] = dlogprobs[src];
    if (dentropy_c) dentropy_c[r] = dentropy ? dentropy[src] : 0.f;
  }
}

// One workgroup per row of d_hidden: the compact row, or zeros.
__global__ __launch_bounds__(256) void scatter_rows_kernel(const uint4* __restrict__ d_hidden_c,
                                                           const int32_t* __restrict__ row_rank,
                                                           int row_vec, uint4* __restrict__ d_hidden) {
  const int n = blockIdx.x;
  const int r = row_rank[n];
  uint4* dst_row = d_hidden + (int64_t)n * row_vec;
  if (r < 0) {
    for (int c = threadIdx.x; c < row_vec; c += 256) dst_row[c] = make_uint4(0, 0, 0, 0);
    return;
  }
  const uint4* src_row = d_hidden_c + (int64_t)r * row_vec;
  for (int c = threadIdx.x; c < row_vec; c += 256) dst_row[c] = src_row[c];
}

// x *= scale[0] in place on bf16 values, eight per thread and access; nothing is read or written when the
// factor is exactly one (the factor lives on the device: the host does not know it without waiting).
// A second array `y` in the same launch (may be empty).
__global__ __launch_bounds__(256) void scale_bf16_kernel(uint4* __restrict__ x, int64_t n_vec, uint4* __restrict__ y,
                                                         int64_t n_y, const float* __restrict__ scale) {
  const float s = scale[0];
  if (s == 1.f) return;
  auto scaled = [s](uint4 v) {
    uint32_t* w = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = pack_bf16(__uint_as_float(w[k] << 16) * s, __uint_as_float(w[k] & 0xffff0000u) * s);
    return v;
  };
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t i = i0; i < n_vec; i += step) x[i] = scaled(x[i]);
  for (int64_t i = i0; i < n_y; i += step) y[i] = scaled(y[i]);
}

}  // namespace axon

using namespace axon;

namespace {

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
// Vocabulary chunk of a backward that is not told one: every chunk costs one read-modify-write pass over the fp32
// dHidden partial sums and its own launches, so as much of the vocabulary as keeps a chunk's bf16 dlogits within
// the 2 GiB that 32768 columns take at 32768 tokens.
constexpr int64_t kDefaultVocabChunk = 32768;
constexpr int64_t kDefaultChunkElems = int64_t(1) << 30;
constexpr int64_t kAlign = 256;
constexpr int kCus = 256;
using SlowLoop = RegLoop<32>;

// Leading dimensions whose byte offsets inside a tile (256 rows K-contiguous, 64 K-major) stay below 2^30
constexpr int64_t kMaxLd = 1 << 21, kMaxLdKMajor = 1 << 23;
// A K-contiguous operand of the DMA loop: 16-byte vectors, and rows at least a k-tile apart (the descriptor's end and
// the scalar offsets of its instructions are multiples of the row stride; rows closer than that, an expanded or an
// overlapping view, go through registers).
inline bool kcontig_ok(const void* p, int64_t ld) {
  return ld >= DmaLoop::kBK && ld < kMaxLd && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}
inline bool dma_ok(const GemmOperands& g) {
  return (g.k % DmaLoop::kBK) == 0 && kcontig_ok(g.a, g.lda) && kcontig_ok(g.b, g.ldb);
}

template <typename K>
int set_lds(K kernel) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             kGemmLdsBytes) == hipSuccess
             ? AXON_OK
             : AXON_ERR_LAUNCH;
}

// Launch kernel<DmaLoop> or kernel<SlowLoop> over all tiles of the problem.
#define AXON_LAUNCH_GEMM(KERNEL, G, P, ST) AXON_LAUNCH_GEMM_PLUS(KERNEL, G, P, ST, 0)
// with EXTRA workgroups more than tiles where the fast loop is taken
#define AXON_LAUNCH_GEMM_PLUS(KERNEL, G, P, ST, EXTRA)                                            \
  do {                                                                                            \
    const int tiles_m_ = ((G).m_rows + kTile - 1) / kTile, tiles_n_ = ((G).n_rows + kTile - 1) / kTile; \
    if (dma_ok(G)) {                                                                              \
      if (set_lds(KERNEL<DmaLoop>) != AXON_OK) return AXON_ERR_LAUNCH;                            \
      hipLaunchKernelGGL(KERNEL<DmaLoop>, dim3(tiles_m_ * tiles_n_ + (EXTRA)), dim3(kGemmThreads), \
                         kGemmLdsBytes, ST, G, P, tiles_m_, tiles_n_);                            \
    } else {                                                                                      \
      if (set_lds(KERNEL<SlowLoop>) != AXON_OK) return AXON_ERR_LAUNCH;                           \
      hipLaunchKernelGGL(KERNEL<SlowLoop>, dim3(tiles_m_ * tiles_n_), dim3(kGemmThreads),         \
                         kGemmLdsBytes, ST, G, P, tiles_m_, tiles_n_);                            \
    }                                                                                             \
    AXON_CHECK_LAUNCH();                                                                          \
  } while (0)

struct FwdWs {
  float* stats;
  int parts;
  int64_t bytes;
};
FwdWs fwd_ws(int64_t n, int64_t vocab, void* base) {
  FwdWs w;
  w.parts = (int)(round_up(vocab, kTile) / kTile) * 2;
  w.stats = static_cast<float*>(base);
  w.bytes = round_up((int64_t)w.parts * n * 12, kAlign);
  return w;
}

// The stash of a forward for its backward: the tiles' fp16 sub-tiles, then the per-part maxima
// (which the forward then writes there instead of into its workspace).
struct StashWs {
  uint4* tiles;
  float* pm;
  int tiles_m, tiles_n;
  int64_t bytes;
};
StashWs stash_ws(int64_t n, int64_t v, void* base) {
  StashWs w{};
  if (n <= 0) return w;
  w.tiles_m = (int)(round_up(v, kTile) / kTile);
  w.tiles_n = (int)(round_up(n, kTile) / kTile);
  const int64_t tile_bytes = (int64_t)w.tiles_m * w.tiles_n * kStashTileBytes;
  w.tiles = static_cast<uint4*>(base);
  w.pm = reinterpret_cast<float*>(static_cast<char*>(base) + tile_bytes);
  w.bytes = tile_bytes + round_up((int64_t)w.tiles_m * 2 * n * 4, kAlign);
  return w;
}
// The logits that a block's forward keeps in fp32 (kKeepLogits), for the shapes of its main loop; 0 for others.
int64_t logits_bytes(int64_t n, int64_t h, int64_t v) {
  if (n <= 0 || h % DmaLoop::kBK != 0 || h >= kMaxLd) return 0;
  return (round_up(v, kTile) / kTile) * (round_up(n, kTile) / kTile) * kLogitsTileBytes;
}
// The whole-call operator (axon_lmhead_fwd / _bwd) keeps a stash for the shapes its callers have always got
// one for; the block entry points take any shape.
bool stash_of_all_tokens(int64_t n, int64_t h, int64_t v) {
  return n > 0 && (h % 64 != 0 || n < kTile || v < kTile || (n % 4 == 0 && v % 4 == 0));
}

// How many workgroups share a tile's reduction.  dHidden has few tiles (tokens x hidden) and a long reduction (the
// vocabulary): with one workgroup per tile 700 tokens x 4096 keep 48 of the 256 CUs busy and 6007 x 896 keep 96.
// The plan minimises an estimate in thirds of a microsecond.  A k-tile takes 1.33 us per workgroup when all CUs work
// (the part is power-limited then) and 1.0 us when few do; a round of workgroups costs 6 us beside its k-tiles
// (first loads, epilogue); a tile part costs 0.1 us of memory time (256 KB written, then read by
// split_sum_kernel).  Measured (sums included): 48 tiles, K = 151936, 2396 us with one part and 579 with 5; 96
// tiles 2475 and 1183 with 8; 384 tiles (8192 x 2880), K = 201088, 7662 and 6525 with 2; 512 tiles (8192 x 4096)
// stay whole.
// At most kMaxUnits tile parts (three rounds, 200 MB of partial sums, which the Infinity Cache holds).
// A part has at least kMinPartTiles k-tiles: below that its first loads and its epilogue are a quarter of its time.
constexpr int kMaxSplits = 64, kMaxUnits = 3 * kCus, kMinPartTiles = 32;
struct SplitPlan { int splits, k_split; };
// The most parts that a reduction of kt k-tiles is planned in, whatever the number of tiles: the plan's bound and
// what the workspace has room for.
int64_t max_splits(int64_t kt) {
  const int64_t longest = kt / kMinPartTiles;
  return longest < 1 ? 1 : longest < kMaxSplits ? longest : kMaxSplits;
}
SplitPlan split_plan(int64_t tiles, int64_t k) {
  const int64_t kt = (k + 63) / 64, most = max_splits(kt);
  SplitPlan best{1, (int)(kt * 64)};
  int64_t best_cost = INT64_MAX;
  for (int s = 1; s <= most && (s == 1 || tiles * s <= kMaxUnits); ++s) {
    const int64_t per = (kt + s - 1) / s, parts = (kt + per - 1) / per;  // every part gets k-tiles
    if (parts != s) continue;
    const int64_t units = tiles * s, full = units / kCus, rem = units % kCus;
    const int64_t cost = per * 4 * full + (rem ? per * 3 + per * rem / kCus : 0) + 18 * (full + (rem ? 1 : 0)) +
                         (s > 1 ? units / 3 : 0);
    if (cost < best_cost) { best_cost = cost; best = SplitPlan{s, (int)(per * 64)}; }
  }
  return best;
}

// Whether the half-filled last tiles of an output product are computed as half tiles.  What that saves falls with the
// number of tiles beside them; what it costs grows with the reduction: a half tile runs ahead of the whole ones, with
// which it no longer shares operand slices in the L2 (dWeight more than dHidden, whose parts keep an XCD on one part
// of k). Whole / half, ms: dWeight hidden 896 (4 tiles) 3001 tokens (47 k-tiles) 0.671 / 0.611, 8192 1.67 / 1.58,
// 12288 2.53 / 2.45, 16381 3.42 / 3.47; hidden 2880 (12 tiles) 700 tokens 0.847 / 0.789, 3001 2.60 / 2.57, 6007 4.92
// / 4.96, 16381 13.1 / 13.9.  dHidden 896 6007 tokens (297 k-tiles) 1.28 / 1.20, 16381 (2374) 3.26 / 3.13; 2880 3001
// tokens (629) 2.66 / 2.64, 6007 (1571) 6.21 / 6.22, 8192 (1571) 6.72 / 6.76, 16381 (3142) 13.3 / 13.5.
constexpr int64_t kHalfEdgeDw = 768, kHalfEdgeDh = 12288;  // most k-tiles times tiles
bool half_edge(int64_t k, int64_t h, int64_t most) {
  return (h - 1) % kTile < kTile / 2 && (k + 63) / 64 * (round_up(h, kTile) / kTile) <= most;
}

struct BwdWs {
  __bf16 *hT, *dl, *dlT;
  float4* dh_acc;  // dHidden partial sums in tile order: the parts of a split reduction, or carried over the chunks
  int64_t dh_parts;  // how many 256 KB tile parts dh_acc holds
  int64_t v_pad, n_pad, chunk, bytes;
  int64_t ld_n, ld_c;  // leading dimensions of hT/dlT, dl: padded by kLdPad elements
  int chunks;
  // The dWeight GEMM reads dl [token][vocab] as it lies, as its K-major operand: no vocab-major copy
  // (dlT is null).
  bool dl_kmajor;
};
// Rows a power of two apart land on the same L2 sets and memory channels; 128 bytes of padding
// per row moves consecutive rows to consecutive cache lines (+5..13 % on a stand-alone GEMM with
// power-of-two leading dimensions, within noise on the whole backward).
constexpr int64_t kLdPad = 64;
constexpr int64_t kMaxVocabChunk = 1 << 20;  // keeps dl's leading dimension inside kMaxLd
// `n`: the tokens the workspace holds (one call's, or the span of a group of blocks whose weight
// gradient is formed by one GEMM)
BwdWs bwd_ws(int64_t n, int64_t h, int64_t vocab, int64_t chunk, void* base) {
  BwdWs w;
  w.v_pad = round_up(vocab, kTile);
  w.n_pad = round_up(n, kTile);
  w.chunk = chunk;
  if (w.chunk <= 0) {
    const int64_t fit = kDefaultChunkElems / (w.n_pad > 0 ? w.n_pad : kTile) / kTile * kTile;
    w.chunk = fit > kDefaultVocabChunk ? fit : kDefaultVocabChunk;
  }
  if (w.chunk > w.v_pad) w.chunk = w.v_pad;
  if (w.chunk > kMaxVocabChunk) w.chunk = kMaxVocabChunk;
  // not so that a last chunk of less than a tile is left, which would need the second copy of the dlogits
  if (chunk <= 0)
    while (w.chunk > kDefaultVocabChunk && (vocab - 1) % w.chunk + 1 < kTile) w.chunk -= kTile;
  w.chunks = (int)((vocab + w.chunk - 1) / w.chunk);
  w.ld_n = w.n_pad + kLdPad;
  w.ld_c = w.chunk + kLdPad;
  const int64_t last_rows = vocab - (int64_t)(w.chunks - 1) * w.chunk;
  w.dl_kmajor = h >= kTile && last_rows >= kTile && vocab % 8 == 0 && w.ld_n < kMaxLd;
  char* p = static_cast<char*>(base);
  int64_t off = 0;
  w.hT = reinterpret_cast<__bf16*>(p + off);  off += round_up(h * w.ld_n * 2, kAlign);
  w.dl = reinterpret_cast<__bf16*>(p + off);  off += round_up(w.n_pad * w.ld_c * 2, kAlign);
  w.dlT = nullptr;
  if (!w.dl_kmajor) {
    w.dlT = reinterpret_cast<__bf16*>(p + off);
    off += round_up(w.chunk * w.ld_n * 2, kAlign);
  }
  const int64_t dh_tiles = (round_up(h, kTile) / kTile) * (w.n_pad / kTile);
  // room for the parts of any call over at most n tokens (dh_plan), or for one part per tile
  const int64_t most = max_splits(((w.chunks > 1 ? w.chunk : vocab) + 63) / 64);
  int64_t parts = most < 2 ? 0 : dh_tiles * most < kMaxUnits ? dh_tiles * most : kMaxUnits;
  if (w.chunks > 1 && parts < dh_tiles) parts = dh_tiles;
  w.dh_acc = reinterpret_cast<float4*>(p + off);
  w.dh_parts = parts;
  off += parts * kTileAccVecs * 16;
  w.bytes = off;
  return w;
}

// dHidden of a call over `n` tokens: how its tiles' reductions are shared, and the tile parts that it keeps in dh_acc.
struct DhPlan { SplitPlan split; int64_t parts; };
DhPlan dh_plan(const BwdWs& w, int64_t n, int64_t h, int64_t v) {
  const int64_t tiles = (round_up(h, kTile) / kTile) * (round_up(n, kTile) / kTile);
  const SplitPlan split = split_plan(tiles, w.chunks > 1 ? w.chunk : v);
  return DhPlan{split, (w.chunks > 1 || split.splits > 1) ? tiles * split.splits : 0};
}

// Which of the backward's two output products take half tiles: dHidden, each of whose parts reduces over k_split of the
// vocabulary, and dWeight, which reduces over k_dw tokens (the partial sums that are carried from block to block hold
// whole tiles: `carried`).  A hidden size below a tile has no half tiles, nor has dWeight from the vocab-major copy.
struct HalfEdges { bool dh, dw; };
HalfEdges half_edges(const BwdWs& w, const SplitPlan& dh, int64_t h, int64_t k_dw, bool carried) {
  return HalfEdges{h >= kTile && half_edge(dh.k_split, h, kHalfEdgeDh),
                   w.dl_kmajor && !carried && half_edge(k_dw, h, kHalfEdgeDw)};
}

// Whether dWeight over k_dw tokens (padded to whole k-tiles) and vc vocabulary rows is formed from rows of hT held in
// registers (dweight_rows.h): no partial sums carried, dlogits read as they lie, offsets in 32 bits, a long enough walk.
bool dw_by_rows(const BwdWs& w, int64_t h, int64_t vc, int64_t k_dw, bool carried) {
  return !carried && w.dl_kmajor && k_dw <= kDwRowsMaxK && h <= kDwRowsMaxHidden &&
         h * w.ld_n * 2 < (int64_t(1) << 31) && dw_rows_worth(h, vc, k_dw);
}

// Bytes for a call over `n` tokens.  The default chunk shrinks in steps while n grows, so a shorter call can need a
// little more: the most of any call over at most n tokens (beyond 32768 the chunk stays the same).
int64_t bwd_ws_bytes(int64_t n, int64_t h, int64_t vocab, int64_t chunk) {
  int64_t bytes = bwd_ws(n, h, vocab, chunk, nullptr).bytes;
  if (chunk <= 0)
    for (int64_t m = kTile; m < n && m <= kDefaultChunkElems / kDefaultVocabChunk; m += kTile) {
      const int64_t b = bwd_ws(m, h, vocab, chunk, nullptr).bytes;
      bytes = b > bytes ? b : bytes;
    }
  return bytes;
}

// Optional per-phase timing with HIP events on the launch stream (used by the *_timed entry points
// only).  Recording does not synchronise: the events are read when the caller collects them.  A
// null timer costs nothing.
struct PhaseTimer {
  struct Rec { hipEvent_t a, b; int phase; };
  hipStream_t st;
  std::vector<Rec> recs;
  Rec cur{};
  bool open = false;
  int base = 0;  // added to the phase ids of the spans being recorded (0 forward, 4 backward)
  explicit PhaseTimer(hipStream_t s) : st(s) {}
  void begin(int ph) {
    if (hipEventCreate(&cur.a) != hipSuccess) return;
    if (hipEventCreate(&cur.b) != hipSuccess) { (void)hipEventDestroy(cur.a); return; }
    cur.phase = base + ph;
    (void)hipEventRecord(cur.a, st);
    open = true;
  }
  void end() {
    if (!open) return;
    (void)hipEventRecord(cur.b, st);
    recs.push_back(cur);
    open = false;
  }
  // synchronises the stream; adds elapsed ms and launch counts per phase, forgets the spans
  void collect(float* ms, int32_t* launches, int n_phases) {
    (void)hipStreamSynchronize(st);
    for (const Rec& r : recs) {
      float t = 0.f;
      (void)hipEventElapsedTime(&t, r.a, r.b);
      if (r.phase < n_phases) {
        ms[r.phase] += t;
        launches[r.phase] += 1;
      }
      (void)hipEventDestroy(r.a);
      (void)hipEventDestroy(r.b);
    }
    recs.clear();
  }
};
struct Span {  // RAII: one timed span around the launches in scope
  PhaseTimer* t;
  Span(PhaseTimer* timer, int ph) : t(timer) { if (t) t->begin(ph); }
  ~Span() { if (t) t->end(); }
};

int check_head_shape(int64_t n, int64_t h, int64_t v) {
  if (n < 0 || h <= 0 || v <= 0) return AXON_ERR_ARG;
  if (h % 32 != 0) return AXON_ERR_SHAPE;
  if (n >= (1 << 30) || v >= (1 << 30) || h >= (1 << 24)) return AXON_ERR_SHAPE;
  return AXON_OK;
}

int launch_store(const GemmOperands& g, const StoreParams& sp, hipStream_t st) {
  AXON_LAUNCH_GEMM(gemm_store_kernel, g, sp, st);
  return AXON_OK;
}

// The same with operands that are K-major ([k][rows], see DmaLoopT): the rows are fetched as 16-byte
// vectors, so the leading dimension and the base are multiples of 8 elements.  The DMA loop only.  A
// K-contiguous side beside a K-major one is readable, and zero, up to the next multiple of 64 of k.
inline bool kmajor_ok(const void* p, int64_t ld) {
  return ld % 8 == 0 && ld < kMaxLdKMajor && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}
template <class Loop>
int launch_store_loop(const GemmOperands& g, const StoreParams& sp, hipStream_t st) {
  const int tiles_m = (g.m_rows + kTile - 1) / kTile, tiles_n = (g.n_rows + kTile - 1) / kTile;
  if (set_lds(gemm_store_kernel<Loop>) != AXON_OK) return AXON_ERR_LAUNCH;
  hipLaunchKernelGGL(gemm_store_kernel<Loop>, dim3(tiles_m * tiles_n * sp.splits), dim3(kGemmThreads), kGemmLdsBytes, st, g,
                     sp, tiles_m, tiles_n);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}
int launch_store_kmajor(const GemmOperands& g, const StoreParams& sp, bool a_kmajor, bool b_kmajor,
                        hipStream_t st) {
  if (!a_kmajor && !b_kmajor) return launch_store(g, sp, st);
  if (b_kmajor && (g.ldb < kTile || (a_kmajor && g.lda < kTile))) return AXON_ERR_SHAPE;
  if (!(a_kmajor ? kmajor_ok(g.a, g.lda) : kcontig_ok(g.a, g.lda)) ||
      !(b_kmajor ? kmajor_ok(g.b, g.ldb) : kcontig_ok(g.b, g.ldb)))
    return AXON_ERR_SHAPE;
  if (a_kmajor && b_kmajor) return launch_store_loop<DmaLoopT<true, true>>(g, sp, st);
  if (a_kmajor && g.lda < kTile) return launch_store_loop<DmaLoopT<true, false, true>>(g, sp, st);
  if (a_kmajor) return launch_store_loop<DmaLoopT<true, false>>(g, sp, st);
  return launch_store_loop<DmaLoopT<false, true>>(g, sp, st);
}

int launch_transpose(const void* in, int64_t ld_in, int rows, int cols, void* out, int64_t ld_out,
                     int rows_pad, hipStream_t st) {
  if ((ld_in | ld_out) % 8 != 0 ||
      ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15))
    return AXON_ERR_ARG;
  const dim3 grid((rows_pad + 63) / 64, (cols + 63) / 64);
  hipLaunchKernelGGL(transpose_bf16_kernel, grid, dim3(256), 0, st,
                     static_cast<const uint16_t*>(in), ld_in, rows, cols,
                     static_cast<uint16_t*>(out), ld_out, rows_pad);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

// The forward's tiles that are computed in halves of 128 vocabulary rows: those of a last round that would occupy at
// most half of the compute units, so that it takes half as long.  594 tiles, 2.3 rounds: 187 tokens x 896 x 151936 87
// us for 80, 187 x 4096 305 for 288; 128 tiles (250 x 2048 x 32768) 44 for 35.  A last round over more than half of
// them would become two.  Not behind many whole rounds, which then no longer split evenly over the XCDs' ranges of
// the walk and read more from beyond the L2 (8192 x 4096 x 151936 18 to 21 GB for 15).  Whole / half, ms, at hidden
// 4096 x 151936: 9.3 rounds 0.942 / 0.907, 16.2 1.574 / 1.545, 32.5 3.068 / 3.034, 37.1 3.581 / 3.609, 74.3 6.99 /
// 7.13.
constexpr int64_t kHalvedRounds = 36;
int halved_tiles(int64_t n, int64_t v) {
  const int64_t tiles = (round_up(v, kTile) / kTile) * (round_up(n, kTile) / kTile), rest = tiles % kCus;
  return rest <= kCus / 2 && tiles < kHalvedRounds * kCus ? (int)rest : 0;
}

// A call of few tokens has one column of tiles; up to 192 of them it is computed in tiles of 192 or 128 tokens, whose
// products and statistics take three quarters or half of the time: what is left is reading the weight.  Forward with
// 256 / these, us: hidden 896 x 151936 64 tokens 75 / 68, 128 79 / 68, 129 79.5 / 72.7, 192 87 / 81; 2880 x 201088 64
// tokens 243 / 233, 128 250 / 236, 129 249 / 242, 192 262 / 253; 4096 x 151936 128 259 / 245, 192 275 / 270; 2048 x 32768
// 128 35.2 / 33.7, 192 37.2 / 35.5; 1024 x 50257 the same within what runs differ.
int narrow_columns(int64_t n) { return n <= 128 ? 4 : n <= 192 ? 6 : kBlocks; }

template <bool SOFTCAP, Keep KEEP, int BN>
__global__ __launch_bounds__(kGemmThreads) void lmhead_fwd_narrow_kernel(GemmOperands g, FwdParams p, int tiles_m,
                                                                         int tiles_n) {
  fwd_body<DmaLoopT<false, false, false, kBlocks, BN>, SOFTCAP, KEEP>(g, p, tiles_m, tiles_n);
}

template <bool SOFTCAP, Keep KEEP>
int launch_fwd_narrow(const GemmOperands& g, const FwdParams& p, hipStream_t st) {
  auto* const kernel = narrow_columns(g.n_rows) == 4 ? lmhead_fwd_narrow_kernel<SOFTCAP, KEEP, 4>
                                                     : lmhead_fwd_narrow_kernel<SOFTCAP, KEEP, 6>;
  const int tiles_m = (g.m_rows + kTile - 1) / kTile;
  if (set_lds(kernel) != AXON_OK) return AXON_ERR_LAUNCH;
  hipLaunchKernelGGL(kernel, dim3(tiles_m + p.halved), dim3(kGemmThreads), kGemmLdsBytes, st, g, p, tiles_m, 1);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

template <bool SOFTCAP>
int launch_fwd_logits(const GemmOperands& g, const FwdParams& p, hipStream_t st) {
  const int tiles_m = (g.m_rows + kTile - 1) / kTile, tiles_n = (g.n_rows + kTile - 1) / kTile;
  if (!dma_ok(g)) return AXON_ERR_SHAPE;
  if (set_lds(lmhead_fwd_logits_kernel<SOFTCAP>) != AXON_OK) return AXON_ERR_LAUNCH;
  hipLaunchKernelGGL(lmhead_fwd_logits_kernel<SOFTCAP>, dim3(tiles_m * tiles_n + p.halved), dim3(kGemmThreads),
                     kGemmLdsBytes, st, g, p, tiles_m, tiles_n);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

int fwd_impl(const void* hidden, const void* weight, const void* labels, int labels_i64, int64_t n,
             int64_t h, int64_t v, float inv_temp, float softcap, const uint8_t* is_start,
             int64_t last_dst, float* logprobs, float* entropy, float* lse, float* entropy_b,
             void* workspace, int64_t ws_bytes, void* stash, int64_t stash_bytes, void* stream,
             PhaseTimer* timer, bool is_block = false, Keep keep = kKeepStash) {
  int rc = check_head_shape(n, h, v);
  if (rc != AXON_OK) return rc;
  if (n == 0) return AXON_OK;
  if (!hidden || !weight || !labels || !logprobs || !entropy || !lse || !entropy_b || !workspace)
    return AXON_ERR_ARG;
  if (!(inv_temp > 0.f) || !(softcap >= 0.f)) return AXON_ERR_ARG;
  if ((reinterpret_cast<uintptr_t>(hidden) | reinterpret_cast<uintptr_t>(weight)) & 15)
    return AXON_ERR_ARG;
  char* base = reinterpret_cast<char*>(round_up(reinterpret_cast<int64_t>(workspace), kAlign));
  FwdWs w = fwd_ws(n, v, base);
  if ((base - static_cast<char*>(workspace)) + w.bytes > ws_bytes) return AXON_ERR_WORKSPACE;
  const hipStream_t st = (hipStream_t)stream;
  StashWs sw{};
  float* pm = nullptr;
  if (stash) {
    if (reinterpret_cast<uintptr_t>(stash) & 15) return AXON_ERR_ARG;
    if (keep == kKeepLogits) {
      const int64_t bytes = logits_bytes(n, h, v);
      if (bytes == 0) return AXON_ERR_SHAPE;
      if (bytes > stash_bytes) return AXON_ERR_WORKSPACE;
      sw.tiles = static_cast<uint4*>(stash);
    } else {
      if (!is_block && !stash_of_all_tokens(n, h, v)) return AXON_ERR_SHAPE;
      sw = stash_ws(n, v, stash);
      if (sw.bytes > stash_bytes) return AXON_ERR_WORKSPACE;
      pm = sw.pm;  // the backward needs the per-part maxima as well: they live in the stash
    }
  }

  GemmOperands g;
  g.a = static_cast<const __bf16*>(weight);  g.lda = h;  g.m_rows = (int)v;
  g.b = static_cast<const __bf16*>(hidden);  g.ldb = h;  g.n_rows = (int)n;
  g.k = (int)h;
  FwdParams p{w.stats, pm, (int)n, (int)v, inv_temp * kLog2e, softcap,
              softcap > 0.f ? 1.f / softcap : 0.f, sw.tiles, dma_ok(g) ? halved_tiles(n, v) : 0};
  {
    Span span(timer, 0);
    if (stash && keep == kKeepLogits) {
      rc = softcap > 0.f ? launch_fwd_logits<true>(g, p, st) : launch_fwd_logits<false>(g, p, st);
      if (rc != AXON_OK) return rc;
    } else if (dma_ok(g) && narrow_columns(n) < kBlocks) {
      rc = stash ? softcap > 0.f ? launch_fwd_narrow<true, kKeepStash>(g, p, st)
                                 : launch_fwd_narrow<false, kKeepStash>(g, p, st)
                 : softcap > 0.f ? launch_fwd_narrow<true, kKeepNone>(g, p, st)
                                 : launch_fwd_narrow<false, kKeepNone>(g, p, st);
      if (rc != AXON_OK) return rc;
    } else if (stash) {
      if (softcap > 0.f)
        AXON_LAUNCH_GEMM_PLUS(lmhead_fwd_softcap_stash_kernel, g, p, st, p.halved);
      else
        AXON_LAUNCH_GEMM_PLUS(lmhead_fwd_stash_kernel, g, p, st, p.halved);
    } else if (softcap > 0.f) {
      AXON_LAUNCH_GEMM_PLUS(lmhead_fwd_softcap_kernel, g, p, st, p.halved);
    } else {
      AXON_LAUNCH_GEMM_PLUS(lmhead_fwd_kernel, g, p, st, p.halved);
    }
  }
  Span span(timer, 1);
#define AXON_FINISH(T, PER)                                                                                       \
  do {                                                                                                           \
    const dim3 grid((unsigned)((n + T * PER - 1) / (T * PER)));                                                  \
    if (labels_i64) AXON_FINISH_L(T, PER, int64_t); else AXON_FINISH_L(T, PER, int32_t);                         \
  } while (0)
#define AXON_FINISH_L(T, PER, LabelT)                                                                            \
  hipLaunchKernelGGL((lmhead_finish_kernel<T, PER, LabelT>), grid, dim3(1024), 0, st, w.stats, w.parts,          \
                     static_cast<const __bf16*>(hidden), static_cast<const __bf16*>(weight),                     \
                     static_cast<const LabelT*>(labels), (int)n, (int)h, (int)v, inv_temp, softcap, lse,         \
                     entropy_b, entropy, logprobs, is_start, (int)last_dst)
  if (n <= 4 * kCus) AXON_FINISH(4, 1);
  else if (n <= 16 * kCus) AXON_FINISH(16, 1);
  else AXON_FINISH(16, 2);
#undef AXON_FINISH_L
#undef AXON_FINISH
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

// A backward over a block of consecutive tokens of a longer stream (one call per block, one stream):
// where the last row's label and gradients live (aligned_pos), and how this block's share of the weight
// gradient leaves: the blocks of a step add up in one fp32 array, the last one rounds the sum to bf16.
enum { kDwStore = 0, kDwFirst = 1, kDwAdd = 2, kDwLast = 3 };
struct BlockArgs {
  bool is_block = false;  // a stash for any shape, as the caller decides; else the shapes of stash_of_all_tokens
  Keep keep = kKeepStash;  // what the buffer beside the forward's holds
  int64_t last_dst = 0;
  int dw_mode = kDwStore;
  float* dw_acc = nullptr;  // axon_lmhead_block_dw_acc_bytes of fp32 partial sums, tile order (modes other than kDwStore)
  // Several consecutive blocks may share ONE weight-gradient GEMM (a longer reduction, fewer passes over
  // the fp32 partial sums): each keeps its dlogits and its transposed hidden rows in the workspace, at
  // `group_pos` tokens from the start (a multiple of 256, the blocks before it rounded up to that), and
  // the GEMM runs with the block that says `dw_now` over everything up to its end.  `ws_tokens`: the
  // tokens the workspace was sized for (0: this call's), the same for every call that shares it.
  int64_t group_pos = 0;
  int dw_now = 1;
  int64_t ws_tokens = 0;
};

int bwd_impl(const float* dlogprobs, const float* dentropy, const void* hidden, const void* weight,
             const void* labels, int labels_i64, const float* lse, const float* entropy_b,
             int64_t n, int64_t h, int64_t v, float inv_temp, float softcap,
             const uint8_t* is_start, void* d_hidden, void* d_weight, int64_t chunk, void* workspace,
             int64_t ws_bytes, const void* stash, int64_t stash_bytes, void* stream, PhaseTimer* timer,
             const BlockArgs& blk = BlockArgs()) {
  int rc = check_head_shape(n, h, v);
  if (rc != AXON_OK) return rc;
  if (chunk < 0 || chunk % kTile != 0) return AXON_ERR_ARG;
  if (!weight) return AXON_ERR_ARG;
  if (blk.dw_mode < kDwStore || blk.dw_mode > kDwLast) return AXON_ERR_ARG;
  if (blk.dw_mode != kDwStore && (!blk.dw_acc || (reinterpret_cast<uintptr_t>(blk.dw_acc) & 15) || n == 0))
    return AXON_ERR_ARG;
  const bool dw_bf16 = blk.dw_now && (blk.dw_mode == kDwStore || blk.dw_mode == kDwLast);
  if (dw_bf16 && !d_weight) return AXON_ERR_ARG;
  const hipStream_t st = (hipStream_t)stream;
  if (n == 0) return axon_fill_zero(d_weight, v * h * 2, stream);
  if (!dlogprobs || !hidden || !labels || !lse || !entropy_b || !d_hidden || !workspace)
    return AXON_ERR_ARG;
  if (!(inv_temp > 0.f) || !(softcap >= 0.f)) return AXON_ERR_ARG;
  if ((reinterpret_cast<uintptr_t>(hidden) | reinterpret_cast<uintptr_t>(weight) |
       reinterpret_cast<uintptr_t>(d_hidden) | (dw_bf16 ? reinterpret_cast<uintptr_t>(d_weight) : 0)) & 15)
    return AXON_ERR_ARG;
  const int64_t pos = blk.group_pos, n_tile = round_up(n, kTile);
  const int64_t ws_tokens = blk.ws_tokens > 0 ? blk.ws_tokens : n;
  if (pos < 0 || pos % kTile != 0 || pos + n_tile > round_up(ws_tokens, kTile)) return AXON_ERR_ARG;
  char* base = reinterpret_cast<char*>(round_up(reinterpret_cast<int64_t>(workspace), kAlign));
  const BwdWs w = bwd_ws(ws_tokens, h, v, chunk, base);
  if ((base - static_cast<char*>(workspace)) + w.bytes > ws_bytes) return AXON_ERR_WORKSPACE;
  const DhPlan dh = dh_plan(w, n, h, v);
  const SplitPlan plan = dh.split;
  if (dh.parts > w.dh_parts) return AXON_ERR_WORKSPACE;
  // blocks that share a weight-gradient GEMM keep their dlogits of the whole vocabulary side by side
  if ((pos > 0 || !blk.dw_now) && !(w.dl_kmajor && w.chunks == 1)) return AXON_ERR_ARG;
  StashWs sw{};
  if (stash) {
    if (reinterpret_cast<uintptr_t>(stash) & 15) return AXON_ERR_ARG;
    if (!blk.is_block && !stash_of_all_tokens(n, h, v)) return AXON_ERR_SHAPE;
    sw = stash_ws(n, v, const_cast<void*>(stash));
    const int64_t bytes = blk.keep == kKeepLogits ? logits_bytes(n, h, v) : sw.bytes;
    if (bytes == 0) return AXON_ERR_SHAPE;
    if (bytes > stash_bytes) return AXON_ERR_WORKSPACE;
  }

  // the hidden states K-contiguous for the weight gradient, zeros up to the tile border
  {
    Span span(timer, 0);
    rc = launch_transpose(hidden, h, (int)n, (int)h, w.hT + pos, w.ld_n, (int)n_tile, st);
    if (rc != AXON_OK) return rc;
  }
  const int64_t n_red = round_up(n, 64);  // reduction length of B3 (from this block's first token)
  const int64_t tiles_h = round_up(h, kTile) / kTile;
  const HalfEdges half = half_edges(w, plan, h, pos + n_red, blk.dw_mode != kDwStore);
  __bf16* const dl = w.dl + pos * w.ld_c;  // this block's rows

  for (int ci = 0; ci < w.chunks; ++ci) {
    const int64_t v0 = (int64_t)ci * w.chunk;
    const int64_t vc = (v - v0 < w.chunk) ? (v - v0) : w.chunk;  // valid vocab rows in this chunk
    // B1: dlogit for vocab rows [v0, v0 + vc); zeros beyond the last token (up to n_end) and the last vocabulary row
    {
      Span span(timer, 1);
      GemmOperands g;
      g.a = static_cast<const __bf16*>(weight) + v0 * h;  g.lda = h;  g.m_rows = (int)vc;
      g.b = static_cast<const __bf16*>(hidden);            g.ldb = h;  g.n_rows = (int)n;
      g.k = (int)h;
      DlogitParams p;
      p.lse = lse; p.entropy_b = entropy_b; p.dlogprobs = dlogprobs; p.dentropy = dentropy;
      p.labels = labels; p.labels_i64 = labels_i64;
      p.dl = dl; p.dlT = w.dlT; p.ld_dl = w.ld_c; p.ld_dlT = w.ld_n;
      p.n_tokens = (int)n; p.vocab = (int)v; p.v_begin = (int)v0; p.inv_temp = inv_temp;
      p.cap = softcap; p.inv_cap = softcap > 0.f ? 1.f / softcap : 0.f;
      p.is_start = is_start;
      p.last_dst = (int)blk.last_dst;
      // a block with others behind it in the same weight-gradient GEMM: whole tiles, its rows lie between theirs
      p.n_end = (int)(blk.dw_now ? n_red : n_tile);
      if (stash) {
        const StashSource src{sw.tiles, sw.pm, sw.tiles_n, (int)(v0 / kTile)};
        const unsigned blocks = (unsigned)(round_up(vc, kTile) / kTile) * (unsigned)sw.tiles_n * 8u;
        auto* const kernel = blk.keep == kKeepLogits
                                 ? (softcap > 0.f ? lmhead_dlogit_logits_kernel<true> : lmhead_dlogit_logits_kernel<false>)
                             : softcap > 0.f
                                 ? (dentropy ? lmhead_dlogit_stash_kernel<true, true> : lmhead_dlogit_stash_kernel<true, false>)
                                 : (dentropy ? lmhead_dlogit_stash_kernel<false, true>
                                             : lmhead_dlogit_stash_kernel<false, false>);
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64), 0, st, p, src);
        AXON_CHECK_LAUNCH();
      } else if (softcap > 0.f) {
        AXON_LAUNCH_GEMM(lmhead_dlogit_softcap_kernel, g, p, st);
      } else {
        AXON_LAUNCH_GEMM(lmhead_dlogit_kernel, g, p, st);
      }
    }
    // B2: dHidden[n][h] (+)= sum_v dl[n][v] * W[v0 + v][h], the weight read K-major where it lies
    {
      Span span(timer, 2);
      GemmOperands g;
      g.a = static_cast<const __bf16*>(weight) + v0 * h;  g.lda = h;  g.m_rows = (int)h;
      g.b = dl;  g.ldb = w.ld_c;  g.n_rows = (int)n;
      g.k = (int)vc;
      const bool last = (ci == w.chunks - 1), split = plan.splits > 1;
      StoreParams sp;
      sp.out_bf16 = (last && !split) ? static_cast<__bf16*>(d_hidden) : nullptr;  sp.ld_bf16 = h;
      sp.m_valid = (int)h; sp.n_valid = (int)n;
      sp.tile_acc = (w.chunks > 1 || split) ? w.dh_acc : nullptr;
      sp.accumulate = (ci > 0); sp.keep_f32 = split || !last;
      sp.half_edge = half.dh;
      // a shorter last chunk reaches the first parts only
      sp.k_split = plan.k_split;
      sp.splits = (int)((vc + sp.k_split - 1) / sp.k_split);
      rc = launch_store_kmajor(g, sp, true, false, st);
      if (rc != AXON_OK) return rc;
      if (last && split) {
        const int tiles_m = (int)tiles_h, tiles_n = (int)(n_tile / kTile);
        hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)(tiles_m * tiles_n * (kTileAccVecs / 256))), dim3(256), 0, st,
                           w.dh_acc, plan.splits, tiles_m, tiles_n, (int)h, (int)n,
                           static_cast<__bf16*>(d_hidden), h);
        AXON_CHECK_LAUNCH();
      }
    }
    // B3: dWeight[v0 + v][h] = sum_t dl[t][v] * hT[h][t] over the tokens the workspace holds up to this
    // block's end (dl read as the K-major operand, or its vocab-major copy dlT[v][t])
    if (blk.dw_now) {
      Span span(timer, 3);
      GemmOperands g;
      g.a = w.hT;  g.lda = w.ld_n;  g.m_rows = (int)h;
      if (w.dl_kmajor) { g.b = w.dl;   g.ldb = w.ld_c; }
      else             { g.b = w.dlT;  g.ldb = w.ld_n; }
      g.n_rows = (int)vc;
      g.k = (int)(pos + n_red);
      StoreParams sp;
      sp.tile_acc = blk.dw_mode == kDwStore
                        ? nullptr
                        : reinterpret_cast<float4*>(blk.dw_acc) + (v0 / kTile) * tiles_h * kTileAccVecs;
      sp.out_bf16 = dw_bf16 ? static_cast<__bf16*>(d_weight) + v0 * h : nullptr;  sp.ld_bf16 = h;
      sp.m_valid = (int)h; sp.n_valid = (int)vc;
      sp.accumulate = blk.dw_mode == kDwAdd || blk.dw_mode == kDwLast;
      sp.keep_f32 = blk.dw_mode != kDwLast;
      sp.splits = 1; sp.k_split = g.k;
      sp.half_edge = half.dw;
      rc = dw_by_rows(w, h, vc, g.k, blk.dw_mode != kDwStore) ? launch_dw_rows(g, sp.out_bf16, sp.ld_bf16, st)
                                                              : launch_store_kmajor(g, sp, false, w.dl_kmajor, st);
      if (rc != AXON_OK) return rc;
    }
  }
  return AXON_OK;
}

}  // namespace


extern "C" int axon_seq_start_flags(const int32_t* cu_seqlens, int64_t n_seqs, int64_t n_tokens,
                                    uint8_t* flags, void* stream) {
  if (n_seqs < 0 || n_tokens < 0 || n_tokens >= (int64_t)INT32_MAX || n_seqs >= (int64_t)INT32_MAX)
    return AXON_ERR_SHAPE;
  if (n_tokens == 0) return AXON_OK;
  if (!flags || (n_seqs > 0 && !cu_seqlens)) return AXON_ERR_ARG;
  const int64_t words = (n_tokens + 3) / 4;
  hipLaunchKernelGGL(seq_start_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     cu_seqlens, (int)n_seqs, (int)n_tokens, reinterpret_cast<AnyWord*>(flags));
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_lmhead_active_rows(const float* dlogprobs, const float* dentropy,
                                       const uint8_t* seq_start, int64_t n, int32_t* row_index,
                                       int32_t* row_rank, int32_t* count, void* stream) {
  if (n < 0 || n >= (int64_t)INT32_MAX - 8192) return AXON_ERR_SHAPE;  // the walk steps by 4096
  if (!count) return AXON_ERR_ARG;
  if (n > 0 && (!dlogprobs || !row_index || !row_rank)) return AXON_ERR_ARG;
  hipLaunchKernelGGL(active_rows_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, dlogprobs,
                     dentropy, seq_start, (int)n, row_index, row_rank, count);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_lmhead_gather_rows(const void* hidden, const void* labels, int labels_i64,
                                       const float* lse, const float* entropy_b,
                                       const float* dlogprobs, const float* dentropy,
                                       const uint8_t* seq_start, int64_t n, int64_t h,
                                       const int32_t* row_index, int64_t n_active, void* hidden_c,
                                       void* labels_c, float* lse_c, float* entropy_b_c,
                                       float* dlogprobs_c, float* dentropy_c, void* stream) {
  if (n < 0 || n >= (int64_t)INT32_MAX || n_active < 0 || n_active > n) return AXON_ERR_SHAPE;
  if (h < 8 || h % 8 != 0 || h / 8 >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (n_active == 0) return AXON_OK;
  if (!hidden || !labels || !lse || !entropy_b || !dlogprobs || !row_index || !hidden_c ||
      !labels_c || !lse_c || !entropy_b_c || !dlogprobs_c)
    return AXON_ERR_ARG;
  if ((reinterpret_cast<uintptr_t>(hidden) | reinterpret_cast<uintptr_t>(hidden_c)) & 15)
    return AXON_ERR_ARG;
  const dim3 grid((unsigned)n_active), block(256);
  const hipStream_t st = (hipStream_t)stream;
  if (labels_i64)
    hipLaunchKernelGGL(gather_rows_kernel<int64_t>, grid, block, 0, st,
                       static_cast<const uint4*>(hidden), (int)(h / 8),
                       static_cast<const int64_t*>(labels), lse, entropy_b, dlogprobs, dentropy,
                       seq_start, (int)n, row_index, static_cast<uint4*>(hidden_c),
                       static_cast<int64_t*>(labels_c), lse_c, entropy_b_c, dlogprobs_c, dentropy_c);
  else
    hipLaunchKernelGGL(gather_rows_kernel<int32_t>, grid, block, 0, st,
                       static_cast<const uint4*>(hidden), (int)(h / 8),
                       static_cast<const int32_t*>(labels), lse, entropy_b, dlogprobs, dentropy,
                       seq_start, (int)n, row_index, static_cast<uint4*>(hidden_c),
                       static_cast<int32_t*>(labels_c), lse_c, entropy_b_c, dlogprobs_c, dentropy_c);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_lmhead_scatter_rows(const void* d_hidden_c, const int32_t* row_rank, int64_t n,
                                        int64_t h, void* d_hidden, void* stream) {
  if (n < 0 || n >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (h < 8 || h % 8 != 0 || h / 8 >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (n == 0) return AXON_OK;
  if (!row_rank || !d_hidden) return AXON_ERR_ARG;  // d_hidden_c may be NULL when no row is active
  if ((reinterpret_cast<uintptr_t>(d_hidden_c) | reinterpret_cast<uintptr_t>(d_hidden)) & 15)
    return AXON_ERR_ARG;
  hipLaunchKernelGGL(scatter_rows_kernel, dim3((unsigned)n), dim3(256), 0, (hipStream_t)stream,
                     static_cast<const uint4*>(d_hidden_c), row_rank, (int)(h / 8),
                     static_cast<uint4*>(d_hidden));
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int64_t axon_lmhead_fwd_workspace_bytes(int64_t n, int64_t h, int64_t v) {
  if (check_head_shape(n, h, v) != AXON_OK) return -1;
  return fwd_ws(n, v, nullptr).bytes + kAlign;
}

extern "C" int64_t axon_lmhead_stash_bytes(int64_t n, int64_t h, int64_t v) {
  if (check_head_shape(n, h, v) != AXON_OK) return -1;
  return stash_of_all_tokens(n, h, v) ? stash_ws(n, v, nullptr).bytes : 0;
}

extern "C" int64_t axon_lmhead_block_stash_bytes(int64_t n, int64_t h, int64_t v) {
  if (check_head_shape(n, h, v) != AXON_OK) return -1;
  return stash_ws(n, v, nullptr).bytes;
}

extern "C" int axon_lmhead_fwd(const void* hidden, const void* weight, const void* labels,
                               int labels_i64, int64_t n, int64_t h, int64_t v, float inv_temp,
                               float softcap, const uint8_t* seq_start, float* logprobs,
                               float* entropy, float* lse, float* entropy_b, void* workspace,
                               int64_t ws_bytes, void* stash, int64_t stash_bytes, void* stream) {
  return fwd_impl(hidden, weight, labels, labels_i64, n, h, v, inv_temp, softcap, seq_start, 0,
                  logprobs, entropy, lse, entropy_b, workspace, ws_bytes, stash, stash_bytes, stream,
                  nullptr);
}

extern "C" void* axon_timer_create(void* stream) { return new (std::nothrow) PhaseTimer((hipStream_t)stream); }

extern "C" int axon_timer_collect(void* timer, float* phase_ms, int32_t* phase_launches) {
  if (!timer || !phase_ms || !phase_launches) return AXON_ERR_ARG;
  static_cast<PhaseTimer*>(timer)->collect(phase_ms, phase_launches, 8);
  return AXON_OK;
}

extern "C" void axon_timer_destroy(void* timer) {
  if (!timer) return;
  float ms[8] = {0};
  int32_t n[8] = {0};
  static_cast<PhaseTimer*>(timer)->collect(ms, n, 8);  // releases the events
  delete static_cast<PhaseTimer*>(timer);
}

extern "C" int axon_lmhead_fwd_timed(const void* hidden, const void* weight, const void* labels,
                                     int labels_i64, int64_t n, int64_t h, int64_t v,
                                     float inv_temp, float softcap, const uint8_t* seq_start,
                                     float* logprobs, float* entropy, float* lse,
                                     float* entropy_b, void* workspace, int64_t ws_bytes,
                                     void* stash, int64_t stash_bytes, void* stream, void* timer) {
  if (!timer) return AXON_ERR_ARG;
  PhaseTimer* t = static_cast<PhaseTimer*>(timer);
  if (t->st != (hipStream_t)stream) return AXON_ERR_ARG;
  t->base = 0;
  return fwd_impl(hidden, weight, labels, labels_i64, n, h, v, inv_temp, softcap, seq_start, 0, logprobs,
                  entropy, lse, entropy_b, workspace, ws_bytes, stash, stash_bytes, stream, t);
}

extern "C" int64_t axon_lmhead_bwd_workspace_bytes(int64_t n, int64_t h, int64_t v,
                                                   int64_t chunk) {
  if (check_head_shape(n, h, v) != AXON_OK) return -1;
  if (chunk < 0 || chunk % kTile != 0) return -1;
  return bwd_ws_bytes(n, h, v, chunk) + kAlign;
}

extern "C" int axon_lmhead_bwd(const float* dlogprobs, const float* dentropy, const void* hidden,
                               const void* weight, const void* labels, int labels_i64,
                               const float* lse, const float* entropy_b, int64_t n, int64_t h,
                               int64_t v, float inv_temp, float softcap, const uint8_t* seq_start,
                               void* d_hidden, void* d_weight, int64_t chunk, void* workspace,
                               int64_t ws_bytes, const void* stash, int64_t stash_bytes, void* stream) {
  return bwd_impl(dlogprobs, dentropy, hidden, weight, labels, labels_i64, lse, entropy_b, n, h, v,
                  inv_temp, softcap, seq_start, d_hidden, d_weight, chunk, workspace, ws_bytes,
                  stash, stash_bytes, stream, nullptr);
}

extern "C" int axon_lmhead_bwd_timed(const float* dlogprobs, const float* dentropy,
                                     const void* hidden, const void* weight, const void* labels,
                                     int labels_i64, const float* lse, const float* entropy_b,
                                     int64_t n, int64_t h, int64_t v, float inv_temp,
                                     float softcap, const uint8_t* seq_start, void* d_hidden,
                                     void* d_weight, int64_t chunk, void* workspace,
                                     int64_t ws_bytes, const void* stash, int64_t stash_bytes,
                                     void* stream, void* timer) {
  if (!timer) return AXON_ERR_ARG;
  PhaseTimer* t = static_cast<PhaseTimer*>(timer);
  if (t->st != (hipStream_t)stream) return AXON_ERR_ARG;
  t->base = 4;
  return bwd_impl(dlogprobs, dentropy, hidden, weight, labels, labels_i64, lse, entropy_b, n, h, v,
                  inv_temp, softcap, seq_start, d_hidden, d_weight, chunk, workspace, ws_bytes, stash,
                  stash_bytes, stream, t);
}

extern "C" int axon_gemm_nt_bf16(const void* a, int64_t lda, const void* b, int64_t ldb, float* out,
                                 int64_t ldo, int64_t m, int64_t n, int64_t k, void* stream) {
  if (!a || !b || !out) return AXON_ERR_ARG;
  if (m <= 0 || n <= 0 || k <= 0) return AXON_ERR_ARG;
  if (k % 32 != 0 || lda % 8 != 0 || ldb % 8 != 0 || m % 4 != 0 || ldo % 4 != 0)
    return AXON_ERR_SHAPE;
  if (m >= (1 << 30) || n >= (1 << 30)) return AXON_ERR_SHAPE;
  GemmOperands g;
  g.a = static_cast<const __bf16*>(a);  g.lda = lda;  g.m_rows = (int)m;
  g.b = static_cast<const __bf16*>(b);  g.ldb = ldb;  g.n_rows = (int)n;
  g.k = (int)k;
  StoreParams sp;
  sp.out_f32 = out; sp.ld_f32 = ldo;
  sp.m_valid = (int)m; sp.n_valid = (int)n;
  sp.k_split = (int)k;
  return launch_store(g, sp, (hipStream_t)stream);
}

// The K-major forms of the plain GEMM keep the domain their documentation states.
static bool gemm_kmajor_domain(const GemmOperands& g, bool a_kmajor, bool b_kmajor) {
  return (!a_kmajor && !b_kmajor) || (g.m_rows >= kTile && g.n_rows >= kTile && g.k % 64 == 0 &&
                                      (!a_kmajor || g.m_rows % 8 == 0) && (!b_kmajor || g.n_rows % 8 == 0));
}

extern "C" int axon_gemm_bf16(const void* a, int64_t lda, int a_kmajor, const void* b, int64_t ldb,
                              int b_kmajor, float* out, int64_t ldo, int64_t m, int64_t n, int64_t k,
                              void* stream) {
  if (!a || !b || !out) return AXON_ERR_ARG;
  if (m <= 0 || n <= 0 || k <= 0) return AXON_ERR_ARG;
  if (k % 32 != 0 || lda % 8 != 0 || ldb % 8 != 0 || m % 4 != 0 || ldo % 4 != 0) return AXON_ERR_SHAPE;
  if (m >= (1 << 30) || n >= (1 << 30)) return AXON_ERR_SHAPE;
  GemmOperands g;
  g.a = static_cast<const __bf16*>(a);  g.lda = lda;  g.m_rows = (int)m;
  g.b = static_cast<const __bf16*>(b);  g.ldb = ldb;  g.n_rows = (int)n;
  g.k = (int)k;
  if (!gemm_kmajor_domain(g, a_kmajor != 0, b_kmajor != 0)) return AXON_ERR_SHAPE;
  StoreParams sp;
  sp.out_f32 = out; sp.ld_f32 = ldo;
  sp.m_valid = (int)m; sp.n_valid = (int)n;
  sp.k_split = (int)k;
  return launch_store_kmajor(g, sp, a_kmajor != 0, b_kmajor != 0, (hipStream_t)stream);
}

// ----------------------------------------------------------------------------
// One step as token blocks: forward (with stash), loss and backward of one block of consecutive
// tokens before the next block's forward, so that what is kept from a forward to its backward is
// one block's stash whatever the number of tokens.  One call per block and phase, all on one stream.
// ----------------------------------------------------------------------------
namespace {
PhaseTimer* block_timer(void* timer, void* stream, int base, int* rc) {
  *rc = AXON_OK;
  if (!timer) return nullptr;
  PhaseTimer* t = static_cast<PhaseTimer*>(timer);
  if (t->st != (hipStream_t)stream) { *rc = AXON_ERR_ARG; return nullptr; }
  t->base = base;
  return t;
}
bool last_dst_ok(int64_t last_dst, int64_t n) { return last_dst <= n && last_dst > -(int64_t(1) << 30); }
}  // namespace

extern "C" int64_t axon_lmhead_block_dw_acc_bytes(int64_t h, int64_t v) {
  if (check_head_shape(0, h, v) != AXON_OK) return -1;
  return (round_up(h, kTile) / kTile) * (round_up(v, kTile) / kTile) * kTileAccVecs * 16;
}

extern "C" int axon_lmhead_bwd_dlogit_copies_of(int64_t n, int64_t h, int64_t v, int64_t chunk) {
  if (check_head_shape(n, h, v) != AXON_OK || chunk < 0 || chunk % kTile != 0) return -1;
  return bwd_ws(n, h, v, chunk, nullptr).dl_kmajor ? 1 : 2;
}

extern "C" int axon_lmhead_bwd_dlogit_copies(int64_t h, int64_t v, int64_t chunk) {
  return axon_lmhead_bwd_dlogit_copies_of(kTile, h, v, chunk == 0 ? kDefaultVocabChunk : chunk);
}

extern "C" int64_t axon_lmhead_bwd_dhidden_parts(int64_t n, int64_t ws_tokens, int64_t h, int64_t v, int64_t chunk,
                                                 int64_t* reserved) {
  int rc = check_head_shape(n, h, v);
  if (rc == AXON_OK) rc = check_head_shape(ws_tokens, h, v);
  if (rc != AXON_OK) return rc;
  if (!reserved || chunk < 0 || chunk % kTile != 0 || n > ws_tokens) return AXON_ERR_ARG;
  const BwdWs w = bwd_ws(ws_tokens, h, v, chunk, nullptr);
  *reserved = w.dh_parts;
  return n > 0 ? dh_plan(w, n, h, v).parts : 0;
}

extern "C" int axon_lmhead_bwd_half_tiles(int64_t n, int64_t ws_tokens, int64_t h, int64_t v, int64_t chunk) {
  int rc = check_head_shape(n, h, v);
  if (rc == AXON_OK) rc = check_head_shape(ws_tokens, h, v);
  if (rc != AXON_OK) return rc;
  if (n == 0 || chunk < 0 || chunk % kTile != 0 || n > ws_tokens) return AXON_ERR_ARG;
  const BwdWs w = bwd_ws(ws_tokens, h, v, chunk, nullptr);
  const HalfEdges half = half_edges(w, dh_plan(w, n, h, v).split, h, round_up(n, 64), false);
  return (half.dh ? 1 : 0) + (half.dw && !dw_by_rows(w, h, v < w.chunk ? v : w.chunk, round_up(n, 64), false) ? 2 : 0);
}

extern "C" int axon_lmhead_bwd_dweight_by_rows(int64_t n, int64_t ws_tokens, int64_t h, int64_t v, int64_t chunk) {
  int rc = check_head_shape(n, h, v);
  if (rc == AXON_OK) rc = check_head_shape(ws_tokens, h, v);
  if (rc != AXON_OK) return rc;
  if (n == 0 || chunk < 0 || chunk % kTile != 0 || n > ws_tokens) return AXON_ERR_ARG;
  const BwdWs w = bwd_ws(ws_tokens, h, v, chunk, nullptr);
  return dw_by_rows(w, h, v < w.chunk ? v : w.chunk, round_up(n, 64), false) ? 1 : 0;
}

extern "C" int axon_lmhead_block_can_group(int64_t h, int64_t v, int64_t chunk) {
  if (check_head_shape(0, h, v) != AXON_OK || chunk < 0 || chunk % kTile != 0) return 0;
  const BwdWs w = bwd_ws(kTile, h, v, chunk > 0 ? chunk : kDefaultVocabChunk, nullptr);
  return (w.dl_kmajor && w.chunks == 1) ? 1 : 0;
}

extern "C" int axon_lmhead_block_begin(const void* weight, int64_t h, int64_t v, int64_t chunk,
                                       void* workspace, int64_t /*ws_bytes*/, void* stream, void* timer) {
  int rc = check_head_shape(0, h, v);
  if (rc != AXON_OK) return rc;
  if (chunk < 0 || chunk % kTile != 0) return AXON_ERR_ARG;
  if (!weight || !workspace || (reinterpret_cast<uintptr_t>(weight) & 15)) return AXON_ERR_ARG;
  (void)block_timer(timer, stream, 4, &rc);
  return rc;
}

extern "C" int64_t axon_lmhead_block_logits_bytes(int64_t n, int64_t h, int64_t v) {
  if (check_head_shape(n, h, v) != AXON_OK) return -1;
  return logits_bytes(n, h, v);
}

static int block_fwd(const void* hidden, const void* weight, const void* labels, int labels_i64, int64_t n,
                     int64_t h, int64_t v, float inv_temp, float softcap, const uint8_t* seq_start,
                     int64_t last_dst, float* logprobs, float* entropy, float* lse, float* entropy_b,
                     void* workspace, int64_t ws_bytes, void* stash, int64_t stash_bytes, void* stream,
                     void* timer, Keep keep) {
  if (!last_dst_ok(last_dst, n)) return AXON_ERR_ARG;
  int rc;
  PhaseTimer* t = block_timer(timer, stream, 0, &rc);
  if (rc != AXON_OK) return rc;
  return fwd_impl(hidden, weight, labels, labels_i64, n, h, v, inv_temp, softcap, seq_start, last_dst,
                  logprobs, entropy, lse, entropy_b, workspace, ws_bytes, stash, stash_bytes, stream, t, true, keep);
}

extern "C" int axon_lmhead_block_fwd(const void* hidden, const void* weight, const void* labels, int labels_i64,
                                     int64_t n, int64_t h, int64_t v, float inv_temp, float softcap,
                                     const uint8_t* seq_start, int64_t last_dst, float* logprobs,
                                     float* entropy, float* lse, float* entropy_b, void* workspace,
                                     int64_t ws_bytes, void* stash, int64_t stash_bytes, void* stream,
                                     void* timer) {
  return block_fwd(hidden, weight, labels, labels_i64, n, h, v, inv_temp, softcap, seq_start, last_dst,
                   logprobs, entropy, lse, entropy_b, workspace, ws_bytes, stash, stash_bytes, stream, timer,
                   kKeepStash);
}

extern "C" int axon_lmhead_block_fwd_logits(const void* hidden, const void* weight, const void* labels,
                                            int labels_i64, int64_t n, int64_t h, int64_t v, float inv_temp,
                                            float softcap, const uint8_t* seq_start, int64_t last_dst,
                                            float* logprobs, float* entropy, float* lse, float* entropy_b,
                                            void* workspace, int64_t ws_bytes, void* stash, int64_t stash_bytes,
                                            void* stream, void* timer) {
  return block_fwd(hidden, weight, labels, labels_i64, n, h, v, inv_temp, softcap, seq_start, last_dst,
                   logprobs, entropy, lse, entropy_b, workspace, ws_bytes, stash, stash_bytes, stream, timer,
                   kKeepLogits);
}

static int block_bwd(const float* dlogprobs, const float* dentropy, const void* hidden, const void* weight,
                     const void* labels, int labels_i64, const float* lse, const float* entropy_b, int64_t n,
                     int64_t h, int64_t v, float inv_temp, float softcap, const uint8_t* seq_start,
                     int64_t last_dst, void* d_hidden, void* d_weight, float* dw_acc, int dw_mode,
                     int /*wt_ready*/, int64_t group_pos, int dw_now, int64_t ws_tokens, int64_t chunk,
                     void* workspace, int64_t ws_bytes, const void* stash, int64_t stash_bytes, void* stream,
                     void* timer, Keep keep) {
  if (!last_dst_ok(last_dst, n) || n <= 0) return AXON_ERR_ARG;
  int rc;
  PhaseTimer* t = block_timer(timer, stream, 4, &rc);
  if (rc != AXON_OK) return rc;
  BlockArgs blk;
  blk.is_block = true;
  blk.keep = keep;
  blk.last_dst = last_dst;
  blk.dw_mode = dw_mode;
  blk.dw_acc = dw_acc;
  blk.group_pos = group_pos;
  blk.dw_now = dw_now != 0;
  blk.ws_tokens = ws_tokens;
  return bwd_impl(dlogprobs, dentropy, hidden, weight, labels, labels_i64, lse, entropy_b, n, h, v,
                  inv_temp, softcap, seq_start, d_hidden, d_weight, chunk, workspace, ws_bytes, stash,
                  stash_bytes, stream, t, blk);
}

extern "C" int axon_lmhead_block_bwd(const float* dlogprobs, const float* dentropy, const void* hidden,
                                     const void* weight, const void* labels, int labels_i64, const float* lse,
                                     const float* entropy_b, int64_t n, int64_t h, int64_t v, float inv_temp,
                                     float softcap, const uint8_t* seq_start, int64_t last_dst, void* d_hidden,
                                     void* d_weight, float* dw_acc, int dw_mode, int wt_ready,
                                     int64_t group_pos, int dw_now, int64_t ws_tokens, int64_t chunk,
                                     void* workspace, int64_t ws_bytes, const void* stash, int64_t stash_bytes,
                                     void* stream, void* timer) {
  return block_bwd(dlogprobs, dentropy, hidden, weight, labels, labels_i64, lse, entropy_b, n, h, v, inv_temp,
                   softcap, seq_start, last_dst, d_hidden, d_weight, dw_acc, dw_mode, wt_ready, group_pos,
                   dw_now, ws_tokens, chunk, workspace, ws_bytes, stash, stash_bytes, stream, timer,
                   kKeepStash);
}

extern "C" int axon_lmhead_block_bwd_logits(const float* dlogprobs, const float* dentropy, const void* hidden,
                                            const void* weight, const void* labels, int labels_i64,
                                            const float* lse, const float* entropy_b, int64_t n, int64_t h,
                                            int64_t v, float inv_temp, float softcap, const uint8_t* seq_start,
                                            int64_t last_dst, void* d_hidden, void* d_weight, float* dw_acc,
                                            int dw_mode, int wt_ready, int64_t group_pos, int dw_now,
                                            int64_t ws_tokens, int64_t chunk, void* workspace, int64_t ws_bytes,
                                            const void* stash, int64_t stash_bytes, void* stream, void* timer) {
  return block_bwd(dlogprobs, dentropy, hidden, weight, labels, labels_i64, lse, entropy_b, n, h, v, inv_temp,
                   softcap, seq_start, last_dst, d_hidden, d_weight, dw_acc, dw_mode, wt_ready, group_pos,
                   dw_now, ws_tokens, chunk, workspace, ws_bytes, stash, stash_bytes, stream, timer,
                   kKeepLogits);
}

extern "C" int axon_scale_bf16_pair_unless_one(void* x, int64_t nx, void* y, int64_t ny, const float* scale, void* stream) {
  if (nx < 0 || nx % 8 != 0 || ny < 0 || ny % 8 != 0) return AXON_ERR_SHAPE;
  if (nx == 0 && ny == 0) return AXON_OK;
  if ((nx && !x) || (ny && !y) || !scale || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15))
    return AXON_ERR_ARG;
  const int64_t most = nx > ny ? nx / 8 : ny / 8, blocks = (most + 255) / 256;
  hipLaunchKernelGGL(scale_bf16_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                     (hipStream_t)stream, static_cast<uint4*>(x), nx / 8, static_cast<uint4*>(y), ny / 8, scale);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_scale_bf16_unless_one(void* x, int64_t n, const float* scale, void* stream) {
  return axon_scale_bf16_pair_unless_one(x, n, nullptr, 0, scale, stream);
}
