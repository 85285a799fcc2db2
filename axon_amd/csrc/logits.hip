// The non-fused branch of the trainer's forward: the model has already written the [tokens, vocab] logits;
// per token, log_softmax(logits)[label] and the entropy come out of ONE read of the row (online max /
// sum / sum-times-logit, as in the fused head), and the backward turns the row into its gradient in one
// more read and one write (in place when asked to).  HBM-bound: 2 or 4 bytes per logit forward, twice that
// plus the write backward.
#include "common.h"
#include <type_traits>

namespace axon {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf16_to_f32(unsigned short h) { return __uint_as_float((uint32_t)h << 16); }
// two floats to bf16, round to nearest even, NaN kept (one v_cvt_pk_bf16_f32; in integer arithmetic eight
// instructions per value, which is what held the gradient kernel back)
__device__ __forceinline__ uint32_t f32x2_to_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

template <typename T> struct Row;
template <> struct Row<float> {
  static constexpr int kPer = 4;
  // CACHED: the vector stays in the caches behind (plain load) instead of passing them by
  template <bool CACHED = false>
  __device__ static void load(const float* p, float (&v)[8]) {
    const f32x4* const q = reinterpret_cast<const f32x4*>(p);
    const f32x4 x = CACHED ? *q : __builtin_nontemporal_load(q);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
  __device__ static float one(const float* p) { return *p; }
  __device__ static void store(float* p, const float (&v)[8]) {
    const f32x4 x = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(p));
  }
  __device__ static void store_one(float* p, float v) { *p = v; }
};
template <> struct Row<unsigned short> {
  static constexpr int kPer = 8;
  template <bool CACHED = false>
  __device__ static void load(const unsigned short* p, float (&v)[8]) {
    const u16x8* const q = reinterpret_cast<const u16x8*>(p);
    const u16x8 x = CACHED ? *q : __builtin_nontemporal_load(q);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf16_to_f32(x[j]);
  }
  __device__ static float one(const unsigned short* p) { return bf16_to_f32(*p); }
  __device__ static void store(unsigned short* p, const float (&v)[8]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 x = {f32x2_to_bf16(v[0], v[1]), f32x2_to_bf16(v[2], v[3]), f32x2_to_bf16(v[4], v[5]),
                     f32x2_to_bf16(v[6], v[7])};
    __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(p));
  }
  __device__ static void store_one(unsigned short* p, float v) { *p = (unsigned short)f32x2_to_bf16(v, 0.f); }
};

// Running statistics of a set of logits y (log2 units): M >= every y, s = sum 2^(y-M), e = sum 2^(y-M)(y-M).
struct Stats { float M, s, e; };

constexpr float kTiny = -150.f;  // 2^-150 flushes to zero: a logit that far below the maximum (or -inf) adds nothing

// Folds N logits (natural units) at once: one rescale at most, then four arithmetic instructions and one
// exponential per logit.
template <int N>
__device__ __forceinline__ void fold(Stats& a, const float (&z)[8]) {
  float m = z[0];
#pragma unroll
  for (int j = 1; j < N; ++j) m = fmaxf(m, z[j]);
  m *= kLog2e;
  if (m > a.M) {  // rescale what is there to the new reference
    const float d = fmaxf(a.M - m, kTiny), f = __builtin_amdgcn_exp2f(d);
    a.e = f * fmaf(a.s, d, a.e);
    a.s = a.s * f;
    a.M = m;
  }
  // four independent partial sums: the additions of consecutive logits do not wait for one another
  float s4[4] = {a.s, 0.f, 0.f, 0.f}, e4[4] = {a.e, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float d = fmaxf(fmaf(z[j], kLog2e, -a.M), kTiny), f = __builtin_amdgcn_exp2f(d);
    s4[j & 3] += f;
    e4[j & 3] = fmaf(f, d, e4[j & 3]);
  }
  a.s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  a.e = (e4[0] + e4[1]) + (e4[2] + e4[3]);
}
__device__ __forceinline__ Stats merge(Stats a, Stats b) {
  const float Mn = fmaxf(a.M, b.M);
  const float d1 = fmaxf(a.M - Mn, kTiny), d2 = fmaxf(b.M - Mn, kTiny);
  const float f1 = __builtin_amdgcn_exp2f(d1), f2 = __builtin_amdgcn_exp2f(d2);
  Stats r;
  r.M = Mn;
  r.e = f1 * fmaf(a.s, d1, a.e) + f2 * fmaf(b.s, d2, b.e);
  r.s = a.s * f1 + b.s * f2;
  return r;
}
constexpr float kFloor = -1e30f;  // below any logit; finite, so that differences stay finite

// What one workgroup does of a row: the 16-byte vectors [q_lo, q_hi) of the row's aligned middle, counted from
// element `head` on, and its share of the n_scalar elements outside it (before `head`, then behind the last vector).
// An odd vocabulary puts every row on another boundary, so a row's first vector starts at its first 16-byte boundary
// and not at its first element.
struct RowSpan {
  int head, n_vec, n_scalar, q_lo, q_hi;
  template <typename T>
  __device__ __forceinline__ RowSpan(const T* row, int vocab, bool vec_ok, int part, int parts) {
    constexpr int kPer = Row<T>::kPer;
    const int off = (int)((reinterpret_cast<uintptr_t>(row) & 15) / sizeof(T));
    head = min((kPer - off) & (kPer - 1), vocab);
    n_vec = vec_ok ? (vocab - head) / kPer : 0;
    n_scalar = vocab - n_vec * kPer;
    q_lo = (int)((int64_t)n_vec * part / parts);
    q_hi = (int)((int64_t)n_vec * (part + 1) / parts);
  }
  template <typename T>
  __device__ __forceinline__ int scalar(int i) const { return i < head ? i : i + n_vec * Row<T>::kPer; }
};

template <typename T, typename LabelT>
__device__ __forceinline__ void write_stats(Stats st, int t, const T* row, int vocab, const LabelT* labels,
                                            float* logprob, float* entropy, float* lse) {
  const float L = __log2f(st.s), d = st.e / st.s;
  const float lse_v = (st.M + L) * kLn2;
  lse[t] = lse_v;
  if (entropy != nullptr) entropy[t] = (L - d) * kLn2;  // lse - sum p z, the common max cancelled
  if (logprob != nullptr) {
    const int64_t lab = (int64_t)labels[t];
    logprob[t] = (lab >= 0 && lab < vocab) ? Row<T>::one(row + lab) - lse_v : 0.f;
  }
}

// Workgroup (part, row): blockIdx.x = row * parts + part.  One part writes the row's results, several leave their
// statistics in ws[row][part][3] for logits_merge_kernel.  Bound by memory, 6.0 to 6.6 TB/s from 1100 rows on.
// 2047 x 50257 bf16 39 us for 81 (rows off a 16-byte boundary), 187 x 151936 bf16 20 for 31, 300 x 151936 fp32 32 for 58.
// Rows from `cached_from` on are left in the 256 MB cache in front of the memory, for the backward to find: a
// non-temporal load does not allocate there.  The rows before them, which would be evicted again, pass it by (all
// rows cached: 116 us for 106 at 2047 x 151936 bf16, for the lines that are written back to make room).
template <typename T, typename LabelT>
__global__ __launch_bounds__(kBlock) void logits_stats_kernel(
    const T* __restrict__ logits, int64_t ld, int vocab, const LabelT* __restrict__ labels,
    float* __restrict__ logprob, float* __restrict__ entropy, float* __restrict__ lse, int parts,
    float* __restrict__ ws, int cached_from) {
  __shared__ float red[3][kBlock / kWave];
  const int t = blockIdx.x / parts, part = blockIdx.x - t * parts;
  const T* row = logits + (int64_t)t * ld;
  constexpr int kPer = Row<T>::kPer;
  const RowSpan sp(row, vocab, true, part, parts);
  Stats st{kFloor, 0.f, 0.f};
  const T* body = row + sp.head;
  auto walk = [&](auto cached) {
    constexpr bool kCached = decltype(cached)::value;
    int q = sp.q_lo + threadIdx.x;
    for (; q + kBlock < sp.q_hi; q += 2 * kBlock) {  // two loads in flight per thread
      float v0[8], v1[8];
      Row<T>::template load<kCached>(body + (uint32_t)q * kPer, v0);
      Row<T>::template load<kCached>(body + (uint32_t)(q + kBlock) * kPer, v1);
      fold<kPer>(st, v0);
      fold<kPer>(st, v1);
    }
    for (; q < sp.q_hi; q += kBlock) {
      float v[8];
      Row<T>::template load<kCached>(body + (uint32_t)q * kPer, v);
      fold<kPer>(st, v);
    }
  };
  if (t >= cached_from) walk(std::true_type{}); else walk(std::false_type{});
  for (int i = part * kBlock + threadIdx.x; i < sp.n_scalar; i += parts * kBlock) {
    const float v[8] = {Row<T>::one(row + sp.scalar<T>(i))};
    fold<1>(st, v);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    Stats o;
    o.M = __shfl_down(st.M, off, kWave);
    o.s = __shfl_down(st.s, off, kWave);
    o.e = __shfl_down(st.e, off, kWave);
    st = merge(st, o);
  }
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (lane == 0) { red[0][wave] = st.M; red[1][wave] = st.s; red[2][wave] = st.e; }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kBlock / kWave; ++w) st = merge(st, Stats{red[0][w], red[1][w], red[2][w]});
  if (parts > 1) {
    float* o = ws + (int64_t)blockIdx.x * 3;
    o[0] = st.M; o[1] = st.s; o[2] = st.e;
    return;
  }
  write_stats(st, t, row, vocab, labels, logprob, entropy, lse);
}

// One wavefront per row folds the row's parts (at most kMaxParts), in a fixed tree.
constexpr int kMaxParts = 64;
template <typename T, typename LabelT>
__global__ __launch_bounds__(kWave) void logits_merge_kernel(
    const float* __restrict__ ws, int parts, const T* __restrict__ logits, int64_t ld, int vocab,
    const LabelT* __restrict__ labels, float* __restrict__ logprob, float* __restrict__ entropy,
    float* __restrict__ lse) {
  const int t = blockIdx.x, lane = threadIdx.x;
  Stats st{kFloor, 0.f, 0.f};
  if (lane < parts) {
    const float* o = ws + ((int64_t)t * parts + lane) * 3;
    st = Stats{o[0], o[1], o[2]};
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    Stats o;
    o.M = __shfl_down(st.M, off, kWave);
    o.s = __shfl_down(st.s, off, kWave);
    o.e = __shfl_down(st.e, off, kWave);
    st = merge(st, o);
  }
  if (lane == 0) write_stats(st, t, logits + (int64_t)t * ld, vocab, labels, logprob, entropy, lse);
}

// dlogits[j] = g_lp (onehot_j - p_j) - g_ent p_j (log p_j + H),  p_j = exp(z_j - lse).
// dlogits may be the logits' own storage: every element is read before it is written by the same thread.  Rows, and
// the vectors of a row, are walked from the last to the first: the end of what the forward read last is still in the 256 MB cache in front of the
// memory (its cached_from), and the loads and stores here, which pass that cache by, leave it there until it is
// read.  Bound by memory: 2047 x 151936 bf16 208 us for 247 with a forward that leaves nothing, 4096 x 50257 151 for
// 186, 1600 x 151936 fp32 355 for 404; where a short batch is split into parts 32 x 151936 takes 9.3 us for 53, 187 x
// 151936 24 for 78; rows of an odd vocabulary, read from their first 16-byte boundary on, 2047 x 50257 bf16 93 us for
// 166.
template <typename T, typename LabelT>
__global__ __launch_bounds__(kBlock) void logits_grad_kernel(
    const T* logits, int64_t ld, int vocab, const LabelT* __restrict__ labels,
    const float* __restrict__ lse, const float* __restrict__ entropy, const float* __restrict__ g_logprob,
    const float* __restrict__ g_entropy, T* dlogits, int64_t ld_d, int vec_ok, int parts) {
  const int b = gridDim.x - 1 - blockIdx.x;
  const int t = b / parts, part = b - t * parts;
  const T* row = logits + (int64_t)t * ld;
  T* out = dlogits + (int64_t)t * ld_d;
  constexpr int kPer = Row<T>::kPer;
  const float lse_v = lse[t];
  const float g_lp = g_logprob ? g_logprob[t] : 0.f;
  const float g_en = g_entropy ? g_entropy[t] : 0.f;
  const float H = g_entropy ? entropy[t] : 0.f;
  const int64_t lab64 = g_logprob ? (int64_t)labels[t] : -1;
  const int lab = (lab64 >= 0 && lab64 < vocab) ? (int)lab64 : -1;
  auto grad = [&](float z) {
    const float lp = z - lse_v;
    const float p = __expf(lp);
    // a probability of 0 takes nothing from the entropy, also where its log is -inf
    return p * ((p > 0.f) ? fmaf(-g_en, lp + H, -g_lp) : -g_lp);
  };
  // vec_ok: the row of dlogits sits on the same offset from a 16-byte boundary as the row of logits
  const RowSpan sp(row, vocab, vec_ok != 0, part, parts);
  const T* body = row + sp.head;
  T* body_out = out + sp.head;
  const int lab_b = lab < sp.head ? -1 : lab - sp.head;
  auto finish = [&](int q, float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) v[j] = grad(v[j]);
    const int in_vec = lab_b - q * kPer;
    if ((unsigned)in_vec < (unsigned)kPer) {
#pragma unroll
      for (int j = 0; j < kPer; ++j) v[j] += (j == in_vec) ? g_lp : 0.f;
    }
    Row<T>::store(body_out + (uint32_t)q * kPer, v);
  };
  int q = sp.q_hi - 1 - (int)threadIdx.x;
  for (; q - kBlock >= sp.q_lo; q -= 2 * kBlock) {  // two loads in flight per thread
    float v0[8], v1[8];
    Row<T>::load(body + (uint32_t)q * kPer, v0);
    Row<T>::load(body + (uint32_t)(q - kBlock) * kPer, v1);
    finish(q, v0);
    finish(q - kBlock, v1);
  }
  for (; q >= sp.q_lo; q -= kBlock) {
    float v[8];
    Row<T>::load(body + (uint32_t)q * kPer, v);
    finish(q, v);
  }
  for (int i = part * kBlock + threadIdx.x; i < sp.n_scalar; i += parts * kBlock) {
    const int j = sp.scalar<T>(i);
    Row<T>::store_one(out + j, grad(Row<T>::one(row + j)) + (j == lab ? g_lp : 0.f));
  }
}

}  // namespace axon

using namespace axon;

namespace {

// Workgroups per row.  The part holds 2048 of these workgroups at once; from three quarters of that on a row is left
// to one (2047 x 151936 bf16, forward + backward: 343 us with one, 343 with two, 353 with four).  Fewer rows are split
// into about 8192 pieces, of at least eight vectors per thread each (1500 x 128264 bf16: 228 us for 242 with 4096
// pieces and with one per row, 700 x 151936: 126 for 130 and 148, 300 x 151936 fp32: 104 for 110 and 187).
int row_parts(int64_t n, int64_t vocab, int elem_bytes) {
  if (n >= 1536) return 1;
  const int64_t fill = 8192 / (n > 0 ? n : 1), work = vocab * elem_bytes / (8 * 16 * kBlock);
  const int64_t p = fill < work ? fill : work;
  return (int)(p < 1 ? 1 : (p < kMaxParts ? p : kMaxParts));
}

// The forward pays for a split with a second launch: rows of less than 128 KB, which one workgroup reads in about as
// long, are left whole (32 x 151936 bf16, 300 KB, is split; 50257 and 32768 are not).
int fwd_parts(int64_t n, int64_t vocab, int elem_bytes) {
  return vocab * elem_bytes < 131072 ? 1 : row_parts(n, vocab, elem_bytes);
}

// How much of the rows a forward leaves in the cache in front of the memory for its backward: the size of that cache.
// Forward + backward at 2047 x 151936 bf16: 354 us with nothing, 333 with 128 MB, 323 with 192, 316 with 224, 314 with
// 256, 321 with 400; 4096 x 50257 (411 MB) 263, 246, 240, 233, 231, 232; a backward that does not come costs up to 2 us.
constexpr int64_t kCacheBytes = int64_t(256) << 20;

// every row of b sits on the same offset from a 16-byte boundary as the row of a
bool same_offsets(const void* a, int64_t ld_a, const void* b, int64_t ld_b, int64_t n, int elem_bytes) {
  const uintptr_t d = reinterpret_cast<uintptr_t>(a) ^ reinterpret_cast<uintptr_t>(b);
  return (d & 15) == 0 && (n <= 1 || ((ld_a - ld_b) * elem_bytes) % 16 == 0);
}

int check_logits(const void* logits, int dtype, int64_t ld, int64_t n, int64_t v) {
  if (n < 0 || v <= 0 || ld < v) return AXON_ERR_ARG;
  if (dtype != AXON_LOGITS_F32 && dtype != AXON_LOGITS_BF16) return AXON_ERR_ARG;
  if (n >= (int64_t)INT32_MAX || v >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (n > 0 && !logits) return AXON_ERR_ARG;
  return AXON_OK;
}

}  // namespace

extern "C" int64_t axon_logits_fwd_workspace_bytes(int dtype, int64_t n, int64_t vocab) {
  if (n < 0 || vocab <= 0 || (dtype != AXON_LOGITS_F32 && dtype != AXON_LOGITS_BF16)) return AXON_ERR_ARG;
  const int parts = fwd_parts(n, vocab, dtype == AXON_LOGITS_F32 ? 4 : 2);
  return parts > 1 ? n * parts * 3 * (int64_t)sizeof(float) : 0;
}

static int logits_fwd(const void* logits, int dtype, int64_t ld, int64_t n, int64_t vocab, const void* labels,
                      int labels_i64, float* logprob, float* entropy, float* lse, float* workspace, bool bwd_follows,
                      void* stream) {
  int rc = check_logits(logits, dtype, ld, n, vocab);
  if (rc != AXON_OK) return rc;
  if (n == 0) return AXON_OK;
  if (!lse || (logprob && !labels)) return AXON_ERR_ARG;
  const hipStream_t st = (hipStream_t)stream;
  const int eb = dtype == AXON_LOGITS_F32 ? 4 : 2;
  const int parts = workspace ? fwd_parts(n, vocab, eb) : 1;
  const int64_t cached = bwd_follows ? kCacheBytes / (vocab * eb) : 0;
  const int cached_from = (int)(cached < n ? n - cached : 0);
  const dim3 grid((unsigned)(n * parts)), blk(kBlock);
#define AXON_STATS(T, L)                                                                               \
  do {                                                                                                 \
    hipLaunchKernelGGL((logits_stats_kernel<T, L>), grid, blk, 0, st, static_cast<const T*>(logits), ld, \
                       (int)vocab, static_cast<const L*>(labels), logprob, entropy, lse, parts, workspace, cached_from); \
    if (parts > 1)                                                                                     \
      hipLaunchKernelGGL((logits_merge_kernel<T, L>), dim3((unsigned)n), dim3(kWave), 0, st, workspace, parts, \
                         static_cast<const T*>(logits), ld, (int)vocab, static_cast<const L*>(labels), \
                         logprob, entropy, lse);                                                       \
  } while (0)
  if (dtype == AXON_LOGITS_F32) {
    if (labels_i64) AXON_STATS(float, int64_t); else AXON_STATS(float, int32_t);
  } else {
    if (labels_i64) AXON_STATS(unsigned short, int64_t); else AXON_STATS(unsigned short, int32_t);
  }
#undef AXON_STATS
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_logits_fwd_ws(const void* logits, int dtype, int64_t ld, int64_t n, int64_t vocab,
                                  const void* labels, int labels_i64, float* logprob, float* entropy,
                                  float* lse, float* workspace, void* stream) {
  return logits_fwd(logits, dtype, ld, n, vocab, labels, labels_i64, logprob, entropy, lse, workspace, false, stream);
}

extern "C" int axon_logits_fwd_train(const void* logits, int dtype, int64_t ld, int64_t n, int64_t vocab,
                                     const void* labels, int labels_i64, float* logprob, float* entropy,
                                     float* lse, float* workspace, void* stream) {
  return logits_fwd(logits, dtype, ld, n, vocab, labels, labels_i64, logprob, entropy, lse, workspace, true, stream);
}

extern "C" int axon_logits_fwd(const void* logits, int dtype, int64_t ld, int64_t n, int64_t vocab,
                               const void* labels, int labels_i64, float* logprob, float* entropy,
                               float* lse, void* stream) {
  return axon_logits_fwd_ws(logits, dtype, ld, n, vocab, labels, labels_i64, logprob, entropy, lse, nullptr, stream);
}

extern "C" int axon_logits_bwd(const void* logits, int dtype, int64_t ld, int64_t n, int64_t vocab,
                               const void* labels, int labels_i64, const float* lse,
                               const float* entropy, const float* g_logprob, const float* g_entropy,
                               void* dlogits, int64_t ld_d, void* stream) {
  int rc = check_logits(logits, dtype, ld, n, vocab);
  if (rc != AXON_OK) return rc;
  if (n == 0) return AXON_OK;
  if (!lse || !dlogits || ld_d < vocab) return AXON_ERR_ARG;
  if ((g_logprob && !labels) || (g_entropy && !entropy)) return AXON_ERR_ARG;
  const hipStream_t st = (hipStream_t)stream;
  const int eb = dtype == AXON_LOGITS_F32 ? 4 : 2;
  const int vec_ok = same_offsets(logits, ld, dlogits, ld_d, n, eb), parts = row_parts(n, vocab, eb);
  const dim3 grid((unsigned)(n * parts)), blk(kBlock);
#define AXON_GRAD(T, L)                                                                            \
  hipLaunchKernelGGL((logits_grad_kernel<T, L>), grid, blk, 0, st, static_cast<const T*>(logits), ld,  \
                     (int)vocab, static_cast<const L*>(labels), lse, entropy, g_logprob, g_entropy,    \
                     static_cast<T*>(dlogits), ld_d, vec_ok, parts)
  if (dtype == AXON_LOGITS_F32) {
    if (labels_i64) AXON_GRAD(float, int64_t); else AXON_GRAD(float, int32_t);
  } else {
    if (labels_i64) AXON_GRAD(unsigned short, int64_t); else AXON_GRAD(unsigned short, int32_t);
  }
#undef AXON_GRAD
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}
