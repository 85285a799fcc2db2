// (b) Ragged segmented reductions over cu_seqlens, token-parallel.
//
// Every workgroup streams a contiguous chunk of slots with 16-byte loads.  A
// thread folds its four slots, then the wave runs a segmented shuffle reduction
// keyed by row id (row ids are non-decreasing across lanes), and the first lane
// of each run adds the run total to the per-row output with one atomic.  A row
// that spans several waves costs one atomic per wave, so load balance does not
// depend on the row-length distribution.
//
// The partial sums of a long row arrive in whatever order its wavefronts finish, and float addition
// is not associative.  The counts are sums of small integers (exact in any order) and the flags are
// ORs; the sums are added as 64-bit fixed-point integers in units of 2^-32, whose addition is
// associative, so a row's sum comes out the same bits on every run however many wavefronts it
// spans.  A partial of 2^20 or more in magnitude, an infinity or a NaN goes to a float slot beside
// it (whether that slot ends up finite, infinite or NaN does not depend on the order either).  A
// finishing pass turns the two into the fp32 sum.  Rounding a partial to 2^-32 is finer than the
// fp32 rounding of any row sum of 2^-8 or more in magnitude.
#include "common.h"

namespace axon {

struct Seg {
  int row;
  float cnt, sum;
  int flag;
};

struct RowSumAcc {
  unsigned long long* fixed;  // [n_rows] two's-complement sums in units of 2^-32
  float* big;                 // [n_rows] what does not fit the fixed-point range
};
constexpr float kRowSumUnit = 4294967296.f;  // 2^32
constexpr float kRowSumLimit = 1048576.f;    // 2^20 per partial: 2^52 units, 2^11 such partials fit 63 bits

__device__ __forceinline__ void row_sum_add(const RowSumAcc& acc, int row, float v) {
  if (fabsf(v) < kRowSumLimit)
    atomicAdd(acc.fixed + row, (unsigned long long)__float2ll_rn(v * kRowSumUnit));
  else
    atomicAdd(acc.big + row, v);
}

__global__ __launch_bounds__(256) void row_sum_finish_kernel(RowSumAcc acc, int64_t n_rows,
                                                             float* __restrict__ sum) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_rows) return;
  const double fixed = (double)(long long)acc.fixed[r] * (1.0 / 4294967296.0);
  sum[r] = (float)((double)acc.big[r] + fixed);
}

__device__ __forceinline__ void seg_flush(const Seg& s, float* cnt, const RowSumAcc& sum, int32_t* flag) {
  if (s.row < 0) return;
  if (cnt != nullptr && s.cnt != 0.f) atomicAdd(cnt + s.row, s.cnt);
  if (sum.fixed != nullptr && s.sum != 0.f) row_sum_add(sum, s.row, s.sum);
  if (flag != nullptr && s.flag) atomicOr(flag + s.row, 1);
}

// Segmented reduction across the wave; lanes hold (row, values) with rows sorted.
__device__ __forceinline__ void seg_wave_reduce_flush(Seg s, float* cnt, const RowSumAcc& sum,
                                                      int32_t* flag) {
  const int lane = threadIdx.x & (kWave - 1);
  // the common case: the whole wavefront sits in one row (rows are mostly longer than 256 slots)
  const int first = __builtin_amdgcn_readfirstlane(s.row);
  if (first >= 0 && __builtin_amdgcn_readlane(s.row, kWave - 1) == first) {  // rows are sorted across lanes
    Seg t;
    t.row = first;
    t.cnt = wave_sum_to_last(s.cnt);
    t.sum = wave_sum_to_last(s.sum);
    t.flag = (flag != nullptr) ? (__ballot(s.flag != 0) != 0) : 0;
    if (lane == kWave - 1) seg_flush(t, cnt, sum, flag);
    return;
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int r2 = __shfl_down(s.row, off, kWave);
    const float c2 = __shfl_down(s.cnt, off, kWave);
    const float s2 = __shfl_down(s.sum, off, kWave);
    const int f2 = __shfl_down(s.flag, off, kWave);
    if (lane + off < kWave && r2 == s.row) {
      s.cnt += c2;
      s.sum += s2;
      s.flag |= f2;
    }
  }
  const int prev = __shfl_up(s.row, 1, kWave);
  if (lane == 0 || prev != s.row) seg_flush(s, cnt, sum, flag);
}

template <int MK>
__global__ __launch_bounds__(kBlock) void row_stats_kernel(
    const float* __restrict__ a, const float* __restrict__ b, const void* __restrict__ mask,
    const int32_t* __restrict__ cu, int64_t n_rows, int64_t n_slots, int64_t uniform_len,
    int flag_mode, float thr, float* cnt, RowSumAcc sum, int32_t* flag) {
  __shared__ int32_t lds_cu[kLdsRows];
  const int64_t c0 = (int64_t)blockIdx.x * kChunk;
  const int64_t c1 = min(c0 + (int64_t)kChunk, n_slots);
  RowFinder rf;
  const bool whole = (c1 - c0 == kChunk);
  // whole chunk: every load is issued before the first use (twelve 16-byte requests in flight per
  // thread), and before the row search, whose chain of dependent loads then runs under them
  float av_[kIter][4], bv_[kIter][4], mv_[kIter][4];
  if (whole) {
#pragma unroll
    for (int it = 0; it < kIter; ++it) {
      const int64_t i = c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec;
      load4(a, i, av_[it]);
      if (b != nullptr) load4(b, i, bv_[it]);
      else bv_[it][0] = bv_[it][1] = bv_[it][2] = bv_[it][3] = 0.f;
      load_mask4<MK>(mask, i, mv_[it]);
    }
  }
  rf.init(cu, n_rows, uniform_len, c0, c1, lds_cu);

  // the slots of one vector of four -> the wavefront's segmented sums
  auto fold = [&](int64_t i, const float (&av)[4], const float (&bv)[4], const float (&mv)[4]) {
    Seg s{-1, 0.f, 0.f, 0};
    if (i < c1) {
      int r = rf.row(i);
      int64_t rend = rf.row_end(r);
      s.row = r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t p = i + j;
        if (p >= n_slots) break;
        if (p >= rend) {  // slot belongs to a later row: flush and restart
          seg_flush(s, cnt, sum, flag);
          r = rf.row(p);
          rend = rf.row_end(r);
          s = Seg{r, 0.f, 0.f, 0};
        }
        const float d = av[j] - bv[j];
        const float m = mv[j];
        s.cnt += m;
        // masked_sum in the reference zeroes values outside the mask before the
        // multiply, so NaN/Inf in padding never reaches the sum.
        s.sum += (m != 0.f) ? d * m : 0.f;
        if (flag_mode == 1) s.flag |= (m != 0.f && d < thr);
        if (flag_mode == 2) s.flag |= (m != 0.f && fabsf(d) > thr);
      }
    }
    seg_wave_reduce_flush(s, cnt, sum, flag);
  };
  if (whole) {
#pragma unroll
    for (int it = 0; it < kIter; ++it)
      fold(c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec, av_[it], bv_[it], mv_[it]);
    return;
  }
#pragma unroll 1
  for (int it = 0; it < kIter; ++it) {
    const int64_t i = c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec;
    float av[4] = {0.f, 0.f, 0.f, 0.f}, bv[4] = {0.f, 0.f, 0.f, 0.f}, mv[4] = {0.f, 0.f, 0.f, 0.f};
    if (i < c1) {
      const bool full = (i + kVec <= n_slots);
      if (full) {
        load4(a, i, av);
        if (b != nullptr) load4(b, i, bv);
        load_mask4<MK>(mask, i, mv);
      } else {
        for (int j = 0; j < 4; ++j) {
          const bool ok = i + j < n_slots;
          av[j] = ok ? a[i + j] : 0.f;
          bv[j] = (ok && b != nullptr) ? b[i + j] : 0.f;
          mv[j] = ok ? load_mask1<MK>(mask, i + j) : 0.f;
        }
      }
    }
    fold(i, av, bv, mv);
  }
}

struct GroupCfg {
  int64_t n_groups;
  float eps;
  int mode;  // 0 centred, 1 centred and divided by the standard deviation, 2 RLOO, 3 GPG
};

// GRPO / RLOO / GPG scalar of a row with score x in a group of c rows with mean mu and deviation sd (advantage.py:78-146,
// 336-371); alpha: rows over rows with a non-zero score.
__device__ __forceinline__ float group_scalar_of(const GroupCfg& g, float x, float c, float mu, float sd, float alpha) {
  float v;
  if (g.mode == 2) {  // (n*s - S) / (n - 1), S = n * mean
    v = (c * x - c * mu) / fmaxf(c - 1.f, 1.f);
  } else if (g.mode == 3) {  // alpha * (s - mean) / f_norm, eps carries f_norm; singletons have mean 0 and keep their score
    return alpha * (x - mu) / g.eps;
  } else {
    v = g.mode ? (x - mu) / (sd + g.eps) : (x - mu);
  }
  return v * ((c > 1.f) ? 1.f : 0.f);
}

// group_mean_std + GRPO scalar, one workgroup.
__global__ __launch_bounds__(1024) void group_stats_kernel(
    const float* __restrict__ scores, const int64_t* __restrict__ gidx, int64_t n_rows,
    int64_t n_groups, float eps, int norm_by_std, float* mean, float* stdv, float* count,
    float* scalar) {
  __shared__ int nonzero;  // rows with a non-zero score (GPG's alpha)
  if (threadIdx.x == 0) nonzero = 0;
  __syncthreads();
  // phase 1: count -> count[], s1 -> mean[], s2 -> stdv[] (zero-filled by caller)
  for (int64_t i = threadIdx.x; i < n_rows; i += blockDim.x) {
    const int64_t g = gidx[i];
    const float x = scores[i];
    if (norm_by_std == 3 && x != 0.f) atomicAdd(&nonzero, 1);
    if (g < 0 || g >= n_groups) continue;
    atomicAdd(count + g, 1.f);
    atomicAdd(mean + g, x);
    atomicAdd(stdv + g, x * x);
  }
  __threadfence();
  __syncthreads();
  // phase 2: finalise per group
  for (int64_t g = threadIdx.x; g < n_groups; g += blockDim.x) {
    const float c = count[g], s1 = mean[g], s2 = stdv[g];
    const float cc = fmaxf(c, 1.f);
    float mu = s1 / cc;
    const float var = (s2 - (s1 * s1) / cc) / fmaxf(c - 1.f, 1.f);
    float sd = sqrtf(fmaxf(var, eps));
    if (c <= 1.f) { mu = 0.f; sd = 1.f; }
    mean[g] = mu;
    stdv[g] = sd;
  }
  __threadfence();
  __syncthreads();
  if (scalar == nullptr) return;
  for (int64_t i = threadIdx.x; i < n_rows; i += blockDim.x) {
    const int64_t g = gidx[i];
    if (g < 0 || g >= n_groups) { scalar[i] = 0.f; continue; }
    const float x = scores[i];
    const float alpha = (float)n_rows / (float)max(nonzero, 1);
    scalar[i] = group_scalar_of(GroupCfg{n_groups, eps, norm_by_std}, x, count[g], mean[g], stdv[g], alpha);
  }
}

// Row sums and, in the workgroup that ends last, the group statistics and the per-row scalar of the group-based
// estimators: with row_broadcast_kernel behind it an advantage is two launches, no zero fills and no float atomics
// in memory.  A wavefront owns a row (double accumulators per lane, then a fixed tree; a workgroup a very long one), four 16-byte loads in flight;
// the grid is bounded so that its tickets stay cheap.  The groups' sums are formed in LDS by
// double atomics, whose order is not fixed: mean and variance are right, and the same on every run, to c * 2^-53 of
// (sum of squares / variance) for a group of c rows; below 2^-24, the rounding of the fp32 results, while the scores' common
// offset is under some 5000 standard deviations.  (The separate kernels, and the reference, add in fp32.)
// 128 x 1024 slots, 16 groups: 7.5 us where fill, row pass, finish and group kernel took 6.9 + 1.3 + 10.9 and two fills;
// 8.4 M slots in 9000 rows, 1150 groups: 33 for 27 + 4.7 + 80 (40 with one row after the other in the last workgroup).
constexpr int kScoreGroups = 2048;  // 40 KB of LDS
constexpr int kScoreBlocks = 512;  // what fits the part at once: a wavefront with a short row takes another one
// A row of more than kLongRow slots is summed by the whole workgroup of the wavefront that meets it (on its first 64
// trips): a wavefront needs 0.5 us per 1024 slots, which a packed batch, of which the host knows the mean length only,
// pays for its longest row alone.  Whole operator, 9000 rows of 500 slots and one of 2^20: 110 us, 593 with a wavefront per row
// and 221 with the separate kernels; one of 65536: 42, 68 and 179.  Workgroups of many long rows take one after the other, so that
// the line lies where half the rows of the longest mean length that comes here can be beyond it: from 8192 on, 512 rows
// of 16384 took 48 us for 34.
constexpr int kScoreThreads = 1024, kLongRow = 32768;

__global__ __launch_bounds__(kScoreThreads) void group_scores_kernel(
    const float* __restrict__ a, const int32_t* __restrict__ cu, int64_t n_rows, int64_t n_slots, int64_t uniform_len,
    const int64_t* __restrict__ gidx, GroupCfg g, float* scores, float* __restrict__ scalar, unsigned* ticket) {
  __shared__ double sums[kScoreGroups][2];
  __shared__ int count[kScoreGroups];
  __shared__ int last, nonzero;
  constexpr int kWaves = kScoreThreads / kWave;
  __shared__ double part[kWaves];
  __shared__ uint64_t long_trips[kWaves];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  auto span = [&](int64_t r, int64_t& t0, int64_t& t1) {
    t0 = uniform_len > 0 ? r * uniform_len : (int64_t)cu[r];
    t1 = uniform_len > 0 ? t0 + uniform_len : (int64_t)cu[r + 1];
    t0 = min(max(t0, (int64_t)0), n_slots);
    t1 = min(max(t1, t0), n_slots);
  };
  // this thread's share of a row that `n` threads add up, `id` of them: whole vectors, and the row's edges
  auto share = [&](int64_t t0, int64_t t1, int id, auto n_c) -> double {
    constexpr int n = decltype(n_c)::value;
    double acc = 0.0;
    const int64_t b0 = min((t0 + 3) & ~(int64_t)3, t1), b1 = max(t1 & ~(int64_t)3, b0);  // whole vectors
    // the row's edges and its first four vectors per thread are on their way before anything is added
    const float e0 = id < b0 - t0 ? a[t0 + id] : 0.f, e1 = id < t1 - b1 ? a[b1 + id] : 0.f;
    for (int64_t p = b0 + id * kVec; p < b1; p += 4 * n * kVec) {
      float v[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) load4(a, min(p + u * n * kVec, b1 - kVec), v[u]);  // a valid vector; dropped below
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double x = ((double)v[u][0] + (double)v[u][1]) + ((double)v[u][2] + (double)v[u][3]);
        acc += p + u * n * kVec < b1 ? x : 0.0;
      }
    }
    return acc + ((double)e0 + (double)e1);
  };
  auto put = [&](int64_t r, double v) {
    __hip_atomic_store(scores + r, (float)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto row_of = [&](int trip, int w) { return ((int64_t)trip * gridDim.x + blockIdx.x) * kWaves + w; };
  uint64_t longs = 0;  // this wavefront's trips whose row is left to the whole workgroup
  for (int trip = 0;; ++trip) {
    const int64_t r = row_of(trip, wave);
    if (r >= n_rows) break;
    int64_t t0, t1;
    span(r, t0, t1);
    if (t1 - t0 > kLongRow && trip < 64) {
      longs |= 1ull << trip;
      continue;
    }
    const double acc = wave_sum_d(share(t0, t1, lane, std::integral_constant<int, kWave>{}));
    if (lane == 0) put(r, acc);
  }
  if (lane == 0) long_trips[wave] = longs;
  __syncthreads();
  // the same rows for every thread of the workgroup
  for (uint64_t with = __ballot(lane < kWaves && long_trips[lane % kWaves] != 0); with != 0; with &= with - 1) {
    const int w = __builtin_ctzll(with);
    for (uint64_t m = long_trips[w]; m != 0; m &= m - 1) {
      const int64_t r = row_of(__builtin_ctzll(m), w);
      int64_t t0, t1;
      span(r, t0, t1);
      const double acc = wave_sum_d(share(t0, t1, (int)threadIdx.x, std::integral_constant<int, kScoreThreads>{}));
      if (lane == 0) part[wave] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        double sum = 0.0;
        for (int u = 0; u < kWaves; ++u) sum += part[u];
        put(r, sum);
      }
      __syncthreads();
    }
  }
  // the scores' write-through stores are acknowledged before the workgroup draws its ticket (publish_row_take_ticket)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0)
  __syncthreads();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if (threadIdx.x == 0) {
    const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = (t == gridDim.x - 1);
    if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
    nonzero = 0;
  }
  const int n_groups = (int)g.n_groups;
  for (int i = threadIdx.x; i < n_groups; i += blockDim.x) { sums[i][0] = 0.0; sums[i][1] = 0.0; count[i] = 0; }
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  // Up to 1024 rows: a thread has one.  More: eight consecutive rows per thread and trip, their loads all in flight (a
  // load from behind a dropped cache is a microsecond).  Rows of a group lie next to one another as a rule: a thread adds
  // up its run of a group in registers and adds to LDS once per run, and the threads of a wavefront rarely meet on one
  // address.  (With 128 rows eight in a row per thread cost 2.5 us more than one.)
  const int per = n_rows <= blockDim.x ? 1 : 8;
  auto each_eight = [&](auto&& f) {
    for (int64_t i0 = per * (int64_t)threadIdx.x; i0 < n_rows; i0 += 8 * (int64_t)blockDim.x) {
      int64_t k[8];
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t i = min(i0 + u, n_rows - 1);  // a valid row; dropped by f
        k[u] = gidx[i];
        x[u] = scores[i];
      }
      f(i0, k, x);
    }
  };
  each_eight([&](int64_t i0, const int64_t (&k)[8], const float (&x)[8]) {
    int run = -1, c = 0, nz = 0;
    double s1 = 0.0, s2 = 0.0;
    auto flush = [&]() {
      if (run < 0) return;
      atomicAdd(&count[run], c);
      atomicAdd(&sums[run][0], s1);
      atomicAdd(&sums[run][1], s2);
    };
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (u >= per || i0 + u >= n_rows) break;
      nz += x[u] != 0.f ? 1 : 0;
      if (k[u] < 0 || k[u] >= n_groups) continue;
      if ((int)k[u] != run) {
        flush();
        run = (int)k[u];
        c = 0;
        s1 = s2 = 0.0;
      }
      ++c;
      s1 += (double)x[u];
      s2 += (double)x[u] * (double)x[u];
    }
    flush();
    if (g.mode == 3 && nz != 0) atomicAdd(&nonzero, nz);
  });
  __syncthreads();
  for (int k = threadIdx.x; k < n_groups; k += blockDim.x) {  // sums -> mean and deviation, singletons 0 and 1
    const double c = (double)count[k], cc = fmax(c, 1.0);
    const double s1 = sums[k][0], s2 = sums[k][1];
    const float var = (float)((s2 - s1 * s1 / cc) / fmax(c - 1.0, 1.0));
    const bool one = count[k] <= 1;
    sums[k][0] = one ? 0.0 : s1 / cc;
    sums[k][1] = one ? 1.0 : (double)sqrtf(fmaxf(var, g.eps));
  }
  __syncthreads();
  const float alpha = (float)n_rows / (float)max(nonzero, 1);
  each_eight([&](int64_t i0, const int64_t (&k)[8], const float (&x)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (u >= per || i0 + u >= n_rows) break;
      const bool ok = k[u] >= 0 && k[u] < n_groups;
      const int q = ok ? (int)k[u] : 0;
      const float v = group_scalar_of(g, x[u], (float)count[q], (float)sums[q][0], (float)sums[q][1], alpha);
      scalar[i0 + u] = ok ? v : 0.f;
    }
  });
}

template <int MK>
__global__ __launch_bounds__(kBlock) void row_broadcast_kernel(
    const float* __restrict__ row_scalar, const void* __restrict__ mask,
    const int32_t* __restrict__ cu, int64_t n_rows, int64_t n_slots, int64_t uniform_len,
    float clamp_abs, float* __restrict__ out) {
  __shared__ int32_t lds_cu[kLdsRows];
  const int64_t c0 = (int64_t)blockIdx.x * kChunk;
  const int64_t c1 = min(c0 + (int64_t)kChunk, n_slots);
  RowFinder rf;
  if (c1 - c0 == kChunk) {
    // whole chunk: the mask loads of all four steps are in flight before the row search
    float mv[kIter][4];
#pragma unroll
    for (int it = 0; it < kIter; ++it)
      load_mask4<MK>(mask, c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec, mv[it]);
    rf.init(cu, n_rows, uniform_len, c0, c1, lds_cu);
#pragma unroll
    for (int it = 0; it < kIter; ++it) {
      const int64_t i = c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec;
      int r = rf.row(i);
      int64_t rend = rf.row_end(r);
      float sc = row_scalar[r];
      float o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (i + j >= rend) {
          r = rf.row(i + j);
          rend = rf.row_end(r);
          sc = row_scalar[r];
        }
        float v = sc * mv[it][j];
        if (clamp_abs > 0.f) v = fminf(fmaxf(v, -clamp_abs), clamp_abs);
        o[j] = v;
      }
      store4(out, i, o);
    }
    return;
  }
  rf.init(cu, n_rows, uniform_len, c0, c1, lds_cu);
#pragma unroll 1
  for (int it = 0; it < kIter; ++it) {
    const int64_t i = c0 + ((int64_t)it * kBlock + threadIdx.x) * kVec;
    if (i >= c1) continue;
    int r = rf.row(i);
    int64_t rend = rf.row_end(r);
    float sc = row_scalar[r];
    float mv[4], o[4];
    const bool full = (i + kVec <= n_slots);
    if (full) load_mask4<MK>(mask, i, mv);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t p = i + j;
      if (p >= n_slots) break;
      if (p >= rend) {
        r = rf.row(p);
        rend = rf.row_end(r);
        sc = row_scalar[r];
      }
      const float m = full ? mv[j] : load_mask1<MK>(mask, p);
      float v = sc * m;
      if (clamp_abs > 0.f) v = fminf(fmaxf(v, -clamp_abs), clamp_abs);
      o[j] = v;
    }
    if (full) store4(out, i, o);
    else
      for (int j = 0; j < 4 && i + j < n_slots; ++j) out[i + j] = o[j];
  }
}

__global__ __launch_bounds__(kBlock) void fill_zero_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

}  // namespace axon

using namespace axon;

static inline int grid_for(int64_t n_slots) { return (int)((n_slots + kChunk - 1) / kChunk); }

// out[i] = x[i] * s1[0] * (s2 ? s2[0] : 1): the chain rule of a scalar loss whose per-token gradient the
// forward left unscaled (the factors live on the device).
__global__ __launch_bounds__(kBlock) void scale_by_scalars_kernel(const float* __restrict__ x,
                                                                  const float* __restrict__ s1,
                                                                  const float* __restrict__ s2,
                                                                  float* __restrict__ out, int64_t n) {
  const float f = s1[0] * (s2 != nullptr ? s2[0] : 1.f);
  const int64_t n4 = n / 4;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    const float4 v = reinterpret_cast<const float4*>(x)[i];
    reinterpret_cast<float4*>(out)[i] = make_float4(v.x * f, v.y * f, v.z * f, v.w * f);
  }
  const int64_t t = n4 * 4 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) out[t] = x[t] * f;
}

extern "C" int axon_scale_f32(const float* x, const float* s1, const float* s2, float* out, int64_t n,
                              void* stream) {
  if (n < 0) return AXON_ERR_SHAPE;
  if (n == 0) return AXON_OK;
  if (!x || !s1 || !out) return AXON_ERR_ARG;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) return AXON_ERR_ARG;
  const int64_t blocks = (n / 4 + kBlock - 1) / kBlock;
  const unsigned grid = (unsigned)(blocks < 1 ? 1 : blocks < 4096 ? blocks : 4096);
  hipLaunchKernelGGL(scale_by_scalars_kernel, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, x, s1, s2,
                     out, n);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_fill_zero(void* ptr, int64_t n_bytes, void* stream) {
  if (n_bytes < 0 || (n_bytes & 3) != 0) return AXON_ERR_ARG;
  if (n_bytes == 0) return AXON_OK;
  if (ptr == nullptr) return AXON_ERR_ARG;
  const int64_t n = n_bytes / 4;
  int64_t nb = (n + kBlock - 1) / kBlock;
  const int grid = (int)(nb < 4096 ? nb : 4096);
  hipLaunchKernelGGL(fill_zero_kernel, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream,
                     (uint32_t*)ptr, n);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

static int check_rows(const int32_t* cu, int64_t n_rows, int64_t n_slots, int64_t uniform_len) {
  if (n_rows < 0 || n_slots < 0 || uniform_len < 0) return AXON_ERR_ARG;
  if (n_rows >= (int64_t)INT32_MAX || n_slots >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (uniform_len == 0 && cu == nullptr && n_slots > 0) return AXON_ERR_ARG;
  if (uniform_len > 0 && n_rows * uniform_len != n_slots) return AXON_ERR_SHAPE;
  if (uniform_len == 0 && n_rows == 0 && n_slots > 0) return AXON_ERR_SHAPE;  // tokens that belong to no row
  return AXON_OK;
}

extern "C" int64_t axon_row_stats_workspace_bytes(int64_t n_rows) {
  return n_rows < 0 ? -1 : n_rows * 12;
}

extern "C" int axon_row_stats(const float* a, const float* b, const void* mask, int mask_kind,
                              const int32_t* cu, int64_t n_rows, int64_t n_slots,
                              int64_t uniform_len, int flag_mode, float thr, float* cnt,
                              float* sum, int32_t* flag, void* sum_workspace, void* stream) {
  int rc = check_rows(cu, n_rows, n_slots, uniform_len);
  if (rc != AXON_OK) return rc;
  if (n_slots == 0 || n_rows == 0) return AXON_OK;
  if (a == nullptr) return AXON_ERR_ARG;
  if (flag_mode < 0 || flag_mode > 2) return AXON_ERR_ARG;
  if (flag_mode != 0 && flag == nullptr) return AXON_ERR_ARG;
  if (mask_kind != AXON_MASK_F32 && mask_kind != AXON_MASK_I64) return AXON_ERR_ARG;
  if (sum != nullptr && (sum_workspace == nullptr || (reinterpret_cast<uintptr_t>(sum_workspace) & 7)))
    return AXON_ERR_WORKSPACE;
  RowSumAcc acc{nullptr, nullptr};
  if (sum != nullptr) {
    acc.fixed = static_cast<unsigned long long*>(sum_workspace);
    acc.big = reinterpret_cast<float*>(acc.fixed + n_rows);
  }
  const dim3 g(grid_for(n_slots)), blk(kBlock);
  if (mask_kind == AXON_MASK_F32)
    hipLaunchKernelGGL(row_stats_kernel<AXON_MASK_F32>, g, blk, 0, (hipStream_t)stream, a, b, mask,
                       cu, n_rows, n_slots, uniform_len, flag_mode, thr, cnt, acc, flag);
  else
    hipLaunchKernelGGL(row_stats_kernel<AXON_MASK_I64>, g, blk, 0, (hipStream_t)stream, a, b, mask,
                       cu, n_rows, n_slots, uniform_len, flag_mode, thr, cnt, acc, flag);
  AXON_CHECK_LAUNCH();
  if (sum != nullptr) {
    hipLaunchKernelGGL(row_sum_finish_kernel, dim3((unsigned)((n_rows + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, acc, n_rows, sum);
    AXON_CHECK_LAUNCH();
  }
  return AXON_OK;
}

extern "C" int axon_group_stats(const float* scores, const int64_t* gidx, int64_t n_rows,
                                int64_t n_groups, float eps, int norm_by_std, float* mean,
                                float* stdv, float* count, float* scalar, void* stream) {
  if (n_rows < 0 || n_groups < 0) return AXON_ERR_ARG;
  if (n_rows >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (n_rows == 0 || n_groups == 0) return AXON_OK;
  if (!scores || !gidx || !mean || !stdv || !count) return AXON_ERR_ARG;
  hipLaunchKernelGGL(group_stats_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, scores, gidx,
                     n_rows, n_groups, eps, norm_by_std, mean, stdv, count, scalar);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_group_advantage(const float* rewards, const void* mask, int mask_kind, const int32_t* cu,
                                    int64_t n_rows, int64_t n_slots, int64_t uniform_len, const int64_t* gidx,
                                    int64_t n_groups, float eps, int mode, float clamp_abs, float* row_scratch,
                                    float* out, float* partials, void* stream) {
  int rc = check_rows(cu, n_rows, n_slots, uniform_len);
  if (rc != AXON_OK) return rc;
  if (n_slots == 0 || n_rows == 0) return AXON_OK;
  if (n_groups <= 0 || n_groups > kScoreGroups) return AXON_ERR_SHAPE;
  if (!rewards || !gidx || !row_scratch || !out || !partials || mode < 0 || mode > 3) return AXON_ERR_ARG;
  if (reinterpret_cast<uintptr_t>(rewards) & 15) return AXON_ERR_ARG;
  constexpr int kWaves = kScoreThreads / kWave;
  const int64_t blocks = (n_rows + kWaves - 1) / kWaves;
  hipLaunchKernelGGL(group_scores_kernel, dim3((unsigned)(blocks < kScoreBlocks ? blocks : kScoreBlocks)), dim3(kScoreThreads), 0,
                     (hipStream_t)stream, rewards, cu, n_rows, n_slots, uniform_len, gidx,
                     GroupCfg{n_groups, eps, mode}, row_scratch, row_scratch + n_rows,
                     reinterpret_cast<unsigned*>(partials + kTicketsOffset));
  AXON_CHECK_LAUNCH();
  return axon_row_broadcast_mask(row_scratch + n_rows, mask, mask_kind, cu, n_rows, n_slots, uniform_len, clamp_abs, out,
                                 stream);
}

extern "C" int axon_row_broadcast_mask(const float* row_scalar, const void* mask, int mask_kind,
                                       const int32_t* cu, int64_t n_rows, int64_t n_slots,
                                       int64_t uniform_len, float clamp_abs, float* out,
                                       void* stream) {
  int rc = check_rows(cu, n_rows, n_slots, uniform_len);
  if (rc != AXON_OK) return rc;
  if (n_slots == 0 || n_rows == 0) return AXON_OK;
  if (!row_scalar || !out) return AXON_ERR_ARG;
  if (mask_kind != AXON_MASK_F32 && mask_kind != AXON_MASK_I64) return AXON_ERR_ARG;
  const dim3 g(grid_for(n_slots)), blk(kBlock);
  if (mask_kind == AXON_MASK_F32)
    hipLaunchKernelGGL(row_broadcast_kernel<AXON_MASK_F32>, g, blk, 0, (hipStream_t)stream,
                       row_scalar, mask, cu, n_rows, n_slots, uniform_len, clamp_abs, out);
  else
    hipLaunchKernelGGL(row_broadcast_kernel<AXON_MASK_I64>, g, blk, 0, (hipStream_t)stream,
                       row_scalar, mask, cu, n_rows, n_slots, uniform_len, clamp_abs, out);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}
