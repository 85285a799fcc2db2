// The few values between the kernels of one training step (head forward, loss, head backward): launches over one
// block's tokens or a handful of scalars, each in the place of a chain of tensor operations.  A launch over so little
// is about 5 us of GPU time behind another one, whatever it does, and as much host time; a step over 700 tokens, 2.2
// ms most of which are three matrix products, had 39 launches and has 22 with these.
#include "common.h"

namespace axon {

// Gradients of one block's tokens from the loss kernel's array (without the factor acc[5], see axon_policy_loss) and from
// the side terms' (factor side[5]).  Element by element: a block's positions begin anywhere in the step's arrays.
__global__ __launch_bounds__(kBlock) void step_grads_kernel(const float* __restrict__ grad, const float* __restrict__ acc,
                                                            const float* __restrict__ agg_w,
                                                            const float* __restrict__ grad_kl,
                                                            const float* __restrict__ side, float entropy_coef,
                                                            float kl_coef, int64_t n, float* __restrict__ g_lp,
                                                            float* __restrict__ g_en) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float g = grad[i] * acc[5];
  if (grad_kl != nullptr) g += kl_coef * (grad_kl[i] * side[5]);
  g_lp[i] = g;
  if (g_en != nullptr) g_en[i] = agg_w[i] * (side[5] * -entropy_coef);
}

// The step's scalars from its blocks' sums [n_blocks][16] (eight of the loss, eight of the side terms): their totals, the
// loss, and the first and last offset of the packed layout.
__global__ __launch_bounds__(kWave) void step_scalars_kernel(const float* __restrict__ blocks, int n_blocks,
                                                             float entropy_coef, float kl_coef,
                                                             const int32_t* __restrict__ cu, int64_t n_seqs,
                                                             double* __restrict__ out, float* __restrict__ loss) {
  const int k = threadIdx.x;
  float s = 0.f;
  if (k < 16)
    for (int b = 0; b < n_blocks; ++b) s += blocks[b * 16 + k];
  if (k < 16) reinterpret_cast<float*>(out)[k] = s;
  const float entropy = __shfl(s, 8, kWave), kl = __shfl(s, 9, kWave);
  if (k == 0) {
    float l = s;
    if (entropy_coef != 0.f) l -= entropy * entropy_coef;
    if (kl_coef != 0.f) l += kl * kl_coef;
    loss[0] = l;
    out[8] = cu != nullptr ? (double)cu[0] : 0.0;
    out[9] = cu != nullptr ? (double)cu[n_seqs] : 0.0;
  }
}

}  // namespace axon

using namespace axon;

extern "C" int axon_step_grads(const float* grad, const float* acc, const float* agg_w, const float* grad_kl,
                               const float* side, float entropy_coef, float kl_coef, int64_t n, float* g_lp, float* g_en,
                               void* stream) {
  if (n < 0 || n >= (int64_t)INT32_MAX) return AXON_ERR_SHAPE;
  if (n == 0) return AXON_OK;
  if (!grad || !acc || !g_lp || ((g_en || grad_kl) && !side) || (g_en && !agg_w)) return AXON_ERR_ARG;
  hipLaunchKernelGGL(step_grads_kernel, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, (hipStream_t)stream,
                     grad, acc, agg_w, grad_kl, side, entropy_coef, kl_coef, n, g_lp, g_en);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}

extern "C" int axon_step_scalars(const float* blocks, int64_t n_blocks, float entropy_coef, float kl_coef,
                                 const int32_t* cu_seqlens, int64_t n_seqs, double* out, float* loss, void* stream) {
  if (n_blocks <= 0 || n_blocks >= (1 << 24) || n_seqs < 0) return AXON_ERR_SHAPE;
  if (!blocks || !out || !loss || (reinterpret_cast<uintptr_t>(out) & 7)) return AXON_ERR_ARG;
  hipLaunchKernelGGL(step_scalars_kernel, dim3(1), dim3(kWave), 0, (hipStream_t)stream, blocks, (int)n_blocks, entropy_coef,
                     kl_coef, cu_seqlens, n_seqs, out, loss);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}
