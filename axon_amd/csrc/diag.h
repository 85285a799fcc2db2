// What the kernels that form the mismatch diagnostics share: the layout of the per-workgroup token partials and of the
// per-row sums, and the pass over the rows (diag.hip) that turns both into the reported sums.
#pragma once
#include "common.h"

namespace axon {

constexpr int kDiagSums = 23;    // token-level sums, see axon_amd.h
constexpr int kDiagMinMax = 6;   // max e, min e, max |pa-ps|, min |pa-ps|, max |lr|, min |lr|
constexpr int kDiagStride = 32;  // floats per workgroup in `partials`
constexpr int kDiagRowVals = 6;  // cnt, sum old, sum sampler, sum lr, sum e, sum token-rejected

struct DiagCfg {
  int is_mode, rs_mode;  // 0 off, 1 token, 2 sequence, 3 geometric (rs only)
  int with_gap;          // also the off-policy diagnostics (out[42..49], [59], [69]), from the sums of old and sampler
  float is_lo, is_hi, rs_lo, rs_hi;                  // ratio thresholds
  float log_is_lo, log_is_hi, log_rs_lo, log_rs_hi;  // fp32 log of the same
};

struct DiagWorkspace {
  float* row_vals;  // [kDiagRowVals][n_rows]
  float* partials;  // [token_blocks][kDiagStride]
  double* parts;    // the row pass's per-workgroup results
};
DiagWorkspace diag_workspace(float* base, int64_t n_rows, int64_t token_blocks);
int64_t diag_workspace_bytes(int64_t n_rows, int64_t token_blocks);
int launch_diag_rows(const DiagWorkspace& w, int token_blocks, int64_t n_rows, const DiagCfg& cfg, double* out,
                     hipStream_t st);

}  // namespace axon
