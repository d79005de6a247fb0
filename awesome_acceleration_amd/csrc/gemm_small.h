// The projections of a decode step of few sequences (csrc/gemm_small.hip),
// reached from aac_gemm_nt's own choice of tiling and from
// aac_rmsnorm_gemm_nt.
#pragma once

#include "aac_common.h"

namespace aac {
namespace gs {

struct Args {
  const u16* x;  // [m, k] rows; with a norm: the block output before the residual add
  const u16* w;
  u16* y;
  int64_t x_stride, w_stride, y_stride;  // elements
  int32_t m, k;
  int32_t n_tiles;   // tiles along the output columns
  int32_t silu_off;  // gate/up pairing: W row of up column 0 (= I)
  const u16* res;    // residual added before the norm, or null
  u16* res_out;      // x + res, rounded
  const u16* norm_w; // null: no norm
  float eps;
};

// Whether the small-batch kernel takes y [m, n] = x w^T of depth k (see
// gemm_small.hip for where the line lies).
bool small_takes(int m, int n, int k);
int launch_small(const Args& a, int n_out, bool silu, bool f16, hipStream_t st);

}  // namespace gs
}  // namespace aac
