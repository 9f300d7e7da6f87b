// gemm_q6k.hip -- the fused-dequant bf16 GEMM (gemm_core.hpp) for Q6_K
// weights: more than 64 tokens, rows of whole block pairs (n_cols % 512 == 0).
// swamp_gemm_dq_route says which of those calls come here; without scratch the
// others do too.
#include "gemm_core.hpp"

size_t swamp_gemm_q6k_scratch_bytes(int m, int n_rows, int n_cols) {
  return swamp::scratch_round(plan_bf16<SWAMP_Q6_K>(m, n_rows, n_cols).part_bytes);
}

int swamp_launch_gemm_q6k(const void *d_w, const void *d_x, float *d_y, int m, int n_rows,
                          int n_cols, swamp::Scratch &sc, hipStream_t s) {
  if (!swamp::q6k_gemm_fusable(m, n_cols)) return SWAMP_EWORKSPACE;
  return launch_bf16<SWAMP_Q6_K>(static_cast<const uint8_t *>(d_w),
                                 static_cast<const uint16_t *>(d_x), d_y, m, n_rows, n_cols, sc, s);
}
