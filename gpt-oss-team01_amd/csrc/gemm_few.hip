// bf16-weight instantiations of the few-row GEMM kernel.
#include "gemm_few_kernel.hpp"

namespace gptoss {
int run_gemm_few(const GemmParams &p, bool gather, int epi, int rows_per_tile, int max_tiles, hipStream_t s) {
  if (gather && epi == EPI_SWIGLU) return launch_few_gemm<true, EPI_SWIGLU, false>(p, rows_per_tile, max_tiles, s);
  if (!gather && epi == EPI_F32) return launch_few_gemm<false, EPI_F32, false>(p, rows_per_tile, max_tiles, s);
  if (!gather && epi == EPI_MIXED && !p.tiles) return launch_few_gemm<false, EPI_MIXED, false>(p, rows_per_tile, max_tiles, s);
  if (!gather && epi == EPI_PARTIAL && !p.tiles) return launch_few_gemm<false, EPI_PARTIAL, false>(p, rows_per_tile, max_tiles, s);
  return fail(GPTOSS_ERR_DIM, "run_gemm: no few-row kernel for this form (gather=%d epi=%d)", (int)gather, epi);
}
}  // namespace gptoss
