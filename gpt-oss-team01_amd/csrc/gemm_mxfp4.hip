// MXFP4-weight instantiations of the grouped GEMM kernel, and their dispatch.
#include <algorithm>
#include <mutex>

#include "gemm_few_kernel.hpp"
#include "gemm_mxfp4_kernel.hpp"

namespace gptoss {
GPTOSS_GEMM_INSTANTIATE(2, true, EPI_SWIGLU, true)
GPTOSS_GEMM_INSTANTIATE(2, false, EPI_F32, true)

static hipError_t set_attrs() {
  hipError_t err = hipSuccess;
  GPTOSS_GEMM_SET_ATTR(2, true, EPI_SWIGLU, true)
  GPTOSS_GEMM_SET_ATTR(2, false, EPI_F32, true)
  return err;
}

// Up to so many work items, one per CU, an item's own latencies are the launch: the streaming kernel, with eight waves and
// four slabs in flight for an item, is the faster one (4096 x 1536, 4 experts of 60 rows 66 us against 72, second product
// of 8 experts of 75 rows, 2880 x 2880, 28 against 30; with 391 items 44 against 39, 348 items 109 against 97).
constexpr int FP4_ITEM_PER_CU = 256;

template <bool GATHER, int EPI>
static int dispatch_rows(const GemmParams &p, int rows_per_tile, int max_tiles, hipStream_t s) {
  if (rows_per_tile == 32 && gemm_few_applies(p, rows_per_tile, max_tiles)) return launch_few_gemm<GATHER, EPI, true>(p, rows_per_tile, max_tiles, s);
  if (p.tiles && rows_per_tile <= 64)
    return (long long)max_tiles * p.n_col_tiles <= FP4_ITEM_PER_CU ? launch_gemm<2, GATHER, EPI, true>(p, max_tiles, s)
                                                                   : launch_mxfp4<GATHER, EPI>(p, max_tiles, s);
  return fail(GPTOSS_ERR_DIM, "run_gemm: unsupported rows_per_tile %d", rows_per_tile);
}

static int dispatch(const GemmParams &p, bool gather, int epi, int rows_per_tile, int max_tiles, hipStream_t s) {
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static bool done[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "run_gemm: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!done[dev]) GPTOSS_HIP(set_attrs());
    done[dev] = true;
  }
  if (gather && epi == EPI_SWIGLU) return dispatch_rows<true, EPI_SWIGLU>(p, rows_per_tile, max_tiles, s);
  if (!gather && epi == EPI_F32) return dispatch_rows<false, EPI_F32>(p, rows_per_tile, max_tiles, s);
  return fail(GPTOSS_ERR_DIM, "run_gemm: unsupported combination (gather=%d epi=%d)", (int)gather, epi);
}

// a library of model classes without MXFP4 experts is linked without this file
static const bool registered = [] {
  run_gemm_mxfp4 = dispatch;
  return true;
}();
}  // namespace gptoss
