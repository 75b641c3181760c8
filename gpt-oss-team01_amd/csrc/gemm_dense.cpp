// Host side of the dense bf16 GEMMs (kernel dispatch) and the weight repacking kernel.  The GEMM kernels
// themselves are in gemm_kernel.hpp and gemm_tall_kernel.hpp.
#include <math.h>
#include <stdlib.h>

#include <mutex>

#include "common.hpp"
#include "gemm.hpp"

namespace gptoss {

// Repack row-major [n_out, n_in] matrices into fragment order:
//   dst[((nb*KS + ks)*64 + lane)*8 + j] = W[row(nb*32 + lane%32)][ks*16 + (lane/32)*8 + j]
// With GLU pairing, virtual row v of a 32-row block maps to pair (v/32)*16 + v%16, gate for the
// first 16 virtual rows and up for the second 16.
template <typename SRC>
__global__ __launch_bounds__(256) void pack_weight_kernel(const SRC *__restrict__ src,
                                                          bf16_t *__restrict__ dst, int n_out,
                                                          int n_in, int glu) {
  const int ksteps = n_in / 16;
  const size_t frags_per_mat = (size_t)(n_out / 32) * ksteps;
  const size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x;  // one (fragment, lane) per thread
  const size_t frag = gid >> 6;
  const int lane = (int)(gid & 63);
  const int mat = blockIdx.y;
  if (frag >= frags_per_mat) return;
  const int nb = (int)(frag / ksteps), ks = (int)(frag - (size_t)nb * ksteps);
  int v = nb * 32 + (lane & 31);
  int row = v;
  if (glu) row = 2 * ((v >> 5) * 16 + (v & 15)) + ((v >> 4) & 1);
  const SRC *sp = src + ((size_t)mat * n_out + row) * n_in + ks * 16 + (lane >> 5) * 8;
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if constexpr (sizeof(SRC) == 4) {
      o[j] = pack_bf16x2((float)sp[2 * j], (float)sp[2 * j + 1]);
    } else {
      o[j] = (uint32_t)sp[2 * j] | ((uint32_t)sp[2 * j + 1] << 16);
    }
  }
  u32x4 *dp = reinterpret_cast<u32x4 *>(dst + ((size_t)mat * frags_per_mat + frag) * 512 + lane * 8);
  *dp = u32x4{o[0], o[1], o[2], o[3]};
}

// Host-side dispatcher of the form without gather.  rows_per_tile selects the kernel.
template <int MBMAX, bool GATHER, int EPI, bool FP4>
int launch_gemm(const GemmParams &p, int max_tiles, hipStream_t s);  // gemm_bf16.hip, gemm_mixed_bf16.hip

template <int EPI>
static int dispatch_rows(const GemmParams &p, int rows_per_tile, int max_tiles, hipStream_t s) {
  switch (rows_per_tile) {
    case 32: return launch_gemm<1, false, EPI, false>(p, max_tiles, s);
    case 64: return launch_gemm<2, false, EPI, false>(p, max_tiles, s);
    case 96: return launch_gemm<3, false, EPI, false>(p, max_tiles, s);
    case 128: return launch_gemm<4, false, EPI, false>(p, max_tiles, s);
    case 160: return launch_gemm<5, false, EPI, false>(p, max_tiles, s);
  }
  return fail(GPTOSS_ERR_DIM, "run_gemm: unsupported rows_per_tile %d", rows_per_tile);
}

hipError_t gemm_set_attrs_bf16();        // gemm_bf16.hip
hipError_t gemm_set_attrs_mixed_bf16();  // gemm_mixed_bf16.hip

// Raises the dynamic-LDS limit of every such kernel on the calling thread's current device, the
// first time that device launches one.
static int gemm_prepare_device() {
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static bool done[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "run_gemm: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  std::lock_guard<std::mutex> lock(mu);
  if (!done[dev]) {
    GPTOSS_HIP(gemm_set_attrs_bf16());
    GPTOSS_HIP(gemm_set_attrs_mixed_bf16());
    done[dev] = true;
  }
  return GPTOSS_OK;
}

// Estimated us of a launch, for choosing its kernel, row tile and parts.  `blocks`: 32-column blocks of all its work items,
// `slabs`: 64-k slabs an item walks.  A round of work items takes a part of its own (first loads, epilogue) beside its slabs,
// and both take longer the more CUs are at it: terms per round and terms per full round's worth of items.
// Streaming kernels (gemm_kernel.hpp): items of MB 32-row blocks x 256 columns, 256 to a round.
// Few-row kernels (gemm_few_kernel.hpp): 128 columns per workgroup, 256 to a round; up to 512 blocks a workgroup is one block.
// Fitted to every tile and every number of parts that a launch could have, weights from HBM: 27 shapes of 512-16384 columns
// and K 256-8192 at 34 row counts of 8-2047, and 12 shapes at 26 with their K cut as well; 4 to 12 % rms (64 rows in several
// rounds: 5 % on top, as what they gain at a tie is less than what they lose).  With one fixed part per launch, products of
// short K or narrow N took up to 37 % longer than on streaming kernels alone (us: 1280 x 1280 with its K cut, 257 rows
// 11.1 instead of 8.1; 2048 x 256, 257 rows 8.0 instead of 6.3).
// The few-row kernels have become faster since, tiles of up to 16 rows by up to a third (gemm_few_kernel.hpp), which the fit leaves
// out: uncut products of up to 8 / 16 rows take 0.79 / 0.85 of few_us' time, where the streaming kernels take 1.12 of streaming_us', so
// these look better there than they are.  What that costs is stated at the rules that use it; how often to cut the K of so
// few rows is by partial_us.
static double streaming_us(int mb, long long blocks, int slabs) {
  // [mb - 1]: launch; per round, and per slab of it; per full round's items, and per slab of them
  static const double t[5][5] = {{3.2, 0.63, 0.496, 1.8, 0.028}, {3.5, 1.35, 0.533, 3.3, 0.106}, {4.0, 2.5, 0.578, 3.8, 0.145},
                                 {4.3, 3.7, 0.635, 3.9, 0.222}, {5.0, 5.0, 0.724, 3.5, 0.303}};
  const double *c = t[mb - 1];
  return c[0] + (double)((blocks + 2047) / 2048) * (c[1] + c[2] * slabs) + blocks / 2048.0 * (c[3] + c[4] * slabs);
}

static double few_us(int mb, long long blocks, int slabs) {
  if (blocks <= FEW_SOLO_BLOCKS) {
    const double full = (double)blocks / FEW_SOLO_BLOCKS;
    return mb == 1 ? 3.6 + 0.078 * slabs + full * (1.3 + 0.142 * slabs) : 5.0 + 0.239 * slabs + full * (1.8 + 0.079 * slabs);
  }
  const double rounds = (double)((blocks + 1023) / 1024), full = blocks / 1024.0;
  return mb == 1 ? 3.4 + rounds * (1.1 + 0.175 * slabs) + full * (0.7 + 0.071 * slabs)
                 : 3.9 + rounds * (1.58 + 0.191 * slabs) + full * (1.15 + 0.147 * slabs);
}

// The few-row kernels on up to 8 or 16 rows, K cut into parts: 59 shapes of 512-16384 columns and K 512-12288 at every number of parts
// up to 16, weights from HBM, 1 / 6 / 8 / 12 / 16 rows; 4 to 5 % rms (some of 9 to 16 rows beyond 512 blocks 8).  256 blocks to a round.
static double partial_us(int rows, long long blocks, int slabs) {
  // [rows > 8][more than FEW_SOLO_BLOCKS]: launch; per round, and per slab of it; per full round's blocks, and per slab of them
  static const double t[2][2][5] = {{{2.6, 0.76, 0.035, -0.2, 0.1}, {2.6, 0.46, 0.047, -0.048, 0.096}},
                                    {{2.9, 0.065, 0.056, 0.49, 0.091}, {2.9, 1.0, 0.0021, -0.62, 0.15}}};
  const double *c = t[rows > 8][blocks > FEW_SOLO_BLOCKS], full = blocks / 256.0;
  return c[0] + (double)((blocks + 255) / 256) * (c[1] + c[2] * slabs) + full * (c[3] + c[4] * slabs);
}

// Uncut dense problems: the kernel that is estimated to be the faster one with this row tile.
static bool dense_few(int rows_per_tile, int tiles, int N, int K) {
  const int mb = rows_per_tile / 32;
  return mb <= 2 && few_us(mb, (long long)tiles * (N / 32), K / 64) < streaming_us(mb, (long long)tiles * gemm_col_tiles(N) * 8, K / 64);
}

int run_gemm_dense(const GemmParams &p, int epi, int rows_per_tile, int max_tiles, hipStream_t s) {
  // output and operand offsets inside the kernels are 32-bit element counts
  const long long max_rows = p.tiles ? (long long)max_tiles * rows_per_tile : p.dense_rows;
  GPTOSS_REQUIRE(max_rows * p.N < (1ll << 32) && max_rows * p.K < (1ll << 32), GPTOSS_ERR_DIM,
                 "run_gemm: rows x columns must stay below 2^32 elements (rows<=%lld N=%d K=%d)", max_rows, p.N, p.K);
  if (rows_per_tile == 256) return run_gemm_tall(p, epi, max_tiles, max_rows, s);
  if (epi != EPI_ARGMAX && gemm_few_applies(p, rows_per_tile, max_tiles) &&
      (p.tiles ? grouped_few(rows_per_tile, max_tiles, p.N) : epi == EPI_PARTIAL || dense_few(rows_per_tile, max_tiles, p.N, p.K)))
    return run_gemm_few(p, false, epi, rows_per_tile, max_tiles, s);
  int prc = gemm_prepare_device();
  if (prc != GPTOSS_OK) return prc;
  if (epi == EPI_F32) return dispatch_rows<EPI_F32>(p, rows_per_tile, max_tiles, s);
  if (epi == EPI_MIXED && p.tiles == nullptr) return dispatch_rows<EPI_MIXED>(p, rows_per_tile, max_tiles, s);
  if (epi == EPI_PARTIAL && p.tiles == nullptr) return dispatch_rows<EPI_PARTIAL>(p, rows_per_tile, max_tiles, s);
  if (epi == EPI_ARGMAX && p.tiles == nullptr && p.amax_val && p.amax_idx)
    return dispatch_rows<EPI_ARGMAX>(p, rows_per_tile, max_tiles, s);
  return fail(GPTOSS_ERR_DIM, "run_gemm: unsupported combination (dense, epi=%d)", epi);
}

// The same for the 256-row kernel (gemm_tall_kernel.hpp): rounds of 32 tiles per XCD, the last one in halves of a tile where
// they leave half of its workgroups idle.  A CU's slab takes longer the more CUs multiply (the chip is at its power limit).
// Within 6 % of 63 products: 9 shapes of 1024-24576 columns and K 512-10240 at 7 row counts of 2048-8000, at fewer rows within 8 %.
static double tall_tiles_us(double tiles, int slabs) {
  const int mine = (int)ceil(tiles / 8), rest = mine % 32;
  double us = 4.0 + mine / 32 * (11.5 + 1.44 * slabs);
  if (rest && 2 * rest <= 32) us += 9.0 + (0.39 + 0.45 * rest / 16.0) * slabs;
  else if (rest) us += 11.5 + (0.54 + 0.9 * rest / 32.0) * slabs;
  return us;
}
static double tall_us(int B, int N, int K) { return tall_tiles_us(cdiv(B, 256) * cdiv(N, 256), K / 64); }

double grouped_us(int rows_per_tile, double tiles, bool few, int N, int K) {
  // (tiles of several experts share no weights: a tenth more)
  if (rows_per_tile == 256) return 1.1 * tall_tiles_us(tiles * cdiv(N, 256), K / 64);
  return few ? few_us(rows_per_tile / 32, (long long)(tiles * (N / 32)), K / 64)
             : streaming_us(rows_per_tile / 32, (long long)(tiles * gemm_col_tiles(N) * 8), K / 64);
}

// GPTOSS_DENSE_TALL_MIN_ROWS: rows from which a dense fp32-output GEMM uses the 256-row kernel, in place of the estimates
static int dense_tall_min_rows() {
  static const int v = [] {
    const char *e = getenv("GPTOSS_DENSE_TALL_MIN_ROWS");
    return e ? atoi(e) : 0;
  }();
  return v;
}

// Whether a dense product is one for the 256-row kernel, given the best estimate of the others, which is up to a fifth too high
// for products of a thousand rows: below 2048 rows the 256-row kernel has to be clearly ahead, above clearly behind.  Timed with
// both at 630 products (18 shapes of 512-65536 columns, K 256-10240, 256-8000 rows) against 256-row tiles from 2048 rows on: 5 %
// less time on average (8192 x 2048, 2047 rows 86 -> 62 us, 16640 x 2048, 1500 rows 123 -> 106; 1024 x 10240, 4100 rows 118 -> 105).
// Two are slower, 4128 x 256 with 4000 and 4096 rows, 32 -> 33.5: the others' estimate leaves out what writes of short K cost.  A
// margin of 1.15 instead of 1.1 mends these and costs more elsewhere (5120 x 2880, 3100 rows 97 -> 112, 2560 x 320, 2500 rows
// 14.7 -> 17.5).  Missed by the estimates: 65536 x 1024, 600 rows, 122 instead of 100.
static bool dense_tall(int B, int N, int K, double other_us) {
  if (dense_tall_min_rows() > 0) return B >= dense_tall_min_rows();
  return tall_us(B, N, K) < (B < 2048 ? 0.88 : 1.1) * other_us;
}

// rows from which the classifier's arg-max GEMM uses it (measured, vocabulary 201088 x 2880: 256 rows
// 360 -> 295 us, 512 rows 716 -> 556, 1024 rows 1194 -> 986-1007, 2048 rows 2319 -> 1859)
static int argmax_tall_min_rows() {
  static const int v = [] {
    const char *e = getenv("GPTOSS_ARGMAX_TALL_MIN_ROWS");
    const int n = e ? atoi(e) : 0;
    return n > 0 ? n : 256;
  }();
  return v;
}

// Row tile of a dense GEMM below the 256-row kernels: the one with the least estimated time; ties go to the larger tile
// (fewer re-reads of the weights).  Timed with every tile at the 918 sizes above, with the kernels that the estimates were fitted to:
// 1 % slower than the best one on average and 16 % faster than the streaming kernels alone (5120 x 2880, 97 / 200 / 364 rows 32 / 32 /
// 33 -> 19 / 21 / 22 us).  With the present ones, 53 shapes of 512-16384 columns and K 256-8192, 1 to 32 rows: less than 1 % slower than the
// better of both kernels, which is the few-row one at all of them.  The estimates leave
// out what a second row tile costs in reads of the weights, so from 65 column tiles on up to 128 rows are one tile:
// 24576 x 2880, 65 / 128 rows 65 / 69 us with tiles of 64, 46 / 54 with one.  Hundreds of column tiles (an unembedding) fill
// the chip at any size: one tile up to 96 rows, then 128, measured best at 1024.
static int dense_rows_per_tile(int B, int n_col_tiles, int N, int K, int epi, double *us) {
  auto estimate = [&](int mb) {
    const int tiles = cdiv(B, 32 * mb);
    return epi != EPI_ARGMAX && dense_few(32 * mb, tiles, N, K) ? few_us(mb, (long long)tiles * (N / 32), K / 64)
                                                                : streaming_us(mb, (long long)tiles * n_col_tiles * 8, K / 64);
  };
  if (n_col_tiles >= 128 || epi == EPI_ARGMAX || (n_col_tiles > 64 && B <= 128)) {
    const int rpt = B <= 96 ? (int)align_up(B, 32) : n_col_tiles >= 64 ? 128 : 0;
    if (rpt) {
      *us = estimate(rpt / 32);
      return rpt;
    }
  }
  int rpt = 160;
  for (int mb = 1; mb <= 5; mb++) {
    const double t = estimate(mb);
    if (mb == 1 || t <= *us) {
      *us = t;
      rpt = 32 * mb;
    }
    if (B <= 32 * mb) break;
  }
  return rpt;
}

static GemmParams dense_params(const bf16_t *A, const bf16_t *W, const float *bias, void *out, int B, int N, int K) {
  GemmParams g{};
  g.A = A;
  g.W = W;
  g.bias = bias;
  g.out = out;
  g.tiles = nullptr;
  g.dense_rows = g.max_tile_rows = B;
  g.N = N;
  g.K = K;
  g.n_col_tiles = gemm_col_tiles(N);
  return g;
}

// C[B, N] = A[B, K] . W[N, K]^T (+ bias): the dense GEMMs of a step (QKV and output projections,
// classifier), with the kernel and row tile chosen from the batch size.
int dense_gemm(const bf16_t *A, const bf16_t *W, const float *bias, void *out, int epi, int B, int N,
               int K, hipStream_t s, float *amax_val, int *amax_idx, int *amax_tiles) {
  GemmParams g = dense_params(A, W, bias, out, B, N, K);
  g.amax_val = amax_val;
  g.amax_idx = amax_idx;
  double us = 0.0;
  int rpt = dense_rows_per_tile(B, g.n_col_tiles, N, K, epi, &us);
  if ((epi == EPI_ARGMAX ? B >= argmax_tall_min_rows() : dense_tall(B, N, K, us)) && gemm_tall_applies(g, false, epi) &&
      gemm_tall_shape_ok(N, K, B))
    rpt = 256;
  if (epi == EPI_ARGMAX) {
    GPTOSS_REQUIRE(amax_tiles, GPTOSS_ERR_NULL, "dense_gemm: the arg-max form reports its pairs per row");
    *amax_tiles = rpt == 256 ? 2 * g.n_col_tiles : g.n_col_tiles;
  }
  return run_gemm_dense(g, epi, rpt, cdiv(B, rpt), s);
}

int dense_gemm_mixed(const bf16_t *A, const bf16_t *W, float *out, const GemmBf16Range *ranges, int n_ranges, int B,
                     int N, int K, hipStream_t s) {
  GPTOSS_REQUIRE(n_ranges >= 0 && n_ranges <= 2, GPTOSS_ERR_DIM, "dense_gemm_mixed: %d ranges", n_ranges);
  GemmParams g = dense_params(A, W, nullptr, out, B, N, K);
  bool wide = true;   // rows that the 256-row kernel can write 16 bytes at a time
  for (int i = 0; i < n_ranges; i++) {
    g.range[i] = ranges[i];
    wide = wide && ranges[i].ld % 8 == 0 && aligned(ranges[i].out, 16);
    GPTOSS_REQUIRE(ranges[i].from % 32 == 0 && ranges[i].to % 32 == 0 && ranges[i].ld % 4 == 0 && aligned(ranges[i].out, 8),
                   GPTOSS_ERR_DIM, "dense_gemm_mixed: ranges are whole 32-column blocks of aligned rows");
  }
  double us = 0.0;
  int rpt = dense_rows_per_tile(B, g.n_col_tiles, N, K, EPI_MIXED, &us);
  if (dense_tall(B, N, K, us) && wide && gemm_tall_applies(g, false, EPI_MIXED) && gemm_tall_shape_ok(N, K, B)) rpt = 256;
  return run_gemm_dense(g, EPI_MIXED, rpt, cdiv(B, rpt), s);
}

// Few rows and few columns leave most CUs without a work item while those that have one walk all of K.
// Cutting K makes more items; what it costs is a part per round and the reading of the partial sums.  All row tiles and parts timed
// at the 312 sizes above, with the kernels that the estimates were fitted to:
// the chosen ones take 2 % longer than the best ones on average and are 15 % faster than with streaming kernels alone (2048 x 2048,
// 8 / 400 / 1024 rows 7.0 / 14.6 / 21.8 -> 4.7 / 11.5 / 17.5 us).  Up to 8 / 16 rows, where partial_us decides, the chosen parts
// take 1 % longer than the best, by few_us 9 / 7 % (2048 x 12288, 8 rows, 16 parts 11.7 us, four 10.3; 4096 x 2048 eight 6.7, one or two
// 5.5-5.8; 2880 x 4096 eleven 7.6, two 6.7); 17 to 32 rows 5 %.
int dense_gemm_partial(const bf16_t *A, const bf16_t *W, float *out, size_t max_elems, int *parts, int B, int N, int K,
                       hipStream_t s) {
  *parts = 1;
  GemmParams g = dense_params(A, W, nullptr, out, B, N, K);
  if (B >= 2048) return dense_gemm(A, W, nullptr, out, EPI_F32, B, N, K, s);
  const int nslab = K / 64;
  double best = 0.0;
  int rpt = 32, splits = 1, slabs = nslab;
  for (int mb = 1; mb <= 5; mb++) {
    if (mb > 1 && 32 * (mb - 1) >= B) break;
    for (int want = 1; want <= GEMM_MAX_PARTS; want++) {
      const int per = cdiv(nslab, want), n = cdiv(nslab, per);
      // (an item prefetches two slabs of the next one, so no part may have fewer)
      if (n != want || (n > 1 && (per < 4 || nslab - per * (n - 1) < 2 || (size_t)n * B * N > max_elems))) continue;
      const int tiles = cdiv(B, 32 * mb);
      const bool few = n == 1 ? dense_few(32 * mb, tiles, N, K) : mb <= 2;   // as run_gemm_dense has it
      const double cost = (few ? B <= 16 ? partial_us(B, (long long)(N / 32) * n, per) : few_us(mb, (long long)tiles * (N / 32) * n, per)
                               : streaming_us(mb, (long long)tiles * g.n_col_tiles * 8 * n, per)) +
                          (n - 1) * (double)B * N * 4 / 5e6;
      if ((mb == 1 && n == 1) || cost < best) {
        best = cost;
        rpt = 32 * mb;
        splits = n;
        slabs = per;
      }
    }
  }
  if (splits == 1) return run_gemm_dense(g, EPI_F32, rpt, cdiv(B, rpt), s);
  g.k_splits = splits;
  g.split_slabs = slabs;
  *parts = splits;
  return run_gemm_dense(g, EPI_PARTIAL, rpt, cdiv(B, rpt), s);
}

}  // namespace gptoss

using namespace gptoss;

extern "C" size_t gptoss_packed_weight_bytes(int n_mat, int n_out, int n_in) {
  if (n_mat <= 0 || n_out <= 0 || n_in <= 0) return 0;
  return (size_t)n_mat * n_out * n_in * sizeof(bf16_t);
}

extern "C" int gptoss_pack_weight(const void *src, void *dst, int n_mat, int n_out, int n_in,
                                  int flags, void *stream) {
  GPTOSS_REQUIRE(src && dst, GPTOSS_ERR_NULL, "pack_weight: null pointer");
  const int glu = (flags & GPTOSS_PACK_GLU) ? 1 : 0;
  GPTOSS_REQUIRE(n_mat >= 1 && n_out > 0 && n_in > 0 && n_out % 32 == 0 && n_in % 64 == 0, GPTOSS_ERR_DIM,
                 "pack_weight: need n_out %% 32 == 0 and n_in %% 64 == 0 (n_out=%d n_in=%d)", n_out, n_in);
  GPTOSS_REQUIRE(aligned(src, 16) && aligned(dst, 16), GPTOSS_ERR_ALIGN,
                 "pack_weight: pointers must be 16-byte aligned");
  size_t threads = (size_t)(n_out / 32) * (n_in / 16) * 64;
  dim3 grid((unsigned)((threads + 255) / 256), n_mat);
  hipStream_t s = (hipStream_t)stream;
  if (flags & GPTOSS_PACK_SRC_FP32)
    pack_weight_kernel<float><<<grid, 256, 0, s>>>((const float *)src, (bf16_t *)dst, n_out, n_in, glu);
  else
    pack_weight_kernel<bf16_t><<<grid, 256, 0, s>>>((const bf16_t *)src, (bf16_t *)dst, n_out, n_in, glu);
  GPTOSS_LAUNCH_CHECK("pack_weight_kernel");
  return GPTOSS_OK;
}
