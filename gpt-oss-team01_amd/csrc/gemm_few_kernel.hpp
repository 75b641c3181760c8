// GEMMs of a few rows for gfx950: the same products as gemm_kernel.hpp for row tiles of at most 32 or 64 rows.
//
//   C[rows, N] = A[rows, K] . W[N, K]^T      a decoding step of few sequences, a short prompt, an expert's few tokens
//
// Nothing but reading W takes time here, so what counts is how many bytes of W are on their way at any moment, from how
// many CUs.  The streaming kernels give 256 columns to a workgroup of eight waves with two 4 KB slabs of W in flight
// each, on a grid of one workgroup per CU: one token's four experts are then 92 (first product) and 48 (second) work
// items on 256 CUs.  Here a workgroup is 128 columns, or 32 (below), the grid has one for every work item, and a wave
// has eight slabs in flight.  To have the registers for that, A does not pass through them slab by slab: chunks of eight
// slabs (64 rows, MXFP4: four) are staged in LDS, one barrier each, and W's loads stay in flight across it.  Operand
// roles, order of the sum over K and epilogues are those of the streaming kernels, so a row has the same bits whichever
// kernel computes it.
// Measured, 2880 x 2880 experts, streaming kernels -> these (us): one token, both products 36 + 32 -> 24 + 14, MXFP4
// block 60 -> 43; 27 tokens 156 + 91 -> 157 + 81 (5.9-6.8 TB/s either way); MXFP4 block of 12 tokens 114 -> 87.
// Dense 5120 x 2880: one row 31 -> 9, 32 rows 33 -> 11, 64 rows 37 -> 16, 200 rows 32 -> 21.
// (A read straight from memory in operand order, without LDS: one token 60, but 12 tokens on MXFP4 127,
// because A is then four times the bytes of W.  One wave with 16 rows for MXFP4's small tiles: nine tokens 86.0 -> 87.6,
// twelve 87.8 -> 93.5.)
#pragma once
#include "gemm_kernel.hpp"

namespace gptoss {

// A workgroup: WAVES 32-column blocks, one per wave, times tiles of at most ROWS rows.
//   4 x 32, 4 x 64   the waves share the staged rows
//   1 x 8            one wave can stage so few rows by itself, and four times as many workgroups fill the chip: one
//                    token's block 68 -> 59 us, eight tokens' 178 -> 176
//   1 x 32, 1 x 64   the same for launches of at most FEW_SOLO_BLOCKS blocks, on the registers of two waves

constexpr int FEW_RING = 8;   // 64-k slabs of W that a wave keeps in flight
constexpr int few_chunk(int rows, bool fp4) { return rows <= 32 && !fp4 ? 8 : 4; }   // slabs of A that are staged together: one barrier each
constexpr int few_row(int rows, bool fp4) { return few_chunk(rows, fp4) * BK + 8; }   // padded row of a staged chunk in bf16 elements
constexpr int few_ahead(int rows) { return rows <= 32 ? 4 : 2; }       // k-steps whose operands are read from LDS ahead
// Waves per SIMD.  A single wave that stages 32 rows or more needs the registers of two.  MXFP4: expanding the codes takes
// as long as the products, and a third wave fills in for it (a slab of W is five registers); with two waves, sixteen slabs
// in flight and chunks of eight, 12 tokens took 95 us instead of 87, 600 on 128 experts 410 instead of 394.
constexpr int few_occupancy(int waves, int rows, bool fp4) { return waves == 1 && rows > 8 ? 1 : fp4 ? 3 : 2; }

typedef __amdgpu_buffer_rsrc_t few_rsrc_t;
// cache policy of a buffer load: the non-temporal bit
constexpr int FEW_NT = 2;
// A's buffer: offsets from here on read as zeros
constexpr uint32_t FEW_A_BYTES = 0x80000000u;

__device__ __forceinline__ few_rsrc_t few_buffer(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

template <int WAVES, int ROWS, bool GATHER, int EPI, bool FP4, bool ONCE>
__device__ __forceinline__ void few_block(const GemmParams &p, bf16_t *lds, int mat, int row0, int rows, int cb, int slab0,
                                          int nslab, void *out) {
  constexpr int RING = FEW_RING;
  constexpr int RB = (ROWS + 31) / 32, CHUNK = few_chunk(ROWS, FP4), ROW = few_row(ROWS, FP4), AHEAD = few_ahead(ROWS);
  constexpr int WQ = FP4 ? 1 : 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, kslab = K / BK;
  const bool live = cb * 32 < N;   // the last workgroup of a row tile may have waves to spare

  // W: the block's slabs lie one behind the other.  Slabs past the end are requested all the same (every load of the
  // loop is unconditional) and read as zeros without touching memory: they lie outside the buffer.  (The part of an
  // offset that is checked against the buffer's size is the one in the vector register, so the slab goes there.)
  const size_t mat_bytes = FP4 ? (size_t)N * K / 2 + (size_t)N * K / 32 : (size_t)N * K * 2;
  const char *mb = reinterpret_cast<const char *>(p.W) + (size_t)mat * mat_bytes;
  constexpr int SLAB = FP4 ? 1024 : 4096;
  const few_rsrc_t wb = few_buffer(mb + ((size_t)cb * kslab + slab0) * SLAB, live ? nslab * SLAB : 0);
  const few_rsrc_t sb = few_buffer(FP4 ? mb + (size_t)N * K / 2 + ((size_t)cb * kslab + slab0) * 64 : mb,   // MXFP4 scales
                                   FP4 && live ? nslab * 64 : 0);
  u32x4 w[RING][WQ];
  uint32_t sc[RING];
  auto load_w = [&](int s, auto r) {
    constexpr int R = decltype(r)::value;
#pragma unroll
    for (int q = 0; q < WQ; q++)
      w[R][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, lane * 16 + s * SLAB + q * 1024, 0, ONCE ? FEW_NT : 0));
    if constexpr (FP4) sc[R] = __builtin_amdgcn_raw_buffer_load_b16(sb, (lane & 31) * 2 + s * 64, 0, ONCE ? FEW_NT : 0);
  };
  // which rows of A the tile's rows are: before W, because loads return in order
  int id = row0 + min(lane, rows - 1);
  if (GATHER) id = p.row_ids[id];
  static_for<0, RING>([&](auto r) { load_w(decltype(r)::value, r); });
  const few_rsrc_t bb = few_buffer(p.bias && live ? p.bias + (size_t)mat * N + cb * 32 : nullptr, p.bias && live ? 128 : 0);
  const int bias = __builtin_amdgcn_raw_buffer_load_b32(bb, (lane & 31) * 4, 0, 0);

  // A: the workgroup copies chunks of ROWS rows x CHUNK slabs, a wave 1 KB (one row or two) per load.  Rows beyond the
  // tile's and k beyond K are zeros, again from outside the buffer.
  constexpr int PIECES = CHUNK * 8, PER = 64 / PIECES;   // 16-byte pieces of a row; rows of a load instruction
  constexpr int NA = ROWS / PER / WAVES;
  const few_rsrc_t ab = few_buffer(p.A + (size_t)slab0 * BK, FEW_A_BYTES);
  if (GATHER) id = (uint32_t)id / (uint32_t)p.top_k;
  uint32_t a_off[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int r = (wave + WAVES * i) * PER + lane / PIECES;
    int src = __builtin_amdgcn_readlane(id, (wave + WAVES * i) * PER);
    if (PER == 2) src = lane < PIECES ? src : __builtin_amdgcn_readlane(id, (wave + WAVES * i) * PER + 1);
    a_off[i] = r < rows ? (uint32_t)src * (uint32_t)K * 2u : FEW_A_BYTES;
  }
  u32x4 areg[NA];
  auto load_a = [&](int c) {
    const int k = c * (CHUNK * BK) + lane % PIECES * 8;
#pragma unroll
    for (int i = 0; i < NA; i++)
      areg[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ab, k < nslab * BK ? a_off[i] + k * 2 : FEW_A_BYTES, 0, 0));
  };
  auto store_a = [&](int c) {
    bf16_t *d = lds + (c & 1) * (ROWS * ROW) + (wave * PER + lane / PIECES) * ROW + lane % PIECES * 8;
#pragma unroll
    for (int i = 0; i < NA; i++) *reinterpret_cast<u32x4 *>(d + WAVES * PER * i * ROW) = areg[i];
  };
  load_a(0);
  store_a(0);
  __syncthreads();

  f32x16 acc[RB];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int x = 0; x < 16; x++) acc[i][x] = 0.f;
  const bf16_t *a_src = lds + min(lane & 31, ROWS - 1) * ROW + (lane >> 5) * 8;
  // the operands of AHEAD k-steps are read while the AHEAD before them are multiplied: group G of them into set G & 1
  bf16x8 af[2][AHEAD][RB];
  auto read_a = [&](int c, auto gg) {
    constexpr int G = decltype(gg)::value;
#pragma unroll
    for (int x = 0; x < AHEAD; x++)
#pragma unroll
      for (int i = 0; i < RB; i++)
        af[G & 1][x][i] = as_bf16x8(*reinterpret_cast<const u32x4 *>(a_src + (c & 1) * (ROWS * ROW) + i * 32 * ROW +
                                                                     (G * AHEAD + x) % (CHUNK * 4) * 16));
  };
  read_a(0, std::integral_constant<int, 0>{});
  for (int s = 0; s < nslab; s += RING)
    static_for<0, RING>([&](auto rr) {
      constexpr int R = decltype(rr)::value;
      const int c = (s + R) / CHUNK;
      if constexpr (R % CHUNK == 0) load_a(c + 1);
      static_for<0, 4 / AHEAD>([&](auto hh) {
        constexpr int G = R * 4 / AHEAD + decltype(hh)::value;
        if constexpr ((G + 1) * AHEAD % (CHUNK * 4) != 0) read_a(c, std::integral_constant<int, G + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < AHEAD; x++) {
          constexpr int K0 = decltype(hh)::value * AHEAD;
          bf16x8 b;
          if constexpr (FP4) b = as_bf16x8(fp4_expand(w[R][0][K0 + x], fp4_scale((sc[R] >> (8 * ((K0 + x) >> 1))) & 0xffu)));
          else b = as_bf16x8(w[R][(K0 + x) % WQ]);
#pragma unroll
          for (int i = 0; i < RB; i++)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, af[G & 1][x][i], acc[i], 0, 0, 0);
        }
      });
      load_w(s + R + RING, rr);
      __builtin_amdgcn_sched_barrier(0);   // the order of the loads is the order of their uses
      if constexpr (R % CHUNK == CHUNK - 1) {
        store_a(c + 1);
        __syncthreads();
        read_a(c + 1, std::integral_constant<int, (R + 1) % RING * 4 / AHEAD>{});
      }
    });
  if (!live) return;
  auto bias_of = [&](int j) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(bias, j)); };
  if constexpr (EPI == EPI_PARTIAL) {
    GemmParams q = p;
    q.out = out;
    epilogue_rows<RB, EPI_F32>(q, row0, rows, cb * 32, lane, acc, bias_of);
  } else {
    epilogue_rows<RB, EPI>(p, row0, rows, cb * 32, lane, acc, bias_of);
  }
}

// Work items are (row tile, 32-column block) pairs; every XCD has a contiguous part of them, so that the row tiles of
// one expert, which multiply the same blocks of W one after the other, find them in that XCD's L2.
// ALONE: no expert has a second tile, so that the item's number says which tile it is, and what a workgroup has to know
// before its first load of W comes in one round trip to memory instead of three, one behind the other.  MoE blocks: one
// token 48.7 -> 47.9 us, four 123.2 -> 121.0, MXFP4 weights one 33.0 -> 32.4, twelve 86.0 -> 85.2.
template <int WAVES, int ROWS, bool GATHER, int EPI, bool FP4, bool ALONE>
__global__ __launch_bounds__(WAVES * 64, few_occupancy(WAVES, ROWS, FP4)) void few_gemm_kernel(GemmParams p) {
  constexpr int BM = ROWS <= 32 ? 32 : 64;   // rows of a dense problem's tile
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * ROWS * few_row(ROWS, FP4)];
  const const_as<int> tiles = constant_ptr(p.tiles);
  const int n_blk = (p.N / 32 + WAVES - 1) / WAVES;
  int part = 0, tile, cb, mat = 0, row0, rows;
  bool once;
  if constexpr (ALONE) {
    tile = blockIdx.y;   // the grid has a row for every tile that the list has room for
    cb = blockIdx.x;
    int n_tiles = tiles[0];
    mat = tiles[1 + 3 * tile];
    row0 = tiles[2 + 3 * tile];
    rows = tiles[3 + 3 * tile];
    once = true;
    // together, and with the arguments that W's address takes: the compiler would load them behind the branch
    asm volatile("" : "+s"(n_tiles), "+s"(mat), "+s"(row0), "+s"(rows) : "s"(p.W), "s"(p.N), "s"(p.K), "s"(p.A), "s"(p.row_ids));
    if (tile >= n_tiles) return;
  } else {
    const int n_tiles = p.tiles ? tiles[0] : (p.dense_rows + BM - 1) / BM;
    const int tile_items = n_tiles * n_blk;
    const int total = EPI == EPI_PARTIAL ? tile_items * p.k_splits : tile_items;
    const int chunk = (total + 7) >> 3;
    const int j = blockIdx.x >> 3;
    int work = (blockIdx.x & 7) * chunk + j;
    if (j >= chunk || work >= total) return;
    if (EPI == EPI_PARTIAL) {
      part = work / tile_items;
      work -= part * tile_items;
    }
    if (p.tiles) {
      if (p.xcd_bounds) {   // the tiles of an expert's block are walked column block by column block
        const int info = constant_ptr(p.xcd_bounds)[XCD_BOUNDS_INTS + work / n_blk];
        const int first = info >> 8, th = info & 255;
        const int v = work - first * n_blk;
        cb = v / th;
        tile = first + (v - cb * th);
        once = th == 1;
      } else {
        tile = work / n_blk;
        cb = work - tile * n_blk;
        once = false;
      }
      mat = tiles[1 + 3 * tile];
      row0 = tiles[2 + 3 * tile];
      rows = tiles[3 + 3 * tile];
    } else {
      cb = work / n_tiles;
      tile = work - cb * n_tiles;
      row0 = tile * BM;
      rows = min(BM, p.dense_rows - row0);
      once = n_tiles == 1;
    }
  }
  int slab0 = 0, nslab = p.K / BK;
  void *out = p.out;
  if (EPI == EPI_PARTIAL) {
    slab0 = part * p.split_slabs;
    nslab = min(p.split_slabs, nslab - slab0);
    out = reinterpret_cast<float *>(p.out) + (size_t)part * p.dense_rows * p.N;
  }
  // wave-uniform, and known to be: buffer resources live in scalar registers
  mat = __builtin_amdgcn_readfirstlane(mat);
  cb = __builtin_amdgcn_readfirstlane(cb * WAVES + (threadIdx.x >> 6));
  row0 = __builtin_amdgcn_readfirstlane(row0), rows = __builtin_amdgcn_readfirstlane(rows);
  slab0 = __builtin_amdgcn_readfirstlane(slab0), nslab = __builtin_amdgcn_readfirstlane(nslab);
  if (ALONE || once) few_block<WAVES, ROWS, GATHER, EPI, FP4, true>(p, lds, mat, row0, rows, cb, slab0, nslab, out);
  else few_block<WAVES, ROWS, GATHER, EPI, FP4, false>(p, lds, mat, row0, rows, cb, slab0, nslab, out);
}

template <int WAVES, int ROWS, bool GATHER, int EPI, bool FP4>
int launch_few_waves(const GemmParams &p, int max_tiles, hipStream_t s) {
  constexpr int BM = ROWS <= 32 ? 32 : 64;
  const long long total = (long long)max_tiles * cdiv(p.N / 32, WAVES) * (EPI == EPI_PARTIAL ? p.k_splits : 1);
  if (total == 0) return GPTOSS_OK;
  const unsigned grid = (unsigned)((total + 7) / 8) * 8;
  {
    TraceScope ts(FP4 ? (GATHER ? "gemm1_gather_swiglu_mxfp4" : "gemm_f32_mxfp4")
                      : (GATHER ? "gemm1_gather_swiglu" : "gemm_f32"), s);
    bool alone = false;
    if constexpr (EPI == EPI_SWIGLU || EPI == EPI_F32) {
      alone = p.tiles && p.max_tile_rows > 0 && p.max_tile_rows <= BM;
      if (alone) few_gemm_kernel<WAVES, ROWS, GATHER, EPI, FP4, true><<<dim3(cdiv(p.N / 32, WAVES), max_tiles), WAVES * 64, 0, s>>>(p);
    }
    if (!alone) few_gemm_kernel<WAVES, ROWS, GATHER, EPI, FP4, false><<<grid, WAVES * 64, 0, s>>>(p);
  }
  GPTOSS_LAUNCH_CHECK("few_gemm_kernel");
  return GPTOSS_OK;
}

template <bool GATHER, int EPI, bool FP4>
int launch_few_gemm(const GemmParams &p, int rows_per_tile, int max_tiles, hipStream_t s) {
  // few blocks: workgroups of four would leave most CUs without one (2880 x 5120, 32 rows: 20 us on 40 CUs, 11 on 160)
  const long long blocks = (long long)max_tiles * (p.N / 32) * (EPI == EPI_PARTIAL ? p.k_splits : 1);
  const bool solo = blocks <= FEW_SOLO_BLOCKS;
  if constexpr (!FP4)
    if (rows_per_tile == 64)
      return solo ? launch_few_waves<1, 64, GATHER, EPI, FP4>(p, max_tiles, s) : launch_few_waves<4, 64, GATHER, EPI, FP4>(p, max_tiles, s);
  if (p.max_tile_rows && p.max_tile_rows <= 8) return launch_few_waves<1, 8, GATHER, EPI, FP4>(p, max_tiles, s);
  return solo ? launch_few_waves<1, 32, GATHER, EPI, FP4>(p, max_tiles, s) : launch_few_waves<4, 32, GATHER, EPI, FP4>(p, max_tiles, s);
}

}  // namespace gptoss
