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
// Measured, 2880 x 2880 experts, streaming kernels -> these (us): one token, both products 36 + 32 -> 24 + 14 (21 + 13 with what follows), MXFP4
// block 60 -> 43; 27 tokens 156 + 91 -> 157 + 81 (5.9-6.8 TB/s either way); MXFP4 block of 12 tokens 114 -> 87.
// Dense 5120 x 2880: one row 31 -> 9, 32 rows 33 -> 11, 64 rows 37 -> 16, 200 rows 32 -> 21.
//
// One wave per CU, as a small launch has it, is bound by what comes one behind the other: a chain of 32x32x16 matrix
// instructions on one accumulator takes 54 cycles for each, 220 for a slab, and a CU reads about 40 GB/s with 32 KB in
// flight however many other CUs are idle.  bf16 tiles of up to 16 rows, and some of 32 (few_narrow), are therefore
// multiplied by 16x16x32 instructions, several accumulators side by side, 35 cycles for the same 32 k of 32 columns; their
// sums have the same bits (k in the same order, eight at a time).  A lane's operand is then another 16 bytes of the packed
// slab, nothing is exchanged.  And launches that leave CUs idle give each half block of 16 columns a workgroup.
// Measured, 1 / 12 / 24 rows, before -> now (us): 2880 x 4096 9.6 / 12.9 / 13.1 -> 7.1 / 8.6 / 11.1, 2048 x 2048
// 5.7 / 8.1 / 8.3 -> 4.7 / 5.2 / 7.2, 5120 x 2880 7.8 / 10.8 / 10.9 -> 7.5 / 8.5 / 11.0, 16384 x 2048 13.0 / 15.0 / 15.3 ->
// 12.9 / 13.5 / 14.9; MoE block of 2880 x 2880, 1 / 4 / 12 / 30 tokens 46.3 / 118 / 217 / 253 -> 45.3 / 116 / 214 / 250.
// (A read straight from memory in operand order, without LDS: one token 60, but 12 tokens on MXFP4 127,
// because A is then four times the bytes of W.  One wave with 16 rows for MXFP4's small tiles: nine tokens 86.0 -> 87.6,
// twelve 87.8 -> 93.5.)
#pragma once
#include "gemm_kernel.hpp"
#include "moe_gating.hpp"

namespace gptoss {

// A workgroup: WAVES 32-column blocks, one per wave, times tiles of at most ROWS rows.
//   4 x 32, 4 x 64   the waves share the staged rows
//   4 x 16           the same for 9 to 16 rows, half the staging: MXFP4 block of 9 / 12 / 16 tokens 77.5 / 79.9 / 81.9 -> 73.6 /
//                    75.8 / 77.8 us, 128 experts 95.6 / 112 / 135 -> 89.2 / 105 / 126
//   1 x 8            one wave can stage so few rows by itself, and four times as many workgroups fill the chip: one
//                    token's block 68 -> 59 us, eight tokens' 178 -> 176
//   1 x 16, 1 x 32, 1 x 64   the same for launches of at most FEW_SOLO_BLOCKS blocks, on the registers of two waves
// COLS = 16 (1 x 8, 1 x 16, 1 x 32): half a block per workgroup.

// 64-k slabs of W that a wave keeps in flight: 32 KB of whole blocks, or of half ones where a staged chunk is small
// enough for a second one to be on its way too (2880 x 4096, one row 8.3 -> 7.1 us; whole blocks gain nothing from more:
// 9.5 -> 9.6)
constexpr int few_ring(int rows, int cols) { return rows <= 8 && cols == 16 ? 16 : 8; }
constexpr int few_chunk(int rows, bool fp4) { return rows <= 32 && !fp4 ? 8 : 4; }   // slabs of A that are staged together: one barrier each
constexpr int few_row(int rows, bool fp4) { return few_chunk(rows, fp4) * BK + 8; }   // padded row of a staged chunk in bf16 elements
constexpr int few_ahead(int rows) { return rows <= 32 ? 4 : 2; }       // k-steps whose operands are read from LDS ahead
// Waves per SIMD.  A single wave that stages 32 rows or more needs the registers of two.  MXFP4: expanding the codes takes
// as long as the products, and a third wave fills in for it (a slab of W is five registers); with two waves, sixteen slabs
// in flight and chunks of eight, 12 tokens took 95 us instead of 87, 600 on 128 experts 410 instead of 394.
constexpr int few_occupancy(int waves, int rows, bool fp4) { return waves == 1 && rows > 8 ? 1 : fp4 ? 3 : 2; }

// Products by 16x16x32 instructions.  Not for whole blocks of 32 rows on one wave: with four accumulators and twice the
// operand sets, 5120 x 2880 takes 11.7 instead of 10.9 us at 24 rows.  Not for MXFP4, whose codes have to be exchanged between
// lanes for it (four waves: 12 tokens 75.8 -> 76.9 us, 27 93.1 -> 96.6; one wave: one token 30.7 -> 33.7).
constexpr bool few_narrow(int waves, int rows, int cols, bool fp4) {
  return !fp4 && (rows <= 16 || cols == 16 || (waves == 4 && rows <= 32));
}
constexpr int FEW_CUS = 256;   // compute units

typedef __amdgpu_buffer_rsrc_t few_rsrc_t;
// cache policy of a buffer load: the non-temporal bit
constexpr int FEW_NT = 2;
// A's buffer: offsets from here on read as zeros
constexpr uint32_t FEW_A_BYTES = 0x80000000u;

__device__ __forceinline__ few_rsrc_t few_buffer(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// Epilogue of a block of at most 16 rows: lane l has row l % 16 and channels half * 16 + l / 16 * 4 + 0..3 of both halves.
// bias: of a lane's channels, or of its pairs (EPI_SWIGLU).  The arithmetic of epilogue_rows.
template <int NH, int EPI>
__device__ __forceinline__ void narrow_epilogue(const GemmParams &p, int row0, int rows, int n0, int lane, const f32x4 (&acc)[NH],
                                                const f32x4 (&bias)[NH], void *out) {
  const int row = lane & 15, c = lane >> 4 << 2;
  if (row >= rows) return;
  if constexpr (EPI == EPI_SWIGLU) {
    static_assert(NH == 2, "a pair's gate and up lie in the two halves");
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = glu(p.glu, acc[0][q] + bias[q >> 1][q * 2 & 3], acc[1][q] + bias[q >> 1][(q * 2 & 3) + 1]);
    *reinterpret_cast<u32x2 *>(reinterpret_cast<bf16_t *>(out) + (size_t)(row0 + row) * (p.N >> 1) + (n0 >> 1) + c) =
        u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  } else {
#pragma unroll
    for (int h = 0; h < NH; h++) {
      f32x4 v;
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = acc[h][q] + bias[h][q];
      bool done = false;
      if constexpr (EPI == EPI_MIXED) {
#pragma unroll
        for (int x = 0; x < 2; x++) {
          const GemmBf16Range &rg = p.range[x];
          if (!done && n0 >= rg.from && n0 < rg.to) {   // wave-uniform
#pragma unroll
            for (int q = 0; q < 4; q++)
              if (rg.relu_squared) {
                v[q] = fmaxf(v[q], 0.f);
                v[q] *= v[q];
              }
            *reinterpret_cast<u32x2 *>(rg.out + (size_t)(row0 + row) * rg.ld + (n0 - rg.from) + h * 16 + c) =
                u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            done = true;
          }
        }
      }
      if (!done) *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(out) + (size_t)(row0 + row) * p.N + n0 + h * 16 + c) = v;
    }
  }
}

template <int WAVES, int ROWS, int COLS, bool GATHER, int EPI, bool FP4, bool ONCE>
__device__ __forceinline__ void few_block(const GemmParams &p, bf16_t *lds, int mat, int row0, int rows, int cb, int slab0,
                                          int nslab, void *out, const int *row_ids = nullptr) {
  constexpr int RING = few_ring(ROWS, COLS);
  constexpr bool NARROW = few_narrow(WAVES, ROWS, COLS, FP4);
  constexpr int RB = NARROW ? (ROWS + 15) / 16 : (ROWS + 31) / 32, RBLK = NARROW ? 16 : 32, CHUNK = few_chunk(ROWS, FP4), ROW = few_row(ROWS, FP4);
  constexpr int KSTEPS = NARROW ? 2 : 4, AHEAD = NARROW ? 2 : few_ahead(ROWS);   // matrix instructions' k-steps in a slab
  constexpr int NH = NARROW ? COLS / 16 : 1;                                      // column halves of a narrow block
  constexpr int WQ = FP4 ? 1 : NARROW ? 2 * NH : 4;
  static_assert(COLS == 32 || (COLS == 16 && NARROW), "a wave has a block or a half of one");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, kslab = K / BK;
  const bool live = cb * COLS < N;   // the last workgroup of a row tile may have waves to spare

  const int blk = cb * COLS / 32;
  // W: the block's slabs lie one behind the other.  Slabs past the end are requested all the same (every load of the
  // loop is unconditional) and read as zeros without touching memory: they lie outside the buffer.  (The part of an
  // offset that is checked against the buffer's size is the one in the vector register, so the slab goes there.)
  const size_t mat_bytes = FP4 ? (size_t)N * K / 2 + (size_t)N * K / 32 : (size_t)N * K * 2;
  const char *mb = reinterpret_cast<const char *>(p.W) + (size_t)mat * mat_bytes;
  constexpr int SLAB = FP4 ? 1024 : 4096;
  const few_rsrc_t wb = few_buffer(mb + ((size_t)blk * kslab + slab0) * SLAB, live ? nslab * SLAB : 0);
  const few_rsrc_t sb = few_buffer(FP4 ? mb + (size_t)N * K / 2 + ((size_t)blk * kslab + slab0) * 64 : mb,   // MXFP4 scales
                                   FP4 && live ? nslab * 64 : 0);
  u32x4 w[RING][WQ];
  uint32_t sc[RING];
  // a lane's first 16 bytes of a slab, and how far apart they are: narrow, fragment q & 1 of a k-step is its column half
  const int group = lane >> 4;
  const uint32_t w_lane = NARROW ? (group >> 1) * 1024 + (group & 1) * 512 + (lane & 15) * 16 + (COLS == 16 ? (cb & 1) * 256 : 0) : lane * 16;
  auto w_at = [](int q) { return NARROW ? q / NH * 2048 + q % NH * 256 : q * 1024; };
  auto load_w = [&](int s, auto r) {
    constexpr int R = decltype(r)::value;
#pragma unroll
    for (int q = 0; q < WQ; q++)
      w[R][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, w_lane + s * SLAB + w_at(q), 0, ONCE ? FEW_NT : 0));
    if constexpr (FP4) sc[R] = __builtin_amdgcn_raw_buffer_load_b16(sb, (lane & 31) * 2 + s * 64, 0, ONCE ? FEW_NT : 0);
  };
  // which rows of A the tile's rows are: before W, because loads return in order
  int id = row0 + min(lane, rows - 1);
  if (GATHER) id = row_ids ? row_ids[id] : p.row_ids[id];
  static_for<0, RING>([&](auto r) { load_w(decltype(r)::value, r); });
  const few_rsrc_t bb = few_buffer(p.bias && live ? p.bias + (size_t)mat * N + cb * COLS : nullptr, p.bias && live ? COLS * 4 : 0);
  int bias = 0;
  f32x4 bias4[NH];
  if constexpr (NARROW) {
#pragma unroll
    for (int h = 0; h < NH; h++)
      bias4[h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(bb, EPI == EPI_SWIGLU ? group * 32 + h * 16 : group * 16 + h * 64, 0, 0));
  } else {
    bias = __builtin_amdgcn_raw_buffer_load_b32(bb, (lane & 31) * 4, 0, 0);
  }

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
  constexpr int SETS = RING / 8;   // chunks of A that are requested ahead, each into a register set of its own
  u32x4 areg[SETS][NA];
  auto load_a = [&](int c, auto set) {
    const int k = c * (CHUNK * BK) + lane % PIECES * 8;
#pragma unroll
    for (int i = 0; i < NA; i++)
      areg[decltype(set)::value][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ab, k < nslab * BK ? a_off[i] + k * 2 : FEW_A_BYTES, 0, 0));
  };
  auto store_a = [&](int c, auto set) {
    bf16_t *d = lds + (c & 1) * (ROWS * ROW) + (wave * PER + lane / PIECES) * ROW + lane % PIECES * 8;
#pragma unroll
    for (int i = 0; i < NA; i++) *reinterpret_cast<u32x4 *>(d + WAVES * PER * i * ROW) = areg[decltype(set)::value][i];
  };
  static_assert(RING % (CHUNK * SETS) == 0, "the set of a chunk is known where it is used");
  static_for<0, SETS>([&](auto set) { load_a(decltype(set)::value, set); });
  store_a(0, std::integral_constant<int, 0>{});
  __syncthreads();

  f32x16 acc[RB];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int x = 0; x < 16; x++) acc[i][x] = 0.f;
  f32x4 acc4[RB][NH];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int h = 0; h < NH; h++) acc4[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16_t *a_src = NARROW ? lds + min(lane & 15, ROWS - 1) * ROW + group * 8
                               : lds + min(lane & 31, ROWS - 1) * ROW + (lane >> 5) * 8;
  // the operands of AHEAD k-steps are read while the AHEAD before them are multiplied: group G of them into set G & 1
  bf16x8 af[2][AHEAD][RB];
  auto read_a = [&](int c, auto gg) {
    constexpr int G = decltype(gg)::value;
#pragma unroll
    for (int x = 0; x < AHEAD; x++)
#pragma unroll
      for (int i = 0; i < RB; i++)
        af[G & 1][x][i] = as_bf16x8(*reinterpret_cast<const u32x4 *>(a_src + (c & 1) * (ROWS * ROW) + i * RBLK * ROW +
                                                                     (G * AHEAD + x) % (CHUNK * KSTEPS) * (BK / KSTEPS)));
  };
  read_a(0, std::integral_constant<int, 0>{});
  for (int s = 0; s < nslab; s += RING)
    static_for<0, RING>([&](auto rr) {
      constexpr int R = decltype(rr)::value;
      const int c = (s + R) / CHUNK;
      if constexpr (R % CHUNK == 0) load_a(c + SETS, std::integral_constant<int, R / CHUNK % SETS>{});
      static_for<0, KSTEPS / AHEAD>([&](auto hh) {
        constexpr int G = R * KSTEPS / AHEAD + decltype(hh)::value;
        if constexpr ((G + 1) * AHEAD % (CHUNK * KSTEPS) != 0) read_a(c, std::integral_constant<int, G + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < AHEAD; x++) {
          constexpr int K0 = decltype(hh)::value * AHEAD;
          if constexpr (NARROW) {
#pragma unroll
            for (int h = 0; h < NH; h++)
#pragma unroll
              for (int i = 0; i < RB; i++)
                acc4[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[R][((K0 + x) * NH + h) % WQ]), af[G & 1][x][i], acc4[i][h], 0, 0, 0);
            continue;
          }
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
        store_a(c + 1, std::integral_constant<int, (R / CHUNK + 1) % SETS>{});
        __syncthreads();
        read_a(c + 1, std::integral_constant<int, (R + 1) % RING * KSTEPS / AHEAD>{});
      }
    });
  if (!live) return;
  if constexpr (NARROW) {
#pragma unroll
    for (int i = 0; i < RB; i++) narrow_epilogue<NH, EPI>(p, row0 + i * 16, rows - i * 16, cb * COLS, lane, acc4[i], bias4, out);
    return;
  }
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
template <int WAVES, int ROWS, int COLS, bool GATHER, int EPI, bool FP4, bool ALONE>
__global__ __launch_bounds__(WAVES * 64, few_occupancy(WAVES, ROWS, FP4)) void few_gemm_kernel(GemmParams p) {
  constexpr int BM = ROWS <= 32 ? 32 : 64;   // rows of a dense problem's tile
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * ROWS * few_row(ROWS, FP4)];
  const const_as<int> tiles = constant_ptr(p.tiles);
  const int n_blk = (p.N / COLS + WAVES - 1) / WAVES;
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
  if (ALONE || once) few_block<WAVES, ROWS, COLS, GATHER, EPI, FP4, true>(p, lds, mat, row0, rows, cb, slab0, nslab, out);
  else few_block<WAVES, ROWS, COLS, GATHER, EPI, FP4, false>(p, lds, mat, row0, rows, cb, slab0, nslab, out);
}

// The first product of up to ROUTED_TOKENS tokens, whose workgroups gate and group them from the router's partial products, each
// for itself: a chain of 2 us in front of a product of 19 (one token, 4 of 32 experts, 2880 x 5760, between events 22.9 -> 24.8 us,
// MXFP4 12.4 -> 15.0), in place of a launch, whose workgroup everybody waited for, with that chain and 3 us more.  The grid's
// first row of workgroups has no tile: one leaves the routing's results, and what the kernels behind this one read, the others
// add a norm's residual to x.
template <int NJ, bool FP4>   // experts per lane
__global__ __launch_bounds__(64, few_occupancy(1, 8, FP4)) void few_routed_kernel(GemmParams p, RoutedFew r) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * 8 * few_row(8, FP4)];
  __shared__ float weight[ROUTED_TOKENS * 8];
  __shared__ int expert[ROUTED_TOKENS * 8], sorted[ROUTED_TOKENS * 8];
  const int lane = threadIdx.x, sub = lane & 31, E = r.router.E, k = r.router.k, B = r.router.B, P = B * k;
  const bool publish = blockIdx.y == 0;
  if (publish && blockIdx.x != 0) {
    if (r.residual)
      for (int i = ((blockIdx.x - 1) * 64 + lane) * 4; i < r.x_count; i += (gridDim.x - 1) * 64 * 4) {
        f32x4 v = *reinterpret_cast<const f32x4 *>(r.x + i);
        const f32x4 d = *reinterpret_cast<const f32x4 *>(r.residual + i);
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = __fadd_rn(v[q], d[q]);
        *reinterpret_cast<f32x4 *>(r.x + i) = v;
      }
    return;
  }
  // two tokens at a time
  constexpr int PASSES = ROUTED_TOKENS / 2;
  PartialLogit x[PASSES][NJ];
#pragma unroll
  for (int i = 0; i < PASSES; i++)
    if (2 * i < B)
#pragma unroll
      for (int j = 0; j < NJ; j++) x[i][j].load(r.router, 2 * i + (lane >> 5), sub + 32 * j);
#pragma unroll
  for (int i = 0; i < PASSES; i++)
    if (2 * i < B) {
      const int row = 2 * i + (lane >> 5);
      float v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const int e = sub + 32 * j;
        v[j] = e < E ? x[i][j].sum(r.router) : -INFINITY;
        if (publish && row < B && e < E) r.logits[(size_t)row * E + e] = v[j];
      }
      const int o = row < B ? row * k : 0;
      topk_softmax_group<NJ>(v, sub, E, k, row < B, weight + o, expert + o);
    }
  __syncthreads();
  // a pair per lane: pairs of lower experts, earlier ones and all of its own
  const int e = lane < P ? expert[lane] : 0x7fffffff;
  int lower = 0, before = 0, same = 0;
  for (int q = 0; q < P; q++) {
    const int other = __builtin_amdgcn_readlane(e, q);
    lower += other < e ? 1 : 0;
    same += other == e ? 1 : 0;
    before += other == e && q < lane ? 1 : 0;
  }
  const uint64_t firsts = __ballot(lane < P && before == 0);
  const int n_tiles = __popcll(firsts);
  int mine = 0;   // the pair's tile: experts before its own
  for (uint64_t f = firsts; f != 0; f &= f - 1) mine += __builtin_amdgcn_readlane(e, __builtin_ctzll(f)) < e ? 1 : 0;
  if (publish) {
    const RouterGroup &g = r.group;
    if (lane < P) {
      r.topk_w[lane] = weight[lane];
      r.topk_i[lane] = e;
      g.sorted_pair_ids[lower + before] = lane;
      g.inv_perm[lane] = lower + before;
      if (before == 0) {
        int *tp = g.tiles + 1 + 3 * mine;
        tp[0] = e;
        tp[1] = lower;
        tp[2] = same;
        g.xcd_bounds[XCD_BOUNDS_INTS + mine] = (mine << 8) | 1;
      }
    }
    if (lane < 9) g.xcd_bounds[lane] = (lane * n_tiles) << 13;   // eight parts of equal length, as group_by_one_wave
    if (lane == 0) g.tiles[0] = n_tiles;
    for (int x = lane; x <= E; x += 64) {
      int n = 0;
      for (int q = 0; q < P; q++) n += expert[q] < x ? 1 : 0;
      g.expert_offsets[x] = n;
    }
    return;
  }
  const int tile = blockIdx.y - 1;
  if (tile >= n_tiles) return;
  const uint64_t of_tile = __ballot(lane < P && mine == tile);
  const int one = __builtin_ctzll(of_tile);
  const int mat = __builtin_amdgcn_readlane(e, one), row0 = __builtin_amdgcn_readlane(lower, one), rows = __popcll(of_tile);
  if (lane < P) sorted[lower + before] = lane;
  __syncthreads();
  few_block<1, 8, 32, true, EPI_SWIGLU, FP4, true>(p, lds, mat, row0, rows, blockIdx.x, 0, p.K / BK, p.out, sorted);
}

template <bool FP4>
int launch_few_routed(const GemmParams &p, int max_tiles, hipStream_t s) {
  const RoutedFew &r = *p.routed;
  GPTOSS_REQUIRE(r.router.B >= 1 && r.router.B <= ROUTED_TOKENS && r.router.k <= 8 && r.router.E <= ROUTED_EXPERTS && p.N % 32 == 0 && p.N >= 64, GPTOSS_ERR_DIM,
                 "run_gemm: %d tokens over %d experts are not routed here", r.router.B, r.router.E);
  {
    TraceScope ts(FP4 ? "gemm1_gather_swiglu_mxfp4" : "gemm1_gather_swiglu", s);
    const dim3 grid(p.N / 32, max_tiles + 1);
    if (r.router.E <= 32) few_routed_kernel<1, FP4><<<grid, 64, 0, s>>>(p, r);
    else few_routed_kernel<4, FP4><<<grid, 64, 0, s>>>(p, r);
  }
  GPTOSS_LAUNCH_CHECK("few_routed_kernel");
  return GPTOSS_OK;
}

template <int WAVES, int ROWS, int COLS, bool GATHER, int EPI, bool FP4>
int launch_few_waves(const GemmParams &p, int max_tiles, hipStream_t s) {
  constexpr int BM = ROWS <= 32 ? 32 : 64;
  const long long total = (long long)max_tiles * cdiv(p.N / COLS, WAVES) * (EPI == EPI_PARTIAL ? p.k_splits : 1);
  if (total == 0) return GPTOSS_OK;
  const unsigned grid = (unsigned)((total + 7) / 8) * 8;
  {
    TraceScope ts(FP4 ? (GATHER ? "gemm1_gather_swiglu_mxfp4" : "gemm_f32_mxfp4")
                      : (GATHER ? "gemm1_gather_swiglu" : "gemm_f32"), s);
    bool alone = false;
    if constexpr (EPI == EPI_SWIGLU || EPI == EPI_F32) {
      alone = p.tiles && p.max_tile_rows > 0 && p.max_tile_rows <= BM;
      if (alone) few_gemm_kernel<WAVES, ROWS, COLS, GATHER, EPI, FP4, true><<<dim3(cdiv(p.N / COLS, WAVES), max_tiles), WAVES * 64, 0, s>>>(p);
    }
    if (!alone) few_gemm_kernel<WAVES, ROWS, COLS, GATHER, EPI, FP4, false><<<grid, WAVES * 64, 0, s>>>(p);
  }
  GPTOSS_LAUNCH_CHECK("few_gemm_kernel");
  return GPTOSS_OK;
}

template <bool GATHER, int EPI, bool FP4>
int launch_few_gemm(const GemmParams &p, int rows_per_tile, int max_tiles, hipStream_t s) {
  if constexpr (GATHER && EPI == EPI_SWIGLU)
    if (p.routed) return launch_few_routed<FP4>(p, max_tiles, s);
  // few blocks: workgroups of four would leave most CUs without one (2880 x 5120, 32 rows: 20 us on 40 CUs, 11 on 160)
  const long long blocks = (long long)max_tiles * (p.N / 32) * (EPI == EPI_PARTIAL ? p.k_splits : 1);
  const bool solo = blocks <= FEW_SOLO_BLOCKS;
  if constexpr (!FP4)
    if (rows_per_tile == 64)
      return solo ? launch_few_waves<1, 64, 32, GATHER, EPI, FP4>(p, max_tiles, s) : launch_few_waves<4, 64, 32, GATHER, EPI, FP4>(p, max_tiles, s);
  const int rows = p.max_tile_rows ? p.max_tile_rows : 32;
  if constexpr (!FP4) {
    // Half blocks where they are fewer rounds on the CUs than whole ones of twice the time: 90 blocks one half round instead
    // of one, 360 three halves instead of two, 160 or 256 no fewer (5120 x 2880, one row 7.5 us whole, 7.7 in halves).  From
    // 17 rows on staging A takes longer than a half block's W, and only CUs that would be idle gain: 320 blocks of two
    // tiles 14.4 us whole, 20.3 in halves.  A gated pair has its columns in both halves.
    if constexpr (EPI != EPI_SWIGLU)
      if (solo && (rows > 16 ? blocks <= FEW_CUS / 2 : (blocks - 1) % FEW_CUS < FEW_CUS / 2)) {
        if (rows <= 8) return launch_few_waves<1, 8, 16, GATHER, EPI, FP4>(p, max_tiles, s);
        if (rows <= 16) return launch_few_waves<1, 16, 16, GATHER, EPI, FP4>(p, max_tiles, s);
        return launch_few_waves<1, 32, 16, GATHER, EPI, FP4>(p, max_tiles, s);
      }
    if (rows > 8 && rows <= 16)
      return solo ? launch_few_waves<1, 16, 32, GATHER, EPI, FP4>(p, max_tiles, s) : launch_few_waves<4, 16, 32, GATHER, EPI, FP4>(p, max_tiles, s);
  }
  if (FP4 && rows > 8 && rows <= 16 && !solo) return launch_few_waves<4, 16, 32, GATHER, EPI, FP4>(p, max_tiles, s);
  if (rows <= 8) return launch_few_waves<1, 8, 32, GATHER, EPI, FP4>(p, max_tiles, s);
  return solo ? launch_few_waves<1, 32, 32, GATHER, EPI, FP4>(p, max_tiles, s) : launch_few_waves<4, 32, 32, GATHER, EPI, FP4>(p, max_tiles, s);
}

}  // namespace gptoss
