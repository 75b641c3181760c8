// The grouped GEMM on MXFP4 weights for tiles of more than a few rows (gfx950).
//
// With a quarter of bf16's bytes per weight the streaming kernel's form (gemm_kernel.hpp: a wave has 32 columns and every
// row of the tile) is bound by LDS: each matrix instruction takes a fresh fragment of A, 128 bytes a cycle for the four
// SIMDs, which is all that LDS gives.  Here a wave has 64 columns, so a fragment of A feeds two instructions, and a
// workgroup of four waves 256 columns x up to 64 rows.
//   A and W go from memory straight into LDS in stages of 64 k, W as codes and scales (a wave reads back its own only and
//   expands it in registers).  The loads are inline assembly: every wait for them is counted by hand.
//   Three or four workgroups share a CU: one's first loads, its waits behind a barrier and its epilogue lie behind the
//   others' matrix instructions.
// Operand roles, order over k and epilogues are those of the other kernels, so results are bit-identical to theirs.
//
// Measured against the streaming kernel with 64-row tiles (both products, 2880 x 2880, us): 128 experts, 4096 tokens
// 707 + 380 -> 595 + 327 (Zipf 1.1), 700 + 377 -> 576 + 314 (uniform), 850 tokens 275 + 151 -> 234 + 131; 32 experts, 4096
// tokens 586 + 317 -> 495 + 272, 500 tokens 118 + 77 -> 101 + 62.  4096 tokens on all of 4 experts (no tile with less than
// 64 rows) 637 + 361 -> 454 + 248: 1.2 PFLOP/s, matrix cores 67 and 57 % busy (775 and 456 thousand cycles), waves waiting 45 %
// of their cycles; what is left is waves that wait for each other at the barriers, and tiles and rounds that are not full.
// Not kept: tiles of 128 rows (two workgroups a CU, two waves per SIMD: 4096 tokens 964 -> 1036), 96 rows (1058), W straight
// into registers a stage ahead (955 -> 995: the registers of a wave more), a higher priority for the waves that multiply
// (within 1 %).
#pragma once
#include "gemm_tall_kernel.hpp"

namespace gptoss {

// Stages, all but one of them in flight, and the workgroups of a CU that they leave room for.
template <int STAGES_, int PER_CU_>
struct Fp4Tile {
  static constexpr int RB = 2, BM = RB * 32;           // row blocks of 32, rows
  static constexpr int THREADS = 256, CB = 2;          // four waves of two 32-column blocks
  static constexpr int STAGES = STAGES_, AHEAD = STAGES - 1, PER_CU = PER_CU_;
  // a stage: 128 bytes of every row, then 2 KB of codes and 256 bytes of scales per wave
  static constexpr int W_OFF = BM * 128, S_OFF = W_OFF + 4 * CB * 1024, STAGE = S_OFF + 4 * 256;
  static constexpr int SMEM = STAGES * STAGE;
  static_assert(SMEM * PER_CU <= 160 * 1024, "LDS of a CU");
};

// From so many work items on (an upper bound: every expert's last tile counts) four workgroups of two stages, below three of
// three: a launch of many rounds gains from the fourth one, one of few loses more in its last round, where CUs have less than
// four items left (first / second product, three / four: 8832 / 4608 items 605 / 339 -> 576 / 314 us, 6624 / 3456 520 / 288 ->
// 495 / 272, 2323 / 1212 183 / 102 -> 180 / 101, 1955 / 1020 126 / 70 -> 134 / 84).
constexpr int FP4_MANY_ITEMS = 3000;

// 4 bytes per lane to LDS, as tall_load
__device__ __forceinline__ void fp4_load_scales(unsigned lds, uint32_t voff, tall_rsrc_t base, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(base), "s"(soff)
               : "memory");
}

// A work item, and where this wave's share of its loads comes from.
template <class T>
struct Fp4Item {
  int mat, row0, rows, ct;
  tall_rsrc_t codes, scales;   // of the wave's first column block
  int second;                  // its second block's distance in blocks (0: there is none, the first again)
  uint32_t a[T::RB];           // byte offsets of this lane's piece of the A rows it loads (gather: pair ids until they are needed)
};

template <class T, bool GATHER, int EPI>
__global__ __launch_bounds__(256, T::PER_CU) void mxfp4_gemm_kernel(GemmParams p) {
  constexpr int RB = T::RB, CB = T::CB, STAGE = T::STAGE;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, nslab = K / BK;
  const unsigned lds_base =
      __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)lds);

  // ---- work list: that of grouped_gemm_kernel (gemm_kernel.hpp), grouped problems only ---------------
  const const_as<int> tiles = constant_ptr(p.tiles), bounds = constant_ptr(p.xcd_bounds);
  const int total = tiles[0] * p.n_col_tiles;
  const int per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7;
  int lo, hi;
  if (p.xcd_bounds) {
    auto item = [&](int b) { return (b >> 16) * p.n_col_tiles + (((b & 0xffff) * p.n_col_tiles) >> 16); };
    lo = item(bounds[xcd]);
    hi = item(bounds[xcd + 1]);
  } else {
    const int chunk = (total + 7) >> 3;
    lo = xcd * chunk;
    hi = min(total, lo + chunk);
  }
  int j = blockIdx.x >> 3;
  auto valid = [&](int jj) { return lo + jj < hi; };
  if (!valid(j)) return;

  const size_t code_bytes = (size_t)N * K / 2, mat_bytes = code_bytes + (size_t)N * K / 32;
  auto decode = [&](int jj, Fp4Item<T> &t) {
    const int work = lo + jj;
    int tile = work / p.n_col_tiles;
    t.ct = work - tile * p.n_col_tiles;
    if (p.tile_block > 1 && p.xcd_bounds) {
      const int info = bounds[XCD_BOUNDS_INTS + tile], first = info >> 8, th = info & 255;
      const int v = work - first * p.n_col_tiles;
      t.ct = v / th;
      tile = first + (v - t.ct * th);
    }
    t.ct = __builtin_amdgcn_readfirstlane(t.ct);
    t.mat = __builtin_amdgcn_readfirstlane(tiles[1 + 3 * tile]);
    t.row0 = __builtin_amdgcn_readfirstlane(tiles[2 + 3 * tile]);
    t.rows = __builtin_amdgcn_readfirstlane(tiles[3 + 3 * tile]);
    const int last = N / 32 - 1, block = min(t.ct * 8 + w * CB, last);   // (a wave beyond N repeats the last block)
    const unsigned char *m = reinterpret_cast<const unsigned char *>(p.W) + (size_t)t.mat * mat_bytes;
    t.codes = tall_buffer(m + (size_t)block * nslab * 1024);
    t.scales = tall_buffer(m + code_bytes + (size_t)block * nslab * 64);
    t.second = min(1, last - block);
    // load instruction q of the four waves moves rows q * 32 .. + 31 of the tile, rows past the last one repeat it
#pragma unroll
    for (int q = 0; q < RB; q++) {
      const int r = min((q * 4 + w) * 8 + (lane >> 3), t.rows - 1);
      t.a[q] = GATHER ? p.row_ids[t.row0 + r] : t.row0 + r;
    }
  };
  uint32_t inv_k = 0;
  if constexpr (GATHER) inv_k = pair_inverse(p.top_k);
  // the lane at piece p of row r fetches piece p ^ ((r >> 1) & 7): fragment reads are free of bank conflicts
  const uint32_t piece = (uint32_t)(((lane & 7) ^ ((w * 8 + (lane >> 3)) >> 1 & 7)) << 4);
  auto a_offsets = [&](Fp4Item<T> &t) {
#pragma unroll
    for (int q = 0; q < RB; q++) t.a[q] = (GATHER ? pair_token(t.a[q], inv_k) : t.a[q]) * (uint32_t)K * 2u + piece;
  };

  const tall_rsrc_t abuf = tall_buffer(p.A);
  // loads of slab s into `stage`: one per row block of the tile, two of codes, one of scales
  auto load_w = [&](const Fp4Item<T> &t, unsigned stage, int s) {
    const uint32_t voff = lane * 16, far = (uint32_t)(t.second * nslab);
    tall_load<0>(stage + T::W_OFF + w * (CB * 1024), voff, t.codes, (uint32_t)s * 1024u);
    tall_load<1024>(stage + T::W_OFF + w * (CB * 1024), voff, t.codes, (uint32_t)(s + far) * 1024u);
    // lanes 0-15 the first block's, 16-31 the second's, and both again
    fp4_load_scales(stage + T::S_OFF + w * 256, (lane & 15) * 4 + ((lane >> 4) & 1) * far * 64u, t.scales, (uint32_t)s * 64u);
  };
  auto load_first = [&](const Fp4Item<T> &t) {   // the first slabs of an item
    const int mb = (t.rows + 31) >> 5;
#pragma unroll
    for (int s = 0; s < T::AHEAD; s++) {
      if (s >= nslab) break;
      const unsigned stage = lds_base + s * STAGE;
      static_for<0, RB>([&](auto q) {
        constexpr int Q = decltype(q)::value;
        if (Q < mb) tall_load<Q * 4096>(stage + w * 1024, t.a[Q], abuf, s * 128);
      });
      load_w(t, stage, s);
    }
  };

  const int h = lane >> 5, sw = ((lane & 31) >> 1) & 7;
  const unsigned a_rd = (lane & 31) * 128, c_rd = T::W_OFF + w * (CB * 1024) + lane * 16, s_rd = T::S_OFF + w * 256 + (lane & 31) * 2;
  unsigned a_k[4];   // the lane's piece of k-step x
#pragma unroll
  for (int x = 0; x < 4; x++) a_k[x] = a_rd + (unsigned)(((2 * x + h) ^ sw) << 4);

  Fp4Item<T> cur, nxt;
  // One item with MB row blocks.
  auto run = [&](auto mb) {
    constexpr int MB = decltype(mb)::value;
    const bool live = (cur.ct * 8 + w * CB) * 32 < N;
    f32x16 acc[CB][MB];
#pragma unroll
    for (int i = 0; i < CB; i++)
#pragma unroll
      for (int r = 0; r < MB; r++)
#pragma unroll
        for (int x = 0; x < 16; x++) acc[i][r][x] = 0.f;
    unsigned at = 0, ahead = T::AHEAD * STAGE;   // stages of slab s and of slab s + AHEAD
    for (int s = 0; s < nslab; s++) {
      const bool more = s + T::AHEAD < nslab;
      if (more) {
        const unsigned stage = lds_base + ahead;
        static_for<0, MB>([&](auto q) {
          constexpr int Q = decltype(q)::value;
          tall_load<Q * 4096>(stage + w * 1024, cur.a[Q], abuf, (uint32_t)(s + T::AHEAD) * 128u);
        });
        load_w(cur, stage, s + T::AHEAD);
      }
      if (live) {
        const unsigned char *st = lds + at;
        u32x4 c[CB];
        float scale[CB][2];
#pragma unroll
        for (int i = 0; i < CB; i++) {
          c[i] = *reinterpret_cast<const u32x4 *>(st + c_rd + i * 1024);
          const uint32_t e = *reinterpret_cast<const unsigned short *>(st + s_rd + i * 64);
          scale[i][0] = fp4_scale(e & 0xffu);
          scale[i][1] = fp4_scale(e >> 8);
        }
        bf16x8 a[2][MB];
#pragma unroll
        for (int r = 0; r < MB; r++) a[0][r] = as_bf16x8(*reinterpret_cast<const u32x4 *>(st + a_k[0] + r * 4096));
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          if (kk < 3) {
#pragma unroll
            for (int r = 0; r < MB; r++)
              a[(kk + 1) & 1][r] = as_bf16x8(*reinterpret_cast<const u32x4 *>(st + a_k[kk < 3 ? kk + 1 : 0] + r * 4096));
          }
#pragma unroll
          for (int i = 0; i < CB; i++) {
            const bf16x8 b = as_bf16x8(fp4_expand(c[i][kk], scale[i][kk >> 1]));
#pragma unroll
            for (int r = 0; r < MB; r++) acc[i][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a[kk & 1][r], acc[i][r], 0, 0, 0);
          }
        }
      }
      // slab s + 1 has landed, the loads behind it may be on their way
      if (more) wait_vmcnt<(T::AHEAD - 1) * (MB + 3)>();
      else wait_vmcnt<0>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      at = at == T::AHEAD * STAGE ? 0 : at + STAGE;
      ahead = ahead == T::AHEAD * STAGE ? 0 : ahead + STAGE;
    }
    // every wave is past its last read: the next item's first slabs travel during the epilogue
    if (nxt.rows > 0) load_first(nxt);
#pragma unroll
    for (int i = 0; i < CB; i++) {
      const int n0 = (cur.ct * 8 + w * CB + i) * 32;
      if (n0 < N) epilogue_store<MB, EPI, true>(p, cur.mat, cur.row0, cur.rows, n0, lane, acc[i]);
    }
  };

  decode(j, cur);
  a_offsets(cur);
  load_first(cur);
  while (true) {
    const int jn = j + per_xcd;
    const bool more = valid(jn);
    nxt = cur;
    nxt.rows = 0;
    if (more) {
      decode(jn, nxt);
      a_offsets(nxt);
    }
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    const int mb = (cur.rows + 31) >> 5;
    bool done = false;
    static_for<1, RB + 1>([&](auto m) {
      if (!done && mb == decltype(m)::value) {
        run(m);
        done = true;
      }
    });
    if (!more) break;
    j = jn;
    cur = nxt;
  }
}

template <class T, bool GATHER, int EPI>
static int launch_mxfp4_tile(const GemmParams &p, long long items, hipStream_t s) {
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static bool raised[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "run_gemm: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  auto kern = mxfp4_gemm_kernel<T, GATHER, EPI>;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!raised[dev]) {
      GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM));
      raised[dev] = true;
    }
  }
  const int grid = (int)std::min<long long>((items + 7) / 8 * 8, 256 * T::PER_CU);
  if (grid == 0) return GPTOSS_OK;
  {
    TraceScope ts(GATHER ? "gemm1_gather_swiglu_mxfp4" : "gemm_f32_mxfp4", s);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(T::THREADS), T::SMEM, s, p);
  }
  GPTOSS_LAUNCH_CHECK("mxfp4_gemm_kernel");
  return GPTOSS_OK;
}

template <bool GATHER, int EPI>
static int launch_mxfp4(const GemmParams &p, int max_tiles, hipStream_t s) {
  const long long items = (long long)max_tiles * p.n_col_tiles;
  return items >= FP4_MANY_ITEMS ? launch_mxfp4_tile<Fp4Tile<2, 4>, GATHER, EPI>(p, items, s)
                                 : launch_mxfp4_tile<Fp4Tile<3, 3>, GATHER, EPI>(p, items, s);
}

}  // namespace gptoss
