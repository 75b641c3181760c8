// The grouped / dense bf16 GEMM for MANY rows (prompt passes: thousands of rows, ~1000 per expert),
// where the launch is bound by the matrix cores and not by streaming W.
//
// gemm_kernel.hpp feeds every MFMA one fresh LDS fragment (a wave owns 32 columns and all rows of
// the tile), which caps it at ~70 % of the MFMA rate before anything else is counted.  Here a
// workgroup of four waves (one per SIMD) owns a 256 x 256 tile and a wave a 128 x 128 quarter of
// it: 4 W fragments and 4 A fragments per k-step feed 16 MFMAs, half a fragment per MFMA.  Both
// operands go from global memory straight into LDS with buffer_load_dwordx4 .. lds (no staging
// registers, no LDS store instructions), and the load pipeline runs on from one work item into
// the next.
//   W: stages of 32 k in four buffers, three in flight, in the same packed fragment order as
//      everywhere else (a fragment lands in LDS as it is read).
//   A: chunks of 64 k in three buffers, two in flight: a load instruction moves 8 rows x 128 bytes,
//      whole cache lines.  (Rows of 64 bytes, one 32-k stage at a time, fetch every line twice, once per half:
//      the loads of A then cost 2-3 times those of W, 55-65 us of a 265 us launch.)  The eight
//      16-byte pieces of a row are XOR-swizzled by (row >> 1) & 7, so fragment reads are free of
//      bank conflicts; the token gather of GEMM1 is a per-lane row offset of the load.
// The loads are inline assembly, invisible to the compiler's wait counting, and the loop has no
// other vector memory operation: every s_waitcnt vmcnt(N) is counted by hand (N = loads issued
// behind the one waited for; stores of the previous item's epilogue that are still in flight only
// make a wait stricter).
// Same operand roles (W fragment first: lane = token row, registers = channels), same k order and
// the same epilogue code as gemm_kernel.hpp, so the results are bit-identical to it.  Three forms:
// gather + SwiGLU (GEMM1 of a prompt pass), plain fp32 output (GEMM2, the projections), and the row
// arg-max of the classifier, which writes no products at all and is the fastest of the three.
//
// A tile costs what its rows are worth: its row blocks go to the two wave rows in turn, and the loop has a form for 1, 2, 3 and
// 4 blocks of a wave.  One block takes about 0.55 of a full tile (fragment reads and the same loads), two 0.6, three 0.75.  And
// where an XCD's last round of work items leaves half of its workgroups idle, its items are cut into halves of their rows.
// Before -> now (us): 2880 x 4096, 2048 rows (12 tiles per XCD for 32 workgroups) 77 -> 57, 2048 x 10240 164 -> 111, 5120 x
// 2880, 3100 rows 129 -> 112, 8000 (2.5 rounds) 211 -> 199; 16640 x 2048, 8000 rows (8.1) 485 -> 469; 8192 x 2048 (whole rounds)
// 227 -> 228; MoE block of 4500 tokens 1104 -> 1020, 5000 1129 -> 1070, 5999 1268 -> 1252, 4096 and 5000 under Zipf 1.1
// 1003 -> 922 and 1173 -> 1109.  (Idle CUs at the end of a launch leave the others power, so a round saved is worth less than
// its share.)
// gemm_tall.hip instantiates the forms without the gather, gemm_tall_grouped.hip the one with it.
#pragma once
#include <algorithm>
#include <mutex>

#include "gemm_kernel.hpp"

namespace gptoss {

constexpr int TALL_THREADS = 256;
constexpr int TALL_BK = 32;   // k of a W stage; an A chunk is two of them

// A workgroup is WR x WC waves (four in all), a wave RB x CB blocks of 32 x 32 outputs.
template <int WR_, int WC_, int RB_, int CB_>
struct TallShape {
  static_assert(WR_ * WC_ == 4, "four waves, one per SIMD");
  static constexpr int WR = WR_, WC = WC_, RB = RB_, CB = CB_;
  static constexpr int BM = WR * RB * 32, BN = WC * CB * 32;
  static constexpr int NSTW = 4;                        // W stage buffers, NSTW - 1 in flight
  static constexpr int W_BYTES = WC * CB * 2048;        // a W stage: a column block's two k-steps are 2 KB
  static constexpr int A_BYTES = BM * 128;              // an A chunk: 128 bytes of every row
  static constexpr int A_OFF = NSTW * W_BYTES;          // three A chunk buffers behind the W stages
  static constexpr int SMEM = A_OFF + 3 * A_BYTES;      // 160 KB for the 256 x 256 tile: all of a CU's LDS
  static constexpr int LW = WC * CB * 2 / 4;            // load instructions per wave: W fragments of a stage,
  static constexpr int LA = BM / 8 / 4;                 // 8-row pieces of an A chunk
  static_assert(WC * CB * 2 % 4 == 0 && BM % 32 == 0, "the loads are shared out evenly");
  static_assert(SMEM <= 160 * 1024, "LDS of a CU");
  static constexpr int NM = RB * CB, NR = RB + CB;      // MFMAs and fragment reads of a k-step
  static_assert(LW % 2 == 0 && LA % 4 == 0, "a k-step issues half a W stage and a quarter of an A chunk");
  static_assert(NM >= NR + 2 * (LA / 4 + LW / 2), "room for a k-step's reads and loads between its MFMAs");
  static constexpr int STEP = WR * 32;                  // rows from one of a wave's blocks to the next: the waves take them in turn
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
typedef uint32_t tall_rsrc_t __attribute__((ext_vector_type(4)));   // a buffer resource in scalar registers
__device__ __forceinline__ tall_rsrc_t tall_buffer(const void *base) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  return tall_rsrc_t{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v),
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32) & 0xffffu), 0xffffffffu, 0x00020000u};
}

// 16 bytes per lane, from the buffer's base + voff + soff to LDS address lds + ADD + 16 * lane: load_to_lds (common.hpp) in
// three instructions.  With one wave per SIMD an instruction takes four cycles of which only those in the shadow of a
// matrix instruction are free, seven instructions or so: an address of 64 bits per load, added up in scalar registers,
// made the ten instructions of a load outlast it.  A tile of K = 2880 takes 110 thousand cycles instead of 120 (its matrix
// instructions alone 92), and the chip, at its power limit, runs them at 1.65 GHz instead of 1.75: block of 5999 tokens
// 1344 -> 1311 us, of 4500 1152 -> 1120.
template <int ADD>
__device__ __forceinline__ void tall_load(unsigned lds, uint32_t voff, tall_rsrc_t base, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(base),
               "s"(soff), "n"(ADD)
               : "memory", "scc");
}

// The token of a pair: id / top_k by a multiplication.  inv = 2^32 / k rounded up (k = 1: 0) is off by e / k with e = inv k -
// 2^32 < k, which adds id e / (k 2^32) to the quotient: less than the 1 / k that can be missing to the next whole number while
// id e < 2^32.  A call has fewer than 2^31 / 64 pairs (a row has at least 64 elements) and k <= MOE_MAX_TOP.
__host__ __device__ constexpr uint32_t pair_inverse(uint32_t k) { return 0xffffffffu / k + 1u; }
__host__ __device__ constexpr uint32_t pair_token(uint32_t id, uint32_t inv) { return inv ? (uint32_t)((uint64_t)id * inv >> 32) : id; }
constexpr bool pair_tokens_exact() {
  constexpr uint64_t pairs = (1ull << 31) / 64;
  for (uint32_t k = 1; k <= MOE_MAX_TOP; k++) {
    const uint32_t inv = pair_inverse(k);
    if (k > 1 && (pairs - 1) * ((uint64_t)inv * k - (1ull << 32)) >= 1ull << 32) return false;
    for (uint64_t id = k; id < pairs; id *= 2) {
      const uint32_t m = (uint32_t)(id / k * k);
      if (pair_token(m, inv) != m / k || pair_token(m - 1, inv) != (m - 1) / k || pair_token(m + k - 1, inv) != m / k) return false;
    }
  }
  return true;
}
static_assert(pair_tokens_exact(), "a pair's token by multiplication");

// where one work item's operands come from, for this wave's share of the loads
template <class SH>
struct TallSrc {
  static constexpr int WB = SH::LW / 2;   // column blocks: both k-steps of a stage of each
  tall_rsrc_t w;       // the tile's first column block
  uint32_t wo[WB];     // byte offsets of the wave's column blocks from there
  uint32_t a[SH::LA];  // byte offsets of this lane's piece of the A rows it loads
  int mat, row0, rows, ct;
};

// Epilogue of a wave's CB x RB blocks.  A lane holds one row and four consecutive columns per register quad, so stored
// from where they lie an instruction's 64 pieces of 16 bytes go to 32 rows, and with a row of a multiple of 4 KB (8192
// or 16384 columns) to one and the same memory channel.  fp32 and bf16 columns go through LDS instead, 32 rows of a
// column block at a time, and leave in whole lines: 8000 x 8192 x 2048 262 -> 236 us, 8192 x 16384 x 2048 678 -> 490,
// 8192 x 5120 x 2880 235 -> 222.  (Not the gated form: rows of a quarter of the bytes, and its biases read once per row
// block instead of once cost more than the stores gain: block of 5999 tokens 1318 -> 1403 us.)
// buf: 8 KB of the A buffer that the next item's first stage fills again.  It is the part that this wave's own loads go
// to, and they are issued after its reads here; the other waves read it after a barrier.  Pieces of 16 bytes are
// XOR-swizzled by their row.
template <class SH, int EPI>
__device__ __forceinline__ void tall_epilogue(const GemmParams &p, unsigned char *buf, int mat, int row0, int rows, int c0,
                                              int lane, f32x16 (&acc)[SH::CB][SH::RB]) {
  constexpr int RB = SH::RB, CB = SH::CB;
  static_assert(SH::LA * 1024 >= 32 * 128, "32 rows of a column block in fp32");
  const int N = p.N, tok = lane & 31, h = lane >> 5;
  const const_as<float> bp = constant_ptr(p.bias ? p.bias + (size_t)mat * N + c0 : nullptr);
  // a row of the staged block is P pieces of 16 bytes
  auto put = [&](auto pieces, int piece, auto v) {
    constexpr int P = decltype(pieces)::value;
    unsigned char *d = buf + tok * (P * 16) + ((piece ^ (tok & (P - 1))) << 4);
    if constexpr (sizeof(v) == 8) d += h * 8;   // two lanes share a piece
    *reinterpret_cast<decltype(v) *>(d) = v;
  };
  // rows of the wave's block r: `width` 16-byte pieces of them are real, out = first byte of the first row
  auto flush = [&](auto pieces, int r, int width, unsigned char *out, size_t ld) {
    constexpr int P = decltype(pieces)::value, PER = 64 / P;   // rows of a store instruction
#pragma unroll
    for (int i = 0; i < 32 / PER; i++) {
      const int row = i * PER + lane / P, piece = lane % P;
      const u32x4 v = *reinterpret_cast<const u32x4 *>(buf + row * (P * 16) + ((piece ^ (row & (P - 1))) << 4));
      if (r * SH::STEP + row < rows && piece < width) *reinterpret_cast<u32x4 *>(out + (size_t)(r * SH::STEP + row) * ld + piece * 16) = v;
    }
  };
  // the compiler copies accumulators out of their AGPRs early, and spills, unless they are pinned until they are used
  auto pin = [&](int i, int r) { asm volatile("" : "+a"(acc[i][r])); };
  using P8 = std::integral_constant<int, 8>;
  using P4 = std::integral_constant<int, 4>;
  if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
    for (int i = 0; i < CB; i++) {
#pragma unroll
      for (int r = 0; r < RB; r++) pin(i, r);
      if (c0 + i * 32 < N) epilogue_store<RB, EPI, true, SH::STEP>(p, mat, row0, rows, c0 + i * 32, lane, acc[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < CB; i++) {
      const int n0 = c0 + i * 32;
#pragma unroll
      for (int r = 0; r < RB; r++) pin(i, r);
      if (n0 < N) {
        float bv[16];
#pragma unroll
        for (int x = 0; x < 16; x++) {
          const int c = i * 32 + (x >> 2) * 8 + (x & 3);
          const float lo = bp ? bp[c] : 0.f, hi = bp ? bp[c + 4] : 0.f;
          bv[x] = h ? hi : lo;
        }
        bool half = false;
        GemmBf16Range to;
        if constexpr (EPI == EPI_MIXED) {
          const bool in0 = n0 >= p.range[0].from && n0 < p.range[0].to, in1 = n0 >= p.range[1].from && n0 < p.range[1].to;
          half = in0 || in1;
          to.from = in1 ? p.range[1].from : p.range[0].from;
          to.out = in1 ? p.range[1].out : p.range[0].out;
          to.ld = in1 ? p.range[1].ld : p.range[0].ld;
          to.relu_squared = in1 ? p.range[1].relu_squared : p.range[0].relu_squared;
        }
        if (EPI == EPI_MIXED && half) {
#pragma unroll
          for (int r = 0; r < RB; r++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
              float v[4];
#pragma unroll
              for (int q = 0; q < 4; q++) {
                v[q] = acc[i][r][g * 4 + q] + bv[g * 4 + q];
                if (to.relu_squared) {
                  v[q] = fmaxf(v[q], 0.f);
                  v[q] *= v[q];
                }
              }
              put(P4{}, g, u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])});
            }
            flush(P4{}, r, 4, reinterpret_cast<unsigned char *>(to.out + (size_t)row0 * to.ld + (n0 - to.from)), (size_t)to.ld * 2);
          }
        } else {
#pragma unroll
          for (int r = 0; r < RB; r++) {
#pragma unroll
            for (int g = 0; g < 4; g++)
              put(P8{}, g * 2 + h, f32x4{acc[i][r][g * 4] + bv[g * 4], acc[i][r][g * 4 + 1] + bv[g * 4 + 1],
                                         acc[i][r][g * 4 + 2] + bv[g * 4 + 2], acc[i][r][g * 4 + 3] + bv[g * 4 + 3]});
            flush(P8{}, r, 8, reinterpret_cast<unsigned char *>(p.out) + ((size_t)row0 * N + n0) * 4, (size_t)N * 4);
          }
        }
      }
    }
  }
}

template <class SH, bool GATHER, int EPI>
__global__ __launch_bounds__(TALL_THREADS, 1) void tall_gemm_kernel(GemmParams p) {
  constexpr int RB = SH::RB, CB = SH::CB, LW = SH::LW, LA = SH::LA, LW1 = SH::LW / 2, LA1 = SH::LA / 4;
  constexpr int NR = SH::NR;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w / SH::WC, wc = w % SH::WC;   // the wave's part of the tile
  const int K = p.K, N = p.N;
  const int S = K / TALL_BK;                    // even: K % 64 == 0
  const unsigned lds_base =
      __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)lds);

  // ---- work list: the order of grouped_gemm_kernel (gemm_kernel.hpp), with tiles of BM rows --------
  const const_as<int> tiles = constant_ptr(p.tiles), bounds = constant_ptr(p.xcd_bounds);
  const int n_tiles = p.tiles ? tiles[0] : (p.dense_rows + SH::BM - 1) / SH::BM;
  const int total = n_tiles * p.n_col_tiles;
  const int per_xcd = gridDim.x >> 3;
  const int xcd = blockIdx.x & 7;
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
  // An XCD's items in its last round, if they leave half of its workgroups without one, are cut into two halves of their rows
  const int whole = (hi - lo) - (hi - lo) % per_xcd, rest = hi - lo - whole;
  const bool halves = 2 * rest <= per_xcd;
  const int mine = halves ? whole + 2 * rest : hi - lo;
  int j = blockIdx.x >> 3;
  auto valid = [&](int jj) { return jj < mine; };
  if (!valid(j)) return;
  // which tile, which matrix, and this wave's share of the W loads
  auto decode = [&](int jj, TallSrc<SH> &t) {
    const bool part = halves && jj >= whole;
    const int work = lo + (part ? whole + ((jj - whole) >> 1) : jj);
    int tile;
    if (p.tiles && p.tile_block > 1 && p.xcd_bounds) {
      const int info = bounds[XCD_BOUNDS_INTS + work / p.n_col_tiles];
      const int first = info >> 8, th = info & 255;
      const int v = work - first * p.n_col_tiles;
      t.ct = v / th;
      tile = first + (v - t.ct * th);
    } else if (p.tiles) {
      tile = work / p.n_col_tiles;
      t.ct = work - tile * p.n_col_tiles;
    } else {
      // dense: blocks of eight row tiles are walked column tile by column tile, so that what an XCD's 32 workgroups read
      // at a time are the rows of eight tiles and the weights of four, not of 32 and one (8000 x 8192 x 2048: 315 -> 262
      // us, 8192 x 16384 x 2048: 806 -> 678, 8192 x 5120 x 2880: 241 -> 235)
      const int grp = work / (8 * p.n_col_tiles), v = work - grp * 8 * p.n_col_tiles;
      const int th = min(8, n_tiles - grp * 8);
      t.ct = v / th;
      tile = grp * 8 + (v - t.ct * th);
    }
    if (p.tiles) {
      t.mat = tiles[1 + 3 * tile];
      t.row0 = tiles[2 + 3 * tile];
      t.rows = tiles[3 + 3 * tile];
    } else {
      t.mat = 0;
      t.row0 = tile * SH::BM;
      t.rows = min(SH::BM, p.dense_rows - t.row0);
    }
    if (part) {   // whole row blocks; where there is but one the second half has no rows, and is no item
      const int first = min(t.rows, ((t.rows + 63) >> 6) * 32);
      if (((jj - whole) & 1) == 0) t.rows = first;
      else {
        t.row0 += t.rows > first ? first : 0;
        t.rows -= first;
      }
    }
    t.ct = __builtin_amdgcn_readfirstlane(t.ct);
    t.mat = __builtin_amdgcn_readfirstlane(t.mat);
    t.row0 = __builtin_amdgcn_readfirstlane(t.row0);
    t.rows = __builtin_amdgcn_readfirstlane(t.rows);
    // W fragment f of a stage = (column block f / 2 of the tile, k-step f % 2); a block beyond N repeats the last one
    const int first = t.ct * (SH::WC * CB);
    t.w = tall_buffer(reinterpret_cast<const unsigned char *>(p.W) + ((size_t)t.mat * N + (size_t)first * 32) * K * 2);
#pragma unroll
    for (int q = 0; q < TallSrc<SH>::WB; q++)
      t.wo[q] = (uint32_t)min(w * TallSrc<SH>::WB + q, N / 32 - 1 - first) * (uint32_t)K * 64u;
  };
  // A: load instruction q of this wave moves 8 tile rows, eight lanes per row and one 16-byte piece
  // per lane: the lane at position p of row r fetches piece p ^ ((r >> 1) & 7).  Rows past the
  // tile's last one repeat it (their results are not stored).  The pair ids of a gathered tile are
  // read through the constant address space: scalar loads, which the vector-memory counter of the
  // hand-counted waits does not see.
  // Eight ids are one scalar load, four of which are requested together: id by id, with a wait for each group of rows, an
  // item began with 3.6 us of its 87 (block of 4500 tokens 1081 -> 1073 us, of 5999 1260 -> 1254).  A tile of fewer than
  // eight rows reads on behind them, into what follows in the workspace, and does not use it.
  uint32_t inv_k = 0;
  if constexpr (GATHER) inv_k = pair_inverse(p.top_k);
  auto a_offsets = [&](TallSrc<SH> &t) {
    typedef int ids_t __attribute__((ext_vector_type(8), aligned(4)));
    const int last = t.rows - 1, group = lane >> 3;
    auto offset = [&](int src, int r) {
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      return ((uint32_t)src * (uint32_t)K) * 2u + (uint32_t)c * 16u;
    };
    if constexpr (GATHER) {
      static_assert(LA % 4 == 0, "four row groups at a time");
#pragma unroll
      for (int q0 = 0; q0 < LA; q0 += 4) {
        ids_t v[4];
        int base[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          base[q] = max(min((w * LA + q0 + q) * 8, last - 7), 0);
          v[q] = *(const_as<ids_t>)(p.row_ids + t.row0 + base[q]);
        }
        asm volatile("" : "+s"(v[0]), "+s"(v[1]), "+s"(v[2]), "+s"(v[3]));
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int r = (w * LA + q0 + q) * 8 + group, j = min(r, last) - base[q];
          int src = v[q][0];
#pragma unroll
          for (int i = 1; i < 8; i++) src = j == i ? v[q][i] : src;
          t.a[q0 + q] = offset((int)pair_token(src, inv_k), r);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < LA; q++) {
        const int r = (w * LA + q) * 8 + group;
        t.a[q] = offset(t.row0 + min(r, last), r);
      }
    }
  };

  const uint32_t voff_w = lane * 16;
  const tall_rsrc_t abuf = tall_buffer(p.A);
  // the wave's parts of W buffer `buf` and of A buffer `buf`
  auto w_dst = [&](int buf) { return lds_base + buf * SH::W_BYTES + w * LW * 1024; };
  auto a_dst = [&](int buf) { return lds_base + SH::A_OFF + buf * SH::A_BYTES + w * LA * 1024; };

  f32x16 acc[CB][RB];   // [column block][row block]
  const int sw = ((lane & 31) >> 1) & 7, h = lane >> 5;
  const unsigned a_rd = SH::A_OFF + (wr * 32 + (lane & 31)) * 128;
  unsigned a_k[4];      // where the lane finds its piece of k-step x of a chunk
#pragma unroll
  for (int x = 0; x < 4; x++) a_k[x] = (unsigned)(((2 * x + h) ^ sw) << 4);
  const unsigned w_rd = (wc * CB) * 2 * 1024 + lane * 16;
  bf16x8 F[2][NR];      // two fragment sets: [0, CB) W column blocks, [CB, CB + RB) A row blocks
  // fragment read number i of a k-step, in the order the MFMAs want them: W0, every A, the other W;
  // x = the k-step's number inside its A chunk, NB = row blocks of the wave
  auto rd = [&](auto nb, int wbuf, int kk, int abuf, int x, int set, int i) {
    constexpr int NB = decltype(nb)::value;
    const int f = i == 0 ? 0 : (i <= NB ? CB + i - 1 : i - NB);
    if (f < CB)
      F[set][f] = as_bf16x8(*reinterpret_cast<const u32x4 *>(lds + wbuf * SH::W_BYTES + w_rd + (f * 2 + kk) * 1024));
    else
      F[set][f] = as_bf16x8(
          *reinterpret_cast<const u32x4 *>(lds + abuf * SH::A_BYTES + a_rd + (f - CB) * SH::STEP * 128 + a_k[x]));
  };
  // One k-step: NB * CB MFMAs out of fragment set `set`; with the first of them the fragment reads of
  // the next k-step (into the other set), behind those its loads, loads(0), loads(1), ...
  auto kstep = [&](auto nb, int set, int wbuf, int kk, int abuf, int x, auto &&loads) {
    constexpr int NB = decltype(nb)::value, M = NB * CB, R = NB + CB, L = LA1 + LW1;
    constexpr int PER = (R + L <= M) ? 1 : 2;                                // reads per MFMA
    constexpr int FIRST = PER == 1 ? R : (M - L > 0 ? M - L : 0);            // MFMA that the first load stands behind
    constexpr int APART = FIRST + 2 * (L - 1) < M ? 2 : 1;
    static_assert(FIRST + APART * (L - 1) < M && PER * M >= R, "every read and load has its place");
#pragma unroll
    for (int m = 0; m < M; m++) {
      acc[m / NB][m % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(F[set][m / NB], F[set][CB + m % NB],
                                                                    acc[m / NB][m % NB], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < PER; i++)
        if (m * PER + i < R) rd(nb, wbuf, kk, abuf, x, set ^ 1, m * PER + i);
      if (m >= FIRST && (m - FIRST) % APART == 0) loads((m - FIRST) / APART);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  TallSrc<SH> cur, nxt;
  decode(j, cur);
  if (cur.rows == 0) return;
  a_offsets(cur);
  // The first loads go out in the order the stage loop would have issued them, so that its waits
  // count right from the first stage on: chunk 0 and W stage 0, then a quarter of chunk 1 with
  // every half of W stages 1 and 2.
  static_assert(LW1 == 2 && TallSrc<SH>::WB == 2, "half a W stage is one column block of the wave");
  static_for<0, LA>([&](auto q) { tall_load<decltype(q)::value * 1024>(a_dst(0), cur.a[decltype(q)::value], abuf, 0); });
  static_for<0, LW>([&](auto q) {
    constexpr int Q = decltype(q)::value;
    tall_load<Q * 1024>(w_dst(0), voff_w + (Q & 1) * 1024, cur.w, cur.wo[Q >> 1]);
  });
  static_for<0, 4>([&](auto xx) {
    constexpr int X = decltype(xx)::value;
    static_for<0, LA1>([&](auto q) {
      constexpr int Q = X * LA1 + decltype(q)::value;
      tall_load<Q * 1024>(a_dst(1), cur.a[Q], abuf, 128);
    });
    static_for<0, LW1>([&](auto q) {
      constexpr int Q = (X & 1) * LW1 + decltype(q)::value;
      tall_load<Q * 1024>(w_dst(1 + (X >> 1)), voff_w + (Q & 1) * 1024, cur.w, cur.wo[Q >> 1] + (1 + (X >> 1)) * 2048);
    });
  });
  wait_vmcnt<4 * (LA1 + LW1)>();   // chunk 0 and stage 0 have landed; the loads behind them may be on their way
  __builtin_amdgcn_s_barrier();
  int g = 0;   // running stage count (even at the start of every item): W buffer g & 3
  int ab = 0;  // A buffer of the current chunk: the running chunk count modulo 3
  // what the loop requests next: a W stage, of the current item or the next one, and an A chunk
  tall_rsrc_t ws = cur.w;
  uint32_t wo[2] = {cur.wo[0] + 3 * 2048, cur.wo[1] + 3 * 2048}, ao = 2 * 128;
  const uint32_t voff_w1 = voff_w + 1024;
  while (true) {
    const int jn = j + per_xcd;
    bool more = valid(jn);
    if (more) {
      decode(jn, nxt);
      more = nxt.rows > 0;   // (an empty half belongs to the last round, so nothing comes behind it)
    }
    if (more) a_offsets(nxt);
    else nxt = cur;  // past the last item the pipeline requests this item's first loads again, and drops them
#pragma unroll
    for (int i = 0; i < CB; i++)
#pragma unroll
      for (int r = 0; r < RB; r++)
#pragma unroll
        for (int x = 0; x < 16; x++) acc[i][r][x] = 0.f;
    // the loop over K for NB row blocks of the wave
    auto walk = [&](auto nb) {
      for (int s = 0; s < S; s += 2, g += 2) {
        // ---- even stage s: the first half of A chunk s / 2 --------------------------------------
        const int ab1 = ab == 2 ? 0 : ab + 1, ab2 = ab1 == 2 ? 0 : ab1 + 1;
        // from here on the A chunks that are requested (two ahead) are the next item's, and so is every W stage from the
        // middle of this round on
        const bool wrap = s + 4 >= S;
        if (s + 4 == S) ao = 0;
        const unsigned ad = a_dst(ab2);
        // Every k-step issues a quarter of A chunk s / 2 + 2, into the buffer that chunk s / 2 - 1 left
        // (every wave is past the barrier of the stage that read it last), and half of a W stage,
        // behind the fragment reads
        auto loads = [&](int m, auto xx, int wbuf, auto hh) {
          constexpr int X = decltype(xx)::value, H = decltype(hh)::value;
          static_for<0, LA1>([&](auto q) {
            constexpr int Q = X * LA1 + decltype(q)::value;
            if (m == decltype(q)::value) tall_load<Q * 1024>(ad, wrap ? nxt.a[Q] : cur.a[Q], abuf, ao);
          });
          if (m == LA1) tall_load<2 * H * 1024>(w_dst(wbuf), voff_w, ws, wo[H]);
          if (m == LA1 + 1) {
            tall_load<(2 * H + 1) * 1024>(w_dst(wbuf), voff_w1, ws, wo[H]);
            wo[H] += 2048;
          }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        kstep(nb, 0, g & 3, 1, ab, 1, [&](int m) { loads(m, I0{}, (g + 3) & 3, I0{}); });
        // behind W stage s+1 were issued the loads of two k-steps of stage s-1 and of one of stage s
        wait_vmcnt<3 * (LA1 + LW1)>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        kstep(nb, 1, (g + 1) & 3, 0, ab, 2, [&](int m) { loads(m, I1{}, (g + 3) & 3, I1{}); });
        if (s + 4 == S) {   // W stage s + 3 was this item's last
          ws = nxt.w;
          wo[0] = nxt.wo[0];
          wo[1] = nxt.wo[1];
        }
        // ---- odd stage s+1: the second half of the chunk -----------------------------------------
        kstep(nb, 0, (g + 1) & 3, 1, ab, 3, [&](int m) { loads(m, I2{}, (g + 4) & 3, I0{}); });
        // W stage s+2, and with it the A chunk that the next stage starts (its last loads went out in
        // front of that stage's), must have landed
        wait_vmcnt<3 * (LA1 + LW1)>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        kstep(nb, 1, (g + 2) & 3, 0, ab1, 0, [&](int m) { loads(m, I3{}, (g + 4) & 3, I1{}); });
        ao += 128;
        ab = ab1;
      }
    };
    // The first fragments (those that the item before has read with its last k-step are not kept across its epilogue, and
    // may be of fewer blocks).
#pragma unroll
    for (int i = 0; i < NR; i++) rd(std::integral_constant<int, RB>{}, g & 3, 0, ab, 0, 0, i);
    __builtin_amdgcn_sched_barrier(0);
    // A wave takes every second row block of the tile, so a tile of few rows has few for each of them.
    const int nb = (cur.rows + SH::STEP - 1) / SH::STEP;
    if (nb >= RB) walk(std::integral_constant<int, RB>{});
    else if (nb == 3) walk(std::integral_constant<int, 3>{});
    else if (nb == 2) walk(std::integral_constant<int, 2>{});
    else walk(std::integral_constant<int, 1>{});
    // epilogue: the wave's column blocks, each with its row blocks.  The empty asm pins a column
    // block's accumulators in their AGPRs until the block before it has been stored: left alone,
    // the compiler copies every accumulator to VGPRs where the stage loop ends, and spills.
    if constexpr (EPI == EPI_ARGMAX) {
      // Row-wise arg-max of the wave's CB x 32 columns without writing the products.  A lane holds
      // one row of each row block and 16 channels of each column block: it scans them in ascending
      // column order with a strict >, so the lowest column wins a tie; the two half-waves are merged
      // with the same rule, and the first 32 lanes write the (value, column) pair of their rows for
      // this half of the column tile.
      float bv[RB];
      int bi[RB];
#pragma unroll
      for (int r = 0; r < RB; r++) {
        bv[r] = -INFINITY;
        bi[r] = 0x7fffffff;
      }
      const const_as<float> bias = constant_ptr(p.bias);
#pragma unroll
      for (int i = 0; i < CB; i++) {
#pragma unroll
        for (int r = 0; r < RB; r++) asm volatile("" : "+a"(acc[i][r]));
        const int n0 = cur.ct * SH::BN + (wc * CB + i) * 32;
        if (n0 < N) {
#pragma unroll
          for (int gq = 0; gq < 16; gq++) {
            const int c_lo = n0 + (gq >> 2) * 8 + (gq & 3), c_hi = c_lo + 4;
            float b = 0.f;
            if (p.bias) {
              const float b_lo = bias[c_lo], b_hi = bias[c_hi];
              b = h ? b_hi : b_lo;
            }
            const int col = h ? c_hi : c_lo;
#pragma unroll
            for (int r = 0; r < RB; r++) {
              const float v = acc[i][r][gq] + b;
              if (v > bv[r]) {
                bv[r] = v;
                bi[r] = col;
              }
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < RB; r++) {
        const float ov = lane_xor<32>(bv[r]);
        const int oi = lane_xor<32>(bi[r]);
        if (ov > bv[r] || (ov == bv[r] && oi < bi[r])) {
          bv[r] = ov;
          bi[r] = oi;
        }
        const int row = r * SH::STEP + wr * 32 + lane;
        if (lane < 32 && row < cur.rows) {
          const size_t o = (size_t)(cur.row0 + row) * (SH::WC * p.n_col_tiles) + cur.ct * SH::WC + wc;
          p.amax_val[o] = bv[r];
          p.amax_idx[o] = bi[r];
        }
      }
    } else {
      unsigned char *buf = lds + SH::A_OFF + (ab == 0 ? 2 : ab - 1) * SH::A_BYTES + w * LA * 1024;
      tall_epilogue<SH, EPI>(p, buf, cur.mat, cur.row0 + wr * 32, cur.rows - wr * 32,
                             cur.ct * SH::BN + wc * CB * 32, lane, acc);
    }
    if (!more) break;
    j = jn;
    cur = nxt;
  }
  // loads into LDS are still in flight: the workgroup must not give its LDS back before they land
  wait_vmcnt<0>();
}

template <class SH, bool GATHER, int EPI>
static int launch_tall(const GemmParams &p, int max_tiles, hipStream_t s) {
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static bool raised[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "run_gemm: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  auto kern = tall_gemm_kernel<SH, GATHER, EPI>;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!raised[dev]) {
      GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     SH::SMEM));
      raised[dev] = true;
    }
  }
  GemmParams q = p;
  q.n_col_tiles = cdiv(p.N, SH::BN);
  const long long items = (long long)max_tiles * q.n_col_tiles;
  int grid = (int)std::min<long long>(16 * ((items + 7) / 8), 256);   // room for the halves of an XCD's items
  if (grid == 0) return GPTOSS_OK;
  {
    TraceScope ts(EPI == EPI_ARGMAX ? "gemm_argmax" : GATHER ? "gemm1_gather_swiglu" : "gemm_f32", s);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(TALL_THREADS), SH::SMEM, s, q);
  }
  GPTOSS_LAUNCH_CHECK("tall_gemm_kernel");
  return GPTOSS_OK;
}

// The shape in use.  Tiles of 128 rows for the dense GEMMs of a decode step of 1024 rows (128 x 96,
// 128, 160 and 192 columns, on an earlier form of this kernel with 32-k stages for both operands)
// came out bit-identical as well, and 3-4 us ahead of the streaming kernels' 41-43 us on the two
// projections of the 20B shape: a wave that owns 3 to 6 output blocks has 4 to 6 fragment reads per
// k-step of 100-200 cycles and nothing else to run while they are on their way, so even without any
// load or store such a launch takes 21-28 us where its MFMAs alone take 15.  128 x 128 tiles with two
// workgroups per CU (80 KB of LDS each, on this form of the kernel) did not move that either: 48 and
// 41 us against 43 and 43.  Not worth a second dispatch rule.
using Tall256 = TallShape<2, 2, 4, 4>;   // 256 x 256

}  // namespace gptoss
