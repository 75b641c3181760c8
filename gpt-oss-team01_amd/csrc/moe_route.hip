// MoE routing for gfx950: router GEMM (bf16 MFMA 16x16x32), top-k + softmax gating with exchanges
// between lanes in registers, and a stable counting sort of the (token,slot) pairs by expert built from wave
// ballots and an LDS histogram (no global atomics), which also emits the tile list that the
// grouped GEMMs schedule from.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"
#include "moe_gating.hpp"

namespace gptoss {

__device__ __forceinline__ uint64_t same_expert_mask(int e, bool valid, int nbits) {
  uint64_t mask = __ballot(valid);
  for (int b = 0; b < nbits; b++) {
    bool bit = (e >> b) & 1;
    uint64_t bal = __ballot(valid && bit);
    mask &= bit ? bal : ~bal;
  }
  return mask;
}

// Exclusive prefix sum over up to 256 values held 4 per lane by one wave (lane l owns entries
// 4l..4l+3); returns the lane's own exclusive prefixes through ex[] and the grand total.
__device__ __forceinline__ int wave_scan4(const int (&v)[4], int (&ex)[4]) {
  const int lane = threadIdx.x & 63;
  int sum = v[0] + v[1] + v[2] + v[3];
  // inside the rows of 16 lanes (row_shr 1, 2, 4, 8; nothing enters from outside), then the last lane of rows 0 and 2 to
  // rows 1 and 3, then lane 31 to the upper half
  int inc = sum;
  inc += __builtin_amdgcn_mov_dpp(inc, 0x111, 0xf, 0xf, true);
  inc += __builtin_amdgcn_mov_dpp(inc, 0x112, 0xf, 0xf, true);
  inc += __builtin_amdgcn_mov_dpp(inc, 0x114, 0xf, 0xf, true);
  inc += __builtin_amdgcn_mov_dpp(inc, 0x118, 0xf, 0xf, true);
  inc += __builtin_amdgcn_update_dpp(0, inc, 0x142, 0xa, 0xf, false);
  inc += __builtin_amdgcn_update_dpp(0, inc, 0x143, 0xc, 0xf, false);
  int run = inc - sum;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    ex[i] = run;
    run += v[i];
  }
  return __builtin_amdgcn_readlane(inc, 63);
}

// From the experts' pair counts total[E] (LDS): the experts' offsets into offs[E+1] (LDS), and, when
// `publish` is set, to memory together with the number of tiles and the cut positions
// of the work list.  Called by one whole wave (wave 0 of a workgroup); cost_pre / tile_pre are E
// ints of LDS scratch each, tile_pre the experts' first tiles, for group_tiles.
__device__ __forceinline__ void group_finish(const int *total, int *offs, int *cost_pre, int *tile_pre, int E,
                                             bool publish, int *__restrict__ expert_offsets,
                                             int *__restrict__ tiles, int rows_per_tile,
                                             int *__restrict__ xcd_bounds, int cost0) {
  const int lane = threadIdx.x & 63;
  int cnt[4], nt[4], off_ex[4], tile_ex[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int e = lane * 4 + i;
    cnt[i] = (e < E) ? total[e] : 0;
    nt[i] = (rows_per_tile > 0) ? (cnt[i] + rows_per_tile - 1) / rows_per_tile : 0;
  }
  const int all = wave_scan4(cnt, off_ex);
  const int n_tiles = wave_scan4(nt, tile_ex);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int e = lane * 4 + i;
    if (e < E) {
      offs[e] = off_ex[i];
      if (publish) expert_offsets[e] = off_ex[i];
      tile_pre[e] = tile_ex[i];
    }
  }
  if (lane == 0) {
    offs[E] = all;
    if (publish) expert_offsets[E] = all;
    if (publish && tiles != nullptr && rows_per_tile > 0) tiles[0] = n_tiles;
  }
  // Where to cut the tile list into 8 parts (one per XCD) of equal estimated cost: a tile costs
  // cost0 + 2 per 32-row block (half units), all work items of a tile cost the same, and a cut may
  // fall inside a tile (between two of its column tiles), hence the 16-bit fraction.
  if (publish && xcd_bounds != nullptr && tiles != nullptr && rows_per_tile > 0) {
    const int cfull = cost0 + 2 * (rows_per_tile / 32);
    auto last_cost = [&](int count, int n) { return cost0 + 2 * ((count - (n - 1) * rows_per_tile + 31) / 32); };
    int cost[4], cpre[4];
#pragma unroll
    for (int i = 0; i < 4; i++) cost[i] = (nt[i] > 0) ? (nt[i] - 1) * cfull + last_cost(cnt[i], nt[i]) : 0;
    const int ctot = wave_scan4(cost, cpre);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int e = lane * 4 + i;
      if (e < E) cost_pre[e] = cpre[i];
    }
    // lane x finds cut x: the last expert whose cost prefix is <= x/8 of the total has a tile under
    // the cut (experts without rows share their successor's prefix).  All quantities fit 32 bits:
    // ctot < 2^15 tiles * (cost0 + 16).
    if (lane < 8) {
      int bound = 0;
      if (ctot > 0) {
        const int target = (lane * ctot) >> 3;
        int lo = 0, hi = E - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (cost_pre[mid] <= target) lo = mid;
          else hi = mid - 1;
        }
        const int count = offs[lo + 1] - offs[lo];
        const int nte = (count + rows_per_tile - 1) / rows_per_tile;
        // float quotient (operands < 2^24) with a one-step correction instead of integer division
        const int a = target - cost_pre[lo];
        const float rcp_cfull = __builtin_amdgcn_rcpf((float)cfull);
        int t = (int)((float)a * rcp_cfull);
        t -= (t * cfull > a) ? 1 : 0;
        t += ((t + 1) * cfull <= a) ? 1 : 0;
        t = min(t, nte - 1);
        const int rest = a - t * cfull;
        const float inv = (t == nte - 1) ? __builtin_amdgcn_rcpf((float)last_cost(count, nte)) : rcp_cfull;
        bound = ((tile_pre[lo] + t) << 16) | min(65535, (int)((float)rest * 65536.0f * inv));
      }
      xcd_bounds[lane] = bound;
    }
    if (lane == 0) xcd_bounds[8] = n_tiles << 16;
  }
}

// The tile list and every tile's block, by all threads of a workgroup, a tile each, from what group_finish left in LDS.  (An
// expert's lane writing its tiles one after the other took most of the kernel where experts had many: scatter kernel, 4096 tokens
// on all of 4 experts, 64-row tiles, 30.8 -> 5.9 us; 128 experts under Zipf 1.1 20.4 -> 6.8; 5999 tokens on 32, 256-row tiles,
// 11.7 -> 6.4; sorting kernel, 1024 tokens 10.8 -> 9.6.)
__device__ __forceinline__ void group_tiles(const int *total, const int *offs, const int *tile_pre, int E,
                                            int *__restrict__ tiles, int rows_per_tile, int *__restrict__ xcd_bounds) {
  if (tiles == nullptr || rows_per_tile <= 0) return;
  const int n_tiles = tile_pre[E - 1] + (total[E - 1] + rows_per_tile - 1) / rows_per_tile;
  for (int tile = threadIdx.x; tile < n_tiles; tile += blockDim.x) {
    int e = 0, hi = E - 1;   // the last expert whose first tile is no later (experts without rows share their successor's)
    while (e < hi) {
      const int mid = (e + hi + 1) >> 1;
      if (tile_pre[mid] <= tile) e = mid;
      else hi = mid - 1;
    }
    const int first = tile_pre[e], t = tile - first, count = total[e];
    int *tp = tiles + 1 + 3 * tile;
    tp[0] = e;
    tp[1] = offs[e] + t * rows_per_tile;
    tp[2] = min(rows_per_tile, count - t * rows_per_tile);
    if (xcd_bounds != nullptr) {   // the block of up to MOE_TILE_BLOCK tiles of this expert that the tile belongs to
      const int b0 = t - t % MOE_TILE_BLOCK, nt = (count + rows_per_tile - 1) / rows_per_tile;
      xcd_bounds[XCD_BOUNDS_INTS + tile] = ((first + b0) << 8) | min(MOE_TILE_BLOCK, nt - b0);
    }
  }
}

constexpr int ROUTER_GROUP_PAIRS = ROUTER_GROUP_TOKENS * 8;

// Stable grouping of at most ROUTER_GROUP_PAIRS pairs by one wave: what group_sort_kernel writes for them.  No expert has
// more than ROUTER_GROUP_TOKENS rows, so every expert that has any is one tile and a block of its own, and the work list
// is cut into eight parts of equal length.
__device__ __forceinline__ void group_by_one_wave(const int *topk_i, int P, int E, int *lds, const RouterGroup &g) {
  int *total = lds, *offs = total + 256;   // [256] each
  const int lane = threadIdx.x & 63;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int i = 0; i < 4; i++) total[lane * 4 + i] = 0;
  constexpr int STEPS = ROUTER_GROUP_PAIRS / 64;
  int e[STEPS], rank[STEPS];
#pragma unroll
  for (int u = 0; u < STEPS; u++) {
    if (u * 64 < P) {
      const int p = u * 64 + lane;
      const bool valid = p < P;
      e[u] = valid ? topk_i[p] : 0;
      const uint64_t mask = same_expert_mask(e[u], valid, g.nbits);
      rank[u] = valid ? total[e[u]] + __popcll(mask & lt_mask) : 0;
      // all lanes have read the counts before the lowest lane of each expert updates them (wave-ordered LDS operations)
      if (valid && (mask & lt_mask) == 0) total[e[u]] += __popcll(mask);
    }
  }
  // one scan for both prefixes: rows in the low half, experts with rows (= tiles) in the high half
  int v[4], ex[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int c = total[lane * 4 + i];
    v[i] = c | (c > 0 ? 1 << 16 : 0);
  }
  const int n_tiles = wave_scan4(v, ex) >> 16;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int x = lane * 4 + i, off = ex[i] & 0xffff, t = ex[i] >> 16;
    offs[x] = off;
    if (x <= E) g.expert_offsets[x] = off;
    if (v[i]) {
      int *tp = g.tiles + 1 + 3 * t;
      tp[0] = x;
      tp[1] = off;
      tp[2] = v[i] & 0xffff;
      g.xcd_bounds[XCD_BOUNDS_INTS + t] = (t << 8) | 1;
    }
  }
  if (lane < 9) g.xcd_bounds[lane] = (lane * n_tiles) << 13;   // tile << 16 | fraction
  if (lane == 0) g.tiles[0] = n_tiles;
  if (lane == 0 && E == 256) g.expert_offsets[E] = P;
#pragma unroll
  for (int u = 0; u < STEPS; u++) {
    const int p = u * 64 + lane;
    if (p < P) {
      const int dst = offs[e[u]] + rank[u];
      g.sorted_pair_ids[dst] = p;
      g.inv_perm[p] = dst;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Router GEMM: logits[B,E] = t[B,H] . Wr[E,H]^T + br, and the gating of the tokens, 32 lanes per token, while the logits are
// still in LDS.
// ------------------------------------------------------------------------------------------------
// k-steps whose operands a wave requests before its first MFMA: as many as ~150 registers hold,
// so that a hidden size of 2880 with up to 32 experts is a single round of loads
constexpr int router_steps(int nb) { return nb <= 2 ? 12 : (nb <= 4 ? 7 : (nb <= 8 ? 4 : 2)); }

// What norm_router_kernel does first: x += residual, t = RMSNorm(x) * weight for the
// workgroup's own token rows.
struct RouterNorm {
  float *x;               // [B,H] residual stream, updated in place
  const float *residual;  // [B,H] or nullptr
  const float *weight;    // [H]
  bf16_t *t_out;          // [B,H]
};

// x += residual, t = RMSNorm(x) * weight for `rows` rows from r0 on, t to memory and to t_rows in LDS: the arithmetic of
// rmsnorm_rows_kernel, 256 threads per row, the same element-to-thread assignment and summation order, so t is the same to the
// bit; as many rows at a time as the workgroup has 256 threads.  SHARED: other workgroups norm the same rows, so x stays as it is,
// and t is stored by one of them (store_t).  requested(): called once, when the first rows are on their way.
template <bool W_EARLY, bool SHARED, class Requested>
__device__ __forceinline__ void norm_rows(const RouterNorm &nrm, bf16_t *t_rows, int r0, int rows, int B, int H, bool store_t,
                                          Requested &&requested) {
  constexpr int VPT = 4;  // rows of up to 4096 floats
  __shared__ double nred[2][4];
  const int grp = threadIdx.x >> 8, tg = threadIdx.x & 255, groups = blockDim.x >> 8;  // groups of 256 threads, a row each
  f32x4 nw[VPT];
#pragma unroll
  for (int i = 0; i < VPT; i++)
    if (W_EARLY) nw[i] = *reinterpret_cast<const f32x4 *>(nrm.weight + min((tg + 256 * i) * 4, H - 4));
  for (int rr = 0; rr < rows; rr += groups) {
    const int lr = rr + grp;
    const bool live = lr < rows && r0 + lr < B;
    const size_t row = (size_t)(r0 + lr) * H;
    // no load under a condition, so that a row's are all on their way together (lanes past its end read its last elements)
    const size_t src = (size_t)min(r0 + min(lr, rows - 1), B - 1) * H;
    f32x4 v[VPT], res[VPT];
#pragma unroll
    for (int i = 0; i < VPT; i++) {
      const int h = min((tg + 256 * i) * 4, H - 4);
      v[i] = *reinterpret_cast<const f32x4 *>(nrm.x + src + h);
      res[i] = *reinterpret_cast<const f32x4 *>((nrm.residual ? nrm.residual : nrm.x) + src + h);
    }
    if (rr == 0) requested();
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < VPT; i++) {
      const int h = (tg + 256 * i) * 4;
      if (live && h < H) {
        if (nrm.residual) {
#pragma unroll
          for (int q = 0; q < 4; q++) v[i][q] = __fadd_rn(v[i][q], res[i][q]);
          if (!SHARED) *reinterpret_cast<f32x4 *>(nrm.x + row + h) = v[i];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) ss += (double)__fmul_rn(v[i][q], v[i][q]);
      }
    }
    ss = lanes_sum(ss);
    if ((threadIdx.x & 63) == 0) nred[grp][(threadIdx.x >> 6) & 3] = ss;
    __syncthreads();
    ss = nred[grp][0] + nred[grp][1] + nred[grp][2] + nred[grp][3];
    ss /= H;
    ss += 1e-5f;
    const double inv = (double)(1.0f / sqrtf((float)ss));
#pragma unroll
    for (int i = 0; i < VPT; i++) {
      const int h = (tg + 256 * i) * 4;
      if (live && h < H) {
        if (!W_EARLY) nw[i] = *reinterpret_cast<const f32x4 *>(nrm.weight + h);
        f32x4 o;
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = (float)((double)nw[i][q] * (inv * (double)v[i][q]));
        const u32x2 pk = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        if (!SHARED || store_t) *reinterpret_cast<u32x2 *>(nrm.t_out + row + h) = pk;
        *reinterpret_cast<u32x2 *>(t_rows + (size_t)lr * H + h) = pk;
      }
    }
    __syncthreads();   // nred is reused by the next pair of rows; after the last pair: t_rows complete
  }
}

// What follows the products of a workgroup of ROUTER_WAVES waves, 32 lanes per token row (`live`: it is one): the sum of the
// waves' parts and the bias, published, and gated if the workgroup has all experts.
template <int NB>
__device__ __forceinline__ void router_gate(float (*red)[16][NB * 16 + 1], const float (&bias)[(NB + 1) / 2],
                                            float *__restrict__ logits, int r0, int e0, bool live, bool has_bias, int B, int E, int k,
                                            float *__restrict__ topk_w, int *__restrict__ topk_i, const RouterGroup &grp) {
  constexpr int NJ = (NB + 1) / 2;
  const int row = threadIdx.x >> 5, sub = threadIdx.x & 31;
  float v[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int col = sub + 32 * j, e = e0 + col;
    float x = -INFINITY;
    if (e < E && col < NB * 16) {
      x = 0.f;
#pragma unroll
      for (int w = 0; w < ROUTER_WAVES; w++) x += red[w][row][col];
      if (has_bias) x += bias[j];
      if (live) logits[(size_t)(r0 + row) * E + e] = x;
    }
    v[j] = x;
  }
  if (topk_w != nullptr) {
    const size_t o = (size_t)(live ? r0 + row : 0) * k;
    __shared__ int ids[ROUTER_GROUP_PAIRS];
    topk_softmax_group<NJ>(v, sub, E, k, live, topk_w + o, topk_i + o, grp.expert_offsets ? ids + row * k : nullptr);
    if (grp.expert_offsets != nullptr) {   // one workgroup holds every token
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) group_by_one_wave(ids, B * k, E, reinterpret_cast<int *>(red), grp);
    }
  }
}

// The router behind a norm: the workgroup first normalises its
// rows (norm_rows) and multiplies them from LDS, with the experts' weights, meanwhile requested, from registers: one launch and one read of t less than norm kernel + router kernel.
// A small launch is a chain of waits for memory, so all that does not depend on each other is requested at once: the
// router's weights and biases, a row's elements, its residual and the norm's weights.  (With a branch for each of the
// row's parts they came one behind the other.)  One row of 2880, 4 experts 8.4 -> 7.3 us, 33 rows 10.6 -> 8.4
// (6.1 with two rows per workgroup, run_norm_router).
template <int NB>   // 16-expert column blocks held per wave
__global__ __launch_bounds__(ROUTER_WAVES * 64) void norm_router_kernel(
    const bf16_t *__restrict__ wr, const float *__restrict__ br,
    float *__restrict__ logits, int B, int H, int E, int k, float *__restrict__ topk_w,
    int *__restrict__ topk_i, int rows_per_wg, RouterNorm nrm, RouterGroup grp) {
  __shared__ float red[ROUTER_WAVES][16][NB * 16 + 1];
  extern __shared__ __attribute__((aligned(16))) unsigned char t_rows_raw[];  // [rows_per_wg][H] bf16
  // The wave's number has to be a scalar: matrix instructions do not look at the mask of active lanes, so a wave skips the
  // k-steps that are not its own only by a branch, and for a condition on a lane's value the compiler leaves the branch
  // out where masking looks cheaper (one matrix instruction under it, no wait: its products were added all the same).
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows_per_wg <= 16 token rows are this workgroup's; the other MFMA rows repeat the last of them
  const int r0 = blockIdx.x * rows_per_wg;
  const int arow = min(r0 + min(lane & 15, rows_per_wg - 1), B - 1);
  const int kq = (lane >> 4) * 8;
  constexpr int ROUTER_MAX_STEPS = router_steps(NB);
  const int ksteps = H / 32;
  // In two halves: while one is multiplied, the other's loads are on their way.  More than 128 experts leave no registers for it.
  constexpr int SETS = NB <= 8 ? 2 : 1, HALF = (ROUTER_MAX_STEPS + SETS - 1) / SETS, STRIDE = HALF * ROUTER_WAVES;
  u32x4 a[SETS][HALF], b[SETS][HALF][NB];
  auto load_b = [&](int ks0, auto set) {
#pragma unroll
    for (int u = 0; u < HALF; u++) {
      const int ks = min(ks0 + u * ROUTER_WAVES, ksteps - 1);
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        int e = min(nb * 16 + (lane & 15), E - 1);
        b[decltype(set)::value][u][nb] = *reinterpret_cast<const u32x4 *>(wr + (size_t)e * H + ks * 32 + kq);
      }
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, SETS - 1>;
  // the bias of the experts that the lane sums up in the end
  const int row = threadIdx.x >> 5, sub = threadIdx.x & 31;
  constexpr int NJ = (NB + 1) / 2;
  float bias[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) bias[j] = br ? br[min(sub + 32 * j, E - 1)] : 0.f;
  // the router's weights do not wait for the norm (more than 128 experts: no registers to hold them meanwhile).  Loads return
  // in order, so the bias is in front of them, and a wave without a k-step requests none: behind twelve steps' loads in each
  // of eight waves, of which H = 64 has work for two, 32 / 128 experts took 7.0 / 9.1 us instead of 3.1 / 3.7.
  constexpr bool EARLY = NB <= 8;
  static_assert(EARLY || SETS == 1, "two sets are requested early");
  if (EARLY && wave < ksteps) load_b(wave, S0{});
  if (SETS == 2 && EARLY && wave + STRIDE < ksteps) load_b(wave + STRIDE, S1{});
  bf16_t *t_rows = reinterpret_cast<bf16_t *>(t_rows_raw);
  norm_rows<(NB < 8), false>(nrm, t_rows, r0, rows_per_wg, B, H, true, [] {});   // (W_EARLY where registers allow)
  const bf16_t *ap = t_rows + (size_t)(arow - r0) * H + kq;
  f32x4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto load_a = [&](int ks0, auto set) {
#pragma unroll
    for (int u = 0; u < HALF; u++)
      a[decltype(set)::value][u] = *reinterpret_cast<const u32x4 *>(ap + min(ks0 + u * ROUTER_WAVES, ksteps - 1) * 32);
  };
  auto multiply = [&](int ks0, auto set) {
#pragma unroll
    for (int u = 0; u < HALF; u++) {
      if (ks0 + u * ROUTER_WAVES < ksteps) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
          acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[decltype(set)::value][u]),
                                                            as_bf16x8(b[decltype(set)::value][u][nb]), acc[nb], 0, 0, 0);
      }
    }
  };
  if constexpr (SETS == 1) {
    for (int ks0 = wave; ks0 < ksteps; ks0 += STRIDE) {
      if (!EARLY || ks0 != wave) load_b(ks0, S0{});
      load_a(ks0, S0{});
      multiply(ks0, S0{});
    }
  } else if (wave < ksteps) {
    load_a(wave, S0{});
    if (wave + STRIDE < ksteps) load_a(wave + STRIDE, S1{});
    for (int ks0 = wave; ks0 < ksteps; ks0 += 2 * STRIDE) {
      multiply(ks0, S0{});
      if (ks0 + 2 * STRIDE < ksteps) {
        load_b(ks0 + 2 * STRIDE, S0{});
        load_a(ks0 + 2 * STRIDE, S0{});
      }
      if (ks0 + STRIDE >= ksteps) break;
      multiply(ks0 + STRIDE, S1{});
      if (ks0 + 3 * STRIDE < ksteps) {
        load_b(ks0 + 3 * STRIDE, S1{});
        load_a(ks0 + 3 * STRIDE, S1{});
      }
    }
  }
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave][(lane >> 4) * 4 + i][nb * 16 + (lane & 15)] = acc[nb][i];
  __syncthreads();
  router_gate<NB>(red, bias, logits, r0, 0, row < rows_per_wg && r0 + row < B, br != nullptr, B, E, k, topk_w, topk_i, grp);
}

// The router: one workgroup = 16 token rows x all experts (or 16 of them, where they are shared out among workgroups); its 8
// waves split the K loop (k-steps of 32, interleaved) and reduce through LDS; with topk_w it also gates its tokens.
// The operands come through LDS.  In operand order a load takes 16 bytes of
// 16 rows by every four lanes in a row, and a CU reads 36 KB a us that way; of whole rows 64 bytes a cycle (all CUs at work on what
// their L2s hold: 110 KB a us).  So the workgroup's 16 rows and its experts' come in stages of 512 bytes a row, one k-step for each
// wave, straight into LDS, and are taken from there.  More than 64 experts come in parts of a stage, so that three
// buffers have room; 32 experts' three buffers leave room for a second workgroup (6000 tokens 13.2 -> 12.5).  Operands straight into registers in operand order -> this,
// all experts in one workgroup, 2880 inputs (us): 32 experts, 27 / 1024 / 4096 tokens 8.3 /
// 8.9 / 10.4 -> 5.0 / 5.6 / 6.3, 64 16.0 / 16.7 / 18.2 -> 7.1 / 7.9 / 8.4, 128 27.2 / 26.0 / 27.5 -> 12.3 / 13.0 / 14.3; 2048 inputs and four
// 4.1 / 4.5 / 6.5 -> 3.9 / 3.9 / 6.1.  Same bits.
template <int NB>
struct RouterStages {
  static constexpr int PARTS = (NB + 3) / 4, BLOCKS = NB / PARTS;   // parts of a stage, 16-expert blocks of a part
  static constexpr int ROWS = 16 + BLOCKS * 16, BYTES = ROWS * 512, LOADS = ROWS / 16;   // loads: per wave, two rows each
  static constexpr int COUNT = NB == 1 ? 4 : 3;                       // buffers, all but one of them on their way
  static constexpr int RED = ROUTER_WAVES * 16 * (NB * 16 + 1) * 4;   // the waves' sums, when the loop is over
  static constexpr int SMEM = COUNT * BYTES > RED ? COUNT * BYTES : RED;
  static_assert(SMEM + 1024 <= 160 * 1024, "LDS of a CU");
};

template <int N>
__device__ __forceinline__ void router_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// LARGE: experts or 16 rows of 4 GiB and more, which gptoss_router_gemm takes.  Offsets of 64 bits cost the others up to 6 % (256
// experts of 1024 inputs, 1024 tokens 10.7 -> 11.3 us).
template <int NB, bool LARGE>
__global__ __launch_bounds__(ROUTER_WAVES * 64) void router_gemm_kernel(
    const bf16_t *__restrict__ t, const bf16_t *__restrict__ wr, const float *__restrict__ br, float *__restrict__ logits, int B,
    int H, int E, int k, float *__restrict__ topk_w, int *__restrict__ topk_i, int rows_per_wg, RouterGroup grp) {
  const int e0 = blockIdx.y * (NB * 16);   // first expert of the workgroup; it gates only if it has them all
  using S = RouterStages<NB>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = blockIdx.x * rows_per_wg, ksteps = H / 32, n_stages = (ksteps + ROUTER_WAVES - 1) / ROUTER_WAVES;
  const int row = threadIdx.x >> 5, sub = threadIdx.x & 31;
  constexpr int NJ = (NB + 1) / 2;
  float bias[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) bias[j] = br ? br[min(e0 + sub + 32 * j, E - 1)] : 0.f;
  // Load x of the wave moves rows 16 x + 2 wave and the next of a buffer: token rows with x = 0 (those beyond the workgroup's
  // repeat its last one), then experts'.  Position j of row r holds piece j ^ (r & 15), so that a fragment's lanes hit
  // different banks.  (The compiler does not count these loads.)
  const int pair = 2 * wave + (lane >> 5), piece = (lane & 31) ^ pair;
  using Place = std::conditional_t<LARGE, const unsigned char *, uint32_t>;   // of a row: its address, or its offset in bytes
  auto place = [&](const bf16_t *base, int row) {
    if constexpr (LARGE) return reinterpret_cast<const unsigned char *>(base + (size_t)row * H);
    else return (uint32_t)row * (uint32_t)H * 2u;
  };
  auto load = [&](unsigned to, Place from, const bf16_t *base) {
    if constexpr (LARGE) load_to_lds(to, from);
    else load_to_lds(to, from, base);
  };
  const bf16_t *a_src = t + (size_t)r0 * H;
  const Place a_row = place(a_src, min(min(pair, rows_per_wg - 1), B - 1 - r0));
  Place e_row[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) e_row[nb] = place(wr, min(e0 + nb * 16 + pair, E - 1));
  const unsigned lds_base =
      __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)lds) + wave * 1024;
  auto request = [&](int st, auto part, int buf) {
    constexpr int P = decltype(part)::value;
    const uint32_t at = (uint32_t)st * 512u + (st * 256 + piece * 8 < H ? piece * 16 : 0);   // (beyond a row's end: nobody's)
    const unsigned to = lds_base + buf * S::BYTES;
    load(to, a_row + at, a_src);
#pragma unroll
    for (int x = 0; x < S::BLOCKS; x++) load(to + (x + 1) * 8192, e_row[P * S::BLOCKS + x] + at, wr);
  };
  f32x4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned char *frag = lds + (lane & 15) * 512 + (((wave * 4 + (lane >> 4)) ^ (lane & 15)) << 4);
  // parts are numbered through: part u of the loop is part u % PARTS of stage u / PARTS
  const int total = n_stages * S::PARTS;
  static_for<0, S::COUNT - 1>([&](auto u) {
    constexpr int U = decltype(u)::value;
    if (U < total) request(U / S::PARTS, std::integral_constant<int, U % S::PARTS>{}, U);
  });
  int buf = 0, ahead = S::COUNT - 1;
  for (int st = 0; st < n_stages; st++) {
    static_for<0, S::PARTS>([&](auto part) {
      constexpr int P = decltype(part)::value;
      const int u = st * S::PARTS + P;
      // part u has landed when no more than the COUNT - 2 behind it are on their way; behind the barrier it has for every
      // wave, and nobody reads the buffer of the part before any more
      if (u + S::COUNT - 1 <= total) router_wait<(S::COUNT - 2) * S::LOADS>();
      else router_wait<0>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      constexpr int Q = P + S::COUNT - 1;
      if (u + S::COUNT - 1 < total) request(st + Q / S::PARTS, std::integral_constant<int, Q % S::PARTS>{}, ahead);
      if (st * ROUTER_WAVES + wave < ksteps) {
        const unsigned char *f = frag + buf * S::BYTES;
        const bf16x8 a = as_bf16x8(*reinterpret_cast<const u32x4 *>(f));
#pragma unroll
        for (int x = 0; x < S::BLOCKS; x++)
          acc[P * S::BLOCKS + x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, as_bf16x8(*reinterpret_cast<const u32x4 *>(f + (x + 1) * 8192)), acc[P * S::BLOCKS + x], 0, 0, 0);
      }
      buf = buf + 1 == S::COUNT ? 0 : buf + 1;
      ahead = ahead + 1 == S::COUNT ? 0 : ahead + 1;
    });
  }
  __syncthreads();   // the buffers have been read
  typedef float Sums[16][NB * 16 + 1];
  Sums *red = reinterpret_cast<Sums *>(lds);
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave][(lane >> 4) * 4 + i][nb * 16 + (lane & 15)] = acc[nb][i];
  __syncthreads();
  router_gate<NB>(red, bias, logits, r0, e0, row < rows_per_wg && r0 + row < B, br != nullptr, B, E, k, topk_w, topk_i, grp);
}

// The partial products that the waves of router_gemm_kernel add up, of at most 16 tokens: a workgroup is one of its waves over
// 16 experts.  One workgroup for all of them waits for the experts' weights, of which a CU gets 36 KB a us; here 8 to 128 CUs
// share them.  Whoever gates adds the parts up (PartialLogit).  NORM: every workgroup norms the few rows for itself, in the time
// that its weights take, and t is an output; what adds the residual to x comes behind (few_routed_kernel).
// Between events, which add 4 us: 2880 inputs, 32 experts, one token 11.8 us with the gating -> 6.2 without; of 12 tokens the
// whole routing, in two launches instead of one, takes 4.6 us less.
template <bool NORM>
__global__ __launch_bounds__(NORM ? 512 : 64) void router_parts_kernel(const bf16_t *__restrict__ t, const bf16_t *__restrict__ wr,
                                                                       float *__restrict__ parts, int B, int H, int E, RouterNorm nrm) {
  constexpr int STEPS = 12;
  extern __shared__ __attribute__((aligned(16))) unsigned char t_rows_raw[];   // NORM: [B][H] bf16
  const int lane = threadIdx.x & 63, wave = blockIdx.x, e0 = blockIdx.y * 16;
  const bool multiplies = !NORM || __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0;
  const int kq = (lane >> 4) * 8, ksteps = H / 32, arow = min(lane & 15, B - 1);
  const bf16_t *ap = t + (size_t)arow * H + kq, *bp = wr + (size_t)min(e0 + (lane & 15), E - 1) * H + kq;
  u32x4 a[STEPS], b[STEPS];
  auto load = [&](const bf16_t *from, u32x4 (&to)[STEPS], int ks0) {
#pragma unroll
    for (int u = 0; u < STEPS; u++) to[u] = *reinterpret_cast<const u32x4 *>(from + min(ks0 + u * ROUTER_WAVES, ksteps - 1) * 32);
  };
  if constexpr (NORM) {
    bf16_t *t_rows = reinterpret_cast<bf16_t *>(t_rows_raw);
    norm_rows<true, true>(nrm, t_rows, 0, B, B, H, wave == 0 && e0 == 0, [&] {
      if (multiplies) load(bp, b, wave);
    });
    if (!multiplies) return;
    ap = t_rows + (size_t)arow * H + kq;
  } else {
    load(bp, b, wave);
  }
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ks0 = wave; ks0 < ksteps; ks0 += ROUTER_WAVES * STEPS) {
    if (ks0 != wave) load(bp, b, ks0);
    load(ap, a, ks0);
#pragma unroll
    for (int u = 0; u < STEPS; u++)
      if (ks0 + u * ROUTER_WAVES < ksteps) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[u]), as_bf16x8(b[u]), acc, 0, 0, 0);
  }
  const int e = e0 + (lane & 15);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = (lane >> 4) * 4 + i;
    if (row < B && e < E) parts[((size_t)wave * B + row) * E + e] = acc[i];
  }
}

// ------------------------------------------------------------------------------------------------
// Stand-alone gating from logits in memory: 32 lanes per token, two tokens per wave.
// ------------------------------------------------------------------------------------------------
template <int NJ, int KMAX = 8>
__global__ __launch_bounds__(256) void topk_softmax_kernel(const float *__restrict__ logits, int B,
                                                           int E, int k, float *__restrict__ topk_w,
                                                           int *__restrict__ topk_i) {
  const int sub = threadIdx.x & 31;
  const int token = (blockIdx.x * 256 + threadIdx.x) >> 5;
  const bool live = token < B;
  const float *row = logits + (size_t)(live ? token : 0) * E;
  float v[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    int e = sub + 32 * j;
    v[j] = (live && e < E) ? row[e] : -INFINITY;
  }
  const size_t o = (size_t)(live ? token : 0) * k;
  topk_softmax_group<NJ, KMAX>(v, sub, E, k, live, topk_w + o, topk_i + o);
}

// ------------------------------------------------------------------------------------------------
// Stable counting sort of P = B*k pairs by expert in ONE workgroup of 1024 threads (16 waves).
// Each wave owns a contiguous range of pairs.  Inside a 64-pair step the lanes holding the same
// expert are found with log2(E) ballots; the lowest such lane adds their count to the wave's own
// LDS histogram row, so no atomics are needed and the order is the pair order (stable).
// ------------------------------------------------------------------------------------------------
constexpr int SORT_THREADS = 1024;
constexpr int SORT_WAVES = SORT_THREADS / 64;

constexpr int SORT_CHUNK = 8;  // 64-pair steps whose expert ids a wave requests at once

__global__ __launch_bounds__(SORT_THREADS) void group_sort_kernel(
    const int *__restrict__ topk_i, int P, int E, int nbits, int *__restrict__ expert_offsets,
    int *__restrict__ sorted_pair_ids, int *__restrict__ inv_perm, int *__restrict__ tiles,
    int rows_per_tile, int *__restrict__ xcd_bounds, int cost0) {
  extern __shared__ int smem[];
  int *hist = smem;                    // [SORT_WAVES][E] per-wave counts, then per-wave cursors
  int *total = hist + SORT_WAVES * E;  // [E]
  int *offs = total + E;               // [E+1]
  int *cost_pre = offs + E + 1;        // [E] exclusive prefix of the experts' estimated cost
  int *tile_pre = cost_pre + E;        // [E] first tile of every expert
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

  for (int i = threadIdx.x; i < SORT_WAVES * E; i += SORT_THREADS) hist[i] = 0;
  __syncthreads();

  const int steps_total = (P + 63) / 64;
  const int steps_per_wave = (steps_total + SORT_WAVES - 1) / SORT_WAVES;
  const int p_begin = wave * steps_per_wave * 64;
  const int p_end = min(P, p_begin + steps_per_wave * 64);
  int *myhist = hist + wave * E;

  // expert ids of SORT_CHUNK steps are requested together, so their latencies overlap
  auto load_chunk = [&](int p0, int (&e)[SORT_CHUNK]) {
#pragma unroll
    for (int u = 0; u < SORT_CHUNK; u++) {
      const int p = p0 + u * 64 + lane;
      e[u] = (p < p_end) ? topk_i[p] : -1;
    }
  };

  for (int p0 = p_begin; p0 < p_end; p0 += 64 * SORT_CHUNK) {
    int e[SORT_CHUNK];
    load_chunk(p0, e);
#pragma unroll
    for (int u = 0; u < SORT_CHUNK; u++) {
      if (p0 + u * 64 < p_end) {  // wave-uniform
        const bool valid = (e[u] >= 0 && e[u] < E);
        const uint64_t mask = same_expert_mask(e[u], valid, nbits);
        if (valid && (mask & lt_mask) == 0) myhist[e[u]] += __popcll(mask);
      }
    }
  }
  __syncthreads();

  // per expert: exclusive prefix over waves (turns counts into in-expert start ranks), and totals
  for (int e = threadIdx.x; e < E; e += SORT_THREADS) {
    int run = 0;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; w++) {
      int c = hist[w * E + e];
      hist[w * E + e] = run;
      run += c;
    }
    total[e] = run;
  }
  __syncthreads();

  // expert offsets, tile list and cut positions: wave 0
  if (wave == 0)
    group_finish(total, offs, cost_pre, tile_pre, E, true, expert_offsets, tiles, rows_per_tile, xcd_bounds, cost0);
  __syncthreads();
  group_tiles(total, offs, tile_pre, E, tiles, rows_per_tile, xcd_bounds);

  for (int p0 = p_begin; p0 < p_end; p0 += 64 * SORT_CHUNK) {
    int e[SORT_CHUNK];
    load_chunk(p0, e);
#pragma unroll
    for (int u = 0; u < SORT_CHUNK; u++) {
      if (p0 + u * 64 < p_end) {
        const int p = p0 + u * 64 + lane;
        const bool valid = (e[u] >= 0 && e[u] < E);
        const uint64_t mask = same_expert_mask(e[u], valid, nbits);
        if (valid) {
          const int rank = myhist[e[u]] + __popcll(mask & lt_mask);
          const int dst = offs[e[u]] + rank;
          sorted_pair_ids[dst] = p;
          inv_perm[p] = dst;
        }
        // all lanes of the wave have read myhist before the leaders update it (wave-ordered LDS ops)
        if (valid && (mask & lt_mask) == 0) myhist[e[u]] += __popcll(mask);
      }
    }
  }
}


// ---- the same sort by many workgroups (prompt passes, large batches) ---------------------------
// One workgroup of 16 waves per 1024 pairs, one 64-pair step per wave.  First kernel: every pair's
// rank among the pairs of its expert inside its workgroup (to rank[], which may be inv_perm) and
// the workgroup's pair count per expert (wg_hist [G][E]).  Second kernel: every workgroup sums the
// counts of the workgroups before it, derives the experts' offsets and scatters its pairs;
// workgroup 0 also writes the offsets, the tile list and the cut positions.  The order inside an
// expert is (workgroup, wave, lane) = pair order, as in the one-workgroup kernel.
constexpr int SORT_PARALLEL_MIN_PAIRS = 8192;

__global__ __launch_bounds__(SORT_THREADS) void group_count_kernel(const int *__restrict__ topk_i, int P, int E,
                                                                   int nbits, int *__restrict__ wg_hist,
                                                                   int *__restrict__ rank) {
  extern __shared__ int smem[];  // [SORT_WAVES][E]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int i = threadIdx.x; i < SORT_WAVES * E; i += SORT_THREADS) smem[i] = 0;
  __syncthreads();
  const int p = blockIdx.x * SORT_THREADS + threadIdx.x;
  const int e = (p < P) ? topk_i[p] : -1;
  const bool valid = (e >= 0 && e < E);
  const uint64_t mask = same_expert_mask(e, valid, nbits);
  if (valid && (mask & lt_mask) == 0) smem[wave * E + e] = __popcll(mask);
  __syncthreads();
  for (int x = threadIdx.x; x < E; x += SORT_THREADS) {
    int run = 0;
#pragma unroll
    for (int w = 0; w < SORT_WAVES; w++) {
      const int c = smem[w * E + x];
      smem[w * E + x] = run;
      run += c;
    }
    wg_hist[(size_t)blockIdx.x * E + x] = run;
  }
  __syncthreads();
  if (valid) rank[p] = smem[wave * E + e] + __popcll(mask & lt_mask);
}

__global__ __launch_bounds__(SORT_THREADS) void group_scatter_kernel(
    const int *__restrict__ topk_i, int P, int E, const int *__restrict__ wg_hist, const int *rank,
    int *__restrict__ expert_offsets, int *__restrict__ sorted_pair_ids, int *inv_perm, int *__restrict__ tiles,
    int rows_per_tile, int *__restrict__ xcd_bounds, int cost0) {
  extern __shared__ int smem[];
  int *before = smem;          // [E] pairs of the expert in the workgroups before this one
  int *total = before + E;     // [E]
  int *offs = total + E;       // [E+1]
  int *cost_pre = offs + E + 1;
  int *tile_pre = cost_pre + E;
  const int wave = threadIdx.x >> 6;
  const int G = gridDim.x;
  for (int x = threadIdx.x; x < E; x += SORT_THREADS) {
    int run = 0, mine = 0;
    constexpr int AT_ONCE = 8;
    for (int g0 = 0; g0 < G; g0 += AT_ONCE) {
      int c[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; i++) c[i] = wg_hist[(size_t)min(g0 + i, G - 1) * E + x];
#pragma unroll
      for (int i = 0; i < AT_ONCE; i++) {
        if (g0 + i == (int)blockIdx.x) mine = run;
        run += g0 + i < G ? c[i] : 0;
      }
    }
    before[x] = mine;
    total[x] = run;
  }
  __syncthreads();
  if (wave == 0)
    group_finish(total, offs, cost_pre, tile_pre, E, blockIdx.x == 0, expert_offsets, tiles, rows_per_tile,
                 xcd_bounds, cost0);
  __syncthreads();
  if (blockIdx.x == 0) group_tiles(total, offs, tile_pre, E, tiles, rows_per_tile, xcd_bounds);
  const int p = blockIdx.x * SORT_THREADS + threadIdx.x;
  const int e = (p < P) ? topk_i[p] : -1;
  if (e >= 0 && e < E) {
    const int dst = offs[e] + before[e] + rank[p];   // rank may alias inv_perm: read before the write below
    sorted_pair_ids[dst] = p;
    inv_perm[p] = dst;
  }
}


// Gating of at most ROUTER_GROUP_TOKENS tokens from their logits (PARTS: from the router's partial products, and the logits), and
// their grouping: the end of router_gemm_kernel, for experts that several workgroups shared.
template <int NJ, bool PARTS>
__global__ __launch_bounds__(512) void topk_group_kernel(float *__restrict__ logits, RouterParts parts, int B, int E, int k,
                                                         float *__restrict__ topk_w, int *__restrict__ topk_i, RouterGroup grp) {
  __shared__ int ids[ROUTER_GROUP_PAIRS], lds[512];
  const int row = threadIdx.x >> 5, sub = threadIdx.x & 31;
  const bool live = row < B;
  float v[NJ];
  if constexpr (PARTS) {
    PartialLogit x[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) x[j].load(parts, row, sub + 32 * j);
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int e = sub + 32 * j;
      v[j] = e < E ? x[j].sum(parts) : -INFINITY;
      if (live && e < E) logits[(size_t)row * E + e] = v[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const float x = logits[(size_t)min(row, B - 1) * E + min(sub + 32 * j, E - 1)];
      v[j] = sub + 32 * j < E ? x : -INFINITY;
    }
  }
  const size_t o = (size_t)(live ? row : 0) * k;
  topk_softmax_group<NJ>(v, sub, E, k, live, topk_w + o, topk_i + o, ids + row * k);
  __syncthreads();
  if (threadIdx.x < 64) group_by_one_wave(ids, B * k, E, lds, grp);
}

// Behind a norm in the router's kernel, where no workgroup holds every token: 5.2 us by group_sort_kernel, 2.1 by one wave.
__global__ __launch_bounds__(64) void group_few_kernel(const int *__restrict__ topk_i, int P, int E, RouterGroup g) {
  __shared__ int lds[512];
  group_by_one_wave(topk_i, P, E, lds, g);
}

// gating only: logits [B,E] -> top-k weights and ids
int run_topk_softmax(const float *logits, int B, int E, int k, float *topk_w, int *topk_i, hipStream_t s) {
  dim3 grid(cdiv(B * 32, 256)), block(256);
  int nj = cdiv(E, 32);
  TraceScope ts("topk_softmax", s);
  if (k > 8) topk_softmax_kernel<8, MOE_MAX_TOP><<<grid, block, 0, s>>>(logits, B, E, k, topk_w, topk_i);
  else if (nj <= 1) topk_softmax_kernel<1><<<grid, block, 0, s>>>(logits, B, E, k, topk_w, topk_i);
  else if (nj <= 2) topk_softmax_kernel<2><<<grid, block, 0, s>>>(logits, B, E, k, topk_w, topk_i);
  else if (nj <= 4) topk_softmax_kernel<4><<<grid, block, 0, s>>>(logits, B, E, k, topk_w, topk_i);
  else topk_softmax_kernel<8><<<grid, block, 0, s>>>(logits, B, E, k, topk_w, topk_i);
  GPTOSS_LAUNCH_CHECK("topk_softmax_kernel");
  return GPTOSS_OK;
}

// Token rows of a workgroup: as few as leave no more workgroups than CUs.  Up to there their number makes little difference (2880
// inputs, 32 experts, 512 / 1024 tokens in groups of four 5.5 / 5.9 us, of eight 5.5 / 5.6, of 16 5.4 / 5.5), because a workgroup takes the time
// of its experts' weights whatever its rows are; beyond it they come in rounds: 1400 tokens, 32 / 128 experts, 7.6 / 23.6, 5.7 / 12.6 and
// 5.6 / 12.6, 3000 11.0 / 34.4, 8.0 / 23.8 and 6.1 / 13.1.
static int router_rows_per_wg(int B) {
  int rows_per_wg = 4;
  while (rows_per_wg < 16 && cdiv(B, rows_per_wg) > 256) rows_per_wg *= 2;
  return rows_per_wg;
}
// With the norm in front (norm_router_applies): two rows at a time by a workgroup, so four even where that is more of them.
static int norm_router_rows_per_wg(int B) {
  int rows_per_wg = 16;
  while (rows_per_wg > 4 && cdiv(B, rows_per_wg) < 256) rows_per_wg >>= 1;
  return rows_per_wg;
}

// 16-expert column blocks of the kernel instance that holds all experts
static int router_col_blocks(int E) {
  const int nb = cdiv(E, 16);
  return nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : nb <= 8 ? 8 : 16;
}

// Whether a workgroup takes 16 experts instead of all of them.  That saves the loads and the parts of a stage one behind the other
// (router_gemm_kernel) and costs a second launch, which gates (up to 16 tokens: and groups).  MoE block with narrow experts, all
// experts in one workgroup -> shared out, us:
//   more than 128 experts  2880 inputs, 256 experts, 17 / 512 tokens 77.4 / 168 -> 61.6 / 148, 1024 41.6 / 66.7 -> 35.0 / 61.9, 512 28.3 / 37.7
//                          -> 25.5 / 35.4, 256 26.7 / 32.5 -> 25.1 / 31.4, 64 24.0 / 25.2 -> 22.8 / 24.9; 192 of 512 28.2 / 37.4 -> 25.5 / 35.2
//   65 to 128              2880 inputs, 128 experts 46.4 / 97.7 -> 40.4 / 90.4, 1024 27.2 / 44.2 -> 25.5 / 42.6, 96 experts 27.3 / 43.6 -> 26.0 /
//                          42.2, 512 24.4 / 33.4 -> 24.0 / 33.1; but 256 23.6 / 28.6 -> 23.8 / 29.4
//   33 to 64               4096 inputs, 64 experts 46.1 / 88.2 -> 44.3 / 85.4, 2880 37.8 / 73.0 -> 36.9 / 71.3, 33 experts 35.8 / 68.4 -> 34.4 /
//                          67.6; but 2048, 48 experts 30.6 / 49.2 -> 30.4 / 49.3, 1792, 49 30.1 / 48.3 -> 30.1 / 48.6, 1024, 64 24.2 / 35.7 ->
//                          24.8 / 36.5, 512 22.0 / 31.4 -> 22.9 / 32.3
// Up to 512 tokens: at 1000 it is 0 to 5 % (256 experts of 64 inputs, 1500 / 4000 tokens 26.9 / 33.9 -> 29.2 / 39.7).
static bool router_splits(int B, int H, int E) { return E > 32 && B <= 512 && (E > 128 || H >= (E > 64 ? 512 : 2112)); }

// Rows of a workgroup of 16 experts: as few as leave no more than a workgroup per CU.  Up to there their number makes no difference
// (logits of 1 to 100 tokens over 64 to 128 experts of 1024 and 2880 inputs within 4 % with 4, 8 or 16), beyond it they come in rounds: 128
// experts of 2880 inputs, 256 / 512 / 1024 tokens in groups of four 5.9 / 10.5 / 18.2 us, of eight 4.6 / 5.9 / 10.1, of 16 4.5 / 4.7 / 6.2.
static int router_split_rows(int B, int E) {
  int rows = 4;
  while (rows < 16 && cdiv(B, rows) * cdiv(E, 16) > 256) rows *= 2;
  return rows;
}

int run_router_parts(const void *t, const void *w_router, float *parts, int B, int H, int E, hipStream_t s) {
  GPTOSS_REQUIRE(B >= 1 && B <= ROUTER_GROUP_TOKENS, GPTOSS_ERR_DIM, "router: no partial products of %d tokens", B);
  TraceScope ts("router_parts", s);
  router_parts_kernel<false><<<dim3(ROUTER_WAVES, cdiv(E, 16)), 64, 0, s>>>((const bf16_t *)t, (const bf16_t *)w_router, parts, B, H, E, RouterNorm{});
  GPTOSS_LAUNCH_CHECK("router_parts_kernel");
  return GPTOSS_OK;
}

bool norm_router_parts_apply(int B, int H, const float *x, const float *residual, const float *weight, const void *t_out) {
  return B >= 1 && B <= ROUTED_TOKENS && H % 32 == 0 && H <= 4096 && aligned(x, 16) && aligned(weight, 16) && aligned(t_out, 16) &&
         (!residual || aligned(residual, 16));
}

int run_norm_router_parts(const float *x, const float *residual, const float *weight, void *t_out, const void *w_router,
                          float *parts, int B, int H, int E, hipStream_t s) {
  GPTOSS_REQUIRE(norm_router_parts_apply(B, H, x, residual, weight, t_out), GPTOSS_ERR_DIM,
                 "norm + router: no partial products of this form (B=%d H=%d)", B, H);
  TraceScope ts("norm_router_parts", s);
  const RouterNorm nrm{const_cast<float *>(x), residual, weight, (bf16_t *)t_out};
  router_parts_kernel<true><<<dim3(ROUTER_WAVES, cdiv(E, 16)), B == 1 ? 256 : 512, (size_t)B * H * 2, s>>>(
      nrm.t_out, (const bf16_t *)w_router, parts, B, H, E, nrm);
  GPTOSS_LAUNCH_CHECK("router_parts_kernel (with norm)");
  return GPTOSS_OK;
}

template <int NB, bool LARGE>
static int launch_router_rows(const bf16_t *t, const bf16_t *wr, const float *br, float *logits, int B, int H, int E, int k,
                         float *topk_w, int *topk_i, int rows_per_wg, int shares, const RouterGroup &grp, hipStream_t s) {
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static bool raised[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "router: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  auto kern = router_gemm_kernel<NB, LARGE>;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!raised[dev]) {
      GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     RouterStages<NB>::SMEM));
      raised[dev] = true;
    }
  }
  hipLaunchKernelGGL(kern, dim3(cdiv(B, rows_per_wg), shares), dim3(ROUTER_WAVES * 64), RouterStages<NB>::SMEM, s, t, wr, br, logits, B, H, E,
                     k, topk_w, topk_i, rows_per_wg, grp);
  GPTOSS_LAUNCH_CHECK("router_gemm_kernel");
  return GPTOSS_OK;
}
template <int NB, class... Args>
static int launch_router(const bf16_t *t, const bf16_t *wr, const float *br, float *logits, int B, int H, int E, const Args &...more) {
  const bool large = (size_t)std::max(E, 16) * H * 2 > (1ull << 32);
  return (large ? launch_router_rows<NB, true> : launch_router_rows<NB, false>)(t, wr, br, logits, B, H, E, more...);
}

// logits (+ optional gating of the same tokens), in one launch unless many experts are shared out and gated as well
int run_router(const void *t, const void *w_router, const float *b_router, float *logits, int B,
               int H, int E, int k, float *topk_w, int *topk_i, hipStream_t s, const RouterGroup *group, float *parts) {
  const RouterGroup grp = group ? *group : RouterGroup{};
  const int rows_per_wg = grp.expert_offsets ? ROUTER_GROUP_TOKENS : router_rows_per_wg(B);
  GPTOSS_REQUIRE(!grp.expert_offsets || (topk_w && router_groups(B, k)), GPTOSS_ERR_DIM, "router: %d tokens are not grouped here", B);
  const bf16_t *tp = (const bf16_t *)t, *wp = (const bf16_t *)w_router;
  int nb = cdiv(E, 16);
  if (topk_w && k > 8) {   // more experts per token than the fused gating holds
    const int rc = run_router(t, w_router, b_router, logits, B, H, E, k, nullptr, nullptr, s);
    return rc != GPTOSS_OK ? rc : run_topk_softmax(logits, B, E, k, topk_w, topk_i, s);
  }
  // Few tokens: the products of a kernel of their own for any number of experts, one launch more for those that one workgroup had.
  // The whole block, us: 32 experts, 5 / 16 tokens 53.4 / 84.2 -> 49.6 / 78.6 (MXFP4, 2880 x 2880), 21.2 / 27.1 -> 17.4 / 22.6 (640 x
  // 256); 128 61.9 / 126.7 -> 59.4 / 123.9; 256 of 1024 inputs 24.4 / 30.7 -> 22.5 / 29.3; 16 of 4096 32.9 / 41.5 -> 28.6 / 32.4; four and eight
  // from eight tokens on: 42.5 / 53.5 -> 43.9 / 51.7 and 27.9 / 36.0 -> 28.1 / 34.2.
  if (grp.expert_offsets && parts && topk_w && (E >= 16 || B >= 8)) {
    int rc = run_router_parts(t, w_router, parts, B, H, E, s);
    if (rc != GPTOSS_OK) return rc;
    const RouterParts rp{parts, b_router, B, E, k};
    TraceScope ts("topk_group", s);
    auto launch = [&](auto kern) { kern<<<1, 512, 0, s>>>(logits, rp, B, E, k, topk_w, topk_i, grp); };
    if (nb <= 2) launch(topk_group_kernel<1, true>);
    else if (nb <= 4) launch(topk_group_kernel<2, true>);
    else if (nb <= 8) launch(topk_group_kernel<4, true>);
    else launch(topk_group_kernel<8, true>);
    GPTOSS_LAUNCH_CHECK("topk_group_kernel");
    return GPTOSS_OK;
  }
  if (router_splits(B, H, E) && topk_w) {
    const int rows = router_split_rows(B, E);
    {
      TraceScope ts("router_gemm", s);
      const int rc = launch_router<1>(tp, wp, b_router, logits, B, H, E, k, nullptr, nullptr, rows, nb, RouterGroup{}, s);
      if (rc != GPTOSS_OK) return rc;
    }
    if (!grp.expert_offsets) return run_topk_softmax(logits, B, E, k, topk_w, topk_i, s);
    TraceScope ts("topk_group", s);
    auto launch = [&](auto kern) { kern<<<1, 512, 0, s>>>(logits, RouterParts{}, B, E, k, topk_w, topk_i, grp); };
    // (up to 64 experts are shared out only with so many inputs that the products have room as parts)
    if (nb <= 8) launch(topk_group_kernel<4, false>);
    else launch(topk_group_kernel<8, false>);
    GPTOSS_LAUNCH_CHECK("topk_group_kernel");
    return GPTOSS_OK;
  }
  TraceScope ts(topk_w ? "router_gemm_topk" : "router_gemm", s);
  // Logits alone need no launch more for experts that are shared out: up to 1024 tokens that is the faster form at every size (us, one
  // workgroup for all -> shared out: 80 experts of 96 inputs, 9 tokens 3.6 -> 2.3; 136 of 288, 513 tokens 6.6 -> 3.0; 64 of 2880, 1024
  // tokens 7.5 -> 4.7; 256 of 2880, 1 / 1024 tokens 20.7 / 23.4 -> 4.2 / 11.7).  Beyond, each share reads the tokens again: 1025 tokens over
  // 64 of 7168 13.4 -> 15.3, 2000 over 256 of 1024 10.5 -> 11.8.
  if (!topk_w && E > 32 && B <= 1024)
    return launch_router<1>(tp, wp, b_router, logits, B, H, E, k, nullptr, nullptr, router_split_rows(B, E), nb, RouterGroup{}, s);
  if (nb <= 1) return launch_router<1>(tp, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, 1, grp, s);
  if (nb <= 2) return launch_router<2>(tp, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, 1, grp, s);
  if (nb <= 4) return launch_router<4>(tp, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, 1, grp, s);
  if (nb <= 8) return launch_router<8>(tp, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, 1, grp, s);
  return launch_router<16>(tp, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, 1, grp, s);
}


template <int NB>
static int launch_norm_router(const RouterNorm &nrm, const bf16_t *wp, const float *b_router, float *logits, int B, int H,
                              int E, int k, float *topk_w, int *topk_i, int rows_per_wg, size_t dyn, hipStream_t s,
                              const RouterGroup &grp) {
  // the kernel's LDS (router partial sums + the rows of t) exceeds what a launch gets by default
  constexpr int MAX_DEV = 64;
  static std::mutex mu;
  static size_t raised[MAX_DEV];
  int dev = 0;
  GPTOSS_HIP(hipGetDevice(&dev));
  GPTOSS_REQUIRE(dev >= 0 && dev < MAX_DEV, GPTOSS_ERR_STATE, "router: device ordinal %d outside 0..%d", dev, MAX_DEV - 1);
  auto kern = norm_router_kernel<NB>;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (raised[dev] < dyn) {
      GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)dyn));
      raised[dev] = dyn;
    }
  }
  TraceScope ts("norm_router_gemm_topk", s);
  hipLaunchKernelGGL(kern, dim3(cdiv(B, rows_per_wg)), dim3(ROUTER_WAVES * 64), dyn, s, wp, b_router, logits, B, H,
                     E, k, topk_w, topk_i, rows_per_wg, nrm, grp);
  GPTOSS_LAUNCH_CHECK("norm_router_kernel");
  return GPTOSS_OK;
}

// Whether a norm in front of more than 32 experts is a kernel of its own.  Behind it in one kernel (norm_router_kernel) all experts'
// loads come in operand order, in rounds; behind one of its own the router takes either form.  Block with narrow experts, one kernel ->
// two and shared out, us: 2880 inputs, 64 experts, 512 tokens 80.2 -> 71.3, 128 104 -> 87.0; one round: 1024 inputs, 64 experts, 256
// tokens 36.3 -> 34.3, 33 experts 35.9 -> 36.6, 96 experts, 400 tokens 44.5 -> 46.0, 512 inputs, 192 experts, 400 tokens 38.1 -> 43.1.
static bool norm_apart(int B, int H, int E) {
  if (E <= 32) return false;
  const bool one_round = H / 32 <= ROUTER_WAVES * router_steps(router_col_blocks(E));
  return one_round ? E > 48 && H >= 256 && B <= 256 : B <= 512;
}

bool norm_router_applies(int B, int H, int E, const float *x, const float *residual, const float *weight,
                         const void *t_out) {
  const int nb = router_col_blocks(E);
  const size_t lds = (size_t)ROUTER_WAVES * 16 * (nb * 16 + 1) * 4 + (size_t)norm_router_rows_per_wg(B) * H * 2 + 640;   // (and the pair ids)
  // With more than four rows per workgroup (batches of more than ~1000 rows) the rows a workgroup
  // normalises one after the other cost more than the launch the fusion saves (8192 rows: 2.58 ms
  // per 24 layers against 2.23 ms for the two kernels; 1024 rows: 0.63 against 0.71 ms).
  return B > 0 && !norm_apart(B, H, E) && norm_router_rows_per_wg(B) <= 4 && H % 32 == 0 && H <= 4096 && lds <= 160 * 1024 && aligned(x, 16) && aligned(weight, 16) &&
         aligned(t_out, 16) && (!residual || aligned(residual, 16));
}

// x += residual; t_out = RMSNorm(x) * weight; logits = t_out . Wr^T + br; gating: one launch
int run_norm_router(float *x, const float *residual, const float *weight, void *t_out, const void *w_router,
                    const float *b_router, float *logits, int B, int H, int E, int k, float *topk_w, int *topk_i,
                    hipStream_t s, const RouterGroup *group) {
  const RouterGroup grp = group ? *group : RouterGroup{};
  GPTOSS_REQUIRE(!grp.expert_offsets || (router_groups(B, k) && B <= ROUTER_GROUP_NORM_TOKENS), GPTOSS_ERR_DIM,
                 "norm + router: %d tokens are not grouped here", B);
  GPTOSS_REQUIRE(norm_router_applies(B, H, E, x, residual, weight, t_out), GPTOSS_ERR_DIM,
                 "norm + router: shape or alignment outside the fused kernel's range (H=%d E=%d)", H, E);
  // A workgroup norms two rows at a time, so up to 512 rows are two each, unless one workgroup groups them all: with four,
  // 4 experts, 6 / 33 / 500 rows 7.4 / 7.6 / 8.7 us, with two 5.8 / 5.9 / 7.2; 32 experts 11.6 / 11.9 / 12.9 and 10.1 /
  // 10.2 / 11.4.
  const bool grouped = group && group->expert_offsets;
  const int rows_per_wg = !grouped && cdiv(B, 2) <= 256 ? 2 : norm_router_rows_per_wg(B);
  const RouterNorm nrm{x, residual, weight, (bf16_t *)t_out};
  const bf16_t *wp = (const bf16_t *)w_router;
  const size_t dyn = (size_t)rows_per_wg * H * 2;
  const int nb = cdiv(E, 16);
  if (nb <= 1) return launch_norm_router<1>(nrm, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, dyn, s, grp);
  if (nb <= 2) return launch_norm_router<2>(nrm, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, dyn, s, grp);
  if (nb <= 4) return launch_norm_router<4>(nrm, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, dyn, s, grp);
  if (nb <= 8) return launch_norm_router<8>(nrm, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, dyn, s, grp);
  return launch_norm_router<16>(nrm, wp, b_router, logits, B, H, E, k, topk_w, topk_i, rows_per_wg, dyn, s, grp);
}

}  // namespace gptoss

using namespace gptoss;

extern "C" int gptoss_router_gemm(const void *t, const void *w_router, const float *b_router,
                                  float *logits, int B, int H, int E, void *stream) {
  GPTOSS_REQUIRE(t && w_router && logits, GPTOSS_ERR_NULL, "router_gemm: null pointer");
  GPTOSS_REQUIRE(B >= 0 && H > 0 && H % 32 == 0 && E >= 1 && E <= 256, GPTOSS_ERR_DIM,
                 "router_gemm: need H %% 32 == 0 and 1 <= E <= 256 (B=%d H=%d E=%d)", B, H, E);
  GPTOSS_REQUIRE(aligned(t, 16) && aligned(w_router, 16), GPTOSS_ERR_ALIGN,
                 "router_gemm: t and w_router must be 16-byte aligned");
  if (B == 0) return GPTOSS_OK;
  return run_router(t, w_router, b_router, logits, B, H, E, 0, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int gptoss_moe_max_tiles(int B, int k, int E, int rows_per_tile) {
  if (rows_per_tile <= 0 || B < 0 || k <= 0 || E <= 0) return 0;
  long long P = (long long)B * k;
  return (int)(P / rows_per_tile) + E;
}

static int moe_route_impl(const float *logits, int B, int E, int k, float *topk_w, int *topk_i,
                          int *expert_offsets, int *sorted_pair_ids, int *inv_perm, int *tiles,
                          int rows_per_tile, int *xcd_bounds, int tile_cost0_x2, void *stream, bool gate,
                          int *sort_scratch);

// grouping only: topk_i was already written by the fused router kernel
int gptoss::run_group(int B, int E, int k, float *topk_w, int *topk_i, int *expert_offsets,
                      int *sorted_pair_ids, int *inv_perm, int *tiles, int rows_per_tile,
                      int *xcd_bounds, int tile_cost0_x2, hipStream_t s, int *sort_scratch) {
  // the cut positions hold the tile index in 15 bits
  if (gptoss_moe_max_tiles(B, k, E, rows_per_tile) >= 32768) xcd_bounds = nullptr;
  if (B > 0 && router_groups(B, k) && xcd_bounds && tiles && rows_per_tile >= ROUTER_GROUP_TOKENS && E >= 1 && E <= 256) {
    RouterGroup g;
    g.expert_offsets = expert_offsets;
    g.sorted_pair_ids = sorted_pair_ids;
    g.inv_perm = inv_perm;
    g.tiles = tiles;
    g.xcd_bounds = xcd_bounds;
    g.nbits = 0;
    while ((1 << g.nbits) < E) g.nbits++;
    TraceScope ts("group_sort", s);
    group_few_kernel<<<1, 64, 0, s>>>(topk_i, B * k, E, g);
    GPTOSS_LAUNCH_CHECK("group_few_kernel");
    return GPTOSS_OK;
  }
  return moe_route_impl(nullptr, B, E, k, topk_w, topk_i, expert_offsets, sorted_pair_ids, inv_perm,
                        tiles, rows_per_tile, xcd_bounds, tile_cost0_x2, s, false, sort_scratch);
}

extern "C" int gptoss_moe_route(const float *logits, int B, int E, int k, float *topk_w,
                                int *topk_i, int *expert_offsets, int *sorted_pair_ids,
                                int *inv_perm, int *tiles, int rows_per_tile, void *stream) {
  return moe_route_impl(logits, B, E, k, topk_w, topk_i, expert_offsets, sorted_pair_ids, inv_perm,
                        tiles, rows_per_tile, nullptr, 0, stream, true, nullptr);
}

static int moe_route_impl(const float *logits, int B, int E, int k, float *topk_w, int *topk_i,
                          int *expert_offsets, int *sorted_pair_ids, int *inv_perm, int *tiles,
                          int rows_per_tile, int *xcd_bounds, int tile_cost0_x2, void *stream, bool gate,
                          int *sort_scratch) {
  GPTOSS_REQUIRE(expert_offsets, GPTOSS_ERR_NULL, "moe_route: null pointer");
  GPTOSS_REQUIRE(B <= 0 || ((logits || !gate) && topk_w && topk_i && sorted_pair_ids && inv_perm),
                 GPTOSS_ERR_NULL, "moe_route: null pointer");
  const int max_top = gate ? 8 : MOE_MAX_TOP;
  GPTOSS_REQUIRE(E >= 1 && E <= 256 && k >= 1 && k <= max_top && k <= E && B >= 0, GPTOSS_ERR_DIM,
                 "moe_route: need 1 <= k <= min(%d,E), E <= 256 (B=%d E=%d k=%d)", max_top, B, E, k);
  GPTOSS_REQUIRE((long long)B * k < (1ll << 30), GPTOSS_ERR_DIM, "moe_route: B*k too large");
  bool tile_ok = rows_per_tile >= 0 && rows_per_tile <= 256 && rows_per_tile % 32 == 0;
  GPTOSS_REQUIRE(tile_ok, GPTOSS_ERR_DIM, "moe_route: rows_per_tile must be 0 or a multiple of 32 up to 256");
  GPTOSS_REQUIRE(rows_per_tile == 0 || tiles, GPTOSS_ERR_NULL, "moe_route: tiles is NULL");
  hipStream_t s = (hipStream_t)stream;
  if (B > 0 && gate) {
    int rc = run_topk_softmax(logits, B, E, k, topk_w, topk_i, s);
    if (rc != GPTOSS_OK) return rc;
  }
  int nbits = 0;
  while ((1 << nbits) < E) nbits++;
  size_t smem = sizeof(int) * ((size_t)SORT_WAVES * E + E + (E + 1) + 2 * (size_t)E);
  const int P = B * k;
  if (sort_scratch != nullptr && P >= SORT_PARALLEL_MIN_PAIRS) {
    const int G = cdiv(P, SORT_THREADS);
    TraceScope ts("group_sort", s);
    group_count_kernel<<<G, SORT_THREADS, sizeof(int) * SORT_WAVES * E, s>>>(topk_i, P, E, nbits, sort_scratch,
                                                                           inv_perm);
    GPTOSS_LAUNCH_CHECK("group_count_kernel");
    group_scatter_kernel<<<G, SORT_THREADS, sizeof(int) * (5 * (size_t)E + 1), s>>>(
        topk_i, P, E, sort_scratch, inv_perm, expert_offsets, sorted_pair_ids, inv_perm,
        rows_per_tile ? tiles : nullptr, rows_per_tile, xcd_bounds, tile_cost0_x2);
    GPTOSS_LAUNCH_CHECK("group_scatter_kernel");
    return GPTOSS_OK;
  }
  {
    TraceScope ts("group_sort", s);
    group_sort_kernel<<<1, SORT_THREADS, smem, s>>>(topk_i, B * k, E, nbits, expert_offsets,
                                                    sorted_pair_ids, inv_perm,
                                                    rows_per_tile ? tiles : nullptr, rows_per_tile,
                                                    xcd_bounds, tile_cost0_x2);
  }
  GPTOSS_LAUNCH_CHECK("group_sort_kernel");
  return GPTOSS_OK;
}
