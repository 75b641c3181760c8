// Host side of the MoE block: workspace layout and the launch sequence
// router GEMM -> top-k/softmax -> stable grouping + tile list -> grouped GEMM1 (+gather, +SwiGLU)
// -> grouped GEMM2 -> ordered weighted combine.  Nothing here synchronises or allocates.
#include <math.h>
#include <stdlib.h>

#include <algorithm>

#include "common.hpp"
#include "gemm.hpp"
#include "glue.hpp"

namespace gptoss {

struct MoeWorkspace {
  float *logits, *topk_w;
  int *topk_i, *expert_offsets, *sorted_pair_ids, *inv_perm, *tiles, *xcd_bounds, *sort_scratch;
  bf16_t *act;
  float *y2;
  size_t bytes;
};

static MoeWorkspace carve(void *base, int B, int E, int k, int H, int I) {
  MoeWorkspace w;
  size_t off = 0;
  auto take = [&](size_t n) {
    size_t o = off;
    off += align_up(n, 256);
    return reinterpret_cast<unsigned char *>(base) + o;
  };
  const size_t P = (size_t)B * k;
  w.logits = (float *)take((size_t)B * E * 4);
  w.topk_w = (float *)take(P * 4);
  w.topk_i = (int *)take(P * 4);
  w.expert_offsets = (int *)take((size_t)(E + 1) * 4);
  w.sorted_pair_ids = (int *)take(P * 4);
  w.inv_perm = (int *)take(P * 4);
  w.tiles = (int *)take((1 + 3 * (P / 32 + E)) * 4);
  w.xcd_bounds = (int *)take((XCD_BOUNDS_INTS + P / 32 + E) * 4);
  w.sort_scratch = (int *)take(group_sort_scratch_ints(B, k, E) * 4);
  w.act = (bf16_t *)take(P * I * 2);
  w.y2 = (float *)take(P * H * 4);
  w.bytes = off;
  return w;
}

// Row-tile size for B*k pairs over E experts.
// bf16 weights (32, 64, 128 or 160 rows): the smallest tile that holds an average expert's rows
// plus 2.5 standard deviations of a uniform routing, so that nearly every expert is a single tile
// and its weights are streamed exactly once; the kernel is bound by that stream.
// MXFP4 weights (32 or 64 rows): tiles of at most 64 rows, three or four workgroups of which share a CU
// (gemm_mxfp4_kernel.hpp); an expert's few row tiles are walked column tile by column tile
// (tile_block), so its weights still come from HBM once.
static int env_int(const char *name, int dflt) {
  const char *e = getenv(name);
  const int n = e ? atoi(e) : 0;
  return n > 0 ? n : dflt;
}
// Whether a bf16 MoE block uses the 256-row kernels of gemm_tall.hip, by its average rows per expert.
// From 416 on they gain 2-23 % (both routings, uniform and Zipf 1.1; 2880 x 2880, 32 experts of 437 rows 877 -> 790 us) where there
// is work for the whole chip: blocks of 1024 x 512 on 16 experts lose 13 %, blocks of four times the arithmetic gain, so small ones
// from 512 on.
// From 165 to 248 an expert's rows are two 160-row tiles and one of 256, but only while the routing is uniform (2880 x 2880, 32
// experts, uniform / Zipf 0.6 / 1.1, streaming kernels = 1: 165 rows 0.90 / 1.03 / 1.05, 177 0.85 / 1.07 / 1.06, 189 0.84 / 1.08 /
// 1.05, 201 0.82 / 1.03 / 1.05, 213 0.85 / 1.04 / 1.01, 225 0.87 / 1.03 / 0.98, 243 0.92 / 1.02 / 0.99; 500 us at 177, 560 at 213).  So
// from 213 on, where preferences like a trained router's lose nothing, and with as much arithmetic as that: of smaller blocks those
// lose up to 18 %, of 7 sizes beyond the line uniform routings gain 5 to 16 %, Zipf 0.6 and 1.1 1 % on average, at most 3 % lost.
// Where every token takes every expert, so that no expert has more rows than another, from 165 on and with 40 % of that arithmetic.
// Above 248 two tiles of either (275 rows 692 / - / 737 -> 790 / - / 704 us, 325 837 / - / 802 -> 861 / - / 784).
static int moe_tall_forced() {
  static const int v = env_int("GPTOSS_MOE_TALL_MIN_ROWS", 0);
  return v;
}
static bool moe_tall(long long pairs, int E, int k, int N, int K) {
  if (const int v = moe_tall_forced()) return pairs >= (long long)v * E;
  const double work = (double)pairs * N * K;
  if (pairs >= (long long)(work >= (double)(1ll << 34) ? 416 : 512) * E) return true;
  return work >= (k == E ? 2.0 : 5.0) * (1ll << 34) && pairs >= (k == E ? 165ll : 213ll) * E && pairs <= 248ll * E;
}

int moe_rows_per_tile(int B, int k, int E, bool mxfp4) {
  double avg = (double)B * k / E;
  // Every token on every expert: nothing to deviate.  Short of that the deviation is sqrt(avg (1 - k / E)), but a margin cut
  // to that is too small: 380 tokens, 4 of 32 experts, 312 -> 361 us with tiles of 64; 166 tokens, 2 of 16, 74 -> 81.
  double need = k == E ? avg : avg + 2.5 * sqrt(avg);

  if (need <= 32) return 32;
  if (need <= 64) return 64;
  if (mxfp4) return 64;
  if (need <= 128) return 128;
  return 160;
}

// Row tiles of E experts with `avg` rows each on average, spread as a uniform routing spreads them.
static double expected_tiles(int k, int E, double avg, int rows_per_tile) {
  if (k == E) return E * ceil(avg / rows_per_tile);
  const double s = sqrt(2 * avg * (1 - (double)k / E));
  double n = 1;
  for (int m = 1; m * rows_per_tile <= 2 * avg + 64; m++) n += 0.5 * erfc((m * rows_per_tile + 0.5 - avg) / s);
  return E * n;
}

// The row tile of a bf16 block, given the one that holds an expert's rows: where tiles of that size are work for fewer than two
// rounds of the CUs, the one that makes both products shortest by the estimates of gemm_dense.cpp.  Smaller tiles put more
// CUs to work (an item of 160 rows is a CU's for 20 to 50 us), and where every token takes every expert, so that the tiles are known,
// 256 rows may save a round.  Blocks in us, before -> after: 4 of 4 experts, 2048 x 1024, 70 / 135 / 240 rows each 61 / 73 / 75 -> 39 / 42 /
// 44, 2880 x 2880, 100 / 330 rows 102 / 192 -> 82 / 131; 4 of 16, 1024 x 512, 60 / 200 rows 45 / 61 -> 35 / 51; two of 4, 4096 x 1536, 70 rows
// 93 -> 64.
// Every token on every expert: it has to be ahead by 11 %, the estimates' error.  Of 890 blocks of random sizes none takes more than 2 %
// longer; ahead by a tenth, 70 rows of 2816 x 4800 on five lose 3 %, and by 15 %, 21 blocks do without what they gain, four experts of 165 to 190
// rows, 2880 x 2880, 177 -> 105 us.
// Experts that are chosen: by a quarter, and by 12 % with a fifth more tiles than a uniform routing makes (or as many as there can be): 6
// experts of 106 rows of 2624 x 2688 have 12 tiles of 64, one round of the CUs, or 13, and two.  Below 64 rows on average the default's tiles
// are mostly of no more blocks than one of 64 rows, and cost no more: there by a quarter as well with those more.  188 blocks that the first
// condition alone sends to other tiles, uniform, Zipf 0.6 and 1.1: half of them are sent there, 20 % faster on average, at worst 3 % slower; all of them,
// 12 %, and up to 21 %.
static int small_block_rows(int dflt, int B, int k, int E, int H, int I, bool tall) {
  const double avg = (double)B * k / E;
  if (dflt <= 64 || dflt == 256 || expected_tiles(k, E, avg, dflt) * gemm_col_tiles(2 * I) >= 512) return dflt;
  auto us = [&](int rpt, double more) {
    const int max_tiles = gptoss_moe_max_tiles(B, k, std::min(E, B * k), rpt);
    const double expected = expected_tiles(k, E, avg, rpt), tiles = std::min(expected * more, std::max(expected, (double)max_tiles));
    return grouped_us(rpt, tiles, grouped_few(rpt, max_tiles, 2 * I), 2 * I, H) + grouped_us(rpt, tiles, grouped_few(rpt, max_tiles, H), H, I);
  };
  int best = dflt;
  const double dflt_us = us(dflt, 1.0), at_most = (avg >= 64 ? 0.88 : 0.75) * dflt_us;
  double least = (k == E ? 0.89 : 0.75) * dflt_us;
  for (int rpt : {32, 64, 128, 160, 256}) {
    // (tiles of 32 rows read the weights again and again: not beyond two rounds of the few-row kernels)
    if ((rpt == 256 && (!tall || k != E)) || (rpt == 32 && expected_tiles(k, E, avg, 32) * (2 * I / 32) > 2560)) continue;
    const double t = us(rpt, 1.0);
    if (t < least && (k == E || us(rpt, 1.2) < at_most)) {
      least = t;
      best = rpt;
    }
  }
  return best;
}

// Fixed part of a work item's cost, in half units of one 32-row block of arithmetic, used to cut
// the work list into 8 equally expensive parts.  With bf16 weights an item is dominated by
// streaming its 1.5 MB of W whatever its row count (16 + blocks); with MXFP4 weights, a quarter of
// the bytes, the arithmetic weighs more (5 + blocks).  Both constants are the measured optimum on a
// Zipf-skewed routing; a uniform routing is indifferent to them.
constexpr int MOE_TILE_COST0_X2_BF16 = 32;
constexpr int MOE_TILE_COST0_X2_MXFP4 = 10;

static int check_moe(const gptoss_moe_weights *w, const void *t, int B, float *out, void *ws,
                     size_t ws_bytes, int max_top) {
  GPTOSS_REQUIRE(w && t && out, GPTOSS_ERR_NULL, "moe_forward: null pointer");
  GPTOSS_REQUIRE(w->w_router && w->w1 && w->w2, GPTOSS_ERR_NULL, "moe_forward: null weight pointer");
  const int E = w->n_experts, k = w->top_k, H = w->hidden, I = w->intermediate;
  GPTOSS_REQUIRE(B >= 0 && E >= 1 && E <= 256 && k >= 1 && k <= max_top && k <= E, GPTOSS_ERR_DIM,
                 "moe_forward: need 1 <= k <= min(%d,E), E <= 256 (B=%d E=%d k=%d)", max_top, B, E, k);
  GPTOSS_REQUIRE(aligned(t, 16), GPTOSS_ERR_ALIGN, "moe_forward: t must be 16-byte aligned");
  GPTOSS_REQUIRE(H > 0 && I > 0 && H % 64 == 0 && I % 64 == 0, GPTOSS_ERR_DIM,
                 "moe_forward: need hidden %% 64 == 0 and intermediate %% 64 == 0 (H=%d I=%d)", H, I);
  GPTOSS_REQUIRE((long long)B * k * (long long)(H > I ? H : I) < (1ll << 31), GPTOSS_ERR_DIM,
                 "moe_forward: B*k*max(H,I) must stay below 2^31");
  GPTOSS_REQUIRE(aligned(t, 16) && aligned(out, 16) && aligned(w->w1, 16) && aligned(w->w2, 16) &&
                     aligned(w->w_router, 16),
                 GPTOSS_ERR_ALIGN, "moe_forward: pointers must be 16-byte aligned");
  GPTOSS_REQUIRE(ws != nullptr && aligned(ws, 256), GPTOSS_ERR_WORKSPACE,
                 "moe_forward: workspace missing or not 256-byte aligned");
  size_t need = gptoss_moe_workspace_bytes(B, E, k, H, I);
  GPTOSS_REQUIRE(ws_bytes >= need, GPTOSS_ERR_WORKSPACE,
                 "moe_forward: workspace has %zu bytes, needs %zu", ws_bytes, need);
  return GPTOSS_OK;
}

}  // namespace gptoss

using namespace gptoss;

extern "C" size_t gptoss_moe_workspace_bytes(int B, int E, int k, int H, int I) {
  if (B < 0 || E <= 0 || k <= 0 || H <= 0 || I <= 0) return 0;
  return carve(nullptr, B, E, k, H, I).bytes;
}

extern "C" int gptoss_moe_workspace_views(void *workspace, int B, int E, int k, int H, int I,
                                          float **logits, float **topk_w, int **topk_i,
                                          int **expert_offsets, int **sorted_pair_ids,
                                          int **inv_perm) {
  GPTOSS_REQUIRE(workspace, GPTOSS_ERR_NULL, "moe_workspace_views: null workspace");
  GPTOSS_REQUIRE(B >= 0 && E > 0 && k > 0 && H > 0 && I > 0, GPTOSS_ERR_DIM,
                 "moe_workspace_views: bad dimensions");
  MoeWorkspace w = carve(workspace, B, E, k, H, I);
  if (logits) *logits = w.logits;
  if (topk_w) *topk_w = w.topk_w;
  if (topk_i) *topk_i = w.topk_i;
  if (expert_offsets) *expert_offsets = w.expert_offsets;
  if (sorted_pair_ids) *sorted_pair_ids = w.sorted_pair_ids;
  if (inv_perm) *inv_perm = w.inv_perm;
  return GPTOSS_OK;
}

static int moe_forward_impl(const gptoss_moe_weights *w, const void *t, int B, float *out,
                            int accumulate, void *workspace, size_t workspace_bytes, void *stream,
                            int mxfp4, const float *norm_w = nullptr, bf16_t *norm_out = nullptr,
                            const MoePreNorm *pre = nullptr, const GluForm *glu = nullptr,
                            const TanhNorm *tanh_norm = nullptr) {
  int rc = check_moe(w, t, B, out, workspace, workspace_bytes, glu ? MOE_MAX_TOP : 8);
  if (rc != GPTOSS_OK) return rc;
  if (B == 0) return GPTOSS_OK;
  const int E = w->n_experts, k = w->top_k, H = w->hidden, I = w->intermediate;
  hipStream_t s = (hipStream_t)stream;
  MoeWorkspace ws = carve(workspace, B, E, k, H, I);
  int rpt = moe_rows_per_tile(B, k, E, mxfp4 != 0);
  // a prompt pass, hundreds of rows per expert: bound by the matrix cores, not by streaming W
  // (the kernels address a row of A by a 32-bit byte offset: batches beyond that stay on the streaming kernels)
  const long long tall_rows = ((long long)B * k / 256 + E) * 256;
  if (!mxfp4) {
    const bool tall = gemm_tall_shape_ok(2 * I, H, tall_rows) && gemm_tall_shape_ok(H, I, tall_rows);
    if (tall && moe_tall((long long)B * k, E, k, 2 * I, H)) rpt = 256;
    if (!moe_tall_forced()) rpt = small_block_rows(rpt, B, k, E, H, I, tall);
  }
  // (no more experts have a row than there are rows)
  const int max_tiles = gptoss_moe_max_tiles(B, k, std::min(E, B * k), rpt);
  // Each expert's row tiles are walked in blocks of up to MOE_TILE_BLOCK, column tile by column
  // tile, so the workgroups of an XCD share a column tile of the expert's weights among the block's
  // row tiles instead of streaming it once per row tile.  With one tile per expert (a decode step
  // under uniform routing) the order is the plain one; a skewed routing (Zipf 0.6-1.1 over 32
  // experts, seven of them above 160 rows) runs the layer 7 % faster, prompt passes 2-4 %.
  const int tile_block = MOE_TILE_BLOCK;

  // router GEMM with the gating of its own 16 tokens fused in, then the stable grouping, in the same launch for a few
  // tokens (with `pre`, the residual add and RMSNorm that produce t run in it as well)
  const int cost0 = mxfp4 ? MOE_TILE_COST0_X2_MXFP4 : MOE_TILE_COST0_X2_BF16;
  RouterGroup grp;
  grp.sorted_pair_ids = ws.sorted_pair_ids;
  grp.inv_perm = ws.inv_perm;
  grp.tiles = ws.tiles;
  grp.xcd_bounds = ws.xcd_bounds;
  grp.nbits = 0;
  while ((1 << grp.nbits) < E) grp.nbits++;
  // A few tokens: the router's products are spread over CUs (router_parts_kernel), if the second product's output, which comes
  // later, has room for them.  A router of few inputs is little to spread (block, us: 128 inputs, 8 experts of 1024, 8 / 16 tokens
  // +6 / +4 %, one of 128 +9 / +7 %; 64 inputs, 16 experts 3 to 11 %; 32 experts of 128 inputs -5 to -15 %).
  float *parts = router_parts_floats(B, E) <= (size_t)B * k * H && (H >= 256 || E * H >= 4096) ? ws.y2 : nullptr;
  // Up to four are gated and grouped by the workgroups of the first product (few_routed_kernel); the norm in front runs in the
  // router's kernel.  The block by one launch less, us: 2880 x 2880, one token on 4 of 32 experts 45.9 -> 40.6, two 68.4 -> 63.8,
  // four 120.5 -> 116.2, in MXFP4 31.6 -> 26.8, 38.2 -> 33.6, 49.6 -> 46.6, one on 128 experts 31.6 -> 27.9, with the norm one on 32
  // experts 48.5 -> 43.0, on 128 (1024 wide) 30.5 -> 25.5.  Each workgroup repeats the gating, so three and four tokens go this way
  // only where that is little, up to 32 experts, and where the router's own kernel has a large matrix to read: 128 experts, four
  // tokens 51.4 -> 54.4, four experts of 2880 inputs 42.8 -> 43.5, eight of 2048 27.9 -> 28.2; 32 of 640 20.6 -> 18.2.
  // More than 32 experts take four values a lane, and more workgroups than the chip holds at once gate in a second round: two
  // tokens on 8 of 48 experts of 768 x 2880, 3060 workgroups, +6 %, one token, 1620, -5 %; up to 2048.
  RoutedFew routed{RouterParts{parts, w->b_router, B, E, k}, ws.logits, ws.topk_w, ws.topk_i, grp};
  routed.group.expert_offsets = ws.expert_offsets;
  if (pre) {
    routed.x = pre->x;
    routed.residual = pre->residual;
    routed.x_count = B * H;
  }
  const bool gated_at_once = E <= 32 || (long long)(max_tiles + 1) * (2 * I / 32) <= 2048;
  const bool few = (B <= 2 || (B <= ROUTED_TOKENS && E <= 32 && H * E >= 20480)) && k <= 8 && E <= ROUTED_EXPERTS && rpt == 32 && parts && gated_at_once &&
                   (long long)max_tiles * 32 * H * 2 < (1ll << 31) &&
                   (!pre || norm_router_parts_apply(B, H, pre->x, pre->residual, pre->weight, t));
  if (few) {
    rc = pre ? run_norm_router_parts(pre->x, pre->residual, pre->weight, const_cast<void *>(t), w->w_router, parts, B, H, E, s)
             : run_router_parts(t, w->w_router, parts, B, H, E, s);
    if (rc != GPTOSS_OK) return rc;
    // (from 16 experts on, more tokens than that kernel groups have their norm in front of router_parts_kernel: 2880 x 2880, 32
    // experts, 5 / 12 / 16 tokens 102.8 / 142.1 / 174.6 -> 99.5 / 138.7 / 171.5 us, 1024 wide 25.3 / 31.0 / 30.8 -> 21.0 / 27.1 / 27.2; with
    // eight experts 18.5 / 19.3 / 19.2 -> 16.9 / 18.9 / 18.9 and four 46.8 / 51.4 / 58.5 -> 47.7 / 52.2 / 59.2)
  } else if (pre && !(parts && E >= 16 && B > ROUTER_GROUP_NORM_TOKENS && router_groups(B, k)) &&
             norm_router_applies(B, H, E, pre->x, pre->residual, pre->weight, t)) {
    if (router_groups(B, k) && B <= ROUTER_GROUP_NORM_TOKENS) grp.expert_offsets = ws.expert_offsets;
    rc = run_norm_router(pre->x, pre->residual, pre->weight, const_cast<void *>(t), w->w_router, w->b_router,
                         ws.logits, B, H, E, k, ws.topk_w, ws.topk_i, s, &grp);
  } else {
    if (pre) {
      rc = run_rmsnorm(pre->x, pre->residual, pre->weight, (bf16_t *)const_cast<void *>(t), nullptr, B, H, s);
      if (rc != GPTOSS_OK) return rc;
    }
    if (router_groups(B, k)) grp.expert_offsets = ws.expert_offsets;
    rc = run_router(t, w->w_router, w->b_router, ws.logits, B, H, E, k, ws.topk_w, ws.topk_i, s, &grp, parts);
  }
  if (rc == GPTOSS_OK && !few && !grp.expert_offsets)
    rc = run_group(B, E, k, ws.topk_w, ws.topk_i, ws.expert_offsets, ws.sorted_pair_ids, ws.inv_perm,
                   ws.tiles, rpt, ws.xcd_bounds, cost0, s, ws.sort_scratch);
  if (rc != GPTOSS_OK) return rc;
  const int *bounds = max_tiles < 32768 ? ws.xcd_bounds : nullptr;

  GemmParams g1{};
  g1.A = (const bf16_t *)t;
  g1.row_ids = ws.sorted_pair_ids;
  g1.top_k = k;
  g1.W = (const bf16_t *)w->w1;
  g1.w_mxfp4 = mxfp4;
  g1.bias = w->b1;
  g1.out = ws.act;
  g1.tiles = ws.tiles;
  g1.tile_block = tile_block;
  g1.xcd_bounds = bounds;
  g1.max_tile_rows = B;   // a token takes an expert once
  g1.routed = few ? &routed : nullptr;
  g1.N = 2 * I;
  g1.K = H;
  g1.n_col_tiles = gemm_col_tiles(2 * I);
  if (glu) g1.glu = *glu;
  else g1.glu.limit = w->swiglu_limit;
  rc = run_gemm(g1, true, EPI_SWIGLU, rpt, max_tiles, s);
  if (rc != GPTOSS_OK) return rc;

  GemmParams g2{};
  g2.A = ws.act;
  g2.W = (const bf16_t *)w->w2;
  g2.w_mxfp4 = mxfp4;
  g2.bias = w->b2;
  g2.out = ws.y2;
  g2.tiles = ws.tiles;
  g2.tile_block = tile_block;
  g2.xcd_bounds = bounds;
  g2.max_tile_rows = B;
  g2.N = H;
  g2.K = I;
  g2.n_col_tiles = gemm_col_tiles(H);
  rc = run_gemm(g2, false, EPI_F32, rpt, max_tiles, s);
  if (rc != GPTOSS_OK) return rc;

  return run_combine(ws.y2, ws.topk_w, ws.inv_perm, out, B, H, k, accumulate, norm_w, norm_out, s, tanh_norm);
}

int gptoss::moe_forward_norm(const gptoss_moe_weights *w, const void *t, int B, float *out, void *workspace,
                             size_t workspace_bytes, hipStream_t s, int mxfp4, const float *norm_w,
                             bf16_t *norm_out, const MoePreNorm *pre) {
  return moe_forward_impl(w, t, B, out, 1, workspace, workspace_bytes, s, mxfp4, norm_w, norm_out, pre);
}

int gptoss::moe_forward_glu(const gptoss_moe_weights *w, const GluForm &glu, const void *t, int B, float *out,
                            void *workspace, size_t workspace_bytes, hipStream_t s, const TanhNorm &norm, bf16_t *norm_out) {
  return moe_forward_impl(w, t, B, out, 1, workspace, workspace_bytes, s, 0, nullptr, norm_out, nullptr, &glu, &norm);
}

extern "C" int gptoss_moe_forward(const gptoss_moe_weights *w, const void *t, int B, float *out,
                                  int accumulate, void *workspace, size_t workspace_bytes,
                                  void *stream) {
  return moe_forward_impl(w, t, B, out, accumulate, workspace, workspace_bytes, stream, 0);
}

extern "C" int gptoss_moe_forward_mxfp4(const gptoss_moe_weights *w, const void *t, int B, float *out,
                                        int accumulate, void *workspace, size_t workspace_bytes,
                                        void *stream) {
  return moe_forward_impl(w, t, B, out, accumulate, workspace, workspace_bytes, stream, 1);
}
