// Recurrent mixers for gfx950: gated delta rules (one decay per head, or one per key channel), the
// state-space recurrence and retention (a fixed decay per head, plain writes), with the short
// convolutions in front of them and the gated norms behind.
//
// The recurrence of a head acts on a K x V state whose V columns are independent of each other, so a
// column lives in 8 lanes of a wave (K / 8 rows each, in registers) and a wave owns 16 columns (8 where
// there is little to share out): for a step of one token the launch streams every state once through
// the chip, 16 bytes per lane and request; for a stretch of a prompt the state stays in registers while
// the tokens go by, their keys, queries and gates staged in LDS and shared by the workgroup's columns.
// Everything is fp32, and the tokens are taken one after the other, so a sequence's results are bit for
// bit the same however it is cut into steps.  Long stretches of a prompt run in retention.hip (retention) and scan_chunks.hip
// (state space) instead, which equal this to rounding.
#include <type_traits>

#include "recurrent_device.hpp"

namespace gptoss {

__device__ __forceinline__ float wave_sum_f(float v) {
  return lanes_sum(v);
}

// ---- short convolution ---------------------------------------------------------------------------
// Input of channel c, j tokens before row r (offset `off` in its sequence's stretch, position `pos`).
__device__ __forceinline__ float conv_input(const ShortConv &c, const float *in, int ld_in, const float *state,
                                            int row, int off, int pos, int slot, int ch, int j) {
  if (j > pos) return 0.f;
  if (j <= off) return in[(size_t)(row - j) * ld_in + c.col + ch];
  // state[taps - 2] is the input right before the stretch
  return state[((size_t)slot * (c.taps - 1) + (c.taps - 1 + off - j)) * c.channels + ch];
}

// One wave per (rows, head): heads of unit_dim channels that become unit vectors first, then the remaining
// channels in pieces of 64.  A wave takes RT consecutive rows, whose inputs it requests together and
// slides the taps over (TAPS 0: any number of taps, inputs read tap by tap).
template <int TAPS, int RT>
__global__ __launch_bounds__(256) void short_conv_kernel(ShortConv c, const int *__restrict__ slots,
                                                         const int *__restrict__ lens,
                                                         const int *__restrict__ offset,
                                                         const float *__restrict__ in, int ld_in,
                                                         const float *__restrict__ state, float *__restrict__ out,
                                                         int ld_out, int units, int n) {
  constexpr int PIECES = SCAN_MAX_KEY / 64;
  const int row0 = blockIdx.y * RT, lane = threadIdx.x & 63;
  const int unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;
  const bool norm = unit < 2 * c.n_unit;
  const int unit_ch = 2 * c.n_unit * c.unit_dim;
  const int ch0 = norm ? unit * c.unit_dim : unit_ch + (unit - 2 * c.n_unit) * 64;
  const int width = norm ? c.unit_dim : min(64, c.channels - ch0);
  const int live = min(RT, n - row0);
  int off[RT], pos[RT], slot[RT];
#pragma unroll
  for (int r = 0; r < RT; r++) {
    const int row = row0 + min(r, live - 1);
    off[r] = offset[row];
    pos[r] = lens[row] - 1;
    slot[r] = slots[row];
  }
  float v[PIECES][RT], ss[RT];
#pragma unroll
  for (int r = 0; r < RT; r++) ss[r] = 0.f;
#pragma unroll
  for (int i = 0; i < PIECES; i++) {
    if (64 * i >= width) break;
    const int d = lane + 64 * i, ch = ch0 + min(d, width - 1);
    const float bias = c.bias ? c.bias[ch] : 0.f;
    if constexpr (TAPS > 0) {
      float w[TAPS], x[RT], past[TAPS];   // past[j]: the input j + 1 tokens back
#pragma unroll
      for (int j = 0; j < TAPS; j++) w[j] = c.weight[(size_t)ch * TAPS + (TAPS - 1 - j)];
#pragma unroll
      for (int r = 0; r < RT; r++) x[r] = in[(size_t)(row0 + min(r, live - 1)) * ld_in + c.col + ch];
#pragma unroll
      for (int r = 0; r < RT; r++) {
        if (r == 0 || off[r] == 0) {   // wave-uniform: the first row here, or of its sequence in this step
#pragma unroll
          for (int j = 0; j + 1 < TAPS; j++)
            past[j] = conv_input(c, in, ld_in, state, row0 + min(r, live - 1), off[r], pos[r], slot[r], ch, j + 1);
        }
        float a = bias;
#pragma unroll
        for (int j = TAPS - 1; j >= 1; j--) a = fmaf(w[j], past[j - 1], a);
        a = fmaf(w[0], x[r], a);
#pragma unroll
        for (int j = TAPS - 2; j >= 1; j--) past[j] = past[j - 1];
        if (TAPS > 1) past[0] = x[r];
        v[i][r] = d < width ? silu_f(a) : 0.f;
        ss[r] = fmaf(v[i][r], v[i][r], ss[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < RT; r++) {
        float a = bias;
        for (int j = c.taps - 1; j >= 0; j--)
          a = fmaf(c.weight[(size_t)ch * c.taps + (c.taps - 1 - j)],
                   conv_input(c, in, ld_in, state, row0 + min(r, live - 1), off[r], pos[r], slot[r], ch, j), a);
        v[i][r] = d < width ? silu_f(a) : 0.f;
        ss[r] = fmaf(v[i][r], v[i][r], ss[r]);
      }
    }
  }
  float scale[RT];
#pragma unroll
  for (int r = 0; r < RT; r++) scale[r] = 1.f;
  if (norm) {
#pragma unroll
    for (int r = 0; r < RT; r++)
      scale[r] = (unit < c.n_unit ? c.unit_scale : 1.f) / sqrtf(wave_sum_f(ss[r]) + 1e-6f);
  }
#pragma unroll
  for (int i = 0; i < PIECES; i++) {
    if (64 * i >= width) break;
    const int d = lane + 64 * i;
#pragma unroll
    for (int r = 0; r < RT; r++)
      if (r < live && d < width) out[(size_t)(row0 + r) * ld_out + ch0 + d] = v[i][r] * scale[r];
  }
}

// ---- recurrence ----------------------------------------------------------------------------------
template <int NI, int KIND, bool ONE, int CPL>
__global__ __launch_bounds__(256) void scan_kernel(Scan p, const RowSeg *__restrict__ segs, int n_seg) {
  __shared__ __attribute__((aligned(16))) ScanLds<NI, KIND, ONE, CPL> l;
  // workgroups in order of (head, column block, sequence); those of the convolutions' states come last
  constexpr int COLS = 32 * CPL;
  const int blocks = (p.V + COLS - 1) / COLS;
  const int seg_id = blockIdx.x % n_seg, unit = blockIdx.x / n_seg;
  const RowSeg seg = segs[seg_id];
  if (unit >= p.heads * blocks) {
    advance_conv_state(p, seg, unit - p.heads * blocks, gridDim.x / n_seg - p.heads * blocks);
    return;
  }
  const int h = unit / blocks;
  scan_stretch<NI, KIND, ONE, CPL>(p, seg, h, (unit - h * blocks) * COLS, l);
}

// ---- gated output norm ---------------------------------------------------------------------------
__device__ __forceinline__ float gated_value(const GatedNorm &g, float y, float gate) {
  return g.gate_first ? y * silu_f(gate) : y;
}

// One wave per (row, group), any size and alignment.
template <typename OUT>
__global__ __launch_bounds__(256) void gated_norm_kernel(GatedNorm g) {
  const int row = blockIdx.y, lane = threadIdx.x & 63;
  const int group = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (group >= g.groups) return;
  const float *y = g.y + (size_t)row * g.ld_y + group * g.size;
  const float *gate = g.gate + (size_t)row * g.ld_gate + group * g.size;
  const float *w = g.weight ? g.weight + (g.weight_per_group ? group * g.size : 0) : nullptr;
  float ss = 0.f;
  for (int d = lane; d < g.size; d += 64) {
    const float v = gated_value(g, y[d], gate[d]);
    ss += v * v;
  }
  const float inv = 1.f / sqrtf(wave_sum_f(ss) / g.size + g.eps);
  OUT *out = (OUT *)g.out + (size_t)row * g.ld_out + g.out_col + group * g.size;
  for (int d = lane; d < g.size; d += 64) {
    float v = gated_value(g, y[d], gate[d]) * inv * (w ? w[d] : 1.f);
    if (!g.gate_first) v *= g.sigmoid_gate ? sigmoid_f(gate[d]) : silu_f(gate[d]);
    v *= g.scale;
    if constexpr (sizeof(OUT) == 2) out[d] = f32_to_bf16(v);
    else out[d] = v;
  }
}

// Groups of at most 4 * LANES * VPT values whose rows are 16-byte aligned: LANES lanes hold a group in
// registers, a wave 64 / LANES groups.
template <typename OUT, int LANES, int VPT>
__global__ __launch_bounds__(256) void gated_norm_vec_kernel(GatedNorm g) {
  const int row = blockIdx.y, l = threadIdx.x % LANES;
  const int group = blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  const bool live = group < g.groups;
  const int at = (live ? group : 0) * g.size;
  const float *y = g.y + (size_t)row * g.ld_y + at, *gate = g.gate + (size_t)row * g.ld_gate + at;
  const float *w = g.weight ? g.weight + (g.weight_per_group ? at : 0) : nullptr;
  f32x4 v[VPT], z[VPT], wv[VPT];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; i++) {
    const int d = (l + LANES * i) * 4;
    v[i] = z[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    wv[i] = f32x4{1.f, 1.f, 1.f, 1.f};
    if (d < g.size) {
      v[i] = *reinterpret_cast<const f32x4 *>(y + d);
      z[i] = *reinterpret_cast<const f32x4 *>(gate + d);
      if (w) wv[i] = *reinterpret_cast<const f32x4 *>(w + d);
    }
  }
#pragma unroll
  for (int i = 0; i < VPT; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[i][e] = gated_value(g, v[i][e], z[i][e]);
      ss = fmaf(v[i][e], v[i][e], ss);
    }
  ss = lanes_sum<LANES>(ss);
  const float inv = 1.f / sqrtf(ss / g.size + g.eps);
  if (!live) return;
  OUT *out = (OUT *)g.out + (size_t)row * g.ld_out + g.out_col + at;
#pragma unroll
  for (int i = 0; i < VPT; i++) {
    const int d = (l + LANES * i) * 4;
    if (d < g.size) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        o[e] = v[i][e] * inv * wv[i][e];
        if (!g.gate_first) o[e] *= g.sigmoid_gate ? sigmoid_f(z[i][e]) : silu_f(z[i][e]);
        o[e] *= g.scale;
      }
      if constexpr (sizeof(OUT) == 2)
        *reinterpret_cast<u32x2 *>(out + d) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      else *reinterpret_cast<f32x4 *>(out + d) = o;
    }
  }
}

__global__ __launch_bounds__(256) void column_map_kernel(const float *__restrict__ in, int ld_in, int col, int width,
                                                         int relu_squared, float *__restrict__ out, int ld_out) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  const size_t row = blockIdx.y;
  if (d >= width) return;
  float v = in[row * ld_in + col + d];
  if (relu_squared) {
    v = fmaxf(v, 0.f);
    v *= v;
  }
  out[row * ld_out + d] = v;
}

// ---- launches ------------------------------------------------------------------------------------
int run_short_conv(const ShortConv &c, const StepRows &r, const float *in, int ld_in, const float *state,
                   float *out, int ld_out, hipStream_t s) {
  GPTOSS_REQUIRE(c.unit_dim <= SCAN_MAX_KEY && c.taps >= 1, GPTOSS_ERR_DIM,
                 "short_conv: heads of at most %d channels, at least one tap (%d, %d)", SCAN_MAX_KEY, c.unit_dim, c.taps);
  const int plain = c.channels - 2 * c.n_unit * c.unit_dim;
  const int units = 2 * c.n_unit + cdiv(plain, 64);
  TraceScope ts("short_conv", s);
  auto go = [&](auto kern, int rt) {
    kern<<<dim3(cdiv(units, 4), cdiv(r.n, rt)), 256, 0, s>>>(c, r.slots, r.lens, r.offset, in, ld_in, state, out, ld_out,
                                                             units, r.n);
  };
  const bool many = r.longest > 1 && r.n >= 256;
  if (c.taps == 4) many ? go(short_conv_kernel<4, 8>, 8) : go(short_conv_kernel<4, 1>, 1);
  else if (c.taps == 3) many ? go(short_conv_kernel<3, 8>, 8) : go(short_conv_kernel<3, 1>, 1);
  else if (c.taps == 2) many ? go(short_conv_kernel<2, 8>, 8) : go(short_conv_kernel<2, 1>, 1);
  else go(short_conv_kernel<0, 1>, 1);
  GPTOSS_LAUNCH_CHECK("short_conv_kernel");
  return GPTOSS_OK;
}

template <int NI, int KIND>
static void launch_scan_kind(const Scan &p, const StepRows &r, hipStream_t s) {
  // The convolutions' states: a thread per channel.  With as many workgroups as a head has column blocks, one or two, a
  // decoding step waited for them: four sequences, 4096 channels and 32 heads of 128 x 64 15.6 -> 5.2 us.
  const int conv = KIND == SCAN_RETENTION ? 0 : cdiv(p.conv_desc.channels, 256);
  auto grid = [&](int cols) { return dim3((unsigned)(r.n_seg * (p.heads * cdiv(p.V, cols) + conv))); };
  // Stretches of few heads and sequences: with two columns per lane half of the chip would be idle, or every SIMD have
  // one wave, which issues an instruction every seven cycles (8 prompts of 1000 and 16 heads of 128 x 128, 256 workgroups
  // against 512: delta rule 455 -> 409 us, per key channel 544 -> 521; 32 heads of 128 x 64, state space 383 -> 342).
  // Beyond 256 a lane's second column costs less than a second workgroup: 12 prompts of 500, delta rule 336 against 360 us
  // with one column, per key channel 403 / 450, state space 249 / 228; 16 prompts 359 / 429, 444 / 539, 279 / 346.
  const bool few = (long long)r.n_seg * p.heads * cdiv(p.V, 64) <= 256;
  if (r.longest == 1) scan_kernel<NI, KIND, true, 2><<<grid(64), 256, 0, s>>>(p, r.segs, r.n_seg);
  else if (few) scan_kernel<NI, KIND, false, 1><<<grid(32), 256, 0, s>>>(p, r.segs, r.n_seg);
  else scan_kernel<NI, KIND, false, 2><<<grid(64), 256, 0, s>>>(p, r.segs, r.n_seg);
}

template <int NI>
static void launch_scan(const Scan &p, const StepRows &r, hipStream_t s) {
  switch (p.kind) {
    case SCAN_DELTA: launch_scan_kind<NI, SCAN_DELTA>(p, r, s); break;
    case SCAN_CHANNEL_DELTA: launch_scan_kind<NI, SCAN_CHANNEL_DELTA>(p, r, s); break;
    case SCAN_STATE_SPACE: launch_scan_kind<NI, SCAN_STATE_SPACE>(p, r, s); break;
    case SCAN_RETENTION: launch_scan_kind<NI, SCAN_RETENTION>(p, r, s); break;
  }
}

int run_scan(const Scan &scan, const StepRows &r, hipStream_t s) {
  Scan p = scan;
  p.vec = scan_reads_wide(p);
  GPTOSS_REQUIRE(!p.rot.table || (p.kind == SCAN_RETENTION && r.longest == 1 && p.vec && !p.rot.interleaved &&
                                  p.rot.dims % 8 == 0 && p.rot.dims <= p.K),
                 GPTOSS_ERR_DIM, "scan: only steps of one row per sequence rotate queries and keys, in groups of four dimensions");
  GPTOSS_REQUIRE(p.K >= 1 && p.K <= SCAN_MAX_KEY && p.V >= 1 && p.key_heads >= 1 && p.heads % p.key_heads == 0,
                 GPTOSS_ERR_DIM, "scan: key dimension %d (at most %d), %d heads over %d", p.K, SCAN_MAX_KEY, p.heads,
                 p.key_heads);
  GPTOSS_REQUIRE(r.n_seg * ((long long)p.heads * cdiv(p.V, 32) + cdiv(p.conv_desc.channels, 256)) < (1ll << 31), GPTOSS_ERR_DIM,
                 "scan: too many workgroups");
  static const char *names[] = {"scan_delta", "scan_channel_delta", "scan_state_space", "scan_retention"};
  TraceScope ts(names[p.kind], s);
  switch (scan_key_pad(p.K) / 32) {
    case 1: launch_scan<1>(p, r, s); break;
    case 2: launch_scan<2>(p, r, s); break;
    case 3: launch_scan<3>(p, r, s); break;
    case 4: launch_scan<4>(p, r, s); break;
    case 5: launch_scan<5>(p, r, s); break;
    case 6: launch_scan<6>(p, r, s); break;
    case 7: launch_scan<7>(p, r, s); break;
    default: launch_scan<8>(p, r, s); break;
  }
  GPTOSS_LAUNCH_CHECK("scan_kernel");
  return GPTOSS_OK;
}

template <typename OUT>
static void launch_gated_norm(const GatedNorm &g, int n, hipStream_t s) {
  const bool vec = g.size % 4 == 0 && g.ld_y % 4 == 0 && g.ld_gate % 4 == 0 && g.ld_out % 4 == 0 && g.out_col % 4 == 0 &&
                   aligned(g.y, 16) && aligned(g.gate, 16) && aligned(g.weight, 16) && aligned(g.out, 16);
  if (vec && g.size <= 64) gated_norm_vec_kernel<OUT, 16, 1><<<dim3(cdiv(g.groups, 16), n), 256, 0, s>>>(g);
  else if (vec && g.size <= 128) gated_norm_vec_kernel<OUT, 32, 1><<<dim3(cdiv(g.groups, 8), n), 256, 0, s>>>(g);
  else if (vec && g.size <= 256) gated_norm_vec_kernel<OUT, 64, 1><<<dim3(cdiv(g.groups, 4), n), 256, 0, s>>>(g);
  else if (vec && g.size <= 512) gated_norm_vec_kernel<OUT, 64, 2><<<dim3(cdiv(g.groups, 4), n), 256, 0, s>>>(g);
  else if (vec && g.size <= 1024) gated_norm_vec_kernel<OUT, 64, 4><<<dim3(cdiv(g.groups, 4), n), 256, 0, s>>>(g);
  else gated_norm_kernel<OUT><<<dim3(cdiv(g.groups, 4), n), 256, 0, s>>>(g);
}

int run_gated_norm(const GatedNorm &g, int n, hipStream_t s) {
  TraceScope ts("gated_norm", s);
  if (g.out_f32) launch_gated_norm<float>(g, n, s);
  else launch_gated_norm<bf16_t>(g, n, s);
  GPTOSS_LAUNCH_CHECK("gated_norm_kernel");
  return GPTOSS_OK;
}

int run_column_map(const float *in, int ld_in, int col, int width, bool relu_squared, float *out, int ld_out, int n,
                   hipStream_t s) {
  TraceScope ts(relu_squared ? "relu_squared" : "column_copy", s);
  column_map_kernel<<<dim3(cdiv(width, 256), n), 256, 0, s>>>(in, ld_in, col, width, relu_squared, out, ld_out);
  GPTOSS_LAUNCH_CHECK("column_map_kernel");
  return GPTOSS_OK;
}

}  // namespace gptoss
