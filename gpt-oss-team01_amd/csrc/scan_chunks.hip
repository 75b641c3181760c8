// The state-space recurrence over stretches of a prompt on gfx950, in chunks of 32 tokens on the matrix cores, in fp32
// throughout (v_mfma_f32_16x16x4).  With t, s counting from the chunk's first token, S the state in front of it, c_t the sum of
// the logarithms of the decays up to and with token t and u_s = dt_s v_s what token s writes,
//   o_t = e^(c_t) S^T q_t + sum_{s <= t} e^(c_t - c_s) (k_s . q_t) u_s
//   S  <- e^(c_31) S + sum_s e^(c_31 - c_s) k_s u_s^T
//
// The sums c are kept in double, so that a difference of two is as exact as one decay's logarithm; every weight is
// e^(difference) <= 1, whatever the decays.
//
// A workgroup of four waves has 64 columns of one head's state of one sequence, a wave 16 of them, in registers.  Reduction
// indices are taken four at a time as a 16x16 result lies in its lanes (lane group c = lane >> 4 has rows 4 c .. + 3): state,
// u and token products are operands of the next product without a shuffle, and an operand's four values are one 16-byte read.
//
// Token by token (recurrent.hip) a state element takes three vector instructions a token, and the reads of keys and queries
// fill LDS at the same time; here it takes two products at twice the vector units' rate.  Measured, token by token -> here (us),
// 32 heads of 128 x 64: 8 prompts of 1000 tokens 281 -> 139, 16 of 260 116 -> 68, one 65 -> 41; 8 heads of 128 x 16, one of 1000
// 220 -> 133; 4 of 256 x 64 424 -> 250.  With one wave per SIMD what lies between the products is not hidden (LDS reads are
// requested a group of products ahead, the tokens' decays two chunks); the second workgroup that a CU has room for, up to 128
// keys, is there from 9 sequences of 32 heads on.
//
// A matrix instruction adds its products to a sum one behind the other, so sums over the state's keys are four and over a tile's
// eight, added up in the end, what the chunk's tokens give is summed up by itself, and a token's own key times query, most of its
// output where decays are strong, is made in double by the wave that has no tile.  Errors of the outputs against 64 bits, times
// those token by token, five sizes, 500 tokens: random keys 0.70 on average, with decays of 0 to 0.9 0.76, as the layers make them
// 0.74 and 0.83, of a common direction 0.79 and 1.00, that drift 0.70 and 1.02; of the states 0.5 to 1.0.  With one sum over the
// state's keys, two over a tile's and no part by itself the outputs had 0.96 and 1.44, 1.18 and 1.49, 1.14 and 1.47, 1.08 and 1.55,
// in 8 % less time.
//
// Not for the delta rules, although a chunk can be made of them as well (u is then the solution of a triangular system; 412 ->
// 222 us with a decay per head, 449 -> 273 with one per channel).  What a token writes there takes off what the state has along
// its key.  Token by token every rounding is taken off with it by the next token; in a chunk the tokens' parts are summed up as
// they are, larger than their sum where keys agree.  Errors of the outputs against 64 bits, times those token by token, five
// sizes, 500 tokens: random keys 0.7 to 1.3, keys of a common direction or that drift 2.2 to 6.8 (per channel 1.6 to 2.8).  With
// every product and the system's solution in double an emulation still has 1.7 to 2.2.
#include "recurrent_device.hpp"

namespace gptoss {

constexpr int CHUNK = 32;

// floats of LDS
template <int NI>
struct ChunkLds {
  static constexpr int KP = 32 * NI, ROW = KP + 4;
  static constexpr int Q = 0, K = CHUNK * ROW, STAGE = 2 * CHUNK * ROW;   // two stages
  static constexpr int P = 2 * STAGE;         // 16x16 tiles of token products, 64 lanes x 4 values
  static constexpr int CUM = P + 3 * 256;     // [2][CHUNK] doubles, then per token
  static constexpr int FROM = CUM + 4 * CHUNK, OUT = FROM + 2 * CHUNK, STEP = OUT + 2 * CHUNK, OWN = STEP + 2 * CHUNK,
                       FLOATS = OWN + CHUNK;   // (OWN: of the present chunk)
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// inclusive sums over 32 lanes, of both halves of the wave
__device__ __forceinline__ double prefix32(double v) {
  auto add = [&](auto ctrl, auto rows) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (uint32_t)u, decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (uint32_t)(u >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
    v += __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  };
  using All = std::integral_constant<int, 0xf>;
  add(std::integral_constant<int, 0x111>{}, All{});   // row_shr 1, 2, 4, 8: lanes without a source add nothing
  add(std::integral_constant<int, 0x112>{}, All{});
  add(std::integral_constant<int, 0x114>{}, All{});
  add(std::integral_constant<int, 0x118>{}, All{});
  add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});   // the last lane of rows 0 and 2 to rows 1 and 3
  return v;
}

__device__ __forceinline__ f32x4 sum_of_eight(const f32x4 (&x)[2][4]) {
  return ((x[0][0] + x[1][0]) + (x[0][1] + x[1][1])) + ((x[0][2] + x[1][2]) + (x[0][3] + x[1][3]));
}

// What tokens write, where some of it is not finite.  A product with a whole tile would take its zeros above the diagonal times
// an infinity and give every token of the chunk no number, those in front of the infinity too; here only the tokens in front of
// a token give it something.
__device__ __forceinline__ bool any_not_finite(float sum) { return __ballot(sum * 0.f != 0.f) != 0; }
__device__ __forceinline__ f32x4 tile_below(f32x4 acc, const float *a, f32x4 b, int lane) {
  const int n = lane & 15, c = lane >> 4;
#pragma unroll 1
  for (int g = 0; g < 4; g++)
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const int s = 4 * g + f;
      const float from = __shfl(b[f], g * 16 + n);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int t = 4 * c + e;
        if (s < t) acc[e] = fmaf(a[(g * 16 + t) * 4 + f], from, acc[e]);
      }
    }
  return acc;
}

template <int NI>
__global__ __launch_bounds__(256, NI <= 4 ? 2 : 1) void scan_chunk_kernel(Scan p, const RowSeg *__restrict__ segs, int n_seg) {
  using L = ChunkLds<NI>;
  constexpr int KP = L::KP, ROW = L::ROW, NB = 2 * NI;   // 16-key blocks of the state
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int seg_id = blockIdx.x % n_seg, unit = blockIdx.x / n_seg, blocks = (p.V + 63) / 64;
  const RowSeg seg = segs[seg_id];
  if (unit >= p.heads * blocks) {   // workgroups of the convolutions' states come last
    advance_conv_state(p, seg, unit - p.heads * blocks, gridDim.x / n_seg - p.heads * blocks);
    return;
  }
  // Shorter ones token by token, as in a step without a long one: the same bits.  In this launch, because one behind the other
  // takes longer (us, both in one / shorter ones first / all token by token: a prompt of 48 and 7 of 30, 32 heads of 128 x 64
  // 14.7 / 25.7 / 17.3, 8 heads of 64 x 16 8.8 / 15.9 / 10.3; a prompt of 48 beside 15 / 100 decoding rows, 32 heads 19.7 / 26.6 / 23.9
  // and 50.3 / 54.1 / 55.0; the exception is hundreds of decoding rows of narrow heads: 500 beside 200 tokens, 32 heads of 128 x 16
  // 137 / 105 / 162).
  if (seg.n < SCAN_CHUNK_ROWS) {
    using Tokens = ScanLds<NI, SCAN_STATE_SPACE, false, 2>;
    static_assert(sizeof(Tokens) <= L::FLOATS * sizeof(float));
    const int h = unit / blocks;
    scan_stretch<NI, SCAN_STATE_SPACE, false, 2>(p, seg, h, (unit - h * blocks) * 64, *reinterpret_cast<Tokens *>(lds));
    return;
  }
  const int h = unit / blocks, kh = h / (p.heads / p.key_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, c = lane >> 4;
  const int c0 = (unit - h * blocks) * 64 + wave * 16, col = min(c0 + n, p.V - 1);   // columns c0 .. + 15 of the wave
  const bool live = c0 + n < p.V;
  const float rate = expf(p.a_log[h]), bias = p.dt_bias[h], skip = p.d_skip[h];

  f32x4 S[NB];   // keys 16 b + 4 c + e of column c0 + n
  float *st = p.state + (((size_t)seg.slot * p.heads + h) * p.V + col) * KP + 4 * c;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    S[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (seg.pos0 > 0 && live) S[b] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(st + 16 * b));
  }

  // The next chunk's inputs travel through registers while the current one is worked on.  Addresses: a base per chunk and a
  // 32-bit offset per lane, its token's part by a product of 24 bits (a 64-bit product each takes as long as 16 others).
  f32x4 rk[NI], rq[NI];
  float rv[2][4];
  const uint32_t ld4 = 4 * p.ld_conv;
  auto fetch = [&](int t0) {
    const int T = min(CHUNK, seg.n - t0);
    const char *rows = reinterpret_cast<const char *>(p.conv + (size_t)(seg.row0 + t0) * p.ld_conv);
    const char *ks = rows + 4 * (size_t)(p.k_col + kh * p.K), *qs = rows + 4 * (size_t)(p.q_col + kh * p.K);
    const char *vs = rows + 4 * (size_t)(p.v_col + h * p.V);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int idx = tid + 256 * i, t = min(idx / (KP / 4), T - 1), d = min(idx % (KP / 4) * 4, p.K - 4);
      const uint32_t at = __umul24(t, ld4) + 4 * d;
      rk[i] = *reinterpret_cast<const f32x4 *>(ks + at);
      rq[i] = *reinterpret_cast<const f32x4 *>(qs + at);
    }
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        rv[x][e] = *reinterpret_cast<const float *>(vs + __umul24(min(16 * x + 4 * c + e, T - 1), ld4) + 4 * col);
  };
  // rows and columns outside the problem are zero: they write nothing
  auto put = [&](int t0, int stage) {
    const int T = min(CHUNK, seg.n - t0);
    float *at = lds + stage * L::STAGE;
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int idx = tid + 256 * i, t = idx / (KP / 4), d = idx % (KP / 4) * 4;
      if (T < CHUNK || p.K < KP) {
        const bool out = t >= T || d >= p.K;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          rk[i][e] = out ? 0.f : rk[i][e];
          rq[i][e] = out ? 0.f : rq[i][e];
        }
      }
      *reinterpret_cast<f32x4 *>(at + L::K + t * ROW + d) = rk[i];
      *reinterpret_cast<f32x4 *>(at + L::Q + t * ROW + d) = rq[i];
    }
  };
  // Decays and steps of a chunk's tokens, lane t (and t + 32 again) of the last wave, requested two chunks ahead: it has
  // the least to do while the token products are made.
  float r_decay = 0.f;
  auto fetch_tokens = [&](int t0) {
    r_decay = p.in[(size_t)(seg.row0 + min(t0 + (tid & 31), seg.n - 1)) * p.ld_in + p.decay_col + h];
  };
  auto put_tokens = [&](int t0, int stage) {
    const int t = lane & 31;
    const bool real = t0 + t < seg.n;
    const float dt = softplus_f(r_decay + bias);
    // (Past e^-200, which is zero, no further: the differences behind an infinite sum would be no numbers.)
    const float log_decay = -rate * dt < -200.f ? -200.f : -rate * dt;
    const double cum = prefix32(real ? (double)log_decay : 0.0), all = __shfl(cum, 31);
    if (lane < 32) {
      reinterpret_cast<double *>(lds + L::CUM)[stage * CHUNK + t] = cum;
      lds[L::FROM + stage * CHUNK + t] = exp_f((float)cum);
      lds[L::OUT + stage * CHUNK + t] = exp_f((float)(all - cum));
      lds[L::STEP + stage * CHUNK + t] = real ? dt : 0.f;
    }
  };

  if (wave == 3) fetch_tokens(0);
  fetch(0);
  put(0, 0);
  if (wave == 3) {
    put_tokens(0, 0);
    fetch_tokens(CHUNK);
  }
  int stage = 0;
  for (int t0 = 0; t0 < seg.n; t0 += CHUNK, stage ^= 1) {
    const int T = min(CHUNK, seg.n - t0);
    const bool more = t0 + CHUNK < seg.n;
    float v[2][4];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int e = 0; e < 4; e++) v[x][e] = 16 * x + 4 * c + e < T && live ? rv[x][e] : 0.f;
    __syncthreads();   // this chunk is staged, and nobody reads the other stage or the tiles any more
    if (more) {
      if (wave == 3) {
        put_tokens(t0 + CHUNK, stage ^ 1);
        fetch_tokens(t0 + 2 * CHUNK);
      }
      fetch(t0 + CHUNK);
    }
    const float *q = lds + stage * L::STAGE + L::Q + n * ROW + 4 * c, *k = lds + stage * L::STAGE + L::K + n * ROW + 4 * c;
    const double *cum = reinterpret_cast<const double *>(lds + L::CUM) + stage * CHUNK;
    auto at4 = [&](const float *a) { return *reinterpret_cast<const f32x4 *>(a); };

    // Products of keys (rows) and queries (columns) of tokens, decayed and masked, in tiles (keys', queries') (0, 0), (0, 1), (1, 1),
    // and in the last wave a token's own key times query
    auto product = [&](int sx, int tx, float *to) {
      f32x4 sum[2][4], x[2][2], y[2][2];
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) sum[b][e] = f32x4{0.f, 0.f, 0.f, 0.f};
      auto load = [&](int i) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
          x[i & 1][b] = at4(k + sx * 16 * ROW + 16 * (2 * i + b));
          y[i & 1][b] = at4(q + tx * 16 * ROW + 16 * (2 * i + b));
        }
      };
      load(0);
#pragma unroll
      for (int i = 0; i < NI; i++) {
        if (i + 1 < NI) load(i + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int b = 0; b < 2; b++) sum[b][e] = mfma4(x[i & 1][b][e], y[i & 1][b][e], sum[b][e]);
        __builtin_amdgcn_sched_barrier(0);
      }
      const f32x4 all = sum_of_eight(sum);
      const int t = tx * 16 + n;
      const double ct = cum[t];
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int s = sx * 16 + 4 * c + e;
        const float x = exp_f((float)(ct - cum[s])) * all[e];
        w[e] = s < t ? x : 0.f;
      }
      *reinterpret_cast<f32x4 *>(to + lane * 4) = w;
    };
    if (wave < 3) product(wave == 2, wave > 0, lds + L::P + wave * 256);
    else {
      const float *kt = lds + stage * L::STAGE + L::K + (lane & 31) * ROW + (lane >> 5) * (KP / 2), *qt = kt + (L::Q - L::K);
      double own[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
      for (int d = 0; d < KP / 2; d += 4) {
        const f32x4 a = at4(kt + d), b = at4(qt + d);
#pragma unroll
        for (int e = 0; e < 4; e++) own[e] = fma((double)a[e], (double)b[e], own[e]);
      }
      const double sum = (own[0] + own[1]) + (own[2] + own[3]), all = sum + lane_xor<32>(sum);
      if (lane < 32) lds[L::OWN + lane] = (float)all;
    }
    __syncthreads();

    // what the state in front of the chunk gives: [token][column]
    f32x4 o4[2][4], qx[3][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int e = 0; e < 4; e++) o4[x][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int b) {
#pragma unroll
      for (int x = 0; x < 2; x++) qx[b % 3][x] = at4(q + x * 16 * ROW + 16 * b);
    };
    load(0);
    load(1);
#pragma unroll
    for (int b = 0; b < NB; b++) {
      if (b + 2 < NB) load(b + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int x = 0; x < 2; x++) o4[x][e] = mfma4(qx[b % 3][x][e], S[b][e], o4[x][e]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // what the tokens write
    f32x4 u[2];
#pragma unroll
    for (int x = 0; x < 2; x++) u[x] = at4(lds + L::STEP + stage * CHUNK + 16 * x + 4 * c) * f32x4{v[x][0], v[x][1], v[x][2], v[x][3]};
    auto tile = [&](f32x4 acc, const float *a, f32x4 b) {
      const f32x4 w = at4(a + lane * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) acc = mfma4(w[e], b[e], acc);
      return acc;
    };
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f}, sum = u[0] + u[1];
    f32x4 o[2];   // what the chunk's tokens give later ones
    if (any_not_finite(sum[0] + sum[1] + sum[2] + sum[3])) {
      o[0] = tile_below(zero, lds + L::P, u[0], lane);
      o[1] = tile_below(tile(zero, lds + L::P + 256, u[0]), lds + L::P + 512, u[1], lane);
    } else {
      o[0] = tile(zero, lds + L::P, u[0]);
      o[1] = tile(zero, lds + L::P + 256, u[0]) + tile(zero, lds + L::P + 512, u[1]);
    }
#pragma unroll
    for (int x = 0; x < 2; x++) {
      const f32x4 from = at4(lds + L::FROM + stage * CHUNK + 16 * x + 4 * c), own = at4(lds + L::OWN + 16 * x + 4 * c);
      const f32x4 before = (o4[x][0] + o4[x][1]) + (o4[x][2] + o4[x][3]);
#pragma unroll
      for (int e = 0; e < 4; e++) o[x][e] = fmaf(skip, v[x][e], fmaf(own[e], u[x][e], fmaf(from[e], before[e], o[x][e])));
    }
    char *out = reinterpret_cast<char *>(p.out + (size_t)(seg.row0 + t0) * p.ld_out + h * p.V);
    const uint32_t out4 = 4 * p.ld_out, first = __umul24(4 * c, out4) + 4 * (c0 + n);
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float *to = reinterpret_cast<float *>(out + (16 * x + e) * out4 + first);
        if (T == CHUNK && c0 + 16 <= p.V) *to = o[x][e];
        else if (live && 16 * x + 4 * c + e < T) *to = o[x][e];
      }

    // the state behind the chunk
    const float faded = lds[L::FROM + stage * CHUNK + CHUNK - 1];
#pragma unroll
    for (int x = 0; x < 2; x++) u[x] *= at4(lds + L::OUT + stage * CHUNK + 16 * x + 4 * c);
    const float *keys = lds + stage * L::STAGE + L::K + 4 * c * ROW + n;   // keys of token 4 c, key n
    float kt[2][2][2][4];
    auto load_keys = [&](int i) {
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
          for (int e = 0; e < 4; e++) kt[i & 1][b][x][e] = keys[(16 * x + e) * ROW + 16 * (2 * i + b)];
    };
    load_keys(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      if (i + 1 < NI) load_keys(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; b++) S[2 * i + b] *= faded;
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int b = 0; b < 2; b++) S[2 * i + b] = mfma4(kt[i & 1][b][x][e], u[x][e], S[2 * i + b]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) put(t0 + CHUNK, stage ^ 1);
  }
  if (live) {
#pragma unroll
    for (int b = 0; b < NB; b++) __builtin_nontemporal_store(S[b], reinterpret_cast<f32x4 *>(st + 16 * b));
  }
}

bool scan_chunks_apply(const Scan &p, const StepRows &r) {
  return p.kind == SCAN_STATE_SPACE && r.longest >= SCAN_CHUNK_ROWS && scan_reads_wide(p) && p.K >= 4 && p.K <= SCAN_MAX_KEY &&
         p.ld_conv < (1 << 22) && p.ld_out < (1 << 22);   // (24-bit row pitches)
}

template <int NI>
static int launch_chunks(const Scan &p, const StepRows &r, hipStream_t s) {
  constexpr int bytes = ChunkLds<NI>::FLOATS * (int)sizeof(float);
  auto kern = scan_chunk_kernel<NI>;
  GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  TraceScope ts("scan_state_space", s);
  const size_t grid = (size_t)r.n_seg * (p.heads * cdiv(p.V, 64) + cdiv(p.conv_desc.channels, 256));
  kern<<<(unsigned)grid, 256, bytes, s>>>(p, r.segs, r.n_seg);
  GPTOSS_LAUNCH_CHECK("scan_chunk_kernel");
  return GPTOSS_OK;
}

int run_scan_chunks(const Scan &scan, const StepRows &r, hipStream_t s) {
  Scan p = scan;
  p.vec = 1;   // (scan_chunks_apply)
  GPTOSS_REQUIRE(scan_chunks_apply(p, r) && p.V >= 1 && p.key_heads >= 1 && p.heads % p.key_heads == 0, GPTOSS_ERR_DIM,
                 "scan: kind %d with keys of %d, %d heads over %d does not go by chunks", (int)p.kind, p.K, p.heads, p.key_heads);
  GPTOSS_REQUIRE(r.n_seg * ((long long)p.heads * cdiv(p.V, 64) + cdiv(p.conv_desc.channels, 256)) < (1ll << 31), GPTOSS_ERR_DIM,
                 "scan: too many workgroups");
  switch (scan_key_pad(p.K) / 32) {
    case 1: return launch_chunks<1>(p, r, s);
    case 2: return launch_chunks<2>(p, r, s);
    case 3: return launch_chunks<3>(p, r, s);
    case 4: return launch_chunks<4>(p, r, s);
    case 5: return launch_chunks<5>(p, r, s);
    case 6: return launch_chunks<6>(p, r, s);
    case 7: return launch_chunks<7>(p, r, s);
    default: return launch_chunks<8>(p, r, s);
  }
}

}  // namespace gptoss
