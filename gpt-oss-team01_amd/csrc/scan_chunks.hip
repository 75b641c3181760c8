// The gated delta rules and the state-space recurrence over stretches of a prompt on gfx950, in chunks of 32 tokens (one decay
// per key channel: of 16, further down) on the matrix cores, in fp32 throughout (v_mfma_f32_16x16x4).  With t, s counting from
// the chunk's first token, S the state in front of it, c_t the sum of the logarithms of the decays up to and with token t and
// u_s what token s writes,
//   o_t = e^(c_t) S^T q_t + sum_{s <= t} e^(c_t - c_s) (k_s . q_t) u_s
//   S  <- e^(c_31) S + sum_s e^(c_31 - c_s) k_s u_s^T
// State space: u_s = dt_s v_s.  Delta rule: u_t = beta_t (v_t - e^(c_t) S^T k_t - sum_{s < t} e^(c_t - c_s) (k_s . k_t) u_s), a
// triangular system whose diagonal blocks of 16 are inverted by forward substitution.
//
// The sums c are kept in double, so that a difference of two is as exact as one decay's logarithm; every weight is
// e^(difference) <= 1, whatever the decays.
//
// A workgroup of four waves has 64 columns of one head's state of one sequence, a wave 16 of them, in registers.  Reduction
// indices are taken four at a time as a 16x16 result lies in its lanes (lane group c = lane >> 4 has rows 4 c .. + 3): state,
// u and token products are operands of the next product without a shuffle, and an operand's four values are one 16-byte read.
//
// Token by token (recurrent.hip) a state element takes three (state space) or four vector instructions a token, and the
// reads of keys and queries fill LDS at the same time; here it takes two or three products at twice the vector units' rate.
// Measured, token by token -> here (us): 8 prompts of 1000 tokens, 32 heads of 128 x 64 (state space) 338 -> 152, 16 heads of
// 128 x 128 (delta rule) 412 -> 222; 16 prompts of 260 150 -> 85, 195 -> 121; one 71 -> 42, 82 -> 60.  The products alone are 70
// and 113 us of the first two: with one wave per SIMD what lies between them is not hidden (LDS reads are requested a group of
// products ahead, the tokens' decays two chunks; as the compiler placed them 185 and 270 us), and the second workgroup that a
// CU has room for, up to 128 keys, is there from 9 sequences of 32 heads on.
// Errors against 64 bits, six layers of other sizes, 500 tokens, decays of 0.6 to 0.999 and of 0 to 0.9: 0.82 to 1.10 times
// those of the recurrence token by token, 0.97 on average.
#include "recurrent_device.hpp"

namespace gptoss {

constexpr int CHUNK = 32;

// floats of LDS
template <int NI>
struct ChunkLds {
  static constexpr int KP = 32 * NI, ROW = KP + 4;
  static constexpr int Q = 0, K = CHUNK * ROW, STAGE = 2 * CHUNK * ROW;   // two stages
  // 16x16 tiles, 64 lanes x 4 values: products with the queries, with the keys, inverses of the diagonal blocks
  static constexpr int P = 2 * STAGE, A = P + 3 * 256, INV = A + 3 * 256;
  static constexpr int CUM = INV + 2 * 256;                              // [2][CHUNK] doubles, then per token
  static constexpr int FROM = CUM + 4 * CHUNK, OUT = FROM + 2 * CHUNK, BETA = OUT + 2 * CHUNK, FLOATS = BETA + 2 * CHUNK;
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

// What tokens write, where some of it is not finite.  A product with a whole tile would take its zeros above the diagonal times
// an infinity and give every token of the chunk no number, those in front of the infinity too; here only the tokens in front of
// a token (own: and it itself) give it something.
__device__ __forceinline__ bool any_not_finite(float sum) { return __ballot(sum * 0.f != 0.f) != 0; }
__device__ __forceinline__ f32x4 tile_below(f32x4 acc, const float *a, f32x4 b, bool own, int lane) {
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
        if (s < t || (own && s == t)) acc[e] = fmaf(a[(g * 16 + t) * 4 + f], from, acc[e]);
      }
    }
  return acc;
}

// The inverse of I + A, A a strictly lower triangular tile of 16x16 ((s >> 2, t, s & 3), s < t), by columns: lane n (< 16) has
// column n.  What a row of the inverse gives the later ones is taken off all of them at once, four columns of A in registers at
// a time (AHEAD: the next four requested meanwhile).
template <bool AHEAD>
__device__ __forceinline__ void invert_tile(const float *a, float *inv, float diagonal, int n) {
  f32x4 w[AHEAD ? 2 : 1][16];
  auto load = [&](auto group) {
    constexpr int g = decltype(group)::value;
#pragma unroll
    for (int t = 4 * g + 1; t < 16; t++) w[AHEAD ? g & 1 : 0][t] = *reinterpret_cast<const f32x4 *>(a + (g * 16 + t) * 4);
  };
  float x[16];
#pragma unroll
  for (int t = 0; t < 16; t++) x[t] = t == n ? 1.f : 0.f;
  auto take = [&](auto group) {
    constexpr int g = decltype(group)::value;
    if constexpr (!AHEAD) load(group);
    else if constexpr (g < 3) load(std::integral_constant<int, g + 1>{});
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int t = 4 * g + e + 1; t < 16; t++) x[t] = fmaf(-w[AHEAD ? g & 1 : 0][t][e], x[4 * g + e], x[t]);
  };
  if constexpr (AHEAD) load(std::integral_constant<int, 0>{});
  take(std::integral_constant<int, 0>{});
  take(std::integral_constant<int, 1>{});
  take(std::integral_constant<int, 2>{});
  take(std::integral_constant<int, 3>{});
  float *to = inv + (n >> 2) * 64 + (n & 3);
#pragma unroll
  for (int t = 0; t < 16; t++) to[t * 4] = t == n ? diagonal : x[t];
}

template <int NI, int KIND>
__global__ __launch_bounds__(256, NI <= 4 ? 2 : 1) void scan_chunk_kernel(Scan p, const RowSeg *__restrict__ segs, int n_seg,
                                                                               int fewest) {
  using L = ChunkLds<NI>;
  constexpr bool DELTA = KIND == SCAN_DELTA;
  constexpr int KP = L::KP, ROW = L::ROW, NB = 2 * NI;   // 16-key blocks of the state
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int seg_id = blockIdx.x % n_seg, unit = blockIdx.x / n_seg, blocks = (p.V + 63) / 64;
  const RowSeg seg = segs[seg_id];
  if (seg.n < fewest) return;   // taken elsewhere
  if (unit >= p.heads * blocks) {   // workgroups of the convolutions' states come last
    advance_conv_state(p, seg, unit - p.heads * blocks, gridDim.x / n_seg - p.heads * blocks);
    return;
  }
  const int h = unit / blocks, kh = h / (p.heads / p.key_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, c = lane >> 4;
  const int c0 = (unit - h * blocks) * 64 + wave * 16, col = min(c0 + n, p.V - 1);   // columns c0 .. + 15 of the wave
  const bool live = c0 + n < p.V;
  const float rate = expf(p.a_log[h]), bias = p.dt_bias[h], skip = DELTA ? 0.f : p.d_skip[h];

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
  // Decays and strengths of a chunk's tokens, lane t (and t + 32 again) of the last wave, requested two chunks ahead: it has
  // the least to do while the token products are made.
  float r_decay = 0.f, r_beta = 0.f;
  auto fetch_tokens = [&](int t0) {
    const float *in = p.in + (size_t)(seg.row0 + min(t0 + (tid & 31), seg.n - 1)) * p.ld_in + h;
    r_decay = in[p.decay_col];
    if (DELTA) r_beta = in[p.beta_col];
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
      lds[L::BETA + stage * CHUNK + t] = real ? (DELTA ? sigmoid_f(r_beta) : dt) : 0.f;
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

    // Products of keys (rows) and queries or keys (columns) of tokens, decayed and masked, in tiles (keys', columns') (0, 0),
    // (0, 1), (1, 1).  Delta rule: the first two waves have a diagonal tile of the keys each and its inverse.
    auto product = [&](const float *right, int sx, int tx, bool strict, const float *beta, float *to) {
      f32x4 even = f32x4{0.f, 0.f, 0.f, 0.f}, odd = even, x[2][2], y[2][2];
      auto load = [&](int i) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
          x[i & 1][b] = at4(k + sx * 16 * ROW + 16 * (2 * i + b));
          y[i & 1][b] = at4(right + tx * 16 * ROW + 16 * (2 * i + b));
        }
      };
      load(0);
#pragma unroll
      for (int i = 0; i < NI; i++) {
        if (i + 1 < NI) load(i + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          even = mfma4(x[i & 1][0][e], y[i & 1][0][e], even);
          odd = mfma4(x[i & 1][1][e], y[i & 1][1][e], odd);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const int t = tx * 16 + n;
      const double ct = cum[t];
      const float scale = beta ? beta[t] : 1.f;
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int s = sx * 16 + 4 * c + e;
        const float x = scale * exp_f((float)(ct - cum[s])) * (even[e] + odd[e]);
        w[e] = (strict ? s < t : s <= t) ? x : 0.f;
      }
      *reinterpret_cast<f32x4 *>(to + lane * 4) = w;
    };
    const float *beta = lds + L::BETA + stage * CHUNK;
    if constexpr (!DELTA) {
      if (wave < 3) product(q, wave == 2, wave > 0, false, nullptr, lds + L::P + wave * 256);
    } else if (wave < 2) {
      float *a = lds + L::A + wave * 512;
      product(k, wave, wave, true, beta, a);
      if (lane < 16) invert_tile<true>(a, lds + L::INV + wave * 256, 1.f, n);
    } else if (wave == 2) {
      product(q, 0, 0, false, nullptr, lds + L::P);
      product(q, 0, 1, false, nullptr, lds + L::P + 256);
    } else {
      product(q, 1, 1, false, nullptr, lds + L::P + 512);
      product(k, 0, 1, true, beta, lds + L::A + 256);
    }
    __syncthreads();

    // what the state in front of the chunk gives: [token][column]
    f32x4 o[2], r[2];
#pragma unroll
    for (int x = 0; x < 2; x++) o[x] = r[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 qx[3][2], kx[3][2];
    auto load = [&](int b) {
#pragma unroll
      for (int x = 0; x < 2; x++) {
        qx[b % 3][x] = at4(q + x * 16 * ROW + 16 * b);
        if (DELTA) kx[b % 3][x] = at4(k + x * 16 * ROW + 16 * b);
      }
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
        for (int x = 0; x < 2; x++) {
          o[x] = mfma4(qx[b % 3][x][e], S[b][e], o[x]);
          if (DELTA) r[x] = mfma4(kx[b % 3][x][e], S[b][e], r[x]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    // what the tokens write
    f32x4 u[2];
#pragma unroll
    for (int x = 0; x < 2; x++) {
      const f32x4 from = at4(lds + L::FROM + stage * CHUNK + 16 * x + 4 * c), be = at4(beta + 16 * x + 4 * c);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        o[x][e] *= from[e];
        u[x][e] = be[e] * (DELTA ? v[x][e] - from[e] * r[x][e] : v[x][e]);
      }
    }
    auto tile = [&](f32x4 acc, const float *a, f32x4 b) {
      const f32x4 w = at4(a + lane * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) acc = mfma4(w[e], b[e], acc);
      return acc;
    };
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 w[2] = {u[0], u[1]};
    if constexpr (DELTA) {
      w[0] = tile(zero, lds + L::INV, u[0]);
      w[1] = tile(zero, lds + L::INV + 256, u[1] - tile(zero, lds + L::A + 256, w[0]));
    }
    const f32x4 sum = w[0] + w[1];
    if (any_not_finite(sum[0] + sum[1] + sum[2] + sum[3])) {
      if constexpr (DELTA) {
        w[0] = tile_below(zero, lds + L::INV, u[0], true, lane);
        w[1] = tile_below(zero, lds + L::INV + 256, u[1] - tile(zero, lds + L::A + 256, w[0]), true, lane);
      }
      o[0] = tile_below(o[0], lds + L::P, w[0], true, lane);
      o[1] = tile_below(tile(o[1], lds + L::P + 256, w[0]), lds + L::P + 512, w[1], true, lane);
    } else {
      o[0] = tile(o[0], lds + L::P, w[0]);
      o[1] = tile(o[1], lds + L::P + 256, w[0]);
      o[1] = tile(o[1], lds + L::P + 512, w[1]);
    }
#pragma unroll
    for (int x = 0; x < 2; x++) u[x] = w[x];
    if (!DELTA)
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int e = 0; e < 4; e++) o[x][e] = fmaf(skip, v[x][e], o[x][e]);
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

// ------------------------------------------------------------------------------------------------
// The delta rule with a decay per head and key channel, in chunks of 16 tokens.  The weight between two tokens is now a product
// of decays in every channel, so token products take operands that carry it: with the chunk's tokens halved again and again, a
// pair s < t is split by exactly one boundary, behind the even one and in front of the odd one of two neighbouring blocks of
// 8, 4, 2 or 1; t's key and query carry the decays from the boundary up to and with t, s's key those behind s up to it.  These
// are products of at most eight decays, never quotients, so nothing overflows however strong the decays are.  A wave has a
// block size: the keys of its 8 even tokens times the keys and queries of its 8 odd ones.  The state in front of the chunk
// meets keys and queries that carry the decays from the chunk's first token on, the state behind it keys that carry those up
// to its last.
//
// Four waves have 16 columns of the state each, eight others prepare the next chunk meanwhile.  Between two barriers either the
// operands are made (a thread has a channel of four tokens in registers: products of decays are its own and two exchanges with
// the lanes 16 and 32 further) while the state gives its part and the chunk's block is inverted, or the token products while
// the state is brought up to date.
//
// A SIMD's three waves have 136 products of 32 cycles a chunk, 4400 of the 9000 that it takes; what makes the operands fills the
// rest, LDS first (60 reads and writes of single values for each of its eight waves).  Measured, token by token -> here (us), 16 heads of 128 x 128: 8 prompts of 1000 tokens 449 -> 273, one 353 ->
// 252, 16 of 260 187 -> 158, 16 of 64 52 -> 49; 8 prompts of 1000 within Nezavik 545 -> 320.  With all of it one behind the other
// in four waves 440 (there), with four waves that prepare and eight tokens a thread 376, and with the decays' exponentials in
// branches, as the compiler has them by itself, 391.
// Errors against 64 bits, six shapes, 500 tokens, decays of 0.6 to 0.999 and of 0 to 0.9: 0.75 to 1.02 times those of the
// recurrence token by token, 0.94 on average.  For that a token's own key times query is summed up in double, what is added to a
// token's own part is summed up by itself, and sums over channels are four; as one or two sums and products of tiles that hold the
// own part 1.15, 1.3 where decays are strong.
// ------------------------------------------------------------------------------------------------
constexpr int QUARTER = 4, HALF = 8, SHORT = 16;
constexpr int CHANNEL_MAX_KEY = 160;   // what LDS has room for

// floats of LDS
template <int NI>
struct ChannelLds {
  static constexpr int KP = 32 * NI, ROW = KP + 4, TROW = SHORT + 4;
  // of a chunk, two stages: keys and queries with the decays from its first token on; keys with those up to its last, [channel][token];
  // decays of all its tokens; products with the queries, a tile as above, without those of a
  // token's own key and query; strengths; those
  static constexpr int K = 0, Q = SHORT * ROW, KT = Q + SHORT * ROW, FADE = KT + KP * TROW, P = FADE + KP, BETA = P + 256,
                       OWN = BETA + SHORT, STAGE = OWN + SHORT;
  // while it is prepared: per block size keys of the even tokens [HALF], keys and queries of the odd ones [2 HALF], four of each
  // in turn; decays; products with the keys and their inverse; every token's own product, a row for each 16 channels
  static constexpr int EVEN = 2 * STAGE, ODD = EVEN + 4 * HALF * ROW, DECAY = ODD + 8 * HALF * ROW, A = DECAY + SHORT * ROW,
                       INV = A + 256, DIAG = INV + 256, FLOATS = DIAG + 16 * SHORT;
};
static_assert(ChannelLds<CHANNEL_MAX_KEY / 32>::FLOATS * 4 <= 160 * 1024);

template <int NI>
__global__ __launch_bounds__(768, 1) void scan_channel_kernel(Scan p, const RowSeg *__restrict__ segs, int n_seg, int fewest) {
  using L = ChannelLds<NI>;
  constexpr int ROW = L::ROW, TROW = L::TROW, NB = 2 * NI, NG = (NI + 3) / 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int seg_id = blockIdx.x % n_seg, unit = blockIdx.x / n_seg, blocks = (p.V + 63) / 64;
  const RowSeg seg = segs[seg_id];
  if (seg.n < fewest) return;   // taken elsewhere
  if (unit >= p.heads * blocks) {   // workgroups of the convolutions' states come last, of 256 threads
    if (threadIdx.x < 256) advance_conv_state(p, seg, unit - p.heads * blocks, gridDim.x / n_seg - p.heads * blocks);
    return;
  }
  const int h = unit / blocks, kh = h / (p.heads / p.key_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, c = lane >> 4;
  const uint32_t ld4 = 4 * p.ld_conv;
  auto at4 = [&](const float *a) { return *reinterpret_cast<const f32x4 *>(a); };
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid < 256) lds[L::A + tid] = lds[L::P + tid] = lds[L::STAGE + L::P + tid] = 0.f;   // what no pair s < t writes stays zero

  if (wave >= 4) {
    const int w8 = wave - 4, t8 = tid - 256;
    const float rate = expf(p.a_log[h]);
    // Inputs travel through registers, four channels of a token at a time, and to LDS as they are but for the decays, a chunk
    // before the operands are made of them (loading every thread's own channel instead took 2200 cycles of a chunk's 9700)
    f32x4 bias[NG], rk[NG], rq[NG], rg[NG];
    float r_beta = 0.f;
    auto place = [&](int g, int &t, int &d) {
      const int idx = t8 + 512 * g;
      t = idx / (L::KP / 4);
      d = idx % (L::KP / 4) * 4;
      return t < SHORT;
    };
    int t, d;
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (place(g, t, d))
#pragma unroll
        for (int e = 0; e < 4; e++) bias[g][e] = p.dt_bias[h * p.K + min(d, p.K - 4) + e];
    const uint32_t ldg4 = 4 * p.ld_decay;
    auto fetch = [&](int t0) {
      const int T = min(SHORT, seg.n - t0);
      const char *rows = reinterpret_cast<const char *>(p.conv + (size_t)(seg.row0 + t0) * p.ld_conv);
      const char *ks = rows + 4 * (size_t)(p.k_col + kh * p.K), *qs = rows + 4 * (size_t)(p.q_col + kh * p.K);
      const char *gs = reinterpret_cast<const char *>(p.channel_decay + (size_t)(seg.row0 + t0) * p.ld_decay + h * p.K);
      int t, d;
#pragma unroll
      for (int g = 0; g < NG; g++)
        if (place(g, t, d)) {
          t = min(t, T - 1);
          const uint32_t d4 = 4 * min(d, p.K - 4);
          rg[g] = *reinterpret_cast<const f32x4 *>(gs + __umul24(t, ldg4) + d4);
          rk[g] = *reinterpret_cast<const f32x4 *>(ks + __umul24(t, ld4) + d4);
          rq[g] = *reinterpret_cast<const f32x4 *>(qs + __umul24(t, ld4) + d4);
        }
      if (w8 == 7) r_beta = p.in[(size_t)(seg.row0 + t0 + min(n, T - 1)) * p.ld_in + p.beta_col + h];
    };
    // tokens and channels outside the problem: zero, and no decay
    auto put_inputs = [&](int t0, float *stage) {
      const int T = min(SHORT, seg.n - t0);
      int t, d;
#pragma unroll
      for (int g = 0; g < NG; g++)
        if (place(g, t, d)) {
          const bool real = t < T && d < p.K;
          f32x4 a;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float decay = exp_f(-rate * softplus_f(rg[g][e] + bias[g][e]));
            asm("" : "+v"(decay));   // whether real or not: a branch around each costs more
            a[e] = real ? decay : 1.f;
            rk[g][e] = real ? rk[g][e] : 0.f;
            rq[g][e] = real ? rq[g][e] : 0.f;
          }
          *reinterpret_cast<f32x4 *>(lds + L::DECAY + t * ROW + d) = a;
          *reinterpret_cast<f32x4 *>(stage + L::K + t * ROW + d) = rk[g];
          *reinterpret_cast<f32x4 *>(stage + L::Q + t * ROW + d) = rq[g];
        }
      if (w8 == 7 && lane < SHORT) stage[L::BETA + lane] = lane < T ? sigmoid_f(r_beta) : 0.f;
    };
    // operands: this thread's tokens 4 c .. of channels 16 (w8 + 8 g) + n
    auto put = [&](float *stage) {
      double diag[QUARTER];
#pragma unroll
      for (int i = 0; i < QUARTER; i++) diag[i] = 0.0;
#pragma unroll
      for (int g = 0; g < NG; g++)
        if (w8 + 8 * g < NB) {
          const int ch = 16 * (w8 + 8 * g) + n;
          float a[QUARTER], k[QUARTER], q[QUARTER], until[QUARTER], behind[QUARTER];   // products of decays up to and with a token, behind it
#pragma unroll
          for (int i = 0; i < QUARTER; i++) {
            a[i] = lds[L::DECAY + (c * QUARTER + i) * ROW + ch];
            k[i] = stage[L::K + (c * QUARTER + i) * ROW + ch];
            q[i] = stage[L::Q + (c * QUARTER + i) * ROW + ch];
          }
#pragma unroll
          for (int i = 0; i < QUARTER; i++) {
            diag[i] += (double)k[i] * (double)q[i];
            until[i] = i ? until[i - 1] * a[i] : a[i];
          }
          behind[QUARTER - 1] = 1.f;
#pragma unroll
          for (int i = QUARTER - 2; i >= 0; i--) behind[i] = behind[i + 1] * a[i + 1];
          // of whole quarters: this one, its neighbour in the half, the other half
          const float all = until[QUARTER - 1], beside = lane_xor<16>(all), other = lane_xor<32>(all * beside);
          const float before8 = c & 1 ? beside : 1.f, after8 = c & 1 ? 1.f : beside;
          const float before = c & 2 ? before8 * other : before8, after = c & 2 ? after8 : after8 * other;
          if (c == 0) stage[L::FADE + ch] = all * beside * other;
          f32x4 kt;
#pragma unroll
          for (int i = 0; i < QUARTER; i++) {
            stage[L::K + (c * QUARTER + i) * ROW + ch] = k[i] * (before * until[i]);
            stage[L::Q + (c * QUARTER + i) * ROW + ch] = q[i] * (before * until[i]);
            kt[i] = k[i] * (behind[i] * after);
          }
          *reinterpret_cast<f32x4 *>(stage + L::KT + ch * TROW + c * QUARTER) = kt;
          // `at`: place among the even or the odd tokens
          auto even_token = [&](int l, int at, float key) { lds[L::EVEN + (l * HALF + at) * ROW + ch] = key; };
          auto odd_token = [&](int l, int at, float key, float query) {
            float *to = lds + L::ODD + (l * SHORT + at + (at & 4)) * ROW + ch;
            to[0] = key;
            to[4 * ROW] = query;
          };
          // blocks of 1 and 2 lie within the thread's tokens
          even_token(0, 2 * c, k[0]);
          odd_token(0, 2 * c, k[1] * a[1], q[1] * a[1]);
          even_token(0, 2 * c + 1, k[2]);
          odd_token(0, 2 * c + 1, k[3] * a[3], q[3] * a[3]);
          even_token(1, 2 * c, k[0] * a[1]);
          even_token(1, 2 * c + 1, k[1]);
          odd_token(1, 2 * c, k[2] * a[2], q[2] * a[2]);
          odd_token(1, 2 * c + 1, k[3] * (a[2] * a[3]), q[3] * (a[2] * a[3]));
#pragma unroll
          for (int l = 2; l < 4; l++) {   // quarters, halves
            const bool odd = c & (l == 2 ? 1 : 2);
            const float far = l == 2 ? 1.f : odd ? before8 : after8;
            const int first = l == 2 ? (c >> 1) * 4 : (c & 1) * 4;
            float *to = lds + (odd ? L::ODD + (l * SHORT + 2 * first) * ROW : L::EVEN + (l * HALF + first) * ROW) + ch;
#pragma unroll
            for (int i = 0; i < QUARTER; i++) {
              const float w = far * (odd ? until[i] : behind[i]);
              to[i * ROW] = k[i] * w;
              if (odd) to[(4 + i) * ROW] = q[i] * w;
            }
          }
        }
      // a token's key and query, without decays: sums over the wave's channels
#pragma unroll
      for (int i = 0; i < QUARTER; i++) {
        diag[i] += lane_xor<8>(diag[i]);
        diag[i] += lane_xor<4>(diag[i]);
        diag[i] += lane_xor<2>(diag[i]);
        diag[i] += lane_xor<1>(diag[i]);
      }
      if (n == 0)
#pragma unroll
        for (int i = 0; i < QUARTER; i++) reinterpret_cast<double *>(lds + L::DIAG)[w8 * SHORT + c * QUARTER + i] = diag[i];
    };
    // pairs of tokens that blocks of 2^w8 part: rows the even tokens' keys, columns the odd tokens' keys and queries
    auto products = [&](float *stage) {
      const float *x0 = lds + L::EVEN + (w8 * HALF + (n & 7)) * ROW + 4 * c, *y0 = lds + L::ODD + (w8 * SHORT + n) * ROW + 4 * c;
      f32x4 sum[2][2] = {{zero, zero}, {zero, zero}}, x[2][2], y[2][2];
      auto load = [&](int i) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
          x[i & 1][b] = at4(x0 + 16 * (2 * i + b));
          y[i & 1][b] = at4(y0 + 16 * (2 * i + b));
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
          for (int b = 0; b < 2; b++) sum[b][e & 1] = mfma4(x[i & 1][b][e], y[i & 1][b][e], sum[b][e & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      const int i = (n >> 1 & 4) + (n & 3), low = (1 << w8) - 1, t = ((i & ~low) << 1) + low + 1 + (i & low);
      const bool query = n & 4;
      const float scale = query ? 1.f : stage[L::BETA + t];
      float *to = query ? stage + L::P : lds + L::A;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int j = 4 * c + e, s = ((j & ~low) << 1) + (j & low);
        if (c < 2 && (i & ~low) == (j & ~low)) to[((s >> 2) * 16 + t) * 4 + (s & 3)] = scale * ((sum[0][0][e] + sum[0][1][e]) + (sum[1][0][e] + sum[1][1][e]));
      }
    };
    fetch(0);
    put_inputs(0, lds);
    if (SHORT < seg.n) fetch(SHORT);
    __syncthreads();
    for (int t0 = -SHORT, at = 0; t0 < seg.n; t0 += SHORT, at ^= 1) {   // the chunk at t0 is worked on; the next one:
      const bool more = t0 + SHORT < seg.n;
      float *stage = lds + at * L::STAGE;
      if (more) put(stage);
      __syncthreads();
      if (t0 + 2 * SHORT < seg.n) put_inputs(t0 + 2 * SHORT, lds + (at ^ 1) * L::STAGE);   // whose keys and queries are done with
      if (t0 + 3 * SHORT < seg.n) fetch(t0 + 3 * SHORT);
      if (more && w8 < 4) products(stage);
      if (more && w8 == 4 && lane < SHORT) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < 8; w++) sum += reinterpret_cast<const double *>(lds + L::DIAG)[w * SHORT + n];
        stage[L::OWN + n] = (float)sum;
      }
      __syncthreads();
    }
    return;
  }

  const int c0 = (unit - h * blocks) * 64 + wave * 16, col = min(c0 + n, p.V - 1);   // columns c0 .. + 15 of the wave
  const bool live = c0 + n < p.V;
  f32x4 S[NB];   // keys 16 b + 4 c + e of column c0 + n
  float *st = p.state + (((size_t)seg.slot * p.heads + h) * p.V + col) * L::KP + 4 * c;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    S[b] = zero;
    if (seg.pos0 > 0 && live) S[b] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(st + 16 * b));
  }
  float rv[4];
  auto fetch = [&](int t0) {
    const int T = min(SHORT, seg.n - t0);
    const char *vs = reinterpret_cast<const char *>(p.conv + (size_t)(seg.row0 + t0) * p.ld_conv + p.v_col + h * p.V);
#pragma unroll
    for (int e = 0; e < 4; e++) rv[e] = *reinterpret_cast<const float *>(vs + __umul24(min(4 * c + e, T - 1), ld4) + 4 * col);
  };
  fetch(0);
  for (int i = 0; i < 3; i++) __syncthreads();   // the first chunk is prepared
  for (int t0 = 0, at = 0; t0 < seg.n; t0 += SHORT, at ^= 1) {
    const int T = min(SHORT, seg.n - t0);
    const float *stage = lds + at * L::STAGE;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = 4 * c + e < T && live ? rv[e] : 0.f;
    if (t0 + SHORT < seg.n) fetch(t0 + SHORT);
    // what the state in front of the chunk gives: [token][column]
    const float *q = stage + L::Q + n * ROW + 4 * c, *k = stage + L::K + n * ROW + 4 * c;
    f32x4 o2[4] = {zero, zero, zero, zero}, r2[4] = {zero, zero, zero, zero}, qx[3], kx[3];
    auto load = [&](int b) {
      qx[b % 3] = at4(q + 16 * b);
      kx[b % 3] = at4(k + 16 * b);
    };
    load(0);
    load(1);
#pragma unroll
    for (int b = 0; b < NB; b++) {
      if (b + 2 < NB) load(b + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        o2[e] = mfma4(qx[b % 3][e], S[b][e], o2[e]);
        r2[e] = mfma4(kx[b % 3][e], S[b][e], r2[e]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const f32x4 be = at4(stage + L::BETA + 4 * c), pt = at4(stage + L::P + lane * 4), own = at4(stage + L::OWN + 4 * c);
    f32x4 u, o = (o2[0] + o2[1]) + (o2[2] + o2[3]);
#pragma unroll
    for (int e = 0; e < 4; e++) u[e] = be[e] * (v[e] - ((r2[0][e] + r2[1][e]) + (r2[2][e] + r2[3][e])));
    if (wave == 0 && lane < SHORT) invert_tile<false>(lds + L::A, lds + L::INV, 0.f, n);
    __syncthreads();

    const f32x4 inv = at4(lds + L::INV + lane * 4);
    const float *keys = stage + L::KT + n * TROW + 4 * c, *fade = stage + L::FADE + 4 * c;
    f32x4 kt[2][2], fd[2][2];
    auto load_keys = [&](int i) {
#pragma unroll
      for (int b = 0; b < 2; b++) {
        kt[i & 1][b] = at4(keys + 16 * (2 * i + b) * TROW);
        fd[i & 1][b] = at4(fade + 16 * (2 * i + b));
      }
    };
    load_keys(0);
    // (what is added to a token's own part is summed up by itself: small sums round less)
    f32x4 w = zero;
#pragma unroll
    for (int e = 0; e < 4; e++) w = mfma4(inv[e], u[e], w);
    w += u;
    const bool careful = any_not_finite(w[0] + w[1] + w[2] + w[3]);
    if (careful) {
      w = tile_below(zero, lds + L::INV, u, false, lane) + u;
      o = tile_below(o, stage + L::P, w, false, lane);
    }
    // the state behind the chunk, and what its own tokens give
#pragma unroll
    for (int i = 0; i < NI; i++) {
      if (i + 1 < NI) load_keys(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2; b++) S[2 * i + b] *= fd[i & 1][b];
#pragma unroll
      for (int e = 0; e < 4; e++) {
#pragma unroll
        for (int b = 0; b < 2; b++) S[2 * i + b] = mfma4(kt[i & 1][b][e], w[e], S[2 * i + b]);
        if (i == 0 && !careful) o = mfma4(pt[e], w[e], o);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    char *out = reinterpret_cast<char *>(p.out + (size_t)(seg.row0 + t0) * p.ld_out + h * p.V);
    const uint32_t out4 = 4 * p.ld_out, first = __umul24(4 * c, out4) + 4 * (c0 + n);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      o[e] = fmaf(own[e], w[e], o[e]);
      float *to = reinterpret_cast<float *>(out + e * out4 + first);
      if (T == SHORT && c0 + 16 <= p.V) *to = o[e];
      else if (live && 4 * c + e < T) *to = o[e];
    }
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int b = 0; b < NB; b++) __builtin_nontemporal_store(S[b], reinterpret_cast<f32x4 *>(st + 16 * b));
  }
}

bool scan_chunks_apply(const Scan &p, const StepRows &r) {
  return p.kind != SCAN_RETENTION && r.longest >= SCAN_CHUNK_ROWS && scan_reads_wide(p) && p.K >= 4 &&
         p.K <= (p.kind == SCAN_CHANNEL_DELTA ? CHANNEL_MAX_KEY : SCAN_MAX_KEY) &&
         p.ld_conv < (1 << 22) && p.ld_decay < (1 << 22) && p.ld_out < (1 << 22);   // (24-bit row pitches)
}

template <int NI, int KIND>
static int launch_chunks(const Scan &p, const StepRows &r, int fewest, hipStream_t s) {
  constexpr bool CHANNEL = KIND == SCAN_CHANNEL_DELTA;
  constexpr int bytes = (CHANNEL ? ChannelLds<NI>::FLOATS : ChunkLds<NI>::FLOATS) * (int)sizeof(float);
  auto kern = [] {
    if constexpr (CHANNEL) return scan_channel_kernel<NI>;
    else return scan_chunk_kernel<NI, KIND>;
  }();
  GPTOSS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  TraceScope ts(CHANNEL ? "scan_channel_delta" : KIND == SCAN_DELTA ? "scan_delta" : "scan_state_space", s);
  const size_t grid = (size_t)r.n_seg * (p.heads * cdiv(p.V, 64) + cdiv(p.conv_desc.channels, 256));
  kern<<<(unsigned)grid, CHANNEL ? 768 : 256, bytes, s>>>(p, r.segs, r.n_seg, fewest);
  GPTOSS_LAUNCH_CHECK("scan_chunk_kernel");
  return GPTOSS_OK;
}

template <int KIND>
static int launch_kind(const Scan &p, const StepRows &r, int fewest, hipStream_t s) {
  switch (scan_key_pad(p.K) / 32) {
    case 1: return launch_chunks<1, KIND>(p, r, fewest, s);
    case 2: return launch_chunks<2, KIND>(p, r, fewest, s);
    case 3: return launch_chunks<3, KIND>(p, r, fewest, s);
    case 4: return launch_chunks<4, KIND>(p, r, fewest, s);
    case 5: return launch_chunks<5, KIND>(p, r, fewest, s);
    case 6: return launch_chunks<6, KIND>(p, r, fewest, s);
    default: break;
  }
  if constexpr (KIND != SCAN_CHANNEL_DELTA) {
    if (scan_key_pad(p.K) / 32 == 7) return launch_chunks<7, KIND>(p, r, fewest, s);
    return launch_chunks<8, KIND>(p, r, fewest, s);
  }
  return fail(GPTOSS_ERR_DIM, "scan: keys of %d per channel do not go by chunks", p.K);
}

int run_scan_chunks(const Scan &p, const StepRows &r, hipStream_t s) {
  GPTOSS_REQUIRE(scan_chunks_apply(p, r) && p.V >= 1 && p.key_heads >= 1 && p.heads % p.key_heads == 0, GPTOSS_ERR_DIM,
                 "scan: kind %d with keys of %d, %d heads over %d does not go by chunks", (int)p.kind, p.K, p.heads, p.key_heads);
  GPTOSS_REQUIRE(r.n_seg * ((long long)p.heads * cdiv(p.V, 64) + cdiv(p.conv_desc.channels, 256)) < (1ll << 31), GPTOSS_ERR_DIM,
                 "scan: too many workgroups");
  // Decoding rows beside the stretches: a chunk of one token takes a CU as long as a full one, which is nothing while there are
  // CUs to spare; with more of them than run at a time they go as a step of their own.
  int fewest = 1;
  if ((long long)r.n_singles * p.heads * cdiv(p.V, 64) > 512) {
    StepRows single = r;
    single.segs = r.singles;
    single.n_seg = r.n_singles;
    single.longest = 1;
    GPTOSS_STEP(run_scan(p, single, s));
    fewest = 2;
  }
  switch (p.kind) {
    case SCAN_DELTA: return launch_kind<SCAN_DELTA>(p, r, fewest, s);
    case SCAN_CHANNEL_DELTA: return launch_kind<SCAN_CHANNEL_DELTA>(p, r, fewest, s);
    default: return launch_kind<SCAN_STATE_SPACE>(p, r, fewest, s);
  }
}

}  // namespace gptoss
