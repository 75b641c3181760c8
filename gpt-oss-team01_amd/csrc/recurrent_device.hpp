// What the kernels of the recurrences share (recurrent.hip, scan_chunks.hip).
#pragma once
#include "recurrent.hpp"

namespace gptoss {

// On the hardware's exp2, log2 and reciprocal (about one unit in the last place each), which keeps these
// within a few units: the argument of an exponential that matters is small.
__device__ __forceinline__ float exp_f(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float sigmoid_f(float z) { return __builtin_amdgcn_rcpf(1.f + exp_f(-z)); }
__device__ __forceinline__ float silu_f(float z) { return z * sigmoid_f(z); }
// max(z, 0) + log(1 + e), e = exp(-|z|).  With u = 1 + e rounded, log(u) e / (u - 1) is log(1 + e) to a few
// units in the last place however small e is (W. Kahan's form of log1p).
__device__ __forceinline__ float softplus_f(float z) {
  const float e = exp_f(-fabsf(z)), u = 1.f + e, d = u - 1.f;
  const float l = __builtin_amdgcn_logf(u) * 0.6931471805599453f * e * __builtin_amdgcn_rcpf(d);
  return fmaxf(z, 0.f) + (d == 0.f ? e : l);
}

// The convolution's last taps - 1 inputs after the stretch; one thread owns a channel.  All are read before the first is
// written (they move within the same memory).
__device__ __forceinline__ void advance_conv_state(const Scan &p, const RowSeg &seg, int part, int parts) {
  const ShortConv &c = p.conv_desc;
  const int keep = c.taps - 1;
  for (int ch = part * 256 + threadIdx.x; ch < c.channels; ch += parts * 256) {
    float *st = p.conv_state + (size_t)seg.slot * keep * c.channels + ch;
    auto value = [&](int i) {
      const int t = seg.n - keep + i;   // row of the stretch whose input belongs here; negative: an older one
      if (t >= 0) return p.in[(size_t)(seg.row0 + t) * p.ld_in + c.col + ch];
      return seg.pos0 + t >= 0 ? st[(size_t)(i + seg.n) * c.channels] : 0.f;
    };
    constexpr int ROOM = 8;
    if (keep <= ROOM) {
      float v[ROOM];
#pragma unroll
      for (int i = 0; i < ROOM; i++) v[i] = i < keep ? value(i) : 0.f;
#pragma unroll
      for (int i = 0; i < ROOM; i++)
        if (i < keep) st[(size_t)i * c.channels] = v[i];
    } else {
      for (int i = 0; i < keep; i++) st[(size_t)i * c.channels] = value(i);   // (each is read before an earlier place is written)
    }
  }
}

// sum over 8 consecutive lanes: two exchanges inside a quad, then the mirrored half row
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum8(float v) {
  v = dpp_add<0xB1>(v);    // quad_perm [1,0,3,2]
  v = dpp_add<0x4E>(v);    // quad_perm [2,3,0,1]
  return dpp_add<0x141>(v);  // row_half_mirror
}

constexpr int SCAN_TOKENS = 16;   // tokens staged at a time

// What a lane needs of one token.
template <int NI, bool CHANNEL, int CPL>
struct ScanToken {
  f32x4 k[NI], q[NI], g[CHANNEL ? NI : 1];
  float v[CPL], decay, beta;
};

// LDS of a workgroup: one token more than is staged, as the loop reads a token ahead
template <int NI, int KIND, bool ONE, int CPL>
struct ScanLds {
  static constexpr int KP = 32 * NI, TC = ONE ? 1 : SCAN_TOKENS, COLS = 32 * CPL;
  float k[TC + 1][KP], q[TC + 1][KP], g[KIND == SCAN_CHANNEL_DELTA ? TC + 1 : 1][KP], v[TC + 1][COLS];
  float decay[TC + 1], beta[TC + 1];
};

// The recurrence over one stretch, token by token, for columns c0 .. of head h, by a workgroup of 256 threads.
// CPL: columns per lane; a workgroup has 4 waves x 8 lane groups x CPL columns.  Two share the reads of a
// token's keys and queries; one gives twice the workgroups, where there are few heads and sequences.
// ONE: every sequence has one row (decoding); the launch is then a stream of states through the chip.
template <int NI, int KIND, bool ONE, int CPL>
__device__ __forceinline__ void scan_stretch(const Scan &p, const RowSeg &seg, int h, int c0, ScanLds<NI, KIND, ONE, CPL> &l) {
  constexpr int KP = 32 * NI, TC = ONE ? 1 : SCAN_TOKENS;
  constexpr bool CHANNEL = KIND == SCAN_CHANNEL_DELTA, SSM = KIND == SCAN_STATE_SPACE, RET = KIND == SCAN_RETENTION;
  constexpr int COLS = 32 * CPL;
  constexpr int PIECES = (TC * KP / 4 + 255) / 256, VPIECES = (TC * COLS / 4 + 255) / 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 7;
  const int cw = (wave * 8 + (lane >> 3)) * CPL;   // this lane's first column is c0 + cw
  const bool busy = c0 + wave * 8 * CPL < p.V;   // wave-uniform
  const int kh = h / (p.heads / p.key_heads);
  const float rate = RET ? 0.f : expf(p.a_log[h]);
  const float bias = CHANNEL || RET ? 0.f : p.dt_bias[h];
  const float fixed = RET ? p.head_decay[h] : 0.f;
  const float skip = SSM ? p.d_skip[h] : 0.f;

  f32x4 S[CPL][NI];
  float *st = p.state + (((size_t)seg.slot * p.heads + h) * p.V + c0 + cw) * KP + 4 * j;
#pragma unroll
  for (int c = 0; c < CPL; c++)
#pragma unroll
    for (int i = 0; i < NI; i++) {
      S[c][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (seg.pos0 > 0 && c0 + cw + c < p.V)
        S[c][i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(st + c * KP + 32 * i));
    }

  // the next tokens' inputs travel through registers, four values at a time, while the current ones are
  // worked on; rows and columns outside the problem are read from inside it and replaced by zero
  f32x4 rk[PIECES], rq[PIECES], rg[CHANNEL ? PIECES : 1], rv[VPIECES];
  float r_beta = 0.f, r_decay = 0.f;
  const float *k_src = p.conv + p.k_col + kh * p.K, *q_src = p.conv + p.q_col + kh * p.K;
  const float *v_src = p.conv + p.v_col + h * p.V, *g_src = p.channel_decay + h * p.K;
  auto load4 = [&](const float *row, int d, int limit) {
    f32x4 x;
    if (p.vec) {
      x = *reinterpret_cast<const f32x4 *>(row + min(d, limit - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = row[min(d + e, limit - 1)];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = d + e < limit ? x[e] : 0.f;
    return x;
  };
  auto fetch = [&](int t0) {
    const int T = min(TC, seg.n - t0);
    const size_t first = seg.row0 + t0;
#pragma unroll
    for (int x = 0; x < PIECES; x++) {
      const int idx = tid + 256 * x, t = min(idx / (KP / 4), T - 1), d = idx % (KP / 4) * 4;
      const float *kr = k_src + (first + t) * p.ld_conv, *qr = q_src + (first + t) * p.ld_conv;
      rk[x] = load4(kr, d, p.K);
      rq[x] = load4(qr, d, p.K);
      if constexpr (RET && ONE) {
        const int half = p.rot.table ? p.rot.dims >> 1 : 0;
        if (d < 2 * half) {   // pairs (i, i + half)
          const bool second = d >= half;
          const int i = second ? d - half : d, partner = second ? i : i + half;
          const f32x4 ko = load4(kr, partner, p.K), qo = load4(qr, partner, p.K);
          const f32x4 *at = reinterpret_cast<const f32x4 *>(p.rot.table + ((size_t)seg.pos0 * half + i) * 2);
          const f32x4 cs[2] = {at[0], at[1]};
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float c = cs[e >> 1][2 * (e & 1)], s = (second ? 1.f : -1.f) * cs[e >> 1][2 * (e & 1) + 1];
            rk[x][e] = rk[x][e] * c + ko[e] * s;
            rq[x][e] = rq[x][e] * c + qo[e] * s;
          }
        }
      }
      if (CHANNEL) rg[x] = load4(g_src + (first + t) * p.ld_decay, d, p.K);
    }
#pragma unroll
    for (int x = 0; x < VPIECES; x++) {
      const int idx = tid + 256 * x, t = min(idx / (COLS / 4), T - 1), c = c0 + idx % (COLS / 4) * 4;
      rv[x] = load4(v_src + (first + t) * p.ld_conv, c, p.V);
    }
    if (RET) return;
    const float *ir = p.in + (first + min(tid, T - 1)) * p.ld_in + h;
    if (!SSM) r_beta = ir[p.beta_col];
    if (!CHANNEL) r_decay = ir[p.decay_col];
  };
  auto put = [&]() {
#pragma unroll
    for (int x = 0; x < PIECES; x++) {
      const int idx = tid + 256 * x, t = idx / (KP / 4), d = idx % (KP / 4) * 4;
      if (TC * KP / 4 % 256 == 0 || t < TC) {
        *reinterpret_cast<f32x4 *>(&l.k[t][d]) = rk[x];
        *reinterpret_cast<f32x4 *>(&l.q[t][d]) = rq[x];
        if (CHANNEL) {
          f32x4 g;
#pragma unroll
          for (int e = 0; e < 4; e++)
            g[e] = exp_f(-rate * softplus_f(rg[x][e] + p.dt_bias[h * p.K + min(d + e, p.K - 1)]));
          *reinterpret_cast<f32x4 *>(&l.g[t][d]) = g;
        }
      }
    }
#pragma unroll
    for (int x = 0; x < VPIECES; x++) {
      const int idx = tid + 256 * x;
      if (TC * COLS / 4 % 256 == 0 || idx < TC * COLS / 4)
        *reinterpret_cast<f32x4 *>(&l.v[0][0] + idx * 4) = rv[x];
    }
    if (!RET && tid < TC) {
      if (SSM) {
        const float dt = softplus_f(r_decay + bias);
        l.decay[tid] = exp_f(-rate * dt);
        l.beta[tid] = dt;
      } else {
        l.beta[tid] = sigmoid_f(r_beta);
        if (!CHANNEL) l.decay[tid] = exp_f(-rate * softplus_f(r_decay + bias));
      }
    }
  };
  using Token = ScanToken<NI, CHANNEL, CPL>;
  auto read = [&](Token &x, int t) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      x.k[i] = *reinterpret_cast<const f32x4 *>(&l.k[t][32 * i + 4 * j]);
      x.q[i] = *reinterpret_cast<const f32x4 *>(&l.q[t][32 * i + 4 * j]);
      if (CHANNEL) x.g[i] = *reinterpret_cast<const f32x4 *>(&l.g[t][32 * i + 4 * j]);
    }
#pragma unroll
    for (int c = 0; c < CPL; c++) x.v[c] = l.v[t][cw + c];
    if (!RET) x.beta = l.beta[t];
    if (!CHANNEL && !RET) x.decay = l.decay[t];
  };
  auto advance = [&](const Token &x, float (&o)[CPL]) {
#pragma unroll
    for (int c = 0; c < CPL; c++)
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) S[c][i][e] *= CHANNEL ? x.g[CHANNEL ? i : 0][e] : RET ? fixed : x.decay;
    float u[CPL];
#pragma unroll
    for (int c = 0; c < CPL; c++) {
      if constexpr (RET) {
        u[c] = p.value_scale * x.v[c];
      } else if constexpr (SSM) {
        u[c] = x.beta * x.v[c];
      } else {
        float d0 = 0.f, d1 = 0.f;
#pragma unroll
        for (int i = 0; i < NI; i++) {
          d0 = fmaf(S[c][i][0], x.k[i][0], d0);
          d1 = fmaf(S[c][i][1], x.k[i][1], d1);
          d0 = fmaf(S[c][i][2], x.k[i][2], d0);
          d1 = fmaf(S[c][i][3], x.k[i][3], d1);
        }
        u[c] = x.beta * (x.v[c] - sum8(d0 + d1));
      }
    }
#pragma unroll
    for (int c = 0; c < CPL; c++) {
      float d0 = 0.f, d1 = 0.f;
#pragma unroll
      for (int i = 0; i < NI; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++) S[c][i][e] = fmaf(x.k[i][e], u[c], S[c][i][e]);
        d0 = fmaf(S[c][i][0], x.q[i][0], d0);
        d1 = fmaf(S[c][i][1], x.q[i][1], d1);
        d0 = fmaf(S[c][i][2], x.q[i][2], d0);
        d1 = fmaf(S[c][i][3], x.q[i][3], d1);
      }
      o[c] = sum8(d0 + d1);
      if (SSM) o[c] = fmaf(skip, x.v[c], o[c]);
    }
  };
  // lane j of a group keeps the results of tokens t with t % 8 == j; they are stored eight at a time, those
  // of a piece's last tokens after the next piece has been staged (the wait for its loads would otherwise
  // be one for these stores)
  float keep[CPL];
  int kept = -1;   // first row of the tokens in keep; -1: stored
  auto flush = [&](int rows) {
    if (j < rows) {
      float *dst = p.out + (size_t)(kept + j) * p.ld_out + h * p.V + c0 + cw;
#pragma unroll
      for (int c = 0; c < CPL; c++)
        if (c0 + cw + c < p.V) dst[c] = keep[c];
    }
    kept = -1;
  };
  fetch(0);
  for (int t0 = 0; t0 < seg.n; t0 += TC) {
    const int T = min(TC, seg.n - t0);
    if (t0 > 0) __syncthreads();
    put();
    __syncthreads();
    if (!ONE && t0 + TC < seg.n) fetch(t0 + TC);
    if (!busy) continue;
    if (!ONE && kept >= 0) flush(8);   // a full piece came before
    auto emit = [&](int t, const float (&o)[CPL]) {
#pragma unroll
      for (int c = 0; c < CPL; c++) keep[c] = (t & 7) == j ? o[c] : keep[c];
      if ((t & 7) == 0) kept = seg.row0 + t0 + t;
      if ((t & 7) == 7 && t + 1 < TC) flush(8);
    };
    Token a;
    read(a, 0);
    if constexpr (ONE) {
      float o[CPL];
      advance(a, o);
      emit(0, o);
    } else if constexpr (NI <= 4) {
      // two tokens in registers: the next one's inputs are requested before the current one is worked on
      Token b;
      for (int t = 0; t < T; t += 2) {
        float o[CPL];
        read(b, t + 1);
        advance(a, o);
        emit(t, o);
        if (t + 1 >= T) break;
        read(a, t + 2);
        advance(b, o);
        emit(t + 1, o);
      }
    } else {
      for (int t = 0; t < T; t++) {
        float o[CPL];
        advance(a, o);
        emit(t, o);
        if (t + 1 < T) read(a, t + 1);
      }
    }
  }
  if (busy && kept >= 0) flush(seg.row0 + seg.n - kept);
#pragma unroll
  for (int c = 0; c < CPL; c++)
#pragma unroll
    for (int i = 0; i < NI; i++)
      if (c0 + cw + c < p.V)
        __builtin_nontemporal_store(S[c][i], reinterpret_cast<f32x4 *>(st + c * KP + 32 * i));
}

}  // namespace gptoss
