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

}  // namespace gptoss
