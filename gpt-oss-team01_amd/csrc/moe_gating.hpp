// Gating and grouping of a few tokens on the device (moe_route.hip, gemm_few_kernel.hpp).
#pragma once
#include "common.hpp"
#include "gemm.hpp"

namespace gptoss {

// ------------------------------------------------------------------------------------------------
// Top-k + softmax for one token held by a group of 32 lanes: lane j holds experts j, j+32, ...
// Selection = k rounds ordered by (value desc, expert id asc); softmax over the k picked values with exp in float and the
// sum and division in double (run.cpp:319-337).  Every lane of the group must call; lane s writes pick s.
// A logit that is no number ranks as -infinity: whatever a token's row holds, its picks are k different experts, so that
// its pairs cannot displace those of other tokens.  The weights of a token that picks one are no numbers.
// A small launch waits for this from end to end, so every round is short: values as integers of the same order, their
// largest by five exchanges, its holder by a ballot, and the exponentials and divisions of all picks at once, one per
// lane.  The router kernel, one token over 32 experts 10.8 -> 9.2 us, twelve 12.8 -> 10.8 (before, value and expert went
// through every exchange, and one lane computed all weights).
// ------------------------------------------------------------------------------------------------
template <int NJ, int KMAX = 8>
__device__ __forceinline__ void topk_softmax_group(const float (&v)[NJ], int sub, int E, int k,
                                                   bool live, float *__restrict__ w_out,
                                                   int *__restrict__ i_out, int *i_copy = nullptr) {
  uint32_t key[NJ], nan = 0;   // 0: not to be picked (any longer)
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const bool no_number = v[j] != v[j];
    const uint32_t u = __float_as_uint((no_number ? -INFINITY : v[j]) + 0.f);   // (zeros of either sign are equal)
    key[j] = sub + 32 * j < E ? ((int)u < 0 ? ~u : u | 0x80000000u) : 0u;
    nan |= (no_number ? 1u : 0u) << j;
  }
  float top = 0.f, mine = 0.f;   // the largest value, and pick number `sub`
  int my_id = 0;
  bool no_number = false;
#pragma unroll
  for (int s = 0; s < KMAX; s++) {
    if (s < k) {
      uint32_t best = key[0];
      int slot = 0;
#pragma unroll
      for (int j = 1; j < NJ; j++) {
        slot = key[j] > best ? j : slot;
        best = max(best, key[j]);
      }
      uint32_t all = best;
      butterfly<32>([&](auto m) { all = max(all, lane_xor<decltype(m)::value>(all)); });
      // the lowest expert among those that hold it
      int id = 0;
      bool found = false;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const uint32_t holders = (uint32_t)(__ballot(best == all && slot == j) >> (threadIdx.x & 32));
        if (!found && holders != 0) id = __builtin_ctz(holders) + 32 * j;
        found = found || holders != 0;
      }
      const bool won = (id & 31) == sub;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const bool taken = won && (id >> 5) == j;
        no_number = no_number || (taken && ((nan >> j) & 1u));
        key[j] = taken ? 0u : key[j];
      }
      const float value = __uint_as_float((int)all < 0 ? all & 0x7fffffffu : ~all);
      if (s == 0) top = value;
      mine = sub == s ? value : mine;
      my_id = sub == s ? id : my_id;
    }
  }
  const bool no_numbers = (uint32_t)(__ballot(no_number) >> (threadIdx.x & 32)) != 0;
  const float ex = sub < k ? expf(mine - top) : 0.f;
  double sum = 0.0;
#pragma unroll
  for (int s = 0; s < KMAX; s++) {
    if (s < k) {
      const float lower = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_int(ex), s));
      const float upper = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_int(ex), 32 + s));
      sum += (threadIdx.x & 32) ? upper : lower;
    }
  }
  if (live && sub < k) {
    w_out[sub] = no_numbers ? NAN : (float)((double)ex / sum);
    i_out[sub] = my_id;
    if (i_copy) i_copy[sub] = my_id;
  }
}

// A token's logit of expert e from the router's partial products (RouterParts), in the order of router_gemm_kernel's sum.
struct PartialLogit {
  float part[ROUTER_WAVES], bias;
  __device__ __forceinline__ void load(const RouterParts &r, int row, int e) {
    row = min(row, r.B - 1);
    e = min(e, r.E - 1);
    bias = r.bias ? r.bias[e] : 0.f;
#pragma unroll
    for (int w = 0; w < ROUTER_WAVES; w++) part[w] = r.parts[((size_t)w * r.B + row) * r.E + e];
  }
  __device__ __forceinline__ float sum(const RouterParts &r) const {
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < ROUTER_WAVES; w++) x += part[w];
    return r.bias ? x + bias : x;
  }
};

}  // namespace gptoss
