// Shared device/host helpers for the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "../../include/gptoss_mi355.h"

namespace gptoss {

// ---- error plumbing (host) -------------------------------------------------------------------
void set_error(const char *fmt, ...);
int fail(int code, const char *fmt, ...);

#define GPTOSS_REQUIRE(cond, code, ...)                 \
  do {                                                  \
    if (!(cond)) return ::gptoss::fail(code, __VA_ARGS__); \
  } while (0)

#define GPTOSS_HIP(call)                                                                       \
  do {                                                                                         \
    hipError_t err__ = (call);                                                                 \
    if (err__ != hipSuccess)                                                                   \
      return ::gptoss::fail(GPTOSS_ERR_HIP, "%s: %s (%s:%d)", #call, hipGetErrorString(err__), \
                            __FILE__, __LINE__);                                               \
  } while (0)

#define GPTOSS_LAUNCH_CHECK(name)                                                           \
  do {                                                                                      \
    hipError_t err__ = hipGetLastError();                                                   \
    if (err__ != hipSuccess)                                                                \
      return ::gptoss::fail(GPTOSS_ERR_HIP, "launch %s: %s", name, hipGetErrorString(err__)); \
  } while (0)

// ---- kernel timing hook (host) ----------------------------------------------------------------
// When the calling thread has armed a trace (gptoss_trace_set), every kernel launch made by an
// entry point is bracketed by a start/stop event pair on the launch stream.
struct TraceScope {
  TraceScope(const char *name, hipStream_t stream);
  ~TraceScope();
  int slot;
  hipStream_t stream;
};

static inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// ---- device types ----------------------------------------------------------------------------
typedef uint16_t bf16_t;  // raw bf16 bits
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int WAVE = 64;

__device__ __forceinline__ float bf16_to_f32(bf16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

// round-to-nearest-even, NaN stays NaN: gfx950 converts in hardware (v_cvt_pk_bf16_f32)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  return __builtin_bit_cast(bf16_t, static_cast<__bf16>(f));
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// A pointer to data that nothing writes while the kernel runs, in the constant address space: a load
// through it with a wave-uniform address is a scalar load whatever the kernel stores or clobbers
// elsewhere (a generic pointer falls back to vector loads once the compiler sees a possible writer,
// an asm statement with a memory clobber included).
template <typename T>
using const_as = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ const_as<T> constant_ptr(const T *q) {
  return (const_as<T>)(q);
}

// 16 bytes per lane, from sbase + voff (an unsigned offset) to LDS address lds + 16 * lane.  The compiler does not count these
// loads: whoever reads what they bring waits for the vector-memory counter by itself first.
__device__ __forceinline__ void load_to_lds(unsigned lds, uint32_t voff, const void *sbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(voff), "s"(sbase)
               : "memory");
}
// The same from an address of each lane's own.
__device__ __forceinline__ void load_to_lds(unsigned lds, const void *from) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(from)
               : "memory");
}

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) {
  union {
    u32x4 u;
    bf16x8 b;
  } c;
  c.u = v;
  return c.b;
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }

// ---- exchanges between lanes ---------------------------------------------------------------------
// The value of lane (own ^ M), every lane active: moves inside a row of 16 lanes and swaps of rows, in registers.  A
// shuffle goes through LDS and takes over a hundred cycles, and a reduction waits for six of them one after the other,
// which is what the small kernels of a decoding step did for a good part of their few microseconds.
template <int M>
__device__ __forceinline__ uint32_t lane_xor_bits(uint32_t v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16 || M == 32);
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);    // quad_perm [1,0,3,2]
  if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);    // quad_perm [2,3,0,1]
  if constexpr (M == 4)   // half a row mirrored (^ 7), then every quad mirrored (^ 3)
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
  if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);   // row_ror 8
  if constexpr (M == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);   // [0]: rows 0 0 2 2, [1]: rows 1 1 3 3
    return (threadIdx.x & 16) ? s[0] : s[1];
  }
  if constexpr (M == 32) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);   // [0]: the lower half twice, [1]: the upper
    return (threadIdx.x & 32) ? s[0] : s[1];
  }
}
template <int M, typename T>
__device__ __forceinline__ T lane_xor(T v) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8);
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, lane_xor_bits<M>(__builtin_bit_cast(uint32_t, v)));
  } else {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(T, (uint64_t)lane_xor_bits<M>((uint32_t)(u >> 32)) << 32 | lane_xor_bits<M>((uint32_t)u));
  }
}

// f(integral_constant<M>) for M = N / 2, N / 4, .. 1: the steps of a butterfly over N lanes
template <int N, typename F>
__device__ __forceinline__ void butterfly(F &&f) {
  if constexpr (N > 1) {
    f(std::integral_constant<int, N / 2>{});
    butterfly<N / 2>(f);
  }
}

// The sum over N consecutive lanes (N a power of two), in all of them.
template <int N = WAVE, typename T>
__device__ __forceinline__ T lanes_sum(T v) {
  butterfly<N>([&](auto m) { v += lane_xor<decltype(m)::value>(v); });
  return v;
}

// The largest value of the four lanes n, n + 16, n + 32, n + 48, in all of them, without a trip through LDS.
__device__ __forceinline__ float max_over_quarters(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const uint32_t w = __float_as_uint(m);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// ---- KV cache layout ---------------------------------------------------------------------------
// One array per layer: for every (sequence, kv head) capacity/64 blocks of 64 slots; a block holds
// the K rows of its slots, [64][D] bf16, followed by their V in the operand order of the second
// attention MFMA, [2 groups of 32 slots][D/16][64 lanes][8].  A wave that walks a sequence reads
// one contiguous 256*D-byte unit per 64 slots; position p lives in slot p % capacity.
constexpr int KV_BLOCK = 64;
__host__ __device__ __forceinline__ size_t kv_plane_elems(int cap, int D) { return (size_t)cap * D * 2; }
// first element of the block that holds `slot` of (seq, g)
__device__ __forceinline__ size_t kv_block_off(int seq, int g, int n_kv, int cap, int D, int slot) {
  return ((size_t)(seq * n_kv + g) * (cap >> 6) + (slot >> 6)) * (size_t)(2 * KV_BLOCK * D);
}
// element offsets inside a block
__device__ __forceinline__ int kv_k_elem(int slot, int d, int D) { return (slot & 63) * D + d; }
__device__ __forceinline__ int kv_v_elem(int slot, int d, int D) {
  const int tt = slot & 31, within = tt & 15;
  const int lane = (within >> 2) * 16 + (d & 15);
  const int j = (tt >> 4) * 4 + (within & 3);
  return KV_BLOCK * D + (((slot & 63) >> 5) * (D >> 4) + (d >> 4)) * 512 + lane * 8 + j;
}

// Attention: the reference that a row's weights are taken against, from a block's largest score: raised only by more than RAISE_FROM,
// to the next whole number, so that most blocks behind a row's first rescale nothing, and where one does the factor is a power of
// two, without a rounding.
constexpr float RAISE_FROM = 4.f;
__device__ __forceinline__ bool raises_reference(float m, float top) { return top > m + RAISE_FROM; }
__device__ __forceinline__ float raise_reference(float m, float top) { return raises_reference(m, top) ? ceilf(top) : m; }

// K rows of a block in LDS: piece j (16 bytes) of row r is at j ^ kv_swizzle(r).  LDS serves lanes 0-3, 12-15 and 20-27 of a fragment
// read (16 rows, one piece per quarter) together, then 4-11, 16-19 and 28-31, and the upper half alike, and these hit 16
// different 16-byte slots modulo 256 bytes.
template <int D>
__device__ __forceinline__ int kv_swizzle(int r) {
  static_assert(D == 32 || D == 64);
  return D == 64 ? ((r >> 1) & 7) ^ (r & 4) : ((r >> 2) & 3) ^ ((r >> 1) & 2);
}

// K of a block as it lies, load i / KS, i % KS of a wave its i-th KB, into operands: lane (n, c) of [tb][s] has piece c KS + s of
// row 16 tb + n.  own: KV_BLOCK * D * 2 bytes of LDS that the wave has to itself.  (In operand order a load takes 16 bytes of each of 16
// rows, and a CU reads 36 KB a us that way, of whole lines 110.)
template <int D>
__device__ __forceinline__ void keys_to_operands(u32x4 (&k)[4][D / 32], unsigned char *own) {
  constexpr int KS = D / 32, PIECES = D / 8;
  const int lane = lane_id(), n = lane & 15, c = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4 * KS; i++) {
    const int r = i * (64 / PIECES) + lane / PIECES, j = lane % PIECES;
    *reinterpret_cast<u32x4 *>(own + r * (D * 2) + ((j ^ kv_swizzle<D>(r)) << 4)) = k[i / KS][i % KS];
  }
#pragma unroll
  for (int tb = 0; tb < 4; tb++)
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const int r = tb * 16 + n;
      k[tb][s] = *reinterpret_cast<const u32x4 *>(own + r * (D * 2) + (((c * KS + s) ^ kv_swizzle<D>(r)) << 4));
    }
}

}  // namespace gptoss
