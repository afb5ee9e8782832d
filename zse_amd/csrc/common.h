// Shared by every kernel file.  The library is built twice from the same
// sources: with ZSE_ACT_BF16=1 activations, weights and the cache are
// bfloat16; with ZSE_ACT_BF16=0 they are float and nothing is computed below
// 32 bits.  Residual stream, statistics, scores and logits are float in both.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#ifndef ZSE_ACT_BF16
#error "build with -DZSE_ACT_BF16=0 or 1"
#endif

#if ZSE_ACT_BF16
typedef __bf16 act_t;
#else
typedef float act_t;
#endif

#define ZSE_WAVE 64

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(__bf16 x) { return (float)x; }
template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <>
__device__ __forceinline__ __bf16 from_f32<__bf16>(float x) { return (__bf16)x; }

// A load of 8 or 16 bytes that one block reads once in a launch (a weight, a cached value), marked non-temporal: the
// caches do not make room for it.  A streaming read reaches 6.5 to 6.8 TB/s so, 6.0 to 6.1 without (blocks of 4 or 8
// waves, 100 MB to 1.6 GB); a step of 8 decoded tokens of 27B shapes 10,830 -> 9,760 us, of 8 and 1 of 2B shapes 2,228
// -> 2,160 and 1,655 -> 1,595.
// Only for memory that no later launch finds in the memory side's cache of 256 MB anyway (six layers of width 1,024,
// 250 MB in all, one decoded token 200 -> 204 us; 8 requests of 500 keys in the cache 11.2 -> 11.4), which the runner
// says, and for whole 128-byte lines a load, which the launch looks at: where a wave asks for a line's halves one after
// the other (rows of cached keys, values in pages of 64 keys and more), the second half comes from further away again
// (64 requests of 200 to 3,840 keys with the keys so too 4,880 -> 5,010 us; 64 of 4,000 keys in pages of 128 231 -> 279).
template <typename T>
__device__ __forceinline__ T load_once(const T* p) {
  typedef unsigned words __attribute__((ext_vector_type(sizeof(T) / 4)));
  return __builtin_bit_cast(T, __builtin_nontemporal_load((const words*)p));
}

template <bool ONCE, typename T>
__device__ __forceinline__ T load_maybe_once(const T* p) {
  if constexpr (ONCE) return load_once(p);
  else return *p;
}

// One rotation of a pair by an angle, written so that every kernel that rotates rounds alike
// (a token's values must not depend on how many tokens the step holds or on which kernel took
// it): a product rounded, then one fused multiply-add.
__device__ __forceinline__ void rotate_pair(float a, float b, float sn, float cs, float& ra, float& rb) {
  ra = __fmaf_rn(a, cs, -__fmul_rn(b, sn));
  rb = __fmaf_rn(b, cs, __fmul_rn(a, sn));
}

// Reductions over a wave and a block.  A lane's partner is fetched by a lane permutation of the vector unit (a few
// cycles; through the local memory, as __shfl_xor goes, about a hundred), in the order 32, 16, 8, 4, 2, 1: the sum is
// the same bits in every lane.  Kernels of a few rows are a chain of such steps (us, through the local memory and so: a
// step of one decoded token, 2B shapes, 1,786 and 1,722, of eight 2,423 and 2,355; a model of six layers of width 1,024 234 and 222).
//
// The permutations do not fetch from lanes that are not there: everything down to the running sums, but for wave_sum, wave_max
// and block_sum, is for waves whose 64 lanes are all active (blocks of whole waves, outside of conditions on lanes), as this tree's
// kernels call them: the look at the lanes costs a recurrence that adds up twice a token 2 % (six layers of width 1,024 in 32
// bits, 253 tokens, 3,346 and 3,427 us a step).
// Lane l's partner l ^ 32 or l ^ 16: the pair's two values, in some order.
__device__ __forceinline__ void wave_pair32(float v, float& a, float& b) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
#endif
}
__device__ __forceinline__ void wave_pair16(float v, float& a, float& b) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
#endif
}
// The value of a lane of the same 16: rotated by 8 or 4 (the partner l ^ 8, and l ^ 4 where lanes 8 apart agree), or
// permuted inside groups of four.
#define ZSE_DPP_ROR8 0x128
#define ZSE_DPP_ROR4 0x124
#define ZSE_DPP_XOR2 0x4E
#define ZSE_DPP_XOR1 0xB1
template <int CTRL>
__device__ __forceinline__ float wave_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum16(float v) {      // over the 16 lanes of a row
  v += wave_dpp<ZSE_DPP_ROR8>(v);
  v += wave_dpp<ZSE_DPP_ROR4>(v);
  v += wave_dpp<ZSE_DPP_XOR2>(v);
  v += wave_dpp<ZSE_DPP_XOR1>(v);
  return v;
}
__device__ __forceinline__ float wave_sum_whole(float v) {
  float a = 0.f, b = 0.f;
  wave_pair32(v, a, b);
  wave_pair16(a + b, a, b);
  return wave_sum16(a + b);
}
__device__ __forceinline__ float wave_max_whole(float v) {
  float a = 0.f, b = 0.f;
  wave_pair32(v, a, b);
  wave_pair16(fmaxf(a, b), a, b);
  v = fmaxf(a, b);
  v = fmaxf(v, wave_dpp<ZSE_DPP_ROR8>(v));
  v = fmaxf(v, wave_dpp<ZSE_DPP_ROR4>(v));
  v = fmaxf(v, wave_dpp<ZSE_DPP_XOR2>(v));
  return fmaxf(v, wave_dpp<ZSE_DPP_XOR1>(v));
}
// The same over the lanes that are active: in a wave that lacks some, one after the other.
__device__ __forceinline__ bool wave_is_whole() { return __ballot(1) == ~0ull; }
__device__ __forceinline__ float wave_lane(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
__device__ __forceinline__ float wave_sum(float v) {
  if (wave_is_whole()) return wave_sum_whole(v);
  float t = 0.f;
  for (unsigned long long left = __ballot(1); left; left &= left - 1) t += wave_lane(v, __ffsll(left) - 1);
  return t;
}
__device__ __forceinline__ float wave_max(float v) {
  if (wave_is_whole()) return wave_max_whole(v);
  float t = -INFINITY;
  for (unsigned long long left = __ballot(1); left; left &= left - 1) t = fmaxf(t, wave_lane(v, __ffsll(left) - 1));
  return t;
}

// Sums and maxima over a lane and its partners 16, 32 or both away (in that order).
__device__ __forceinline__ float wave_add32(float v) {
  float a = 0.f, b = 0.f;
  wave_pair32(v, a, b);
  return a + b;
}
__device__ __forceinline__ float wave_max32(float v) {
  float a = 0.f, b = 0.f;
  wave_pair32(v, a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float wave_add16_32(float v) {
  float a = 0.f, b = 0.f;
  wave_pair16(v, a, b);
  return wave_add32(a + b);
}
__device__ __forceinline__ float wave_max16_32(float v) {
  float a = 0.f, b = 0.f;
  wave_pair16(v, a, b);
  return wave_max32(fmaxf(a, b));
}

// Running sums and maxima over a wave's lanes (each lane's own value included): rows of 16 lanes by shifts, then a row's
// last lane handed to the next row, then lane 31 to the upper half.  ``none``: what a lane without a neighbour joins.
template <int CTRL, int ROWS>
__device__ __forceinline__ int wave_shifted(int v, int none) {
  return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);
}
#define ZSE_WAVE_SCAN(v, join, cast, back, none)                        \
  v = join(v, cast(wave_shifted<0x111, 0xf>(back(v), back(none))));     \
  v = join(v, cast(wave_shifted<0x112, 0xf>(back(v), back(none))));     \
  v = join(v, cast(wave_shifted<0x114, 0xf>(back(v), back(none))));     \
  v = join(v, cast(wave_shifted<0x118, 0xf>(back(v), back(none))));     \
  v = join(v, cast(wave_shifted<0x142, 0xa>(back(v), back(none))));     \
  v = join(v, cast(wave_shifted<0x143, 0xc>(back(v), back(none))));
__device__ __forceinline__ int wave_add(int a, int b) { return a + b; }
__device__ __forceinline__ float wave_add(float a, float b) { return a + b; }
__device__ __forceinline__ int wave_running_sum(int v) {
  ZSE_WAVE_SCAN(v, wave_add, int, int, 0)
  return v;
}
__device__ __forceinline__ float wave_running_sum(float v) {
  ZSE_WAVE_SCAN(v, wave_add, __int_as_float, __float_as_int, 0.f)
  return v;
}
__device__ __forceinline__ float wave_running_max(float v) {
  ZSE_WAVE_SCAN(v, fmaxf, __int_as_float, __float_as_int, -INFINITY)
  return v;
}

// Sum over a block of up to 1024 threads; every thread gets the result (each wave adds the waves' sums up for
// itself).  ``scratch`` holds at least 16 floats of LDS; block_sum and block_sum_whole may be called again with the same ones,
// block_sum_once with such that nothing else of the block is reading or writing.  The latter two: blocks of whole waves.
__device__ __forceinline__ float block_sum_once(float v, float* scratch) {
  const int lane = threadIdx.x & (ZSE_WAVE - 1), wave = threadIdx.x / ZSE_WAVE, nw = blockDim.x / ZSE_WAVE;
  v = wave_sum_whole(v);
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  return wave_sum16((lane & 15) < nw ? scratch[lane & 15] : 0.f);
}
__device__ __forceinline__ float block_sum_whole(float v, float* scratch) {
  __syncthreads();
  return block_sum_once(v, scratch);
}
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (ZSE_WAVE - 1), wave = threadIdx.x / ZSE_WAVE;
  const int nw = (blockDim.x + ZSE_WAVE - 1) / ZSE_WAVE;
  __syncthreads();
  v = wave_sum(v);
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  if (blockDim.x % ZSE_WAVE == 0) return wave_sum16((lane & 15) < nw ? scratch[lane & 15] : 0.f);
  v = 0.f;                               // a last wave that is not whole: all waves add up alike
  for (int w = 0; w < nw; w++) v += scratch[w];
  return v;
}

// Requests are rows [q_start[r], q_start[r + 1]) of a step, cut into pieces of ``len`` rows that are numbered
// through all requests.  Where piece x lies: its request, that request's rows and the piece's first row among
// them; false behind the last piece.  All lanes of a wave call it and get the same; 64 requests are added
// up at a time (one request after the other costs a wait for memory each).
struct Piece {
  int r, t0, n, first;
};
__device__ __forceinline__ bool find_piece(const int* __restrict__ q_start, int R, int len, int x, Piece& at) {
  const int lane = threadIdx.x & (ZSE_WAVE - 1);
  int acc = 0;
  for (int r0 = 0; r0 < R; r0 += ZSE_WAVE) {
    const int t0 = q_start[min(r0 + lane, R)], n = q_start[min(r0 + lane + 1, R)] - t0;
    const int end = acc + wave_running_sum((n + len - 1) / len);          // pieces up to this request's last
    const unsigned long long later = __ballot(end > x);
    if (later) {
      const int i = __ffsll(later) - 1;
      const int before = i ? __builtin_amdgcn_readlane(end, i - 1) : acc;
      at.r = r0 + i;
      at.t0 = __builtin_amdgcn_readlane(t0, i);
      at.n = __builtin_amdgcn_readlane(n, i);
      at.first = (x - before) * len;
      return true;
    }
    acc = __builtin_amdgcn_readlane(end, ZSE_WAVE - 1);
  }
  return false;
}

// ---- host side ----
extern thread_local std::string zk_error;
int zk_fail(const char* msg);
int zk_launch_status(const char* what);

#define ZK_REQUIRE(cond, msg) \
  do {                        \
    if (!(cond)) return zk_fail(msg); \
  } while (0)

// The definitions behind the three declarations above and the two functions through which a
// caller asks a library for its last message and its storage type.  Each shared library has
// them once: the kernel libraries in elementwise.hip, a library of a part's own kernels in its
// own source file.
#define ZK_DEFINE_HOST_SIDE                                               \
  thread_local std::string zk_error;                                      \
  int zk_fail(const char* msg) {                                          \
    zk_error = msg;                                                       \
    return -1;                                                            \
  }                                                                       \
  int zk_launch_status(const char* what) {                                \
    hipError_t e = hipGetLastError();                                     \
    if (e != hipSuccess) {                                                \
      zk_error = std::string(what) + ": " + hipGetErrorString(e);         \
      return (int)e;                                                      \
    }                                                                     \
    return 0;                                                             \
  }                                                                       \
  extern "C" const char* zk_last_error() { return zk_error.c_str(); }     \
  extern "C" int zk_act_is_bf16() { return ZSE_ACT_BF16; }
