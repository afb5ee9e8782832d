// bfloat16 matrix products on the matrix cores (MFMA), float accumulation:
//   C[M,N] = A[M,K] * W[N,K]^T        (weights [out, in], both operands K-contiguous)
//
// Three kernels, chosen by M:
//  * skinny (M <= 16, or weights not in strip layout up to 64): the weight matrix is streamed
//    once from HBM.  A block owns a strip of 16 weight rows; its waves split K and each feeds
//    16x16x32 MFMAs straight from global memory: a lane's 16-byte load is exactly its MFMA
//    operand (row = lane % 16, eight k values at 8 * (lane / 16)), so no LDS staging is
//    needed.  Partial sums of the waves meet in LDS.
//  * mid (17 <= M <= 64, strip layout, and some shapes of fewer rows): one to eight strips a block, one to eight waves
//    each, the activations of a k chunk shared through LDS, K split over blocks when N alone gives too few of them.
//  * tile (M > 64, prefill): weights in strip layout by the kernel of gemm_bf16_tiles.h, others by
//    128x128x64 to 256x256x64 block tiles staged through registers and LDS.
// Epilogues: plain store (bf16 or float), soft cap on float output (LM head), and
// the gated activation act(gate) * up over a [2I, K] weight whose first I rows are
// the gate (the feed-forward's first product; the [T, 2I] intermediate never
// reaches memory).
//
// The reference's products are scalar-FMA tiles and a one-warp-per-row GEMV
// (orchestrator/kernels.py:1075-1126, 2077-2107), gate and up separate
// (orchestrator/model_runner.py:1270-1275).
#include "common.h"
#include "gemm_bf16_static.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

// Where a product that splits K over blocks leaves its partial sums.  ``strict``: the split is
// chosen as for the standard workspace (so that the bits do not depend on who brought the
// memory) and refused, not narrowed, when ``bytes`` cannot hold it.
#define ZK_GEMM_WORKSPACE_BYTES ((size_t)320 << 20)
struct GemmWorkspace {
  void* ptr;
  size_t bytes;
  bool strict;
  size_t split_bytes() const { return strict ? ZK_GEMM_WORKSPACE_BYTES : bytes; }
  int too_small(size_t need) const {
    static thread_local char msg[200];
    snprintf(msg, sizeof msg, "zk_gemm_bf16_static: this shape's partial sums need %zu bytes, the "
             "static scratch array holds %zu", need, bytes);
    return zk_fail(msg);
  }
};

#if ZSE_ACT_BF16

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// EPI_PICK (the LM head of a step whose next tokens are the largest logits): nothing of C is
// stored; each strip of 16 columns leaves, per row, its largest value after the soft cap (cap
// <= 0: none) and that value's column in ``partials`` [M][strips] as (float, int), larger value
// first, equal values to the lower column, NaN never, which a joining kernel reduces to one
// column a row: the greedy choice without the logits ever reaching memory.
enum { EPI_NONE = 0, EPI_SOFTCAP = 1, EPI_GELU_TANH = 2, EPI_SILU = 3, EPI_PICK = 4, EPI_RELU = 5, EPI_CLAMPED = 6, EPI_RELU2 = 7,
       EPI_GELU = 8 };

struct Pick {
  float value;
  int column;
};

// A lane's four results x[i] at columns n + i of one row, joined with the lanes 16, 32 and 48
// further on (the other columns of the strip); afterwards every one of the four lanes holds
// the strip's pick.
__device__ __forceinline__ Pick pick_of_strip(const float (&x)[4], int n, int N, float cap) {
  Pick p{-INFINITY, 0x7fffffff};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (n + i >= N) continue;
    const float v = cap > 0.f ? cap * tanhf(x[i] / cap) : x[i];
    if (v > p.value || (p.column == 0x7fffffff && v == v)) {
      p.value = v;
      p.column = n + i;
    }
  }
#pragma unroll
  for (int off = 16; off <= 32; off *= 2) {
    const float ov = __shfl_xor(p.value, off);
    const int oc = __shfl_xor(p.column, off);
    const bool other_valid = oc != 0x7fffffff, mine_valid = p.column != 0x7fffffff;
    if (other_valid && (!mine_valid || ov > p.value || (ov == p.value && oc < p.column))) {
      p.value = ov;
      p.column = oc;
    }
  }
  return p;
}

// What a plain (not gated) product does to a sum before it is stored: the soft cap, the square of
// relu, the gelu with the error function, or nothing.
__device__ __forceinline__ float epi_unary(float x, int epi, float cap) {
  if (epi == EPI_SOFTCAP) return cap * tanhf(x / cap);
  if (epi == EPI_RELU2) {
    const float r = fmaxf(x, 0.f);
    return r * r;
  }
  if (epi == EPI_GELU) return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f));
  return x;
}

// 0.5 g (1 + tanh(u)) = g / (1 + exp(-2 u)): one exponential and one reciprocal instead of the
// library's tanh, which cost a tenth of the prompt's gate|up product; the difference (a few
// units in the last place of a float) vanishes when the result is rounded to 16 bits.
__device__ __forceinline__ float epi_gelu_tanh(float g) {
  const float k = 0.7978845608028654f;
  const float u = k * (g + 0.044715f * g * g * g);
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-2.0f * u));
}
// cap: the limit of the clamped gate (g = min(g, cap), u = clamp(u, -cap, cap): g sigmoid(1.702 g) (u + 1))
__device__ __forceinline__ float epi_gate(float g, float u, int epi, float cap) {
  if (epi == EPI_RELU) return fmaxf(g, 0.f) * u;
  if (epi == EPI_CLAMPED) {
    g = fminf(g, cap);
    u = fminf(fmaxf(u, -cap), cap);
    return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
  }
  return (epi == EPI_GELU_TANH ? epi_gelu_tanh(g) : g / (1.0f + expf(-g))) * u;
}

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; i++) z[i] = (__bf16)0.f;
  return z;
}

// Whether the weights are read past the caches: the caller says that no step finds there what the last one read (w_strip 3).
static bool reads_once(int w_strip) { return (w_strip & 2) != 0; }
template <bool ONCE>
__device__ __forceinline__ bf16x8 load_weights(const void* p) {
  return load_maybe_once<ONCE>((const bf16x8*)p);
}

// An argument of those forms of a kernel that read it: what a kernel is launched with is written and fetched whether it looks at it or
// not, and the launch's own numbers, which the compiler reads behind the arguments, move into another line (a norm's 64 bytes on every
// product of up to 16 rows: steps of 2, 8 and 16 decoded tokens, six layers of width 1,024, 207, 231 and 302 us and 212, 238 and 304).
struct Nothing {};
template <bool READ, typename T>
using ArgumentIf = std::conditional_t<READ, T, Nothing>;

// ------------------------------------------------------------------ the norm in front of a product of one row
// h_out = h + post(sub) and the row next(h_out), as zk_norm_add_norm makes them, to the bit: sub as activations or ``parts`` planes of
// float sums.  Every block of the product works the row out for itself, while its first weights are on their way, and the first
// block stores h_out (elsewhere than h, which the others are still reading).
//
// What it saves is a launch that waits for memory twice and that everything behind it waits for; what it costs is the row's planes read
// by every CU from its L2, which is why it is for one row only (5 planes of 2,304 sums are 55 KB a block).  A step of one decoded token,
// us: six layers of width 1,024 204 -> 184, the 2B shapes 1,565 -> 1,514.
struct RowNorm {
  const void* sub;
  const float* w_post;
  const float* h;
  float* h_out;
  const float* w_next;
  float eps_post, eps_next;
  int parts, uo_post, uo_next, H;
};

// h + x g, rounded in between: as the norm's kernels, where the post norm may be missing, round.
__device__ __forceinline__ float row_joined(float h, float x, float g) {
#pragma clang fp contract(off)
  const float y = x * g;
  return h + y;
}

__device__ __forceinline__ f32x4 load4_act(const __bf16* p) {
  const bf16x4 x = *(const bf16x4*)p;
  return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
}

// The sums run as in norm_add_norm_wide_kernel (WIDE, H >= 2,048: 16 waves, a vector of four a thread) or
// norm_add_norm_fast_kernel (4 waves, up to two vectors a thread), whose waves this block's NW waves take in turn,
// SLOTS each.  H a multiple of 256.  PL: 0, or as many planes asked for (parts <= PL).
// Two halves, because loads come back in the order in which they were asked for: what the row is made of first, then
// (by the caller) the first weights, then the sums, which wait for the former alone (weights first: a step of the 2B
// shapes 1,550 us, so 1,514).  All that forks is fixed at compile time: with branches on the planes and the width the
// compiler waits for every load and keeps rows in scratch memory (4,096 columns of K 2,304 8.0 and 9.1 us in a trace
// of a step).
template <int NW, int SLOTS, bool WIDE, int PL>
struct RowInWork {
  static_assert(WIDE ? NW * SLOTS <= 16 || SLOTS <= 2 : NW == 4 && SLOTS <= 2, "every wave of the kernels above has a place");
  f32x4 v[SLOTS], t[SLOTS][PL > 1 ? PL - 1 : 1], hv[SLOTS], gp[SLOTS], gn[SLOTS];

  // Slot s of this wave: place (wave + s NW) of the wide kernel, or vector s of the narrow one's wave.  Below H for whole waves or not at all.
  static __device__ __forceinline__ int at(int s) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return WIDE ? (wave + s * NW) * 256 + lane * 4 : wave * 256 + lane * 4 + s * 1024;
  }
  static __device__ __forceinline__ bool in(const RowNorm& p, int s) { return __builtin_amdgcn_readfirstlane(at(s)) < p.H; }

  __device__ __forceinline__ void ask(const RowNorm& p) {
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
      if (!in(p, s)) continue;
      const int i = at(s);
      if constexpr (PL == 0) {
        v[s] = load4_act((const __bf16*)p.sub + i);
      } else {
        const float* sf = (const float*)p.sub + i;
        v[s] = *(const f32x4*)sf;
#pragma unroll
        for (int q = 1; q < PL; q++) t[s][q - 1] = *(const f32x4*)(sf + (size_t)min(q, p.parts - 1) * p.H);
      }
      hv[s] = *(const f32x4*)(p.h + i);
      gp[s] = *(const f32x4*)(p.w_post + i);
      gn[s] = *(const f32x4*)(p.w_next + i);
    }
  }

  // the sum of squares as the kernels above have it: a thread's own in order, a wave's by permutations, the waves' in LDS
  __device__ __forceinline__ float total(const RowNorm& p, float* scratch) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
      if (WIDE) ss = 0.f;
      if (in(p, s)) {
#pragma unroll
        for (int e = 0; e < 4; e++) ss += v[s][e] * v[s][e];
      }
      if (WIDE) {
        const float w = wave_sum_whole(ss);
        if (lane == 0 && in(p, s)) scratch[wave + s * NW] = w;
      }
    }
    if (!WIDE) {
      const float w = wave_sum_whole(ss);
      if (lane == 0) scratch[wave] = w;
    }
    __syncthreads();
    // (places without values would add nothing)
    return wave_sum16((lane & 15) < (WIDE ? p.H / 256 : 4) ? scratch[lane & 15] : 0.f);
  }

  // ``row``: H values in LDS, red: 32 floats there; every thread of the block, which may read the row afterwards
  __device__ __forceinline__ void make(const RowNorm& p, __bf16* __restrict__ row, float* __restrict__ red, bool store_h) {
    if constexpr (PL > 0) {
#pragma unroll
      for (int s = 0; s < SLOTS; s++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
          for (int q = 1; q < PL; q++) v[s][e] = q < p.parts ? v[s][e] + t[s][q - 1][e] : v[s][e];
          v[s][e] = (float)(__bf16)v[s][e];
        }
    }
    const float rs = rsqrtf(total(p, red) / (float)p.H + p.eps_post);
#pragma unroll
    for (int s = 0; s < SLOTS; s++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[s][e] = row_joined(hv[s][e], v[s][e] * rs, p.uo_post ? 1.f + gp[s][e] : gp[s][e]);
      }
    const float rs2 = rsqrtf(total(p, red + 16) / (float)p.H + p.eps_next);
#pragma unroll
    for (int s = 0; s < SLOTS; s++) {
      if (!in(p, s)) continue;
      bf16x4 y;
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] = (__bf16)(v[s][e] * rs2 * (p.uo_next ? 1.f + gn[s][e] : gn[s][e]));
      *(bf16x4*)(row + at(s)) = y;
      if (store_h) *(f32x4*)(p.h_out + at(s)) = v[s];
    }
    __syncthreads();
  }
};
// The kernels' template argument: none, or slots + 8 WIDE + 16 PL.
constexpr int row_norm_mode(int slots, bool wide, int pl) { return slots + 8 * wide + 16 * pl; }
template <int NW, int MODE>
using RowOf = RowInWork<MODE ? NW : 4, MODE ? MODE % 8 : 1, MODE ? MODE / 8 % 2 != 0 : false, MODE / 16>;

// ------------------------------------------------------------------ skinny
// What the q|k|v product of decoded tokens does with its results instead of storing them all:
// q and k heads are rotated (pairs (i, i + hd/2), angle position * inv_freq[i]), q goes to C,
// k and v to the token's place in the paged cache.
struct RopeStore {
  const int* positions;
  const int* slot_map;  // null: nothing is stored in the cache (nkv = 0)
  const float* inv_freq;
  __bf16* kcache;
  __bf16* vcache;
  int nh, nkv, hd, bs, v_transposed;
};

__device__ __forceinline__ void store4(__bf16* dst, const float (&x)[4]) {
  bf16x4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = (__bf16)x[i];
  *(bf16x4*)dst = o;
}

// A lane's results 4 kq + i of a strip of 16, row m: lanes 0..31 hold places hpos + 4 kq + i of the
// head's first half, lanes 32..63 their partners in the second.  sn, cs: of the lane's four angles.  All 64 lanes call it.
__device__ __forceinline__ void rope_store(const RopeStore& rs, const f32x4& v, int m, int M, int lane, int head, int hpos, int slot,
                                           const float (&sn)[4], const float (&cs)[4], __bf16* __restrict__ C, int ldc) {
  const int kq = lane >> 4;
  const bool first = kq < 2;
  const int half = rs.hd / 2, at = hpos + 4 * (kq & 1) + (first ? 0 : half);
  float x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    x[i] = (float)(__bf16)v[i];
    const float y = __shfl_xor(x[i], 32);
    if (head < rs.nh + rs.nkv) {
      float ra, rb;
      rotate_pair(first ? x[i] : y, first ? y : x[i], sn[i], cs[i], ra, rb);
      x[i] = first ? ra : rb;
    }
  }
  if (m >= M) return;
  if (head < rs.nh) {
    store4(C + (size_t)m * ldc + (size_t)head * rs.hd + at, x);
    return;
  }
  if (slot < 0) return;
  const int kvh = (head - rs.nh) % rs.nkv;
  const size_t page = slot / rs.bs, off = slot % rs.bs;
  if (head < rs.nh + rs.nkv || !rs.v_transposed) {
    store4((head < rs.nh + rs.nkv ? rs.kcache : rs.vcache) + ((page * rs.nkv + kvh) * rs.bs + off) * rs.hd + at, x);
  } else {
    __bf16* vt = rs.vcache + (page * rs.nkv + kvh) * (size_t)rs.hd * rs.bs + off;
#pragma unroll
    for (int i = 0; i < 4; i++) vt[(size_t)(at + i) * rs.bs] = (__bf16)x[i];
  }
}

// GATED: the block also streams the strip of "up" rows I + n and stores act(g)*u.
// ROPE (M <= 16): W is [(nh + 2 nkv) hd, K]; the block's 16 weight rows are eight places of a
// head's first half and their partners in the rotation, hd/2 rows further on, so that partners
// meet in lanes 32 apart; the results are finished as RopeStore says.  Every result is rounded
// to 16 bits before it is rotated, as the separate product and rotation kernels do, so a
// token's keys are the same bits whichever way it came.
// NORM (one row): the kernel makes the row it multiplies itself (RowInWork), so that a step of one token has no launch between two products.
// EXACT (weights in strip layout, so K is a whole number of 32-wide steps): no load is under a
// condition.  A step past the wave's run reads the run's last step again and its weights are
// set to zero afterwards; a row past M reads row M - 1 (its results are never stored).  Only so
// can the compiler count the loads in flight and let a group's products wait for that group
// alone: with loads under per-lane conditions it waits for every load before each group, and
// the next group's loads, just issued, no longer overlap anything (down projection of 2304 x
// 9216 at 8 rows: 14 us against 9).
// WHOLE (EXACT, up to 16 rows, K in whole groups of 8 steps, every launch of a real model's sizes): a load's address is a scalar that
// moves on from group to group, a lane's own offset that does not, and a constant.  Worked out for each load from its step (clamped, in 64
// bits), the addresses of a group are a hundred instructions that a wave issues one every fourth cycle in
// front of its loads (us, 8 rows: 4,096 columns of K 2,304 6.3 -> 5.5, 2,304 of 2,048
// 5.0 -> 4.4, 2,304 of 9,216 13.3 -> 12.4; a step of 8 decoded tokens of the 2B shapes 2,319 -> 2,278).  The same sums.
// ONCE (WHOLE): weights by loads that leave no trace in the caches (reads_once).
template <int MT, bool GATED, int NW, bool ROPE = false, bool EXACT = false, bool SPLIT = false, bool WHOLE = false, bool ONCE = false, int NORM = 0>
__global__ __launch_bounds__(NW * 64) void gemm_skinny_kernel(const __bf16* __restrict__ A, int lda,
                                                          const __bf16* __restrict__ W,
                                                          void* __restrict__ C, int ldc, int c_is_f32,
                                                          int M, int N, int K, int epi, float cap,
                                                          int w_strip, RopeStore rs,
                                                          float* __restrict__ partials = nullptr, int ksplit = 1,
                                                          ArgumentIf<NORM != 0, RowNorm> norm = {}) {
  static_assert(!NORM || (WHOLE && !SPLIT), "a row made here is multiplied whole");
  __shared__ __align__(16) __bf16 own_row[NORM ? 4096 : 8];
  __shared__ float own_sums[NORM ? 32 : 1];
  static_assert(!ROPE || (MT == 1 && !GATED), "the rotating epilogue takes up to 16 rows");
  static_assert(!WHOLE || (EXACT && MT == 1), "whole groups: strips, up to 16 rows");
  constexpr int NS = GATED ? 2 : 1;
  __shared__ f32x4 red[NW - 1][NS][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kq = lane >> 4;
  // the block's strips of 16 weight rows
  const int strip0 = blockIdx.x, strip1 = N / 16 + blockIdx.x;
  const int n0 = strip0 * 16;
  // Row-major weights: a lane reads row n0 + r at 8 * kq, a 32-wide step further on is 32
  // elements away.  Strip layout: the 64 lanes' pieces of one (strip, step) are one
  // contiguous KB, a step further on is 512 elements away, strips follow each other.
  const int wrow = min(n0 + r, N - 1);
  const int ksteps = (K + 31) / 32;
  const size_t wstep = w_strip ? 512 : 32;
  const __bf16* wp[NS];
  wp[0] = w_strip ? W + (size_t)strip0 * ksteps * 512 + lane * 8 : W + (size_t)wrow * K + kq * 8;
  if (GATED)
    wp[NS - 1] = w_strip ? W + (size_t)strip1 * ksteps * 512 + lane * 8
                         : W + (size_t)(N + wrow) * K + kq * 8;
  int head = 0, hpos = 0;  // ROPE: the head and the first of the block's eight places in its first half
  if (ROPE) {
    const int per_head = rs.hd / 16;
    head = blockIdx.x / per_head;
    hpos = (blockIdx.x % per_head) * 8;
    const int row = head * rs.hd + hpos + (r < 8 ? r : rs.hd / 2 + r - 8);
    wp[0] = w_strip ? W + (size_t)(row / 16) * ksteps * 512 + (16 * kq + row % 16) * 8
                    : W + (size_t)row * K + kq * 8;
  }
  const __bf16* ap[MT];
  bool av[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int m = mt * 16 + r;
    av[mt] = m < M;
    ap[mt] = A + (size_t)min(m, M - 1) * lda + kq * 8;
  }
  f32x4 acc[NS][MT];
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[s][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // the K range is cut into NW equal runs of 32-wide steps, one run a wave.  A wave works in
  // groups of STEPS steps and keeps the next group's loads in flight while it multiplies the
  // current one (two register sets, the loop is unrolled by two to name them).
  constexpr int STEPS = (MT * NS >= 4) ? 4 : 8;
  const int total_steps = (K + 31) / 32;
  const int per_wave = (total_steps + NW - 1) / NW;
  const int s_begin = wave * per_wave, s_end = min(total_steps, s_begin + per_wave);
  // EXACT: whole groups of STEPS steps are shared out among the waves as evenly as they go
  const int total_groups = (total_steps + STEPS - 1) / STEPS;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);      // the same in every lane: loop bounds stay scalar
  // (SPLIT) blockIdx.y takes one of ksplit ranges of the groups, its waves share the range out
  static_assert(!SPLIT || (EXACT && MT == 1 && !GATED && !ROPE), "K is split for plain products of up to 16 rows");
  const int gy0 = SPLIT ? (int)blockIdx.y * total_groups / ksplit : 0;
  const int gy1 = SPLIT ? ((int)blockIdx.y + 1) * total_groups / ksplit : total_groups;
  const int gw0 = gy0 + uwave * (gy1 - gy0) / NW, gw1 = gy0 + (uwave + 1) * (gy1 - gy0) / NW;
  const int run_lo = gw0 * STEPS, run_n = (gw1 - gw0) * STEPS;      // the wave's run of steps
  // WHOLE: the wave's run in each strip and in A (scalars), and where the lane reads in a step of them
  const char* wrun[NS];
  const char* arun = (const char*)A + (size_t)run_lo * 64;
  unsigned wlane = lane * 16;
  const unsigned alane = (unsigned)min(r, M - 1) * (unsigned)lda * 2 + kq * 16;
  if (WHOLE) {
    int first = strip0;
    if (ROPE) {
      first = (head * rs.hd + hpos) / 16;
      const int row = head * rs.hd + hpos + (r < 8 ? r : rs.hd / 2 + r - 8);
      wlane = (unsigned)(row / 16 - first) * (unsigned)ksteps * 1024 + (16 * kq + row % 16) * 16;
    }
    wrun[0] = (const char*)W + ((size_t)first * ksteps + run_lo) * 1024;
    if (GATED) wrun[NS - 1] = (const char*)W + ((size_t)strip1 * ksteps + run_lo) * 1024;
  }
  auto fetch = [&](int s0, bf16x8 (&wf)[NS][STEPS], bf16x8 (&af)[MT][STEPS]) {
    if constexpr (WHOLE) {
      const char* a = arun + (size_t)s0 * 64;
#pragma unroll
      for (int g = 0; g < NS; g++) {
        // (a constant in an address reaches 4 KB)
        const char *lo = wrun[g] + (size_t)s0 * 1024, *hi = lo + 4096;
#pragma unroll
        for (int s = 0; s < STEPS; s++) wf[g][s] = load_weights<ONCE>((s < 4 ? lo + s * 1024 : hi + (s - 4) * 1024) + wlane);
      }
      if (!NORM) {
#pragma unroll
        for (int s = 0; s < STEPS; s++) af[0][s] = *(const bf16x8*)(a + s * 64 + alane);
      }
      return;
    }
    if (EXACT) {
      // A whole group of steps, counted from the start of the wave's run; only the last group
      // of K may hold fewer steps, and then the steps past K read K's last step again and count
      // as zero.
#pragma unroll
      for (int s = 0; s < STEPS; s++) {
        const int step = min(run_lo + s0 + s, total_steps - 1);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) af[mt][s] = *(const bf16x8*)(ap[mt] + step * 32);
#pragma unroll
        for (int g = 0; g < NS; g++) wf[g][s] = *(const bf16x8*)(wp[g] + (size_t)step * wstep);
      }
      if (run_lo + run_n > total_steps) {
#pragma unroll
        for (int s = 0; s < STEPS; s++)
          if (run_lo + s0 + s >= total_steps) {
#pragma unroll
            for (int g = 0; g < NS; g++) wf[g][s] = zero8();
          }
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      const int k = (s0 + s) * 32;
      const bool in = (s0 + s < s_end) && (k + kq * 8 < K);
#pragma unroll
      for (int mt = 0; mt < MT; mt++) af[mt][s] = (in && av[mt]) ? *(const bf16x8*)(ap[mt] + k) : zero8();
#pragma unroll
      for (int g = 0; g < NS; g++) wf[g][s] = in ? *(const bf16x8*)(wp[g] + (size_t)(s0 + s) * wstep) : zero8();
    }
  };
  int at_step = run_lo;        // (NORM) the step of A that the next product takes
  auto multiply = [&](const bf16x8 (&wf)[NS][STEPS], const bf16x8 (&af)[MT][STEPS]) {
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
      for (int g = 0; g < NS; g++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          acc[g][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[g][s], NORM ? *(const bf16x8*)(own_row + (at_step + s) * 32 + kq * 8) : af[mt][s], acc[g][mt], 0, 0, 0);
    if (NORM != 0) at_step += STEPS;
  };
  bf16x8 wf0[NS][STEPS], af0[MT][STEPS], wf1[NS][STEPS], af1[MT][STEPS];
  RowOf<NW, NORM> own;
  if constexpr (NORM != 0) {
    own.ask(norm);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (EXACT) {
    if (gw0 < gw1) fetch(0, wf0, af0);
  } else if (s_begin < s_end) {
    fetch(s_begin, wf0, af0);
  }
  // the angles of the lane's four pairs, worked out by four waves while the first loads are on their way (all by
  // the one that stores, they are 0.7 us that the others wait for)
  __shared__ float2 turn[ROPE ? 4 : 1][64];
  int slot = -1;
  if (ROPE) {
    if (wave == 0 && head >= rs.nh && rs.slot_map) slot = rs.slot_map[min(r, M - 1)];
    if (wave < 4 && head < rs.nh + rs.nkv) {
      float sn, cs;
      sincosf((float)rs.positions[min(r, M - 1)] * rs.inv_freq[hpos + 4 * (kq & 1) + wave], &sn, &cs);
      turn[wave][lane] = make_float2(sn, cs);
    }
  }
  if constexpr (NORM != 0) {
    __builtin_amdgcn_sched_barrier(0);
    own.make(norm, own_row, own_sums, blockIdx.x == 0);
  }
  if (EXACT) {
    // The wave's run is a whole number of groups [gw0, gw1).  In the loop every product follows
    // a fetch, so the number of loads in flight at each wait is known; the last one or two
    // groups have code of their own.  Nothing is loaded twice.  (The scheduling barriers keep
    // the compiler from moving a group's loads down to their first use, which would put each
    // load right in front of the product that waits for it.)
    if (gw0 < gw1) {
      int g = 0;
      const int gw1 = run_n / STEPS;         // groups of the run, counted from its start
      for (; g + 2 < gw1; g += 2) {
        fetch((g + 1) * STEPS, wf1, af1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(wf0, af0);
        __builtin_amdgcn_sched_barrier(0);
        fetch((g + 2) * STEPS, wf0, af0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(wf1, af1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (g + 2 == gw1) {
        fetch((g + 1) * STEPS, wf1, af1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(wf0, af0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(wf1, af1);
      } else {
        multiply(wf0, af0);
      }
    }
  } else {
    for (int s0 = s_begin; s0 < s_end; s0 += 2 * STEPS) {
      if (s0 + STEPS < s_end) fetch(s0 + STEPS, wf1, af1);
      multiply(wf0, af0);
      if (s0 + STEPS >= s_end) break;
      if (s0 + 2 * STEPS < s_end) fetch(s0 + 2 * STEPS, wf0, af0);
      multiply(wf1, af1);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int g = 0; g < NS; g++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) red[wave - 1][g][mt][lane] = acc[g][mt];
  }
  __syncthreads();
  if (wave > 0) return;
  // lane holds rows n = n0 + 4*kq + i (i = 0..3) of column m = mt*16 + r
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int m = mt * 16 + r;
    f32x4 v[NS];
#pragma unroll
    for (int g = 0; g < NS; g++) {
      v[g] = acc[g][mt];
#pragma unroll
      for (int w = 0; w < NW - 1; w++) v[g] += red[w][g][mt][lane];
    }
    if (SPLIT) {
      // the range's partial sums: plane blockIdx.y of [M, npad] floats, to be added up in the
      // order of the ranges by whoever reads them (zk_norm_add_norm, or the joining kernel)
      if (m < M) {
        const size_t npad = (size_t)gridDim.x * 16;
        *(f32x4*)(partials + ((size_t)blockIdx.y * M + m) * npad + n0 + 4 * kq) = v[0];
      }
      continue;
    }
    if (ROPE) {
      float sn[4], cs[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float2 t = turn[ROPE ? i : 0][lane];
        sn[i] = t.x;
        cs[i] = t.y;
      }
      rope_store(rs, v[0], m, M, lane, head, hpos, slot, sn, cs, (__bf16*)C, ldc);
      continue;
    }
    if (!GATED && epi == EPI_PICK) {
      const float x[4] = {v[0][0], v[0][1], v[0][2], v[0][3]};
      const Pick p = pick_of_strip(x, n0 + 4 * kq, N, cap);
      if (kq == 0 && m < M) ((Pick*)partials)[(size_t)m * gridDim.x + blockIdx.x] = p;
      continue;
    }
    if (m >= M) continue;
    if (WHOLE && !c_is_f32 && n0 + 16 <= N && (((uintptr_t)C | (unsigned)ldc * 2) & 7) == 0) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = GATED ? epi_gate(v[0][i], v[NS - 1][i], epi, cap) : epi_unary(v[0][i], epi, cap);
      store4((__bf16*)C + (size_t)m * ldc + n0 + 4 * kq, x);
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int n = n0 + 4 * kq + i;
      if (n >= N) continue;
      float x = v[0][i];
      if (GATED) x = epi_gate(x, v[NS - 1][i], epi, cap);
      else x = epi_unary(x, epi, cap);
      if (c_is_f32) ((float*)C)[(size_t)m * ldc + n] = x;
      else ((__bf16*)C)[(size_t)m * ldc + n] = (__bf16)x;
    }
  }
}

// ------------------------------------------------------------------ tile
// Block tile (32 WMT NWM) x (64 NWN) x 64 with NWM x NWN waves; a wave owns WMT x 2 MFMA tiles
// of 32 x 32.  The k tiles alternate between two LDS buffers: the loads of the next tile are
// issued before the products of the current one and stored after them, one barrier a tile.
#define GT_BK 64
#define GT_LD (GT_BK + 8)

// Blocks that share a weight tile run on one XCD (ids go round-robin over 8 XCDs).
__device__ __forceinline__ void tile_of_block(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
  tn = id / tiles_m;
  tm = id % tiles_m;
}

// The products are taken as W tile x A tile^T, so that a lane holds neighbouring columns of one
// row of C.  Four results of a lane: row lr of the wave's 32 x 32 tiles (i, 0) and (i, 1),
// columns 8 b + 4 lk + e (e = 0..3); x0 belongs to tile (i, 0), x1 to tile (i, 1) (gate and up
// when GATED).
template <int WMT, int NWN, bool GATED>
__device__ __forceinline__ void tile_store_quad(const f32x4& x0, const f32x4& x1, int i, int b,
                                                void* __restrict__ C, int ldc, int c_is_f32, int M, int N,
                                                int m0, int n0, int wm, int wn, int lane, int epi, float cap) {
  const int lr = lane & 31, lk = lane >> 5;
  const int m = m0 + wm * (32 * WMT) + i * 32 + lr;
  if (m >= M) return;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int c = 8 * b + 4 * lk + e;
    if (GATED) {
      const int n = n0 + wn * 32 + c;
      if (n < N) {
        const float x = epi_gate(x0[e], x1[e], epi, cap);
        if (c_is_f32) ((float*)C)[(size_t)m * ldc + n] = x;
        else ((__bf16*)C)[(size_t)m * ldc + n] = (__bf16)x;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int n = n0 + wn * 64 + j * 32 + c;
        if (n >= N) continue;
        float x = j ? x1[e] : x0[e];
        x = epi_unary(x, epi, cap);
        if (c_is_f32) ((float*)C)[(size_t)m * ldc + n] = x;
        else ((__bf16*)C)[(size_t)m * ldc + n] = (__bf16)x;
      }
    }
  }
}

template <int WMT, int NWN, bool GATED>
__device__ __forceinline__ void tile_store(const f32x16 (&acc)[WMT][2], void* __restrict__ C, int ldc,
                                           int c_is_f32, int M, int N, int m0, int n0, int wm, int wn,
                                           int lane, int epi, float cap) {
#pragma unroll
  for (int i = 0; i < WMT; i++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const f32x4 x0 = {acc[i][0][4 * b], acc[i][0][4 * b + 1], acc[i][0][4 * b + 2], acc[i][0][4 * b + 3]};
      const f32x4 x1 = {acc[i][1][4 * b], acc[i][1][4 * b + 1], acc[i][1][4 * b + 2], acc[i][1][4 * b + 3]};
      tile_store_quad<WMT, NWN, GATED>(x0, x1, i, b, C, ldc, c_is_f32, M, N, m0, n0, wm, wn, lane, epi, cap);
    }
}

// The same for a wave whose columns lie inside a 16-bit C with rows that are whole 16-byte pieces:
// the wave's results go through its own piece of LDS (rows of SLD values) and leave as 16 bytes
// a lane, whole 128- or 64-byte runs of a row, instead of two bytes a lane.  Rows from M on are
// left out here.  (A last row of tiles that took the way above instead set the time of a launch
// of one round: 708 x 3072 x 2048 36.7 -> 25.9 us, 535 x 4096 x 2304 33.4 -> 28.4.)
template <int WMT, bool GATED>
__device__ __forceinline__ void tile_store_staged(const f32x16 (&acc)[WMT][2], __bf16* __restrict__ C, int ldc,
                                                  int M, int row0, int col0, int lane, int epi, float cap,
                                                  __bf16* __restrict__ stage) {
  constexpr int COLS = GATED ? 32 : 64, SLD = COLS + 8;
  const int lr = lane & 31, lk = lane >> 5;
#pragma unroll
  for (int i = 0; i < WMT; i++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      float x[4], y[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        x[e] = acc[i][0][4 * b + e];
        y[e] = acc[i][1][4 * b + e];
        if (GATED) x[e] = epi_gate(x[e], y[e], epi, cap);
        else {
          x[e] = epi_unary(x[e], epi, cap);
          y[e] = epi_unary(y[e], epi, cap);
        }
      }
      __bf16* dst = stage + (i * 32 + lr) * SLD + 8 * b + 4 * lk;
      store4(dst, x);
      if (!GATED) store4(dst + 32, y);
    }
  // the wave reads what its other lanes wrote: LDS takes a wave's accesses in order
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int PPR = COLS / 8, RPI = 64 / PPR;      // pieces a row, rows an instruction
  const int prow = lane / PPR, pcol = (lane % PPR) * 8;
#pragma unroll
  for (int r = 0; r < 32 * WMT; r += RPI)
    if (row0 + r + prow < M)
      *(bf16x8*)(C + (size_t)(row0 + r + prow) * ldc + col0 + pcol) = *(const bf16x8*)(stage + (r + prow) * SLD + pcol);
}

template <int WMT, int NWM, int NWN, bool GATED, bool EXACT>
__global__ __launch_bounds__(64 * NWM * NWN, NWM * NWN <= 4 ? 2 : 1) void gemm_tile_kernel(
    const __bf16* __restrict__ A, int lda, const __bf16* __restrict__ W, void* __restrict__ C, int ldc,
    int c_is_f32, int M, int N, int K_all, int epi, float cap, int tiles_m, int tiles_n, int w_strip,
    f32x16* __restrict__ partials, int ksplit, int tile_base) {
  constexpr int T = 64 * NWM * NWN;
  constexpr int BM = 32 * WMT * NWM, BN = 64 * NWN;
  constexpr int RPP = T / 8;                   // rows one pass of the block's threads covers
  constexpr int APT = BM / RPP, BPT = BN / RPP;   // 16-byte pieces a thread moves per k tile
  static_assert(BM % RPP == 0 && BN % RPP == 0 && (T / 64) % 2 == 0, "tile and thread counts do not fit");
  extern __shared__ __align__(16) unsigned char gt_lds[];
  typedef __bf16 (*tile_t)[GT_LD];
  const tile_t tiles = (tile_t)gt_lds;          // buffer b: A rows, then W rows, from row b (BM + BN)
  int tm, tn;
  tile_of_block(blockIdx.x + tile_base, tiles_m, tiles_n, tm, tn);     // a launch takes tiles [tile_base, tile_base + gridDim.x)
  const int m0 = tm * BM;
  constexpr int NCOLS = GATED ? BN / 2 : BN;         // output columns of the block
  const int n0 = tn * NCOLS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / NWN, wn = wave % NWN;
  const int lr = lane & 31, lk = lane >> 5;
  // blockIdx.y takes a range of k tiles (the whole of K unless the launch splits it); the
  // operand pointers start at the range, so below K counts from there
  const int ktiles = (K_all + GT_BK - 1) / GT_BK;
  const int kt0 = (int)((long)blockIdx.y * ktiles / ksplit), kt1 = (int)((long)(blockIdx.y + 1) * ktiles / ksplit);
  const int kbase = kt0 * GT_BK;
  const int K = min(K_all, kt1 * GT_BK) - kbase;

  // piece c = tid + T i of a tile: row c / 8, eight k values at (c % 8) * 8
  const int prow = tid >> 3, pcol = (tid & 7) * 8;
  const __bf16* ga[APT];
  const __bf16* gb[BPT];
#pragma unroll
  for (int i = 0; i < APT; i++) ga[i] = A + (size_t)min(m0 + prow + RPP * i, M - 1) * lda + kbase;
  int brow[BPT], bcol;      // where a thread's pieces of the weight tile land in LDS
  if (w_strip) {
    // a wave copies whole KB blocks: block wave + (T / 64) i of the tile's BN / 16 strips x 2
    // steps, lane l its 16 bytes; the k tile advances by two steps = 1024 elements
    const int tstep = wave & 1;
    const int ksteps = (K_all + 31) / 32;
    const int strips = GATED ? 2 * N / 16 : (N + 15) / 16;
    bcol = tstep * 32 + (lane >> 4) * 8;
#pragma unroll
    for (int i = 0; i < BPT; i++) {
      const int sit = (wave + (T / 64) * i) >> 1;            // strip within the tile
      brow[i] = sit * 16 + (lane & 15);
      int gs;
      if (GATED) gs = sit < BN / 32 ? n0 / 16 + sit : N / 16 + n0 / 16 + (sit - BN / 32);
      else gs = n0 / 16 + sit;
      gs = min(gs, strips - 1);
      gb[i] = W + ((size_t)gs * ksteps + 2 * kt0) * 512 + lane * 8;
    }
  } else {
    bcol = pcol;
#pragma unroll
    for (int i = 0; i < BPT; i++) {
      const int row = prow + RPP * i;
      brow[i] = row;
      int bn;
      if (GATED) bn = row < BN / 2 ? min(n0 + row, N - 1) : N + min(n0 + row - BN / 2, N - 1);
      else bn = min(n0 + row, N - 1);
      gb[i] = W + (size_t)bn * K_all + kbase;
    }
  }
  // a piece's offset from its row's (strip's) first element: tile t, then the place in the tile
  const int boff = w_strip ? (wave & 1) * 512 : pcol, bstep = w_strip ? 1024 : GT_BK;
  f32x16 acc[WMT][2];
#pragma unroll
  for (int i = 0; i < WMT; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

  // Two register sets: the loads of tile t + 2 are issued while tile t is multiplied and tile
  // t + 1 waits in the other set, so a load has a whole tile's products to arrive in.
  bf16x8 ra0[APT], rb0[BPT], ra1[APT], rb1[BPT];
  // EXACT (K a multiple of the k tile): no load is under a condition, so that the compiler
  // can count the loads in flight and wait for the older set alone; a tile beyond K is read
  // from the last tile instead and never multiplied.  Otherwise pieces beyond K are zeros.
  auto fetch = [&](int k0, bf16x8 (&ra)[APT], bf16x8 (&rb)[BPT]) {
    if (EXACT) {
      const int kc = min(k0, K - GT_BK);
      const int aoff = kc + pcol, woff = (kc / GT_BK) * bstep + boff;
#pragma unroll
      for (int i = 0; i < APT; i++) ra[i] = *(const bf16x8*)(ga[i] + aoff);
#pragma unroll
      for (int i = 0; i < BPT; i++) rb[i] = *(const bf16x8*)(gb[i] + woff);
    } else {
      const bool in = k0 + pcol < K, inb = k0 + bcol < K;
#pragma unroll
      for (int i = 0; i < APT; i++) ra[i] = in ? *(const bf16x8*)(ga[i] + k0 + pcol) : zero8();
#pragma unroll
      for (int i = 0; i < BPT; i++) rb[i] = inb ? *(const bf16x8*)(gb[i] + (k0 / GT_BK) * bstep + boff) : zero8();
    }
  };
  auto stash = [&](int buf, const bf16x8 (&ra)[APT], const bf16x8 (&rb)[BPT]) {
#pragma unroll
    for (int i = 0; i < APT; i++) *(bf16x8*)(&tiles[buf * (BM + BN) + prow + RPP * i][pcol]) = ra[i];
#pragma unroll
    for (int i = 0; i < BPT; i++) *(bf16x8*)(&tiles[buf * (BM + BN) + BM + brow[i]][bcol]) = rb[i];
  };
  auto multiply = [&](int buf) {
    if constexpr (NWM * NWN > 8) {
      // sixteen waves: 128 registers a wave, no room for a second set of operands
#pragma unroll
      for (int ks = 0; ks < GT_BK / 16; ks++) {
        bf16x8 fa[WMT], fb[2];
#pragma unroll
        for (int i = 0; i < WMT; i++) fa[i] = *(const bf16x8*)(&tiles[buf * (BM + BN) + wm * (32 * WMT) + i * 32 + lr][ks * 16 + lk * 8]);
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int row = GATED ? j * (BN / 2) + wn * 32 : wn * 64 + j * 32;
          fb[j] = *(const bf16x8*)(&tiles[buf * (BM + BN) + BM + row + lr][ks * 16 + lk * 8]);
        }
#pragma unroll
        for (int i = 0; i < WMT; i++)
#pragma unroll
          for (int j = 0; j < 2; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
      return;
    }
    // the operands of k step ks + 1 are read from LDS while the products of step ks run: two
    // sets of fragments, and a fence that keeps the reads before the products they follow in
    // the source (the compiler would put every read right before its use and wait for it)
    bf16x8 fa[2][WMT], fb[2][2];
    auto read = [&](int ks, bf16x8 (&a)[WMT], bf16x8 (&b)[2]) {
#pragma unroll
      for (int i = 0; i < WMT; i++) a[i] = *(const bf16x8*)(&tiles[buf * (BM + BN) + wm * (32 * WMT) + i * 32 + lr][ks * 16 + lk * 8]);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int row = GATED ? j * (BN / 2) + wn * 32 : wn * 64 + j * 32;
        b[j] = *(const bf16x8*)(&tiles[buf * (BM + BN) + BM + row + lr][ks * 16 + lk * 8]);
      }
    };
    read(0, fa[0], fb[0]);
#pragma unroll
    for (int ks = 0; ks < GT_BK / 16; ks++) {
      if (ks + 1 < GT_BK / 16) read(ks + 1, fa[(ks + 1) & 1], fb[(ks + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0x616);
#pragma unroll
      for (int i = 0; i < WMT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0x616);
    }
  };
  // The loop takes two tiles a turn.  An odd number of tiles: when EXACT the first tile is
  // taken alone before the loop, otherwise the last one is all zeros.
  int kfirst = 0;
  if (EXACT && (K / GT_BK) % 2 == 1) {
    fetch(0, ra0, rb0);
    stash(0, ra0, rb0);
    __syncthreads();
    multiply(0);
    __syncthreads();
    kfirst = GT_BK;
  }
  if (kfirst < K) {
    fetch(kfirst, ra0, rb0);
    stash(0, ra0, rb0);
    fetch(kfirst + GT_BK, ra0, rb0);
    __syncthreads();
  }
  for (int k0 = kfirst; k0 < K; k0 += 2 * GT_BK) {
    // tile k0 is in buffer 0, tile k0 + BK in set 0
    fetch(k0 + 2 * GT_BK, ra1, rb1);
    multiply(0);
    stash(1, ra0, rb0);
    __syncthreads();
    // tile k0 + BK is in buffer 1, tile k0 + 2 BK in set 1
    fetch(k0 + 3 * GT_BK, ra0, rb0);
    multiply(1);
    stash(0, ra1, rb1);
    __syncthreads();
  }
  if (ksplit > 1) {
    // partial sums of this k range, in lane order; the join kernel adds the ranges up
    f32x16* mine = partials + (((size_t)blockIdx.x * ksplit + blockIdx.y) * (NWM * NWN) + wave) * (WMT * 2 * 64) + lane;
#pragma unroll
    for (int i = 0; i < WMT; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) mine[(i * 2 + j) * 64] = acc[i][j];
    return;
  }
  // every wave has passed the loop's last barrier: the tile buffers are free
  if (!c_is_f32 && n0 + NCOLS <= N && ldc % 8 == 0 && (uintptr_t)C % 16 == 0) {
    constexpr int WCOLS = GATED ? 32 : 64;
    tile_store_staged<WMT, GATED>(acc, (__bf16*)C, ldc, M, m0 + wm * (32 * WMT), n0 + wn * WCOLS, lane, epi, cap,
                                  (__bf16*)gt_lds + (size_t)wave * (32 * WMT) * (WCOLS + 8));
    return;
  }
  tile_store<WMT, NWN, GATED>(acc, C, ldc, c_is_f32, M, N, m0, n0, wm, wn, lane, epi, cap);
}

// Second half of a tile product whose K was split over blocks: the ranges are added in order.
// A thread takes four consecutive floats of a lane's accumulator pair (i, 0), (i, 1), so the
// partial sums are read in 16-byte pieces, neighbours by neighbouring threads.
template <int WMT, int NWM, int NWN, bool GATED>
__global__ __launch_bounds__(256) void gemm_tile_join_kernel(
    const f32x4* __restrict__ partials, int ksplit, void* __restrict__ C, int ldc, int c_is_f32, int M,
    int N, int epi, float cap, int tiles_m, int tiles_n, int tile_base, int tile_count) {
  constexpr int BM = 32 * WMT * NWM, BN = 64 * NWN, NW = NWM * NWN;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int b = (int)(idx & 3), lane = (int)((idx >> 2) & 63);
  const int i = (int)((idx >> 8) % WMT), wave = (int)((idx >> 8) / WMT % NW);
  const int tile = (int)((idx >> 8) / (WMT * NW));      // counted from the launch's first tile, as the partial sums are
  if (tile >= tile_count) return;
  int tm, tn;
  tile_of_block(tile + tile_base, tiles_m, tiles_n, tm, tn);
  // float4 index of (tile, range p, wave, pair member j, lane, b): an accumulator is 4 float4
  const size_t per_wave = (size_t)WMT * 2 * 64 * 4;
  if constexpr (!GATED) {
    // Whole columns of a 16-bit C with rows of whole 16-byte pieces: a thread takes the two
    // halves (lanes lr and lr + 32) of eight neighbouring columns of a row, so its store is 16
    // bytes and four threads fill a 64-byte line (the general way below stores two bytes at a
    // time, half a line's bytes from one wave and the other half from another).  The block's
    // 256 threads are (b, lr, j) here; the sums are the same, in the same order.
    const int m0 = tm * BM + (wave / NWN) * (32 * WMT) + i * 32, n0 = tn * BN + (wave % NWN) * 64;
    if (!c_is_f32 && (epi == EPI_NONE || epi == EPI_RELU2 || epi == EPI_GELU) && ldc % 8 == 0 && (uintptr_t)C % 16 == 0 && n0 + 64 <= N) {
      const int lr = lane & 31, j = lane >> 5;
      if (m0 + lr >= M) return;
      const f32x4* at = partials + ((size_t)tile * ksplit * NW + wave) * per_wave + ((size_t)(i * 2 + j) * 64 + lr) * 4 + b;
      f32x4 lo = at[0], hi = at[32 * 4];
      for (int p = 1; p < ksplit; p++) {
        lo += at[(size_t)p * NW * per_wave];
        hi += at[(size_t)p * NW * per_wave + 32 * 4];
      }
      bf16x8 out;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        out[e] = (__bf16)epi_unary(lo[e], epi, cap);
        out[4 + e] = (__bf16)epi_unary(hi[e], epi, cap);
      }
      *(bf16x8*)((__bf16*)C + (size_t)(m0 + lr) * ldc + n0 + j * 32 + 8 * b) = out;
      return;
    }
  }
  const f32x4* src = partials + ((size_t)tile * ksplit * NW + wave) * per_wave + ((size_t)(i * 2) * 64 + lane) * 4 + b;
  f32x4 x0 = src[0], x1 = src[64 * 4];
  for (int p = 1; p < ksplit; p++) {
    x0 += src[(size_t)p * NW * per_wave];
    x1 += src[(size_t)p * NW * per_wave + 64 * 4];
  }
  tile_store_quad<WMT, NWN, GATED>(x0, x1, i, b, C, ldc, c_is_f32, M, N, tm * BM, tn * (GATED ? BN / 2 : BN),
                                   wave / NWN, wave % NWN, lane, epi, cap);
}

template <int WMT, int NWM, int NWN, bool GATED, bool EXACT>
static int launch_tile(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32, int M, int N,
                       int K, int epi, float cap, int w_strip, const GemmWorkspace& wsp, int ksplit,
                       int tail_split, hipStream_t s) {
  constexpr int BM = 32 * WMT * NWM, BN = 64 * NWN;
  constexpr int ncols = GATED ? BN / 2 : BN;
  constexpr size_t lds = (size_t)2 * (BM + BN) * GT_LD * sizeof(__bf16);
  const auto kernel = gemm_tile_kernel<WMT, NWM, NWN, GATED, EXACT>;
  static bool prepared = false;
  if (!prepared) {
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)kernel,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return zk_fail("zk_gemm_bf16: the tile kernel's LDS buffers were refused");
    prepared = true;
  }
  const int tiles_n = (N + ncols - 1) / ncols, tiles_m = (M + BM - 1) / BM;
  ZK_REQUIRE((long long)tiles_m * tiles_n < 2147483647LL, "zk_gemm_bf16: too many tiles");
  // K split over blockIdx.y only as far as the partial sums fit the workspace
  const size_t per_range = (size_t)tiles_m * tiles_n * BM * BN * sizeof(float);
  void* ws = wsp.ptr;
  if (ws == nullptr || (uintptr_t)ws % 64 != 0) ksplit = 1;
  while (ksplit > 1 && per_range * ksplit > wsp.split_bytes()) ksplit--;
  if (ksplit > 1 && per_range * ksplit > wsp.bytes) return wsp.too_small(per_range * ksplit);
  const int tiles = tiles_m * tiles_n;
  // The tail.  The CUs take the tiles in rounds (256 a round for the blocks of eight and sixteen
  // waves, 512 for those of four, two of which share a CU), and a last round with few tiles
  // costs a whole round's time.  Where the caller's model of the times says it pays (a long K:
  // the partial sums of about 256 tile ranges, 16 to 67 MB, cost the same whatever K is), such
  // a last round goes into a launch of its own that splits K into ``tail_split`` ranges, and a
  // join of those tiles alone.
  constexpr int round_blocks = 256 * (NWM * NWN <= 4 ? 2 : 1);
  const int tail = tiles % round_blocks;
  if (ksplit > 1 || tail == 0 || tiles <= round_blocks || ws == nullptr || (uintptr_t)ws % 64 != 0) tail_split = 1;
  if (tail_split > 1 && (size_t)tail * tail_split * BM * BN * sizeof(float) > wsp.split_bytes()) tail_split = 1;
  if (tail_split > 1 && (size_t)tail * tail_split * BM * BN * sizeof(float) > wsp.bytes)
    return wsp.too_small((size_t)tail * tail_split * BM * BN * sizeof(float));
  const int whole = tail_split > 1 ? tiles - tail : tiles;
  kernel<<<dim3(whole, ksplit), 64 * NWM * NWN, lds, s>>>(
      (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, tiles_m, tiles_n, w_strip,
      (f32x16*)ws, ksplit, 0);
  if (ksplit > 1)
    gemm_tile_join_kernel<WMT, NWM, NWN, GATED><<<dim3(tiles * WMT * NWM * NWN), 256, 0, s>>>(
        (const f32x4*)ws, ksplit, C, ldc, c_is_f32, M, N, epi, cap, tiles_m, tiles_n, 0, tiles);
  if (tail_split > 1) {
    kernel<<<dim3(tail, tail_split), 64 * NWM * NWN, lds, s>>>(
        (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, tiles_m, tiles_n, w_strip,
        (f32x16*)ws, tail_split, whole);
    gemm_tile_join_kernel<WMT, NWM, NWN, GATED><<<dim3(tail * WMT * NWM * NWN), 256, 0, s>>>(
        (const f32x4*)ws, tail_split, C, ldc, c_is_f32, M, N, epi, cap, tiles_m, tiles_n, whole, tail);
  }
  return zk_launch_status("zk_gemm_bf16 (tile)");
}

// A caller that passes `parts` takes the partial sums of a split product as they are: planes of
// [M, N] floats at the start of the workspace, nothing in C.  That fits a plain product into a
// 16-bit C whose rows are N long, N a whole number of strips.
static bool joinable_by_reader(int N, int ldc, int c_is_f32, int epi) {
  return N % 16 == 0 && ldc == N && !c_is_f32 && epi == EPI_NONE;
}

// ------------------------------------------------------------------ mid (up to 64 rows)
// A block owns SPB strips (gated: strips of gate and up), KW waves each; all walk K together in chunks of CH 32-wide steps, of which a
// wave multiplies CH / KW, and the activations of a chunk wait in LDS for all of them.  Weights come straight from global memory in
// strip layout, the loads of the next two chunks are in flight while the current one is multiplied.
//
// Why through LDS: straight from memory every wave asks for 16 rows' half lines of 64 bytes a step, which a CU fetches at 13 to 20 bytes
// a cycle, so from some ten rows on the activations and not the weights set the time (9,216 gated columns of K 2,304 at 24 and 64 rows 20 to 21 and
// 33 us, through LDS 16.1 and 18.9).
//
// Which split (the launcher's tables): what counts is the most strips a CU gets, so SPB follows from the number of strips; KW then gives
// the block eight to sixteen waves, because a chunk's chain (reads from LDS, products) takes as long as a load and more waves a SIMD
// fill its waits.  Four waves of a strip and not two of eight strips' four places, one of them idle: 9,216 gated columns of K 2,304 at 24 and
// 64 rows 18.9 -> 16.1 and 22.4 -> 18.9 us; 4,096 of 1,024, which were 64 blocks and a join, 10.0 -> 6.1 and 12.4 -> 7.6; 8,192 of 2,048 18.8 ->
// 13.2 and 21.5 -> 15.0.
//
// Few column blocks of a plain product (N of a few thousand) cannot fill 256 CUs, so blockIdx.y splits K into
// `ksplit` ranges.  Then each block leaves its partial sums in the workspace and a second,
// small kernel adds them in the order of the ranges and applies the epilogue.  (One kernel
// with a ticket per column block, the last block adding up, was measured three times slower:
// the device-wide fences it needs write back and invalidate the L2 of every XCD.)

// A lane's results of one strip and 16 rows: columns n = 16 * strip + 4 * kq + i, row m of A.
template <bool GATED>
__device__ __forceinline__ void mid_store(const f32x4& v, const f32x4& up, int m, void* __restrict__ C, int ldc,
                                          int c_is_f32, int M, int N, int strip, int lane, int epi, float cap,
                                          float* __restrict__ picks, int nstrips) {
  const int kq = lane >> 4;
  if (!GATED && epi == EPI_PICK) {
    const float x[4] = {v[0], v[1], v[2], v[3]};
    const Pick p = pick_of_strip(x, strip * 16 + 4 * kq, N, cap);
    if (kq == 0 && m < M) ((Pick*)picks)[(size_t)m * nstrips + strip] = p;
    return;
  }
  if (m >= M) return;
  float x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = GATED ? epi_gate(v[i], up[i], epi, cap) : epi_unary(v[i], epi, cap);
  const int n = strip * 16 + 4 * kq;
  if (!c_is_f32 && n + 4 <= N && (((uintptr_t)C | (unsigned)ldc * 2) & 7) == 0) {
    store4((__bf16*)C + (size_t)m * ldc + n, x);
    return;
  }
  if (c_is_f32 && n + 4 <= N && (((uintptr_t)C | (unsigned)ldc * 4) & 15) == 0) {
    *(f32x4*)((float*)C + (size_t)m * ldc + n) = f32x4{x[0], x[1], x[2], x[3]};
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (n + i >= N) continue;
    if (c_is_f32) ((float*)C)[(size_t)m * ldc + n + i] = x[i];
    else ((__bf16*)C)[(size_t)m * ldc + n + i] = (__bf16)x[i];
  }
}

// Chains of products that a wave adds up side by side, by its steps of a chunk and by the turns of the loop: where
// fewer waves walk K than before the blocks had shapes, or ranges of it are gone, no sum has longer chains than then.
// The relative error against 64 bits, before, with one chain a wave and so: a head of 256,000 columns of K 2,304 at 17
// to 64 rows 2.0e-7, 2.9e-7 and 2.0e-7; 4,608 columns of K 8,192 at one row, sums left to the reader, 1.1e-7, 1.9e-7
// and 1.05e-7; gated 14,336 of 2,048 at up to 16 rows 1.87e-7, 2.64e-7 and 1.88e-7; gated 2,048 of 4,096 at 17 rows
// 1.5e-7, 1.9e-7 and 1.3e-7.  The times are the same.  One chain where it is no longer than then: blocks of four waves a
// strip and chunks of four steps, heads of up to 16 rows, and the rotating products (4,096 columns of K 2,304: nine steps a
// wave in eight waves, as in two waves and four ranges).
template <int MT, int SPB, int KW, int CH, bool ROPE = false>
struct MidChains {
  static constexpr int by_step = KW == 1 || (MT == 1 && CH == 2 * KW && SPB > 2) ? 2 : 1;
  static constexpr int by_turn = KW == 8 && CH == 8 && !ROPE ? 3 : MT == 1 && SPB == 3 && KW == 4 && CH == 8 ? 2 : 1;
  static constexpr int all = by_step * by_turn;
};

// t[0] + ... + t[N - 1]: neighbours first (PAIRS), or one after the other
template <bool PAIRS, int N>
__device__ __forceinline__ f32x4 sum_of(f32x4 (&t)[N]) {
  if constexpr (PAIRS) {
#pragma unroll
    for (int w = 1; w < N; w *= 2)
#pragma unroll
      for (int k = 0; k + w < N; k += 2 * w) t[k] += t[k + w];
  } else {
#pragma unroll
    for (int k = 1; k < N; k++) t[0] += t[k];
  }
  return t[0];
}

template <int MT, bool GATED, int SPB, int KW, int CH, bool ONCE, bool ROPE = false>
__global__ __launch_bounds__(SPB * KW * 64) void gemm_mid_kernel(const __bf16* __restrict__ A, int lda,
                                                                 const __bf16* __restrict__ W,
                                                                 void* __restrict__ C, int ldc, int c_is_f32,
                                                                 int M, int N, int K, int epi, float cap,
                                                                 float* __restrict__ partials, int ksplit, ArgumentIf<ROPE, RopeStore> rs = {}) {
  static_assert(!ROPE || (!GATED && KW >= MT), "a wave finishes sixteen rows");
  constexpr int NS = GATED ? 2 : 1;
  constexpr int T = SPB * KW * 64, WSTEPS = CH / KW;     // threads; steps of a chunk a wave multiplies
  constexpr int LD = CH * 32 + 16, PPR = CH * 4;         // a row of a chunk in LDS, its 16-byte pieces
  constexpr int PIECES = MT * 16 * PPR, APT = (PIECES + T - 1) / T;
  static_assert(CH % KW == 0, "whole steps a wave");
  // three chunks of activations, and after the loop the waves' sums
  constexpr size_t ACTS = (size_t)3 * MT * 16 * LD * sizeof(__bf16), SUMS = (size_t)SPB * KW * NS * MT * 64 * sizeof(f32x4);
  __shared__ __align__(16) unsigned char lds[ACTS > SUMS ? ACTS : SUMS];
  __bf16(*sA)[MT * 16][LD] = (__bf16(*)[MT * 16][LD])lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int place = wave % SPB, kpart = wave / SPB;
  const int r = lane & 15, kq = lane >> 4;
  const int ksteps = K / 32;
  const int s_begin = (int)((long)blockIdx.y * ksteps / ksplit);
  const int s_end = (int)((long)(blockIdx.y + 1) * ksteps / ksplit);
  const int nstrips = (N + 15) / 16;
  const int strip = blockIdx.x * SPB + place;
  const bool strip_ok = strip < nstrips;
  const int strip_read = min(strip, nstrips - 1);
  const __bf16* wp[NS];
  wp[0] = W + (size_t)strip_read * ksteps * 512 + lane * 8;
  if (GATED) wp[NS - 1] = W + ((size_t)(N / 16) + strip_read) * ksteps * 512 + lane * 8;
  // (ROPE) the strip's rows are eight places of a head's first half and their partners, as in the kernel above
  int head = 0, hpos = 0, slot = -1;
  float sn[4], cs[4];
  if constexpr (ROPE) {
    const int per_head = rs.hd / 16;
    head = strip_read / per_head;
    hpos = (strip_read % per_head) * 8;
    const int row = head * rs.hd + hpos + (r < 8 ? r : rs.hd / 2 + r - 8);
    wp[0] = W + (size_t)(row / 16) * ksteps * 512 + (16 * kq + row % 16) * 8;
  }
  using Chains = MidChains<MT, SPB, KW, CH, ROPE>;
  f32x4 acc[NS][MT][Chains::all];
#pragma unroll
  for (int g = 0; g < NS; g++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int c = 0; c < Chains::all; c++) acc[g][mt][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Every load is issued, none under a condition: a step past the range reads the range's last
  // step again, a row past M row M - 1; activations outside are set to zero afterwards, which
  // makes the product nothing whatever the weights.  (A thread past the pieces takes the last one, as its owner does.)
  auto fetch_a = [&](int s0, bf16x8 (&ra)[APT]) {
#pragma unroll
    for (int j = 0; j < APT; j++) {
      const int q = min(tid + T * j, PIECES - 1), row = q / PPR, piece = q % PPR;
      const bool in = row < M && s0 + piece / 4 < s_end;
      const int step = min(s0 + piece / 4, s_end - 1);
      const bf16x8 v = *(const bf16x8*)(A + (size_t)min(row, M - 1) * lda + step * 32 + (piece % 4) * 8);
      ra[j] = in ? v : zero8();
    }
  };
  auto stash_a = [&](int buf, const bf16x8 (&ra)[APT]) {
#pragma unroll
    for (int j = 0; j < APT; j++) {
      const int q = min(tid + T * j, PIECES - 1);
      *(bf16x8*)(&sA[buf][q / PPR][(q % PPR) * 8]) = ra[j];
    }
  };
  auto fetch_w = [&](int s0, bf16x8 (&wf)[NS][WSTEPS]) {
#pragma unroll
    for (int s = 0; s < WSTEPS; s++)
#pragma unroll
      for (int g = 0; g < NS; g++)
        wf[g][s] = load_weights<ONCE>(wp[g] + (size_t)min(s0 + kpart * WSTEPS + s, s_end - 1) * 512);
  };
  auto multiply = [&](int buf, auto turn, const bf16x8 (&wf)[NS][WSTEPS]) {
#pragma unroll
    for (int s = 0; s < WSTEPS; s++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const bf16x8 af = *(const bf16x8*)(&sA[buf][mt * 16 + r][(kpart * WSTEPS + s) * 32 + kq * 8]);
#pragma unroll
        for (int g = 0; g < NS; g++)
          acc[g][mt][turn % Chains::by_turn * Chains::by_step + s % Chains::by_step] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[g][s], af, acc[g][mt][turn % Chains::by_turn * Chains::by_step + s % Chains::by_step], 0, 0, 0);
      }
  };

  // Chunk c: its activations wait in LDS buffer c % 3, its weights in register set c % 3; the
  // activations of chunk c + 1 are in register set (c + 1) % 2 on their way to LDS.  A turn
  // asks for chunk c + 2, multiplies chunk c, puts chunk c + 1's activations into LDS.
  bf16x8 ra0[APT], ra1[APT], w0[NS][WSTEPS], w1[NS][WSTEPS], w2[NS][WSTEPS];
  fetch_a(s_begin, ra0);
  fetch_w(s_begin, w0);
  fetch_a(s_begin + CH, ra1);
  fetch_w(s_begin + CH, w1);
  if constexpr (ROPE) {
    // the angles of the rows that the wave will finish, while the first loads are on their way
    const int m = min(kpart * 16 + r, M - 1);
    if (kpart < MT) {
      if (head >= rs.nh && rs.slot_map) slot = rs.slot_map[m];
      if (head < rs.nh + rs.nkv) {
        const float pos = (float)rs.positions[m];
#pragma unroll
        for (int i = 0; i < 4; i++) sincosf(pos * rs.inv_freq[hpos + 4 * (kq & 1) + i], &sn[i], &cs[i]);
      }
    }
  }
  stash_a(0, ra0);
  __syncthreads();
#define ZK_MID_TURN(TURN, WCUR, WNEXT2, RA_NEXT2, RA_NEXT1)   \
  fetch_a(s0 + 2 * CH, RA_NEXT2);                             \
  fetch_w(s0 + 2 * CH, WNEXT2);                               \
  multiply(TURN % 3, std::integral_constant<int, TURN>{}, WCUR); \
  s0 += CH;                                                   \
  if (s0 >= s_end) break;                                     \
  stash_a((TURN + 1) % 3, RA_NEXT1);                          \
  __syncthreads();
  for (int s0 = s_begin;;) {
    ZK_MID_TURN(0, w0, w2, ra0, ra1)
    ZK_MID_TURN(1, w1, w0, ra1, ra0)
    ZK_MID_TURN(2, w2, w1, ra0, ra1)
    ZK_MID_TURN(3, w0, w2, ra1, ra0)
    ZK_MID_TURN(4, w1, w0, ra0, ra1)
    ZK_MID_TURN(5, w2, w1, ra1, ra0)
  }
#undef ZK_MID_TURN
  // The waves of a strip lay their sums down (the activation buffers are free once every wave has left the
  // loop) and share the rows out among themselves: sixteen rows a wave, the sums in the order of the
  // chunk's parts, or neighbours first where a wave has several.
  __syncthreads();
  f32x4* sums = (f32x4*)lds + ((size_t)place * KW * NS * MT) * 64 + lane;
#pragma unroll
  for (int g = 0; g < NS; g++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) sums[((kpart * NS + g) * MT + mt) * 64] = sum_of<true>(acc[g][mt]);
  __syncthreads();
  if (!strip_ok) return;
  const size_t npad = (size_t)nstrips * 16;
#pragma unroll
  for (int mt0 = 0; mt0 < MT; mt0 += KW) {
    const int mt = mt0 + kpart, m = mt * 16 + r;
    if (mt >= MT) break;
    f32x4 v[NS];
#pragma unroll
    for (int g = 0; g < NS; g++) {
      f32x4 part[KW];
#pragma unroll
      for (int k = 0; k < KW; k++) part[k] = sums[((k * NS + g) * MT + mt) * 64];
      v[g] = sum_of<(Chains::all > 1)>(part);
    }
    if constexpr (ROPE) {
      rope_store(rs, v[0], m, M, lane, head, hpos, slot, sn, cs, (__bf16*)C, ldc);
      continue;
    }
    if (ksplit > 1) {
      // the range's partial sums: plane (range, g) of [M, npad] floats
      float* planes = partials + (size_t)blockIdx.y * NS * M * npad + strip * 16 + 4 * kq;
#pragma unroll
      for (int g = 0; g < NS; g++)
        if (m < M) *(f32x4*)(planes + ((size_t)g * M + m) * npad) = v[g];
      continue;
    }
    mid_store<GATED>(v[0], v[NS - 1], m, C, ldc, c_is_f32, M, N, strip, lane, epi, cap, partials, nstrips);
  }
}

// The gated product of the kernel above for one row that it makes itself (RowInWork): the same sums, but the row lies in LDS whole, so the waves
// never meet in the loop, and six chunks' weights are on their way.
template <int SPB, int KW, int CH, bool ONCE, int NORM>
__global__ __launch_bounds__(SPB * KW * 64) void gemm_mid_norm_kernel(const __bf16* __restrict__ W, __bf16* __restrict__ C, int N, int K,
                                                                      int epi, RowNorm norm) {
  constexpr int NW = SPB * KW, WSTEPS = CH / KW, DEPTH = 6;
  __shared__ __align__(16) __bf16 row[4096 + CH * 32];
  __shared__ float red[32];
  __shared__ f32x4 sums[NW][2][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int place = wave % SPB, kpart = wave / SPB, kq = lane >> 4;
  const int ksteps = K / 32, nstrips = N / 16;
  const int strip = blockIdx.x * SPB + place, strip_read = min(strip, nstrips - 1);
  const __bf16* wp[2] = {W + (size_t)strip_read * ksteps * 512 + lane * 8, W + (size_t)(nstrips + strip_read) * ksteps * 512 + lane * 8};
  using Chains = MidChains<1, SPB, KW, CH>;
  static_assert(Chains::by_turn == 1, "the loop's turns are not told apart here");
  f32x4 acc[2][Chains::all];
#pragma unroll
  for (int g = 0; g < 2; g++)
#pragma unroll
    for (int c = 0; c < Chains::all; c++) acc[g][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 w[DEPTH][2][WSTEPS];
  // (steps past the end read the last one again; the row is zero there)
  auto fetch = [&](int s0, bf16x8 (&wf)[2][WSTEPS]) {
#pragma unroll
    for (int s = 0; s < WSTEPS; s++)
#pragma unroll
      for (int g = 0; g < 2; g++) wf[g][s] = load_weights<ONCE>(wp[g] + (size_t)min(s0 + kpart * WSTEPS + s, ksteps - 1) * 512);
  };
  auto multiply = [&](int s0, const bf16x8 (&wf)[2][WSTEPS]) {
#pragma unroll
    for (int s = 0; s < WSTEPS; s++) {
      const bf16x8 af = *(const bf16x8*)(row + (s0 + kpart * WSTEPS + s) * 32 + kq * 8);
#pragma unroll
      for (int g = 0; g < 2; g++)
        acc[g][s % Chains::by_step] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[g][s], af, acc[g][s % Chains::by_step], 0, 0, 0);
    }
  };
  RowOf<NW, NORM> own;
  own.ask(norm);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < DEPTH - 1; d++) fetch(d * CH, w[d]);
  __builtin_amdgcn_sched_barrier(0);
  for (int i = K + tid * 8; i < K + CH * 32; i += NW * 64 * 8) *(bf16x8*)(row + i) = zero8();
  own.make(norm, row, red, blockIdx.x == 0);
  for (int s0 = 0; s0 < ksteps;) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
      fetch(s0 + (DEPTH - 1) * CH, w[(d + DEPTH - 1) % DEPTH]);
      multiply(s0, w[d]);
      s0 += CH;
      if (s0 >= ksteps) break;
    }
  }
#pragma unroll
  for (int g = 0; g < 2; g++) sums[place * KW + kpart][g][lane] = sum_of<true>(acc[g]);
  __syncthreads();
  if (kpart > 0 || strip >= nstrips) return;
  f32x4 v[2];
#pragma unroll
  for (int g = 0; g < 2; g++) {
    f32x4 part[KW];
#pragma unroll
    for (int k = 0; k < KW; k++) part[k] = sums[place * KW + k][g][lane];
    v[g] = sum_of<(Chains::all > 1)>(part);
  }
  mid_store<true>(v[0], v[1], lane & 15, C, N, 0, 1, N, strip, lane, epi, 0.f, nullptr, nstrips);
}

// Four neighbouring results of a row, in one store where the address allows it.
__device__ __forceinline__ void store_quad(void* __restrict__ C, int ldc, int c_is_f32, int m, int n, int N, const float (&v)[4]) {
  if (!c_is_f32 && n + 4 <= N && ldc % 4 == 0 && (uintptr_t)C % 8 == 0) {
    store4((__bf16*)C + (size_t)m * ldc + n, v);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (n + i >= N) continue;
    if (c_is_f32) ((float*)C)[(size_t)m * ldc + n + i] = v[i];
    else ((__bf16*)C)[(size_t)m * ldc + n + i] = (__bf16)v[i];
  }
}

// Second half of a mid product whose K was split over blocks: `ksplit`
// ranges of one ([M, npad] floats) or, GATED, two planes each; a thread adds four neighbouring
// columns of a row in the order of the ranges and applies the epilogue.  A reader that adds the
// planes up itself in the same order (zk_norm_add_norm) makes this launch unnecessary.
template <bool GATED>
__global__ __launch_bounds__(256) void gemm_join_kernel(const float* __restrict__ partials, int ksplit,
                                                        void* __restrict__ C, int ldc, int c_is_f32, int M,
                                                        int N, int npad, int epi, float cap) {
  constexpr int NS = GATED ? 2 : 1;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int m = (int)(idx / (npad / 4)), n = (int)(idx % (npad / 4)) * 4;
  if (m >= M) return;
  const size_t plane = (size_t)M * npad;
  const float* at = partials + (size_t)m * npad + n;
  f32x4 x = *(const f32x4*)at, y = x;
  if (GATED) y = *(const f32x4*)(at + plane);
  for (int p = 1; p < ksplit; p++) {
    x += *(const f32x4*)(at + (size_t)p * NS * plane);
    if (GATED) y += *(const f32x4*)(at + ((size_t)p * NS + 1) * plane);
  }
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = GATED ? epi_gate(x[i], y[i], epi, cap) : epi_unary(x[i], epi, cap);
  store_quad(C, ldc, c_is_f32, m, n, N, v);
}

#include "gemm_bf16_tiles.h"

// How a product of up to 64 rows by weights in strips is cut: strips a block, waves a strip, steps a chunk, ranges of K.
struct MidCut {
  int spb, kw, ch, ksplit;
};

// Ranges of K for blocks of ``ch`` steps a chunk: until every CU has a block, a range no shorter than a chunk; two
// blocks a CU where ranges stay long (16 chunks of 8 steps or more: the blocks of a CU then cover each
// other's waits).  More ranges than that cost more in partial sums than they gain.  The
// longest range sets the time, so of the splits with that longest range the one with the
// fewest ranges is taken (8 chunks: 4 ranges of 2 instead of 7 of 1 or 2; measured at the
// shapes of the 2B, 9B and 27B layers with 24 to 64 rows).
static int mid_ranges(int cblocks, int ksteps, int ch) {
  const int chunks = max(1, ksteps / ch);
  int ks = max(1, min(256 / cblocks, chunks));
  if (ch == 8 && chunks / max(1, 512 / cblocks) >= 16) ks = max(1, min(512 / cblocks, chunks));
  const int longest = (chunks + ks - 1) / ks;
  return (chunks + longest - 1) / longest;
}

// The cut follows from the shape alone, and for up to 16 rows not from their number either: a request's bits do not depend on how
// many share its step.
static MidCut mid_cut(bool gated, int M, int N, int K, bool split_ok) {
  const int nstrips = (N + 15) / 16, ksteps = K / 32;
  if (gated) {
    // Few long strips (a lone block would fetch 0.8 MB and more): in ranges, with a join (2,048 columns of K 8,192 at 24 and 64
    // rows 20.1 and 22.0 us, whole 22.2 and 30.8; 512 of 4,096 at 64 14.4 and 16.5, at 24 not: 11.9 and 11.5).  Else whole: a strip a
    // block up to 256 of them, and then as many of two to four as give the fullest CU the least, of equals the more: 512 strips
    // two a block, 576 three, 896 four, 1,152 three, 1,792 four, 2,304 three.  (One a block has every strip fetch all of the
    // activations: us, 32 and 64 rows, one and three a block, 1,152 strips of K 3,072 44 and 69, 43 and 49; 1,792, one and four 65 and
    // 102, 57 and 61.)
    if (split_ok && M > 16 && nstrips <= 192 && (64.0 + 2 * M) * K > 780e3) return {4, 2, 8, mid_ranges((nstrips + 3) / 4, ksteps, 8)};
    int spb = nstrips <= 256 ? 1 : 2;
    auto most = [&](int b) { return (long)(((nstrips + b - 1) / b + 255) / 256) * b; };
    for (int b = 3; b <= 4; b++)
      if (nstrips > 256 && most(b) <= most(spb)) spb = b;
    return spb == 1 ? MidCut{1, 8, 8, 1} : spb == 2 ? MidCut{2, 4, 8, 1} : spb == 3 ? MidCut{3, 4, 4, 1} : MidCut{4, 2, 4, 1};
  }
  // Thousands of strips (a head, wide layers): two strips a block up to 16 rows, eight beyond, where the activations weigh more
  // (256,000 columns of K 2,304, four strips and eight, 24 rows 195 and 192 us, 48 228 and 214, 64 253 and 224).  Where those would be few
  // blocks a CU, three strips of four waves each up to 1,536 (17 and 64 rows of K 4,096, eight strips, four of four waves, three: 1,088 strips
  // 29.8 and 35.3, 33.3 and 43.1, 26.7 and 39.1; before the blocks had shapes 31.8 and 42.6), beyond them four with two waves each up to 48
  // rows and with four from there on (2,560 strips of K 4,096 64 rows, 16 waves a block 72.9, eight 74.3; 17 rows 73.8 and 62.1; before
  // 82.8 and 69.0).  The three rounds of 2,049 to 2,304 strips stay 2 to 8 % behind K of 4,096 and more at 17 to 32 rows.
  if (M <= 16 && nstrips >= 1024) return {2, 8, 16, 1};
  if (nstrips >= 4096) return {8, 1, 4, 1};
  if (nstrips > 1024 && nstrips <= 1536) return {3, 4, 4, 1};
  if (nstrips > 1536 && M <= 48) return {4, 2, 8, 1};
  if (nstrips >= 1024) return {4, 4, 4, 1};
  if (M <= 16) return {3, 4, 8, split_ok ? mid_ranges((nstrips + 2) / 3, ksteps, 8) : 1};
  const int cblocks = (nstrips + 3) / 4;
  if (!split_ok) return {4, 2, 8, 1};
  const int ks = mid_ranges(cblocks, ksteps, 8);
  // ranges of less than 24 steps: chunks of four and twice the waves (us, 24 and 64 rows: 4,096 columns of K 2,304 6.2 -> 5.9 and
  // 7.7 -> 7.4, 2,304 of 2,048 5.2 -> 4.6 and 6.7 -> 6.1)
  if (ks > 1 && ksteps / ks < 24) return {4, 4, 4, mid_ranges(cblocks, ksteps, 4)};
  return {4, 2, 8, ks};
}

// Which products of up to 16 rows take the blocks above; the others feed every wave straight from memory.  us,
// straight and so, 1, 8 and 16 rows.
// Gated: 9,216 columns of K 2,304 16.9, 17.4, 18.9 and 15.7, 15.7, 16.5, 14,336 of 3,584 33.9, 33.2, 37.2 and 33.3,
// 33.1, 33.4; not 8,192 of 2,048 12.6, 12.8, 13.7 and 13.1, 13.1, 13.2, nor 36,864 of 4,608 102, 98, 104 and 105,
// 100, 101.  Their share of the time straight, 1 and 8 rows, K of 1,024, 2,048, 3,072, 4,096: 513 to 768 strips 0.86
// to 1.03 and 0.84 to 0.99; 800 0.96, 0.94, 0.89, 0.97 and 0.91, 0.89, 0.85, 0.96; 896 1.01, 1.00, 0.96, 1.06 and
// 0.94, 0.96, 0.91, 1.01; 960 1.00, 1.01, 0.95, 1.02 and 0.95, 0.98, 0.93, 1.01; 1,024 1.03, 1.04, 0.99, 1.02 and
// 0.99, 1.03, 0.95, 1.00.
// Heads: 256,000 of 2,304 170, 186, 249 and 174, 179, 206; not 32,768 of 1,024 12.2, 13.1, 15.8 and 14.1, 14.5, 15.1.
// Long ones with the partial sums left to the reader: 3,584 of 14,336 17.7, 19.2, 23.5 and 17.2, 17.5, 18.2, 4,608 of
// 36,864 53, 54, 69 and 53, 51, 52; not 2,304 of 9,216 in five ranges 8.6, 9.2, 11.0 and 9.1, 9.3, 9.5.  Their share
// of the time straight, 1 and 8 rows, by strips of K 8,192, 11,008, 14,336: 193 to 384 0.82 to 1.01; 400, where K
// stays whole below 12,288, 1.10 and 1.08, 1.09 and 1.05, 0.93 and 0.89; 512, whose 342 blocks fill a third of a
// second round, 0.99 and 1.00, 1.04 and 1.05, 1.02 and 1.04; 544 to 768 0.87 to 1.00; 832 1.18 and 1.11, 1.17 and
// 1.14, 1.16 and 1.16; 896 to 1,023 0.99 to 1.09.
static bool mid_for_few(bool gated, int N, int K, bool by_reader) {
  const int nstrips = (N + 15) / 16;
  if (gated) return nstrips > 512 && nstrips <= (K % 4096 ? 960 : 800);
  if (nstrips >= 1024) return K >= 2048;
  if (!by_reader || K < 8192 || nstrips <= 192) return false;
  return nstrips <= 384 || (nstrips > 512 && nstrips <= 768) || (nstrips < 512 && mid_ranges((nstrips + 2) / 3, K / 32, 8) > 1);
}

// Bytes of the partial sums of one range.
static size_t mid_range_bytes(bool gated, int M, int N) { return (size_t)(gated ? 2 : 1) * M * ((N + 15) / 16 * 16) * sizeof(float); }

// The cut of a launch: ranges of K only where there is a workspace that 16-byte stores reach and that holds them.  Picks are taken
// from whole sums; up to 16 rows only a reader that adds up the partial sums itself is worth a split.
static MidCut mid_cut_of_launch(bool gated, bool by_reader, int M, int N, int K, int epi, const GemmWorkspace& wsp) {
  const bool split_ok = wsp.ptr != nullptr && (uintptr_t)wsp.ptr % 16 == 0 && epi != EPI_PICK && (M > 16 || by_reader);
  MidCut cut = mid_cut(gated, M, N, K, split_ok);
  while (cut.ksplit > 1 && cut.ksplit * mid_range_bytes(gated, M, N) > wsp.split_bytes()) cut.ksplit--;
  return cut;
}

template <bool GATED>
static int launch_mid(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32, int M, int N,
                      int K, int epi, float cap, int w_strip, const GemmWorkspace& wsp, int* parts, hipStream_t s) {
  const int mt = (M + 15) / 16;
  const int nstrips = (N + 15) / 16, npad = nstrips * 16;
  const bool by_reader = parts != nullptr && joinable_by_reader(N, ldc, c_is_f32, epi);
  const MidCut cut = mid_cut_of_launch(GATED, by_reader, M, N, K, epi, wsp);
  if (cut.ksplit > 1 && cut.ksplit * mid_range_bytes(GATED, M, N) > wsp.bytes) return wsp.too_small(cut.ksplit * mid_range_bytes(GATED, M, N));
  const int ksplit = cut.ksplit;
  float* partials = (float*)wsp.ptr;
  dim3 grid((nstrips + cut.spb - 1) / cut.spb, ksplit);
#define ZK_MID_(MT_, SPB_, KW_, CH_, ONCE_)                                                             \
  gemm_mid_kernel<MT_, GATED, SPB_, KW_, CH_, ONCE_><<<grid, SPB_ * KW_ * 64, 0, s>>>((const __bf16*)A, lda, (const __bf16*)W, C, ldc, \
                                                                                     c_is_f32, M, N, K, epi, cap, partials, ksplit)
#define ZK_MID(MT_, SPB_, KW_, CH_)                                                      \
  do {                                                                                   \
    if (reads_once(w_strip)) ZK_MID_(MT_, SPB_, KW_, CH_, true);                         \
    else ZK_MID_(MT_, SPB_, KW_, CH_, false);                                            \
  } while (0)
// 17 to 64 rows
#define ZK_MID_ROWS(SPB_, KW_, CH_)                   \
  do {                                                \
    if (mt == 2) ZK_MID(2, SPB_, KW_, CH_);           \
    else if (mt == 3) ZK_MID(3, SPB_, KW_, CH_);      \
    else ZK_MID(4, SPB_, KW_, CH_);                   \
  } while (0)
  if (mt == 1) {
    // the cuts of mid_for_few
    if constexpr (GATED) {
      if (cut.spb == 3) ZK_MID(1, 3, 4, 4);
      else ZK_MID(1, 4, 2, 4);
    } else {
      if (cut.spb == 2) ZK_MID(1, 2, 8, 16);
      else ZK_MID(1, 3, 4, 8);
    }
  } else if (cut.spb == 4 && cut.ch == 8) ZK_MID_ROWS(4, 2, 8);
  else if constexpr (GATED) {
    if (cut.spb == 1) ZK_MID_ROWS(1, 8, 8);
    else if (cut.spb == 2) ZK_MID_ROWS(2, 4, 8);
    else if (cut.spb == 3) ZK_MID_ROWS(3, 4, 4);
    else ZK_MID_ROWS(4, 2, 4);
  } else {
    if (cut.spb == 8) ZK_MID_ROWS(8, 1, 4);
    else if (cut.spb == 3) ZK_MID_ROWS(3, 4, 4);
    else ZK_MID_ROWS(4, 4, 4);
  }
#undef ZK_MID_ROWS
#undef ZK_MID
#undef ZK_MID_
  if (ksplit > 1) {
    if (by_reader) {
      *parts = ksplit;
      return zk_launch_status("zk_gemm_bf16 (mid)");
    }
    const size_t quads = (size_t)M * (npad / 4);
    gemm_join_kernel<GATED><<<(unsigned)((quads + 255) / 256), 256, 0, s>>>(partials, ksplit, C, ldc, c_is_f32, M, N,
                                                                          npad, epi, cap);
  }
  return zk_launch_status("zk_gemm_bf16 (mid)");
}

template <bool GATED>
static int launch_skinny(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32, int M,
                         int N, int K, int epi, float cap, int w_strip, const GemmWorkspace& wsp, int* parts,
                         hipStream_t s) {
  const int mt = (M + 15) / 16;
  dim3 grid((N + 15) / 16);
  // A strip is a block, and the blocks of a CU share its way to memory: the kernel takes as
  // long as the CU with the most blocks.  288 strips (N = 4608) leave 32 of the 256 CUs with two
  // blocks and the rest with one, twice the time of an even spread; 144 strips leave 112 CUs
  // idle.  Splitting K into ks ranges makes ks times the blocks of 1/ks the length, and the time
  // of the fullest CU goes with ceil(strips ks / 256) / ks.  That pays where strips are more
  // than the CUs and spread unevenly (N = 4608 with K = 36864 at 8 rows: 87 -> 50 us with eight
  // ranges), and where they are fewer and long (blocks of four waves; us, 1 and 8 rows, without the reader's
  // half a microsecond and more: 144 strips of 9,216 in five ranges 10.3 -> 9.2 and 12.3 -> 9.8, 128 of 8,192 in two 9.3 -> 8.2 and
  // 11.2 -> 8.4, 64 of 4,096 in four 4.1 -> 3.5 and 5.3 -> 3.7), not where they are short (128 of 2,048 in two 3.4 -> 3.5 and
  // 3.9 -> 3.7) or nearly fill the chip (224 of 14,336 in eight 19.1 -> 19.2 and 20.1 -> 20.5).
  // Only where the reader adds up the partial sums itself (the norm kernel, through `parts`):
  // a joining launch would cost what the split gains.
  int ksplit = 1;
  float* partials = (float*)wsp.ptr;
  const size_t npad = (size_t)grid.x * 16;
  bool few_long = false;
  if (!GATED && mt == 1 && w_strip && parts != nullptr && partials != nullptr &&
      (uintptr_t)partials % 16 == 0 && joinable_by_reader(N, ldc, c_is_f32, epi)) {
    auto longest = [&](int ks) { return (double)(((long)grid.x * ks + 255) / 256) / ks; };
    if (grid.x <= 256) {
      // microseconds: the fullest CU at 25 KB, the chip at 6.1 MB, the reader's additions
      const double kb = K * 0.032, chip = grid.x * kb / 6100;
      auto price = [&](int ks) { return std::max(longest(ks) * kb / 25, chip) + (ks > 1 ? 0.5 + 0.05 * ks : 0.0); };
      double best = price(1) - 1.5;
      for (int ks = 2; ks <= 6 && K / ks >= 1024 && (size_t)ks * M * npad * sizeof(float) <= wsp.split_bytes(); ks++)
        if (price(ks) < best) {
          best = price(ks);
          ksplit = ks;
          few_long = true;
        }
    } else {
      double best = longest(1);
      for (int ks = 2; ks <= 8; ks *= 2) {
        if (K / ks < 1024 || (size_t)ks * M * npad * sizeof(float) > wsp.split_bytes()) break;
        if (longest(ks) < 0.97 * best && longest(ks) <= 0.85 * longest(1)) {
          best = longest(ks);
          ksplit = ks;
        }
      }
    }
    if (ksplit > 1 && (size_t)ksplit * M * npad * sizeof(float) > wsp.bytes)
      return wsp.too_small((size_t)ksplit * M * npad * sizeof(float));
    grid.y = ksplit;
  }
  // rows of A within reach of a lane's own offset
  const bool whole = w_strip && mt == 1 && K % 256 == 0 && lda <= (1 << 26);
  // few strips: eight waves a strip keep enough loads in flight
  const bool wide = !few_long && (long)grid.x * ksplit < 512 && K / ksplit >= 2048 && mt <= 2;
  const bool once = reads_once(w_strip);
#define ZK_SKINNY(MT_, NW_)                                                                           \
  do {                                                                                                \
    if (MT_ == 1 && whole && once)                                                                    \
      gemm_skinny_kernel<1, GATED, NW_, false, true, false, true, true><<<grid, NW_ * 64, 0, s>>>(    \
          (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, RopeStore{}, \
          partials, 1);                                                                               \
    else if (MT_ == 1 && whole)                                                                       \
      gemm_skinny_kernel<1, GATED, NW_, false, true, false, true><<<grid, NW_ * 64, 0, s>>>(          \
          (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, RopeStore{}, \
          partials, 1);                                                                               \
    else if (w_strip)                                                                                      \
      gemm_skinny_kernel<MT_, GATED, NW_, false, true><<<grid, NW_ * 64, 0, s>>>(                     \
          (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, RopeStore{}, \
          partials, 1);                                                                               \
    else                                                                                              \
      gemm_skinny_kernel<MT_, GATED, NW_><<<grid, NW_ * 64, 0, s>>>(                                  \
          (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, RopeStore{}, \
          partials, 1);                                                                               \
  } while (0)
#define ZK_SPLIT(NW_, WHOLE_, ONCE_)                                                                        \
  gemm_skinny_kernel<1, false, NW_, false, true, true, WHOLE_, ONCE_><<<grid, NW_ * 64, 0, s>>>(             \
      (const __bf16*)A, lda, (const __bf16*)W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, RopeStore{}, partials, ksplit)
  if (ksplit > 1) {
    if constexpr (!GATED) {
      if (wide) { if (whole && once) ZK_SPLIT(8, true, true); else if (whole) ZK_SPLIT(8, true, false); else ZK_SPLIT(8, false, false); }
      else { if (whole && once) ZK_SPLIT(4, true, true); else if (whole) ZK_SPLIT(4, true, false); else ZK_SPLIT(4, false, false); }
    }
  } else if (mt == 1) { if (wide) ZK_SKINNY(1, 8); else ZK_SKINNY(1, 4); }
  else if (mt == 2) { if (wide) ZK_SKINNY(2, 8); else ZK_SKINNY(2, 4); }
  else if (mt == 3) ZK_SKINNY(3, 4);
  else ZK_SKINNY(4, 4);
#undef ZK_SKINNY
#undef ZK_SPLIT
  if (ksplit > 1) *parts = ksplit;
  return zk_launch_status("zk_gemm_bf16 (skinny)");
}

// The q|k|v product of up to 16 decoded tokens with the rotation and the cache store as its
// epilogue: W [(nh + 2 nkv) hd, K] (row-major or strip layout), q rotated into Q [M, ldq] at
// columns [0, nh hd), k rotated and v as it is into the cache at slot_map[m] (a negative slot
// stores nothing).  The same bits as zk_gemm_bf16 followed by zk_rope_cache_write.  nkv may be 0
// (a mixer that reads another's cache); then slot_map and the caches are not used.
extern "C" int zk_qkv_rope_bf16_supports(int M, int K, int hd, int rotary_dim) {
  return M >= 1 && M <= 16 && K % 8 == 0 && hd % 16 == 0 && rotary_dim == hd;
}

extern "C" int zk_qkv_rope_bf16(const void* A, int lda, const void* W, void* Q, int ldq, int M, int K,
                                int w_strip, const int* positions, const int* slot_map,
                                const float* inv_freq, void* kcache, void* vcache, int nh, int nkv, int hd,
                                int bs, int v_transposed, void* stream) {
  ZK_REQUIRE(M >= 1 && M <= 16 && K > 0 && K % 8 == 0 && lda % 8 == 0 && lda >= K,
             "zk_qkv_rope_bf16: 1 to 16 rows, K and lda multiples of 8");
  ZK_REQUIRE(nh > 0 && nkv >= 0 && hd > 0 && hd % 16 == 0, "zk_qkv_rope_bf16: head_dim must be a multiple of 16");
  ZK_REQUIRE(ldq >= nh * hd && ldq % 4 == 0, "zk_qkv_rope_bf16: ldq too small or not a multiple of 4");
  ZK_REQUIRE(!w_strip || K % 32 == 0, "zk_qkv_rope_bf16: strip layout needs K % 32 == 0");
  ZK_REQUIRE(positions && inv_freq, "zk_qkv_rope_bf16: positions and inv_freq are needed");
  ZK_REQUIRE(nkv == 0 || (slot_map && kcache && vcache && bs > 0), "zk_qkv_rope_bf16: the cache is needed");
  ZK_REQUIRE(((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0) && ((uintptr_t)Q % 8 == 0),
             "zk_qkv_rope_bf16: operands must be 16-byte aligned");
  const int N = (nh + 2 * nkv) * hd;
  RopeStore rs{positions, nkv ? slot_map : nullptr, inv_freq, (__bf16*)kcache, (__bf16*)vcache, nh, nkv, hd, bs,
               v_transposed};
  dim3 grid(N / 16);
  hipStream_t s = (hipStream_t)stream;
  const bool whole = w_strip && K % 256 == 0 && lda <= (1 << 26);
  const bool once = reads_once(w_strip);
#define ZK_QKV(NW_, EX_, WH_, ONCE_)                                                                                          \
  gemm_skinny_kernel<1, false, NW_, true, EX_, false, WH_, ONCE_><<<grid, NW_ * 64, 0, s>>>((const __bf16*)A, lda, (const __bf16*)W, Q, \
                                                                                    ldq, 0, M, N, K, EPI_NONE, 0.f, w_strip, rs)
  if (grid.x < 512 && K >= 2048) {
    if (whole && once) ZK_QKV(8, true, true, true); else if (whole) ZK_QKV(8, true, true, false);
    else if (w_strip) ZK_QKV(8, true, false, false); else ZK_QKV(8, false, false, false);
  } else {
    if (whole && once) ZK_QKV(4, true, true, true); else if (whole) ZK_QKV(4, true, true, false);
    else if (w_strip) ZK_QKV(4, true, false, false); else ZK_QKV(4, false, false, false);
  }
#undef ZK_QKV
  return zk_launch_status("zk_qkv_rope_bf16");
}

// The same for 17 to 64 rows (weights in strips): a strip of a head's places and their partners a block, or two, K
// whole.  Against the product with K in ranges and the rotation that adds them up it is a launch less (us, 24, 40 and
// 64 rows, two launches and this: 4,096 columns of K 2,304 11.3, 12.5, 13.8 and 9.8, 11.2, 12.4; 8,192 of 3,584 16.7,
// 18.0, 20.3 and 14.3, 16.1, 18.9; 1,536 of 1,024 9.8, 10.4, 11.8 and 5.8, 6.7, 7.3).  Rounds to 16 bits in front of
// the rotation, as those do.
// K whole has an end where the ranges fill the chip better (this one's share of the two launches' time, 17 to 64
// rows, heads of 64 and 128 channels, of 256 in brackets): 96 to 320 strips K 2,304 0.82 to 1.03 (0.59 to 0.90),
// 3,072 0.93 to 1.11 (0.74 to 0.98), 3,584 0.99 to 1.17 (0.73 to 1.02), 4,096 0.98 to 1.24 (0.85 to 1.08), 5,120 1.10
// to 1.40 (0.92 to 1.25); 384 and 448 4,096 0.90 to 0.98 (0.85 to 0.95), 4,608 0.98 to 1.09; 512 4,608 0.95 to 1.02,
// 5,120 0.97 to 1.05; 640 up to 32 rows 768 to 2,304 0.79 to 1.01, 3,072 0.95 to 1.05, from 33 rows 1.03 to 1.40.
extern "C" int zk_qkv_rope_rows_bf16_pays(int M, int N, int K, int hd) {
  const int strips = N / 16;
  return K <= (strips > 512 ? (M <= 32 ? 2304 : 0) : strips >= 480 ? 4608 : strips >= 384 ? 4096 : hd >= 256 ? 3584 : 2560);
}

extern "C" int zk_qkv_rope_rows_bf16_supports(int M, int K, int hd, int rotary_dim) {
  return M > 16 && M <= 64 && K > 0 && K % 32 == 0 && hd % 16 == 0 && rotary_dim == hd;
}

extern "C" int zk_qkv_rope_rows_bf16(const void* A, int lda, const void* W, void* Q, int ldq, int M, int K, int w_strip,
                                     const int* positions, const int* slot_map, const float* inv_freq, void* kcache, void* vcache, int nh,
                                     int nkv, int hd, int bs, int v_transposed, void* stream) {
  ZK_REQUIRE(M > 16 && M <= 64 && K > 0 && K % 32 == 0 && lda % 8 == 0 && lda >= K && w_strip,
             "zk_qkv_rope_rows_bf16: 17 to 64 rows, weights in strips, lda a multiple of 8");
  ZK_REQUIRE(nh > 0 && nkv >= 0 && hd > 0 && hd % 16 == 0, "zk_qkv_rope_rows_bf16: head_dim must be a multiple of 16");
  ZK_REQUIRE(ldq >= nh * hd && ldq % 4 == 0, "zk_qkv_rope_rows_bf16: ldq too small or not a multiple of 4");
  ZK_REQUIRE(positions && inv_freq, "zk_qkv_rope_rows_bf16: positions and inv_freq are needed");
  ZK_REQUIRE(nkv == 0 || (slot_map && kcache && vcache && bs > 0), "zk_qkv_rope_rows_bf16: the cache is needed");
  ZK_REQUIRE(((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0) && ((uintptr_t)Q % 8 == 0),
             "zk_qkv_rope_rows_bf16: operands must be 16-byte aligned");
  const int N = (nh + 2 * nkv) * hd, mt = (M + 15) / 16;
  RopeStore rs{positions, nkv ? slot_map : nullptr, inv_freq, (__bf16*)kcache, (__bf16*)vcache, nh, nkv, hd, bs, v_transposed};
  hipStream_t s = (hipStream_t)stream;
#define ZK_ROPE_(MT_, SPB_, ONCE_)                                                                                        \
  gemm_mid_kernel<MT_, false, SPB_, 8, 8, ONCE_, true><<<(N / 16 + SPB_ - 1) / SPB_, SPB_ * 512, 0, s>>>(                  \
      (const __bf16*)A, lda, (const __bf16*)W, Q, ldq, 0, M, N, K, EPI_NONE, 0.f, nullptr, 1, rs)
#define ZK_ROPE(SPB_, ONCE_)                      \
  do {                                            \
    if (mt == 2) ZK_ROPE_(2, SPB_, ONCE_);        \
    else if (mt == 3) ZK_ROPE_(3, SPB_, ONCE_);   \
    else ZK_ROPE_(4, SPB_, ONCE_);                \
  } while (0)
  if (N / 16 <= 256) { if (reads_once(w_strip)) ZK_ROPE(1, true); else ZK_ROPE(1, false); }
  else { if (reads_once(w_strip)) ZK_ROPE(2, true); else ZK_ROPE(2, false); }
#undef ZK_ROPE
#undef ZK_ROPE_
  return zk_launch_status("zk_qkv_rope_rows_bf16");
}

// The two products behind a norm, for one row that the product makes itself: what zk_norm_add_norm (sub, up to 6
// planes, w_post, h, w_next) followed by zk_qkv_rope_bf16, or by zk_gemm_bf16 with a gated epilogue, gives, to the
// bit.  h_out: the new stream, elsewhere than h.  sub must not lie where the product writes.  Weights in strips, K a
// multiple of 256 up to 4,096.
static int row_norm_of(RowNorm& p, const void* sub, int sub_parts, const float* w_post, float eps_post, int uo_post, const float* h, float* h_out,
                       const float* w_next, float eps_next, int uo_next, int K) {
  ZK_REQUIRE(K > 0 && K % 256 == 0 && K <= 4096, "zk_norm product: K must be a multiple of 256 up to 4096");
  ZK_REQUIRE(sub_parts >= 0 && sub_parts <= 6, "zk_norm product: up to 6 planes of partial sums");
  ZK_REQUIRE(sub && h && h_out && w_post && w_next && h != h_out, "zk_norm product: sub, h, another h_out, w_post and w_next are needed");
  ZK_REQUIRE((((uintptr_t)sub | (uintptr_t)h | (uintptr_t)h_out | (uintptr_t)w_next | (uintptr_t)w_post) & 15) == 0,
             "zk_norm product: operands must be 16-byte aligned");
  p = RowNorm{sub, w_post, h, h_out, w_next, eps_post, eps_next, sub_parts, uo_post, uo_next, K};
  return 0;
}

// Where that is no slower than the two launches (a chain of either, one row, K of 2,048 to 4,096; its share of their time by planes of
// partial sums).  Below K of 2,048 0.7 to 0.96 everywhere.  Rotating: up to 256 strips 0.81 to 0.94; 288 to 448 0.76 to 0.92 with up to four
// planes and 1.02 to 1.07 with six, whose loads no longer fit beside the weights'; 512 0.86 to 0.95; 576 to 896 0.81 to 1.00 without planes and
// 0.97 to 1.17 with them (eight waves' rows by four).  Gated straight from memory likewise: 256 and 512 strips 0.85 to 0.95; 1,024 to 2,304
// 0.94 to 1.01 without planes, 0.93 to 1.05 with them.  Gated by blocks: of three strips K 2,048 0.92 to 0.99, 2,304 to 2,816 0.95 to 1.03, 3,072
// 1.01 to 1.07, 3,328 and 3,584 0.97 to 1.02, 3,840 and 4,096 1.01 to 1.05; of four 2,048 0.97 to 1.00, beyond 1.00 to 1.11.
static bool norm_product_pays(bool gated, int N, int K, int sub_parts) {
  if (K <= 0 || K % 256 || K > 4096 || sub_parts > 6) return false;
  const int nstrips = N / 16;
  if (gated && mid_for_few(true, N, K, false)) {
    if (K < 2048) return false;
    return mid_cut(true, 1, N, K, false).spb == 3 ? K <= 2816 || (K > 3072 && K <= 3584) : K <= 2048;
  }
  if (K < 2048) return true;
  return nstrips < 512 ? sub_parts <= 4 || nstrips <= 256 : nstrips == 512 || sub_parts == 0;
}

// Whether zk_norm_gated_bf16 (N columns), or zk_norm_qkv_rope_bf16 (N columns of q, k and v), is to take a row of so many planes.
extern "C" int zk_norm_product_supports(int N, int K, int sub_parts) { return norm_product_pays(true, N, K, sub_parts); }
extern "C" int zk_norm_rope_product_supports(int N, int K, int sub_parts) { return norm_product_pays(false, N, K, sub_parts); }

#define ZK_NORM_MODES(NW_, SLOTS_, WIDE_)                                                          \
  do {                                                                                             \
    if (reads_once(w_strip)) {                                                                     \
      if (sub_parts == 0) ZK_LAUNCH(NW_, true, row_norm_mode(SLOTS_, WIDE_, 0));                   \
      else if (sub_parts <= 4) ZK_LAUNCH(NW_, true, row_norm_mode(SLOTS_, WIDE_, 4));              \
      else ZK_LAUNCH(NW_, true, row_norm_mode(SLOTS_, WIDE_, 6));                                  \
    } else {                                                                                       \
      if (sub_parts == 0) ZK_LAUNCH(NW_, false, row_norm_mode(SLOTS_, WIDE_, 0));                  \
      else if (sub_parts <= 4) ZK_LAUNCH(NW_, false, row_norm_mode(SLOTS_, WIDE_, 4));             \
      else ZK_LAUNCH(NW_, false, row_norm_mode(SLOTS_, WIDE_, 6));                                 \
    }                                                                                              \
  } while (0)

extern "C" int zk_norm_qkv_rope_bf16(const void* sub, int sub_parts, const float* w_post, float eps_post, int uo_post, const float* h,
                                     void* h_out, const float* w_next, float eps_next, int uo_next, const void* W, void* Q, int ldq,
                                     int K, int w_strip, const int* positions, const int* slot_map, const float* inv_freq, void* kcache,
                                     void* vcache, int nh, int nkv, int hd, int bs, int v_transposed, void* stream) {
  RowNorm p;
  if (int rc = row_norm_of(p, sub, sub_parts, w_post, eps_post, uo_post, h, (float*)h_out, w_next, eps_next, uo_next, K)) return rc;
  ZK_REQUIRE(w_strip, "zk_norm_qkv_rope_bf16: weights in strips");
  ZK_REQUIRE(nh > 0 && nkv >= 0 && hd > 0 && hd % 16 == 0, "zk_norm_qkv_rope_bf16: head_dim must be a multiple of 16");
  ZK_REQUIRE(ldq >= nh * hd && ldq % 4 == 0, "zk_norm_qkv_rope_bf16: ldq too small or not a multiple of 4");
  ZK_REQUIRE(positions && inv_freq, "zk_norm_qkv_rope_bf16: positions and inv_freq are needed");
  ZK_REQUIRE(nkv == 0 || (slot_map && kcache && vcache && bs > 0), "zk_norm_qkv_rope_bf16: the cache is needed");
  ZK_REQUIRE((uintptr_t)W % 16 == 0 && (uintptr_t)Q % 8 == 0, "zk_norm_qkv_rope_bf16: operands must be 16-byte aligned");
  const int N = (nh + 2 * nkv) * hd;
  RopeStore rs{positions, nkv ? slot_map : nullptr, inv_freq, (__bf16*)kcache, (__bf16*)vcache, nh, nkv, hd, bs, v_transposed};
  dim3 grid(N / 16);
  hipStream_t s = (hipStream_t)stream;
#define ZK_LAUNCH(NW_, ONCE_, MODE_)                                                                                           \
  gemm_skinny_kernel<1, false, NW_, true, true, false, true, ONCE_, MODE_><<<grid, NW_ * 64, 0, s>>>(                           \
      nullptr, K, (const __bf16*)W, Q, ldq, 0, 1, N, K, EPI_NONE, 0.f, w_strip, rs, nullptr, 1, p)
  // as zk_qkv_rope_bf16: eight waves for few long strips, else four
  if (grid.x < 512 && K >= 2048) ZK_NORM_MODES(8, 2, true);
  else if (K >= 2048) ZK_NORM_MODES(4, 4, true);
  else if (K > 1024) ZK_NORM_MODES(4, 2, false);
  else ZK_NORM_MODES(4, 1, false);
#undef ZK_LAUNCH
  return zk_launch_status("zk_norm_qkv_rope_bf16");
}

extern "C" int zk_norm_gated_bf16(const void* sub, int sub_parts, const float* w_post, float eps_post, int uo_post, const float* h,
                                  void* h_out, const float* w_next, float eps_next, int uo_next, const void* W, void* C, int N, int K,
                                  int epi, int w_strip, void* stream) {
  RowNorm p;
  if (int rc = row_norm_of(p, sub, sub_parts, w_post, eps_post, uo_post, h, (float*)h_out, w_next, eps_next, uo_next, K)) return rc;
  ZK_REQUIRE(w_strip && N > 0 && N % 16 == 0, "zk_norm_gated_bf16: weights in strips, N a multiple of 16");
  ZK_REQUIRE(epi == EPI_GELU_TANH || epi == EPI_SILU || epi == EPI_RELU, "zk_norm_gated_bf16: not a gated epilogue without a limit");
  ZK_REQUIRE((uintptr_t)W % 16 == 0 && (uintptr_t)C % 16 == 0, "zk_norm_gated_bf16: operands must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  if (mid_for_few(true, N, K, false)) {
    // as launch_mid for up to 16 rows: 513 to 1,024 strips, three or four a block
    const MidCut cut = mid_cut(true, 1, N, K, false);
    dim3 grid((N / 16 + cut.spb - 1) / cut.spb);
    ZK_REQUIRE(K >= 2048 && (cut.spb == 3 || cut.spb == 4), "zk_norm_gated_bf16: no kernel for so many strips of this length");
#define ZK_LAUNCH(NW_, ONCE_, MODE_)                                                                                                     \
  gemm_mid_norm_kernel<NW_ == 12 ? 3 : 4, NW_ == 12 ? 4 : 2, 4, ONCE_, MODE_><<<grid, NW_ * 64, 0, s>>>((const __bf16*)W, (__bf16*)C, N, K, epi, p)
    if (cut.spb == 4) ZK_NORM_MODES(8, 2, true);
    else if (K > 3072) ZK_NORM_MODES(12, 2, true);
    else ZK_NORM_MODES(12, 1, true);
#undef ZK_LAUNCH
    return zk_launch_status("zk_norm_gated_bf16 (mid)");
  }
  // as launch_skinny
  dim3 grid(N / 16);
#define ZK_LAUNCH(NW_, ONCE_, MODE_)                                                                                  \
  gemm_skinny_kernel<1, true, NW_, false, true, false, true, ONCE_, MODE_><<<grid, NW_ * 64, 0, s>>>(                  \
      nullptr, K, (const __bf16*)W, C, N, 0, 1, N, K, epi, 0.f, w_strip, RopeStore{}, nullptr, 1, p)
  if ((long)grid.x < 512 && K >= 2048) ZK_NORM_MODES(8, 2, true);
  else if (K >= 2048) ZK_NORM_MODES(4, 4, true);
  else if (K > 1024) ZK_NORM_MODES(4, 2, false);
  else ZK_NORM_MODES(4, 1, false);
#undef ZK_LAUNCH
  return zk_launch_status("zk_norm_gated_bf16 (skinny)");
}

// Strip layout of a [N, K] weight matrix, K % 32 == 0: rows in strips of 16 (the last strip
// padded with zeros), each (strip, 32-wide k step) one KB in which lane l = 16 * kq + r holds
// W[16 * strip + r][32 * step + 8 * kq .. + 8], i.e. exactly what the 64 lanes of a wave load
// for one 16x16x32 MFMA; steps follow each other, then strips.  A wave that streams its run
// of steps reads contiguous memory instead of sixteen rows K elements apart, which keeps
// every memory channel busy whatever K is (row strides of 4096 or 18432 bytes do not).
__global__ void strip_layout_kernel(const __bf16* __restrict__ src, __bf16* __restrict__ dst, int N, int K,
                                    size_t pieces) {
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= pieces) return;
  const int ksteps = K / 32;
  const size_t block = q >> 6;
  const int l = (int)(q & 63);
  const int n = (int)(block / ksteps) * 16 + (l & 15);
  const int k = (int)(block % ksteps) * 32 + (l >> 4) * 8;
  *(bf16x8*)(dst + q * 8) = n < N ? *(const bf16x8*)(src + (size_t)n * K + k) : zero8();
}

// dst holds ceil(N / 16) * 16 rows of K elements.
extern "C" int zk_strip_layout(const void* src, void* dst, int N, int K, void* stream) {
  ZK_REQUIRE(N > 0 && K > 0 && K % 32 == 0, "zk_strip_layout: K must be a positive multiple of 32");
  const size_t pieces = (size_t)((N + 15) / 16) * 16 * K / 8;
  ZK_REQUIRE((pieces + 255) / 256 < 2147483647ull, "zk_strip_layout: matrix too large");
  strip_layout_kernel<<<(unsigned)((pieces + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      (const __bf16*)src, (__bf16*)dst, N, K, pieces);
  return zk_launch_status("zk_strip_layout");
}

// epi: 0 none, 1 soft cap (cap > 0), 2 gelu_tanh gate, 3 silu gate, 5 relu gate, 6 clamped gate (cap: its limit).  For the gated
// epilogues W is [2N, K] (gate rows, then up rows) and C is [M, N].
// w_strip: not 0: W is in strip layout (zk_strip_layout); 3: and belongs to a model too large for the memory side's cache, so that products of up to
// 64 rows read it past the caches (the same bits either way).  Strip layout needs K % 32 == 0 and, for the
// gated epilogues, N % 16 == 0.
// The workspace may be null; then K is never split over blocks.  It serves one launch at a time.
// parts (may be null): a caller whose next kernel can add partial sums up itself passes a place
// for their number.  0 comes back when the result is in C as usual; P > 0 when C was not
// written and the workspace starts with P planes of [M, N] floats, to be added in order and
// rounded to 16 bits (zk_norm_add_norm reads them so), before the next product overwrites them.
extern "C" size_t zk_gemm_bf16_workspace() { return ZK_GEMM_WORKSPACE_BYTES; }

// A tile variant (0: 128 x 128 blocks of four waves, 1: 64 x 128, 2: 128 x 256 of eight,
// 3: 256 x 256 of sixteen) with K split into ks ranges, and a model of its time in microseconds:
// the CU with the most blocks works through them one after the other, a block costs a start-up
// and a time per 64-wide k tile, a lone block a CU differs from one of several by a factor,
// and a split adds a joining kernel that moves the partial sums.  The constants are fitted to
// measurements (see where it is used).
struct TileChoice { int v, ks; };
static double tile_cost(TileChoice c, int M, int N, int K, bool gated, size_t room, int* tail_split = nullptr) {
  if (tail_split) *tail_split = 1;
  static const int BM[4] = {128, 64, 128, 256}, BN[4] = {128, 128, 256, 256};
  static const double start[4] = {0.0, 0.0, 0.974, 4.75}, per_ktile[4] = {0.522, 0.344, 0.881, 1.48},
                      lone[4] = {1.274, 1.432, 0.994, 0.903};
  const double launch = 3.774, join_start = 4.183, join_per_mb = 0.553;
  const int ncols = gated ? BN[c.v] / 2 : BN[c.v];
  const long tiles = (long)((M + BM[c.v] - 1) / BM[c.v]) * ((N + ncols - 1) / ncols);
  const double range_bytes = (double)tiles * BM[c.v] * BN[c.v] * 4.0;
  int ks = c.ks;
  while (ks > 1 && range_bytes * ks > (double)room) ks--;     // as the launcher will clamp it
  if (ks != c.ks) return 1e30;                                  // priced under the split it becomes
  if (ks > 1 && (K + GT_BK - 1) / GT_BK < 2 * ks) return 1e30;  // no ranges of less than two k tiles
  const int ktiles_all = (K + GT_BK - 1) / GT_BK;
  const int ktiles = (ktiles_all + ks - 1) / ks;
  const long per_cu = (tiles * ks + 255) / 256;
  double t = launch + per_cu * (start[c.v] + ktiles * per_ktile[c.v]) * (per_cu == 1 ? lone[c.v] : 1.0);
  if (ks > 1) t += join_start + ks * range_bytes / 1e6 * join_per_mb;
  // a last round of few tiles is launched apart with K in ranges (launch_tile has the rule)
  const long round_blocks = c.v <= 1 ? 512 : 256, tail = tiles % round_blocks;
  if (ks == 1 && tiles > round_blocks && tail > 0 && 2 * tail <= round_blocks && room > 0) {
    const double tile_bytes = (double)BM[c.v] * BN[c.v] * 4.0;
    int ts = (int)(round_blocks / tail < 8 ? round_blocks / tail : 8);
    while (ts > 1 && (ktiles_all / ts < 4 || tail * ts * tile_bytes > (double)room)) ts--;
    if (ts > 1) {
      const long tail_per_cu = (tail * ts + 255) / 256;
      const double apart =
          launch + (double)((tiles - tail) / 256) * (start[c.v] + ktiles_all * per_ktile[c.v]) + 3.0 +
          tail_per_cu * (start[c.v] + (ktiles_all + ts - 1) / ts * per_ktile[c.v]) * (tail_per_cu == 1 ? lone[c.v] : 1.0) +
          join_start + ts * tail * tile_bytes / 1e6 * join_per_mb;
      if (apart < 0.95 * t) {
        t = apart;
        if (tail_split) *tail_split = ts;
      }
    }
  }
  // No faster than memory delivers: the blocks of a weight tile's column walk through all of
  // the activations, which come from memory once per column when they are too many to stay in
  // the memory-side cache (4096 rows of K = 36864: 302 MB, 36 columns of 128: 11 GB).
  const double a_mb = (double)M * K * 2.0 / 1e6, w_mb = (gated ? 2.0 : 1.0) * N * K * 2.0 / 1e6;
  const double traffic_mb = w_mb + a_mb * (a_mb > 128.0 ? (double)((N + ncols - 1) / ncols) : 1.0);
  const double memory = traffic_mb / 6.0;          // 6 TB/s
  return t > memory ? t : memory;
}

// Tiles that pass through registers (weights row by row, or K not whole stages): which block, how
// many ranges of K, of the last round's tiles.  (The figures are from before weights in strips had tiles of
// their own: layer shapes, whose weights are in strips, no longer come here.)
struct StagedCut {
  int variant, ksplit, tail_split;      // 0: 128 x 128, 1: 64 x 128, 2: 128 x 256, 3: 256 x 256
};
static StagedCut staged_cut(int M, int N, int K, bool gated, size_t room) {
  // 128 x 128 blocks of four waves (two share a CU) or 128 x 256 blocks of eight (one a CU,
  // about 1.2 times the rate).  What counts is the CU with the most blocks; a lone small block
  // runs at about 0.8 of the rate of two.  The constants are measured (M = 512 and 2048 with
  // N = 2304 to 18432): the rule picked the faster of the two in each of those.
  const int tiles_m = (M + 127) / 128;
  const long nb_small = (long)tiles_m * ((N + (gated ? 64 : 128) - 1) / (gated ? 64 : 128));
  const long nb_wide = (long)tiles_m * ((N + (gated ? 128 : 256) - 1) / (gated ? 128 : 256));
  const long per_cu_small = (nb_small + 255) / 256, per_cu_wide = (nb_wide + 255) / 256;
  const double cost_small = per_cu_small * 16384.0 / (per_cu_small == 1 ? 0.8 : 1.0);
  const double cost_wide = per_cu_wide * 32768.0 / 1.2;
  const bool wide = cost_wide < cost_small;
  const bool exact = K % GT_BK == 0;
  // Few small blocks: split K over blocks until about 320 blocks exist, a range no shorter than
  // 8 k tiles, and the partial sums (4 M N bytes a range, written and read) no more than W.
  auto ranges = [&](long blocks) {
    int ks = (int)(320 / blocks);
    ks = min(ks, (K + GT_BK - 1) / GT_BK / 8);
    ks = min(ks, K / (4 * M));
    return max(ks, 1);
  };
  int ksplit = (!wide && nb_small < 160) ? ranges(nb_small) : 1;
  // few rows and a K too short to split: 128 x 128 tiles leave half of the CUs or more without
  // a block; 64-row tiles make twice as many (they lose to a split of K where K allows one)
  const bool low = !wide && M > 64 && nb_small * ksplit <= 128;
  if (low) ksplit = ranges((long)((M + 63) / 64) * (nb_small / tiles_m));
  // 256 x 256 blocks of sixteen waves where there are tiles enough.  A 128 x 256 x 64 step moves 48 KB
  // into a CU for 4.2 MFLOP, a 256 x 256 block a third fewer bytes per flop.  Measured against 128 x 256: 0.88 of its
  // time with many rounds of tiles (4096 x 36864 x 4608 gated), 0.91 at 2048 x 9216 x 2304 gated
  // (2.25 rounds), 1.4 at 2048 x 4096 x 2304 (half a round: half of the CUs idle).  The rule:
  // time = (rounds, at least one, + 0.15) x time of a tile.
  int variant = wide ? 2 : low ? 1 : 0;       // 128 x 128, 64 x 128, 128 x 256, 256 x 256
  if (wide && exact) {
    const long nb_big = (long)((M + 255) / 256) * ((N + (gated ? 128 : 256) - 1) / (gated ? 128 : 256));
    auto rounds_cost = [](long nb, double unit) { return ((nb > 256 ? nb / 256.0 : 1.0) + 0.15) * unit; };
    if (rounds_cost(nb_big, 2.0 * 0.8836 * 32768.0 / 1.2) < rounds_cost(nb_wide, 32768.0 / 1.2)) variant = 3;
  }
  // The rules above are right for the shapes they were made on and miss elsewhere: long K with
  // few hundred rows wants more ranges of K than they allow, narrow products of thousands of
  // rows (N = 2304 to 4608) the 256 x 256 blocks.  So every variant and split is priced by a
  // model of its time fitted to a sweep of 1339 measured (rows, shape, variant, split)
  // combinations (2B, 9B and 27B layer shapes, 96 to 4096 rows; 10 % rms error), and the model's
  // choice replaces the rules' when it promises at least 12 % (with that margin it was never
  // more than 3 % slower than the rules on the sweep, and 5 % faster in the sum).
  {
    const TileChoice rule{variant, ksplit};
    const double rule_cost = tile_cost(rule, M, N, K, gated, room);
    TileChoice best = rule;
    double best_cost = rule_cost;
    static const int splits[] = {1, 2, 3, 4, 6, 8};
    for (int v = 0; v < (exact ? 4 : 3); v++)
      for (int ks : splits) {
        const TileChoice c{v, ks};
        const double t = tile_cost(c, M, N, K, gated, room);
        if (t < best_cost) { best = c; best_cost = t; }
      }
    if (best_cost * 1.12 < rule_cost) { variant = best.v; ksplit = best.ks; }
  }
  int tail_split = 1;
  tile_cost(TileChoice{variant, ksplit}, M, N, K, gated, room, &tail_split);
  return StagedCut{variant, ksplit, tail_split};
}

// The bytes of partial sums for which the static array (strict) refuses a product of tiles that pass
// through registers: 0, or more than the array holds.  As launch_tile has it.
static size_t staged_sums(int M, int N, int K, bool gated, const GemmWorkspace& wsp) {
  StagedCut c = staged_cut(M, N, K, gated, wsp.split_bytes());
  static const int BM[4] = {128, 64, 128, 256}, BN[4] = {128, 128, 256, 256};
  const int ncols = gated ? BN[c.variant] / 2 : BN[c.variant], round = c.variant <= 1 ? 512 : 256;
  const int tiles = ((M + BM[c.variant] - 1) / BM[c.variant]) * ((N + ncols - 1) / ncols), tail = tiles % round;
  const size_t tile = (size_t)BM[c.variant] * BN[c.variant] * sizeof(float);
  while (c.ksplit > 1 && tile * tiles * c.ksplit > wsp.split_bytes()) c.ksplit--;
  size_t need = c.ksplit > 1 ? tile * tiles * c.ksplit : 0;
  if (c.ksplit <= 1 && c.tail_split > 1 && tail > 0 && tiles > round && tile * tail * c.tail_split <= wsp.split_bytes())
    need = tile * tail * c.tail_split;
  return need > wsp.bytes ? need : 0;
}

static int gemm_bf16_run(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32,
                         int M, int N, int K, int epi, float cap, int w_strip, const GemmWorkspace& wsp,
                         int* parts, void* stream) {
  ZK_REQUIRE(M >= 0 && N > 0 && K > 0, "zk_gemm_bf16: bad sizes");
  ZK_REQUIRE(K % 8 == 0 && lda % 8 == 0, "zk_gemm_bf16: K and lda must be multiples of 8");
  ZK_REQUIRE(lda >= K && ldc >= N, "zk_gemm_bf16: leading dimensions too small");
  ZK_REQUIRE(epi >= 0 && epi <= EPI_GELU, "zk_gemm_bf16: unknown epilogue");
  ZK_REQUIRE((epi != EPI_SOFTCAP && epi != EPI_CLAMPED) || cap > 0.f, "zk_gemm_bf16: soft cap or clamp limit must be positive");
  ZK_REQUIRE(((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "zk_gemm_bf16: operands must be 16-byte aligned");
  const bool gated = epi == EPI_GELU_TANH || epi == EPI_SILU || epi == EPI_RELU || epi == EPI_CLAMPED;
  ZK_REQUIRE(!w_strip || (K % 32 == 0 && (!gated || N % 16 == 0)), "zk_gemm_bf16: strip layout needs K % 32 == 0 (and N % 16 == 0 when gated)");
  if (parts) *parts = 0;
  if (M == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (w_strip && M <= 64 && (M > 16 || mid_for_few(gated, N, K, parts != nullptr && joinable_by_reader(N, ldc, c_is_f32, epi)))) {
    return gated ? launch_mid<true>(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, wsp, parts, s)
                 : launch_mid<false>(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, wsp, parts, s);
  }
  if (M <= 64) {
    return gated ? launch_skinny<true>(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, wsp, parts, s)
                 : launch_skinny<false>(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, wsp, parts, s);
  }
  // more than 64 rows by weights in strips, K in whole stages (and offsets of a tile's rows that 31 bits hold)
  if (w_strip && K % 64 == 0 && lda <= (1 << 22)) {
    const bool aligned = wsp.ptr != nullptr && (uintptr_t)wsp.ptr % 16 == 0;
    const bool by_reader = parts != nullptr && joinable_by_reader(N, ldc, c_is_f32, epi);
    const TileCut cut = tile_cut(gated, by_reader, M, N, K, aligned ? wsp.split_bytes() : 0);
    // (what the static array is refused for stays what it was before the tiles had other shapes)
    if (wsp.strict)
      if (const size_t need = staged_sums(M, N, K, gated, wsp)) return wsp.too_small(need);
    const TileProduct p{A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap};
    return launch_cut(cut, gated, p, (float*)wsp.ptr, wsp.bytes, parts, s);
  }
  const bool exact = K % GT_BK == 0;
  const size_t room = (wsp.ptr != nullptr && (uintptr_t)wsp.ptr % 64 == 0) ? wsp.split_bytes() : 0;
  const StagedCut cut = staged_cut(M, N, K, gated, room);
  const int variant = cut.variant, ksplit = cut.ksplit, tail_split = cut.tail_split;
#define ZK_TILE_(W_, M_, N_, G_, E_) \
  launch_tile<W_, M_, N_, G_, E_>(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, wsp, ksplit, tail_split, s)
#define ZK_TILE(W_, M_, N_)                                                                            \
  (gated ? (exact ? ZK_TILE_(W_, M_, N_, true, true) : ZK_TILE_(W_, M_, N_, true, false))             \
         : (exact ? ZK_TILE_(W_, M_, N_, false, true) : ZK_TILE_(W_, M_, N_, false, false)))
  if (variant == 3) return gated ? ZK_TILE_(2, 4, 4, true, true) : ZK_TILE_(2, 4, 4, false, true);
  if (variant == 2) return ZK_TILE(2, 2, 4);
  if (variant == 1) return ZK_TILE(1, 2, 2);
  return ZK_TILE(2, 2, 2);
#undef ZK_TILE
#undef ZK_TILE_
}

// Which tile (its number in tile_shapes) and how many ranges of K, of the last round's tiles alone, a product of more
// than 64 rows by weights in strips, K a multiple of 64, takes with the standard workspace (``by_reader``: the caller
// passes ``parts``), and which tile the columns behind the whole rounds take (-1: the same).  For tests that mean to
// reach each of them.
extern "C" int zk_gemm_bf16_tile_cut(int gated, int by_reader, int M, int N, int K, int* shape, int* ks,
                                     int* tail_ks, int* rest) {
  ZK_REQUIRE(M > 64 && N > 0 && K > 0 && K % 64 == 0, "zk_gemm_bf16_tile_cut: no tile product of this size");
  const TileCut c = tile_cut(gated != 0, by_reader != 0, M, N, K, ZK_GEMM_WORKSPACE_BYTES);
  *shape = c.shape;
  *ks = c.ks;
  *tail_ks = c.tail_ks;
  *rest = c.rest;
  return 0;
}

// Whether a product of up to 64 rows by weights in strips takes the blocks of gemm_mid_kernel with this workspace, and how it is cut:
// strips a block, waves a strip, steps a chunk, ranges of K.  ``epi`` and ``by_reader`` as above.  For tests.
extern "C" int zk_gemm_bf16_mid_cut(int epi, int by_reader, int M, int N, int K, const void* ws, size_t ws_bytes, int* cut) {
  const bool gated = epi == EPI_GELU_TANH || epi == EPI_SILU || epi == EPI_RELU || epi == EPI_CLAMPED;
  if (M < 1 || M > 64 || (M <= 16 && !mid_for_few(gated, N, K, by_reader != 0))) return 0;
  const MidCut c = mid_cut_of_launch(gated, by_reader != 0, M, N, K, epi, GemmWorkspace{const_cast<void*>(ws), ws_bytes, false});
  cut[0] = c.spb;
  cut[1] = c.kw;
  cut[2] = c.ch;
  cut[3] = c.ksplit;
  return 1;
}

extern "C" int zk_gemm_bf16(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32,
                            int M, int N, int K, int epi, float cap, int w_strip, void* ws,
                            size_t ws_bytes, int* parts, void* stream) {
  ZK_REQUIRE(epi != EPI_PICK, "zk_gemm_bf16: the picking epilogue belongs to zk_head_pick_bf16");
  return gemm_bf16_run(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip, GemmWorkspace{ws, ws_bytes, false},
                       parts, stream);
}

// ---- the LM head of a greedy step: the largest logit's column of every row, no logits stored
//
// One block a row joins the strips' picks: larger value first, equal values to the lower
// column, NaN never; a row without any valid value gets column 0 (as zk_argmax does).
__global__ __launch_bounds__(1024) void pick_join_kernel(const Pick* __restrict__ picks, int nstrips,
                                                         int* __restrict__ ids) {
  __shared__ float sv[16];
  __shared__ int sc[16];
  const Pick* row = picks + (size_t)blockIdx.x * nstrips;
  Pick best{-INFINITY, 0x7fffffff};
  auto better = [](const Pick& a, const Pick& b) {       // a before b
    if (a.column == 0x7fffffff) return false;
    return b.column == 0x7fffffff || a.value > b.value || (a.value == b.value && a.column < b.column);
  };
  // eight loads of a thread on their way at a time (a place past the end reads the last pick
  // again, which changes nothing): with one block a row the time is the trips to memory
  for (int i0 = threadIdx.x; i0 < nstrips; i0 += 8 * 1024) {
    Pick p[8];
#pragma unroll
    for (int j = 0; j < 8; j++) p[j] = row[min(i0 + j * 1024, nstrips - 1)];
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (better(p[j], best)) best = p[j];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const Pick o{__shfl_xor(best.value, off), __shfl_xor(best.column, off)};
    if (better(o, best)) best = o;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sv[wave] = best.value;
    sc[wave] = best.column;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) {
      const Pick o{sv[w], sc[w]};
      if (better(o, best)) best = o;
    }
    ids[blockIdx.x] = best.column == 0x7fffffff ? 0 : best.column;
  }
}

extern "C" size_t zk_head_pick_bf16_workspace(int M, int N) {
  return (size_t)(M > 0 ? M : 0) * (size_t)((N + 15) / 16) * sizeof(Pick);
}

// ids[m] = the column of the largest value of row m of A W^T after the soft cap (cap <= 0: no
// cap): what zk_gemm_bf16 with the soft-cap epilogue followed by zk_argmax gives, bit for bit,
// without the [M, N] logits.  1 to 64 rows; more than 16 need W in strip layout.  ``picks``:
// zk_head_pick_bf16_workspace(M, N) bytes of scratch, 16-byte aligned.
extern "C" int zk_head_pick_bf16(const void* A, int lda, const void* W, int M, int N, int K, float cap, int w_strip,
                                 void* picks, size_t picks_bytes, void* ids, void* stream) {
  ZK_REQUIRE(M >= 1 && M <= 64, "zk_head_pick_bf16: 1 to 64 rows");
  ZK_REQUIRE(M <= 16 || w_strip, "zk_head_pick_bf16: more than 16 rows need the weights in strip layout");
  ZK_REQUIRE(picks != nullptr && (uintptr_t)picks % 16 == 0 && ids != nullptr, "zk_head_pick_bf16: no scratch or no result");
  ZK_REQUIRE(picks_bytes >= zk_head_pick_bf16_workspace(M, N), "zk_head_pick_bf16: scratch too small");
  if (int rc = gemm_bf16_run(A, lda, W, nullptr, N, 1, M, N, K, EPI_PICK, cap, w_strip,
                             GemmWorkspace{picks, picks_bytes, false}, nullptr, stream))
    return rc;
  pick_join_kernel<<<M, 1024, 0, (hipStream_t)stream>>>((const Pick*)picks, (N + 15) / 16, (int*)ids);
  return zk_launch_status("zk_head_pick_bf16");
}

// ---- the same product for callers that cannot allocate (declared in gemm_bf16_static.h)
//
// The partial sums of a product that splits K go to a statically allocated array instead of a
// workspace the caller brings.  Every GPU holds its own copy of the array at its own address;
// host code never uses the array's name as an address, only the pointer that
// hipGetSymbolAddress gave for the device that is current.
static __device__ __align__(256) unsigned char scratch[ZK_GEMM_STATIC_SCRATCH_BYTES];

#define ZK_MAX_DEVICES 64
static void* scratch_of_device[ZK_MAX_DEVICES];     // null until the device's set-up has run
static std::mutex scratch_mutex;

// The array's address on the current device, asked for once per device.
static int static_scratch(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return zk_fail("zk_gemm_bf16_static: no current device");
  ZK_REQUIRE(dev >= 0 && dev < ZK_MAX_DEVICES, "zk_gemm_bf16_static: device index out of range");
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_of_device[dev] == nullptr) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      return zk_fail("zk_gemm_bf16_static: hipGetSymbolAddress of the scratch array failed");
    }
    scratch_of_device[dev] = ptr;
  }
  *out = scratch_of_device[dev];
  return 0;
}

extern "C" size_t zk_gemm_bf16_static_bytes() { return ZK_GEMM_STATIC_SCRATCH_BYTES; }

extern "C" int zk_gemm_bf16_static_init() {
  void* ptr = nullptr;
  return static_scratch(&ptr);
}

extern "C" int zk_gemm_bf16_static(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32,
                                   int M, int N, int K, int epi, float cap, int w_strip, void* stream) {
  void* ptr = nullptr;
  if (int rc = static_scratch(&ptr)) return rc;
  // strict: K is split exactly as zk_gemm_bf16 splits it with its standard workspace, so the
  // results have the same bits; a split whose partial sums do not fit the array is refused.
  // Nothing in the array has to start at zero: each range's plane is written in full by the
  // product kernel before the joining kernel of the same call reads it.
  ZK_REQUIRE(epi != EPI_PICK, "zk_gemm_bf16_static: the picking epilogue belongs to zk_head_pick_bf16");
  return gemm_bf16_run(A, lda, W, C, ldc, c_is_f32, M, N, K, epi, cap, w_strip,
                       GemmWorkspace{ptr, ZK_GEMM_STATIC_SCRATCH_BYTES, true}, nullptr, stream);
}

#endif  // ZSE_ACT_BF16
