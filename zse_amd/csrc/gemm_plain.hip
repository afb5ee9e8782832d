// Plain matrix product C[M,N] = A[M,K] * W[N,K]^T with float accumulation and no reduced
// precision: the 32-bit path's product and, in the bf16 library, the twin that the tuned
// kernels are checked against.  Weights are [out, in] row-major as in the reference
// (orchestrator/kernels.py:1075-1126, a 32x32 shared-memory tile per block).  The sum over K
// runs in a fixed order for every output element, whatever M is, so a row's result does not
// depend on which other rows are in the batch.
#include "common.h"

#include <algorithm>
#include <cmath>

#if ZSE_ACT_BF16
#define GP_BM 64
#define GP_BN 64
#define GP_BK 16

template <typename TA, typename TC>
__global__ __launch_bounds__(256) void gemm_plain_kernel(const TA* __restrict__ A, int lda,
                                                         const TA* __restrict__ W,
                                                         TC* __restrict__ C, int ldc, int M, int N,
                                                         int K) {
  __shared__ float sA[GP_BK][GP_BM + 1];
  __shared__ float sW[GP_BK][GP_BN + 1];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * GP_BM, n0 = blockIdx.x * GP_BN;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += GP_BK) {
    for (int i = threadIdx.x; i < GP_BM * GP_BK; i += 256) {
      const int r = i / GP_BK, c = i % GP_BK;
      const int m = m0 + r, n = n0 + r, k = k0 + c;
      sA[c][r] = (m < M && k < K) ? to_f32(A[(size_t)m * lda + k]) : 0.f;
      sW[c][r] = (n < N && k < K) ? to_f32(W[(size_t)n * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GP_BK; kk++) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) a[i] = sA[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; j++) b[j] = sW[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int n = n0 + tx * 4 + j;
      if (n < N) C[(size_t)m * ldc + n] = from_f32<TC>(acc[i][j]);
    }
  }
}

#else

// The 32-bit product on the 32-bit matrix cores (16x16x4, float in, float out).
//
// A block owns 16 MF x 16 NF of C and its waves, eight of them, share K out: wave w takes the 32-wide
// steps w, w + 8, .., every wave the whole tile, and their sums meet in LDS, (w, w + 4), then
// (w, w + 2), then (w, w + 1).  So the order of a sum follows from K alone and the tile may
// follow from M and N.  Operands come straight from memory: in a 16-wide piece of K the four
// products take k = 4 (lane / 16) + e, e = 0..3, from both sides, so a lane's float4 of a row
// is its operand of four products and a load takes 64-byte runs of sixteen rows.  A product is
// 32 cycles long, a load of 16 bytes a lane 16: at 4 x 4 pieces the matrix cores are the bound,
// below that L2 (a 2 x 2 tile reads twice the bytes per flop).
//
// Measured (us; before: 64 x 64 tiles of scalar multiply-adds through LDS, one block a tile):
//   M = 303: 1024 x 4096 and 1024 x 1024 (average)  452 -> 42;  8192 x 1024  217 -> 87;
//   1536 x 1024  191 -> 20;  M = 4: 32768 x 1024  207 -> 28.  By f32_tile's choice: 1024 x 4096 61 -> 41, 1024 x 1024
//   18.7 -> 14.2, 8192 x 1024 86 -> 67, 1536 x 1024 19.3 -> 17.2.
// The error against 64 bits is no larger than the scalar sum's (eight shorter sums added up).
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef f32x4 f32x4_any __attribute__((aligned(4)));       // the loads take any float's address

// HOW: 3: K is a whole number of steps; 2: a multiple of four; 1: four or more; 0: fewer, every value is
// loaded on its own.  The loads of the next H pieces of a wave's run are on their way while the
// current ones are multiplied, so nothing may look at them before: with HOW = 1 and 2 what lies
// behind K is set to zero right before it is multiplied.  (2048 x 5000 x 200: 84 us with 2, 99 with 1;
// 2048 x 4096 x 1023: 253 with 1, 390 value by value.)
// WAVES: 8, or 1 or 2 where K has no more steps (waves without a step would bring zeros, so the sum
// is the same): 2048 x 5000 with K = 16 53 -> 21 us, with K = 64 52 -> 27; scalar multiply-adds took 25 and 44.
template <int MF, int NF, int H, int AHEAD, int HOW, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gemm_f32_kernel(const float* __restrict__ A, int lda,
                                                              const float* __restrict__ W,
                                                              float* __restrict__ C, int ldc, int M, int N,
                                                              int K, int tiles_m, int tiles_n) {
  __shared__ f32x4 part[WAVES > 1 ? WAVES / 2 : 1][MF * NF][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  // the blocks that share a strip of W run on one XCD, one after the other (ids go round-robin over 8)
  int id = blockIdx.x;
  const int total = tiles_m * tiles_n;
  if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
  const int m0 = id % tiles_m * (16 * MF), n0 = id / tiles_m * (16 * NF);
  const float* ap[MF];
  const float* wp[NF];
#pragma unroll
  for (int i = 0; i < MF; i++) ap[i] = A + (size_t)min(m0 + 16 * i + r, M - 1) * lda;
#pragma unroll
  for (int j = 0; j < NF; j++) wp[j] = W + (size_t)min(n0 + 16 * j + r, N - 1) * K;
  const int steps = (K + 31) / 32;

  auto piece = [&](const float* row, int k) {
    f32x4 v;
    if (HOW == 3) {
      v = *(const f32x4_any*)(row + k);
    } else if (HOW > 0) {       // the last four values where the piece reaches past them
      v = *(const f32x4_any*)(row + min(k, K - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = k + e < K ? row[k + e] : 0.f;
    }
    return v;
  };
  // The wave's run, counted in units of H pieces of 16: two pieces make one of its 32-wide
  // steps.  (A unit past the last reads inside the matrix again and is not multiplied: no load
  // is under a condition.)
  const int units = (steps - wave + WAVES - 1) / WAVES * (2 / H);
  auto fetch = [&](int u, f32x4 (&af)[MF][H], f32x4 (&wf)[NF][H]) {
    const int p = min(u, units - 1) * H;
    const int k = (wave + p / 2 * WAVES) * 32 + p % 2 * 16 + 4 * q;
#pragma unroll
    for (int h = 0; h < H; h++) {
#pragma unroll
      for (int i = 0; i < MF; i++) af[i][h] = piece(ap[i], k + 16 * h);
#pragma unroll
      for (int j = 0; j < NF; j++) wf[j][h] = piece(wp[j], k + 16 * h);
    }
  };
  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; i++)
#pragma unroll
    for (int j = 0; j < NF; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // W is the first operand: a lane then holds columns 4 q + 0..3 of row r of C
  auto multiply = [&](int u, f32x4 (&a)[MF][H], f32x4 (&w)[NF][H]) {
    if (HOW == 1 || HOW == 2) {
#pragma unroll
      for (int h = 0; h < H; h++) {
        const int p = u * H + h;
        const int over = (wave + p / 2 * WAVES) * 32 + p % 2 * 16 + 4 * q + 4 - K;       // values of the piece behind K
        if (over <= 0) continue;
        auto cut = [&](f32x4& v) {         // what was loaded are the row's last four values
          if (HOW == 2) v = f32x4{0.f, 0.f, 0.f, 0.f};       // all of them belong to the piece before
          else
            v = f32x4{over == 1 ? v[1] : over == 2 ? v[2] : over == 3 ? v[3] : 0.f,
                      over == 1 ? v[2] : over == 2 ? v[3] : 0.f, over == 1 ? v[3] : 0.f, 0.f};
        };
#pragma unroll
        for (int i = 0; i < MF; i++) cut(a[i][h]);
#pragma unroll
        for (int j = 0; j < NF; j++) cut(w[j][h]);
      }
    }
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < MF; i++)
#pragma unroll
          for (int j = 0; j < NF; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][h][e], a[i][h][e], acc[i][j], 0, 0, 0);
  };
  // Unit u lies in register set u % AHEAD; the loads of the next AHEAD - 1 units are on their
  // way.  (No branch lies between a load and its product inside the loop: the load would be
  // sunk behind it.)
  f32x4 a[AHEAD][MF][H], w[AHEAD][NF][H];
  if (wave < steps) {
#pragma unroll
    for (int t = 0; t < AHEAD - 1; t++) fetch(t, a[t], w[t]);
    int u = 0;
    for (; u + AHEAD <= units; u += AHEAD) {
#pragma unroll
      for (int t = 0; t < AHEAD; t++) {
        fetch(u + t + AHEAD - 1, a[(t + AHEAD - 1) % AHEAD], w[(t + AHEAD - 1) % AHEAD]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(u + t, a[t], w[t]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int t = 0; t < AHEAD - 1; t++)
      if (u + t < units) multiply(u + t, a[t], w[t]);
  }
#pragma unroll
  for (int half = WAVES / 2; half > 0; half /= 2) {
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++) part[wave - half][i * NF + j][lane] = acc[i][j];
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int i = 0; i < MF; i++)
#pragma unroll
        for (int j = 0; j < NF; j++) acc[i][j] += part[wave][i * NF + j][lane];
    }
    __syncthreads();
  }
  if (wave > 0) return;
  const bool whole = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
#pragma unroll
  for (int i = 0; i < MF; i++) {
    const int m = m0 + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NF; j++) {
      const int n = n0 + 16 * j + 4 * q;
      float* dst = C + (size_t)m * ldc + n;
      if (whole && n + 4 <= N) *(f32x4*)dst = acc[i][j];
      else
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < N) dst[e] = acc[i][j][e];
    }
  }
}

// LONG: K of 512 or more only.  STEPS: K in whole steps of 32 only.
template <int MF, int NF, int H, int AHEAD, bool LONG = false, bool STEPS = false>
static int launch_f32(const float* A, int lda, const float* W, float* C, int ldc, int M, int N, int K,
                      hipStream_t s) {
  const int tiles_m = (M + 16 * MF - 1) / (16 * MF);
  auto kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 3, 8>;
  if constexpr (!STEPS) {
    if (K % 4) kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 1, 8>;
    else if (K % 32) kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 2, 8>;
  }
  if constexpr (!LONG) {
    if (K < 4) kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 0, 1>;
    else if (K <= 32) kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 1, 1>;
    else if (K <= 64) kernel = gemm_f32_kernel<MF, NF, H, AHEAD, 1, 2>;
  }
  const int waves = K <= 32 ? 1 : K <= 64 ? 2 : 8;
  // a launch of 2^32 threads or more would run its low 32 bits only: columns are taken 2^22 tiles at a time
  const long long most = (long long)std::max((1 << 22) / tiles_m, 1) * (16 * NF);
  for (long long n = 0; n < N; n += most) {
    const int cols = (int)std::min(most, N - n), tiles_n = (cols + 16 * NF - 1) / (16 * NF);
    kernel<<<dim3(tiles_m * tiles_n), 64 * waves, 0, s>>>(A, lda, W + n * K, C + n, ldc, M, cols, K, tiles_m, tiles_n);
  }
  return zk_launch_status("zk_gemm_plain");
}

// More than sixteen rows, K of 512 or more: the tile with the least price.  A launch takes as many rounds as the CU
// with the most blocks has, whatever a block's registers would allow (303 x 1024 x 4096: 320 blocks of 32 x 32 61 us, 224 of
// 48 x 32 41): a block alone already takes what its CU gets from its L2.  Microseconds, fitted to 17 to 2,048
// rows by thirteen weights (512 to 18,432 columns, K of 1,024 to 9,216; the last two to 17 to 2,048 rows of 512 to
// 32,768 columns, K of 512 to 9,216): a round's start, and for every 1,024 of K one round's time and that of several.  The
// tile it names takes 1.009 times the best one's time in the mean and 0.81 of that of 32 x 32 and 64 x 64 alone, 0.98
// times the old rule's speed at the least.  The last two fill rounds that the others leave half empty (us, without and with
// them: 303 x 8192 x 1024, 640 blocks of 64 x 64 or 512 of 80 x 64, 77.6 and 66.9; 150 rows 45 and 36;
// 64 x 8192 x 1024, 256 blocks of 64 x 32, 20.8 and 18.3; 303 x 1536 x 1024 19.6 and 17.2), but for K in whole steps of
// 32 only: else they keep a part of what they work on in scratch memory (128 x 18432 x 520 36.8 and 58.4, 64 x 8192 x 1000 17.3 and
// 22.3, 303 x 18432 x 514 122 and 137).  64 x 32 up to K = 2,560 (256 x 2048 x 4096 62.9 by 32 x 32 and 66.4), the price of 80 x 64 with
// 3 % on top: over some 450 shapes at which the choice then differs from the other tiles' it is 1.02 times their best at the most, 0.89 in the mean.
// The sums are the same bits.  (``longest``: 0, or the longest K, in whole steps.)
struct F32Tile { int mf, nf; double start, lone, several; int longest; };
static const F32Tile f32_tiles[] = {
    {1, 1, 0.88, 3.65, 3.47, 0},
    {1, 2, 1.39, 5.45, 5.16, 0},
    {2, 2, 0.74, 8.06, 7.45, 0},
    {3, 2, 2.54, 8.66, 8.68, 0},
    {2, 3, 2.71, 8.94, 8.55, 0},
    {3, 4, 0.00, 22.29, 21.65, 0},
    {4, 4, 2.23, 23.23, 22.63, 0},
    {4, 2, 2.28, 11.92, 14.20, 2560},
    {5, 4, 7.54, 25.33, 25.27, 1 << 30}};
static int f32_tile(int M, int N, int K) {
  int best = 0;
  double best_time = 1e30;
  const double t_mem = ((double)N * K + (double)M * K + (double)M * N) * 4e-6 / 5.0;
  for (int i = 0; i < (int)(sizeof(f32_tiles) / sizeof(f32_tiles[0])); i++) {
    const F32Tile& t = f32_tiles[i];
    if (t.longest && (K % 32 || K > t.longest)) continue;
    const long blocks = (long)((M + 16 * t.mf - 1) / (16 * t.mf)) * ((N + 16 * t.nf - 1) / (16 * t.nf)), rounds = (blocks + 255) / 256;
    const double work = rounds * (t.start + (rounds == 1 ? t.lone : t.several) * K / 1024.0);
    const double time = sqrt(sqrt(work * work * work * work + t_mem * t_mem * t_mem * t_mem));
    if (time < best_time) best = i, best_time = time;
  }
  return best;
}

// The tile's rows and columns; for tests.
extern "C" int zk_gemm_plain_tile(int M, int N, int K, int* rows, int* columns) {
  if (M <= 16 || N <= 0 || K < 512) return 0;
  const F32Tile& t = f32_tiles[f32_tile(M, N, K)];
  *rows = 16 * t.mf;
  *columns = 16 * t.nf;
  return 1;
}
#endif  // ZSE_ACT_BF16

extern "C" int zk_gemm_plain(const void* A, int lda, const void* W, void* C, int ldc, int c_is_f32,
                             int M, int N, int K, void* stream) {
  ZK_REQUIRE(M >= 0 && N > 0 && K > 0, "zk_gemm_plain: bad sizes");
  ZK_REQUIRE(lda >= K && ldc >= N, "zk_gemm_plain: leading dimensions too small");
  if (M == 0) return 0;
  ZK_REQUIRE((M + 63) / 64 <= 65535, "zk_gemm_plain: too many rows");
  hipStream_t s = (hipStream_t)stream;
#if ZSE_ACT_BF16
  dim3 grid((N + GP_BN - 1) / GP_BN, (M + GP_BM - 1) / GP_BM);
  if (c_is_f32)
    gemm_plain_kernel<act_t, float><<<grid, 256, 0, s>>>((const act_t*)A, lda, (const act_t*)W,
                                                         (float*)C, ldc, M, N, K);
  else
    gemm_plain_kernel<act_t, act_t><<<grid, 256, 0, s>>>((const act_t*)A, lda, (const act_t*)W,
                                                         (act_t*)C, ldc, M, N, K);
  return zk_launch_status("zk_gemm_plain");
#else
  // Few rows or a short K: 64 x 64 where the CUs then work through four rounds of blocks or more (2048 x 8192 x 1024:
  // 433 us against 459 with 32 x 32, but 303 x 8192 x 1024, 2.5 rounds: 83 against 77), 32 x 32
  // otherwise; up to sixteen rows two strips of sixteen columns where every CU then has two
  // blocks (4 x 32768 x 1024: 21.5 against 24.0 us), one where it has not (1 x 1024 x 4096: 10.8
  // against 18.1).
  auto blocks = [&](int mf, int nf) { return (long)((M + 16 * mf - 1) / (16 * mf)) * ((N + 16 * nf - 1) / (16 * nf)); };
  const float *a = (const float*)A, *w = (const float*)W;
  if (M > 16 && K >= 512) {
    switch (f32_tile(M, N, K)) {
      case 0: return launch_f32<1, 1, 2, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 1: return launch_f32<1, 2, 2, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 2: return launch_f32<2, 2, 1, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 3: return launch_f32<3, 2, 2, 2, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 4: return launch_f32<2, 3, 2, 2, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 5: return launch_f32<3, 4, 2, 2, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 6: return launch_f32<4, 4, 2, 2, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
      case 7: return launch_f32<4, 2, 2, 2, true, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
      default: return launch_f32<5, 4, 2, 2, true, true>(a, lda, w, (float*)C, ldc, M, N, K, s);
    }
  }
  if (M > 16 && blocks(4, 4) >= 1024) return launch_f32<4, 4, 1, 3>(a, lda, w, (float*)C, ldc, M, N, K, s);
  if (M > 16) return launch_f32<2, 2, 1, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
  if (blocks(1, 2) >= 512) return launch_f32<1, 2, 2, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
  return launch_f32<1, 1, 2, 2>(a, lda, w, (float*)C, ldc, M, N, K, s);
#endif
}
