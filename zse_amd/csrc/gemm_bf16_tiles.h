// The tile product of more than 64 rows by weights in the strip layout (included by
// gemm_bf16.hip, which defines the epilogues): one kernel over wave tiles of TM x TN squares of
// 32 x 32, the launcher, and the joining kernel of tiles whose K was split.
#pragma once

#define ZK_LDS_AS __attribute__((address_space(3)))

// How the tiles of a launch are dealt to blocks.  The first ``whole`` tiles in K ranges
// ``ks``, and ``tail`` tiles from the ``from``-th on (a last round that would leave most CUs idle) in
// ``tail_ks`` ranges, all in one grid.  ``gm``: rows of tiles of a group (tile_at).  ``col0``, ``cols``: the
// launch's columns.
struct TileGrid {
  int tiles_m, tiles_n, gm, whole, ks, from, tail, tail_ks, col0, cols;
};

// Blocks go round-robin over the 8 XCDs by their number; this gives each XCD a run of
// neighbouring places instead.
__device__ __forceinline__ int xcd_run(int id, int total) {
  const int x = id % 8, q = total / 8, r = total % 8;
  return x * q + min(x, r) + id / 8;
}

// Places in groups of gm rows of tiles, column by column inside a group.  What an XCD works
// on at a time is then near a square of gm x (blocks / gm) tiles, which needs the fewest
// distinct rows and columns through its L2.  (Whole columns instead of groups, 4096 x 4096 x
// 16384 with 16 rows of tiles: 571 us; groups of 8, 6, 4, 2: 429, 425, 424, 432; the library
// product of the same process: 367.)
__device__ __forceinline__ void tile_at(int place, const TileGrid& g, int& tm, int& tn) {
  const int group = place / (g.gm * g.tiles_n), in = place - group * g.gm * g.tiles_n;
  const int rows = min(g.gm, g.tiles_m - group * g.gm);
  tn = in / rows;
  tm = group * g.gm + in % rows;
}

// The order in which a half of a stage is issued: a product, then an LDS read, for each of the
// NR reads; a product, then a copy, for each of the NL copies; the products that are left.  A
// 32 x 32 x 16 product keeps the matrix unit busy for 32 cycles, so what stands between two of
// them costs nothing; issued in a row in front of the products (as the compiler would), the
// reads and copies left the matrix unit idle for their length.
template <int R, int NR, int NM, int NL>
__device__ __forceinline__ void interleave() {
  if constexpr (R < NR + NL) {
    constexpr int T = NR + NL;
    constexpr int m = T <= NM ? 1 : (R + 1) * NM / T - R * NM / T;
    if constexpr (m > 0) __builtin_amdgcn_sched_group_barrier(0x008, m, 0);       // products
    __builtin_amdgcn_sched_group_barrier(R < NR ? 0x100 : 0x020, 1, 0);           // an LDS read, a copy
    interleave<R + 1, NR, NM, NL>();
  } else if constexpr (NM > NR + NL) {
    __builtin_amdgcn_sched_group_barrier(0x008, NM - NR - NL, 0);
  }
}

// Block tile (32 TM NWM) x (32 TN NWN), NWM x NWN waves; NSA stages of A and NSB of W, 64 k values
// each, in LDS; MB blocks a CU.  Operands are copied from memory straight into LDS (16 bytes a
// lane, no registers hold a tile on its way).  A block meets once a stage; a wave reads the operands
// of the next 16 k while it multiplies the present ones, also right after that meeting.
//
// In stage s the copies of A's stage s + NSA - 1 and then of W's stage s + NSB - 1 are issued, into the
// buffers of stage s - 1.  A wave waits before a meeting for its own copies of stage s + 1 and for its own
// reads of stage s; the meeting then says that every wave's copies are there and that nobody
// reads the buffers that the next copies go to.  The meeting stands behind the first half of the last 16 k's products,
// whose operands have come back by then, and the other half goes on beside the first reads of stage s + 1
// (before all of them, behind a quarter, half, three quarters, all: 1, 0.998, 0.989 to 0.994, 0.991, 0.996 of the time in the mean
// over 96 products of 80 to 2,048 rows).  W, which comes from memory, may be further ahead than A, which the L2s or the
// memory-side cache hold: 256 x 256 tiles have room for two stages and three.
//
// What bounds it: the way from memory to the L2s (hence tile_at) and from the L2s into the CUs, where
// half a line costs as much as a whole one.  Stages of 32 k, whose copies of A are 64-byte
// pieces of a row, ran at 0.29 us a step of 128 x 128 x 32 whether one or two blocks shared the CU; with the 128-byte
// pieces of 64 k 2048 x 4096 x 2304 takes 36.9 us instead of 41.5 (tiles of 128 x 256) and 535 x 2304 x 9216 in four
// ranges 32.9 instead of 41.4.  Many full rounds of 256 x 256 tiles reach 1.2 to 1.35 PFLOP/s
// (4096 x 4096 x 16384 in 412 us; the library product 367 to 425 from one process to the next).  In the two whole rounds of
// 2048 x (2 x 9216) x 2304 a CU's matrix units are busy for 0.75 of its cycles, at 1.6 GHz of 2.4.
//
// LDS: W's strips lie as in memory, 1 KB for 32 k: [k piece of 8][row 16][8 values]; an operand
// read (row lane % 32, k piece lane / 32) takes whole 256-byte runs.  A: a copy takes 8 rows x
// 64 k, eight lanes a row; lane c of a row fetches k piece c ^ (row / 2 % 8), so that of the sixteen
// rows that a read takes at once no two lie in the same banks.
//
// The products are taken as W tile x A tile^T: a lane holds, of row lane % 32 of a square, the
// columns 8 b + 4 (lane / 32) + e.  GATED: the first TN / 2 squares of a wave are gate columns,
// the others the same columns of up.
template <int TM, int TN, int NWM, int NWN, int NSA, int NSB, int MB, bool GATED>
__global__ __launch_bounds__(64 * NWM * NWN, MB) void gemm_tile_direct_kernel(
    const __bf16* __restrict__ A, int lda, const __bf16* __restrict__ W, void* __restrict__ C, int ldc,
    int c_is_f32, int M, int N, int K, int epi, float cap, float* __restrict__ partials, TileGrid g) {
  // (the host's pass knows no buffer descriptors)
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = 32 * TM * NWM, BN = 32 * TN * NWN, NW = NWM * NWN;
  constexpr int CA = BM / 8, CB = BN / 8;                               // 1 KB pieces of a stage
  constexpr int LPA = (CA + NW - 1) / NW, LPB = (CB + NW - 1) / NW;     // a wave's (the last may be copied twice)
  constexpr int SA = CA * 1024, SB = CB * 1024, WBASE = NSA * SA;       // bytes of a stage; W's place behind A's
  constexpr int OC = GATED ? BN / 2 : BN, NG = GATED ? 2 : 1;           // output columns
  static_assert(NSA >= 2 && NSA <= NSB, "W is as far ahead as A or further");
  static_assert(!GATED || TN % 2 == 0, "gate and up columns are paired inside a wave");
  extern __shared__ __align__(16) unsigned char gd_lds[];
  const int first = g.whole * g.ks;
  const bool tail = (int)blockIdx.x >= first;
  const int ks = tail ? g.tail_ks : g.ks, part_tiles = tail ? g.tail : g.whole;
  const int place = tail ? xcd_run(blockIdx.x - first, part_tiles * ks) : xcd_run(blockIdx.x, first);
  const int range = place / part_tiles;
  const int tile = place - range * part_tiles + (tail ? g.from : 0);
  int tm, tn;
  tile_at(tile, g, tm, tn);
  const int m0 = tm * BM, n0 = g.col0 + tn * OC;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NWN, wn = wave % NWN;
  const int lr = lane & 31, lk = lane >> 5;
  const int kstages = K / 64;
  const int k0 = (int)((long)range * kstages / ks), ns = (int)((long)(range + 1) * kstages / ks) - k0;
  // Copies.  A: one descriptor, a byte offset a piece and lane; W: a descriptor a piece.  Rows
  // past M and strips past the end read the last ones again; their results are not stored.
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)(A + (size_t)m0 * lda + (size_t)k0 * 64), 0, 0x7fffffff, 0x00027000);
  __amdgpu_buffer_rsrc_t rw[LPB];
  int va[LPA], la[LPA], lw[LPB];
#pragma unroll
  for (int c = 0; c < LPA; c++) {
    const int piece = min(wave + c * NW, CA - 1), row = piece * 8 + (lane >> 3);
    la[c] = piece * 1024;
    va[c] = (min(m0 + row, M - 1) - m0) * lda * 2 + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
  }
#pragma unroll
  for (int c = 0; c < LPB; c++) {
    const int piece = min(wave + c * NW, CB - 1), at = piece >> 1;       // two pieces a strip
    lw[c] = WBASE + piece * 1024;
    const int strips = (N + 15) / 16;
    int strip;
    if (GATED) strip = at < BN / 32 ? min(n0 / 16 + at, strips - 1) : strips + min(n0 / 16 + at - BN / 32, strips - 1);
    else strip = min(n0 / 16 + at, strips - 1);
    rw[c] = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (((size_t)strip * kstages + k0) * 2 + (piece & 1)) * 512), 0, 0x7fffffff, 0x00027000);
  }
  const int vw = lane * 16;
  // a stage past the end: the last one again, into a buffer nobody reads
  auto copy_a = [&](int buf, int stage) {
    stage = min(stage, ns - 1);
#pragma unroll
    for (int c = 0; c < LPA; c++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (ZK_LDS_AS void*)(gd_lds + buf + la[c]), 16, va[c], stage * 128, 0, 0);
  };
  auto copy_w = [&](int buf, int stage) {
    stage = min(stage, ns - 1);
#pragma unroll
    for (int c = 0; c < LPB; c++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw[c], (ZK_LDS_AS void*)(gd_lds + buf + lw[c]), 16, vw, stage * 2048, 0, 0);
  };
  int a_at[4];
#pragma unroll
  for (int q = 0; q < 4; q++) a_at[q] = (wm * (32 * TM) + lr) * 128 + (((q * 2 + lk) ^ ((lr >> 1) & 7)) * 16);
  const int w_at = WBASE + (wn * (GATED ? TN / 2 : TN) * 2 + (lr >> 4)) * 2048 + lk * 256 + (lr & 15) * 16;
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
  bf16x8 fa[2][TM], fb[2][TN];
  auto read = [&](int buf_a, int buf_w, int q) {
#pragma unroll
    for (int i = 0; i < TM; i++) fa[q & 1][i] = *(const bf16x8*)(gd_lds + buf_a + a_at[q] + i * 4096);
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int at = GATED && j >= TN / 2 ? (BN / 32) * 2048 + (j - TN / 2) * 4096 : j * 4096;
      fb[q & 1][j] = *(const bf16x8*)(gd_lds + buf_w + w_at + q * 512 + at);
    }
  };
  constexpr int NM = TM * TN, NR = TM + TN;
  auto products = [&](int q, int from, int to) {
#pragma unroll
    for (int x = 0; x < NM; x++)
      if (x >= from && x < to)
        acc[x / TN][x % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[q][x % TN], fa[q][x / TN], acc[x / TN][x % TN], 0, 0, 0);
  };
  // copies in flight that the wait of a meeting leaves: those issued after A's of stage s + 1
  constexpr int LEFT = (NSA - 2) * (LPA + LPB) + (NSB > NSA ? LPB : 0);
  // the copies that stages -(NSB - 1) .. -1 would have issued
#pragma unroll
  for (int t = 1 - NSB; t < 0; t++) {
    if (t + NSA - 1 >= 0) copy_a((t + NSA - 1) * SA, t + NSA - 1);
    __builtin_amdgcn_sched_barrier(0);          // the wait below counts on this order
    copy_w((t + NSB - 1) * SB, t + NSB - 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  // (the barrier as text: before one it knows, the compiler waits for every load in flight)
#define ZK_TILE_MEET() asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory")
  ZK_TILE_MEET();
  read(0, 0, 0);
  int ba = 0, bw = 0;
  for (int s = 0; s < ns; s++) {
    const int next_a = ba + SA == NSA * SA ? 0 : ba + SA, before_a = ba == 0 ? (NSA - 1) * SA : ba - SA;
    const int next_w = bw + SB == NSB * SB ? 0 : bw + SB, before_w = bw == 0 ? (NSB - 1) * SB : bw - SB;
    __builtin_amdgcn_sched_barrier(0);
    products(0, 0, NM);
    read(ba, bw, 1);
    copy_a(before_a, s + NSA - 1);
    interleave<0, NR, NM, LPA>();
    __builtin_amdgcn_sched_barrier(0);
    products(1, 0, NM);
    read(ba, bw, 2);
    copy_w(before_w, s + NSB - 1);
    interleave<0, NR, NM, LPB>();
    __builtin_amdgcn_sched_barrier(0);
    products(0, 0, NM);
    read(ba, bw, 3);
    interleave<0, NR, NM, 0>();
    __builtin_amdgcn_sched_barrier(0);
    products(1, 0, NM / 2);
    __builtin_amdgcn_sched_barrier(0);
    ZK_TILE_MEET();
    products(1, NM / 2, NM);
    read(next_a, next_w, 0);
    interleave<0, NR, NM - NM / 2, 0>();
    __builtin_amdgcn_sched_barrier(0);
    ba = next_a;
    bw = next_w;
  }
#undef ZK_TILE_MEET
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                              // the buffers are free for the results' way out
  const int wc = wn * (GATED ? TN / 2 : TN) * 32;        // the wave's first column in the tile
  if (ks > 1) {
    // The range's partial sums in planes (range, gate or up).  Every tile split: planes of [M, the launch's
    // columns rounded up to 16]; the tail alone: of [tail tile, BM, OC].
    const int npad = (g.cols + 15) / 16 * 16, ld = tail ? OC : npad;
    const size_t plane = tail ? (size_t)g.tail * BM * OC : (size_t)M * npad;
    float* mine = partials + (size_t)range * NG * plane +
                  (tail ? (size_t)(tile - g.from) * BM * OC : (size_t)m0 * npad + n0 - g.col0);
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int row = wm * 32 * TM + i * 32 + lr;
      if (m0 + row >= M) continue;
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int gate = GATED && j >= TN / 2 ? 1 : 0, col = wc + (j - gate * (TN / 2)) * 32 + 4 * lk;
#pragma unroll
        for (int b = 0; b < 4; b++)
          if (tail || n0 - g.col0 + col + 8 * b < npad)
            *(f32x4*)(mine + gate * plane + (size_t)row * ld + col + 8 * b) =
                f32x4{acc[i][j][4 * b], acc[i][j][4 * b + 1], acc[i][j][4 * b + 2], acc[i][j][4 * b + 3]};
      }
    }
    return;
  }
  constexpr int COLS = GATED ? 16 * TN : 32 * TN, TS = GATED ? TN / 2 : TN;      // columns, squares a wave stores
  // Rows of whole 16-byte pieces of a 16-bit C leave through LDS, 32 rows of the wave at a time,
  // 16 bytes a lane (a last row of tiles that stored two bytes a lane set the time of a launch of one round:
  // 708 x 3072 x 2048 36.7 -> 25.9 us).
  const bool whole_pieces = !c_is_f32 && N % 8 == 0 && ldc % 8 == 0 && (uintptr_t)C % 16 == 0;
  auto store_rows = [&](auto value) {
    constexpr int SLD = COLS + 8, PPR = COLS / 8;
    static_assert(NW * 32 * SLD * 2 <= NSA * SA + NSB * SB, "no room for the results' way out");
    __bf16* stage = (__bf16*)gd_lds + (size_t)wave * 32 * SLD;
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int j = 0; j < TS; j++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
          float x[4];
#pragma unroll
          for (int e = 0; e < 4; e++) x[e] = value(acc[i][j][4 * b + e], acc[i][GATED ? j + TS : j][4 * b + e]);
          store4(stage + lr * SLD + j * 32 + 8 * b + 4 * lk, x);
        }
      // the wave reads what its other lanes wrote: LDS takes a wave's accesses in order
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int p0 = 0; p0 < 32 * PPR; p0 += 64) {
        const int p = p0 + lane, row = p / PPR, col = (p % PPR) * 8;
        const int m = m0 + wm * 32 * TM + i * 32 + row, n = n0 + wc + col;
        if (m < M && n < N) *(bf16x8*)((__bf16*)C + (size_t)m * ldc + n) = *(const bf16x8*)(stage + row * SLD + col);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };
  // The epilogues of a few instructions have an unrolled copy each.  All of them behind one
  // choice per element, tanh and erf among them, made the way out 10 to 20 us of instruction
  // fetches (2048 x 2304 x 2048 in tiles of 192 x 128: 38 us, of which the products are 20).
  if (whole_pieces && !GATED && epi == EPI_NONE) return store_rows([](float x, float) { return x; });
  if (whole_pieces && GATED && epi == EPI_GELU_TANH) return store_rows([](float x, float y) { return epi_gelu_tanh(x) * y; });
  if (whole_pieces && GATED && epi == EPI_SILU) return store_rows([&](float x, float y) { return epi_gate(x, y, EPI_SILU, cap); });
  // The others, and any other C: the sums through LDS, the epilogue in a loop of few instructions.
  constexpr int FLD = 32 * TN + 4;
  static_assert(NW * 32 * FLD * 4 <= NSA * SA + NSB * SB, "no room for the sums' way out");
  float* stage = (float*)gd_lds + (size_t)wave * 32 * FLD;
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int b = 0; b < 4; b++)
        *(f32x4*)(stage + lr * FLD + j * 32 + 8 * b + 4 * lk) =
            f32x4{acc[i][j][4 * b], acc[i][j][4 * b + 1], acc[i][j][4 * b + 2], acc[i][j][4 * b + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
    for (int p = lane; p < 32 * (COLS / 4); p += 64) {
      const int row = p / (COLS / 4), col = p % (COLS / 4) * 4;
      const int m = m0 + wm * 32 * TM + i * 32 + row, n = n0 + wc + col;
      if (m >= M || n >= N) continue;
      const float* x = stage + row * FLD + col;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = GATED ? epi_gate(x[e], x[COLS + e], epi, cap) : epi_unary(x[e], epi, cap);
      store_quad(C, ldc, c_is_f32, m, n, N, v);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
#endif
}

// The tail's tiles: their ranges added in order, the epilogue, the result.  A thread takes four
// neighbouring columns of a row.
template <bool GATED>
__global__ __launch_bounds__(256) void gemm_tail_join_kernel(const float* __restrict__ partials, void* __restrict__ C, int ldc,
                                                             int c_is_f32, int M, int N, int epi, float cap, TileGrid g, int BM,
                                                             int OC) {
  constexpr int NG = GATED ? 2 : 1;
  const int quads = BM * OC / 4;                          // a whole number of blocks
  const int idx = blockIdx.x * 256 + threadIdx.x, t = idx / quads, in = idx - t * quads;
  const int row = in / (OC / 4), col = in % (OC / 4) * 4;
  int tm, tn;
  tile_at(g.from + t, g, tm, tn);
  const int m = tm * BM + row, n = tn * OC + col;
  if (m >= M || n >= N) return;
  const size_t plane = (size_t)g.tail * BM * OC;
  const float* at = partials + (size_t)t * BM * OC + (size_t)row * OC + col;
  f32x4 x = *(const f32x4*)at, y = x;
  if (GATED) y = *(const f32x4*)(at + plane);
  for (int p = 1; p < g.tail_ks; p++) {
    x += *(const f32x4*)(at + (size_t)p * NG * plane);
    if (GATED) y += *(const f32x4*)(at + ((size_t)p * NG + 1) * plane);
  }
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = GATED ? epi_gate(x[i], y[i], epi, cap) : epi_unary(x[i], epi, cap);
  store_quad(C, ldc, c_is_f32, m, n, N, v);
}

struct TileProduct {
  const void* A;
  int lda;
  const void* W;
  void* C;
  int ldc, c_is_f32, M, N, K, epi;
  float cap;
};

// The block tiles.  Wide ones move the fewest bytes into a CU for a product, small ones fill
// the CUs where rows or columns are few; deep stages where one block has a CU to itself.
//   squares of a wave, waves, stages of A and W, blocks a CU; a block's start and end in us, a
//   step of 32 k of one block a CU, of two
#define ZK_TILE_SHAPES(X)                                                    \
  X(0, 4, 2, 2, 4, 2, 3, 1, 7.17, 0.7034, 0.0000)    /* 256 x 256 */ \
  X(1, 2, 2, 2, 4, 3, 3, 1, 4.97, 0.3931, 0.0000)    /* 128 x 256 */ \
  X(2, 2, 2, 4, 2, 3, 4, 1, 4.98, 0.3712, 0.0000)    /* 256 x 128 */ \
  X(3, 3, 2, 2, 4, 2, 3, 1, 5.61, 0.6003, 0.0000)    /* 192 x 256 */ \
  X(4, 3, 2, 2, 2, 3, 5, 1, 4.79, 0.3087, 0.0000)    /* 192 x 128 */ \
  X(5, 2, 2, 2, 2, 4, 5, 1, 3.57, 0.2353, 0.0000)    /* 128 x 128 */ \
  X(6, 2, 2, 2, 2, 2, 3, 2, 3.24, 0.2920, 0.4684)    /* 128 x 128, two */ \
  X(7, 3, 2, 1, 4, 3, 3, 1, 4.37, 0.3452, 0.0000)    /* 96 x 256 */ \
  X(8, 1, 2, 2, 4, 4, 4, 1, 3.10, 0.2832, 0.0000)    /* 64 x 256 */ \
  X(9, 1, 2, 2, 2, 3, 3, 2, 2.24, 0.1629, 0.3194)    /* 64 x 128, two */
struct TileShape {
  int bm, bn, blocks;
  double start, step, step_two;
};
static const TileShape tile_shapes[] = {
#define ZK_SHAPE(V, TM, TN, NWM, NWN, NSA, NSB, MB, START, STEP, STEP2) {32 * TM * NWM, 32 * TN * NWN, MB, START, STEP, STEP2},
    ZK_TILE_SHAPES(ZK_SHAPE)
#undef ZK_SHAPE
};
static const int tile_shape_count = sizeof(tile_shapes) / sizeof(tile_shapes[0]);

static int tile_group(int tiles_m) {
  const int groups = (tiles_m + 5) / 6;
  return (tiles_m + groups - 1) / groups;
}

// Partial sums of ``ks`` ranges of the whole product, of the tail alone (bytes).
static size_t tile_sums(bool gated, int M, int N, int ks) {
  return ks > 1 ? (size_t)ks * (gated ? 2 : 1) * M * ((N + 15) / 16 * 16) * sizeof(float) : 0;
}
static size_t tail_sums(int v, int tail, int ks) {
  return ks > 1 ? (size_t)ks * tail * tile_shapes[v].bm * tile_shapes[v].bn * sizeof(float) : 0;
}

// ``room``: the bytes that the last round's partial sums may take; where they take more, its tiles go a few at a time.
template <int TM, int TN, int NWM, int NWN, int NSA, int NSB, int MB, bool GATED>
static int launch_direct(const TileProduct& p, int col0, int cols, int ks, int tail_ks, float* sums, size_t room, int* parts, hipStream_t s) {
  constexpr int BM = 32 * TM * NWM, BN = 32 * TN * NWN, OC = GATED ? BN / 2 : BN;
  constexpr size_t lds = (size_t)(NSA * BM + NSB * BN) * 128;
  static_assert(lds * MB <= 160 * 1024, "the blocks of a CU do not fit its LDS");
  const auto kernel = gemm_tile_direct_kernel<TM, TN, NWM, NWN, NSA, NSB, MB, GATED>;
  static bool prepared = false;
  if (!prepared) {
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return zk_fail("zk_gemm_bf16: the tile kernel's LDS buffers were refused");
    prepared = true;
  }
  TileGrid g;
  g.tiles_m = (p.M + BM - 1) / BM;
  g.tiles_n = (cols + OC - 1) / OC;
  ZK_REQUIRE((long long)g.tiles_m * g.tiles_n * max(ks, tail_ks) < 2147483647LL, "zk_gemm_bf16: too many tiles");
  g.gm = tile_group(g.tiles_m);
  const int tiles = g.tiles_m * g.tiles_n, tail = tail_ks > 1 ? tiles % (256 * MB) : 0;
  const int most = (int)min((size_t)tail, max(room / ((size_t)tail_ks * BM * BN * sizeof(float)), (size_t)1));
  g.whole = g.from = tiles - tail;
  g.ks = ks;
  g.tail_ks = max(tail_ks, 1);
  g.col0 = col0;
  g.cols = cols;
  do {
    g.tail = min(most, tiles - g.from);
    kernel<<<g.whole * ks + g.tail * g.tail_ks, 64 * NWM * NWN, lds, s>>>(
        (const __bf16*)p.A, p.lda, (const __bf16*)p.W, p.C, p.ldc, p.c_is_f32, p.M, p.N, p.K, p.epi, p.cap, sums, g);
    if (g.tail > 0)
      gemm_tail_join_kernel<GATED><<<g.tail * (BM * OC / 1024), 256, 0, s>>>(sums, p.C, p.ldc, p.c_is_f32, p.M, p.N, p.epi, p.cap,
                                                                             g, BM, OC);
    g.whole = 0;
    g.from += g.tail;
  } while (g.from < tiles);
  if (ks > 1) {
    if (parts && joinable_by_reader(p.N, p.ldc, p.c_is_f32, p.epi)) {
      *parts = ks;
    } else {
      const int npad = (cols + 15) / 16 * 16;
      const size_t quads = (size_t)p.M * (npad / 4);
      gemm_join_kernel<GATED><<<(unsigned)((quads + 255) / 256), 256, 0, s>>>(sums, ks, (char*)p.C + (size_t)col0 * (p.c_is_f32 ? 4 : 2), p.ldc,
                                                                            p.c_is_f32, p.M, cols, npad, p.epi, p.cap);
    }
  }
  return zk_launch_status("zk_gemm_bf16 (tile)");
}

// How a product is cut.  ``rest``: the tile of the columns behind the whole rounds, a launch of their own
// (-1: all columns by ``shape``).
struct TileCut {
  int shape, ks, tail_ks, rest;
};

// The columns that whole rounds of a shape's tiles take.
static int whole_columns(int v, bool gated, int M, int N) {
  const TileShape& t = tile_shapes[v];
  const int oc = gated ? t.bn / 2 : t.bn, tiles_m = (M + t.bm - 1) / t.bm, slots = 256 * t.blocks;
  return (int)((long)tiles_m * ((N + oc - 1) / oc) / slots * slots / tiles_m) * oc;
}

// The time of a cut in microseconds, and the cut with the least.  A CU works through its blocks one
// after the other (or two at a time), each with a start and a time a step; the memory's time
// joins by the cubes; a split adds its partial sums, written, and read by a joining launch or by
// the kernel that follows (``by_reader``).  The constants are fitted to 15,800 measured (rows,
// shape, cut) of the layers of the 2B, 9B and 27B models and of widths 1,024 and 2,048, 70 to 4,096
// rows, weights from memory: 12 % rms, and the cut it names takes 1.02 to 1.03 times the best
// one's time in the mean.  Against the tiles and the rule before (128 x 128 and 64 x 128 tiles through
// registers, 128 x 256 and 256 x 256 copied in stages of 32 k, whole columns to an XCD): 0.82 of the
// time in the geometric mean with joining launches, 0.77 where the reader joins; the most that was
// lost is 4 to 7 % (448 to 1,024 rows by 4608 x 36864).
//
// A gated product by 256 x 256 tiles whose last round is not full may take the columns behind the whole
// rounds by a smaller tile, in a launch of its own (5.5 us: it begins when the first has drained; 10.5 by
// tiles of which two share a CU, 4.5 to 8 us slower there than their price).  The
// ranges of a last round of such tiles write and read two planes of sums, which a joining launch adds up:
// 2048 x (2 x 9216) x 2304 161 us with four ranges, 145 with 128 x 128 tiles for the last eighth; 1024 rows 98 -> 87.
// 94 measured (rows, shape) of 150 to 4,096 rows that it takes: 0.97 of the time in the mean, 1.007 at the worst.
// Not taken where it lost: products without a gate (3,600 x 4608 x 4096 126 -> 132 us), whole rounds of other
// tiles (512 x (2 x 9216) x 2304 by 256 x 128 48.5 -> 55.8), short K (2,400 x (2 x 4096) x 1024 46.3 -> 47.9 at a price of 2 to 4).
static double tile_time(const TileCut& c, bool gated, bool by_reader, int M, int N, int K) {
  const TileShape& t = tile_shapes[c.shape];
  const int oc = gated ? t.bn / 2 : t.bn;
  const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + oc - 1) / oc), slots = 256 * t.blocks;
  auto rounds = [](const TileShape& t, long blocks, double steps) {
    const double one = t.start + steps * t.step, full = t.blocks == 2 ? t.start + steps * t.step_two : one;
    const long slots = 256 * t.blocks, rest = blocks % slots;
    return (double)(blocks / slots) * full + (rest == 0 ? 0.0 : rest <= 256 ? one : full);
  };
  const double steps = K / 32.0, mb = 1e-6, rows_out = (double)M * N;
  const double sums = c.ks > 1 ? (gated ? 2.0 : 1.0) * c.ks * rows_out * 4.0 * mb : 0.0;
  double t_blocks;
  if (c.rest >= 0) {
    const TileShape& u = tile_shapes[c.rest];
    const int ou = gated ? u.bn / 2 : u.bn, cols = whole_columns(c.shape, gated, M, N);
    t_blocks = rounds(t, (long)((M + t.bm - 1) / t.bm) * (cols / oc), steps) + (u.blocks == 2 ? 10.5 : 5.5) +
               rounds(u, (long)((M + u.bm - 1) / u.bm) * ((N - cols + ou - 1) / ou), steps);
  } else if (c.tail_ks > 1) {
    const long tail = tiles % slots;
    t_blocks = rounds(t, tiles - tail, steps) + rounds(t, tail * c.tail_ks, steps / c.tail_ks) + 3.5 +
               (double)tail * c.tail_ks * t.bm * t.bn * 4.0 * mb / 5.0;
  } else {
    t_blocks = rounds(t, tiles * c.ks, steps / c.ks);
  }
  const double t_mem = ((double)(gated ? 2 : 1) * N * K * 2.0 * mb + (double)M * K * 2.0 * mb + rows_out * 2.0 * mb + sums) / 4.15;
  double time = 1.65 + cbrt(t_blocks * t_blocks * t_blocks + t_mem * t_mem * t_mem);
  if (c.ks > 1) time += by_reader ? 0.2 * sums : 3.1 + 0.1425 * sums;
  return time;
}

static TileCut tile_cut(bool gated, bool by_reader, int M, int N, int K, size_t room) {
  static const int splits[] = {2, 3, 4, 5, 6, 8};
  TileCut best{0, 1, 1, -1};
  double best_time = 1e30;
  auto price = [&](const TileCut& c) {
    const double t = tile_time(c, gated, by_reader, M, N, K);
    if (t < best_time) best = c, best_time = t;
  };
  for (int v = 0; v < tile_shape_count; v++) {
    const TileShape& t = tile_shapes[v];
    if (t.bm > 64 && 2L * t.bm > 3L * M) continue;
    const int oc = gated ? t.bn / 2 : t.bn;
    const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + oc - 1) / oc), slots = 256 * t.blocks, tail = tiles % slots;
    price(TileCut{v, 1, 1, -1});
    // ranges of at least 256 k, no more blocks than about a round and a half; a last round no more
    // than half full, cut to one round at the most
    for (int ks : splits)
      if (5 * tiles * ks <= 8 * slots && K / ks >= 256 && tile_sums(gated, M, N, ks) <= room) price(TileCut{v, ks, 1, -1});
    if (tiles > slots && tail > 0 && 2 * tail <= slots)
      for (int ks : {2, 4, 8})
        if (10 * tail * ks <= 11 * slots && K / ks >= 256 && tail_sums(v, (int)tail, ks) <= room) price(TileCut{v, 1, ks, -1});
    if (gated && v == 0 && tiles > slots && tail > 0 && whole_columns(v, gated, M, N) > 0)
      for (int u = 0; u < tile_shape_count; u++)
        if (u != v) price(TileCut{v, 1, 1, u});
  }
  return best;
}

static int launch_columns(int v, bool gated, const TileProduct& p, int col0, int cols, int ks, int tail_ks, float* sums, size_t room,
                          int* parts, hipStream_t s) {
  switch (v) {
#define ZK_SHAPE(V, TM, TN, NWM, NWN, NSA, NSB, MB, START, STEP, STEP2)                                                       \
  case V:                                                                                           \
    return gated ? launch_direct<TM, TN, NWM, NWN, NSA, NSB, MB, true>(p, col0, cols, ks, tail_ks, sums, room, parts, s)    \
                 : launch_direct<TM, TN, NWM, NWN, NSA, NSB, MB, false>(p, col0, cols, ks, tail_ks, sums, room, parts, s);
    ZK_TILE_SHAPES(ZK_SHAPE)
#undef ZK_SHAPE
  }
  return zk_fail("zk_gemm_bf16: no such tile");
}

// ``room``: the bytes at ``sums``.  A cut whose partial sums take more is made some columns (or some of the last round's
// tiles) at a time: the ranges of K, and the order in which an element's sums are added, are those of the whole
// product, and so are the bits.
static int launch_cut(const TileCut& c, bool gated, const TileProduct& p, float* sums, size_t room, int* parts, hipStream_t s) {
  if (c.rest >= 0) {
    const int cols = whole_columns(c.shape, gated, p.M, p.N);
    if (int rc = launch_columns(c.shape, gated, p, 0, cols, 1, 1, sums, room, parts, s)) return rc;
    return launch_columns(c.rest, gated, p, cols, p.N - cols, 1, 1, sums, room, parts, s);
  }
  if (tile_sums(gated, p.M, p.N, c.ks) <= room) return launch_columns(c.shape, gated, p, 0, p.N, c.ks, c.tail_ks, sums, room, parts, s);
  const int oc = gated ? tile_shapes[c.shape].bn / 2 : tile_shapes[c.shape].bn;
  const int cols = (int)(room / tile_sums(gated, p.M, oc, c.ks)) * oc;
  // (of 64 cuts whose sums for one tile's columns are more than the static array's 16 MiB, all are refused before)
  ZK_REQUIRE(cols > 0, "zk_gemm_bf16: no room for the partial sums of one tile's columns");
  for (int n = 0; n < p.N; n += cols)
    if (int rc = launch_columns(c.shape, gated, p, n, min(cols, p.N - n), c.ks, 1, sums, room, nullptr, s)) return rc;
  return 0;
}
