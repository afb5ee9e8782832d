// The kernels of attention_bf16.hip as templates over the sizes of a head's keys (HD16 sixteens) and of
// its values (VD16), and what launches them for one pair of sizes.  attention_bf16.hip holds those whose
// sizes are equal, attention_bf16_uneven.hip those of values half or twice as wide as keys, so
// that the two compile side by side.
#pragma once
#include "common.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

#if ZSE_ACT_BF16

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define ATT_CHUNK 64
#define ATT_DECODE_SPAN 128    // keys of a partial result of a decoded token on 16-wide tiles
#define ATT_DECODE_LONG_FROM 4096      // 256 instead where a request's table holds this many keys or more
#define ATT_SHORT_WAVES 4      // waves of a block of a portion of few rows
#define ATT_MOST_RANGES 8      // ranges of keys a block of rows of a portion is cut into, at most

struct AttnParams {
  const __bf16* q;
  int q_stride;
  const __bf16* kcache;   // [page][nkv][bs][hd]
  const __bf16* vcache;   // [page][nkv >> v_shift][vd][bs]
  int v_shift;            // 2^v_shift neighbouring key heads share one value head (0: a value head per key head)
  const int* block_table;
  int max_blocks;
  const int* q_start;     // [R + 1]
  const int* ctx_len;     // [R]
  __bf16* out;            // [T][nh][vd]
  float* part_o;          // split: [slot][vd]
  float* part_ml;         // split: [slot][2]
  int nh, nkv, hd, bs;
  int vd;                 // channels of a value (and of the output's heads); hd: of a query or key
  int bs_shift;           // page size is 1 << bs_shift in the tuned kernels
  float scale, softcap;
  // scores in the log2 domain: with a cap c,  s2 = c2 * tanh(k2 * dot / 2)  computed as
  // c2 * (1 - 2 / (exp2(k2 * dot) + 1)),  k2 = 2 * scale / c * log2(e),  c2 = c * log2(e);
  // without a cap  s2 = k1 * dot,  k1 = scale * log2(e).  Probabilities are exp2(s2 - m2).
  float k1, k2, c2;
  int window;
  int tpw;                // tokens a wave owns
  int r_begin;            // first request of this launch
  int nchunks;            // split: chunks the grid covers
  int from_window;        // decode: block 0 of a request is the one its window begins in
  int chunk;              // portions with their keys in ranges: tiles of a range; decoded tokens in blocks of 256 keys: a wave's keys
  int mask_chunk;         // > 0: a row sees the keys of its own chunk of this many positions only (no window then)
  int keep;               // beside its window a row sees the first ``keep`` keys of its sequence
  int sink;               // 1: a key of score 0 without a value joins every row's denominator
  const float* sinks;     // [nh] (may be null): exp(sinks[h]) joins head h's denominator, with no key and no value
  const __bf16* gate;     // (may be null) row t's numbers per head at gate + t * gate_ld; head h's output is
  int gate_ld;            // multiplied by the sigmoid of the h-th
  int wide_weights;       // 1: a weight meets the values as two bf16 numbers, its rounded value and what the
                          // rounding left (16 bits of mantissa instead of 8; one more product a tile)
};

// The query head that is the hq-th of key head kvh.  Without shared values: kvh * g + hq.  With
// 2^v_shift maps of keys over one value head, key head (v, m) serves map m of the g query heads
// of value head v, and a query head's maps lie side by side: ((v * g + hq) << v_shift) + m.
__device__ __forceinline__ int q_head_of(const AttnParams& p, int kvh, int hq) {
  const int g = p.nh / p.nkv;
  return (((kvh >> p.v_shift) * g + hq) << p.v_shift) | (kvh & ((1 << p.v_shift) - 1));
}

// The first key a row at position ``pos`` sees.  It never decreases as pos grows, which is all
// the kernels' bounds over groups and blocks of rows rest on.
__device__ __forceinline__ int first_key(const AttnParams& p, int pos) {
  if (p.mask_chunk > 0) return pos - pos % p.mask_chunk;
  return p.window > 0 ? max(0, pos - p.window + 1) : 0;
}

// The tiles of 32 keys that rows whose first key (but for the kept ones) is key_lo walk up to key_hi: those
// of the kept first keys, then from key_lo's on.  Tile i begins at key_of(i), 0 <= i < count.
struct KeyTiles {
  int kept, lo, count;
  __device__ __forceinline__ KeyTiles(const AttnParams& p, int key_lo, int key_hi) {
    lo = key_lo / 32;
    kept = min((p.keep + 31) / 32, lo);
    count = key_hi < 0 ? 0 : kept + key_hi / 32 - lo + 1;
  }
  __device__ __forceinline__ int key_of(int i) const { return 32 * (i < kept ? i : lo + i - kept); }
};

// What a head's sink adds to a row's sum of weights: 2^(sink - m), scores and maximum in the log2 domain.
__device__ __forceinline__ float sink_weight(const float* sinks, int unit_sink, int head, float m) {
  if (sinks) return __builtin_amdgcn_exp2f(sinks[head] * 1.4426950408889634f - m);
  return unit_sink ? __builtin_amdgcn_exp2f(-m) : 0.f;
}

// The sigmoid of a row's gate for a head.
__device__ __forceinline__ float gate_factor(const __bf16* gate, int gate_ld, int row, int head) {
  if (!gate) return 1.f;
  return 1.f / (1.f + __expf(-(float)gate[(size_t)row * gate_ld + head]));
}

// What a row's sum of weighted values is multiplied by: 1 over the sum of its weights, and its gate.
__device__ __forceinline__ float row_factor(const AttnParams& p, int row, int head, float l, float m) {
  return gate_factor(p.gate, p.gate_ld, row, head) / (l + sink_weight(p.sinks, p.sink, head, m));
}

__device__ __forceinline__ float score_log2(const AttnParams& p, float dot) {
  if (p.softcap > 0.f) {
    const float e = __builtin_amdgcn_exp2f(p.k2 * dot);
    return p.c2 * (1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f));
  }
  return p.k1 * dot;
}

// Portions: which (group, KV head) a block takes.  Blocks go to the 8 XCDs in turn by their
// number, and every XCD has an L2 of its own; blocks that read the same keys and values (those
// of one KV head) are therefore given to as few XCDs as possible, so that what one of them has
// fetched is in the L2 for the others instead of crossing from the memory side once per block.
__device__ __forceinline__ void portion_block(int& bx, int& by) {
  const int gx = gridDim.x, gy = gridDim.y;
  bx = blockIdx.x;
  by = blockIdx.y;
  const int total = gx * gy;
  if (total % 8) return;
  const int lin = blockIdx.x + gx * blockIdx.y, xcd = lin & 7, slot = lin >> 3;
  if (gy <= 8 && 8 % gy == 0) {            // 8 / gy XCDs a head
    const int per = 8 / gy;
    by = xcd % gy;
    bx = slot * per + xcd / gy;
  } else if (gy % 8 == 0) {                // gy / 8 heads an XCD
    const int heads = gy / 8;
    by = xcd + 8 * (slot % heads);
    bx = slot / heads;
  }
}

template <int HD16, int VD16, bool SPLIT, bool PAIR>
__global__ __launch_bounds__(256, (HD16 <= 8 && VD16 <= 8 && !PAIR) ? 2 : 1) void attn_mfma_kernel(AttnParams p) {
  constexpr int DT = (VD16 + 1) / 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 31, lk = lane >> 5;
  const int r = p.r_begin + blockIdx.z;
  int block_x = blockIdx.x, kvh = blockIdx.y;
  if (!SPLIT) portion_block(block_x, kvh);
  const int qs = p.q_start[r], n = p.q_start[r + 1] - qs;
  if (n <= 0) return;
  const int start = p.ctx_len[r] - n;
  // portions: a block owns one group of rows and its four waves take every fourth tile of
  // keys (their results are joined at the end).  Or (PAIR, for portions whose groups would
  // need a second, half-empty round of blocks) two groups: one from the end of the portion,
  // which sees many keys, and its mirror from the start, which sees few, so that every block
  // has about the same work; the four waves are shared out between the two by their numbers
  // of key tiles (3 + 1, 2 + 2 or 1 + 3), a group's waves taking its tiles in turn.
  // Decoded tokens: a wave owns one chunk of keys.
  int gi = 0, phase = wave, nphase = 4, first_wave = 0;        // group, and the wave's place among its waves
  int na_block = 4;                                            // waves of the block's first group
  // single groups: the last group of a portion sees the most keys and goes first, so that the
  // blocks still running at the end are the short ones
  if (!SPLIT && !PAIR) gi = (n + p.tpw - 1) / p.tpw - 1 - block_x;
  if (PAIR) {
    const int groups = (n + p.tpw - 1) / p.tpw;
    if (block_x >= (groups + 1) / 2) return;           // the whole block is past the portion
    const int ga = groups - 1 - block_x, gb = block_x;
    if (ga != gb) {
      auto tiles_of = [&](int gr) {
        const int lo = start + gr * p.tpw, hi = start + min(n, (gr + 1) * p.tpw) - 1;
        return KeyTiles(p, first_key(p, lo), hi).count;
      };
      const int ta = tiles_of(ga), tb = tiles_of(gb);
      const int na = min(3, max(1, (4 * ta + (ta + tb) / 2) / (ta + tb)));
      na_block = na;
      if (wave < na) { gi = ga; phase = wave; nphase = na; }
      else { gi = gb; phase = wave - na; nphase = 4 - na; first_wave = na; }
    } else {
      gi = ga;
    }
  }
  const int chunk = SPLIT ? block_x * 4 + wave : 0;
  const int t0 = gi * p.tpw;
  if (!PAIR && (gi < 0 || t0 >= n)) return;
  const int g = p.nh / p.nkv;
  const int tok = lr / g, hq = lr - tok * g;
  const int ntok = min(p.tpw, n - t0);
  const bool row_ok = tok < ntok;
  const int trow = qs + t0 + (row_ok ? tok : 0);
  const int pos = start + t0 + (row_ok ? tok : 0);
  const int head = q_head_of(p, kvh, row_ok ? hq : 0);
  const int pos_lo = start + t0, pos_hi = start + t0 + ntok - 1;
  int key_lo = first_key(p, pos_lo);
  int key_hi = pos_hi;
  if (SPLIT) {
    key_lo = chunk * ATT_CHUNK < p.keep ? chunk * ATT_CHUNK : max(key_lo, chunk * ATT_CHUNK);
    key_hi = min(key_hi, chunk * ATT_CHUNK + ATT_CHUNK - 1);
  }
  if (SPLIT && key_lo > key_hi) return;
  const int row_lo = first_key(p, pos);
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  const int hd = p.hd, vd = p.vd, bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv;

  bf16x8 qf[HD16];
  {
    const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * hd + lk * 8;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++) {
      if (row_ok) qf[ks] = *(const bf16x8*)(qr + ks * 16);
      else
#pragma unroll
        for (int e = 0; e < 8; e++) qf[ks][e] = (__bf16)0.f;
    }
  }
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int e = 0; e < 16; e++) o[dt][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  // where the lane's channels dt * 32 + lr lie in a (page, kv head) block of the transposed V cache
  int vrow[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++) vrow[dt] = min(dt * 32 + lr, vd - 1) << bsh;
  const bool capped = p.softcap > 0.f;
  // keys every row of the group sees (none beyond the first row's position, none before the
  // last row's window; no range at all unless every lane holds a row): tiles inside this range
  // need no mask
  const int all_hi = ntok * g == 32 ? pos_lo : -1;
  const int all_lo = first_key(p, pos_hi);

  // The pages of a tile are looked up a tile ahead as well, so that no load waits for a table
  // entry: the lane's key row, and the four places its V pieces come from.
  struct TilePages { int k, va[2], vb[2]; };
  auto look_up = [&](int key0, TilePages& pg) {
    pg.k = table[min(key0 + lr, key_hi) >> bsh];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      pg.va[h] = table[min(key0 + h * 16 + 4 * lk, key_hi & ~3) >> bsh];
      pg.vb[h] = table[min(key0 + h * 16 + 8 + 4 * lk, key_hi & ~3) >> bsh];
    }
  };
  auto load_k = [&](int key0, int page, bf16x8 (&kf)[HD16]) {
    const int kk = min(key0 + lr, key_hi);
    const __bf16* kr = p.kcache + ((((size_t)max(page, 0) * nkv + kvh) << bsh) + (kk & bmask)) * hd + lk * 8;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++) kf[ks] = *(const bf16x8*)(kr + ks * 16);
  };
  auto tile = [&](int key0, const TilePages& pg, int knext, TilePages& pn) {
    bf16x8 kf[HD16];
    load_k(key0, pg.k, kf);
    look_up(knext, pn);
    // ---- S^T = K Q^T
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qf[ks], s, 0, 0, 0);
    // ---- V^T pieces for this tile (issued early; used after the softmax)
    bf16x8 vf[DT][2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int ka = min(key0 + h * 16 + 4 * lk, key_hi & ~3), kb = min(key0 + h * 16 + 8 + 4 * lk, key_hi & ~3);
      const int pa = max(pg.va[h], 0), pb = max(pg.vb[h], 0);
      const __bf16* vpa = p.vcache + ((((size_t)pa * (nkv >> p.v_shift) + (kvh >> p.v_shift)) * vd) << bsh) + (ka & bmask);
      const __bf16* vpb = p.vcache + ((((size_t)pb * (nkv >> p.v_shift) + (kvh >> p.v_shift)) * vd) << bsh) + (kb & bmask);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const bf16x4 va = *(const bf16x4*)(vpa + vrow[dt]);
        const bf16x4 vb = *(const bf16x4*)(vpb + vrow[dt]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          vf[dt][h][e] = va[e];
          vf[dt][h][4 + e] = vb[e];
        }
      }
    }
    // ---- scale, cap, mask, running softmax (one query row per lane)
    float mt = -INFINITY;
    if (capped) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float ex = __builtin_amdgcn_exp2f(p.k2 * s[e]);
        s[e] = p.c2 * (1.f - 2.f * __builtin_amdgcn_rcpf(ex + 1.f));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] *= p.k1;
    }
    if (key0 < all_lo || key0 + 31 > all_hi || key0 < key_lo || key0 + 31 > key_hi) {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int key = key0 + 8 * j + 4 * lk + i;
          const bool ok = row_ok && (key >= row_lo || key < p.keep) && key <= pos && key <= key_hi;
          s[4 * j + i] = ok ? s[4 * j + i] : -INFINITY;
        }
    }
#pragma unroll
    for (int e = 0; e < 16; e++) mt = fmaxf(mt, s[e]);
    mt = wave_max32(mt);
    const float m_new = mt > m_run + 8.f ? mt : m_run;      // the reference follows the maximum lazily
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const bool moved = m_new > m_run;
    const float corr = moved ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.f;
    float rs = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const float pe = __builtin_amdgcn_exp2f(s[e] - m_use);
      s[e] = pe;
      rs += pe;
    }
    rs = wave_add32(rs);
    l_run = l_run * corr + rs;
    m_run = m_new;
    bf16x8 pb[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int e = 0; e < 8; e++) pb[h][e] = (__bf16)s[8 * h + e];
    // ---- O^T = corr * O^T + V^T P^T  (the maximum rarely rises by the threshold after a
    // row's first tiles; said so, the compiler keeps the accumulators where the products
    // want them instead of moving all of them on every tile)
    if (__builtin_expect(__any(moved), 0)) {
      // in the accumulation registers, where the products keep them: written so, the compiler
      // does not copy all of them to ordinary registers on every tile for this rare path
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          float t;
          asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\tv_accvgpr_write_b32 %0, %1"
                       : "+a"(o[dt][e]), "=&v"(t)
                       : "v"(corr));
        }
    }
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt][0], pb[0], o[dt], 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt][1], pb[1], o[dt], 0, 0, 0);
    }
    if (p.wide_weights) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 8; e++) pb[h][e] = (__bf16)(s[8 * h + e] - (float)pb[h][e]);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt][0], pb[0], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt][1], pb[1], o[dt], 0, 0, 0);
      }
    }
  
  };
  {
    // (a chunk of a decoded token has its tiles one behind the other, kept keys among them or not)
    KeyTiles ts(p, key_lo, key_hi);
    if (SPLIT) {
      ts.kept = 0;
      ts.count = key_hi / 32 - ts.lo + 1;
    }
    const int step = SPLIT ? 1 : nphase;
    int i = SPLIT ? 0 : phase;
    TilePages p0, p1;
    if (i < ts.count) look_up(ts.key_of(i), p0);
    for (; i < ts.count; i += 2 * step) {
      tile(ts.key_of(i), p0, ts.key_of(i + step), p1);
      if (i + step >= ts.count) break;
      tile(ts.key_of(i + step), p1, ts.key_of(i + 2 * step), p0);
    }
  }
  if (SPLIT) {
    if (!row_ok) return;
    const size_t slot = ((size_t)(r - p.r_begin) * p.nh + head) * p.nchunks + chunk;
    if (lk == 0) {
      p.part_ml[slot * 2] = m_run;
      p.part_ml[slot * 2 + 1] = l_run;
    }
    float* po = p.part_o + slot * vd;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int d = dt * 32 + 8 * j + 4 * lk;
        if (d < vd) *(f32x4*)(po + d) = f32x4{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
      }
  } else {
    // join a group's waves: common maximum and sum per row, then the accumulators of the
    // group's other waves reach its first wave through LDS, one wave a round (a slot a group)
    extern __shared__ float dyn[];
    float* sm_ml = dyn;                          // [4][32][2]
    float* sm_o = dyn + 4 * 32 * 2;              // [2][DT * 16][64]
    if (lk == 0) {
      sm_ml[(wave * 32 + lr) * 2] = m_run;
      sm_ml[(wave * 32 + lr) * 2 + 1] = l_run;
    }
    __syncthreads();
    float m_all = -INFINITY;
    for (int w = first_wave; w < first_wave + nphase; w++) m_all = fmaxf(m_all, sm_ml[(w * 32 + lr) * 2]);
    float l_all = 0.f;
    for (int w = first_wave; w < first_wave + nphase; w++) {
      const float mw = sm_ml[(w * 32 + lr) * 2];
      l_all += mw == -INFINITY ? 0.f : sm_ml[(w * 32 + lr) * 2 + 1] * __builtin_amdgcn_exp2f(mw - m_all);
    }
    const float f = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_all);
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int e = 0; e < 16; e++) o[dt][e] *= f;
    float* slot = sm_o + (size_t)(first_wave ? 1 : 0) * DT * 16 * 64;
    const int rounds = max(na_block, 4 - na_block) - 1;
    for (int step = 1; step <= rounds; step++) {
      if (phase == step) {
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
          for (int e = 0; e < 16; e++) slot[(dt * 16 + e) * 64 + lane] = o[dt][e];
      }
      __syncthreads();
      if (phase == 0 && step < nphase) {
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
          for (int e = 0; e < 16; e++) o[dt][e] += slot[(dt * 16 + e) * 64 + lane];
      }
      __syncthreads();
    }
    if (phase != 0 || !row_ok) return;
    const float inv = row_factor(p, trow, head, l_all, m_all);
    __bf16* orow = p.out + ((size_t)trow * p.nh + head) * vd;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int d = dt * 32 + 8 * j + 4 * lk;
        if (d < vd) {
          bf16x4 w;
#pragma unroll
          for (int i = 0; i < 4; i++) w[i] = (__bf16)(o[dt][4 * j + i] * inv);
          *(bf16x4*)(orow + d) = w;
        }
      }
  }
}

// Long portions.  A block of NW waves owns NW groups of rows that follow each other in one
// request (NW * tpw tokens times the g heads of a KV head), every wave one group, and all of
// them walk the same keys: a tile of 32 keys and its values come from the cache once a block,
// wait in LDS and serve every wave (attn_mfma_kernel fetches them once a group of 32 rows:
// with many groups the way from L2 to the CUs then sets the time).  No join: a wave sees all
// the keys of its rows.  Two buffers: the loads of the next tile are in flight while the
// current one is multiplied, and one barrier a tile suffices.
//   sK [2][32 keys][hd + 8]       a lane's piece for the first product is 16 bytes of a key's row
//   sV [2][vd][32 + 8]            a channel's 32 keys in the order the second product wants:
//                                 piece 2h + lk = keys 16h + 4lk + (0..3), 16h + 8 + 4lk + (0..3)
// The padding of 16 bytes a row keeps the 16-byte reads of 16 lanes on different banks.
// Pages of at least 8 keys (a 16-byte piece of the transposed V holds 8 keys of one page).
//
// SPLIT: a launch of few blocks with many keys each (a prompt of a few thousand tokens and few
// heads) cuts the keys of a block of rows into ranges of p.chunk tiles, counted from the
// block's first tile; blockIdx.x is (block of rows) * p.nchunks + range.  A block then leaves
// (max, sum, O) of its range for every row, as the chunks of a decoded token do, and
// attn_portion_join_kernel joins a row's ranges in their order.
template <int HD16, int VD16, int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64, (HD16 <= 8 && VD16 <= 8 && NW <= 4) ? 2 : 1) void attn_shared_kernel(AttnParams p) {
  constexpr int HD = HD16 * 16, VD = VD16 * 16, DT = (VD16 + 1) / 2;
  constexpr int KLD = HD + 8, VLD = 32 + 8;
  constexpr int NT = NW * 64;
  constexpr int PIECES = 4 * HD, V_PIECES = 4 * VD;     // 16-byte pieces of a K tile, and of a V tile
  constexpr int PPT = (PIECES + NT - 1) / NT, VPT = (V_PIECES + NT - 1) / NT;           // pieces of each a thread moves
  constexpr int CPK = HD / 8;                           // pieces of a key's row
  extern __shared__ __attribute__((aligned(16))) unsigned char shared_raw[];
  __bf16* sK = (__bf16*)shared_raw;                     // [2][32][KLD]
  __bf16* sV = sK + 2 * 32 * KLD;                       // [2][VD][VLD]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, lk = lane >> 5;
  const int r = p.r_begin + blockIdx.z;
  int block_x, kvh;
  portion_block(block_x, kvh);
  const int qs = p.q_start[r], n = p.q_start[r + 1] - qs;
  if (n <= 0) return;
  const int start = p.ctx_len[r] - n;
  const int per_block = NW * p.tpw;
  // the last rows of a portion see the most keys and go first
  const int rows_x = SPLIT ? block_x / p.nchunks : block_x;
  const int range = SPLIT ? block_x - rows_x * p.nchunks : 0;
  const int bi = (n + per_block - 1) / per_block - 1 - rows_x;
  if (bi < 0) return;
  const int g = p.nh / p.nkv;
  // the block's keys: from the window of its first row to its last row
  const int blk_lo = start + bi * per_block, blk_hi = start + min(n, (bi + 1) * per_block) - 1;
  const int key_lo = first_key(p, blk_lo), key_hi = blk_hi;
  const KeyTiles ts(p, key_lo, key_hi);
  int tile_i = 0, tile_end = ts.count;
  if (SPLIT) {
    tile_i = range * p.chunk;
    if (tile_i >= ts.count) return;                    // the block of rows has fewer ranges
    tile_end = min(ts.count, tile_i + p.chunk);
  }
  // the wave's rows
  const int t0 = bi * per_block + wave * p.tpw;
  const int ntok = max(0, min(p.tpw, n - t0));
  const int tok = lr / g, hq = lr - tok * g;
  const bool row_ok = tok < ntok;
  const int trow = qs + (row_ok ? t0 + tok : 0);
  const int pos = start + (row_ok ? t0 + tok : 0);
  const int head = q_head_of(p, kvh, row_ok ? hq : 0);
  const int pos_lo = start + t0, pos_hi = start + t0 + ntok - 1;          // ntok == 0: no keys at all
  const int row_lo = first_key(p, pos);
  const int all_hi = ntok * g == 32 ? pos_lo : -1;
  const int all_lo = first_key(p, pos_hi);
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  const int bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv;

  bf16x8 qf[HD16];
  {
    const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * HD + lk * 8;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++) {
      if (row_ok) qf[ks] = *(const bf16x8*)(qr + ks * 16);
      else
#pragma unroll
        for (int e = 0; e < 8; e++) qf[ks][e] = (__bf16)0.f;
    }
  }
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int e = 0; e < 16; e++) o[dt][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // The thread's pieces of a tile.  K: piece q is 8 channels (q % CPK) of key q / CPK.  V: the
  // pieces of a page's part of the tile lie one behind the other in the cache, channel by
  // channel: with tk = min(page size, 32) keys of a page in the tile, piece q is the keys
  // [8c, 8c + 8) of channel d in part q / (HD tk / 8), d = (q / (tk / 8)) % HD, c = q % (tk / 8).
  const int tk_shift = min(bsh, 5);                     // log2 of a page's keys in a tile
  const int cpp_shift = tk_shift - 3;                   // log2 of the pieces of a channel in a page's part
  // What does not change from tile to tile is worked out here, per piece: its place in the page
  // table relative to the tile's first entry, its offset inside a page's block of the cache (the
  // KV head, the key's place in the page, the channels) and its place in LDS.  A tile then costs
  // a piece one table entry and one multiply-add.  (Tiles start at multiples of 32 keys: with
  // pages of up to 32 keys a key's place in its page does not depend on the tile, with larger
  // pages the whole tile lies in one page and the tile's offset in it is the same for all.)
  int k_idx[PPT], v_idx[VPT], k_lds[PPT], v_lds[VPT];
  unsigned k_off[PPT], v_off[VPT];
#pragma unroll
  for (int j = 0; j < PPT; j++) {
    const int q = min(tid + j * NT, PIECES - 1);
    const int kk = q / CPK, col = (q % CPK) * 8;
    k_idx[j] = kk >> bsh;
    k_off[j] = (unsigned)(((kvh << bsh) + (kk & bmask)) * HD + col);
    k_lds[j] = kk * KLD + col;
  }
#pragma unroll
  for (int j = 0; j < VPT; j++) {
    const int q = min(tid + j * NT, V_PIECES - 1);
    const int part = q / (VD << cpp_shift), rem = q - part * (VD << cpp_shift);
    const int d = rem >> cpp_shift;
    const int vk = (part << tk_shift) + ((rem & ((1 << cpp_shift) - 1)) << 3);
    v_idx[j] = vk >> bsh;
    v_off[j] = (unsigned)((((kvh >> p.v_shift) * VD + d) << bsh) + (vk & bmask));
    // keys 8c + (0..3) go to piece 2h of the channel, keys 8c + 4 + (0..3) to piece 2h + 1,
    // both at slot 4 (c % 2), with h = c / 2
    const int c = vk >> 3;
    v_lds[j] = d * VLD + (c >> 1) * 16 + (c & 1) * 4;
  }
  const size_t page_elems = ((size_t)nkv * HD) << bsh;        // of a page of K
  const size_t v_page_elems = ((size_t)(nkv >> p.v_shift) * VD) << bsh;
  const int last_entry = p.max_blocks - 1;
  struct Pages { int k[PPT], v[VPT]; };
  struct Stage { bf16x8 k[PPT], v[VPT]; };
  // A key past the request's last (in its last tile, or in the tile fetched after the last) is
  // read from wherever its table entry points, page 0 where there is none.  It is masked, but
  // its value still meets a weight of 0 in the second product, and 0 x NaN is NaN: the caller
  // keeps page 0 cleared and clears a page before a request first writes to part of it, so
  // what is read here is the request's own or zero, never what another request left.
  auto look_up = [&](int key0, Pages& pg) {
    const int first = key0 >> bsh;
#pragma unroll
    for (int j = 0; j < PPT; j++) pg.k[j] = table[min(first + k_idx[j], last_entry)];
#pragma unroll
    for (int j = 0; j < VPT; j++) pg.v[j] = table[min(first + v_idx[j], last_entry)];
  };
  auto fetch = [&](int key0, const Pages& pg, Stage& st) {
    const unsigned in_page = (unsigned)(key0 & bmask);
#pragma unroll
    for (int j = 0; j < PPT; j++)
      st.k[j] = *(const bf16x8*)(p.kcache + ((size_t)max(pg.k[j], 0) * page_elems + (k_off[j] + in_page * HD)));
#pragma unroll
    for (int j = 0; j < VPT; j++)
      st.v[j] = *(const bf16x8*)(p.vcache + ((size_t)max(pg.v[j], 0) * v_page_elems + (v_off[j] + in_page)));
  };
  auto stash = [&](int buf, const Stage& st) {
    __bf16* kb = sK + buf * 32 * KLD;
    __bf16* vb = sV + buf * VD * VLD;
#pragma unroll
    for (int j = 0; j < PPT; j++)
      if (PIECES % NT == 0 || tid + j * NT < PIECES) *(bf16x8*)(kb + k_lds[j]) = st.k[j];
#pragma unroll
    for (int j = 0; j < VPT; j++) {
      if (V_PIECES % NT == 0 || tid + j * NT < V_PIECES) {
        __bf16* vrow = vb + v_lds[j];
        bf16x4 lo4, hi4;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          lo4[e] = st.v[j][e];
          hi4[e] = st.v[j][4 + e];
        }
        *(bf16x4*)vrow = lo4;
        *(bf16x4*)(vrow + 8) = hi4;
      }
    }
  };
  const bool capped = p.softcap > 0.f;
  auto tile = [&](int buf, int key0) {
    const __bf16* kb = sK + buf * 32 * KLD + lr * KLD + lk * 8;
    const __bf16* vb = sV + buf * VD * VLD + lk * 8;
    // ---- S^T = K Q^T
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(kb + ks * 16), qf[ks], s, 0, 0, 0);
    // ---- scale, cap, mask, running softmax (one query row per lane)
    float mt = -INFINITY;
    if (capped) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float ex = __builtin_amdgcn_exp2f(p.k2 * s[e]);
        s[e] = p.c2 * (1.f - 2.f * __builtin_amdgcn_rcpf(ex + 1.f));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] *= p.k1;
    }
    if (key0 < all_lo || key0 + 31 > all_hi) {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int key = key0 + 8 * j + 4 * lk + i;
          const bool ok = row_ok && (key >= row_lo || key < p.keep) && key <= pos;
          s[4 * j + i] = ok ? s[4 * j + i] : -INFINITY;
        }
    }
#pragma unroll
    for (int e = 0; e < 16; e++) mt = fmaxf(mt, s[e]);
    mt = wave_max32(mt);
    const float m_new = mt > m_run + 8.f ? mt : m_run;      // the maximum is followed lazily
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const bool moved = m_new > m_run;
    const float corr = moved ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.f;
    float rs = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const float pe = __builtin_amdgcn_exp2f(s[e] - m_use);
      s[e] = pe;
      rs += pe;
    }
    rs = wave_add32(rs);
    l_run = l_run * corr + rs;
    m_run = m_new;
    bf16x8 pb[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int e = 0; e < 8; e++) pb[h][e] = (__bf16)s[8 * h + e];
    // ---- O^T = corr O^T + V^T P^T
    if (__builtin_expect(__any(moved), 0)) {
      // in the accumulation registers, where the products keep them
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          float t;
          asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\tv_accvgpr_write_b32 %0, %1"
                       : "+a"(o[dt][e]), "=&v"(t)
                       : "v"(corr));
        }
    }
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      const __bf16* vr = vb + min(dt * 32 + lr, VD - 1) * VLD;
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)vr, pb[0], o[dt], 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(vr + 16), pb[1], o[dt], 0, 0, 0);
    }
    if (p.wide_weights) {
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 8; e++) pb[h][e] = (__bf16)(s[8 * h + e] - (float)pb[h][e]);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const __bf16* vr = vb + min(dt * 32 + lr, VD - 1) * VLD;
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)vr, pb[0], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(vr + 16), pb[1], o[dt], 0, 0, 0);
      }
    }
  };

  // Every wave takes every tile of the block, also the few near the diagonal (or before its
  // window) that none of its rows sees: masked, such a tile adds nothing, and a loop without a
  // branch around the products lets the compiler leave the accumulators where they are (with
  // the branch it copied all of them to ordinary registers on every turn: 852 instead of 1,135 us
  // at 16 heads of 256).  The turn after the last tile fetches that tile again and leaves it
  // unused.
  {
    Pages pg, pn;
    Stage st;
    look_up(ts.key_of(tile_i), pg);
    fetch(ts.key_of(tile_i), pg, st);
    look_up(ts.key_of(tile_i + 1), pn);
    stash(0, st);
    __syncthreads();
    for (int buf = 0; tile_i < tile_end; tile_i++, buf ^= 1) {
      fetch(ts.key_of(tile_i + 1), pn, st);
      look_up(ts.key_of(tile_i + 2), pn);
      tile(buf, ts.key_of(tile_i));
      stash(buf ^ 1, st);
      __syncthreads();
    }
  }
  if (!SPLIT && !row_ok) return;
  if (SPLIT) {
    // A wave's results of its range, as they lie in its registers: 16 bytes a lane, a wave's 64
    // lanes one contiguous KB per (dt, j), so every store is whole lines.  The joining kernel
    // reads them back with the same lanes.  Every lane stores, rows or not.
    const size_t slot = ((((size_t)blockIdx.z * p.nkv + kvh) * (gridDim.x / p.nchunks) + rows_x) * p.nchunks + range) * NW + wave;
    p.part_ml[slot * 128 + lane] = lk == 0 ? m_run : l_run;
    f32x4* po = (f32x4*)p.part_o + slot * (DT * 4 * 64) + lane;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        po[(dt * 4 + j) * 64] = f32x4{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
    return;
  }
  const float inv = row_factor(p, trow, head, l_run, m_run);
  __bf16* orow = p.out + ((size_t)trow * p.nh + head) * VD;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int d = dt * 32 + 8 * j + 4 * lk;
      if (d < VD) {
        bf16x4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (__bf16)(o[dt][4 * j + i] * inv);
        *(bf16x4*)(orow + d) = w;
      }
    }
}

// The order of a quarter of a turn of attn_stream_kernel: a product, two LDS reads for the next
// quarter, a few vector operations; in the second half no more reads, so that the last have arrived when
// the next quarter begins.
template <int MFMAS, int VALUS>
__device__ __forceinline__ void stream_order() {
#pragma unroll
  for (int i = 0; i < MFMAS; i++) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (i < MFMAS / 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, VALUS, 0);
  }
}

// Long portions, heads of 128 and 256 channels: attn_shared_kernel's division of the work (four waves of
// 32 rows, the same tiles of 32 keys, the same results) with the keys and values on their way
// for several tiles, and three tiles in work at a time.
//
// What bounded the other: a turn asked for the next tile and waited for it at its end, so a tile
// took a trip to memory (2.4 to 2.7 us at 256 channels, of which its products are 0.5), and a wave's scores,
// weights and second product followed each other, one wave a SIMD.  Here tiles are copied into
// LDS without passing through registers, keys up to four tiles ahead and values three; and a turn t multiplies tile
// t + 1 by the queries and tile t - 1's weights by its values while the vector unit turns tile t's scores into
// weights.  The page table is read 64 entries at a time into a register.
//
// LDS, a ring of four tiles each.  K: a key's row of HD channels; place p of 16 bytes of row r holds
// piece p ^ (r % 16), so that sixteen rows read at once lie in different banks.  V: [16 keys][channel][the 16 keys' values], the two
// pieces of a channel swapped where its number has bit 3, for the same reason; pages of 16 keys or more, so that a copy
// is one run of such a page.
// Row 8 j + 4 a + i of a score tile is key 16 (j / 2) + 8 a + 4 (j % 2) + i, so that a lane's eight weights of a
// half tile belong to eight neighbouring keys: 16 bytes of a channel of the transposed values.
//
// A masked score is set to the score's least value before the turn and its weight to zero after it; only tiles at an edge
// have any.  Tiles past the range are copied and multiplied, never weighted.  Keys past the block's last page are copied from
// that page: whatever the table holds behind it is neither followed nor multiplied by a weight of 0.
template <int HD16, int VD16, bool SPLIT, bool CAPPED>
__global__ __launch_bounds__(256, (HD16 <= 8 && VD16 <= 8) ? 2 : 1) void attn_stream_kernel(AttnParams p) {
  // (the host's pass knows no address spaces)
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int HD = HD16 * 16, VD = VD16 * 16, DT = VD16 / 2, NW = 4, RING = 4;
  constexpr int KT = 32 * HD * 2, VT = 32 * VD * 2;     // bytes of a tile
  constexpr int KPI = 512 / HD;                         // keys of a copy (1 KB of K)
  constexpr int KW = 8 / KPI, VW = VD / 64;             // copies of a tile a wave issues
  static_assert(HD >= 128 && VD >= 128, "copies of at most four keys");
  extern __shared__ __attribute__((aligned(16))) unsigned char stream_lds[];
  unsigned char* const sV = stream_lds + RING * KT;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lk = lane >> 5;
  const int r = p.r_begin + blockIdx.z;
  int block_x, kvh;
  portion_block(block_x, kvh);
  const int qs = p.q_start[r], n = p.q_start[r + 1] - qs;
  if (n <= 0) return;
  const int start = p.ctx_len[r] - n;
  const int per_block = NW * p.tpw;
  // the last rows of a portion see the most keys and go first
  const int rows_x = SPLIT ? block_x / p.nchunks : block_x;
  const int range = SPLIT ? block_x - rows_x * p.nchunks : 0;
  const int bi = (n + per_block - 1) / per_block - 1 - rows_x;
  if (bi < 0) return;
  const int g = p.nh / p.nkv;
  const int blk_lo = start + bi * per_block, blk_hi = start + min(n, (bi + 1) * per_block) - 1;
  const KeyTiles ts(p, first_key(p, blk_lo), blk_hi);
  int tile_0 = 0, tile_end = ts.count;
  if (SPLIT) {
    tile_0 = range * p.chunk;
    if (tile_0 >= ts.count) return;                    // the block of rows has fewer ranges
    tile_end = min(ts.count, tile_0 + p.chunk);
  }
  const int turns = tile_end - tile_0;
  // the wave's rows
  const int t0 = bi * per_block + wave * p.tpw;
  const int ntok = max(0, min(p.tpw, n - t0));
  const int tok = lr / g, hq = lr - tok * g;
  const bool row_ok = tok < ntok;
  const int trow = qs + (row_ok ? t0 + tok : 0);
  const int pos = start + (row_ok ? t0 + tok : 0);
  const int head = q_head_of(p, kvh, row_ok ? hq : 0);
  // keys [all_lo, all_hi] are seen by every row of the wave.  (What becomes of rows that are not there does not matter; if
  // they made every tile of their wave one to mask, a last block of a few rows, which has the most keys, took 1.5 times as
  // long: 1,500 rows of 8 heads of 256, no ranges, 92 us against 62.)
  const int row_lo = first_key(p, pos);
  const int all_hi = ntok > 0 ? start + t0 : 0x7fffff00;
  const int all_lo = ntok > 0 ? first_key(p, start + t0 + ntok - 1) : 0;
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  const int bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv, last_entry = min(p.max_blocks - 1, blk_hi >> bsh);

  // bytes of a page's key (a page may have 4 GiB and more), and what lies before the key head's part of a page
  const unsigned k_bytes = nkv * HD * 2, v_bytes = (nkv >> p.v_shift) * VD * 2;
  const unsigned char* const k_base = (const unsigned char*)p.kcache + ((size_t)kvh * HD * 2 << bsh);
  const unsigned char* const v_base = (const unsigned char*)p.vcache + ((size_t)(kvh >> p.v_shift) * VD * 2 << bsh);
  // the places of 64 pages, from entry ``first`` of the table on, one a lane; a tile lies in at most two (of 16 keys)
  struct Pages { unsigned lo, hi; int first; };
  auto cover = [&](Pages& e, int key0, const unsigned char* base, unsigned key_bytes) __attribute__((always_inline)) {
    const int first = key0 >> bsh;
    if ((unsigned)(first - e.first) > 60u) {
      e.first = first;
      const uint64_t at = (uint64_t)base + ((uint64_t)(unsigned)max(table[min(first + lane, last_entry)], 0) * key_bytes << bsh);
      e.lo = (unsigned)at;
      e.hi = (unsigned)(at >> 32);
      asm volatile("" : "+v"(e.lo), "+v"(e.hi));        // arrived here, so that no turn waits for loads
    }
  };
  // Copies: K copy c = wave + 4 j is keys KPI c .. of the tile, V copy c 32 channels of the tile's first or last 16 keys.
  // Per copy: its page counted from the tile's first, and a lane's place behind the page's begin (tiles begin at
  // multiples of 32 keys: with pages of up to 32 keys the place does not depend on the tile, with larger ones a tile
  // adds the same for all).  A head's part of a page is at most 4 GiB (stream_takes), so 32 bits hold a place in it.
  unsigned k_off[KW], v_off[VW];
  int k_idx[KW], v_idx[VW];
#pragma unroll
  for (int j = 0; j < KW; j++) {
    const int key = (wave + 4 * j) * KPI, row = key + lane / (64 / KPI);
    k_idx[j] = key >> bsh;
    k_off[j] = (unsigned)((row & bmask) * HD + ((lane % (64 / KPI)) ^ (row & 15)) * 8) * 2;
  }
#pragma unroll
  for (int j = 0; j < VW; j++) {
    const int copy = wave + 4 * j, half = copy / (VD / 32), d = copy % (VD / 32) * 32 + lane / 2;
    const int key = 16 * half + 8 * ((lane & 1) ^ (d >> 3 & 1));
    v_idx[j] = 16 * half >> bsh;
    v_off[j] = (unsigned)((d << bsh) + (key & bmask)) * 2;
  }
  typedef const __attribute__((address_space(1))) void* from_t;
  typedef __attribute__((address_space(3))) void* to_t;
  auto place = [&](const Pages& e, int entry, unsigned off) __attribute__((always_inline)) {
    const uint64_t page = (uint64_t)(unsigned)__builtin_amdgcn_readlane(e.hi, entry) << 32 | (unsigned)__builtin_amdgcn_readlane(e.lo, entry);
    return (from_t)((const unsigned char*)page + off);
  };
  auto copy_k = [&](int slot, int key0, const Pages& e) __attribute__((always_inline)) {
    const int first = (key0 >> bsh) - e.first;
    const unsigned in_page = (unsigned)(key0 & bmask) * (HD * 2);
#pragma unroll
    for (int j = 0; j < KW; j++)
      __builtin_amdgcn_global_load_lds(place(e, first + k_idx[j], k_off[j] + in_page),
                                       (to_t)(stream_lds + slot * KT + (wave + 4 * j) * 1024), 16, 0, 0);
  };
  auto copy_v = [&](int slot, int key0, const Pages& e) __attribute__((always_inline)) {
    const int first = (key0 >> bsh) - e.first;
    const unsigned in_page = (unsigned)(key0 & bmask) * 2;
#pragma unroll
    for (int j = 0; j < VW; j++)
      __builtin_amdgcn_global_load_lds(place(e, first + v_idx[j], v_off[j] + in_page),
                                       (to_t)(sV + slot * VT + (wave + 4 * j) * 1024), 16, 0, 0);
  };

  // (a row that is not there reads another's queries; its scores are masked)
  bf16x8 qf[HD16];
  {
    const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * HD + lk * 8;
#pragma unroll
    for (int ks = 0; ks < HD16; ks++) qf[ks] = *(const bf16x8*)(qr + ks * 16);
  }
  // the values of "tile -1", whose weights are zero, must not be NaN
#pragma unroll
  for (int i = 0; i < VT / 4096; i++) *(f32x4*)(sV + (RING - 1) * VT + (i * 256 + tid) * 16) = f32x4{0.f, 0.f, 0.f, 0.f};
  Pages ek{0, 0, -1000}, ev{0, 0, -1000};
  auto key_of = [&](int t) { return ts.key_of(tile_0 + t); };
  // the copies that turns -4 to -1 would issue (keys of tiles 0 to 3, values of 0 and 1; the waits count on their order)
#pragma unroll 1
  for (int t = -4; t < 0; t++) {
    cover(ek, key_of(t + 4), k_base, k_bytes);
    copy_k(t + 4, key_of(t + 4), ek);
    if (t >= -2) {
      cover(ev, key_of(t + 2), v_base, v_bytes);
      copy_v(t + 2, key_of(t + 2), ev);
    }
  }
  // a lane's weights of a half tile: two a register
  union Weights { bf16x8 v[2]; int w[8]; };
  Weights pb;
#pragma unroll
  for (int e = 0; e < 8; e++) pb.w[e] = 0;
  f32x16 zero;
#pragma unroll
  for (int e = 0; e < 16; e++) zero[e] = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)       // zeros, in 8 bytes of code instead of 128
    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pb.v[0], pb.v[0], zero, 0, 0, 0);
  float m_run = -INFINITY, l_run = 0.f;
  // where a lane reads: its score row's key and the pieces of its half
  const int key_row = 16 * (lr >> 4) + 8 * ((lr >> 2) & 1) + 4 * ((lr >> 3) & 1) + (lr & 3);
  int k_at8[8];
#pragma unroll
  for (int ks = 0; ks < 8; ks++) k_at8[ks] = key_row * HD * 2 + (((ks * 2 + lk) ^ (key_row & 15)) * 16);
  auto k_at = [&](int ks) { return k_at8[ks & 7] + (ks >> 3) * 256; };
  const int v_at = lr * 32 + (lk ^ (lr >> 3 & 1)) * 16;
  // A wait for all but the copies of the last two turns, and a meeting (as text: before a barrier it knows the
  // compiler waits for every load in flight).  The copies of turn t go to the places that turn t - 1 read
  // before its meeting.
#define ZK_STREAM_MEET() asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * (KW + VW)) : "memory")
  ZK_STREAM_MEET();
  f32x16 s = zero;
#pragma unroll
  for (int ks = 0; ks < HD16; ks++)
    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(stream_lds + k_at(ks)), qf[ks], s, 0, 0, 0);
  ZK_STREAM_MEET();                             // every wave has read tile 0, whose place turn 0 writes to
  // What the products so far are multiplied by once a larger maximum was met, right before the next ones
  // (at the end of a turn the branch made the compiler copy all accumulators out and back): in the
  // accumulation registers, where the products keep them.
  float corr = 1.f;
  auto rescale = [&]() __attribute__((always_inline)) {
    if (__builtin_expect(__any(corr != 1.f), 0)) {
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          float x;
          asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\tv_accvgpr_write_b32 %0, %1"
                       : "+a"(o[dt][e]), "=&v"(x)
                       : "v"(corr));
        }
    }
  };
  const float k = CAPPED ? p.k2 : p.k1, c2 = p.c2;
  const float least = k > 0.f ? -INFINITY : k < 0.f ? INFINITY : 0.f;      // times k: the least score
  // A turn goes in quarters: each multiplies the operands that the one before it has read, and turns a part of
  // the scores.  The waves meet before the last quarter, which reads for the next turn's first.
  constexpr int SB = HD16 / 4, PB = VD16 / 4;
  bf16x8 kf[2][SB], vf[2][PB];
  auto read = [&](int t, int b) __attribute__((always_inline)) {
    const unsigned char* kb = stream_lds + ((t + 1) & 3) * KT;
    const unsigned char* vb = sV + ((t + 3) & 3) * VT + v_at;
#pragma unroll
    for (int i = 0; i < SB; i++) kf[b & 1][i] = *(const bf16x8*)(kb + k_at(b * SB + i));
#pragma unroll
    for (int i = 0; i < PB; i++) {
      const int x = b * PB + i;
      vf[b & 1][i] = *(const bf16x8*)(vb + (x / DT) * VD * 32 + (x % DT) * 1024);
    }
  };
  read(0, 0);
  for (int t = 0; t < turns; t++) {
    const int key0 = key_of(t);
    const bool edge = key0 < all_lo || key0 + 31 > all_hi;
    unsigned seen = 0xffffu;
    if (edge) {
      seen = 0;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int key = key0 + 16 * (e >> 3) + 8 * lk + (e & 7);
        const bool ok = row_ok && (key >= row_lo || key < p.keep) && key <= pos;
        seen |= (unsigned)ok << e;
        s[e] = ok ? s[e] : least;
      }
    }
    cover(ek, key_of(t + 4), k_base, k_bytes);
    cover(ev, key_of(t + 2), v_base, v_bytes);
    rescale();
    f32x16 next;
    auto multiply = [&](int b) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < (SB > PB ? SB : PB); i++) {
        if (i < SB) {
          next = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b & 1][i], qf[b * SB + i], b == 0 && i == 0 ? zero : next, 0, 0, 0);
        }
        if (i < PB) {
          const int x = b * PB + i;
          o[x % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[b & 1][i], pb.v[x / DT], o[x % DT], 0, 0, 0);
        }
      }
    };
    // Scores into weights.  Capped: c2 tanh = c2 - 2 c2 r with r = 1 / (2^(k2 dot) + 1), so the largest
    // score has the least r.
    float best = CAPPED ? INFINITY : -INFINITY;
    auto scores = [&](int from) __attribute__((always_inline)) {
#pragma unroll
      for (int e = from; e < from + 8; e++) {
        if (CAPPED) {
          s[e] = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(k * s[e]) + 1.f);
          best = fminf(best, s[e]);
        } else {
          s[e] *= k;
          best = fmaxf(best, s[e]);
        }
      }
    };
    float rs = 0.f, off;
    Weights pn;
    auto weights = [&](int from) __attribute__((always_inline)) {
      bf16x8 w;
#pragma unroll
      for (int e = from; e < from + 8; e++) {
        s[e] = __builtin_amdgcn_exp2f(CAPPED ? fmaf(s[e], -2.f * c2, off) : s[e] + off);
        rs += s[e];
        w[e - from] = (__bf16)s[e];
      }
      pn.v[from / 8] = w;
    };
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    read(t, 1);
    copy_k(t & 3, key_of(t + 4), ek);
    scores(0);
    stream_order<SB + PB, CAPPED ? 5 : 2>();
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    read(t, 2);
    copy_v((t + 2) & 3, key_of(t + 2), ev);
    scores(8);
    stream_order<SB + PB, CAPPED ? 5 : 2>();
    __builtin_amdgcn_sched_barrier(0);
    multiply(2);
    read(t, 3);
    {
      const auto both = __builtin_amdgcn_permlane32_swap(__float_as_int(best), __float_as_int(best), false, false);
      const float a = __int_as_float(both[0]), b = __int_as_float(both[1]);
      best = CAPPED ? fminf(a, b) : fmaxf(a, b);
    }
    const float mt = CAPPED ? fmaf(best, -2.f * c2, c2) : best;
    const float m_new = mt > m_run + 8.f ? mt : m_run;      // the maximum is followed lazily
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    corr = m_new > m_run && m_run > -INFINITY ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.f;     // (nothing to correct yet)
    off = CAPPED ? c2 - m_use : -m_use;
    weights(0);
    stream_order<SB + PB, 5>();
    __builtin_amdgcn_sched_barrier(0);
    ZK_STREAM_MEET();
    multiply(3);
    read(t + 1, 0);
    weights(8);
    stream_order<SB + PB, 4>();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(rs), "+v"(pn.w[0]), "+v"(pn.w[1]), "+v"(pn.w[2]), "+v"(pn.w[3]), "+v"(pn.w[4]), "+v"(pn.w[5]),
                 "+v"(pn.w[6]), "+v"(pn.w[7]));      // here, not on the way without an edge
    if (edge) {
      rs = 0.f;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const bool ok = seen >> e & 1;
        rs += ok ? s[e] : 0.f;
        pn.w[e >> 1] = ok ? pn.w[e >> 1] : pn.w[e >> 1] & (e & 1 ? 0xffff : 0xffff0000);
      }
    }
    {
      const auto both = __builtin_amdgcn_permlane32_swap(__float_as_int(rs), __float_as_int(rs), false, false);
      rs = __int_as_float(both[0]) + __int_as_float(both[1]);
    }
    l_run = l_run * corr + rs;
    m_run = m_new;
    pb = pn;
    s = next;
  }
  rescale();
  {
    const unsigned char* vb = sV + ((turns + 3) & 3) * VT + v_at;
#pragma unroll
    for (int x = 0; x < 2 * DT; x++)
      o[x % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(vb + (x / DT) * VD * 32 + (x % DT) * 1024),
                                                          pb.v[x / DT], o[x % DT], 0, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no copy is on its way into LDS when the block ends
#undef ZK_STREAM_MEET
  if (SPLIT) {
    // a wave's results of its range, as in attn_shared_kernel
    const size_t slot = ((((size_t)blockIdx.z * p.nkv + kvh) * (gridDim.x / p.nchunks) + rows_x) * p.nchunks + range) * NW + wave;
    p.part_ml[slot * 128 + lane] = lk == 0 ? m_run : l_run;
    f32x4* po = (f32x4*)p.part_o + slot * (DT * 4 * 64) + lane;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        po[(dt * 4 + j) * 64] = f32x4{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
    return;
  }
  if (!row_ok) return;
  const float inv = row_factor(p, trow, head, l_run, m_run);
  __bf16* orow = p.out + ((size_t)trow * p.nh + head) * VD;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      bf16x4 w;
#pragma unroll
      for (int i = 0; i < 4; i++) w[i] = (__bf16)(o[dt][4 * j + i] * inv);
      *(bf16x4*)(orow + dt * 32 + 8 * j + 4 * lk) = w;
    }
#endif
}

// Which of a (request, key head)'s blocks a block is.  Blocks go in turn to the 8 XCDs and there to the
// shader engines, 32 in all, so with an even number of them a request the first blocks of all requests
// would share a few and the last ones the others: with requests of uneven lengths, whose last blocks have
// no keys, the first then read half as much again as the average.  They are therefore counted from
// a place of their own.  From one request to the next it moves by 3, through all of them.  From one key
// head to the next it moves by 8, so that the same keys of all heads, which lie side by side in their pages,
// are read by one XCD, on its engines in turn.  (Moved by 1, in launches one after the other over the
// caches of several layers, 64 full requests of 32 heads over 16 of 128 lost a fifth; a launch alone lost 2 %, with
// the same reads, hits and first-level translation misses: which cache or table it is was not found.)
// Measured (us, with the joining launch; from place 0, by 1 further for each head and request, as it is):
// 64 requests of 682 to 8,192 keys, 8 heads over 4 of 256 277, 212, 205; 32 over 16 of 128 510, 450, 401, and
// all of 8,192 keys 737, 901, 745; 64 of 200 to 3,840 keys, 8 over 4 of 256 146, 109, 107.
// An odd number (a window's 17 or 33 blocks) moves them on by itself, and a rotation would undo that (64 requests
// of 200 to 8,000 keys behind a window of 4,096: 153 us without, 168 with).
__device__ __forceinline__ int rotated_block(int blocks) {
  if (blocks % 2) return blockIdx.x;
  return (blockIdx.x + 8 * blockIdx.y + 3 * blockIdx.z) % blocks;
}

// One wave per (request, KV head, 32 keys) for requests that bring one token; a block's four
// waves take 128 neighbouring keys and leave one partial result.  Columns of every tile are
// the g query heads of the KV head (col = lane % 16), rows are keys (first product) or channels
// (second product).  Row 4 a + i of score tile t (a, i = 0..3) is key 8 a + 4 t + i of the 32, so
// that a lane's eight weights belong to eight neighbouring keys, 8 kq + 0..7: its operand of the
// second product, and 16 bytes of a channel of the transposed values.
//
// The time is the way from memory.  A wave has one tile only, so its chain holds one or two waits
// for memory, and blocks are small, so that the CUs get even shares of requests of uneven
// lengths.  Measured (us, with the joining launch, 8 heads over 4 of 256 channels) against blocks
// of four waves with two tiles each one after the other and values in 8-byte pieces: 64 requests
// of 200 to 3,840 keys 146 -> 105 (109 by the order of the blocks alone), of 4,096 keys 192 ->
// 193 (5.6 TB/s), 23 of 130 to 2,000 35.7 -> 27.1, 8 of 4,000 31.6 -> 31.1, 1 of 4,000 13.3 ->
// 11.8.  Eight waves of one tile each: 119, 202, 33.1, 32.9.
template <int HD32, int VD16, bool ONCE>
__global__ __launch_bounds__(256, 4) void attn_decode_kernel(AttnParams p) {
  constexpr int KS = HD32;       // 32-wide steps over head_dim
  constexpr int DT = VD16;       // 16-channel output tiles
  constexpr int NW = 4, SPAN = ATT_DECODE_SPAN;      // waves and keys of a block
  static_assert(SPAN == 32 * NW, "a wave takes 32 keys");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kq = lane >> 4;
  const int r = p.r_begin + blockIdx.z;
  const int kvh = blockIdx.y;
  int block_x = rotated_block(gridDim.x);
  // Where the window is much shorter than the longest context, the grid covers a window's
  // blocks only and counts them from the block the request's window begins in.
  // In front of them come the blocks of the kept first keys, which every request has.
  const int kept_blocks = (p.keep + SPAN - 1) / SPAN;
  if (p.from_window && block_x >= kept_blocks)
    block_x += max(first_key(p, max(p.ctx_len[r] - 1, 0)) / SPAN, kept_blocks) - kept_blocks;
  const int key0 = block_x * SPAN + 32 * wave;
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  constexpr int hd = HD32 * 32, vd = VD16 * 16;
  const int bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv;
  // The pages of the wave's keys are asked for before the request's length is known, beside it:
  // where a key lies follows from the block alone.  A key past the context is masked below; a
  // hole in the table reads page 0, which the caller keeps cleared, and the places of a
  // request's last page behind its last token are cleared too (a masked value still meets a
  // weight of 0 in the second product, and 0 x NaN is NaN).
  int kpage[2], vpage[2];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    kpage[t] = table[min((key0 + 8 * (col >> 2) + 4 * t + (col & 3)) >> bsh, p.max_blocks - 1)];
    vpage[t] = table[min((key0 + 8 * kq + 4 * t) >> bsh, p.max_blocks - 1)];
  }
  const int n = p.q_start[r + 1] - p.q_start[r];
  if (n <= 0) return;
  const int pos = p.ctx_len[r] - 1;
  const int row_lo = first_key(p, pos);
  // a block whose keys all lie past the context or before the window ends here, all its waves
  // alike: the grid is sized for the longest context the caller allows
  if (block_x * SPAN > pos || (block_x * SPAN + SPAN - 1 < row_lo && block_x * SPAN >= p.keep)) return;
  // a wave without keys still meets the others at the barrier
  const bool active = key0 <= pos && (key0 + 31 >= row_lo || key0 < p.keep);
  const int g = p.nh / p.nkv;
  const bool col_ok = col < g;
  const int head = q_head_of(p, kvh, col_ok ? col : 0);
  const int trow = p.q_start[r];

  extern __shared__ __align__(16) unsigned char dec_lds[];
  float* sm_o = (float*)(dec_lds + NW * KS * 64 * sizeof(bf16x8));      // [NW][g][vd]
  constexpr int ML = KS * 64 * sizeof(bf16x8) / sizeof(float);            // a wave's maxima and sums lie where its
  float* sm_ml = (float*)dec_lds;                                         // queries were: [NW] x [16][2], ML apart
  float* so = sm_o + ((size_t)wave * g + col) * vd + 4 * kq;
  float m_run = -INFINITY, l_run = 0.f;
  if (active) {
    // The query operand goes from memory straight to LDS, one 16-byte piece per lane and step.
    // (Columns past the g heads repeat the first head; nothing of them is used.)
    bf16x8(*sq)[64] = (bf16x8(*)[64])dec_lds + wave * KS;
    const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * hd + kq * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(qr + ks * 32),
                                       (__attribute__((address_space(3))) void*)sq[ks], 16, 0, 0);
    bf16x8 kf[2][KS];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int kk = key0 + 8 * (col >> 2) + 4 * t + (col & 3);
      const __bf16* kr = p.kcache + ((((size_t)max(kpage[t], 0) * nkv + kvh) << bsh) + (kk & bmask)) * hd + kq * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) kf[t][ks] = *(const bf16x8*)(kr + ks * 32);
    }
    bf16x8 vf[DT];
    const int vheads = nkv >> p.v_shift, vh = kvh >> p.v_shift;
    const __bf16* va = p.vcache + ((((size_t)max(vpage[0], 0) * vheads + vh) * vd) << bsh) + ((key0 + 8 * kq) & bmask);
    const __bf16* vb = p.vcache + ((((size_t)max(vpage[1], 0) * vheads + vh) * vd) << bsh);
    auto load_v = [&]() {
      if (bsh >= 3) {
#pragma unroll
        for (int dt = 0; dt < DT; dt++) vf[dt] = load_maybe_once<ONCE>((const bf16x8*)(va + ((size_t)(dt * 16 + col) << bsh)));
      } else {         // pages of four keys
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
          const bf16x4 x = *(const bf16x4*)(va + ((size_t)(dt * 16 + col) << bsh)), y = *(const bf16x4*)(vb + ((size_t)(dt * 16 + col) << bsh));
#pragma unroll
          for (int e = 0; e < 4; e++) {
            vf[dt][e] = x[e];
            vf[dt][4 + e] = y[e];
          }
        }
      }
    };
    // Values of 256 channels are asked for after the score products have used up the keys: with
    // both at once a wave has 199 registers, two waves a SIMD, and the CU less on its way (also where blocks are few: 8 requests of
    // 500 keys 11.1 us with the join, beside the keys 12.0; 4 of 3,000 17.1 and 17.8).
    constexpr bool LATE = DT > 8;
    if (!LATE) load_v();
    // the queries are in LDS (the compiler does not know that the reads below depend on them)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][ks], sq[ks][lane], s[t], 0, 0, 0);
    }
    if (LATE) {
      __builtin_amdgcn_sched_barrier(0);
      load_v();
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int key = key0 + 8 * kq + 4 * t + i;
        const float v = score_log2(p, s[t][i]);
        s[t][i] = (col_ok && (key >= row_lo || key < p.keep) && key <= pos) ? v : -INFINITY;
        m_run = fmaxf(m_run, s[t][i]);
      }
    m_run = wave_max16_32(m_run);
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    bf16x8 pb8;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        s[t][i] = __builtin_amdgcn_exp2f(s[t][i] - m_use);
        l_run += s[t][i];
        pb8[4 * t + i] = (__bf16)s[t][i];
      }
    l_run = wave_add16_32(l_run);
    bf16x8 rest8;          // (wide weights) what the rounding left
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) rest8[4 * t + i] = (__bf16)(s[t][i] - (float)pb8[4 * t + i]);
    // the results go to LDS as they come, so that they do not hold registers beside the values
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      f32x4 o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pb8, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      if (p.wide_weights) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], rest8, o, 0, 0, 0);
      if (col_ok) *(f32x4*)(so + dt * 16) = o;
    }
  } else if (col_ok) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++) *(f32x4*)(so + dt * 16) = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the block's waves are joined here, in the order of their keys
  if (col_ok && kq == 0) {
    sm_ml[wave * ML + col * 2] = m_run;
    sm_ml[wave * ML + col * 2 + 1] = l_run;
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < g * vd; idx += NW * 64) {
    const int c = idx / vd, d = idx - c * vd;
    float mw[NW], m = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      mw[w] = sm_ml[w * ML + c * 2];
      m = fmaxf(m, mw[w]);
    }
    float acc = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float e = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - m);
      acc += e * sm_o[((size_t)w * g + c) * vd + d];
      l += e * sm_ml[w * ML + c * 2 + 1];
    }
    const size_t slot = ((size_t)(r - p.r_begin) * p.nh + q_head_of(p, kvh, c)) * p.nchunks + block_x;
    p.part_o[slot * vd + d] = acc;
    if (d == 0) {
      p.part_ml[slot * 2] = m;
      p.part_ml[slot * 2 + 1] = l;
    }
  }
}

// Portions of few rows: 16 rows a block (16 / g tokens of one request times the g query heads of a KV head) on
// 16x16x32 MFMAs, the block's waves take tiles of 32 keys in turn, each with a maximum, a sum and
// results of its own, and are joined in LDS.  Rows are columns of every tile, as in the decode kernel, and
// keys lie in it as there.
//
// What a launch of few rows waits for is one wave's chain: pages, keys, scores, weights, values, the join.  The kernel of 32 rows a
// group walks 5,000 instructions of 32-wide tiles through it and twice the accumulators through
// the join; half the rows a block also double the blocks.  us, that kernel, or tiles shared and joined where these are
// faster, and this: 8 heads over 4 of 256, 7 rows 7.5 and 5.1, 37 11.5 and 5.4, 150 16.2 and 9.3, 512 23.2 and 16.6; 32 over 16 of 128, 37 8.7
// and 4.5, 300 15.5 and 12.4; 16 over 4 of 128, 128 behind 500 keys 17.5 and 12.4.  At 512 rows eight waves a block: 16.1, 30.4 (32 over 16, four
// 23.2), 15.4 (16 over 4, 13.7).
template <int HD32, int VD16, int NW>
__global__ __launch_bounds__(NW * 64, 2) void attn_short_kernel(AttnParams p) {
  constexpr int KS = HD32, DT = VD16, hd = HD32 * 32, vd = VD16 * 16, LD = vd + 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const int r = p.r_begin + blockIdx.z, kvh = blockIdx.y;
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  const int qs = p.q_start[r], n = p.q_start[r + 1] - qs, ctx = p.ctx_len[r];
  const int g = p.nh / p.nkv, tokens = 16 / g;
  const int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * tokens;      // the rows with the most keys first
  if (t0 >= n) return;
  const int start = ctx - n, ntok = min(tokens, n - t0);
  const int tok = col / g, hq = col - tok * g;
  const bool col_ok = tok < ntok;
  const int pos = start + t0 + min(tok, ntok - 1), row_lo = first_key(p, pos);
  const int head = q_head_of(p, kvh, hq), trow = qs + t0 + min(tok, ntok - 1);
  const int key_lo = first_key(p, start + t0), key_hi = start + t0 + ntok - 1;
  const KeyTiles tiles(p, key_lo, key_hi);
  const int bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv, vheads = nkv >> p.v_shift, vh = kvh >> p.v_shift;

  bf16x8 qf[KS];
  const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * hd + kq * 8;
#pragma unroll
  for (int ks = 0; ks < KS; ks++) qf[ks] = *(const bf16x8*)(qr + ks * 32);
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  for (int i = wave; i < tiles.count; i += NW) {
    const int key0 = tiles.key_of(i);
    // (a key behind the block's last: that one's page, which is the request's own.  Asked for a tile ahead, the pages made a wave's
    // registers too many: 512 rows, 8 heads over 4 of 256, 16.7 -> 17.4 us.)
    int kpage[2];
#pragma unroll
    for (int t = 0; t < 2; t++) kpage[t] = table[min(key0 + 8 * (col >> 2) + 4 * t + (col & 3), key_hi) >> bsh];
    const int vpage = table[min(key0 + 8 * kq, key_hi) >> bsh];
    bf16x8 kf[2][KS], vf[DT];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int kk = key0 + 8 * (col >> 2) + 4 * t + (col & 3);
      const __bf16* kr = p.kcache + ((((size_t)max(kpage[t], 0) * nkv + kvh) << bsh) + (kk & bmask)) * hd + kq * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) kf[t][ks] = *(const bf16x8*)(kr + ks * 32);
    }
    const __bf16* va = p.vcache + ((((size_t)max(vpage, 0) * vheads + vh) * vd) << bsh) + ((key0 + 8 * kq) & bmask);
#pragma unroll
    for (int dt = 0; dt < DT; dt++) vf[dt] = *(const bf16x8*)(va + ((size_t)(dt * 16 + col) << bsh));
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][ks], qf[ks], s[t], 0, 0, 0);
    }
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int key = key0 + 8 * kq + 4 * t + e;
        const float v = score_log2(p, s[t][e]);
        s[t][e] = (key >= row_lo || key < p.keep) && key <= pos ? v : -INFINITY;
        top = fmaxf(top, s[t][e]);
      }
    top = fmaxf(m_run, wave_max16_32(top));
    const float m_use = top == -INFINITY ? 0.f : top, corr = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = top;
    float sum = 0.f;
    bf16x8 pb;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float w = __builtin_amdgcn_exp2f(s[t][e] - m_use);
        sum += w;
        pb[4 * t + e] = (__bf16)w;
      }
    l_run = l_run * corr + wave_add16_32(sum);
    if (key0 + 31 > key_hi || key0 < key_lo) {
      // values outside the block's keys may be anything, and a weight of 0 does not make them nothing
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      u4 keep;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int key = key0 + 8 * kq + 2 * e;
        auto in = [&](int k) { return k <= key_hi && (k >= key_lo || k < p.keep); };
        keep[e] = (in(key) ? 0xffffu : 0u) | (in(key + 1) ? 0xffff0000u : 0u);
      }
#pragma unroll
      for (int dt = 0; dt < DT; dt++) vf[dt] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u4, vf[dt]) & keep);
    }
    if (i != wave) {
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] *= corr;
    }
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pb, o[dt], 0, 0, 0);
  }
  // the waves' results: rows of LD floats, then maxima and sums
  extern __shared__ __align__(16) float short_lds[];
  float* ml = short_lds + (size_t)NW * 16 * LD;
  float* so = short_lds + ((size_t)wave * 16 + col) * LD + 4 * kq;
#pragma unroll
  for (int dt = 0; dt < DT; dt++) *(f32x4*)(so + dt * 16) = o[dt];
  if (kq == 0) {
    ml[(wave * 16 + col) * 2] = m_run;
    ml[(wave * 16 + col) * 2 + 1] = l_run;
  }
  __syncthreads();
  // every thread joins four channels of a row at a time
  constexpr int PER_ROW = vd / 4;
  for (int idx = threadIdx.x; idx < 16 * PER_ROW; idx += NW * 64) {
    const int c = idx / PER_ROW, d = idx % PER_ROW * 4, ct = c / g;
    if (ct >= ntok) break;
    float mw[NW], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      mw[w] = ml[(w * 16 + c) * 2];
      m = fmaxf(m, mw[w]);
    }
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float e = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - m);
      acc += e * *(const f32x4*)(short_lds + ((size_t)w * 16 + c) * LD + d);
      l += e * ml[(w * 16 + c) * 2 + 1];
    }
    const int row = qs + t0 + ct, h = q_head_of(p, kvh, c - ct * g);
    const float inv = row_factor(p, row, h, l, m);
    bf16x4 x;
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = (__bf16)(acc[e] * inv);
    *(bf16x4*)(p.out + ((size_t)row * p.nh + h) * vd + d) = x;
  }
}

// One wave per (request, KV head, chunk of 64 keys) for requests that bring one token.
// Columns of every tile are the g query heads of the KV head (col = lane % 16), rows are
// keys (first product) or channels (second product).
//
// For callers whose limit is a long context (ATT_DECODE_LONG_FROM keys a request or more): blocks of
// 256 keys leave half as many partial results as those of 128, whose writing and reading are what
// is left to save once every CU has many blocks.  Figures at decode_in_long_blocks.
template <int HD32, int VD16, bool ONCE>
__global__ __launch_bounds__(256, 2) void attn_decode_long_kernel(AttnParams p) {
  constexpr int KS = HD32;       // 32-wide steps over head_dim
  constexpr int DT = VD16;       // 16-channel output tiles
  // Keys of a wave (64) and of a block.  A number of the launch: with a constant the compiler orders a
  // wave's two tiles otherwise, which loses where the chip is full (us, 64 requests of 4,096 keys, 8 heads over 4
  // of 256 187.2 against 186.1; 8 behind a window of 2,048, 16 over 4 of 128 15.7 against 15.3) and gains with few
  // blocks (8 of 4,096 keys, 8 over 4 of 256 35.8 against 36.7).
  const int wave_keys = p.chunk, span = 4 * wave_keys;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kq = lane >> 4;
  const int r = p.r_begin + blockIdx.z;
  const int kvh = blockIdx.y;
  // Where the window is much shorter than the longest context, the grid covers a window's
  // blocks only and counts them from the block the request's window begins in.
  int block_x = rotated_block(gridDim.x);
  // In front of them come the blocks of the kept first keys, which every request has.
  const int kept_blocks = (p.keep + span - 1) / span;
  if (p.from_window && block_x >= kept_blocks)
    block_x += max(first_key(p, max(p.ctx_len[r] - 1, 0)) / span, kept_blocks) - kept_blocks;
  const int chunk = block_x * 4 + wave;
  const int* table = p.block_table + (size_t)r * p.max_blocks;
  constexpr int hd = HD32 * 32, vd = VD16 * 16;
  const int bsh = p.bs_shift, bmask = p.bs - 1, nkv = p.nkv;
  // The pages of the chunk's (up to two) tiles are asked for before the request's length is
  // known, beside it: where a key lies follows from the chunk alone.  A key past the context is
  // masked below; a hole in the table reads page 0, which the caller keeps cleared, and the
  // places of a request's last page behind its last token are cleared too (a masked value
  // still meets a weight of 0 in the second product, and 0 x NaN is NaN).
  int kpage[2][2], vpage[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int k0 = chunk * wave_keys + 32 * i;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      kpage[i][t] = table[min((k0 + 16 * t + col) >> bsh, p.max_blocks - 1)];
      vpage[i][t] = table[min((k0 + 16 * t + 4 * kq) >> bsh, p.max_blocks - 1)];
    }
  }
  const int n = p.q_start[r + 1] - p.q_start[r];
  if (n <= 0) return;
  const int pos = p.ctx_len[r] - 1;
  const int row_lo = first_key(p, pos);
  // a block whose four chunks all lie past the context or before the window ends here, all
  // its waves alike: the grid is sized for the longest context the caller allows
  const int first_chunk = block_x * 4;
  if (first_chunk * wave_keys > pos ||
      (first_chunk * wave_keys + span - 1 < row_lo && first_chunk * wave_keys >= p.keep)) return;
  const int key_lo = chunk * wave_keys < p.keep ? chunk * wave_keys : max(row_lo, chunk * wave_keys);
  const int key_hi = min(pos, chunk * wave_keys + wave_keys - 1);
  const bool active = key_lo <= key_hi;          // a wave without keys still meets the others at the barrier
  const int g = p.nh / p.nkv;
  const bool col_ok = col < g;
  const int head = q_head_of(p, kvh, col_ok ? col : 0);
  const int trow = p.q_start[r];

  // the query operand waits in LDS (one 16-byte piece per lane and step), not in registers
  __shared__ bf16x8 sq[4][KS][64];
  {
    const __bf16* qr = p.q + (size_t)trow * p.q_stride + (size_t)head * hd + kq * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      bf16x8 t;
      if (col_ok) t = *(const bf16x8*)(qr + ks * 32);
      else
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] = (__bf16)0.f;
      sq[wave][ks][lane] = t;
    }
  }
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int key0 = chunk * wave_keys + 32 * i;
    if (!active || 32 * i >= wave_keys || key0 > key_hi || key0 + 31 < key_lo) continue;
    bf16x8 kf[2][KS];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int kk = key0 + 16 * t + col;
      const int page = max(kpage[i][t], 0);
      const __bf16* kr = p.kcache + ((((size_t)page * nkv + kvh) << bsh) + (kk & bmask)) * hd + kq * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) kf[t][ks] = *(const bf16x8*)(kr + ks * 32);
    }
    bf16x8 vf[DT];
    {
      const int ka = key0 + 4 * kq, kb = key0 + 16 + 4 * kq;
      const int pa = max(vpage[i][0], 0), pb = max(vpage[i][1], 0);
      const __bf16* va_base = p.vcache + ((((size_t)pa * (nkv >> p.v_shift) + (kvh >> p.v_shift)) * vd) << bsh) + (ka & bmask);
      const __bf16* vb_base = p.vcache + ((((size_t)pb * (nkv >> p.v_shift) + (kvh >> p.v_shift)) * vd) << bsh) + (kb & bmask);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const int d = dt * 16 + col;
        const bf16x4 va = load_maybe_once<ONCE>((const bf16x4*)(va_base + ((size_t)d << bsh)));
        const bf16x4 vb = load_maybe_once<ONCE>((const bf16x4*)(vb_base + ((size_t)d << bsh)));
#pragma unroll
        for (int e = 0; e < 4; e++) {
          vf[dt][e] = va[e];
          vf[dt][4 + e] = vb[e];
        }
      }
    }
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][ks], sq[wave][ks][lane], s[t], 0, 0, 0);
    }
    float mt = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int key = key0 + 16 * t + 4 * kq + i;
        float v = score_log2(p, s[t][i]);
        v = (col_ok && (key >= row_lo || key < p.keep) && key <= key_hi) ? v : -INFINITY;
        s[t][i] = v;
        mt = fmaxf(mt, v);
      }
    mt = wave_max16_32(mt);
    const float m_new = fmaxf(m_run, mt);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
    float rs = 0.f;
    bf16x8 pb8;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float pe = __builtin_amdgcn_exp2f(s[t][i] - m_use);
        rs += pe;
        pb8[4 * t + i] = (__bf16)pe;
        s[t][i] = pe;
      }
    rs = wave_add16_32(rs);
    l_run = l_run * corr + rs;
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      o[dt] *= corr;
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pb8, o[dt], 0, 0, 0);
    }
    if (p.wide_weights) {
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) pb8[4 * t + i] = (__bf16)(s[t][i] - (float)pb8[4 * t + i]);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pb8, o[dt], 0, 0, 0);
    }
  }
  // the block's four chunks are joined here, in chunk order: one partial result per 256 keys
  extern __shared__ float dyn[];
  float* sm_ml = dyn;                 // [4][16][2]
  float* sm_o = dyn + 4 * 16 * 2;     // [4][g][vd]
  if (col_ok) {
    if (kq == 0) {
      sm_ml[(wave * 16 + col) * 2] = m_run;
      sm_ml[(wave * 16 + col) * 2 + 1] = l_run;
    }
    float* so = sm_o + ((size_t)wave * g + col) * vd;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) *(f32x4*)(so + dt * 16 + 4 * kq) = o[dt];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < g * vd; idx += 256) {
    const int c = idx / vd, d = idx - c * vd;
    float mw[4], m = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      mw[w] = sm_ml[(w * 16 + c) * 2];
      m = fmaxf(m, mw[w]);
    }
    float acc = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float e = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - m);
      acc += e * sm_o[((size_t)w * g + c) * vd + d];
      l += e * sm_ml[(w * 16 + c) * 2 + 1];
    }
    const size_t slot = ((size_t)(r - p.r_begin) * p.nh + q_head_of(p, kvh, c)) * p.nchunks + block_x;
    p.part_o[slot * vd + d] = acc;
    if (d == 0) {
      p.part_ml[slot * 2] = m;
      p.part_ml[slot * 2 + 1] = l;
    }
  }
}

// One pair of sizes.  what: 0 decoded tokens on 32-wide tiles, 1 pairs of groups a block, 2 a group a block,
// 3 shared tiles with four waves, 4 with eight, 5 with four and the keys in ranges, 6 decoded tokens
// on 16-wide tiles (keys in whole 32s), 7 the same in blocks of 256 keys.
enum AttnWhat { ATT_DECODE_WIDE, ATT_PAIRS, ATT_GROUPS, ATT_SHARED4, ATT_SHARED8, ATT_RANGES, ATT_DECODE, ATT_DECODE_LONG, ATT_SHORT,
                // values past the caches (values_past_caches)
                ATT_DECODE_ONCE, ATT_DECODE_LONG_ONCE };

template <int HD16, int VD16, int NW, bool SPLIT>
static int launch_shared_one(const AttnParams& p, dim3 grid, hipStream_t s) {
  constexpr int HD = HD16 * 16, VD = VD16 * 16;
  constexpr size_t lds = ((size_t)2 * 32 * (HD + 8) + (size_t)2 * VD * (32 + 8)) * sizeof(__bf16);
  static bool prepared = false;
  if (!prepared) {
    if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)attn_shared_kernel<HD16, VD16, NW, SPLIT>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return zk_fail("zk_attention_bf16: the shared-tile kernel's LDS buffers were refused");
    prepared = true;
  }
  attn_shared_kernel<HD16, VD16, NW, SPLIT><<<grid, NW * 64, lds, s>>>(p);
  return zk_launch_status("zk_attention_bf16 (shared tiles)");
}

// What attn_stream_kernel takes of the launches of four groups a block.
static inline bool stream_takes(int hd, int vd, int bs, int wide_weights) {
  return (hd == 128 || hd == 256) && (vd == 128 || vd == 256) && bs >= 16 && bs <= (1 << 23) && !wide_weights;
}

template <int HD16, int VD16, bool SPLIT>
static int launch_stream(const AttnParams& p, dim3 grid, hipStream_t s) {
  constexpr size_t lds = (size_t)4 * 32 * (HD16 + VD16) * 16 * sizeof(__bf16);
  const auto kernel = p.softcap > 0.f ? attn_stream_kernel<HD16, VD16, SPLIT, true> : attn_stream_kernel<HD16, VD16, SPLIT, false>;
  static std::atomic<bool> prepared[2];
  if (lds > 64 * 1024 && !prepared[p.softcap > 0.f]) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return zk_fail("zk_attention_bf16: the stream kernel's LDS was refused");
    prepared[p.softcap > 0.f] = true;
  }
  kernel<<<grid, 256, lds, s>>>(p);
  return zk_launch_status("zk_attention_bf16 (tiles copied ahead)");
}

// the maxima and sums, and the results, of the four waves of a block of 256 keys
static inline size_t decode_long_lds(int g, int vd) { return (4 * 16 * 2 + (size_t)4 * g * vd) * sizeof(float); }

template <int HD16, int VD16>
static int launch_sizes(int what, const AttnParams& p, dim3 grid, hipStream_t s) {
  // the join of a portion's four waves needs [4][32][2] + [2][ceil(vd/32) * 16][64] floats of LDS
  const size_t join = (4 * 32 * 2 + (size_t)2 * ((p.vd + 31) / 32) * 16 * 64) * sizeof(float);
  switch (what) {
    case ATT_DECODE_WIDE: attn_mfma_kernel<HD16, VD16, true, false><<<grid, 256, 0, s>>>(p); break;
    case ATT_PAIRS: attn_mfma_kernel<HD16, VD16, false, true><<<grid, 256, join, s>>>(p); break;
    case ATT_GROUPS: attn_mfma_kernel<HD16, VD16, false, false><<<grid, 256, join, s>>>(p); break;
    case ATT_SHARED4:
      if constexpr (HD16 >= 8 && VD16 >= 8)
        if (stream_takes(p.hd, p.vd, p.bs, p.wide_weights)) return launch_stream<HD16, VD16, false>(p, grid, s);
      return launch_shared_one<HD16, VD16, 4, false>(p, grid, s);
    case ATT_SHARED8:
      if constexpr (HD16 <= 8 && VD16 <= 8) return launch_shared_one<HD16, VD16, 8, false>(p, grid, s);
      else return zk_fail("zk_attention_bf16: eight waves a block take head sizes up to 128");
    case ATT_RANGES:
      if constexpr (HD16 >= 8 && VD16 >= 8)
        if (stream_takes(p.hd, p.vd, p.bs, p.wide_weights)) return launch_stream<HD16, VD16, true>(p, grid, s);
      return launch_shared_one<HD16, VD16, 4, true>(p, grid, s);
    case ATT_SHORT:
      if constexpr (HD16 % 2 == 0) {
        constexpr size_t lds = ((size_t)ATT_SHORT_WAVES * 16 * (VD16 * 16 + 4) + ATT_SHORT_WAVES * 32) * sizeof(float);
        static std::atomic<bool> prepared{false};
        if (lds > 64 * 1024 && !prepared) {
          if (hipFuncSetAttribute((const void*)attn_short_kernel<HD16 / 2, VD16, ATT_SHORT_WAVES>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return zk_fail("zk_attention_bf16: the LDS of the kernel of few rows was refused");
          prepared = true;
        }
        attn_short_kernel<HD16 / 2, VD16, ATT_SHORT_WAVES><<<grid, ATT_SHORT_WAVES * 64, lds, s>>>(p);
        break;
      } else {
        return zk_fail("zk_attention_bf16: the narrow tiles take keys in whole 32s");
      }
    case ATT_DECODE:
    case ATT_DECODE_ONCE:
      if constexpr (HD16 % 2 == 0) {
        const size_t lds = (size_t)4 * (p.nh / p.nkv) * p.vd * sizeof(float) + (size_t)4 * (HD16 / 2) * 64 * sizeof(bf16x8);
        static std::atomic<bool> prepared{false};
        if (lds > 64 * 1024 && !prepared) {      // 16 heads a KV head with values of 256 channels: 96 KB
          if (hipFuncSetAttribute((const void*)attn_decode_kernel<HD16 / 2, VD16, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  96 * 1024) != hipSuccess ||
              hipFuncSetAttribute((const void*)attn_decode_kernel<HD16 / 2, VD16, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  96 * 1024) != hipSuccess)
            return zk_fail("zk_attention_bf16: the decode kernel's LDS was refused");
          prepared = true;
        }
        if (what == ATT_DECODE_ONCE) attn_decode_kernel<HD16 / 2, VD16, true><<<grid, 256, lds, s>>>(p);
        else attn_decode_kernel<HD16 / 2, VD16, false><<<grid, 256, lds, s>>>(p);
        break;
      } else {
        return zk_fail("zk_attention_bf16: the narrow tiles take keys in whole 32s");
      }
    case ATT_DECODE_LONG:
    case ATT_DECODE_LONG_ONCE:
      if constexpr (HD16 % 2 == 0) {
        if (what == ATT_DECODE_LONG_ONCE) attn_decode_long_kernel<HD16 / 2, VD16, true><<<grid, 256, decode_long_lds(p.nh / p.nkv, p.vd), s>>>(p);
        else attn_decode_long_kernel<HD16 / 2, VD16, false><<<grid, 256, decode_long_lds(p.nh / p.nkv, p.vd), s>>>(p);
        break;
      } else {
        return zk_fail("zk_attention_bf16: the narrow tiles take keys in whole 32s");
      }
    default: return zk_fail("zk_attention_bf16: unknown kernel");
  }
  return zk_launch_status("zk_attention_bf16");
}

// attention_bf16_uneven.hip
int attn_launch_uneven(int what, const AttnParams& p, dim3 grid, hipStream_t s);

#endif  // ZSE_ACT_BF16
