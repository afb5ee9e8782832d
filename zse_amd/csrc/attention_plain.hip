// Plain paged attention: one wave per (token, query head), every token of the
// step alike, whether it is a decoded token or one of a prompt portion.  Keys
// and values come only from the cache, through the request's block table.
//
//   s_j = softcap((q . k_j) * scale),   j in [lo, pos],  lo = max(0, pos - window + 1)
//   o   = sum_j softmax(s)_j v_j
//
// With ``chunk`` instead of a window, lo = floor(pos / chunk) * chunk: a query sees the keys of
// its own chunk of positions, counted from position 0.  ``unit_sink``: a sink of score 0 that has
// no value joins the denominator, exp(s_j) / (1 + sum exp(s)).  ``keep``: beside its window a query
// sees the sequence's first ``keep`` keys, at their own positions.  ``gate``: a number z per token and
// query head; the head's output is multiplied by sigmoid(z).
//
// Keys are visited in tiles of 64 aligned to absolute positions, with a
// running maximum and sum, so the order of every sum depends on the token's
// position alone, not on how the step was cut.  Scores, softmax and the output
// sum are float.  The reference's decode kernel has the same shape of work
// (orchestrator/kernels.py:524-671: one block per (sequence, head), block
// table walk, three passes in shared memory); its prefill kernel reads
// contiguous K/V instead (:859-958) and never applies a window (:883).
#include "common.h"

#include <algorithm>
#include <climits>

#define AP_MAX_HD 256

// MAXD: the most channels a head's queries, keys and values have (256, or 1024 for the wide rows
// of a latent cache).  sinks (may be null): float [nh], exp(sink) joins a head's denominator with
// no key and no value.  v_in_k: a value is the first vd channels of its key (no value cache).
template <int MAXD>
__global__ __launch_bounds__(64) void attention_plain_kernel(
    const act_t* __restrict__ q, int q_stride, const act_t* __restrict__ kcache,
    const act_t* __restrict__ vcache, const int* __restrict__ block_table, int max_blocks,
    const int* __restrict__ req_of_token, const int* __restrict__ positions,
    act_t* __restrict__ out, int nh, int nkv, int hd, int vd, int bs, float scale, float softcap,
    int window, int v_transposed, const float* __restrict__ v_freq, int v_interleaved,
    const float* __restrict__ sinks, int v_in_k, int chunk, int unit_sink, int keep, const act_t* __restrict__ gate,
    int gate_ld) {
  __shared__ float sq[MAXD];
  __shared__ float sp[64];
  __shared__ int spage[64];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int pos = positions[t];
  act_t* o = out + ((size_t)t * nh + h) * vd;
  if (pos < 0) {  // padding row
    for (int d = lane; d < vd; d += 64) o[d] = from_f32<act_t>(0.f);
    return;
  }
  const int r = req_of_token[t];
  const int kvh = h / (nh / nkv);
  const int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : chunk > 0 ? pos / chunk * chunk : 0;
  const int* table = block_table + (size_t)r * max_blocks;
  const act_t* qr = q + (size_t)t * q_stride + (size_t)h * hd;
  for (int d = lane; d < hd; d += 64) sq[d] = to_f32(qr[d]);
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  float acc[MAXD / 64] = {};
  // tiles of the kept first keys, then those from the window's first key on
  const int lo_tile = lo / 64 * 64, kept_tiles = (keep + 63) / 64 * 64;
  for (int j0 = keep > 0 ? 0 : lo_tile; j0 <= pos; j0 = (j0 + 64 >= kept_tiles && j0 + 64 < lo_tile) ? lo_tile : j0 + 64) {
    const int j = j0 + lane;
    const bool valid = (j >= lo || j < keep) && j <= pos;
    float s = -INFINITY;
    int page = -1;
    if (valid) {
      page = table[j / bs];
      const act_t* kr = kcache + (((size_t)page * nkv + kvh) * bs + (j % bs)) * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; d++) dot = fmaf(sq[d], to_f32(kr[d]), dot);
      s = dot * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
    }
    const float m_new = fmaxf(m, wave_max_whole(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);  // m = -inf on the first tile: exp(-inf) = 0
    l = l * corr + wave_sum_whole(p);
    m = m_new;
    __syncthreads();
    sp[lane] = p;
    spage[lane] = page;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < MAXD / 64; c++) {
      const int d = lane + c * 64;
      if (d < vd) {
        float a = acc[c] * corr;
        for (int jj = 0; jj < 64; jj++) {
          const int pg = spage[jj];
          if (pg < 0) continue;
          const size_t off = (j0 + jj) % bs;
          act_t v;
          if (v_in_k) {
            v = kcache[(((size_t)pg * nkv + kvh) * bs + off) * hd + d];
          } else {
            const size_t head_base = ((size_t)pg * nkv + kvh) * bs * vd;
            v = v_transposed ? vcache[head_base + (size_t)d * bs + off] : vcache[head_base + off * vd + d];
          }
          a = fmaf(sp[jj], to_f32(v), a);
        }
        acc[c] = a;
      }
    }
  }
  if (sinks != nullptr || unit_sink) {
    const float sk = sinks != nullptr ? sinks[h] : 0.f;
    const float m_new = fmaxf(m, sk);
    const float corr = expf(m - m_new);
    l = l * corr + expf(sk - m_new);
#pragma unroll
    for (int c = 0; c < MAXD / 64; c++) acc[c] *= corr;
  }
  float inv = 1.f / l;
  if (gate != nullptr) inv *= 1.f / (1.f + expf(-to_f32(gate[(size_t)t * gate_ld + h])));
  if (v_freq == nullptr) {
#pragma unroll
    for (int c = 0; c < MAXD / 64; c++) {
      const int d = lane + c * 64;
      if (d < vd) o[d] = from_f32<act_t>(acc[c] * inv);
    }
    return;
  }
  // values were turned by their own positions when they were stored: the sum is turned back
  // by the query's position, pair m by -pos * v_freq[m]
  __syncthreads();
#pragma unroll
  for (int c = 0; c < MAXD / 64; c++) {
    const int d = lane + c * 64;
    if (d < vd) sq[d] = acc[c] * inv;
  }
  __syncthreads();
  const int half = vd / 2;
  for (int m2 = lane; m2 < half; m2 += 64) {
    float sn, cs, ra, rb;
    sincosf(-(float)pos * v_freq[m2], &sn, &cs);
    const int ia = v_interleaved ? 2 * m2 : m2, ib = v_interleaved ? 2 * m2 + 1 : m2 + half;
    rotate_pair(sq[ia], sq[ib], sn, cs, ra, rb);
    o[ia] = from_f32<act_t>(ra);
    o[ib] = from_f32<act_t>(rb);
  }
}

#if !ZSE_ACT_BF16
// The 32-bit path's attention on the 32-bit matrix cores (16x16x4), for heads of whole 16-byte
// pieces.  Sixteen rows, the query heads of one key head times as many neighbouring tokens of
// one request as fit, share every key and value that is read.
//
// Scores are taken as keys x queries: lane l then holds, for the query l % 16, the keys
// 16 f + 4 (l / 16) + e of a tile of 64 (f, e = 0..3), which is just what the second product,
// values x weights, wants as its operand, so nothing is moved between lanes but the maxima and
// sums over the four lanes of a query.  Both products take their sums in the order of the
// registers (k = 4 (l / 16) + e of each piece of 16), keys and values come as 16 bytes a lane.
//
// The keys' tiles of 64, aligned to absolute positions, go round-robin over the block's waves
// (tile j / 64 to wave j / 64 % WAVES); each keeps a running maximum and sum, and the waves'
// sums are joined in their order.  So a row's sums are cut and ordered by its position alone,
// however the step was cut, and rows that share a block do not touch each other: a key that a
// row does not see has weight 0 there, and a tile with such a key and a value that is not finite
// is taken value by value, in the order in which the matrix cores take them.
//
// Bound by the latency of the loads for few tokens and by the matrix cores for many.  Measured
// (us; before: a wave per token and head whose lanes each walked a key's row):
//   303 tokens, 8 heads of 128, contexts of 300 and three of 50 to 700: 852 -> 38.
//   One token, 8 heads over 2 of 128: 1 key 12.4 -> 9.3, 100 keys 57 -> 15, 4,000 keys 2,111 -> 130; 4 heads
//   of 16: 6.9 -> 8.5, 26 -> 11, 884 -> 83; 8 over 4 of 256: 21.7 -> 22.7, 109 -> 27, 6,260 -> 458.  (Heads of up
//   to 64 are slower than before below about ten keys, of 256 below three.)
//
// PACK: launches of many short runs (a step of many requests with a few tokens each).  A run that has a block to itself
// leaves most of its waves without a tile, and with one head a key head most blocks are without a run.  1,000 requests of
// 3 tokens (us; key by key, a run a block, packed): 8 heads of 128 over 2 68, 174, 92; 8 of 64 41, 480, 67; 8 over 4
// of 256 136, 484, 172.  1,500 tokens behind a window of 64, 8 of 64: 99, 159, 50.
//
// ASK: keys and values are asked for without a condition and a piece of 16 ahead of their products (the first values in
// front of the weights), and pieces that no row sees are passed over in the first product too.  For key heads of 65 to
// 128 channels, 8 heads over 2 of 128 (us; keys alone without a condition, and each piece at its turn; both ahead): 303 tokens,
// 300 of them a prompt, 34.9 and 32.5; one token with 4,000 keys 140 and 130; 64 requests of 100 to 3,250 keys 138 and
// 108; 1,000 requests of 3 tokens 498 and 381, with 3 keys 93 and 95; 1,500 tokens 137 and 130, behind a window of 64 61 and 53;
// one token with 1 key 9.4 and 9.3, with 300 or 500 keys, a tile for each wave, 19.5 and 19.9, 23.1 and 23.4 (the keys of pieces behind the
// last are waited for: not asked for under a condition, which costs 303 tokens 26 us).  Not
// for smaller key heads (8 over 4 of 64, 4,000 keys: 92 and 94; with values of 128 34 and 65: the registers
// do not hold both); of 256 the loads in flight do not fit (446 -> 472).
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The value of another lane of the row of 16: 0x110 + n: of the lane n before (none: what is there for it), 0x120 + n: in a circle
template <int WHICH>
__device__ __forceinline__ int row_lane(int v, int none) {
  return __builtin_amdgcn_update_dpp(none, v, WHICH, 0xf, 0xf, false);
}

template <int MAXD, int WAVES, bool ASK, bool PACK>
__global__ __launch_bounds__(64 * WAVES) void attention_f32_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ kcache, const float* __restrict__ vcache,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ req_of_token,
    const int* __restrict__ positions, float* __restrict__ out, int T, int nh, int nkv, int hd, int vd, int bs,
    float scale, float softcap, int window, const float* __restrict__ v_freq, int v_interleaved,
    const float* __restrict__ sinks, int chunk, int unit_sink, int keep, const float* __restrict__ gate, int gate_ld) {
  constexpr int QC = MAXD / 16, VC = MAXD / 64;       // pieces of 16 channels of a query, of 64 of a value
  // A piece of 16 keys that no row of the run sees has weight 0 everywhere: its products are passed over
  // where that was measured to pay (a branch keeps the next piece's loads from being asked for early).
  constexpr bool PASS_VALUES = MAXD <= 128;
  __shared__ float s_acc[WAVES][16][MAXD];
  __shared__ float s_m[WAVES][16], s_l[WAVES][16];
  const int group = nh / nkv, chunks = (group + 15) / 16;
  const int kvh = blockIdx.y / chunks, h0 = blockIdx.y % chunks * 16;       // first of the block's heads in the group
  const int gh = min(16, group - h0), tb = max(1, 16 / group);              // heads, tokens of a block
  const int t0 = blockIdx.x * tb, n_tok = min(tb, T - t0);
  // Lane i of every row of 16 looks at the block's token i, so one wait finds all runs of neighbouring tokens of one
  // request; padding rows (position < 0) belong to none.
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, qd = lane >> 4;
  const int my_pos = positions[t0 + min(r, n_tok - 1)], my_req = req_of_token[t0 + min(r, n_tok - 1)];
  const bool my_live = r < n_tok && my_pos >= 0;
  const unsigned live = (unsigned)__ballot(my_live) & 0xffffu;
  const int req_before = row_lane<0x111>(my_req, -1);          // of the lane before
  unsigned starts = (unsigned)__ballot(my_live && (!(live << 1 >> r & 1) || my_req != req_before)) & 0xffffu;
  if (blockIdx.z == 0 && live != (1u << n_tok) - 1)
    for (int i = 0; i < n_tok; i++)
      if (!(live >> i & 1))
        for (int x = threadIdx.x; x < gh * vd; x += 64 * WAVES)
          out[((size_t)(t0 + i) * nh + (size_t)kvh * group + h0) * vd + x] = 0.f;
  // a run's keys, at its last lane: from the lowest that a token of it sees to its highest position
  auto lowest = [&](int pos) { return window > 0 ? max(pos - window + 1, 0) : chunk > 0 ? pos / chunk * chunk : 0; };
  const int my_run = __popc(starts & ((2u << r) - 1));
  int run_lo = my_live ? lowest(my_pos) : INT_MAX, run_hi = my_live ? my_pos : -1;
  auto widen = [&](int run, int lo, int hi) {
    run_lo = run == my_run ? min(run_lo, lo) : run_lo;
    run_hi = run == my_run ? max(run_hi, hi) : run_hi;
  };
  widen(row_lane<0x111>(my_run, -1), row_lane<0x111>(run_lo, 0), row_lane<0x111>(run_hi, 0));
  widen(row_lane<0x112>(my_run, -1), row_lane<0x112>(run_lo, 0), row_lane<0x112>(run_hi, 0));
  widen(row_lane<0x114>(my_run, -1), row_lane<0x114>(run_lo, 0), row_lane<0x114>(run_hi, 0));
  widen(row_lane<0x118>(my_run, -1), row_lane<0x118>(run_lo, 0), row_lane<0x118>(run_hi, 0));
  // With PACK as many waves as the longest run has tiles take a run (a power of two), and a block takes as many runs
  // at once as it has room for.  A tile's place in the join's order stays its number modulo WAVES.
  int team = WAVES;
  if (PACK) {
    int most = my_live ? run_hi / 64 + 1 - (keep > 0 ? 0 : run_lo / 64) : 0;
    most = max(most, row_lane<0x128>(most, 0));
    most = max(most, row_lane<0x124>(most, 0));
    most = max(most, row_lane<0x122>(most, 0));
    most = __builtin_amdgcn_readfirstlane(max(most, row_lane<0x121>(most, 0)));
    team = most <= 1 ? 1 : most <= 2 ? 2 : most <= 4 ? 4 : WAVES;
  }
  const int runs = __popc(starts);
  for (int z0 = blockIdx.z * (WAVES / team); z0 < runs; z0 += gridDim.z * (WAVES / team)) {
    const bool active = z0 + wave / team < runs;              // a wave without a run still meets the others at the barriers
    unsigned from = starts;
    for (int z = active ? z0 + wave / team : 0; z > 0; z--) from &= from - 1;
    const int run_first = __builtin_ctz(from);
    // the run ends before the next one, before a padding row or with the block's tokens
    const int run_last = __builtin_ctz((from & (from - 1)) | (~live & (~0u << run_first)) | 1u << n_tok) - 1;
    const int run_rows = (run_last - run_first + 1) * gh;
    const int seg_lo = __builtin_amdgcn_readlane(run_lo, run_last), seg_hi = active ? __builtin_amdgcn_readlane(run_hi, run_last) : -1;
    const int row = min(r, run_rows - 1);              // rows past the last repeat it and are not stored
    const int tok = t0 + run_first + row / gh, head = kvh * group + h0 + row % gh;
    const int pos = __shfl(my_pos, run_first + row / gh), lo = lowest(pos);
    const int* table = block_table + (size_t)__builtin_amdgcn_readlane(my_req, run_first) * max_blocks;
    // what the join alone needs waits in a vector register: the loop wants more scalar ones than there are
    int join = run_first | (active ? run_rows : 0) << 8 | team << 16;
    asm volatile("" : "+v"(join));

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 qf[QC];
#pragma unroll
    for (int c = 0; c < QC; c++) {
      const int d = 16 * c + 4 * qd;
      qf[c] = d < hd ? *(const f32x4*)(q + (size_t)tok * q_stride + (size_t)head * hd + d) : zero;
    }
    float m = -INFINITY, l = 0.f;
    f32x4 acc[VC][4];            // [c][e][i]: channel 64 c + 16 qd + 4 i + e of the lane's query
#pragma unroll
    for (int c = 0; c < VC; c++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[c][e] = zero;

    const int lo_tile = seg_lo / 64, kept_tiles = (keep + 63) / 64;
    const int tile0 = keep > 0 ? 0 : lo_tile, tile1 = (seg_hi + 64) / 64;
    auto first_tile = [&](int members) { return tile0 + ((wave - tile0) & (members - 1)); };       // the wave's first tile
    for (int tile = first_tile(team); tile < tile1; tile += WAVES) {
      if (tile >= kept_tiles && tile < lo_tile) continue;
      const int j0 = tile * 64;
      // the cache row of key 16 f + r; a key that no row of the run sees is never read (row -1)
      long long at[4];
#pragma unroll
      for (int f = 0; f < 4; f++) {
        const int j = j0 + 16 * f + r;
        at[f] = -1;
        if (j <= seg_hi && (j >= seg_lo || j < keep)) {
          const int page = table[j / bs];
          if (page >= 0) at[f] = ((long long)page * nkv + kvh) * bs + j % bs;
        }
      }
      auto unseen = [&](int f) { return j0 + 16 * f > seg_hi || (j0 + 16 * f + 15 < seg_lo && j0 + 16 * f >= keep); };
      // ASK: a piece's keys and values are asked for a piece ahead, the first values in front of the weights.  They are
      // held in front of the branches that pass over unseen pieces, behind which the compiler would move their loads.
      f32x4 s[4], k_ahead[2][QC], v_ahead[2][4][VC];
      bool has[2][4];              // the key of a value asked for is in the cache (with PACK found out again: the registers do not hold it)
      auto ask_keys = [&](int f) {
#pragma unroll
        for (int c = 0; c < QC; c++)
          k_ahead[f & 1][c] = *(const f32x4*)(kcache + (size_t)max(at[f], 0LL) * hd + min(16 * c + 4 * qd, hd - 4));
      };
      auto ask_values = [&](int f) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const long long va = __shfl(at[f], 4 * qd + e);
          if (!PACK) has[f & 1][e] = va >= 0;
#pragma unroll
          for (int c = 0; c < VC; c++)
            v_ahead[f & 1][e][c] = *(const f32x4*)(vcache + (size_t)max(va, 0LL) * vd + min(64 * c + 4 * r, vd - 4));
        }
      };
      if (ASK) ask_keys(0);
#pragma unroll
      for (int f = 0; f < 4; f++) {
        s[f] = zero;
        if (ASK) {
          if (f < 3) ask_keys(f + 1);
#pragma unroll
          for (int c = 0; c < QC; c++) asm volatile("" : "+v"(k_ahead[f & 1][c]));
          if (unseen(f)) continue;
        }
        const float* kr = kcache + (size_t)max(at[f], 0LL) * hd;
#pragma unroll
        for (int c = 0; c < QC; c++) {
          const int d = 16 * c + 4 * qd;
          f32x4 k4;
          if (ASK) k4 = at[f] >= 0 && d < hd ? k_ahead[f & 1][c] : zero;
          else k4 = at[f] >= 0 && d < hd ? *(const f32x4*)(kr + d) : zero;
#pragma unroll
          for (int e = 0; e < 4; e++) s[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[e], qf[c][e], s[f], 0, 0, 0);
        }
      }
      if (ASK) ask_values(0);
      float top = -INFINITY;
      bool all = true;             // the lane's query sees all of the lane's keys
#pragma unroll
      for (int f = 0; f < 4; f++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int j = j0 + 16 * f + 4 * qd + e;
          float x = s[f][e] * scale;
          if (softcap > 0.f) x = softcap * tanhf(x / softcap);
          const bool sees = (j >= lo || j < keep) && j <= pos;
          all = all && sees;
          s[f][e] = sees ? x : -INFINITY;
          top = fmaxf(top, s[f][e]);
        }
      top = fmaxf(top, __shfl_xor(top, 16));
      top = fmaxf(top, __shfl_xor(top, 32));
      const float m_new = fmaxf(m, top);
      const float corr = m == m_new ? 1.f : expf(m - m_new);
      float sum = 0.f;
#pragma unroll
      for (int f = 0; f < 4; f++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int j = j0 + 16 * f + 4 * qd + e;
          s[f][e] = (j >= lo || j < keep) && j <= pos ? expf(s[f][e] - m_new) : 0.f;
          sum += s[f][e];
        }
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      l = l * corr + sum;
      m = m_new;
#pragma unroll
      for (int c = 0; c < VC; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[c][e] *= corr;
      const bool whole = __all(all);
#pragma unroll
      for (int f = 0; f < 4; f++) {
        if (ASK) {
          if (f && j0 + 16 * f > seg_hi) break;      // (no wait for a piece behind the last key)
          if (f < 3) ask_values(f + 1);
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int c = 0; c < VC; c++) asm volatile("" : "+v"(v_ahead[f & 1][e][c]));
        }
        if (PASS_VALUES && unseen(f)) continue;
        f32x4 v[4][VC];            // [key 16 f + 4 qd + e][c]: channels 64 c + 4 r ..
        long long va[4];
        bool fine = true;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (!ASK) va[e] = __shfl(at[f], 4 * qd + e);
          const bool there = !ASK ? false : PACK ? __shfl((int)(at[f] >> 32), 4 * qd + e) >= 0 : has[f & 1][e];
#pragma unroll
          for (int c = 0; c < VC; c++) {
            const int d = 64 * c + 4 * r;
            if (ASK) v[e][c] = there && d < vd ? v_ahead[f & 1][e][c] : zero;
            else v[e][c] = va[e] >= 0 && d < vd ? *(const f32x4*)(vcache + (size_t)va[e] * vd + d) : zero;
          }
        }
        if (!whole) {
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int c = 0; c < VC; c++)
#pragma unroll
              for (int x = 0; x < 4; x++) fine = fine && fabsf(v[e][c][x]) < INFINITY;
        }
        if (__all(fine)) {
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int c = 0; c < VC; c++)
#pragma unroll
              for (int x = 0; x < 4; x++)
                acc[c][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e][c][x], s[f][e], acc[c][x], 0, 0, 0);
        } else {
          // rare: each query takes the keys that it sees, in the products' order (0, 4, 8, 12, 1, 5, ..)
          for (int n = 0; n < 16; n++) {
            const int kk = n % 4 * 4 + n / 4, j = j0 + 16 * f + kk;
            const long long av = __shfl(at[f], kk);
            float p = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float x = __shfl(s[f][e], (kk >> 2) * 16 + r);
              if (e == (kk & 3)) p = x;
            }
            if (av < 0 || !((j >= lo || j < keep) && j <= pos)) continue;
#pragma unroll
            for (int c = 0; c < VC; c++)
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const int d = 64 * c + 16 * qd + 4 * i;
                if (d >= vd) continue;
#pragma unroll
                for (int e = 0; e < 4; e++) acc[c][e][i] = fmaf(vcache[(size_t)av * vd + d + e], p, acc[c][e][i]);
              }
          }
        }
      }
    }
    join = __builtin_amdgcn_readfirstlane(join);
    const int first = join & 255, rows = join >> 8 & 255, members = PACK ? join >> 16 : WAVES;
    if (!PACK || first_tile(members) < tile1) {
#pragma unroll
      for (int c = 0; c < VC; c++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          *(f32x4*)&s_acc[wave][r][64 * c + 16 * qd + 4 * i] = f32x4{acc[c][0][i], acc[c][1][i], acc[c][2][i], acc[c][3][i]};
      if (qd == 0) {
        s_m[wave][r] = m;
        s_l[wave][r] = l;
      }
    }
    __syncthreads();
    // a thread joins four channels of a row over the run's waves
    const int wave0 = wave & -members;
    for (int x = threadIdx.x & (64 * members - 1); x < rows * (vd / 4); x += 64 * members) {
      const int rr = x / (vd / 4), d = x % (vd / 4) * 4;
      const int t = t0 + first + rr / gh, h = kvh * group + h0 + rr % gh;
      float part[WAVES], top = -INFINITY, den = 0.f;
      auto holds = [&](int w) { return !PACK || tile0 + ((w - tile0) & (WAVES - 1)) < tile1; };       // the w-th place in the order
      auto at_wave = [&](int w) { return holds(w) ? wave0 + (w & (members - 1)) : wave0; };
#pragma unroll
      for (int w = 0; w < WAVES; w++) {
        part[w] = holds(w) ? s_m[at_wave(w)][rr] : -INFINITY;
        top = fmaxf(top, part[w]);
      }
      f32x4 o = zero;
#pragma unroll
      for (int w = 0; w < WAVES; w++) {
        const float f = part[w] == top ? 1.f : expf(part[w] - top);
        // (written out: the sums' bits are not to hang on what the compiler fuses in which form)
        den = fmaf(holds(w) ? s_l[at_wave(w)][rr] : 0.f, f, den);
        const f32x4 v = holds(w) ? *(const f32x4*)&s_acc[at_wave(w)][rr][d] : zero;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = fmaf(v[e], f, o[e]);
      }
      if (sinks != nullptr || unit_sink) {
        const float sk = sinks != nullptr ? sinks[h] : 0.f;
        const float m_new = fmaxf(top, sk), corr = expf(top - m_new);
        den = den * corr + expf(sk - m_new);
        o *= corr;
      }
      float inv = 1.f / den;
      if (gate != nullptr) inv *= 1.f / (1.f + expf(-gate[(size_t)t * gate_ld + h]));
      o *= inv;
      if (v_freq == nullptr) *(f32x4*)(out + ((size_t)t * nh + h) * vd + d) = o;
      else *(f32x4*)&s_acc[wave0][rr][d] = o;      // a place that no other thread reads
    }
    if (v_freq != nullptr) {
      // values were turned by their own positions when they were stored: the sum is turned back
      // by the query's position, pair m by -pos * v_freq[m]
      __syncthreads();
      const int half = vd / 2;
      for (int x = threadIdx.x & (64 * members - 1); x < rows * half; x += 64 * members) {
        const int rr = x / half, m2 = x % half;
        const int t = t0 + first + rr / gh, h = kvh * group + h0 + rr % gh;
        float sn, cs, ra, rb;
        sincosf(-(float)positions[t] * v_freq[m2], &sn, &cs);
        const int ia = v_interleaved ? 2 * m2 : m2, ib = v_interleaved ? 2 * m2 + 1 : m2 + half;
        rotate_pair(s_acc[wave0][rr][ia], s_acc[wave0][rr][ib], sn, cs, ra, rb);
        out[((size_t)t * nh + h) * vd + ia] = ra;
        out[((size_t)t * nh + h) * vd + ib] = rb;
      }
    }
    if (!PACK) break;                // a block for every run that there can be
    __syncthreads();                 // the next runs' results go where these were
  }
}
#endif  // !ZSE_ACT_BF16

// softcap <= 0: no cap; window <= 0: every earlier key is visible.  v_transposed: V is
// cached as [page][kv head][hd][bs] instead of [page][kv head][bs][hd].
// hd: the size of a head's queries and keys; vd: of its values (the output's too).  v_freq (may
// be null): float [vd / 2], values are cached turned by their positions and the output is turned back.
// sinks (may be null): float [nh].  v_in_k: values are the first vd channels of the keys.
// chunk > 0 (without a window): a query sees the keys of its own chunk of positions only.
// unit_sink: a sink of score 0 joins every head's denominator (not together with sinks).
// keep > 0 (with a window): a query sees the sequence's first ``keep`` keys beside its window.
// gate (may be null): row t's nh numbers lie at gate + t * gate_ld; head h's output times sigmoid of the h-th.
extern "C" int zk_attention_plain_gated(const void* q, int q_stride, const void* kcache, const void* vcache,
                                         const int* block_table, int max_blocks, const int* req_of_token,
                                         const int* positions, void* out, int T, int nh, int nkv, int hd, int vd,
                                         int bs, float scale, float softcap, int window, int v_transposed,
                                         const float* v_freq, int v_interleaved, const float* sinks, int v_in_k,
                                         int chunk, int unit_sink, int keep, const void* gate, int gate_ld, void* stream) {
  ZK_REQUIRE(gate == nullptr || gate_ld >= nh, "zk_attention_plain: gate rows hold a number per head");
  ZK_REQUIRE(keep >= 0 && (keep == 0 || window > 0), "zk_attention_plain: first keys are kept beside a window");
  ZK_REQUIRE(chunk >= 0 && (chunk == 0 || window <= 0), "zk_attention_plain: a chunk or a window, not both");
  ZK_REQUIRE(!unit_sink || sinks == nullptr, "zk_attention_plain: a unit sink or learned sinks, not both");
  ZK_REQUIRE(T >= 0 && nh > 0 && nkv > 0 && hd > 0 && vd > 0 && bs > 0 && max_blocks > 0,
             "zk_attention_plain: bad sizes");
  ZK_REQUIRE(vd <= 1024 && (v_freq == nullptr || vd % 2 == 0), "zk_attention_plain: value size above 1024, or odd with a rotation");
  ZK_REQUIRE(nh % nkv == 0, "zk_attention_plain: heads must be a multiple of kv heads");
  ZK_REQUIRE(hd <= 1024, "zk_attention_plain: head_dim above 1024 is not supported");
  ZK_REQUIRE(nh <= 65535, "zk_attention_plain: too many heads");
  ZK_REQUIRE(q_stride >= nh * hd, "zk_attention_plain: q row stride too small");
  ZK_REQUIRE(!v_in_k || (vd <= hd && !v_transposed), "zk_attention_plain: values inside keys are no wider than the keys");
  if (T == 0) return 0;
#if !ZSE_ACT_BF16
  // Heads of up to 256 channels in whole 16-byte pieces, keys and values in rows of their own:
  // the matrix-core kernel.  Everything else (values inside keys, odd sizes) is taken key by key.
  if (hd <= 256 && vd <= 256 && hd % 4 == 0 && vd % 4 == 0 && q_stride % 4 == 0 && !v_in_k && !v_transposed &&
      ((uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)out) % 16 == 0 &&
      (long long)nkv * ((nh / nkv + 15) / 16) <= 65535) {
    const int group = nh / nkv, tb = group < 16 ? 16 / group : 1, most = hd > vd ? hd : vd;
    // a launch of 2^32 threads or more would run its low 32 bits only: tokens are taken 2^22 blocks at a time
    const int most_tokens = (1 << 22) * tb;
    for (long long t = 0; t < T; t += most_tokens) {
      const int n = T - t < most_tokens ? (int)(T - t) : most_tokens;
      // Where a run a block makes few rounds of blocks, a run has a block to itself; otherwise short runs share blocks,
      // and few blocks are without a run.  From 1,024 blocks on where eight tokens or more share one (64 requests of 3
      // tokens, 8 heads of 64: 20 -> 12 us), from 2,048 on with more than 128 channels (16 requests of 20, 8 over 4 of 256:
      // 1,280 blocks take 28 us and 36 packed, 256 of 3: 3,072 take 128 and 57), else from 4,096 on (1,500 tokens, 8 over
      // 1 of 32: 1,500 blocks take 65 and 75).
      dim3 blocks((n + tb - 1) / tb, nkv * ((group + 15) / 16), tb);
      const long long columns = (long long)blocks.x * blocks.y;
      const bool pack = columns * tb > (tb < 8 ? 4096 : most > 128 ? 2048 : 1024) && tb > 1;
      if (pack) blocks.z = (unsigned)std::min<long long>(tb, (2048 + columns - 1) / columns);
#define ZK_ATTENTION_F32(D_, W_, A_, P_)                                                                               \
  attention_f32_kernel<D_, W_, A_, P_><<<blocks, 64 * W_, 0, (hipStream_t)stream>>>(                                      \
      (const float*)q + t * q_stride, q_stride, (const float*)kcache, (const float*)vcache, block_table,              \
      max_blocks, req_of_token + t, positions + t, (float*)out + t * nh * vd, n, nh, nkv, hd, vd, bs, scale,          \
      softcap, window, v_freq, v_interleaved, sinks, chunk, unit_sink, keep,                                          \
      gate == nullptr ? nullptr : (const float*)gate + t * gate_ld, gate_ld)
#define ZK_ATTENTION_F32_PACK(D_, W_, A_)                                                                             \
  if (pack) ZK_ATTENTION_F32(D_, W_, A_, true);                                                                       \
  else ZK_ATTENTION_F32(D_, W_, A_, false)
      if (most <= 64) {
        ZK_ATTENTION_F32_PACK(64, 8, false);
      } else if (most <= 128 && hd > 64) {
        ZK_ATTENTION_F32_PACK(128, 8, true);
      } else if (most <= 128) {
        ZK_ATTENTION_F32_PACK(128, 8, false);
      } else {
        ZK_ATTENTION_F32_PACK(256, 4, false);
      }
#undef ZK_ATTENTION_F32_PACK
#undef ZK_ATTENTION_F32
    }
    return zk_launch_status("zk_attention_plain");
  }
#endif
  dim3 grid(T, nh);
  if (hd <= AP_MAX_HD && vd <= AP_MAX_HD)
    attention_plain_kernel<AP_MAX_HD><<<grid, 64, 0, (hipStream_t)stream>>>(
        (const act_t*)q, q_stride, (const act_t*)kcache, (const act_t*)vcache, block_table, max_blocks,
        req_of_token, positions, (act_t*)out, nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq,
        v_interleaved, sinks, v_in_k, chunk, unit_sink, keep, (const act_t*)gate, gate_ld);
  else
    attention_plain_kernel<1024><<<grid, 64, 0, (hipStream_t)stream>>>(
        (const act_t*)q, q_stride, (const act_t*)kcache, (const act_t*)vcache, block_table, max_blocks,
        req_of_token, positions, (act_t*)out, nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq,
        v_interleaved, sinks, v_in_k, chunk, unit_sink, keep, (const act_t*)gate, gate_ld);
  return zk_launch_status("zk_attention_plain");
}

extern "C" int zk_attention_plain_kept(const void* q, int q_stride, const void* kcache, const void* vcache,
                                         const int* block_table, int max_blocks, const int* req_of_token,
                                         const int* positions, void* out, int T, int nh, int nkv, int hd, int vd,
                                         int bs, float scale, float softcap, int window, int v_transposed,
                                         const float* v_freq, int v_interleaved, const float* sinks, int v_in_k,
                                         int chunk, int unit_sink, int keep, void* stream) {
  return zk_attention_plain_gated(q, q_stride, kcache, vcache, block_table, max_blocks, req_of_token, positions, out, T,
                                  nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq, v_interleaved,
                                  sinks, v_in_k, chunk, unit_sink, keep, nullptr, 0, stream);
}

extern "C" int zk_attention_plain_masked(const void* q, int q_stride, const void* kcache, const void* vcache,
                                         const int* block_table, int max_blocks, const int* req_of_token,
                                         const int* positions, void* out, int T, int nh, int nkv, int hd, int vd,
                                         int bs, float scale, float softcap, int window, int v_transposed,
                                         const float* v_freq, int v_interleaved, const float* sinks, int v_in_k,
                                         int chunk, int unit_sink, void* stream) {
  return zk_attention_plain_kept(q, q_stride, kcache, vcache, block_table, max_blocks, req_of_token, positions, out, T,
                                 nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq, v_interleaved,
                                 sinks, v_in_k, chunk, unit_sink, 0, stream);
}

extern "C" int zk_attention_plain_sink(const void* q, int q_stride, const void* kcache, const void* vcache,
                                       const int* block_table, int max_blocks, const int* req_of_token,
                                       const int* positions, void* out, int T, int nh, int nkv, int hd, int vd,
                                       int bs, float scale, float softcap, int window, int v_transposed,
                                       const float* v_freq, int v_interleaved, const float* sinks, int v_in_k,
                                       void* stream) {
  return zk_attention_plain_masked(q, q_stride, kcache, vcache, block_table, max_blocks, req_of_token, positions, out, T,
                                   nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq, v_interleaved,
                                   sinks, v_in_k, 0, 0, stream);
}

extern "C" int zk_attention_plain_ext(const void* q, int q_stride, const void* kcache, const void* vcache,
                                      const int* block_table, int max_blocks, const int* req_of_token,
                                      const int* positions, void* out, int T, int nh, int nkv, int hd, int vd,
                                      int bs, float scale, float softcap, int window, int v_transposed,
                                      const float* v_freq, int v_interleaved, void* stream) {
  ZK_REQUIRE(hd <= AP_MAX_HD && vd <= AP_MAX_HD, "zk_attention_plain: head_dim above 256 is not supported");
  return zk_attention_plain_sink(q, q_stride, kcache, vcache, block_table, max_blocks, req_of_token, positions, out, T,
                                 nh, nkv, hd, vd, bs, scale, softcap, window, v_transposed, v_freq, v_interleaved,
                                 nullptr, 0, stream);
}

extern "C" int zk_attention_plain(const void* q, int q_stride, const void* kcache, const void* vcache,
                                  const int* block_table, int max_blocks, const int* req_of_token,
                                  const int* positions, void* out, int T, int nh, int nkv, int hd,
                                  int bs, float scale, float softcap, int window, int v_transposed,
                                  void* stream) {
  return zk_attention_plain_ext(q, q_stride, kcache, vcache, block_table, max_blocks, req_of_token, positions, out, T,
                                nh, nkv, hd, hd, bs, scale, softcap, window, v_transposed, nullptr, 0, stream);
}

#include "packed_call.h"
extern "C" int zk_steplist_register(const char* name, int nargs, void* fn);
static const int attention_plain_sink_entered = zk_steplist_register(
    "zk_attention_plain_sink", zk_packed::Call<zk_attention_plain_sink>::nargs,
    (void*)zk_packed::Call<zk_attention_plain_sink>::call);
static const int attention_plain_masked_entered = zk_steplist_register(
    "zk_attention_plain_masked", zk_packed::Call<zk_attention_plain_masked>::nargs,
    (void*)zk_packed::Call<zk_attention_plain_masked>::call);
static const int attention_plain_kept_entered = zk_steplist_register(
    "zk_attention_plain_kept", zk_packed::Call<zk_attention_plain_kept>::nargs,
    (void*)zk_packed::Call<zk_attention_plain_kept>::call);
static const int attention_plain_gated_entered = zk_steplist_register(
    "zk_attention_plain_gated", zk_packed::Call<zk_attention_plain_gated>::nargs,
    (void*)zk_packed::Call<zk_attention_plain_gated>::call);
static const int attention_plain_ext_entered = zk_steplist_register(
    "zk_attention_plain_ext", zk_packed::Call<zk_attention_plain_ext>::nargs,
    (void*)zk_packed::Call<zk_attention_plain_ext>::call);
