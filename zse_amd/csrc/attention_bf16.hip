// Paged attention on the matrix cores, bfloat16 in, float softmax.
//
// A wave owns up to 32 query rows: TPW consecutive tokens of one request times the g = nh / nkv
// query heads that share a KV head, so every K and V tile it loads serves the
// whole group (the reference's paged_attention_v2 stages a K/V tile once for
// the heads of a group too, orchestrator/kernels.py:687-854, but is never
// launched; the launched kernels read K and V once per query head and hold one
// score per cached token in shared memory, :524-671, :859-958).
//
// Per tile of 32 keys:
//   S^T[key, row]  = K[key, :] . Q[row, :]        32x32x16 MFMA, hd/16 steps
//   scale, soft cap, mask (key <= pos, pos - key < window), running max / sum
//   O^T[d, row]   += V^T[d, key] * P^T[key, row]  32x32x16 MFMA, 2 per 32 channels
// S^T and O^T both keep a query row in a fixed lane (column = lane % 32), so the
// running maximum, sum and rescale are per-lane scalars, and the probabilities
// a lane holds after the first product are exactly its operand for the second:
// the contraction order over keys is permuted to match (slots e < 4 of lane half
// h are keys 4h + e, slots e >= 4 are keys 8 + 4h + e - 4), and V is read with
// the same permutation.  V is therefore cached transposed, [page][kv head][hd][bs],
// so that four consecutive keys of a channel are one 8-byte load.
//
// Portions have these kernels, chosen by the launch's sizes and a price (portion_plan): a group of 32
// rows a block, its four waves sharing out the keys (attn_mfma_kernel: few groups); four or
// eight consecutive groups a block with every tile of keys and values fetched once into LDS for
// all of them (attn_shared_kernel: many groups); and the latter with the keys of a block of rows
// cut into ranges over several blocks, joined by attn_portion_join_kernel (few groups with long
// contexts: a portion of a prompt behind thousands of tokens).  Heads of 128 and 256 channels with
// pages of 16 or more take attn_stream_kernel in place of the shared tiles, in ranges or not, and attn_short_kernel, 16 rows a
// block, where rows and keys are few.
//
// Decoded tokens use a split variant: the keys are cut into chunks aligned to absolute positions,
// each leaves (max, sum, O) and a second kernel joins the chunks in order; the cut never follows
// from the batch, so a request's result is the same whoever shares its step.  With at most 16
// heads a KV head a wave takes 32 keys on 16x16x32 MFMAs and a block of four waves leaves one
// partial result (attn_decode_kernel): a single query token fills only g of a tile's columns,
// and the narrower tile halves both the accumulator registers and the wasted work.  Otherwise a
// wave takes 64 keys on 32x32x16 MFMAs and leaves a result of its own.
//
// A head's values may be half or twice as wide as its keys.  Where a window keeps the sequence's first
// keys in sight, the tiles (or a decoded token's chunks) of those keys come first and are
// followed by the window's.
// The kernels are templates in attention_bf16_kernels.h.
#include "attention_bf16_kernels.h"
#include "packed_call.h"

#include <algorithm>

#if ZSE_ACT_BF16

// Joins the ranges of keys of a portion's rows (attn_shared_kernel, SPLIT), in their order: a
// block of 64 threads per (32 channels of a wave of a block of rows, KV head, request), every
// lane the row and the channels it had in the kernel that wrote the partial results.  The ranges a block of rows
// has follow from its first and last key as there; a range that a row does not see at all (one
// past its position, in a block of rows on the diagonal) has the maximum -inf and weighs nothing.
__global__ __launch_bounds__(64) void attn_portion_join_kernel(AttnParams p, int per_block, int row_blocks, int dts) {
  const int r = p.r_begin + blockIdx.z, kvh = blockIdx.y;
  const int dt = blockIdx.x % dts, ww = blockIdx.x / dts;      // 32 channels of a wave's rows a block
  const int rows_x = ww >> 2, wave = ww & 3;
  const int lane = threadIdx.x, lr = lane & 31, lk = lane >> 5;
  const int qs = p.q_start[r], n = p.q_start[r + 1] - qs;
  if (n <= 0) return;
  const int start = p.ctx_len[r] - n;
  const int bi = (n + per_block - 1) / per_block - 1 - rows_x;
  if (bi < 0) return;
  const int g = p.nh / p.nkv;
  const int t0 = bi * per_block + wave * p.tpw;
  const int ntok = max(0, min(p.tpw, n - t0));
  const int tok = lr / g, hq = lr - tok * g;
  if (tok >= ntok) return;
  const int blk_lo = start + bi * per_block, blk_hi = start + min(n, (bi + 1) * per_block) - 1;
  const int key_lo = first_key(p, blk_lo);
  const int ranges = (KeyTiles(p, key_lo, blk_hi).count - 1) / p.chunk + 1;
  const size_t slot0 = ((((size_t)blockIdx.z * p.nkv + kvh) * row_blocks + rows_x) * p.nchunks) * 4 + wave;
  float m = -INFINITY;
  for (int c = 0; c < ranges; c++) m = fmaxf(m, p.part_ml[(slot0 + (size_t)c * 4) * 128 + lr]);
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
  for (int c = 0; c < ranges; c++) {
    const size_t slot = slot0 + (size_t)c * 4;
    const float mc = p.part_ml[slot * 128 + lr];
    const float w = mc == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mc - m);
    l += w * p.part_ml[slot * 128 + 32 + lr];
    const f32x4* po = (const f32x4*)p.part_o + slot * ((size_t)dts * 4 * 64) + (size_t)dt * 4 * 64 + lane;
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] += w * po[j * 64];
  }
  const int row = qs + t0 + tok, head = q_head_of(p, kvh, hq);
  const float inv = row_factor(p, row, head, l, m);
  __bf16* orow = p.out + ((size_t)row * p.nh + head) * p.vd;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = dt * 32 + 8 * j + 4 * lk;
    if (d < p.vd) {
      bf16x4 w4;
#pragma unroll
      for (int i = 0; i < 4; i++) w4[i] = (__bf16)(acc[j][i] * inv);
      *(bf16x4*)(orow + d) = w4;
    }
  }
}

// Joins the chunks of a decoded token's attention, in chunk order: a block per
// (request, head), a thread per channel; the chunks' weights exp(m_c - m) are computed once.
//
// Its time is the launch and a chain of waits.  With up to 64 parts every wave works the weights out for itself, a
// lane a part, and hands them on as scalars: no local memory, no barrier.  Where the parts are numbered from the sequence's first
// key (``direct``), they are asked for beside the request's length.  (With the kernel that makes the
// parts, us: 1 request of 100 keys, 8 heads over 2 of 128, 8.2 -> 7.6, 8 of 500, 8 over 4 of 256, 11.8 -> 11.1, 24 of 32 to 700 17.6 -> 17.1.)
#define ATT_MAX_CHUNKS 2048      // 262,144 keys in parts of 128
__global__ __launch_bounds__(256) void attn_combine_kernel(const float* __restrict__ part_o,
                                                           const float* __restrict__ part_ml,
                                                           const int* __restrict__ q_start,
                                                           const int* __restrict__ ctx_len,
                                                           __bf16* __restrict__ out, int nh, int hd,
                                                           int window, int r_begin, int nchunks, int span,
                                                           int mask_chunk, int sink, int keep,
                                                           const float* __restrict__ sinks,
                                                           const __bf16* __restrict__ gate, int gate_ld) {
  __shared__ float wgt[ATT_MAX_CHUNKS];
  __shared__ float red[17];
  const int rr = blockIdx.x, head = blockIdx.y, lane = threadIdx.x & 63;
  const int r = r_begin + rr;
  const size_t base = ((size_t)rr * nh + head) * nchunks;
  const int d0 = min((int)threadIdx.x, hd - 1);
  const bool direct = mask_chunk == 0 && (window == 0 || (long long)nchunks * span <= window);
  constexpr int PF = 32, FIRST = 8;
  float pf[PF], ml[2];
  const float* po0 = part_o + base * hd + d0;
  if (direct) {          // (parts past the request's last hold anything; they are not used)
#pragma unroll
    for (int c = 0; c < FIRST; c++) pf[c] = po0[(size_t)min(c, nchunks - 1) * hd];
    const float* at = part_ml + (base + min(lane, nchunks - 1)) * 2;
    ml[0] = at[0];
    ml[1] = at[1];
  }
  const int row = q_start[r], n = q_start[r + 1] - row;
  const int pos = ctx_len[r] - 1;
  if (n <= 0) return;
  const int lo = mask_chunk > 0 ? pos - pos % mask_chunk : window > 0 ? max(0, pos - window + 1) : 0;
  // the parts of the kept first keys, [0, kept), then those from the window's first on, [c0, c1]
  const int c0 = lo / span, c1 = pos / span, kept = min((keep + span - 1) / span, c0);
  auto part_of = [&](int i) { return i < kept ? i : c0 + i - kept; };
  const int np = kept + c1 - c0 + 1;
  // the first partial results of the thread's channel are asked for now: they come in while
  // the weights are worked out (a part past the last is read from the last and not used); the further
  // ones only where there are that many parts (32 asked for always cost 1 to 8 parts 0.3 us a join)
  {
    auto ask = [&](int from, int to) {
#pragma unroll
      for (int c = 0; c < PF; c++)
        if (c >= from && c < to) pf[c] = po0[(size_t)part_of(min(c, np - 1)) * hd];
    };
    if (!direct) ask(0, FIRST);
    if (np > FIRST) ask(FIRST, 16);
    if (np > 16) ask(16, PF);
  }
  __bf16* orow = out + ((size_t)row * nh + head) * hd;
  if (np <= 64) {
    if (!direct) {
      const float* at = part_ml + (base + part_of(min(lane, np - 1))) * 2;
      ml[0] = at[0];
      ml[1] = at[1];
    }
    const bool mine = lane < np;
    const float m = wave_max_whole(mine ? ml[0] : -INFINITY);
    const float w = __builtin_amdgcn_exp2f(ml[0] - m);
    const float l = wave_sum_whole(mine ? ml[1] * w : 0.f);
    const float inv = gate_factor(gate, gate_ld, row, head) / (l + sink_weight(sinks, sink, head, m));
    auto weight = [&](int c) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), c)); };
    if ((int)threadIdx.x < hd) {
      float acc = 0.f;
#pragma unroll
      for (int q = 0; q < PF; q++)
        if (q < np) acc += pf[q] * weight(q);
      for (int c = PF; c < np; c += 8) {      // eight asked for at a time, added up in part order
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = po0[(size_t)part_of(min(c + q, np - 1)) * hd];
#pragma unroll
        for (int q = 0; q < 8; q++)
          if (c + q < np) acc += v[q] * weight(c + q);
      }
      orow[threadIdx.x] = (__bf16)(acc * inv);
    }
    return;
  }
  float m = -INFINITY;
  for (int c = threadIdx.x; c < np; c += 256) m = fmaxf(m, part_ml[(base + part_of(c)) * 2]);
  m = wave_max_whole(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float l = 0.f;
  for (int c = threadIdx.x; c < np; c += 256) {
    const size_t at = (base + part_of(c)) * 2;
    const float w = __builtin_amdgcn_exp2f(part_ml[at] - m);
    wgt[c] = w;
    l += part_ml[at + 1] * w;
  }
  l = block_sum_whole(l, red);
  const float inv = gate_factor(gate, gate_ld, row, head) / (l + sink_weight(sinks, sink, head, m));
  if ((int)threadIdx.x < hd) {
    float acc = 0.f;
#pragma unroll
    for (int q = 0; q < PF; q++) acc += pf[q] * wgt[q];
    int c = PF;
    for (; c + 4 <= np; c += 4) {       // four loads in flight, summed in part order
      const float v0 = po0[(size_t)part_of(c) * hd], v1 = po0[(size_t)part_of(c + 1) * hd];
      const float v2 = po0[(size_t)part_of(c + 2) * hd], v3 = po0[(size_t)part_of(c + 3) * hd];
      acc += v0 * wgt[c];
      acc += v1 * wgt[c + 1];
      acc += v2 * wgt[c + 2];
      acc += v3 * wgt[c + 3];
    }
    for (; c < np; c++) acc += po0[(size_t)part_of(c) * hd] * wgt[c];
    orow[threadIdx.x] = (__bf16)(acc * inv);
  }
}

static int launch_attn(int what, const AttnParams& p, dim3 grid, hipStream_t s) {
  if (p.vd != p.hd) return attn_launch_uneven(what, p, grid, s);
  switch (p.hd / 16) {
    case 1: return launch_sizes<1, 1>(what, p, grid, s);
    case 2: return launch_sizes<2, 2>(what, p, grid, s);
    case 4: return launch_sizes<4, 4>(what, p, grid, s);
    case 8: return launch_sizes<8, 8>(what, p, grid, s);
    case 16: return launch_sizes<16, 16>(what, p, grid, s);
    default: return zk_fail("zk_attention_bf16: head_dim must be 16, 32, 64, 128 or 256");
  }
}

// Bytes the portions' split variant needs behind the decoded tokens' part of the workspace.
// Per (request, KV head, block of rows, range, wave): the wave's accumulators as they lie in
// its registers (ceil(hd / 32) x 16 floats a lane) and 128 floats of maxima and sums.
static size_t portion_split_bytes(long row_blocks, int nkv, int hd, int ranges) {
  const size_t dt = (size_t)(hd + 31) / 32;
  return (size_t)row_blocks * nkv * ranges * 4 * (dt * 16 * 64 + 128) * sizeof(float);
}

// The ranges of keys for a launch of few blocks of rows: tiles a range (0: do not split) and the
// most ranges a block of rows can have.  Priced for one causal request of max_q_len rows ending
// at max_ctx, window or not: blocks(ct) = sum over the blocks of rows of ceil(tiles / ct), and
// the time goes with ceil(blocks / 256) * ct; of equal times the longer range (fewer partial
// results).  No split unless it at least halves the longest block's tiles; at most
// ATT_MOST_RANGES ranges for the longest block of rows the caller's limits allow (bound_tiles),
// which bounds the workspace.
static int portion_ranges(int max_q_len, int max_ctx, int window, int mask_chunk, int keep, int per_block, int nkv,
                          int r_prefill, int bound_tiles) {
  const int row_blocks = (max_q_len + per_block - 1) / per_block;
  auto tiles_of = [&](int bi) {
    const int lo = max_ctx - max_q_len + bi * per_block, hi = std::min(max_ctx, lo + per_block) - 1;
    const int klo = mask_chunk > 0 ? lo - lo % mask_chunk : window > 0 ? std::max(0, lo - window + 1) : 0;
    return std::min((keep + 31) / 32, klo / 32) + hi / 32 - klo / 32 + 1;
  };
  int longest = 0;
  for (int bi = 0; bi < row_blocks; bi++) longest = std::max(longest, tiles_of(bi));
  static const int cands[] = {32, 24, 16, 12, 10, 8, 6, 4};
  int best = 0;
  long best_cost = (long)((long)row_blocks * nkv * r_prefill + 255) / 256 * (longest + 10);
  for (int ct : cands) {
    if (2 * ct > longest || (bound_tiles + ct - 1) / ct > ATT_MOST_RANGES) continue;
    long blocks = 0;
    for (int bi = 0; bi < row_blocks; bi++) blocks += (tiles_of(bi) + ct - 1) / ct;
    blocks *= (long)nkv * r_prefill;
    const long cost = (blocks + 255) / 256 * (ct + 10) + 6;   // a block's start and end, the joining launch: in tiles' worth
    if (cost < best_cost) { best = ct; best_cost = cost; }
  }
  return best;
}

// Heads of 128 and 256 channels on attn_stream_kernel: a group a block (0), four groups a block (4) or the
// latter with the keys in ranges of ``ranges`` tiles (5), by the least of three prices in microseconds.  A
// block costs a start and a time a tile; blocks beyond one a CU (two for 128 channels) take their
// share of the CUs' time, the last ones half of the shortest block's more; ranges add a block's partial
// results, the blocks that find nothing to do and the joining launch.  A block of rows' ranges are neighbours in
// the grid, and blocks go round to the XCDs and their shader engines by number: where 2, 4 or 8 divides the most ranges of a
// block of rows, the first ranges share one half, quarter or eighth of the chip and the last, short or not there,
// another, so each such class is priced on its part (2,048 rows from their first token, 32 heads over 16 of 128: ranges of 32 tiles,
// two a block of rows, 94 us, of 24, three, 82; four groups a block 70).
// The constants are fitted to launches of 40 to 4,096 rows behind up to 8,000 keys, 2 to 16 key heads, one to eight
// requests: over 390 of them the form that is named takes 1.016 times the best one's time in the mean, 1.32 at the
// most (us; group, four, ranges, taken): 8 heads over 4 of 256, 512 rows at 512
// keys 25, 28, 23, ranges; behind 3,584 112, 143, 42, ranges; 4,096 rows 238, 135, 129, ranges; 16 over 8, 2,048 rows 149, 81, 84,
// four; 32 over 16 of 128, 512 rows at 512 keys 16, 21, 25, group; 2,048 rows 168, 70, 82, four.
// ranges: the best cut with ranges, taken or not (0: none); whole: the better kind without; price: of the kind
struct PortionPlan { int kind, ranges, whole; double price; };
static PortionPlan portion_plan(int max_q_len, int max_ctx, int window, int mask_chunk, int keep, int tpw, int nkv, int r_prefill,
                                int bound_tiles, int wide) {
  const bool narrow = wide <= 128;
  const int slots = narrow ? 512 : 256, per_block = 4 * tpw, row_blocks = (max_q_len + per_block - 1) / per_block;
  const long copies = (long)nkv * r_prefill;
  const double start_group = narrow ? 8.7 : 12.0, tile_group = narrow ? 0.64 : 0.77;
  const double start_four = narrow ? 5.5 : 9.5, start_range = narrow ? 6.6 : 11.0, tile_four = narrow ? 0.83 : 1.06;
  const double edges = (narrow ? 1.0 : 0.4) * std::min(max_q_len, per_block) / 32;       // tiles whose scores are masked
  auto tiles_of = [&](int bi) {
    const int lo = max_ctx - max_q_len + bi * per_block, hi = std::min(max_ctx, lo + per_block) - 1;
    const int klo = mask_chunk > 0 ? lo - lo % mask_chunk : window > 0 ? std::max(0, lo - window + 1) : 0;
    return std::min((keep + 31) / 32, klo / 32) + hi / 32 - klo / 32 + 1;
  };
  int longest = 0, shortest = 1 << 30;
  double sum = 0;
  for (int bi = 0; bi < row_blocks; bi++) {
    const int t = tiles_of(bi);
    longest = std::max(longest, t);
    shortest = std::min(shortest, t);
    sum += t;
  }
  auto price = [&](int slots, double blocks, double start, double per_tile, double tiles, int most, int least) {
    const double alone = start + per_tile * most;
    if (blocks <= slots) return alone;
    return std::max(alone, (blocks * start + per_tile * tiles) / slots + 0.5 * (start + per_tile * least));
  };
  PortionPlan best{0, 0, 0, 0};
  const double groups = (max_q_len + tpw - 1) / tpw;
  double best_price = price(slots, groups * copies, start_group, tile_group, sum * copies * groups / row_blocks, longest, shortest);
  const double four = edges + price(slots, (double)row_blocks * copies, start_four, tile_four, sum * copies, longest, shortest);
  if (four < best_price) best = {4, 0, 4, 0}, best_price = four;
  double best_ranges = 1e30;
  static const int cands[] = {64, 48, 40, 32, 24, 16, 12, 10, 8, 6, 4};
  for (int ct : cands) {
    const int most_ranges = (bound_tiles + ct - 1) / ct, classes = most_ranges & -most_ranges;
    if (2 * ct > longest || most_ranges > ATT_MOST_RANGES) continue;
    double blocks[ATT_MOST_RANGES] = {}, tiles[ATT_MOST_RANGES] = {}, t = 0, all = 0;
    for (int bi = 0; bi < row_blocks; bi++)
      for (int i = 0, left = tiles_of(bi); left > 0; i++, left -= ct) {
        blocks[i % classes] += copies;
        tiles[i % classes] += (double)std::min(left, ct) * copies;
      }
    for (int i = 0; i < classes; i++) {
      t = std::max(t, price(slots / classes, blocks[i], start_range, tile_four, tiles[i], ct, std::min(shortest, ct)));
      all += blocks[i];
    }
    t += all * wide * (0.035 / 256) + ((double)row_blocks * copies * most_ranges - all) * 0.005 + 4.0;
    if (t < best_ranges) best.ranges = ct, best_ranges = t;
  }
  best.price = best_price;
  if (best_ranges < best_price) best.kind = 5, best.price = best_ranges;
  return best;
}

// attn_short_kernel's price in microseconds: a start and a time for every tile that the longest block's waves take one after the other;
// blocks beyond one a CU share its way to the L2.  Over 76 launches (7 to 1,024 rows, 8 to 32 heads, up to 2,000 keys in front, one to
// five requests) it is 0.86 to 1.3 times what was measured up to one block a CU, and 0.93 to 1.9 times beyond, where what is close stays
// with the others: 700 rows of 8 heads over 4 of 256, 352 blocks, 28.0 as they are and 30.9; 1,024 of 32 over 16 of 128 35.9 and 61.8.
static double short_price(int max_q_len, int max_ctx, int window, int mask_chunk, int keep, int g, int nkv, int r_prefill, int wide) {
  const int tokens = 16 / g, start = max_ctx - max_q_len, last = start + (max_q_len - 1) / tokens * tokens;
  auto tiles_of = [&](int first) {      // of the block whose first token that is
    const int lo = mask_chunk > 0 ? first - first % mask_chunk : window > 0 ? std::max(0, first - window + 1) : 0;
    return std::min((keep + 31) / 32, lo / 32) + (std::min(max_ctx, first + tokens) - 1) / 32 - lo / 32 + 1;
  };
  int tiles = tiles_of(last);
  // Behind a chunk's beginning the rows see few keys again: where one lies among the rows, the block in front of it has the most (512
  // rows of 8 heads over 4 of 256 that end 256 behind a chunk of 8,192: 8 tiles in the last block, 257 in the longest)
  if (mask_chunk > 0) {
    const int begins = last - last % mask_chunk;
    if (begins > start) tiles = std::max(tiles, tiles_of(start + (begins - 1 - start) / tokens * tokens));
  }
  // (256 channels and more than four tiles a wave: the prices of both kinds are off by as much as they differ, 16 rows behind 500 keys
  // 16.9 as they are and 17.6, 128 rows 20.8 and 19.1)
  if (wide > 128 && tiles > 16) return 1e30;
  const double blocks = (double)((max_q_len + tokens - 1) / tokens) * nkv * r_prefill;
  const double alone = wide > 128 ? 3.6 + 2.8 * ((tiles + 3) / 4) : 3.2 + 1.8 * ((tiles + 3) / 4);
  if (blocks <= 256) return alone;
  // Blocks of one request and key head lie on up to eight XCDs, each of which fetches their keys and values: 7 TB/s, which many requests of
  // few rows reach (32 heads over 16 of 128, 16 requests of 16 rows behind 1,500 keys, 48.2 as they are and 60.6; 32 over 8, 16 of 16
  // behind 400 18.8 and 21.5)
  const double price = alone * (wide > 128 ? 1.3 * blocks / 256 : 1 + 0.45 * (blocks - 256) / 256), each = (max_q_len + tokens - 1) / tokens;
  const double mb = std::min(each, 8.0) * nkv * r_prefill * tiles * 32 * wide * 4 / 1e6;
  return each < 2 ? price : std::max(price, 2 + mb / 7);
}

// 0: the portion kernel is chosen by the sizes; 1: a group of rows a block; 4, 8: shared
// tiles with that many waves a block; 5: shared tiles, four waves, the keys in ranges (as far as
// the workspace allows).  For tests and measurements (process-wide).
static int portion_kernel_mode = 0;

// How a launch of portions runs: which kernel, and with ranges the tiles of one and the most that a
// block of rows has.  ``max_ctx``: the portions' longest context, or (not_theirs) that of all requests of the step, decoded ones
// among them.  ``room``: bytes of workspace for the ranges' partial results.
struct PortionForm {
  AttnWhat what;
  int range_tiles, most_ranges;
};
static PortionForm portion_form(int r_prefill, int max_q_len, int max_ctx, bool not_theirs, int nh, int nkv, int hd, int vd, int bs,
                                int window, int mask_chunk, int keep, int wide_weights, size_t room) {
  const int tpw = 32 / (nh / nkv), per_block = 4 * tpw, wide = std::max(hd, vd), groups = (max_q_len + tpw - 1) / tpw;
  const bool stream = stream_takes(hd, vd, bs, wide_weights);
  // one block a group; two groups a block when that lets every block run at once (256 CUs,
  // one block each) where single groups would need a second round
  const long long single = (long long)groups * nkv * r_prefill, paired = (long long)((groups + 1) / 2) * nkv * r_prefill;
  // Heads of up to 64 channels, pages of 8 keys and wide weights (the others are priced below).  Many groups: tiles
  // shared by the four or eight groups of a block, where that still gives
  // every CU a block (four) or two (eight; head sizes up to 128, whose registers let two
  // waves share a SIMD).  Measured with pages of 8 (us, a group a block and four): 8 heads over 4 of 256, 2,048 rows (512
  // groups) 75 and 112, 3,072 rows (768) 158 and 164, 8,192 rows 878 and 457; 32 over 16 of 128, 512 rows (512) 16 and 25, 1,024
  // rows (1,024) 55 and 44, 4,096 rows 577 and 246 (eight: 223).  The lines are those of these heads; for heads of 64 they
  // lie too low: 32 over 8, 1,024 rows (1,024 groups) 27 and 35, 2,048 rows (2,048) 68 and 63, 4,096 rows (4,096) 219 and 159
  // (eight: 178); 16 over 16, 3,072 rows (1,536) 72 and 93.
  int shared_waves = 0;
  if (bs >= 8 && portion_kernel_mode != 1 && !(stream && portion_kernel_mode == 0)) {
    if (portion_kernel_mode > 1) shared_waves = portion_kernel_mode == 8 ? 8 : 4;
    else if (single >= 4096 && wide <= 128) shared_waves = 8;
    else if (single >= 768) shared_waves = 4;
    if (shared_waves == 8 && wide > 128) shared_waves = 4;       // no room for two waves a SIMD
  }
  // Few blocks of rows with many keys each (a portion of a few hundred rows behind thousands of
  // tokens): four groups a block and the keys in ranges, where the workspace behind the decoded
  // tokens' part holds the ranges' partial results.  By attn_stream_kernel: portion_plan.  The others, with pages of 8 (us, a
  // group a block and ranges): 512 rows behind 3,584 tokens, 8 heads over 4 of 256, 110 and 53, behind 7,680 211 and 80; 32
  // over 16 of 128 92 and 78, 190 and 148; 2,048 rows of 8 heads of 256 from their first token 75 and 61, 1,024 rows 37 and 39.
  if (bs >= 8 && (portion_kernel_mode == 5 || (portion_kernel_mode == 0 && !shared_waves))) {
    // no block of rows has more tiles than this, whatever its request's length
    int bound = (max_ctx + 31) / 32, range_tiles;
    // (a chunk's rows see no more keys than a window of its size would show them)
    const int reach = mask_chunk > 0 ? mask_chunk : window;
    if (reach > 0) bound = std::min(bound, (reach + per_block + 31) / 32 + 1 + (keep + 31) / 32);
    if (stream) {
      const PortionPlan plan = portion_plan(max_q_len, max_ctx, window, mask_chunk, keep, tpw, nkv, r_prefill, bound, wide);
      // few rows and keys: 16 rows a block, where that beats the best of the others, with room for it or not
      if (portion_kernel_mode == 0 && nh / nkv <= 16 &&
          short_price(max_q_len, max_ctx, window, mask_chunk, keep, nh / nkv, nkv, r_prefill, wide) < 0.92 * plan.price)
        return {ATT_SHORT, 0, 0};
      range_tiles = portion_kernel_mode == 5 || plan.kind == 5 ? plan.ranges : 0;
      // Many groups priced by a context that may be another's: no ranges (8 times 128 fresh rows beside 3,840 keys, 32 heads over 16
      // of 128: 26 us, 13 without; 3,584 rows beside 8,192, 16 over 4: 176 and 91).  Few groups do gain from them where the context is theirs.
      if (not_theirs && single >= 768 && portion_kernel_mode == 0) range_tiles = 0;
      shared_waves = std::max(shared_waves, plan.whole);       // without ranges, also where the workspace does not hold them
    } else {
      range_tiles = portion_ranges(max_q_len, max_ctx, window, mask_chunk, keep, per_block, nkv, r_prefill, bound);
    }
    if (range_tiles) {
      const int most_ranges = (bound + range_tiles - 1) / range_tiles;
      const long row_blocks = (long)r_prefill * ((max_q_len + per_block - 1) / per_block);
      if (portion_split_bytes(row_blocks, nkv, vd, most_ranges) <= room) return {ATT_RANGES, range_tiles, most_ranges};
    }
  }
  if (shared_waves) return {shared_waves == 8 ? ATT_SHARED8 : ATT_SHARED4, 0, 0};
  return {single > 256 && paired <= 256 ? ATT_PAIRS : ATT_GROUPS, 0, 0};
}

extern "C" {

int zk_attention_bf16_portion_kernel(int mode) {
  const int before = portion_kernel_mode;
  if (mode == 0 || mode == 1 || mode == 4 || mode == 5 || mode == 8) portion_kernel_mode = mode;
  return before;
}

// Which form a launch of ``r_prefill`` portions takes with ``room`` bytes of workspace behind the decoded tokens' part: 1, 2, 4 or 8
// groups of rows a block, or 5, four with the keys in ranges of *range_tiles tiles.  *stream: 1 by attn_stream_kernel, 2 by
// attn_short_kernel (whose groups have 16 rows).  For tests that mean to reach each of them.
int zk_attention_bf16_portion_form(int r_prefill, int max_q_len, int max_ctx, int not_theirs, int nh, int nkv, int hd, int vd, int bs,
                                   int window, int mask_chunk, int keep, int wide_weights, size_t room, int* range_tiles, int* stream) {
  const PortionForm f = portion_form(r_prefill, max_q_len, max_ctx, not_theirs, nh, nkv, hd, vd, bs, window, mask_chunk, keep, wide_weights, room);
  *range_tiles = f.range_tiles;
  *stream = f.what == ATT_SHORT ? 2 : (f.what == ATT_SHARED4 || f.what == ATT_RANGES) && stream_takes(hd, vd, bs, wide_weights);
  return f.what == ATT_RANGES ? 5 : f.what == ATT_SHARED8 ? 8 : f.what == ATT_SHARED4 ? 4 : f.what == ATT_PAIRS ? 2 : 1;
}

// 1 if the matrix-core kernel takes these sizes, else 0 (the caller then uses the plain kernel).
int zk_attention_bf16_supports(int nh, int nkv, int hd, int bs) {
  if (nkv <= 0 || nh % nkv) return 0;
  const int g = nh / nkv;
  const bool hd_ok = hd == 16 || hd == 32 || hd == 64 || hd == 128 || hd == 256;
  return hd_ok && g <= 32 && bs >= 4 && (bs & (bs - 1)) == 0;
}

// The same for heads whose values have vd channels: as wide as keys, half or twice as wide.
int zk_attention_bf16_supports_values(int nh, int nkv, int hd, int vd, int bs) {
  return zk_attention_bf16_supports(nh, nkv, hd, bs) && (vd == hd || (zk_attention_bf16_supports(nh, nkv, vd, bs) &&
                                                                     (vd == 2 * hd || hd == 2 * vd)));
}

// Bytes of workspace the split variant needs for ``n_decode`` single-token requests.
size_t zk_attention_bf16_workspace(int n_decode, int nh, int hd, int max_ctx) {
  const size_t nchunks = ((size_t)max_ctx + ATT_CHUNK - 1) / ATT_CHUNK;      // an upper bound for both variants
  return (size_t)n_decode * nh * nchunks * (hd + 2) * sizeof(float);
}

// Bytes of workspace that let portions of up to ``max_rows`` rows in all split their keys into
// ranges (a launch of few blocks of rows with long contexts), on top of the decoded tokens'
// part.  A caller that brings less gets the kernels that need none.
size_t zk_attention_bf16_portion_workspace(int max_rows, int nh, int nkv, int hd) {
  if (max_rows <= 0 || nkv <= 0 || nh % nkv || hd <= 0) return 0;
  const int per_block = 4 * std::max(1, 32 / (nh / nkv));
  return portion_split_bytes((max_rows + per_block - 1) / per_block, nkv, hd, ATT_MOST_RANGES) + 256;
}

// Whether decoded tokens of these sizes run on the 16-wide tiles (partial results joined four
// chunks at a time inside a block) or on the 32-wide ones (one partial result a chunk).
static bool decode_on_narrow_tiles(int nh, int nkv, int hd) { return nh / nkv <= 16 && hd % 32 == 0; }

// Whether they go in blocks of 256 keys instead of 128.  By what a runner's limits fix alone (its
// decode_chunk and the width of its block tables), never by a step's requests, because it says where
// a request's sums are cut.  The blocks' queries and results have to fit in 64 KB of LDS.
// Measured (us with the joining launch, blocks of 256 against 128; 8 heads over 4 of 256 channels, A, or 32 over
// 16 of 128, B).  Full contexts of many requests are better off with 256, which leaves half the partial
// results: 64 of 8,192 keys A 357 and 385, B 743 and 810; 64 of 4,096 A 189 and 193, B 372 and 393; below the
// line 64 of 3,072 A 142 and 145, B 283 and 295, of 2,048 A 99.5 and 99.2, B 191 and 197.  Few or uneven requests
// are better off with 128: 1 of 4,096 A 15.1 and 12.1, 8 of 3,000 A 27.8 and 24.7, 8 of 500 to 4,000 24.9 and 21.8,
// 64 of 200 to 3,840 110 and 104, of 200 to 3,000 94 and 85, of 200 to 2,000 65 and 62.  The line lies where the
// loss of full launches by 128 (3 to 4 % under it, 4 to 9 % from 8,192 on) begins to outweigh the rest.
static bool decode_in_long_blocks(int nh, int nkv, int hd, int vd, int bs, int max_blocks, int decode_chunk) {
  return decode_chunk != 32 && (long long)max_blocks * bs >= ATT_DECODE_LONG_FROM &&
         decode_long_lds(nh / nkv, vd) + (size_t)hd / 32 * 4 * 64 * 16 <= 64 * 1024;
}

// Whether decoded tokens' values go past the caches (common.h's load_once) where the caller says that nothing reads
// them again before they have left those anyway: only where a wave's loads take whole lines of a channel's page and
// one block alone reads them.  Pages of up to 32 keys (a wave of the long blocks: 16), no value head under several
// key heads.  us, 64 requests of 4,000 keys, plain loads and these, 8 heads over 4 of 256 channels, pages of 8, 16,
// 32, 64, 128 keys: 201, 198, 198, 206, 231 and 189, 188, 185, 239, 279; 32 over 16 of 128: 393, 392, 388, 397, 400
// and 370, 365, 359, 441, 532; 1 request of 8,000 in long blocks, 8 over 4 of 256, pages of 16, 32, 64: 18.4, 17.5,
// 21.7 and 17.7, 17.9, 22.9; 16 of 64 over 8 whose pairs share values of 128, 64 of 4,000, pages of 16: 113 and 128.
static bool values_past_caches(int once, int bs, int v_shift, bool long_blocks) {
  return once && v_shift == 0 && bs <= (long_blocks ? 16 : 32);
}

// For tests.
extern "C" int zk_attention_bf16_values_past_caches(int once, int nh, int nkv, int hd, int vd, int bs, int max_blocks,
                                                    int decode_chunk, int v_shift) {
  const bool long_blocks = decode_in_long_blocks(nh, nkv, hd, vd, bs, max_blocks, decode_chunk);
  return decode_on_narrow_tiles(nh, nkv, hd) && values_past_caches(once, bs, v_shift, long_blocks);
}

// The longest context the split variant takes for decoded tokens (the joining kernel keeps one
// weight per partial result in LDS).  ``decode_chunk`` as in zk_attention_bf16.
long long zk_attention_bf16_max_context(int nh, int nkv, int hd, int decode_chunk) {
  if (nkv <= 0 || nh % nkv) return 0;
  const int chunk = decode_chunk == 32 ? 32 : ATT_CHUNK;
  return decode_on_narrow_tiles(nh, nkv, hd) ? 4LL * chunk * 1024 : ATT_CHUNK * 1024LL;
}

// Requests [0, r_prefill) hold portions of more than one token (max_q_len the longest);
// requests [r_prefill, R) hold one token each and use the split variant over max_ctx keys.
// decode_chunk: 32 or 64 (0: 64) sets the longest context that decoded tokens on the 16-wide tiles
// take, 131,072 or 262,144 keys.  Their keys are cut after every 128, or with 64 and a table of
// ATT_DECODE_LONG_FROM keys a request or more after every 256: never by what shares the step.
// mask_chunk > 0: a row sees the keys of its own chunk of that many positions (counted from
// position 0) instead of a window; sink: a key of score 0 without a value in every denominator;
// wide_weights: the weights keep 16 bits of mantissa in the product with the values.
// v_shift: 2^v_shift neighbouring key heads read the values of one value head (the value cache
// then holds nkv >> v_shift heads): several maps of keys over the same values.
// vd: channels of a value and of the output's heads (hd, hd / 2 or 2 hd); the workspace functions above
// are asked with vd for their hd.  keep (with a window): a row sees the first ``keep`` keys of its sequence
// beside its window; the caller keeps their pages.
// sinks (may be null; not together with ``sink``): float [nh], exp(sinks[h]) joins head h's denominators.
// gate (may be null): bf16, row t's nh numbers at gate + t * gate_ld; head h's output times sigmoid of the h-th.
// portion_ctx: the longest context among the portions, whose kernel it chooses (0: not known, max_ctx stands for it).
// once: no later launch finds a value that this one reads in the memory side's cache (see values_past_caches; the same bits either way).
int zk_attention_bf16_once(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                           const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                           void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                           int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                           void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                           int v_shift, int vd, int keep, const float* sinks, const void* gate, int gate_ld,
                           int portion_ctx, int once, void* stream) {
  ZK_REQUIRE(portion_ctx >= 0, "zk_attention_bf16: bad context of the portions");
  ZK_REQUIRE(!sink || sinks == nullptr, "zk_attention_bf16: a unit sink or learned sinks, not both");
  ZK_REQUIRE(gate == nullptr || gate_ld >= nh, "zk_attention_bf16: gate rows hold a number per head");
  ZK_REQUIRE(keep >= 0 && (keep == 0 || window > 0), "zk_attention_bf16: first keys are kept beside a window");
  ZK_REQUIRE(v_shift >= 0 && v_shift <= 4 && nkv % (1 << v_shift) == 0, "zk_attention_bf16: key heads in whole groups of a value head");
  ZK_REQUIRE(mask_chunk >= 0 && (mask_chunk == 0 || window == 0), "zk_attention_bf16: a window or a chunk, not both");
  ZK_REQUIRE(R >= 0 && r_prefill >= 0 && r_prefill <= R, "zk_attention_bf16: bad request counts");
  ZK_REQUIRE(zk_attention_bf16_supports_values(nh, nkv, hd, vd, bs), "zk_attention_bf16: sizes not supported "
             "(head_dim 16/32/64/128/256, values as wide, half or twice as wide, at most 32 heads a KV head, page size a power of "
             "two from 4)");
  ZK_REQUIRE(q_stride >= nh * hd && q_stride % 8 == 0 && ((uintptr_t)q % 16 == 0),
             "zk_attention_bf16: q rows must be 16-byte aligned");
  ZK_REQUIRE(max_blocks > 0 && nkv <= 65535 && R <= 65535, "zk_attention_bf16: grid too large");
  ZK_REQUIRE(decode_chunk == 0 || decode_chunk == 32 || decode_chunk == 64,
             "zk_attention_bf16: decode_chunk must be 32 or 64");
  if (R == 0) return 0;
  // everything that can refuse is checked before the first launch
  if (R - r_prefill > 0) {
    ZK_REQUIRE(max_ctx > 0, "zk_attention_bf16: max_ctx must be positive");
    ZK_REQUIRE(max_ctx <= zk_attention_bf16_max_context(nh, nkv, hd, decode_chunk),
               "zk_attention_bf16: context too long for the split variant");
    ZK_REQUIRE(zk_attention_bf16_workspace(R - r_prefill, nh, vd, max_ctx) <= workspace_bytes,
               "zk_attention_bf16: workspace too small for the split partial results");
  }
  if (r_prefill > 0) ZK_REQUIRE(max_q_len > 0, "zk_attention_bf16: max_q_len must be positive");
  hipStream_t s = (hipStream_t)stream;
  AttnParams p;
  p.q = (const __bf16*)q; p.q_stride = q_stride;
  p.kcache = (const __bf16*)kcache; p.vcache = (const __bf16*)vcache_t; p.v_shift = v_shift;
  p.block_table = block_table; p.max_blocks = max_blocks;
  p.q_start = q_start; p.ctx_len = ctx_len; p.out = (__bf16*)out;
  p.nh = nh; p.nkv = nkv; p.hd = hd; p.vd = vd; p.bs = bs; p.keep = keep;
  p.scale = scale; p.softcap = softcap; p.window = window;
  p.from_window = 0;
  p.mask_chunk = mask_chunk; p.sink = sink ? 1 : 0; p.wide_weights = wide_weights ? 1 : 0;
  p.sinks = sinks; p.gate = (const __bf16*)gate; p.gate_ld = gate_ld;
  p.bs_shift = 0;
  while ((1 << p.bs_shift) < bs) p.bs_shift++;
  const float log2e = 1.4426950408889634f;
  p.k1 = scale * log2e;
  p.k2 = softcap > 0.f ? 2.f * scale / softcap * log2e : 0.f;
  p.c2 = softcap * log2e;
  const int g = nh / nkv;
  if (r_prefill > 0) {
    p.tpw = 32 / g; p.r_begin = 0; p.nchunks = 1; p.part_o = nullptr; p.part_ml = nullptr;
    const int groups = (max_q_len + p.tpw - 1) / p.tpw;
    size_t split_at = 0;
    if (R - r_prefill > 0) split_at = (zk_attention_bf16_workspace(R - r_prefill, nh, vd, max_ctx) + 255) / 256 * 256;
    const bool usable = workspace != nullptr && (uintptr_t)workspace % 16 == 0 && split_at < workspace_bytes;
    const PortionForm form = portion_form(r_prefill, max_q_len, portion_ctx ? portion_ctx : max_ctx, !portion_ctx && R > r_prefill, nh, nkv,
                                          hd, vd, bs, window, mask_chunk, keep, wide_weights, usable ? workspace_bytes - split_at : 0);
    int rc;
    if (form.what == ATT_SHORT) {
      const int tokens = 16 / g;
      rc = launch_attn(ATT_SHORT, p, dim3((max_q_len + tokens - 1) / tokens, nkv, r_prefill), s);
    } else if (form.what == ATT_RANGES) {
      const int per_block = 4 * p.tpw, most_ranges = form.most_ranges;
      AttnParams ps = p;
      ps.chunk = form.range_tiles;
      ps.nchunks = most_ranges;
      const int row_blocks = (max_q_len + per_block - 1) / per_block;
      const size_t slots = (size_t)r_prefill * nkv * row_blocks * most_ranges * 4;
      const int dts = (vd + 31) / 32;
      ps.part_o = (float*)((char*)workspace + split_at);
      ps.part_ml = ps.part_o + slots * dts * 16 * 64;
      dim3 grid(row_blocks * most_ranges, nkv, r_prefill);
      rc = launch_attn(ATT_RANGES, ps, grid, s);
      if (rc) return rc;
      attn_portion_join_kernel<<<dim3(row_blocks * 4 * dts, nkv, r_prefill), 64, 0, s>>>(ps, per_block, row_blocks, dts);
      rc = zk_launch_status("zk_attention_bf16 (join of the portions' ranges)");
    } else {
      const int a_block = form.what == ATT_SHARED8 ? 8 : form.what == ATT_SHARED4 ? 4 : form.what == ATT_PAIRS ? 2 : 1;
      rc = launch_attn(form.what, p, dim3((groups + a_block - 1) / a_block, nkv, r_prefill), s);
    }
    if (rc) return rc;
  }
  const int n_dec = R - r_prefill;
  if (n_dec > 0) {
    const int nchunks = (max_ctx + ATT_CHUNK - 1) / ATT_CHUNK;
    p.tpw = 1; p.r_begin = r_prefill; p.nchunks = nchunks;
    p.part_o = (float*)workspace;
    p.part_ml = (float*)workspace + (size_t)n_dec * nh * nchunks * vd;
    dim3 grid((nchunks + 3) / 4, nkv, n_dec);
    int rc = 0;
    int span = ATT_CHUNK;        // keys one partial result covers
    if (decode_on_narrow_tiles(nh, nkv, hd)) {
      // a block joins its four waves: one partial result per block of keys
      const bool long_blocks = decode_in_long_blocks(nh, nkv, hd, vd, bs, max_blocks, decode_chunk);
      p.chunk = ATT_CHUNK;
      span = long_blocks ? 4 * p.chunk : ATT_DECODE_SPAN;
      grid.x = (max_ctx + span - 1) / span;
      p.nchunks = grid.x;
      // a window covers at most ceil(window / span) + 1 blocks of span keys
      const int reach = mask_chunk > 0 ? mask_chunk : window;
      const int window_blocks = reach > 0 ? (reach + span - 1) / span + 1 + (keep + span - 1) / span : 0;
      if (reach > 0 && window_blocks < (int)grid.x) {
        p.from_window = 1;
        grid.x = window_blocks;
      }
      p.part_ml = (float*)workspace + (size_t)n_dec * nh * p.nchunks * vd;
      const bool past = values_past_caches(once, bs, v_shift, long_blocks);
      rc = launch_attn(long_blocks ? (past ? ATT_DECODE_LONG_ONCE : ATT_DECODE_LONG) : past ? ATT_DECODE_ONCE : ATT_DECODE, p, grid, s);
    } else {
      rc = launch_attn(ATT_DECODE_WIDE, p, grid, s);
    }
    if (rc) return rc;
    dim3 cgrid(n_dec, nh);
    attn_combine_kernel<<<cgrid, 256, 0, s>>>(p.part_o, p.part_ml, q_start, ctx_len, (__bf16*)out, nh, vd,
                                              window, r_prefill, p.nchunks, span, mask_chunk, sink, keep, sinks,
                                              (const __bf16*)gate, gate_ld);
    return zk_launch_status("zk_attention_bf16 (combine)");
  }
  return 0;
}

int zk_attention_bf16_step(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                           const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                           void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                           int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                           void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                           int v_shift, int vd, int keep, const float* sinks, const void* gate, int gate_ld,
                           int portion_ctx, void* stream) {
  return zk_attention_bf16_once(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                workspace, workspace_bytes, mask_chunk, sink, wide_weights, v_shift, vd, keep, sinks, gate,
                                gate_ld, portion_ctx, 0, stream);
}

int zk_attention_bf16_gated(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                           const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                           void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                           int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                           void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                           int v_shift, int vd, int keep, const float* sinks, const void* gate, int gate_ld,
                           void* stream) {
  return zk_attention_bf16_step(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                workspace, workspace_bytes, mask_chunk, sink, wide_weights, v_shift, vd, keep, sinks, gate,
                                gate_ld, 0, stream);
}

int zk_attention_bf16_sized(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                           const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                           void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                           int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                           void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                           int v_shift, int vd, int keep, void* stream) {
  return zk_attention_bf16_gated(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                 r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                 workspace, workspace_bytes, mask_chunk, sink, wide_weights, v_shift, vd, keep, nullptr,
                                 nullptr, 0, stream);
}

int zk_attention_bf16_maps(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                           const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                           void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                           int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                           void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                           int v_shift, void* stream) {
  return zk_attention_bf16_sized(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                 r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                 workspace, workspace_bytes, mask_chunk, sink, wide_weights, v_shift, hd, 0, stream);
}

int zk_attention_bf16_masked(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                             const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                             void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                             int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                             void* workspace, size_t workspace_bytes, int mask_chunk, int sink, int wide_weights,
                             void* stream) {
  return zk_attention_bf16_maps(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                workspace, workspace_bytes, mask_chunk, sink, wide_weights, 0, stream);
}

int zk_attention_bf16(const void* q, int q_stride, const void* kcache, const void* vcache_t,
                      const int* block_table, int max_blocks, const int* q_start, const int* ctx_len,
                      void* out, int R, int r_prefill, int max_q_len, int max_ctx, int nh, int nkv,
                      int hd, int bs, float scale, float softcap, int window, int decode_chunk,
                      void* workspace, size_t workspace_bytes, void* stream) {
  return zk_attention_bf16_masked(q, q_stride, kcache, vcache_t, block_table, max_blocks, q_start, ctx_len, out, R,
                                  r_prefill, max_q_len, max_ctx, nh, nkv, hd, bs, scale, softcap, window, decode_chunk,
                                  workspace, workspace_bytes, 0, 0, 0, stream);
}

}  // extern "C"

extern "C" int zk_steplist_register(const char* name, int nargs, void* fn);
static const int zk_attention_bf16_masked_entered = zk_steplist_register(
    "zk_attention_bf16_masked", zk_packed::Call<zk_attention_bf16_masked>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_masked>::call);

static const int zk_attention_bf16_step_entered = zk_steplist_register(
    "zk_attention_bf16_step", zk_packed::Call<zk_attention_bf16_step>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_step>::call);

static const int zk_attention_bf16_once_entered = zk_steplist_register(
    "zk_attention_bf16_once", zk_packed::Call<zk_attention_bf16_once>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_once>::call);

static const int zk_attention_bf16_gated_entered = zk_steplist_register(
    "zk_attention_bf16_gated", zk_packed::Call<zk_attention_bf16_gated>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_gated>::call);

static const int zk_attention_bf16_sized_entered = zk_steplist_register(
    "zk_attention_bf16_sized", zk_packed::Call<zk_attention_bf16_sized>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_sized>::call);

static const int zk_attention_bf16_maps_entered = zk_steplist_register(
    "zk_attention_bf16_maps", zk_packed::Call<zk_attention_bf16_maps>::nargs,
    (void*)zk_packed::Call<zk_attention_bf16_maps>::call);

#endif  // ZSE_ACT_BF16
