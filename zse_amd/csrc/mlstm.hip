// Matrix-memory recurrence (mLSTM of xLSTM), one block per (request, head), token by token.
//
// Per head, with D query/key channels and E value channels, a state (S [D, E], n [D], m) that
// starts at zero and lives as floats in the request's state slot:
//
//   i_t = cap tanh((gi_t + bi) / cap)            f_t = logsigmoid(cap tanh((gf_t + bf) / cap))
//   m_t = max(f_t + m_(t-1), i_t)
//   S_t = exp(f_t + m_(t-1) - m_t) S_(t-1) + exp(i_t - m_t) k_t v_t^T        (n_t likewise with k_t alone)
//   o_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6),      q_t already times D^(-1/2) here
//   out_t = o_t / sqrt(mean(o_t^2) + eps) * g[head] * sigmoid(z_t)
//
// q, k, v and z come from one product in the activation type; gi, gf are float.  Everything
// above is float.  The order of every sum depends on the token alone, so a request's values
// do not depend on how its tokens are cut into steps or on what else a step holds.
#include "common.h"
#include "packed_call.h"

#include <type_traits>

extern "C" int zk_steplist_register(const char* name, int nargs, void* fn);
#define ZK_ENTER(fn) \
  static const int fn##_entered = zk_steplist_register(#fn, zk_packed::Call<fn>::nargs, (void*)zk_packed::Call<fn>::call);

#define MLSTM_THREADS 256

__device__ __forceinline__ float log_sigmoid(float x) {
  // min(x, 0) - log1p(exp(-|x|))
  return fminf(x, 0.f) - log1pf(expf(-fabsf(x)));
}

// DIRECT: S stays in the state slot and every element is read, renewed and written back once per
// token, many loads in flight (steps of single tokens, where staging S through the local memory
// would only add two passes); else S is staged for the step's tokens.  The same arithmetic in
// the same order either way.
template <bool DIRECT>
__global__ __launch_bounds__(MLSTM_THREADS) void mlstm_kernel(
    const act_t* __restrict__ qkvz, int ld, const float* __restrict__ gates, const float* __restrict__ bias_i,
    const float* __restrict__ bias_f, const float* __restrict__ norm_w, float* __restrict__ state, int slot_words,
    int offset_words, const int* __restrict__ q_start, const int* __restrict__ slot_of_req, act_t* __restrict__ out,
    int H, int D, int E, float cap, float eps, float q_scale) {
  extern __shared__ float lds[];
  const int r = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x;
  const int t0 = q_start[r], t1 = q_start[r + 1];
  if (t1 <= t0) return;                       // a padding request of a captured step
  const size_t per_head = (size_t)D * E + D + 1;
  float* st = state + (size_t)slot_of_req[r] * slot_words + offset_words + (size_t)hd * per_head;
  float* S = DIRECT ? st : lds;                // [D][E]
  float* n = DIRECT ? lds : lds + (size_t)D * E;      // [D]
  float* sq = n + D;                           // [D]
  float* sk = sq + D;                          // [D]
  float* sv = sk + D;                          // [E]
  float* part = sv + E;                        // [slices][E]
  float* red = part + MLSTM_THREADS;           // 17 + 1
  if (DIRECT) {
    for (int d = tid; d < D; d += MLSTM_THREADS) n[d] = st[(size_t)D * E + d];
  } else {
    for (int i = tid; i < D * E + D; i += MLSTM_THREADS) lds[i] = st[i];
  }
  float m = st[(size_t)D * E + D];
  const int slices = MLSTM_THREADS / E > 0 ? MLSTM_THREADS / E : 1;     // E <= 256
  const int e = tid % E, sl = tid / E;
  const bool active = sl < slices;
  const int per = (D + slices - 1) / slices;
  const int d0 = sl * per, d1 = min(D, d0 + per);
  const float bi = bias_i[hd], bf = bias_f[hd];
  __syncthreads();
  for (int t = t0; t < t1; t++) {
    const act_t* row = qkvz + (size_t)t * ld;
    for (int d = tid; d < D; d += MLSTM_THREADS) {
      sq[d] = to_f32(row[(size_t)hd * D + d]) * q_scale;
      sk[d] = to_f32(row[(size_t)(H + hd) * D + d]);
    }
    for (int c = tid; c < E; c += MLSTM_THREADS) sv[c] = to_f32(row[(size_t)2 * H * D + (size_t)hd * E + c]);
    const float gi = cap * tanhf((gates[(size_t)t * 2 * H + hd] + bi) / cap);
    const float gf = log_sigmoid(cap * tanhf((gates[(size_t)t * 2 * H + H + hd] + bf) / cap));
    const float m_new = fmaxf(gf + m, gi);
    const float a = expf(gf + m - m_new), b = expf(gi - m_new);
    m = m_new;
    __syncthreads();
    // S and the numerator: a thread owns value channel e and a slice of the key channels
    if (active) {
      const float bv = b * sv[e];
      float acc = 0.f;
      // eight elements of S are asked for before the first of them is written back: the loads
      // of a thread's column are then in flight together (the sums keep their order)
      for (int d = d0; d < d1; d += 8) {
        float old[8];
#pragma unroll
        for (int x = 0; x < 8; x++) old[x] = d + x < d1 ? S[(size_t)(d + x) * E + e] : 0.f;
#pragma unroll
        for (int x = 0; x < 8; x++)
          if (d + x < d1) {
            const float s = fmaf(a, old[x], sk[d + x] * bv);
            S[(size_t)(d + x) * E + e] = s;
            acc = fmaf(s, sq[d + x], acc);
          }
      }
      part[sl * E + e] = acc;
    }
    // n and n . q
    float nq = 0.f;
    for (int d = tid; d < D; d += MLSTM_THREADS) {
      const float v = fmaf(a, n[d], b * sk[d]);
      n[d] = v;
      nq = fmaf(v, sq[d], nq);
    }
    nq = block_sum_whole(nq, red);              // syncs: part[] is complete after it
    const float den = fmaxf(fabsf(nq), expf(-m)) + 1e-6f;
    float o = 0.f;
    if (tid < E) {
      for (int s2 = 0; s2 < slices; s2++) o += part[s2 * E + tid];
      o = o / den;
    }
    const float ms = block_sum_whole(tid < E ? o * o : 0.f, red) / (float)E;
    if (tid < E) {
      const size_t col = (size_t)hd * E + tid;
      const float z = to_f32(row[(size_t)2 * H * D + (size_t)H * E + col]);
      const float y = o / sqrtf(ms + eps) * norm_w[col] * (1.0f / (1.0f + expf(-z)));
      out[(size_t)t * H * E + col] = from_f32<act_t>(y);
    }
    __syncthreads();
  }
  if (DIRECT) {
    for (int d = tid; d < D; d += MLSTM_THREADS) st[(size_t)D * E + d] = n[d];
  } else {
    for (int i = tid; i < D * E + D; i += MLSTM_THREADS) st[i] = lds[i];
  }
  if (tid == 0) st[(size_t)D * E + D] = m;
}

// ---- the same recurrence over chunks of L tokens, for steps that bring portions of prompts.
//
// Inside a chunk that starts from the state (S0, n0, m0), with F_j the sum of the forget gates up
// to token j of the chunk and a_s = i_s - F_s:
//
//   M_j = max(m0, max_{s<=j} a_s)                     m_j = F_j + M_j
//   P_js = (q_j . k_s) exp(a_s - M_j)  for s <= j     g_j = exp(m0 - M_j)
//   S_j^T q_j = g_j S0^T q_j + sum_s P_js v_s         n_j . q_j = g_j n0 . q_j + sum_s P_js
//
// which is the token-by-token recurrence written out (every exponent is <= 0).  At the chunk's
// last token the state becomes g S0 + sum_s exp(a_s - M) k_s v_s^T.  So a chunk is four small
// matrix products (q k^T, P v, q S0, k^T v) instead of L dependent steps.  A block owns 32
// value channels of a head: the recurrence never mixes value channels, only the norm over a
// head's read-out does, and that (with the gain and the output gate) is left to a second
// kernel, which also stores the new n and m: every block of a head computes them, none may
// store them while another still reads the old ones.
#define MLSTM_EC 32

__device__ __forceinline__ void load8(const float* p, float v[8]) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ __forceinline__ void load8(const __bf16* p, float v[8]) {
  typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
  const bf8 a = *(const bf8*)p;
#pragma unroll
  for (int x = 0; x < 8; x++) v[x] = (float)a[x];
}

template <int L>
__global__ __launch_bounds__(MLSTM_THREADS) void mlstm_chunk_kernel(
    const act_t* __restrict__ qkvz, int ld, const float* __restrict__ gates, const float* __restrict__ bias_i,
    const float* __restrict__ bias_f, float* __restrict__ state, int slot_words, int offset_words,
    const int* __restrict__ q_start, const int* __restrict__ slot_of_req, float* __restrict__ o_raw,
    float* __restrict__ nm_new, int H, int D, int E, float cap, float q_scale) {
  constexpr int EC = MLSTM_EC;
  constexpr int TP = L / 16;
  extern __shared__ float lds[];
  const int r = blockIdx.x, hd = blockIdx.y, e0 = blockIdx.z * EC, tid = threadIdx.x;
  const int t0 = q_start[r], t1 = q_start[r + 1];
  if (t1 <= t0) return;
  const int DP = D + 1, LP = L + 1;
  float* Ss = lds;                      // [D][EC]   this block's columns of S
  float* ns = Ss + (size_t)D * EC;      // [D]
  float* Qs = ns + D;                   // [L][DP]
  float* Ks = Qs + (size_t)L * DP;      // [L][DP]
  float* Vs = Ks + (size_t)L * DP;      // [L][EC]
  float* Ps = Vs + (size_t)L * EC;      // [L][LP]
  float* ga = Ps + (size_t)L * LP;      // a_s, then (after the scan) i_s - F_s
  float* gM = ga + L;                   // M_j
  float* gF = gM + L;                   // f_s, then F_j
  float* gden = gF + L;                 // denominators
  float* gw = gden + L;                 // exp(a_s - M_last)
  const size_t per_head = (size_t)D * E + D + 1;
  float* st = state + (size_t)slot_of_req[r] * slot_words + offset_words + (size_t)hd * per_head;
  for (int i = tid; i < D * EC; i += MLSTM_THREADS) {
    const int d = i / EC, e = e0 + i % EC;
    Ss[i] = e < E ? st[(size_t)d * E + e] : 0.f;
  }
  for (int d = tid; d < D; d += MLSTM_THREADS) ns[d] = st[(size_t)D * E + d];
  float m_prev = st[(size_t)D * E + D];
  const float bi = bias_i[hd], bf = bias_f[hd];
  const bool vec8 = D % 8 == 0 && ld % 8 == 0 && (uintptr_t)qkvz % 16 == 0;
  __syncthreads();
  for (int c0 = t0; c0 < t1; c0 += L) {
    const int Lc = min(L, t1 - c0);
    if (vec8) {      // eight channels a load
      const int D8 = D / 8;
      for (int i = tid; i < L * D8; i += MLSTM_THREADS) {
        const int j = i / D8, d = (i % D8) * 8;
        float q[8] = {}, k[8] = {};
        if (j < Lc) {
          const act_t* row = qkvz + (size_t)(c0 + j) * ld;
          load8(row + (size_t)hd * D + d, q);
          load8(row + (size_t)(H + hd) * D + d, k);
        }
#pragma unroll
        for (int x = 0; x < 8; x++) {
          Qs[j * DP + d + x] = q[x] * q_scale;
          Ks[j * DP + d + x] = k[x];
        }
      }
    } else {
      for (int i = tid; i < L * D; i += MLSTM_THREADS) {
        const int j = i / D, d = i % D;
        float q = 0.f, k = 0.f;
        if (j < Lc) {
          const act_t* row = qkvz + (size_t)(c0 + j) * ld;
          q = to_f32(row[(size_t)hd * D + d]) * q_scale;
          k = to_f32(row[(size_t)(H + hd) * D + d]);
        }
        Qs[j * DP + d] = q;
        Ks[j * DP + d] = k;
      }
    }
    for (int i = tid; i < L * EC; i += MLSTM_THREADS) {
      const int j = i / EC, e = e0 + i % EC;
      Vs[i] = (j < Lc && e < E) ? to_f32(qkvz[(size_t)(c0 + j) * ld + (size_t)2 * H * D + (size_t)hd * E + e]) : 0.f;
    }
    if (tid < Lc) {
      const size_t t = c0 + tid;
      ga[tid] = cap * tanhf((gates[t * 2 * H + hd] + bi) / cap);
      gF[tid] = log_sigmoid(cap * tanhf((gates[t * 2 * H + H + hd] + bf) / cap));
    }
    __syncthreads();
    if (tid < ZSE_WAVE) {      // running sums of the forget gates and running maxima of a, over one wave (L <= 64)
      const int j = tid;
      float F = j < Lc ? gF[j] : 0.f;
#pragma unroll
      for (int o = 1; o < ZSE_WAVE; o <<= 1) {
        const float up = __shfl_up(F, o, ZSE_WAVE);
        if (j >= o) F += up;
      }
      const float a = j < Lc ? ga[j] - F : -INFINITY;
      float M = a;
#pragma unroll
      for (int o = 1; o < ZSE_WAVE; o <<= 1) {
        const float up = __shfl_up(M, o, ZSE_WAVE);
        if (j >= o) M = fmaxf(M, up);
      }
      if (j < L) {
        ga[j] = a;
        gM[j] = fmaxf(M, m_prev);
        gF[j] = F;
      }
    }
    __syncthreads();
    {  // P
      // rows pj + 16 a, columns ps + 16 b: neighbouring lanes read neighbouring rows of K
      const int pj = tid / 16, ps = tid % 16;
      float acc[TP][TP] = {};
      for (int d = 0; d < D; d++) {
        float q[TP], k[TP];
#pragma unroll
        for (int x = 0; x < TP; x++) {
          q[x] = Qs[(pj + 16 * x) * DP + d];
          k[x] = Ks[(ps + 16 * x) * DP + d];
        }
#pragma unroll
        for (int a = 0; a < TP; a++)
#pragma unroll
          for (int b = 0; b < TP; b++) acc[a][b] = fmaf(q[a], k[b], acc[a][b]);
      }
#pragma unroll
      for (int a = 0; a < TP; a++)
#pragma unroll
        for (int b = 0; b < TP; b++) {
          const int j = pj + 16 * a, s2 = ps + 16 * b;
          Ps[j * LP + s2] = (s2 <= j && j < Lc) ? acc[a][b] * expf(ga[s2] - gM[j]) : 0.f;
        }
    }
    __syncthreads();
    if (tid < L) {  // denominators
      const int j = tid;
      float nq = 0.f;
      for (int d = 0; d < D; d++) nq = fmaf(ns[d], Qs[j * DP + d], nq);
      nq *= expf(m_prev - gM[j]);
      for (int s2 = 0; s2 <= j; s2++) nq += Ps[j * LP + s2];
      gden[j] = fmaxf(fabsf(nq), expf(-(gF[j] + gM[j]))) + 1e-6f;
      gw[j] = j < Lc ? expf(ga[j] - gM[Lc - 1]) : 0.f;
    }
    {  // read-out: TP rows, columns ec, ec + 1
      const int ec = (tid % 16) * 2, rg = tid / 16;        // rows rg + 16 a
      float acc[TP][2] = {};
      for (int d = 0; d < D; d++) {
        const float s0 = Ss[d * EC + ec], s1 = Ss[d * EC + ec + 1];
#pragma unroll
        for (int a = 0; a < TP; a++) {
          const float q = Qs[(rg + 16 * a) * DP + d];
          acc[a][0] = fmaf(q, s0, acc[a][0]);
          acc[a][1] = fmaf(q, s1, acc[a][1]);
        }
      }
#pragma unroll
      for (int a = 0; a < TP; a++) {
        const float g = expf(m_prev - gM[rg + 16 * a]);
        acc[a][0] *= g;
        acc[a][1] *= g;
      }
      for (int s2 = 0; s2 < Lc; s2++) {
        const float v0 = Vs[s2 * EC + ec], v1 = Vs[s2 * EC + ec + 1];
#pragma unroll
        for (int a = 0; a < TP; a++) {
          const float p = Ps[(rg + 16 * a) * LP + s2];
          acc[a][0] = fmaf(p, v0, acc[a][0]);
          acc[a][1] = fmaf(p, v1, acc[a][1]);
        }
      }
      __syncthreads();          // the denominators are there; every read of Vs is done
#pragma unroll
      for (int a = 0; a < TP; a++) {
        const int j = rg + 16 * a;
        if (j < Lc) {
          float* o = o_raw + ((size_t)(c0 + j) * H + hd) * E;
          if (e0 + ec < E) o[e0 + ec] = acc[a][0] / gden[j];
          if (e0 + ec + 1 < E) o[e0 + ec + 1] = acc[a][1] / gden[j];
        }
      }
    }
    // the state after the chunk's last token
    const float M_last = gM[Lc - 1];
    const float g_last = expf(m_prev - M_last);
    const float m_next = gF[Lc - 1] + M_last;
    for (int i = tid; i < L * EC; i += MLSTM_THREADS) Vs[i] *= gw[i / EC];
    for (int d = tid; d < D; d += MLSTM_THREADS) {
      float acc = 0.f;
      for (int s2 = 0; s2 < Lc; s2++) acc = fmaf(gw[s2], Ks[s2 * DP + d], acc);
      ns[d] = fmaf(g_last, ns[d], acc);
    }
    __syncthreads();
    {
      const int ec = (tid % 16) * 2, dg = (tid / 16) * 4;
      for (int db = 0; db < D; db += 64) {
        float acc[4][2] = {};
        const int d = db + dg;
        for (int s2 = 0; s2 < Lc; s2++) {
          const float v0 = Vs[s2 * EC + ec], v1 = Vs[s2 * EC + ec + 1];
#pragma unroll
          for (int a = 0; a < 4; a++) {
            const float k = d + a < D ? Ks[s2 * DP + d + a] : 0.f;
            acc[a][0] = fmaf(k, v0, acc[a][0]);
            acc[a][1] = fmaf(k, v1, acc[a][1]);
          }
        }
#pragma unroll
        for (int a = 0; a < 4; a++)
          if (d + a < D) {
            float* sp = Ss + (size_t)(d + a) * EC + ec;
            sp[0] = fmaf(g_last, sp[0], acc[a][0]);
            sp[1] = fmaf(g_last, sp[1], acc[a][1]);
          }
      }
    }
    m_prev = m_next;
    __syncthreads();
  }
  for (int i = tid; i < D * EC; i += MLSTM_THREADS) {
    const int d = i / EC, e = e0 + i % EC;
    if (e < E) st[(size_t)d * E + e] = Ss[i];
  }
  if (blockIdx.z == 0) {
    float* nm = nm_new + ((size_t)r * H + hd) * (D + 1);
    for (int d = tid; d < D; d += MLSTM_THREADS) nm[d] = ns[d];
    if (tid == 0) nm[D] = m_prev;
  }
}

// The read-out's norm over each head, gain and output gate; the block of a request's last
// token also stores the head's new n and m.
__global__ __launch_bounds__(64) void mlstm_finish_kernel(
    const float* __restrict__ o_raw, const act_t* __restrict__ qkvz, int ld, const float* __restrict__ norm_w,
    const float* __restrict__ nm_new, float* __restrict__ state, int slot_words, int offset_words,
    const int* __restrict__ req_of_token, const int* __restrict__ q_start, const int* __restrict__ slot_of_req,
    act_t* __restrict__ out, int H, int D, int E, float eps) {
  const int t = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x;
  const float* o = o_raw + ((size_t)t * H + hd) * E;
  float ss = 0.f;
  for (int e = lane; e < E; e += 64) ss = fmaf(o[e], o[e], ss);
  const float inv = 1.0f / sqrtf(wave_sum_whole(ss) / (float)E + eps);
  const act_t* z = qkvz + (size_t)t * ld + (size_t)2 * H * D + (size_t)H * E + (size_t)hd * E;
  for (int e = lane; e < E; e += 64) {
    const float y = o[e] * inv * norm_w[(size_t)hd * E + e] * (1.0f / (1.0f + expf(-to_f32(z[e]))));
    out[((size_t)t * H + hd) * E + e] = from_f32<act_t>(y);
  }
  if (nm_new == nullptr) return;
  const int r = req_of_token[t];
  if (t == q_start[r + 1] - 1) {
    float* st = state + (size_t)slot_of_req[r] * slot_words + offset_words + (size_t)hd * ((size_t)D * E + D + 1) + (size_t)D * E;
    const float* nm = nm_new + ((size_t)r * H + hd) * (D + 1);
    for (int d = lane; d <= D; d += 64) st[d] = nm[d];
  }
}

// ---- the chunks of long portions side by side, in three launches.
//
// The chunk kernel above walks a request's chunks one after the other, since each starts from the
// state the one before left: a head keeps at most a few blocks busy however long the portion.
// What a chunk adds to the state does not depend on that state, though:
//
//   local  (every chunk at once):   A = max_s a_s,  U = sum_s exp(a_s - A) k_s v_s^T,  u likewise,  F = F_L
//   scan   (chunk after chunk, one multiply-add per element of the state):
//          M = max(m0, A),  S0' = exp(m0 - M) S0 + exp(A - M) U,  m0' = F + M;   S0, n0, m0 of every chunk are kept
//   output (every chunk at once):   the read-out of the chunk kernel from the kept S0, n0, m0
//
// Chunks are numbered through the step's requests (request r has ceil(n_r / L) of them).  U is stored where
// the scan then leaves S0 of that chunk.
//
// The products run on the 32-bit matrix cores (16x16x4), whose operands take q, k and P from the
// local memory and S0, v and U straight from and to memory: a wave owns 32 value channels and goes through
// all rows, so each of their elements is fetched once, on its way while the scores are made.  What is
// left is the chain of loads, scores, read-out of one block a head and chunk.  Multiply-adds out of
// the local memory, a block a head, chunk and 32 value channels, the chunks of a request after each other in the scan
// with a wait for memory at each, took (us; 700 tokens and 8 single ones, 16 heads of 64 key and 128 value channels)
// local 17.7, scan 15.1, output 58.0; so 12.0, 13.0 and 19.5 (of which
// the 32-bit matrix cores of the CUs that have a full chunk are busy for 8).
#define MLSTM_EB 128             // value channels a block: 32 for each of its four waves
typedef float mlstm_f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mlstm_f4 mlstm_mfma(float a, float b, mlstm_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Key channels in the local memory: whole groups of 16, the rest zero, and four more that spread the rows over
// the banks (and keep them 16-byte pieces).
__host__ __device__ __forceinline__ int mlstm_pitch(int D) { return (D + 15) / 16 * 16 + 4; }

// Rows [0, L) of a chunk's q (part 0, times ``scale``) or k (part 1) as floats, zero beyond Lc and D.
template <int L>
__device__ __forceinline__ void mlstm_stage(const act_t* __restrict__ qkvz, int ld, int c0, int Lc, int hd, int part, int H, int D,
                                            float scale, float* dst) {
  const int P = mlstm_pitch(D), first = (part * H + hd) * D;
  if (D % 8 == 0 && ld % 8 == 0 && (uintptr_t)qkvz % 16 == 0) {      // eight channels a load
    const int groups = (P - 4) / 8;
    for (int i = threadIdx.x; i < L * groups; i += MLSTM_THREADS) {
      const int j = i / groups, d = (i % groups) * 8;
      float v[8] = {};
      if (j < Lc && d < D) load8(qkvz + (size_t)(c0 + j) * ld + first + d, v);
      *(float4*)(dst + j * P + d) = make_float4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
      *(float4*)(dst + j * P + d + 4) = make_float4(v[4] * scale, v[5] * scale, v[6] * scale, v[7] * scale);
    }
  } else {
    for (int i = threadIdx.x; i < L * (P - 4); i += MLSTM_THREADS) {
      const int j = i / (P - 4), d = i % (P - 4);
      dst[j * P + d] = j < Lc && d < D ? to_f32(qkvz[(size_t)(c0 + j) * ld + first + d]) * scale : 0.f;
    }
  }
}

// The gates of the chunk's token j (lane j of a wave): asked for here ...
struct MlstmGate {
  float i, f, bias_i, bias_f;
};
__device__ __forceinline__ MlstmGate mlstm_gate_load(const float* __restrict__ gates, const float* __restrict__ bias_i,
                                                     const float* __restrict__ bias_f, int c0, int Lc, int hd, int H, int j) {
  const float* g = gates + (size_t)(c0 + min(j, Lc - 1)) * 2 * H + hd;
  return {g[0], g[H], bias_i[hd], bias_f[hd]};
}
// ... and worked out here: a_j (-inf beyond Lc) and the running sum F_j.
__device__ __forceinline__ void mlstm_gates(const MlstmGate& g, int Lc, float cap, int j, float& a, float& F) {
  const float gi = cap * tanhf((g.i + g.bias_i) / cap);
  const float f = log_sigmoid(cap * tanhf((g.f + g.bias_f) / cap));
  F = wave_running_sum(j < Lc ? f : 0.f);
  a = j < Lc ? gi - F : -INFINITY;
}

// Channels e and e + 1 of a row of E (zero from E on and where the row is not there); PAIRS: rows in whole pairs
template <bool PAIRS, typename T>
__device__ __forceinline__ void mlstm_pair(const T* __restrict__ row, int e, int E, bool there, float (&v)[2]) {
  if constexpr (PAIRS) {
    typedef T t2 __attribute__((ext_vector_type(2)));
    const t2 x = *(const t2*)(row + min(e, E - 2));
    v[0] = there && e < E ? to_f32(x[0]) : 0.f;
    v[1] = there && e < E ? to_f32(x[1]) : 0.f;
  } else {
    const float x = to_f32(row[min(e, E - 1)]), y = to_f32(row[min(e + 1, E - 1)]);
    v[0] = there && e < E ? x : 0.f;
    v[1] = there && e + 1 < E ? y : 0.f;
  }
}
template <bool PAIRS>
__device__ __forceinline__ void mlstm_put(float* __restrict__ row, int e, int E, float x, float y) {
  if constexpr (PAIRS) {
    if (e < E) *(float2*)(row + e) = make_float2(x, y);
  } else {
    if (e < E) row[e] = x;
    if (e + 1 < E) row[e + 1] = y;
  }
}

// Tiles of 16 tokens that a chunk of L uses: one, or all of them.
#define MLSTM_TILES(L, Lc, f)                           \
  do {                                                  \
    if ((Lc) <= 16) f(std::integral_constant<int, 1>{}); \
    else f(std::integral_constant<int, (L) / 16>{});    \
  } while (0)

template <int L, bool PAIRS>
__global__ __launch_bounds__(MLSTM_THREADS) void mlstm_local_kernel(
    const act_t* __restrict__ qkvz, int ld, const float* __restrict__ gates, const float* __restrict__ bias_i,
    const float* __restrict__ bias_f, const int* __restrict__ q_start, float* __restrict__ Uw, float* __restrict__ uw,
    float* __restrict__ af, int R, int H, int D, int E, float cap) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int x = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, kq = lane >> 4;
  Piece at_chunk;
  if (!find_piece(q_start, R, L, x, at_chunk)) return;
  const int c0 = at_chunk.t0 + at_chunk.first, Lc = min(L, at_chunk.n - at_chunk.first);
  const int P = mlstm_pitch(D);
  float* Ks = lds;                       // [L][P]
  float* gw = Ks + (size_t)L * P;        // exp(a_s - A)
  const int e0 = blockIdx.z * MLSTM_EB + wave * 32 + 2 * lr;
  const act_t* v0 = qkvz + (size_t)c0 * ld + (size_t)2 * H * D + (size_t)hd * E;
  float* U = Uw + ((size_t)x * H + hd) * D * E;
  auto run = [&](auto tiles) {
    constexpr int KS = decltype(tiles)::value;
    MlstmGate gate;
    if (wave == 0) gate = mlstm_gate_load(gates, bias_i, bias_f, c0, Lc, hd, H, lane);
    mlstm_stage<16 * KS>(qkvz, ld, c0, Lc, hd, 1, H, D, 1.f, Ks);
    float v[KS][4][2];                   // token 16 g + 4 kq + i, channels e0 and e0 + 1
#pragma unroll
    for (int g = 0; g < KS; g++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 16 * g + 4 * kq + i;
        mlstm_pair<PAIRS>(v0 + (size_t)min(row, Lc - 1) * ld, e0, E, row < Lc, v[g][i]);
      }
    if (wave == 0) {
      float a, F;
      mlstm_gates(gate, Lc, cap, lane, a, F);
      const float A = wave_max_whole(a);
      if (lane < L) gw[lane] = lane < Lc ? expf(a - A) : 0.f;
      if (lane == Lc - 1 && blockIdx.z == 0) {
        af[((size_t)x * H + hd) * 2] = A;
        af[((size_t)x * H + hd) * 2 + 1] = F;
      }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < KS; g++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int c = 0; c < 2; c++) v[g][i][c] *= gw[16 * g + 4 * kq + i];
    for (int d0 = 0; d0 < D; d0 += 16) {
      float k[KS][4];
#pragma unroll
      for (int g = 0; g < KS; g++)
#pragma unroll
        for (int i = 0; i < 4; i++) k[g][i] = Ks[(16 * g + 4 * kq + i) * P + d0 + lr];
      mlstm_f4 acc[2] = {};
#pragma unroll
      for (int g = 0; g < KS; g++)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int c = 0; c < 2; c++) acc[c] = mlstm_mfma(k[g][i], v[g][i][c], acc[c]);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int d = d0 + 4 * kq + i;
        if (d < D) mlstm_put<PAIRS>(U + (size_t)d * E, e0, E, acc[0][i], acc[1][i]);
      }
    }
    if (blockIdx.z == 0)                 // u: four threads a channel
      for (int d0 = 0; d0 < D; d0 += MLSTM_THREADS / 4) {
        const int d = d0 + tid / 4;
        float acc = 0.f;
        if (d < D) {
#pragma unroll
          for (int s2 = 0; s2 < 4 * KS; s2++) acc = fmaf(gw[4 * s2 + tid % 4], Ks[(4 * s2 + tid % 4) * P + d], acc);
        }
        acc += wave_dpp<ZSE_DPP_XOR1>(acc);
        acc += wave_dpp<ZSE_DPP_XOR2>(acc);
        if (d < D && tid % 4 == 0) uw[((size_t)x * H + hd) * D + d] = acc;
      }
  };
  MLSTM_TILES(L, Lc, run);
}

// MLSTM_ELEMS elements of a head's state a thread (S, then n, then one more that writes down every chunk's m; the
// state's own m, which all threads read, is renewed by the output kernel).  Eight chunks' U are
// asked for at once: a store of S0 into the place of a U would otherwise hold back the next load.
#define MLSTM_ELEMS 4
__global__ __launch_bounds__(MLSTM_THREADS) void mlstm_scan_kernel(
    float* __restrict__ state, int slot_words, int offset_words, const int* __restrict__ q_start,
    const int* __restrict__ slot_of_req, float* __restrict__ Uw, float* __restrict__ uw, const float* __restrict__ af,
    float* __restrict__ mprev, int L, int H, int D, int E) {
  constexpr int AHEAD = 8, NE = MLSTM_ELEMS;
  const int r = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x & (ZSE_WAVE - 1);
  const int idx0 = blockIdx.z * (MLSTM_THREADS * NE) + threadIdx.x;      // and every MLSTM_THREADS further on
  const int DE = D * E, slot = slot_of_req[r];
  const int t0 = q_start[r], n = q_start[r + 1] - t0;
  int first = 0;                         // chunks of the requests in front of r
  for (int r0 = 0; r0 < r; r0 += ZSE_WAVE) {
    const int q = min(r0 + lane, r - 1);
    const int c = r0 + lane < r ? (q_start[q + 1] - q_start[q] + L - 1) / L : 0;
    first += __builtin_amdgcn_readlane(wave_running_sum(c), ZSE_WAVE - 1);
  }
  if (n <= 0 || idx0 > DE + D) return;
  const int nc = (n + L - 1) / L;
  float* st = state + (size_t)slot * slot_words + offset_words + (size_t)hd * ((size_t)DE + D + 1);
  float m = st[DE + D];
  float val[NE];
  float* p0[NE];                         // the element of chunk 0's U or u, and how far on the next chunk's is
  size_t step[NE];
#pragma unroll
  for (int k = 0; k < NE; k++) {
    const int idx = min(idx0 + k * MLSTM_THREADS, DE + D - 1);      // (past the last: the last again, not stored)
    val[k] = st[idx];
    p0[k] = idx < DE ? Uw + ((size_t)first * H + hd) * DE + idx : uw + ((size_t)first * H + hd) * D + (idx - DE);
    step[k] = (size_t)H * (idx < DE ? DE : D);
  }
  auto mine = [&](int k) { return idx0 + k * MLSTM_THREADS < DE + D; };
  const bool keeps_m = (DE + D - idx0) % MLSTM_THREADS == 0 && DE + D - idx0 < NE * MLSTM_THREADS;
  const float* g0 = af + ((size_t)first * H + hd) * 2;
  for (int c0 = 0; c0 < nc; c0 += AHEAD) {
    float U[AHEAD][NE], A[AHEAD], F[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int ci = min(c0 + i, nc - 1);
#pragma unroll
      for (int k = 0; k < NE; k++) U[i][k] = p0[k][ci * step[k]];
      A[i] = g0[(size_t)ci * H * 2];
      F[i] = g0[(size_t)ci * H * 2 + 1];
    }
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int ci = c0 + i;
      if (ci < nc) {
        const float M = fmaxf(m, A[i]), keep = expf(m - M), add = expf(A[i] - M);
#pragma unroll
        for (int k = 0; k < NE; k++)
          if (mine(k)) {
            p0[k][ci * step[k]] = val[k];                        // the state this chunk starts from
            val[k] = fmaf(keep, val[k], add * U[i][k]);
          }
        if (keeps_m) mprev[(size_t)(first + ci) * H + hd] = m;
        m = F[i] + M;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NE; k++)
    if (mine(k)) st[idx0 + k * MLSTM_THREADS] = val[k];
}

template <int L, bool PAIRS>
__global__ __launch_bounds__(MLSTM_THREADS) void mlstm_output_kernel(
    const act_t* __restrict__ qkvz, int ld, const float* __restrict__ gates, const float* __restrict__ bias_i,
    const float* __restrict__ bias_f, const int* __restrict__ q_start, const float* __restrict__ Sw,
    const float* __restrict__ nw, const float* __restrict__ mprev, float* __restrict__ o_raw, float* __restrict__ state,
    int slot_words, int offset_words, const int* __restrict__ slot_of_req, int R, int H, int D, int E, float cap, float q_scale) {
  constexpr int LP = L + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int x = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, kq = lane >> 4;
  Piece at_chunk;
  if (!find_piece(q_start, R, L, x, at_chunk)) return;
  const int c0 = at_chunk.t0 + at_chunk.first, Lc = min(L, at_chunk.n - at_chunk.first);
  const int P = mlstm_pitch(D);
  float* Qs = lds;                       // [L][P]
  float* Ks = Qs + (size_t)L * P;        // [L][P]
  float* Ps = Ks + (size_t)L * P;        // [L][LP]
  float* ns = Ps + (size_t)L * LP;       // [P]
  float* ga = ns + P;
  float* gM = ga + L;
  float* gF = gM + L;
  float* gden = gF + L;                  // n . q, then the denominators
  const size_t at = (size_t)x * H + hd;
  const int e0 = blockIdx.z * MLSTM_EB + wave * 32 + 2 * lr;
  const float* S0 = Sw + at * D * E;
  const act_t* v0 = qkvz + (size_t)c0 * ld + (size_t)2 * H * D + (size_t)hd * E;
  auto run = [&](auto tiles) {
    constexpr int RT = decltype(tiles)::value;             // tiles of 16 tokens
    MlstmGate gate;
    if (wave == 0) gate = mlstm_gate_load(gates, bias_i, bias_f, c0, Lc, hd, H, lane);
    const float m_prev = mprev[at];
    mlstm_stage<16 * RT>(qkvz, ld, c0, Lc, hd, 0, H, D, q_scale, Qs);
    mlstm_stage<16 * RT>(qkvz, ld, c0, Lc, hd, 1, H, D, 1.f, Ks);
    for (int d = tid; d < P; d += MLSTM_THREADS) ns[d] = d < D ? nw[at * D + d] : 0.f;
    // S0 of 64 key channels and v of the chunk's tokens, on their way from now on
    float sv[4][4][2], v[RT][4][2];
    auto fetch_s = [&](int d0) {
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int d = d0 + 16 * g + 4 * kq + i;
          mlstm_pair<PAIRS>(S0 + (size_t)min(d, D - 1) * E, e0, E, d < D, sv[g][i]);
        }
    };
    fetch_s(0);
#pragma unroll
    for (int g = 0; g < RT; g++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 16 * g + 4 * kq + i;
        mlstm_pair<PAIRS>(v0 + (size_t)min(row, Lc - 1) * ld, e0, E, row < Lc, v[g][i]);
      }
    if (wave == 0) {
      float a, F;
      mlstm_gates(gate, Lc, cap, lane, a, F);
      const float M = fmaxf(wave_running_max(a), m_prev);
      if (lane < L) {
        ga[lane] = a;
        gM[lane] = M;
        gF[lane] = F;
      }
      if (at_chunk.first + Lc == at_chunk.n && lane == Lc - 1 && blockIdx.z == 0)      // the request's last chunk
        state[(size_t)slot_of_req[at_chunk.r] * slot_words + offset_words + (size_t)hd * ((size_t)D * E + D + 1) + (size_t)D * E + D] =
            F + M;
    }
    __syncthreads();
    // P and the denominators: a wave takes every fourth tile of rows, all tiles of columns (zeros behind the diagonal)
    const int KS = (P - 4) / 16;           // groups of 16 key channels
#pragma unroll
    for (int a0 = 0; a0 < (RT + 3) / 4; a0++) {
      const int a = wave + 4 * a0;
      if (a >= RT) break;
      mlstm_f4 acc[RT];
#pragma unroll
      for (int b = 0; b < RT; b++) acc[b] = mlstm_f4{0.f, 0.f, 0.f, 0.f};
      float nq = 0.f;                      // n . q of row lr, the lane's channels
      for (int g = 0; g < KS; g++) {
        const float4 q = *(const float4*)(Qs + (16 * a + lr) * P + 16 * g + 4 * kq), n = *(const float4*)(ns + 16 * g + 4 * kq);
        const float qe[4] = {q.x, q.y, q.z, q.w};
        float ke[RT][4];
#pragma unroll
        for (int b = 0; b < RT; b++) {
          const float4 k = *(const float4*)(Ks + (16 * b + lr) * P + 16 * g + 4 * kq);
          ke[b][0] = k.x, ke[b][1] = k.y, ke[b][2] = k.z, ke[b][3] = k.w;
        }
        nq = fmaf(q.w, n.w, fmaf(q.z, n.z, fmaf(q.y, n.y, fmaf(q.x, n.x, nq))));
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int b = 0; b < RT; b++) acc[b] = mlstm_mfma(qe[i], ke[b][i], acc[b]);
      }
      float ps[4] = {};
#pragma unroll
      for (int b = 0; b < RT; b++) {
        const float as = ga[16 * b + lr];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int j = 16 * a + 4 * kq + i, s2 = 16 * b + lr;
          const float p = (s2 <= j && j < Lc) ? acc[b][i] * expf(as - gM[j]) : 0.f;
          Ps[j * LP + s2] = p;
          ps[i] += p;
        }
      }
      float x0 = 0.f, x1 = 0.f;
      wave_pair32(nq, x0, x1);
      wave_pair16(x0 + x1, x0, x1);
      if (kq == 0) gden[16 * a + lr] = x0 + x1;
#pragma unroll
      for (int i = 0; i < 4; i++) ps[i] = wave_sum16(ps[i]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");      // the wave reads what its other lanes wrote
      __builtin_amdgcn_wave_barrier();
      if (lr < 4) {                        // lane (lr, kq): row 4 kq + lr
        const int j = 16 * a + 4 * kq + lr;
        const float p = lr == 0 ? ps[0] : lr == 1 ? ps[1] : lr == 2 ? ps[2] : ps[3];
        const float den = fmaf(gden[j], expf(m_prev - gM[j]), p);
        gden[j] = 1.0f / (fmaxf(fabsf(den), expf(-(gF[j] + gM[j]))) + 1e-6f);
      }
    }
    __syncthreads();
    mlstm_f4 acc[RT][2];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
      for (int c = 0; c < 2; c++) acc[a][c] = mlstm_f4{0.f, 0.f, 0.f, 0.f};
    for (int d0 = 0; d0 < D; d0 += 64) {
      if (d0) fetch_s(d0);
      const int most = P - 20;             // a group past the last one reads the last again, against zeros
#pragma unroll
      for (int g = 0; g < 4; g++) {
        float qe[RT][4];
#pragma unroll
        for (int a = 0; a < RT; a++) {
          const float4 q = *(const float4*)(Qs + (16 * a + lr) * P + min(d0 + 16 * g, most) + 4 * kq);
          qe[a][0] = q.x, qe[a][1] = q.y, qe[a][2] = q.z, qe[a][3] = q.w;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int a = 0; a < RT; a++)
#pragma unroll
            for (int c = 0; c < 2; c++) acc[a][c] = mlstm_mfma(qe[a][i], sv[g][i][c], acc[a][c]);
      }
    }
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float g = expf(m_prev - gM[16 * a + 4 * kq + i]);
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c][i] *= g;
      }
#pragma unroll
    for (int g = 0; g < RT; g++) {
      float pe[RT][4];
#pragma unroll
      for (int a = g; a < RT; a++) {
        const float4 p = *(const float4*)(Ps + (16 * a + lr) * LP + 16 * g + 4 * kq);
        pe[a][0] = p.x, pe[a][1] = p.y, pe[a][2] = p.z, pe[a][3] = p.w;
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int a = g; a < RT; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) acc[a][c] = mlstm_mfma(pe[a][i], v[g][i][c], acc[a][c]);
    }
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int j = 16 * a + 4 * kq + i;
        if (j < Lc) {
          const float inv = gden[j];
          mlstm_put<PAIRS>(o_raw + ((size_t)(c0 + j) * H + hd) * E, e0, E, acc[a][0][i] * inv, acc[a][1][i] * inv);
        }
      }
  };
  MLSTM_TILES(L, Lc, run);
}

static size_t mlstm_local_lds(int L, int D) { return ((size_t)L * mlstm_pitch(D) + L) * 4; }
static size_t mlstm_output_lds(int L, int D) { return ((size_t)2 * L * mlstm_pitch(D) + (size_t)L * (L + 4) + mlstm_pitch(D) + 4 * L) * 4; }

static size_t mlstm_chunk_lds(int L, int D) {
  return ((size_t)D * MLSTM_EC + D + (size_t)2 * L * (D + 1) + (size_t)L * MLSTM_EC + (size_t)L * (L + 1) + 5 * L + 8) * 4;
}

template <int L>
static int mlstm_chunk_launch(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
                              float* state, int slot_words, int offset_words, const int* q_start,
                              const int* slot_of_req, float* o_raw, float* nm_new, int R, int H, int D, int E,
                              float cap, hipStream_t stream) {
  const size_t lds = mlstm_chunk_lds(L, D);
  static size_t raised = 0;
  if (lds > 48 * 1024 && lds > raised) {
    hipFuncSetAttribute((const void*)mlstm_chunk_kernel<L>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    raised = lds;
  }
  dim3 grid(R, H, (E + MLSTM_EC - 1) / MLSTM_EC);
  mlstm_chunk_kernel<L><<<grid, MLSTM_THREADS, lds, stream>>>((const act_t*)qkvz, ld, gates, bias_i, bias_f, state,
                                                              slot_words, offset_words, q_start, slot_of_req, o_raw,
                                                              nm_new, H, D, E, cap, 1.0f / sqrtf((float)D));
  return zk_launch_status("zk_mlstm_chunked");
}

extern "C" {

size_t zk_mlstm_state_bytes(int H, int D, int E) { return (size_t)H * ((size_t)D * E + D + 1) * 4; }

// qkvz: [T, ld] activations, a row holding q [H, D] | k [H, D] | v [H, E] | z [H, E];
// gates: float [T, 2H] (input gates, then forget gates, before bias and cap); out: [T, H * E].
static int mlstm_run(bool direct, const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
                     const float* norm_w, float* state, int slot_words, int offset_words, const int* q_start,
                     const int* slot_of_req, void* out, int R, int H, int D, int E, float cap, float eps, void* stream) {
  ZK_REQUIRE(R >= 0 && H > 0 && H <= 65535 && D > 0 && E > 0, "zk_mlstm: bad sizes");
  ZK_REQUIRE(E <= MLSTM_THREADS, "zk_mlstm: more than 256 value channels a head are not supported");
  ZK_REQUIRE(ld >= 2 * H * (D + E), "zk_mlstm: rows too short");
  ZK_REQUIRE(cap > 0.f, "zk_mlstm: the gates' cap must be positive");
  ZK_REQUIRE((size_t)slot_words * 4 >= (size_t)offset_words * 4 + zk_mlstm_state_bytes(H, D, E),
             "zk_mlstm: the state does not fit its slot");
  if (R == 0) return 0;
  // a head's S that does not fit the local memory stays in the state slot (the same bits, slower)
  if (!direct && ((size_t)D * E + 3 * D + E + MLSTM_THREADS + 32) * 4 > 150 * 1024) direct = true;
  const size_t lds = ((direct ? 0 : (size_t)D * E) + 3 * D + E + MLSTM_THREADS + 32) * 4;
  ZK_REQUIRE(lds <= 160 * 1024, "zk_mlstm: a head's state does not fit the local memory");
  if (lds > 48 * 1024) {
    static size_t raised = 0;
    if (lds > raised) {
      hipFuncSetAttribute((const void*)mlstm_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      raised = lds;
    }
  }
  dim3 grid(R, H);
  if (direct)
    mlstm_kernel<true><<<grid, MLSTM_THREADS, lds, (hipStream_t)stream>>>(
        (const act_t*)qkvz, ld, gates, bias_i, bias_f, norm_w, state, slot_words, offset_words, q_start, slot_of_req,
        (act_t*)out, H, D, E, cap, eps, 1.0f / sqrtf((float)D));
  else
    mlstm_kernel<false><<<grid, MLSTM_THREADS, lds, (hipStream_t)stream>>>(
        (const act_t*)qkvz, ld, gates, bias_i, bias_f, norm_w, state, slot_words, offset_words, q_start, slot_of_req,
        (act_t*)out, H, D, E, cap, eps, 1.0f / sqrtf((float)D));
  return zk_launch_status("zk_mlstm");
}

int zk_mlstm(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
             const float* norm_w, float* state, int slot_words, int offset_words, const int* q_start,
             const int* slot_of_req, void* out, int R, int H, int D, int E, float cap, float eps, void* stream) {
  return mlstm_run(false, qkvz, ld, gates, bias_i, bias_f, norm_w, state, slot_words, offset_words, q_start, slot_of_req,
                   out, R, H, D, E, cap, eps, stream);
}

// The same for steps in which every request brings one token: the state is renewed where it lies.
// (Right for any step, and bit for bit what zk_mlstm gives; only slower where requests bring more.)
int zk_mlstm_token(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
                   const float* norm_w, float* state, int slot_words, int offset_words, const int* q_start,
                   const int* slot_of_req, void* out, int R, int H, int D, int E, float cap, float eps, void* stream) {
  return mlstm_run(true, qkvz, ld, gates, bias_i, bias_f, norm_w, state, slot_words, offset_words, q_start, slot_of_req,
                   out, R, H, D, E, cap, eps, stream);
}

// The same as zk_mlstm for steps that bring portions: chunks of up to 64 tokens (fewer where
// max_q_len, the longest portion of the step, or the local memory asks for less).  o_raw: float
// [T, H * E] scratch; nm_new: float [R, H, D + 1] scratch.  zk_mlstm_finish must follow.
int zk_mlstm_chunked(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
                     float* state, int slot_words, int offset_words, const int* q_start, const int* slot_of_req,
                     float* o_raw, float* nm_new, int R, int H, int D, int E, float cap, int max_q_len, void* stream) {
  ZK_REQUIRE(R >= 0 && R <= 65535 && H > 0 && H <= 65535 && D > 0 && E > 0, "zk_mlstm_chunked: bad sizes");
  ZK_REQUIRE(D <= 256 && E <= 2048, "zk_mlstm_chunked: heads of more than 256 key channels are not supported");
  ZK_REQUIRE(ld >= 2 * H * (D + E), "zk_mlstm_chunked: rows too short");
  ZK_REQUIRE(cap > 0.f, "zk_mlstm_chunked: the gates' cap must be positive");
  ZK_REQUIRE((size_t)slot_words * 4 >= (size_t)offset_words * 4 + zk_mlstm_state_bytes(H, D, E),
             "zk_mlstm_chunked: the state does not fit its slot");
  if (R == 0) return 0;
  int L = max_q_len <= 16 ? 16 : max_q_len <= 32 ? 32 : 64;
  while (L > 16 && mlstm_chunk_lds(L, D) > 150 * 1024) L /= 2;
  hipStream_t s = (hipStream_t)stream;
#define ZK_CHUNK_(L_) \
  mlstm_chunk_launch<L_>(qkvz, ld, gates, bias_i, bias_f, state, slot_words, offset_words, q_start, slot_of_req, o_raw, \
                         nm_new, R, H, D, E, cap, s)
  return L == 64 ? ZK_CHUNK_(64) : L == 32 ? ZK_CHUNK_(32) : ZK_CHUNK_(16);
#undef ZK_CHUNK_
}

}  // extern "C"

// Tokens a chunk: few enough that the output kernel's block leaves a quarter of the local memory (us, three launches; chunks of 64 and of
// 32: one request of 600, four heads of 40 value channels, 256 key channels 63.9 and 52.2, 224 60.0 and 49.6, 192 51.9 and
// 43.1; eight heads of 256 value channels 75.6 and 73.2, 70.0 and 68.1, 61.5 and 59.5; 2,048 tokens, four heads of 256, 93.4 and
// 97.2, 85.7 and 91.8, 74.4 and 81.3).
static int mlstm_scan_len(int max_q_len, int D) {
  int L = max_q_len <= 16 ? 16 : max_q_len <= 32 ? 32 : 64;
  while (L > 16 && mlstm_output_lds(L, D) > 120 * 1024) L /= 2;
  return L;
}

// Floats of scratch that zk_mlstm_scan needs for a step of T tokens in R requests.
extern "C" size_t zk_mlstm_scan_floats(int T, int R, int H, int D, int E, int max_q_len) {
  const int L = mlstm_scan_len(max_q_len, D);
  const size_t chunks = (size_t)(T + L - 1) / L + R;
  return chunks * H * ((size_t)D * E + D + 3);
}

template <int L, bool PAIRS>
static int mlstm_scan_launch(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f,
                             float* state, int slot_words, int offset_words, const int* q_start, const int* slot_of_req,
                             float* o_raw, float* work, int chunks, int R, int H, int D, int E, float cap, hipStream_t s) {
  float* Uw = work;
  float* uw = Uw + (size_t)chunks * H * D * E;
  float* af = uw + (size_t)chunks * H * D;
  float* mprev = af + (size_t)chunks * H * 2;
  const int zs = (E + MLSTM_EB - 1) / MLSTM_EB;
  const size_t lds_local = mlstm_local_lds(L, D), lds_out = mlstm_output_lds(L, D);
  static size_t raised_local = 0, raised_out = 0;
  if (lds_local > 48 * 1024 && lds_local > raised_local) {
    hipFuncSetAttribute((const void*)mlstm_local_kernel<L, PAIRS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_local);
    raised_local = lds_local;
  }
  if (lds_out > 48 * 1024 && lds_out > raised_out) {
    hipFuncSetAttribute((const void*)mlstm_output_kernel<L, PAIRS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_out);
    raised_out = lds_out;
  }
  mlstm_local_kernel<L, PAIRS><<<dim3(chunks, H, zs), MLSTM_THREADS, lds_local, s>>>(
      (const act_t*)qkvz, ld, gates, bias_i, bias_f, q_start, Uw, uw, af, R, H, D, E, cap);
  if (int rc = zk_launch_status("zk_mlstm_scan (local)")) return rc;
  mlstm_scan_kernel<<<dim3(R, H, (D * E + D + MLSTM_THREADS * MLSTM_ELEMS) / (MLSTM_THREADS * MLSTM_ELEMS)), MLSTM_THREADS, 0, s>>>(
      state, slot_words, offset_words, q_start, slot_of_req, Uw, uw, af, mprev, L, H, D, E);
  if (int rc = zk_launch_status("zk_mlstm_scan (scan)")) return rc;
  mlstm_output_kernel<L, PAIRS><<<dim3(chunks, H, zs), MLSTM_THREADS, lds_out, s>>>(
      (const act_t*)qkvz, ld, gates, bias_i, bias_f, q_start, Uw, uw, mprev, o_raw, state, slot_words, offset_words, slot_of_req, R, H,
      D, E, cap, 1.0f / sqrtf((float)D));
  return zk_launch_status("zk_mlstm_scan (output)");
}

extern "C" {

// zk_mlstm_chunked's work with the chunks of a step side by side (three launches); for steps
// whose portions are several chunks long.  work: zk_mlstm_scan_floats(...) floats of scratch.
// zk_mlstm_finish (with nm_new null: n is stored by the scan, m by the output kernel) must follow.
int zk_mlstm_scan(const void* qkvz, int ld, const float* gates, const float* bias_i, const float* bias_f, float* state,
                  int slot_words, int offset_words, const int* q_start, const int* slot_of_req, float* o_raw, float* work,
                  size_t work_floats, int T, int R, int H, int D, int E, float cap, int max_q_len, void* stream) {
  ZK_REQUIRE(T >= 0 && R >= 0 && R <= 65535 && H > 0 && H <= 65535 && D > 0 && E > 0, "zk_mlstm_scan: bad sizes");
  ZK_REQUIRE(D <= 256 && E <= 2048, "zk_mlstm_scan: heads of more than 256 key channels are not supported");
  ZK_REQUIRE(ld >= 2 * H * (D + E), "zk_mlstm_scan: rows too short");
  ZK_REQUIRE(cap > 0.f, "zk_mlstm_scan: the gates' cap must be positive");
  ZK_REQUIRE((size_t)slot_words * 4 >= (size_t)offset_words * 4 + zk_mlstm_state_bytes(H, D, E),
             "zk_mlstm_scan: the state does not fit its slot");
  ZK_REQUIRE(work != nullptr && work_floats >= zk_mlstm_scan_floats(T, R, H, D, E, max_q_len), "zk_mlstm_scan: too little scratch");
  if (R == 0 || T == 0) return 0;
  const int L = mlstm_scan_len(max_q_len, D);
  const int chunks = (T + L - 1) / L + R;
  hipStream_t s = (hipStream_t)stream;
  // two value channels an access, where every row of them begins on a pair
  const bool pairs = E % 2 == 0 && ld % 2 == 0 && (uintptr_t)qkvz % (2 * sizeof(act_t)) == 0 && (uintptr_t)work % 8 == 0 &&
                     (uintptr_t)o_raw % 8 == 0;
#define ZK_SCAN_(L_)                                                                                                          \
  (pairs ? mlstm_scan_launch<L_, true>(qkvz, ld, gates, bias_i, bias_f, state, slot_words, offset_words, q_start, slot_of_req, \
                                       o_raw, work, chunks, R, H, D, E, cap, s)                                               \
         : mlstm_scan_launch<L_, false>(qkvz, ld, gates, bias_i, bias_f, state, slot_words, offset_words, q_start, slot_of_req, \
                                        o_raw, work, chunks, R, H, D, E, cap, s))
  return L == 64 ? ZK_SCAN_(64) : L == 32 ? ZK_SCAN_(32) : ZK_SCAN_(16);
#undef ZK_SCAN_
}

int zk_mlstm_finish(const float* o_raw, const void* qkvz, int ld, const float* norm_w, const float* nm_new,
                    float* state, int slot_words, int offset_words, const int* req_of_token, const int* q_start,
                    const int* slot_of_req, void* out, int T, int H, int D, int E, float eps, void* stream) {
  ZK_REQUIRE(T >= 0 && H > 0 && H <= 65535 && D > 0 && E > 0, "zk_mlstm_finish: bad sizes");
  if (T == 0) return 0;
  dim3 grid(T, H);
  mlstm_finish_kernel<<<grid, 64, 0, (hipStream_t)stream>>>(o_raw, (const act_t*)qkvz, ld, norm_w, nm_new, state,
                                                            slot_words, offset_words, req_of_token, q_start, slot_of_req,
                                                            (act_t*)out, H, D, E, eps);
  return zk_launch_status("zk_mlstm_finish");
}

}  // extern "C"

ZK_ENTER(zk_mlstm)
ZK_ENTER(zk_mlstm_token)
ZK_ENTER(zk_mlstm_chunked)
ZK_ENTER(zk_mlstm_scan)
ZK_ENTER(zk_mlstm_finish)
