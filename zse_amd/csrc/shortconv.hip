// The short causal convolution over time, channel by channel:
//
//   u = x + in_bias;   y_t = bias + sum_j w[:, j] u_(t - taps + 1 + j);   (+ u_t);   (silu)
//
// rows before a sequence's start being zero (not in_bias).  The taps - 1 rows of u before a
// request's next token are float rows in its state slot, the youngest first; a step reads them for its
// first tokens and renews them.
//
// A thread owns V neighbouring channels (16 bytes of bfloat16) of a run of ``span`` tokens of one
// request and carries the taps - 1 rows before the current token in registers, so a row is read
// once a run.  Runs are counted from the request's first token of the step: only the first of
// them reads the state (span >= taps - 1), and its threads renew it, each its own columns, after
// they have read them.  One launch serves every kind of step.
//
// A block works on one run.  As a rule block (y, z) is run y of request z; where more than half of many such blocks would
// find no run, the runs are numbered through all requests and a block looks for its own (us, the one way and the other: 700
// rows and 8 single ones of 2,048 channels 10.2 and 9.0, 2,000 and 500 single ones of 256 55.8 and 10.0; 2,048 rows of 2,048
// 10.2 and 10.5, 1,000 requests of nine rows of 256 16.7 and 21.4).
//
// Up to 2 million values (3 of 16 bits) the time is the launch and a chain of waits, so a run's rows are all asked for before the
// first is used (us, one after the other and so, taps of 4: 8 rows of 2,048 channels 5.4 and 4.6, 700 and 8 single ones 6.5 and
// 5.6, 60 requests of 20 rows of 1,024 6.3 and 5.6; in 16 bits 700 and 8 of 4,096 6.9 and 6.3); with more values, or of rows that
// are nearly alone, one after the other (2,048 rows of 2,048 in 32 bits 9.3 and 10.1, 200 single rows of 8,192 12.6 and 15.4).
#include "common.h"
#include "packed_call.h"

extern "C" int zk_steplist_register(const char* name, int nargs, void* fn);
#define ZK_ENTER(fn) \
  static const int fn##_entered = zk_steplist_register(#fn, zk_packed::Call<fn>::nargs, (void*)zk_packed::Call<fn>::call);

#define CONV_SPAN 8
#define CONV_MOST_TAPS (CONV_SPAN + 1)

// V channels of a row as they lie in memory, and their values
template <int V>
struct ConvRaw {
  act_t v[V] __attribute__((aligned(sizeof(act_t) * V > 16 ? 16 : sizeof(act_t) * V)));
};
template <int V>
__device__ __forceinline__ ConvRaw<V> conv_raw(const act_t* p) {
  return *(const ConvRaw<V>*)p;
}
template <int V>
__device__ __forceinline__ void conv_values(const ConvRaw<V>& r, float (&v)[V]) {
#pragma unroll
  for (int e = 0; e < V; e++) v[e] = to_f32(r.v[e]);
}
template <int V>
__device__ __forceinline__ void conv_get(const act_t* p, float (&v)[V]) {
  conv_values<V>(conv_raw<V>(p), v);
}
template <int V>
__device__ __forceinline__ void conv_put(act_t* p, const float (&v)[V]) {
  if constexpr (V == 8) {
#if ZSE_ACT_BF16
    typedef __bf16 b8 __attribute__((ext_vector_type(8)));
    b8 q;
#pragma unroll
    for (int e = 0; e < 8; e++) q[e] = (__bf16)v[e];
    *(b8*)p = q;
#else
    *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
#endif
  } else {
    p[0] = from_f32<act_t>(v[0]);
  }
}
template <int V>
__device__ __forceinline__ void conv_get_state(const float* p, float (&v)[V]) {
  if constexpr (V == 8) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
    v[0] = p[0];
  }
}
template <int V>
__device__ __forceinline__ void conv_put_state(float* p, const float (&v)[V]) {
  if constexpr (V == 8) {
    *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
  } else {
    p[0] = v[0];
  }
}

// TAPS: the number of taps where the launch knows it at compile time, 0: ``taps`` (up to 9).  PIECES: runs are numbered through all
// requests, ``columns`` blocks next to each other for each.  AHEAD: a run's rows are all asked for before the first is used
template <int V, int TAPS, bool PIECES, bool AHEAD>
__global__ __launch_bounds__(256) void conv_rows_kernel(const act_t* __restrict__ x, int ld_in,
                                                        const float* __restrict__ in_bias, const float* __restrict__ w,
                                                        const float* __restrict__ bias, float* __restrict__ state,
                                                        int slot_words, int offset_words, const int* __restrict__ q_start,
                                                        const int* __restrict__ slot_of_req, act_t* __restrict__ out,
                                                        int ld_out, int T, int R, int C, int taps_given, int residual,
                                                        int act, int columns) {
  constexpr int MOST = TAPS ? TAPS : CONV_MOST_TAPS, BACK = MOST > 1 ? MOST - 1 : 1;
  const int taps = TAPS ? TAPS : taps_given;
  const int c = ((PIECES ? blockIdx.x % columns : blockIdx.x) * blockDim.x + threadIdx.x) * V;
  auto padding = [&](int from) {         // rows behind the last request: padding of a captured step
    float zero[V];
#pragma unroll
    for (int e = 0; e < V; e++) zero[e] = 0.f;
    for (int t = from; t < T; t++) conv_put<V>(out + (size_t)t * ld_out + c, zero);
  };
  int r, t0, n, first;
  if constexpr (PIECES) {
    Piece run;
    const bool found = find_piece(q_start, R, CONV_SPAN, blockIdx.x / columns, run);      // (all lanes of a wave call it)
    if (c >= C) return;
    if (!found) {
      if (blockIdx.x + columns >= gridDim.x) padding(q_start[R]);
      return;
    }
    r = run.r, t0 = run.t0, n = run.n, first = run.first;
  } else {
    if (c >= C) return;
    r = blockIdx.z, first = blockIdx.y * CONV_SPAN;
    t0 = q_start[r];
    if (r == R) {
      if (first == 0) padding(t0);
      return;
    }
    n = q_start[r + 1] - t0;
    if (first >= n) return;
  }
  const int last = min(n, first + CONV_SPAN);
  float ib[V], b0[V], wt[MOST][V];
#pragma unroll
  for (int e = 0; e < V; e++) {
    ib[e] = in_bias ? in_bias[c + e] : 0.f;
    b0[e] = bias ? bias[c + e] : 0.f;
#pragma unroll
    for (int j = 0; j < MOST; j++) wt[j][e] = j < taps ? w[(size_t)(c + e) * taps + j] : 0.f;
  }
  auto input = [&](int i, float (&v)[V]) {
    conv_get<V>(x + (size_t)(t0 + i) * ld_in + c, v);
#pragma unroll
    for (int e = 0; e < V; e++) v[e] += ib[e];
  };
  ConvRaw<V> rows[AHEAD ? CONV_SPAN : 1];      // (a row past the last: the last again)
  if constexpr (AHEAD) {
#pragma unroll
    for (int i = 0; i < CONV_SPAN; i++) rows[i] = conv_raw<V>(x + (size_t)(t0 + min(first + i, last - 1)) * ld_in + c);
  }
  float* st = taps > 1 ? state + (size_t)slot_of_req[r] * slot_words + offset_words + c : nullptr;
  // back[b]: the row b + 1 places before the current token
  float back[BACK][V];
#pragma unroll
  for (int b = 0; b < BACK; b++)
    if (b < taps - 1) {
      if (first - 1 - b >= 0) input(first - 1 - b, back[b]);
      else conv_get_state<V>(st + (size_t)(b - first) * C, back[b]);      // only in the first run
    }
  if (first == 0 && taps > 1) {
    // the state the next step finds: row a is the row a + 1 places before it, one of this step's
    // rows or one of those just read
#pragma unroll
    for (int a = 0; a < BACK; a++)
      if (a < taps - 1) {
        float v[V];
        if (n - 1 - a >= 0) {
          input(n - 1 - a, v);
        } else {
#pragma unroll
          for (int e = 0; e < V; e++) v[e] = 0.f;
#pragma unroll
          for (int b = 0; b < BACK; b++)
            if (b == a - n) {
#pragma unroll
              for (int e = 0; e < V; e++) v[e] = back[b][e];
            }
        }
        conv_put_state<V>(st + (size_t)a * C, v);
      }
  }
  constexpr int TURN = AHEAD ? CONV_SPAN : 1;
  for (int turn = first; turn < last; turn += TURN) {
#pragma unroll
    for (int k = 0; k < TURN; k++) {
      const int i = turn + k;
      if (i >= last) break;
      float cur[V];
      if constexpr (AHEAD) {
        conv_values<V>(rows[k], cur);
#pragma unroll
        for (int e = 0; e < V; e++) cur[e] += ib[e];
      } else {
        input(i, cur);
      }
      float acc[V];
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] = b0[e];
#pragma unroll
      for (int b = BACK - 1; b >= 0; b--)
        if (b < taps - 1) {
#pragma unroll
          for (int e = 0; e < V; e++) {
            float wj = 0.f;
            if (TAPS) {
              wj = wt[MOST - 2 - b < 0 ? 0 : MOST - 2 - b][e];
            } else {
#pragma unroll
              for (int j = 0; j < MOST; j++) wj = j == taps - 2 - b ? wt[j][e] : wj;
            }
            acc[e] = fmaf(wj, back[b][e], acc[e]);
          }
        }
#pragma unroll
      for (int e = 0; e < V; e++) {
        float wj = wt[0][e];
#pragma unroll
        for (int j = 0; j < MOST; j++) wj = j == taps - 1 ? wt[j][e] : wj;
        acc[e] = fmaf(wj, cur[e], acc[e]);
        if (residual) acc[e] = cur[e] + acc[e];
        if (act == 1) acc[e] = acc[e] / (1.0f + expf(-acc[e]));      // silu
      }
      conv_put<V>(out + (size_t)(t0 + i) * ld_out + c, acc);
#pragma unroll
      for (int b = BACK - 1; b > 0; b--)
#pragma unroll
        for (int e = 0; e < V; e++) back[b][e] = back[b - 1][e];
#pragma unroll
      for (int e = 0; e < V; e++) back[0][e] = cur[e];
    }
  }
}

// How a step's runs are laid out: ``columns`` blocks of ``threads`` for each of ``runs`` runs, of every request or of them all.
struct ConvGrid {
  int threads, columns, runs, by_piece;
};
static ConvGrid conv_grid(int T, int R, int max_q_len, int holders) {      // holders: threads that hold a row between them
  // few runs: narrow blocks, so that they spread over the compute units
  auto threads_of = [&](long long runs) { return (holders + 255) / 256 * runs >= 512 ? 256 : 64; };
  const int most = max_q_len > 0 ? (max_q_len + CONV_SPAN - 1) / CONV_SPAN : 1;
  ConvGrid g{threads_of((long long)most * R), 0, most, 0};
  g.columns = (holders + g.threads - 1) / g.threads;
  // The step's runs, at most (full ones and every request's last), and one for the padding behind the last request.  Finding
  // a run costs 0.2 us, and 0.2 more for every 64 requests: few blocks, or blocks that mostly have a run, do not bring that
  // back.  Over 397 uneven steps this choice takes 0.95 of the time of a block a run and request throughout.
  const long long runs = (long long)T / CONV_SPAN + R + 1, blocks = (long long)most * (R + 1);
  if (most > 1 && g.columns * blocks >= 700 && 2 * runs < blocks && g.columns * runs < 1 << 22) {
    g.threads = threads_of(runs);
    g.columns = (holders + g.threads - 1) / g.threads;
    g.runs = (int)runs;
    g.by_piece = 1;
  }
  return g;
}

extern "C" {

// 1 if a step's runs are numbered through all its requests (``per``: channels a thread holds, 8 or 1).  For tests that mean
// to reach both ways.
int zk_conv_rows_by_piece(int T, int R, int max_q_len, int C, int per) {
  return conv_grid(T, R, max_q_len, (C + per - 1) / per).by_piece;
}

// The most taps zk_conv_rows takes.
int zk_conv_rows_most_taps() { return CONV_MOST_TAPS; }

// x: [T, ld_in] activations, out: [T, ld_out] (another buffer), of which the first C channels take
// part; w: float [C, taps]; in_bias, bias (either may be null): float [C]; the state of request r is
// taps - 1 float rows of C at state[slot_of_req[r] * slot_words + offset_words], renewed by this
// launch.  Requests are rows [q_start[r], q_start[r + 1]) of the step, q_start has R + 1 entries;
// rows behind q_start[R] are padding and come out as 0.  max_q_len: no request brings more tokens
// than this.  residual: the input (with in_bias) is added to the sum; act: 0 none, 1 silu.
int zk_conv_rows(const void* x, int ld_in, const float* in_bias, const float* w, const float* bias, float* state, int slot_words,
                 int offset_words, const int* q_start, const int* slot_of_req, void* out, int ld_out, int T, int R,
                 int max_q_len, int C, int taps, int residual, int act, void* stream) {
  ZK_REQUIRE(T >= 0 && R >= 0 && R < 65535 && C > 0 && taps >= 1 && max_q_len >= 0, "zk_conv_rows: bad sizes");
  ZK_REQUIRE(taps <= CONV_MOST_TAPS, "zk_conv_rows: too many taps");
  ZK_REQUIRE(ld_in >= C && ld_out >= C && (act == 0 || act == 1), "zk_conv_rows: bad strides or activation");
  ZK_REQUIRE(x != out, "zk_conv_rows: not in place");
  ZK_REQUIRE(taps == 1 || (state != nullptr && (long long)slot_words >= (long long)offset_words + (long long)(taps - 1) * C),
             "zk_conv_rows: the state does not fit its slot");
  if (T == 0) return 0;
  auto aligned = [](const void* p, size_t n) { return (uintptr_t)p % n == 0; };
  const bool vec = C % 8 == 0 && ld_in % 8 == 0 && ld_out % 8 == 0 && aligned(x, 16) && aligned(out, 16) &&
                   (taps == 1 || (aligned(state, 16) && slot_words % 4 == 0 && offset_words % 4 == 0));
  ZK_REQUIRE(max_q_len <= 65535 * CONV_SPAN, "zk_conv_rows: too many tokens");
  const int per = vec ? 8 : 1;
  const ConvGrid g = conv_grid(T, R, max_q_len, (C + per - 1) / per);
  const dim3 grid = g.by_piece ? dim3((unsigned)(g.columns * g.runs)) : dim3(g.columns, g.runs, R + 1);
  const bool ahead = max_q_len >= 4 && (long long)T * C <= (ZSE_ACT_BF16 ? 3 << 20 : 2 << 20);      // (see the top)
#define LAUNCH_(V, N, PIECES, AHEAD)                                                                                  \
  conv_rows_kernel<V, N, PIECES, AHEAD><<<grid, g.threads, 0, (hipStream_t)stream>>>(                                 \
      (const act_t*)x, ld_in, in_bias, w, bias, state, slot_words, offset_words, q_start, slot_of_req, (act_t*)out, ld_out, T, R, C, \
      taps, residual, act, g.columns)
#define LAUNCH(V, N, AHEAD)                              \
  do {                                                   \
    if (g.by_piece) LAUNCH_(V, N, true, AHEAD);          \
    else LAUNCH_(V, N, false, AHEAD);                    \
  } while (0)
#define LAUNCH_AHEAD(N) do { if (ahead) LAUNCH(8, N, true); else LAUNCH(8, N, false); } while (0)
  if (vec) {
    if (taps == 2) LAUNCH_AHEAD(2);
    else if (taps == 3) LAUNCH_AHEAD(3);
    else if (taps == 4) LAUNCH_AHEAD(4);
    else LAUNCH(8, 0, false);
  } else {
    LAUNCH(1, 0, false);
  }
#undef LAUNCH_AHEAD
#undef LAUNCH
#undef LAUNCH_
  return zk_launch_status("zk_conv_rows");
}

}  // extern "C"

ZK_ENTER(zk_conv_rows)
