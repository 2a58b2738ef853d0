// Linear recurrences per head whose state is a matrix and whose decay is a vector per token: gated linear attention, and
// (compiled with TIME_MIX) time mixing with a bonus for the current token.
//
// For a request's tokens t = 0, 1, ..., per head, with keys and queries of d channels and values of dv:
//   alpha_t[i] = sigmoid(z_t[i] + b[i]) ^ (1 / tau) = exp(-softplus(-(z_t[i] + b[i])) / tau)
//   S_t[i, j]  = alpha_t[i] S_(t-1)[i, j] + k_t[i] v_t[j],        S_(-1) = 0
//   o_t[j]     = sum_i S_t[i, j] q_t[i] * q_scale
//   y_t[j]     = o_t[j] / sqrt(mean_j o_t[j]^2 + eps) * w[j] * silu(g_t[j])
//
// Time mixing (keys, queries r and values of d):
//   w_t[i]     = exp(-exp(z_t[i] + b[i]))
//   o_t[j]     = sum_i (S_(t-1)[i, j] + u[i] k_t[i] v_t[j]) r_t[i]          (the read-out sees the token's own write only through u)
//   S_t[i, j]  = w_t[i] S_(t-1)[i, j] + k_t[i] v_t[j]
//   y_t[j]     = o_t[j] / sqrt(mean_j o_t[j]^2 + eps) * w_norm[head, j] * silu(g_t[j])
// The bonus' part of o_t is v_t[j] times one number per token, sum_i u[i] k_t[i] r_t[i], which a wave per token forms.
//
// Rows are a step's flattened rows (requests end to end, a request's rows in position order).  q, k, v and g are columns
// of projected rows (ld apart); z is float (the decay's second product, without its bias).
// Decays, their logarithms, S, o, the norm and the gate are float whatever the activation type.
//
// A request's S lives in its state slot, one float32 row per slot laid out [head][j][PARTS * DP]: a column j of S as
// PARTS runs of DP channels (channels at or beyond d are zero and stay zero).  A thread owns one run of one column (of two
// neighbouring columns where DP <= 32): DP (2 DP) numbers of S in registers; the PARTS threads of a column are neighbours in a wave and add their parts of o_t[j] by shuffles in a fixed
// order.  A workgroup is one head of one request (or of one chunk): dv * PARTS threads.  Tokens are taken STAGE at a time:
// the threads put q, k and alpha of the stage's tokens into LDS, a (token, channel) each (and form alpha on the way), everybody walks the
// stage's tokens, o goes to LDS, and a wave per token norms and gates it.
//
// MODE 0: a request's rows in one walk, from its slot and back into it (steps of single tokens: gla_step_kernel).
// Long portions are cut into chunks that run side by side (the recurrence is linear in S):
// MODE 1: a chunk from S = 0; records its final S and the sum of its log alpha per channel.
// gla_combine: walks a request's chunks: chunk c's record becomes the state chunk c starts from,
//              S <- exp(sum log alpha) S + S_c; the request's new state goes into its slot.
// MODE 2: a chunk from the state it starts from; writes y.
#include "common.h"
#include "tile_acts.h"
#include "lane_sums.h"

IFX_DEFINE_LAST_ERROR()

#ifndef TIME_MIX
#define TIME_MIX 0
#endif

#define STAGE 8

struct GlaArgs {
  const void* q; const void* k; const void* v; const void* g;      // the head-0 columns of row 0; rows ld elements apart
  int ld;
  const float* z;          // [T, H * d], or null (steps of single tokens):
  const bf16_t* low;       // ... z_t = w2 low_t with low [T, rank] (rows low_ld apart) and w2 [H * d, rank]
  const bf16_t* w2;
  int low_ld, rank;
  const float* z_bias;     // [H * d] or null
  float inv_tau, q_scale, eps;
  const void* norm_w;      // [dv], or with TIME_MIX [H * dv]
  int norm_dtype;
  const float* bonus;      // TIME_MIX: u [H * d]
  float* state;            // [slots, state_stride]; S at state_offset of a row
  size_t state_stride, state_offset;
  const int* q_start;      // [R]
  const int* q_len;        // [R]
  const int* slots;        // [R]
  void* out;               // [T, H * dv] of the activation type
  int H, d, dv, parts;
  // chunks (MODE 1, 2)
  const int* chunk_req;    // [n_chunks]
  const int* chunk_t0;     // [n_chunks] first row
  const int* chunk_len;    // [n_chunks]
  float* chunk_state;      // [n_chunks, H * dv * parts * DP]
  float* chunk_loga;       // [n_chunks, H * d]
};

__device__ __forceinline__ float log_sigmoid(float x) {      // -softplus(-x), without overflow
  return x >= 0.f ? -log1pf(expf(-x)) : x - log1pf(expf(x));
}

// (a thread's registers hold DP numbers of S: the more of them, the fewer threads a workgroup may have)
#define GLA_MAX_THREADS(DP) ((DP) <= 32 ? 1024 : ((DP) <= 64 ? 512 : 256))

// WHOLE: the parts' channels are all of a head's (parts * DP = d), so nothing is asked of a channel before it is read, and what a thread
// reads of a token from LDS goes in pieces of 16 bytes (4,000 rows of 16 heads of 64 x 128 in chunks: 151 and 222 us -> 98 and 195 for the two
// walks, a third of it the values, which lay in 32 registers; time mixing of 64 requests' prompts 148 -> 93).  With up to 512 threads: it wants 140
// registers, and with 128 of them (1,024 threads) steps of single tokens take 12.4 us for 10.8.
template <typename T, typename TO, int DP, int MODE, int COLS, bool WHOLE>
__global__ __launch_bounds__(WHOLE ? 512 : GLA_MAX_THREADS(DP)) void gla_kernel(GlaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int d = a.d, dv = a.dv, parts = a.parts, H = a.H;
  float* lq = lds;                       // [STAGE][d]
  float* lk = lq + STAGE * d;            // [STAGE][d]
  float* la = lk + STAGE * d;            // [STAGE][d]
  float* lo = la + STAGE * d;            // [STAGE][dv]
  float* lg = lo + STAGE * dv;           // [STAGE][d]: the decays' logarithms (MODE 1 sums them per channel)
  __shared__ float lb[STAGE];            // TIME_MIX: sum_i u[i] k[i] q[i] of a token
  const int unit = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
  int t0, n;
  size_t s_at;                            // where this head's S lies
  float* sbase;
  if (MODE == 0) {
    t0 = a.q_start[unit]; n = a.q_len[unit];
    sbase = a.state + (size_t)a.slots[unit] * a.state_stride + a.state_offset;
  } else {
    t0 = a.chunk_t0[unit]; n = a.chunk_len[unit];
    sbase = a.chunk_state + (size_t)unit * H * dv * parts * DP;
  }
  if (n <= 0) return;
  s_at = (size_t)head * dv * parts * DP;
  // a thread owns COLS neighbouring columns j0 .. j0 + COLS - 1 of S for its run of DP channels: what it reads of a token's
  // q, k and decays from LDS serves COLS columns
  const int j0 = (tid / parts) * COLS, p = tid % parts;
  float S[COLS][DP];
  float* sp = sbase + s_at + ((size_t)j0 * parts + p) * DP;          // (column j0 + c lies c * parts * DP further)
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    if (MODE != 1 && j0 + c < dv) {
#pragma unroll
      for (int i = 0; i < DP; i += 4) {
        const float4 v = *(const float4*)(sp + (size_t)c * parts * DP + i);
        S[c][i] = v.x; S[c][i + 1] = v.y; S[c][i + 2] = v.z; S[c][i + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < DP; ++i) S[c][i] = 0.f;
    }
  }
  const T* rq = (const T*)a.q; const T* rk = (const T*)a.k; const T* rv = (const T*)a.v; const T* rg = (const T*)a.g;
  const int wid = tid / WAVE, lane = tid % WAVE, nw = (blockDim.x + WAVE - 1) / WAVE;
  float loga_sum = 0.f;
  auto put_back = [&]() {
#pragma unroll
    for (int c = 0; c < COLS; ++c)
      if (j0 + c < dv) {
#pragma unroll
        for (int i = 0; i < DP; i += 4)
          *(float4*)(sp + (size_t)c * parts * DP + i) = make_float4(S[c][i], S[c][i + 1], S[c][i + 2], S[c][i + 3]);
      }
  };
  for (int s0 = 0; s0 < n; s0 += STAGE) {
    const int ns = min(STAGE, n - s0);
    // the stage's q, k and decays: one (token, channel) a thread and trip, neighbouring threads on neighbouring channels
    for (int it = tid; it < ns * d; it += blockDim.x) {
      const int tt = it / d, ch = it - tt * d;
      const size_t t = (size_t)(t0 + s0 + tt);
      const float zq = a.z[t * (size_t)(H * d) + head * d + ch] + (a.z_bias ? a.z_bias[head * d + ch] : 0.f);
      const float kq = to_f(rk[t * a.ld + head * d + ch]);
      const float qq = MODE == 1 ? 0.f : to_f(rq[t * a.ld + head * d + ch]);
      const float la_t = TIME_MIX ? -expf(zq) : log_sigmoid(zq) * a.inv_tau;
      if (MODE == 1) lg[it] = la_t;
      la[it] = expf(la_t);
      lk[it] = kq;
      lq[it] = qq * a.q_scale;
    }
    // (a wave's first token's gate and norm weights, up to two of each a lane, come with the stage's own loads)
    float g_early[2], w_early[2];
    if (MODE != 1) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int e = lane + c * WAVE;
        const bool in = wid < ns && e < dv;
        g_early[c] = in ? to_f(rg[(size_t)(t0 + s0 + wid) * a.ld + head * dv + e]) : 0.f;
        w_early[c] = in ? load_dyn(a.norm_w, a.norm_dtype, TIME_MIX ? head * dv + e : e) : 0.f;
      }
    }
    // the values lie where the outputs will: a column's value is read by the lanes that form its output before one of them writes it
    for (int it = tid; it < ns * dv; it += blockDim.x) {
      const int tt = it / dv, c = it - tt * dv;
      lo[it] = to_f(rv[(size_t)(t0 + s0 + tt) * a.ld + head * dv + c]);
    }
    __syncthreads();
    if (MODE == 1 && tid < d)
      for (int tt = 0; tt < ns; ++tt) loga_sum += lg[tt * d + tid];
    if (TIME_MIX && MODE != 1) {
      for (int tt = wid; tt < ns; tt += nw) {
        float b = 0.f;
        for (int c = lane; c < d; c += WAVE) b = fmaf(a.bonus[head * d + c] * lk[tt * d + c], lq[tt * d + c], b);
        b = wave_sum(b);
        if (lane == 0) lb[tt] = b;
      }
      __syncthreads();
    }
#pragma unroll 1
    for (int tt = 0; tt < ns; ++tt) {
      const float* aa = la + tt * d + p * DP;
      const float* kk = lk + tt * d + p * DP;
      const float* qv = lq + tt * d + p * DP;
      float acc[COLS], vt[COLS];
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        acc[c] = 0.f;
        vt[c] = j0 + c < dv ? lo[tt * dv + j0 + c] : 0.f;
      }
      auto channel = [&](int i, float al, float kv, float qq) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          if (TIME_MIX && MODE != 1) acc[c] = fmaf(S[c][i], qq, acc[c]);        // (the read-out comes before the write)
          S[c][i] = fmaf(al, S[c][i], kv * vt[c]);
          if (!TIME_MIX && MODE != 1) acc[c] = fmaf(S[c][i], qq, acc[c]);
        }
      };
      if constexpr (WHOLE) {
#pragma unroll
        for (int i = 0; i < DP; i += 4) {
          const float4 al = *(const float4*)(aa + i), kv = *(const float4*)(kk + i), qq = MODE != 1 ? *(const float4*)(qv + i) : float4{0.f, 0.f, 0.f, 0.f};
          channel(i, al.x, kv.x, qq.x);
          channel(i + 1, al.y, kv.y, qq.y);
          channel(i + 2, al.z, kv.z, qq.z);
          channel(i + 3, al.w, kv.w, qq.w);
        }
      } else {
#pragma unroll
        for (int i = 0; i < DP; ++i)
          if (p * DP + i < d) channel(i, aa[i], kk[i], MODE != 1 ? qv[i] : 0.f);              // (uniform over the lanes that share p)
      }
      if (MODE != 1) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          float r = acc[c];
          for (int o = 1; o < parts; o <<= 1) r += __shfl_xor(r, o, WAVE);
          if (TIME_MIX) r = fmaf(lb[tt], vt[c], r);
          if (j0 + c < dv && p == 0) lo[tt * dv + j0 + c] = r;
        }
      }
    }
    if (MODE == 0 && s0 + STAGE >= n) put_back();          // (on its way while the outputs are formed)
    __syncthreads();
    if (MODE != 1) {
      // a wave per token: the head's norm over dv, its weight, the gate
      for (int tt = wid; tt < ns; tt += nw) {
        const size_t t = (size_t)(t0 + s0 + tt);
        float ss = 0.f;
        for (int c = lane; c < dv; c += WAVE) ss = fmaf(lo[tt * dv + c], lo[tt * dv + c], ss);
        const float inv = rsqrtf(wave_sum(ss) / (float)dv + a.eps);
        int u = 0;
        for (int c = lane; c < dv; c += WAVE, ++u) {
          const bool early = tt == wid && u < 2;
          const float g = early ? (u == 0 ? g_early[0] : g_early[1]) : to_f(rg[t * a.ld + head * dv + c]);
          const float w = early ? (u == 0 ? w_early[0] : w_early[1]) : load_dyn(a.norm_w, a.norm_dtype, TIME_MIX ? head * dv + c : c);
          ((TO*)a.out)[t * (size_t)(H * dv) + head * dv + c] = from_f<TO>(lo[tt * dv + c] * inv * w * act_silu(g));
        }
      }
    }
    __syncthreads();                       // (the next stage's loads overwrite what this stage read)
  }
  if (MODE == 1) put_back();
  if (MODE == 1 && tid < d) a.chunk_loga[(size_t)unit * H * d + head * d + tid] = loga_sum;
}

// Steps of single tokens (a request's tokens one after the other where it has more): a workgroup takes a head of a request.  Bound by S, which is
// read and written once, and for few requests by a trip to memory and the arithmetic behind it.  A thread has four channels of STEP_COLS columns (4,
// and 8 where a head's columns want more than STEP_THREADS threads so), the threads of a column neighbours: a wave's load is 1 KB of contiguous
// memory.  q, k, v and the decays are formed a channel or column a thread and meet in LDS; every load goes out before any is used, without branches
// between them, so that what meets there is waited for while S is on its way.  16 heads of 64 x 128, us by the walk above, whose threads
// have 16 channels, / so, at 1, 16, 32, 48, 64 requests: 5.8 / 4.3, 9.4 / 6.7, 14.1 / 9.2, 17.6 / 12.9, 24.5 / 16.7 (67 MB of S at 64); time mixing of
// 64 x 64 4.2 / 3.9, 5.9 / 5.0, 8.2 / 6.5, 10.6 / 7.7, 12.2 / 8.4.
// LOW: the decays' second product is formed here, too, by as many neighbouring lanes to a channel as there are, from weights that are asked for first: of
// rank 128 6.4 us in two launches / 6.2, 9.2 / 7.7, 15.6 / 10.0, 19.5 / 13.8, 24.4 / 18.8.
#define STEP_THREADS 512
#define LOGIT_MAX 1.329228e36f   // 2^120
#define LOW_AHEAD 2              // runs of 8 that a lane has on their way at once
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 gla_bf16x8;
template <typename T, typename TO, int STEP_COLS, bool LOW>
__global__ __launch_bounds__(STEP_THREADS) __attribute__((amdgpu_waves_per_eu(STEP_COLS == 8 ? 3 : 4))) void gla_step_kernel(GlaArgs a, int KS) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // the token's decays, q, k, TIME_MIX: u k q [4 KS] each, its outputs [dv]
  const int r = blockIdx.x, head = blockIdx.y, n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r], d = a.d, dv = a.dv, H = a.H, dpad = 4 * KS, groups = blockDim.x / KS;
  const int tid = threadIdx.x, lane = tid % WAVE, s = tid % KS, j0 = tid / KS;      // column i of the thread: j0 + groups i
  float *la = lds, *lq = lds + dpad, *lk = lds + 2 * dpad, *lu = lds + 3 * dpad, *lo = lds + 4 * dpad;
  float* sp = a.state + (size_t)a.slots[r] * a.state_stride + a.state_offset + (size_t)head * dv * dpad;      // (the same for all
  const unsigned own = 4 * s;                                                   // threads: a thread's places are 32-bit offsets from it)
  const T *rq = (const T*)a.q + head * d, *rk = (const T*)a.k + head * d, *rv = (const T*)a.v + head * dv, *rg = (const T*)a.g + head * dv;
  const float* u_h = TIME_MIX ? a.bonus + head * d : nullptr;
  const LaneSteps steps = lane_steps(KS);
  const auto weight_of = [&](int c) { return load_dyn(a.norm_w, a.norm_dtype, TIME_MIX ? head * dv + c : c); };
  // LOW: a channel of the decays by ``share`` neighbouring lanes, each its runs of 8 of the rank; else a channel a thread
  int share = 1;
  if (LOW)
    while (2 * share <= WAVE && 2 * share * dpad <= (int)blockDim.x) share *= 2;
  const LaneSteps shares = lane_steps(share);
  const int c0 = min(tid / share, d - 1), per_trip = blockDim.x / share;
  const auto decay = [&](float z) { return expf(TIME_MIX ? -expf(z) : log_sigmoid(z) * a.inv_tau); };
  for (int t = t0; t < t0 + n; ++t) {
    // (the token's rows: bases that all threads share, a thread's places 32-bit offsets from them)
    const T *q_t = rq + (size_t)t * a.ld, *k_t = rk + (size_t)t * a.ld, *v_t = rv + (size_t)t * a.ld, *g_t = rg + (size_t)t * a.ld;
    const bf16_t *low_t = LOW ? a.low + (size_t)t * a.low_ld : nullptr, *w2_h = LOW ? a.w2 + (size_t)head * d * a.rank : nullptr;
    const float* z_t = LOW ? nullptr : a.z + (size_t)t * (H * d) + head * d;
    const unsigned my_value = min(tid, dv - 1);
    // Every load of the token goes out before any is used, without a branch between them (where a thread has nothing it asks for somebody else's): those
    // of the decays ahead, then q, k and v, then S, which arrives last and is waited for last.
    gla_bf16x8 lv[LOW_AHEAD], wv[LOW_AHEAD];      // (of the thread's first channel)
    float z0 = 0.f;
    if constexpr (LOW) {
#pragma unroll
      for (int i = 0; i < LOW_AHEAD; ++i) {
        const int e = min(8 * (tid % share + share * i), a.rank - 8);
        lv[i] = *(const gla_bf16x8*)(low_t + (unsigned)e);
        wv[i] = *(const gla_bf16x8*)(w2_h + (unsigned)(c0 * a.rank + e));
      }
    } else {
      z0 = z_t[(unsigned)c0];
    }
    const float* zb = a.z_bias ? a.z_bias + head * d : (const float*)sp;      // (without a bias: any float, dropped)
    const float zb0 = zb[(unsigned)c0];
    const T v0 = v_t[my_value];
    const unsigned my_channel = min(tid, d - 1);
    const T q0 = q_t[my_channel], k0 = k_t[my_channel];
    const float u0 = TIME_MIX ? u_h[my_channel] : 0.f;
    float4 S[STEP_COLS];      // (a token's own: where a request has several, a thread reads again what it has written)
#pragma unroll
    for (int i = 0; i < STEP_COLS; ++i) S[i] = *(const float4*)(sp + (own + (unsigned)(min(j0 + groups * i, dv - 1) * dpad)));
    const T g = g_t[my_value];
    const float weight = weight_of(my_value);
    for (int c = tid / share; c < dpad; c += per_trip) {          // (LOW: a channel's lanes are of one wave, and go on or leave together)
      const bool first = c == tid / share, in = c < d;
      float z = 0.f;
      if constexpr (LOW) {
        if (first) {
#pragma unroll
          for (int i = 0; i < LOW_AHEAD; ++i) {
            float p = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) p = fmaf((float)lv[i][e], (float)wv[i][e], p);
            z += 8 * (tid % share + share * i) < a.rank ? p : 0.f;
          }
        }
        for (int r8 = 8 * (tid % share + (first ? share * LOW_AHEAD : 0)); r8 < a.rank; r8 += 8 * share) {
          const gla_bf16x8 l = *(const gla_bf16x8*)(low_t + (unsigned)r8), w = *(const gla_bf16x8*)(w2_h + (unsigned)(min(c, d - 1) * a.rank + r8));
#pragma unroll
          for (int e = 0; e < 8; ++e) z = fmaf((float)l[e], (float)w[e], z);
        }
        // (an infinite sum would reach the neighbours' channels as 0 times it: 2^120 decays as it does, and sixty-four of them are finite)
        z = z > LOGIT_MAX ? LOGIT_MAX : z < -LOGIT_MAX ? -LOGIT_MAX : z;
        z = column_sum(z, shares);
      } else {
        z = first ? z0 : z_t[(unsigned)min(c, d - 1)];
      }
      if (a.z_bias) z += first ? zb0 : zb[min(c, d - 1)];
      if (tid % share == 0) la[c] = in ? decay(z) : 0.f;
    }
    // the values lie where the outputs will: a column's is read by its lanes, which are of one wave, before one of them writes the output
    if (tid < dv) lo[tid] = to_f(v0);
    for (int c = tid + blockDim.x; c < dv; c += blockDim.x) lo[c] = to_f(v_t[c]);
    for (int c = tid; c < dpad; c += blockDim.x) {
      const bool first = c == tid;
      const unsigned ch = min(c, d - 1);
      const float q = c < d ? to_f(first ? q0 : q_t[ch]) * a.q_scale : 0.f, k = c < d ? to_f(first ? k0 : k_t[ch]) : 0.f;
      lq[c] = q;
      lk[c] = k;
      if (TIME_MIX) lu[c] = (first ? u0 : u_h[ch]) * k * q;
    }
    LDS_BARRIER();
    const float4 al = *(const float4*)(la + 4 * s), q = *(const float4*)(lq + 4 * s), k = *(const float4*)(lk + 4 * s);
    float b = 0.f;                       // TIME_MIX: sum_i u[i] k[i] q[i]
    if (TIME_MIX) {
      const float4 u = *(const float4*)(lu + 4 * s);
      b = column_sum((u.x + u.y) + (u.z + u.w), steps);
    }
#pragma unroll
    for (int i = 0; i < STEP_COLS; ++i) {
      const int j = j0 + groups * i;
      const float vf = lo[min(j, dv - 1)];
      float o = 0.f;
      if (TIME_MIX) o = (S[i].x * q.x + S[i].y * q.y) + (S[i].z * q.z + S[i].w * q.w);        // (the read-out comes before the write)
      S[i].x = fmaf(al.x, S[i].x, k.x * vf);
      S[i].y = fmaf(al.y, S[i].y, k.y * vf);
      S[i].z = fmaf(al.z, S[i].z, k.z * vf);
      S[i].w = fmaf(al.w, S[i].w, k.w * vf);
      if (j < dv) *(float4*)(sp + (own + (unsigned)(j * dpad))) = S[i];
      if (!TIME_MIX) o = (S[i].x * q.x + S[i].y * q.y) + (S[i].z * q.z + S[i].w * q.w);
      o = column_sum(o, steps);
      if (TIME_MIX) o = fmaf(b, vf, o);
      if (s == 0 && j < dv) lo[j] = o;
    }
    LDS_BARRIER();
    float ss = 0.f;
    for (int c = lane; c < dv; c += WAVE) ss = fmaf(lo[c], lo[c], ss);
    const float inv = rsqrtf(wave_sum(ss) / (float)dv + a.eps);
    TO* out = (TO*)a.out + (size_t)t * (H * dv) + head * dv;
    if (tid < dv) out[tid] = from_f<TO>(lo[tid] * inv * weight * act_silu(to_f(g)));
    for (int c = tid + blockDim.x; c < dv; c += blockDim.x) out[c] = from_f<TO>(lo[c] * inv * weight_of(c) * act_silu(to_f(g_t[c])));
    if (t + 1 < t0 + n) LDS_BARRIER();          // (the next token's decays and outputs overwrite what this one read)
  }
}

// One thread per number of a request's S: walks the request's chunks in order.  chunk_state[c] holds what chunk c
// reaches from zero and receives the state chunk c starts from.
struct CombineArgs {
  float* state; size_t state_stride, state_offset;
  const int* slots; const int* req_chunk0;       // [R + 1]: a request's chunks are req_chunk0[r] .. req_chunk0[r + 1] - 1
  float* chunk_state; const float* chunk_loga;
  int H, d, dv, parts, dp;
};

#define WALK_AHEAD 8
__global__ __launch_bounds__(256) void gla_combine_kernel(CombineArgs a) {
  const size_t per = (size_t)a.H * a.dv * a.parts * a.dp;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= per) return;
  const int r = blockIdx.y;
  const int c0 = a.req_chunk0[r], c1 = a.req_chunk0[r + 1];
  if (c1 <= c0) return;
  const int run = a.parts * a.dp;
  const int i = (int)(e % run), head = (int)(e / run / a.dv);
  float* slot = a.state + (size_t)a.slots[r] * a.state_stride + a.state_offset + e;
  if (i >= a.d) return;                   // (padding: zero for ever)
  float S = *slot;
  for (int k0 = c0; k0 < c1; k0 += WALK_AHEAD) {        // (the loads of several chunks are on their way at once)
    float mine[WALK_AHEAD], keep[WALK_AHEAD];
#pragma unroll
    for (int u = 0; u < WALK_AHEAD; ++u) {
      const int c = min(k0 + u, c1 - 1);
      mine[u] = a.chunk_state[(size_t)c * per + e];
      keep[u] = a.chunk_loga[(size_t)c * a.H * a.d + head * a.d + i];
    }
#pragma unroll
    for (int u = 0; u < WALK_AHEAD; ++u) {
      if (k0 + u >= c1) break;
      a.chunk_state[(size_t)(k0 + u) * per + e] = S;
      S = fmaf(expf(keep[u]), S, mine[u]);
    }
  }
  *slot = S;
}

#if !TIME_MIX
// ---- chunks on the matrix cores ------------------------------------------------------------------------------------------
// A chunk's walk (MODE 1 and 2 for bfloat16 rows, heads of up to 64 x 128) by blocks of 16 tokens, with B_t the sum of the block's log alpha up to
// token t, per channel, and the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: float products, float sums) for every product:
//   o_t = (q_t exp(B_t))^T S + sum_(s <= t) (sum_i q_t[i] exp(B_t - B_7)[i] k_s[i] exp(B_7 - B_s)[i]) v_s
//   S  <- exp(B_15) S + sum_s (k_s exp(B_15 - B_s)) v_s^T
// A workgroup is one head of a chunk; a wave owns 32 columns of S in the instruction's output layout, whose registers are at the same time
// the operand that the read-out wants (with its channels in another order), so S never leaves them.  A block whose decays are strong
// (B_15 below -8 in some channel: exp(B_7 - B_s) would lose digits, and overflow), or that has a value that is not finite (which a weight of zero would hand
// to the tokens before it), is walked token by token as the kernel above does.
// What bounds it is the matrix instruction (88 of 32 cycles a wave and block in MODE 2), the exponentials beside it and the block's four meeting
// points.  Both walks and what joins the chunks, 16 heads of 64 x 128, by the kernel above / here: 4,026 rows of 16 requests 268 / 113 us, 8,192 of
// four 450 / 167, a request of 200 71 / 25.  (With expf() and log1pf() 217 of the 113 us.)  The state against 64 bits, tau 16, decays' logits of
// deviation 1 about 0 and 0.3 about 4, chunks of 32: 9.0e-8 and 2.0e-7 there, 8.5e-8 and 1.6e-7 here; tau 1, 0.3 about 8 2.6e-7 and 2.0e-7, 1 about 2 6.6e-8
// and 7.9e-8.
#define BLOCK 16
#define BLOCK_MIN_DECAY -8.f
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gla_f4;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 gla_bf16x4;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 gla_bf16x8;

// exp(x) for |x| <= 8 by the hardware's exp2 of x log2(e) in two parts, and log_sigmoid by its exp2 and log2: a fifth of the instructions of expf(),
// whose ranges are not needed here, and of log1pf().  What the roundings of 1 + exp(-|x|) and of the exponential's argument lose is put back to first
// order (the second is below 2^-48): where the decays are slow it is all that is left of exp(-|x|).  Relative errors against 64 bits in float steps,
// largest and mean square, log1pf(expf()) : this : without what is put back, logits of 2 to 6 1.2e-7, 3.5e-8 : 1.6e-7, 4.4e-8 : 2.4e-5, 4.9e-6, of 10 to 17
// 1.2e-7, 3.6e-8 : 1.7e-7, 4.6e-8 : 1, 0.29.
__device__ __forceinline__ float exp_rest(float x, float h) { return 0.693147181f * fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269504f, -h)); }
__device__ __forceinline__ float block_exp(float x) {
  const float h = x * 1.44269504f, e = __builtin_amdgcn_exp2f(h);
  return fmaf(e, exp_rest(x, h), e);
}
__device__ __forceinline__ float block_log_sigmoid(float x) {
  const float y = fabsf(x) > 100.f ? -100.f : -fabsf(x), h = y * 1.44269504f;          // (NaN stays; the exponential of infinity has no rest)
  const float e = __builtin_amdgcn_exp2f(h), d = 1.f + e, rest = fmaf(e, exp_rest(y, h), e - (d - 1.f));
  return fminf(x, 0.f) - fmaf(__builtin_amdgcn_logf(d), 0.693147181f, rest * __builtin_amdgcn_rcpf(d));
}
// Over the lanes of a row of 16: those up to this one, and those behind it.  (What a token leaves of its write is summed from the block's end, not
// formed as a difference: the last tokens' sums are then small, and exact to their own last digit.)
#define SHIFTED(v, ctrl) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), (ctrl), 0xf, 0xf, true))
__device__ __forceinline__ float sum_up_to(float v) {
  v += SHIFTED(v, 0x111);
  v += SHIFTED(v, 0x112);
  v += SHIFTED(v, 0x114);
  v += SHIFTED(v, 0x118);
  return v;
}
__device__ __forceinline__ float sum_behind(float v) {
  v = SHIFTED(v, 0x101);
  v += SHIFTED(v, 0x101);
  v += SHIFTED(v, 0x102);
  v += SHIFTED(v, 0x104);
  v += SHIFTED(v, 0x108);
  return v;
}
#undef SHIFTED

template <int MODE>
__global__ __launch_bounds__(256, 2) void gla_blocks_kernel(GlaArgs a) {
  constexpr int D = 64, DV = 128, P = D + 4, PV = DV + 4;
  __shared__ __attribute__((aligned(16))) float lq[BLOCK][P], lk[BLOCK][P], la[BLOCK][P], lqm[MODE == 2 ? BLOCK : 1][P], lkm[MODE == 2 ? BLOCK : 1][P], lv[BLOCK][PV];
  __shared__ __attribute__((aligned(16))) float keep[D];
  __shared__ float squares[4][BLOCK];
  const int unit = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, wid = tid / WAVE, lane = tid % WAVE, i16 = lane % 16, g = lane / 16;
  const int t0 = a.chunk_t0[unit], n = a.chunk_len[unit], H = a.H;
  if (n <= 0) return;
  const bf16_t *rq = (const bf16_t*)a.q, *rk = (const bf16_t*)a.k, *rv = (const bf16_t*)a.v, *rg = (const bf16_t*)a.g;
  // S[ib][jb][r]: channel 16 ib + 4 g + r of column 32 wid + 16 jb + i16
  gla_f4 S[4][2];
  float* sp = a.chunk_state + ((size_t)unit * H + head) * DV * D + (size_t)(32 * wid + i16) * D + 4 * g;
#pragma unroll
  for (int ib = 0; ib < 4; ++ib)
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) S[ib][jb] = MODE == 2 ? *(const gla_f4*)(sp + (size_t)16 * jb * D + 16 * ib) : gla_f4{0.f, 0.f, 0.f, 0.f};
  float w[2][4];
  if (MODE == 2) {
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int r = 0; r < 4; ++r) w[jb][r] = load_dyn(a.norm_w, a.norm_dtype, 32 * wid + 16 * jb + 4 * g + r);
  }
  // a block's rows on their way: token tid / 16, four channels and eight values of it a thread
  // (channels from d on count as zero keys and queries that do not decay)
  const int lt = tid / 16, lc = 4 * (tid % 16), d = a.d, at = head * d + (lc < d ? lc : 0);
  gla_f4 bias = {0.f, 0.f, 0.f, 0.f};
  if (a.z_bias) bias = *(const gla_f4*)(a.z_bias + at);
  gla_bf16x4 nq, nk;
  gla_bf16x8 nv;
  gla_f4 nz;
  gla_bf16x4 ng[2], gate[2];
  auto fetch = [&](int s0) {          // (rows beyond the chunk are asked for as its last)
    const size_t t = t0 + min(s0 + lt, n - 1);
    if (MODE == 2) nq = *(const gla_bf16x4*)(rq + t * a.ld + at);
    nk = *(const gla_bf16x4*)(rk + t * a.ld + at);
    nz = *(const gla_f4*)(a.z + t * (size_t)(H * d) + at);
    nv = *(const gla_bf16x8*)(rv + t * a.ld + head * DV + 2 * lc);
    if (MODE == 2) {
      const size_t tg = t0 + min(s0 + i16, n - 1);
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) ng[jb] = *(const gla_bf16x4*)(rg + tg * a.ld + head * DV + 32 * wid + 16 * jb + 4 * g);
    }
  };
  fetch(0);
  gla_f4 loga = {0.f, 0.f, 0.f, 0.f};          // of the channels ch .. ch + 3 below
  const int ch = 16 * wid + 4 * g;             // with token i16 this thread's of the block's transformed rows
#pragma unroll 1
  for (int s0 = 0; s0 < n; s0 += BLOCK) {
    const bool row = s0 + lt < n, in = row && lc < d;
    gla_f4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = in ? block_log_sigmoid(nz[e] + bias[e]) * a.inv_tau : 0.f;
    *(gla_f4*)&la[lt][lc] = x;
    *(gla_f4*)&lk[lt][lc] = in ? gla_f4{(float)nk[0], (float)nk[1], (float)nk[2], (float)nk[3]} : gla_f4{0.f, 0.f, 0.f, 0.f};
    if (MODE == 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = in ? (float)nq[e] * a.q_scale : 0.f;
      *(gla_f4*)&lq[lt][lc] = x;
      gate[0] = ng[0], gate[1] = ng[1];
    }
    float odd = 0.f;              // NaN where a value is not finite
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = row ? (float)nv[4 * h + e] : 0.f;
        odd = fmaf(x[e], 0.f, odd);
      }
      *(gla_f4*)&lv[lt][2 * lc + 4 * h] = x;
    }
    if (s0 + BLOCK < n) fetch(s0 + BLOCK);
    __syncthreads();
    const gla_f4 mine = *(const gla_f4*)&la[i16][ch];
    gla_f4 upto, whole, half;
    bool walk = !(odd == 0.f);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      upto[e] = sum_up_to(mine[e]);
      whole[e] = __shfl(upto[e], lane | 15, WAVE);
      half[e] = __shfl(upto[e], (lane & 48) + 7, WAVE);
      walk = walk || !(whole[e] > BLOCK_MIN_DECAY);
      loga[e] += whole[e];
    }
    gla_f4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (__syncthreads_or(walk)) {
      const int ns = min(BLOCK, n - s0);
#pragma unroll 1
      for (int tt = 0; tt < ns; ++tt) {
        float v[2], sum[2] = {0.f, 0.f};
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) v[jb] = lv[tt][32 * wid + 16 * jb + i16];
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          if (16 * ib + 4 * g >= d) continue;          // (no channels: zero by a value that is not finite would be none)
          const gla_f4 l = *(const gla_f4*)&la[tt][16 * ib + 4 * g], k = *(const gla_f4*)&lk[tt][16 * ib + 4 * g];
          const gla_f4 q = MODE == 2 ? *(const gla_f4*)&lq[tt][16 * ib + 4 * g] : gla_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float al = expf(l[r]);
#pragma unroll
            for (int jb = 0; jb < 2; ++jb) {
              S[ib][jb][r] = fmaf(al, S[ib][jb][r], k[r] * v[jb]);
              if (MODE == 2) sum[jb] = fmaf(S[ib][jb][r], q[r], sum[jb]);
            }
          }
        }
        if (MODE == 2) {
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) {
            sum[jb] += __shfl_xor(sum[jb], 16, WAVE);
            sum[jb] += __shfl_xor(sum[jb], 32, WAVE);
            if (g == 0) lv[tt][32 * wid + 16 * jb + i16] = sum[jb];          // (in place of the values, this wave's own)
          }
        }
      }
      if (MODE == 2) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) o[jb] = *(const gla_f4*)&lv[i16][32 * wid + 16 * jb + 4 * g];
      }
    } else {
      gla_f4 k = *(const gla_f4*)&lk[i16][ch], kl, km, q1, qm;
      const gla_f4 q = MODE == 2 ? *(const gla_f4*)&lq[i16][ch] : k;
      if (i16 == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) kl[e] = block_exp(whole[e]);
        *(gla_f4*)&keep[ch] = kl;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kl[e] = k[e] * block_exp(sum_behind(mine[e]));
        if (MODE == 2) {
          km[e] = k[e] * block_exp(half[e] - upto[e]);
          qm[e] = q[e] * block_exp(upto[e] - half[e]);
          q1[e] = q[e] * block_exp(upto[e]);
        }
      }
      *(gla_f4*)&lk[i16][ch] = kl;          // (each thread in place of what it read)
      if (MODE == 2) {
        *(gla_f4*)&lq[i16][ch] = q1;
        *(gla_f4*)&lqm[i16][ch] = qm;
        *(gla_f4*)&lkm[i16][ch] = km;
      }
      __syncthreads();
      float v[2][4];
#pragma unroll
      for (int jb = 0; jb < 2; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[jb][r] = lv[4 * g + r][32 * wid + 16 * jb + i16];
      if (MODE == 2) {
        gla_f4 pairs = {0.f, 0.f, 0.f, 0.f};          // what token i16 takes of tokens 4 g + r
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          const gla_f4 ks = *(const gla_f4*)&lkm[i16][16 * ib + 4 * g], qs = *(const gla_f4*)&lqm[i16][16 * ib + 4 * g], qo = *(const gla_f4*)&lq[i16][16 * ib + 4 * g];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            pairs = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[r], qs[r], pairs, 0, 0, 0);
#pragma unroll
            for (int jb = 0; jb < 2; ++jb) o[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[ib][jb][r], qo[r], o[jb], 0, 0, 0);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = 4 * g + r <= i16 ? pairs[r] : 0.f;
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) o[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[jb][r], p, o[jb], 0, 0, 0);
        }
      }
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        const gla_f4 kept = *(const gla_f4*)&keep[16 * ib + 4 * g];
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[ib][jb][r] *= kept[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          const float kt = lk[4 * g + r][16 * ib + i16];
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) S[ib][jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt, v[jb][r], S[ib][jb], 0, 0, 0);
        }
    }
    if (MODE == 2) {
      float ss = 0.f;
#pragma unroll
      for (int jb = 0; jb < 2; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r) ss = fmaf(o[jb][r], o[jb][r], ss);
      ss += __shfl_xor(ss, 16, WAVE);
      ss += __shfl_xor(ss, 32, WAVE);
      if (g == 0) squares[wid][i16] = ss;
    }
    __syncthreads();                         // (and the next block's rows overwrite what this one read)
    if (MODE == 2 && s0 + i16 < n) {
      const float inv = rsqrtf((((squares[0][i16] + squares[1][i16]) + squares[2][i16]) + squares[3][i16]) / (float)DV + a.eps);
      bf16_t* out = (bf16_t*)a.out + (size_t)(t0 + s0 + i16) * (size_t)(H * DV) + head * DV + 32 * wid + 4 * g;
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        gla_bf16x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = (__bf16)(o[jb][r] * inv * w[jb][r] * over_one_plus_exp<false>((float)gate[jb][r], (float)gate[jb][r]));
        *(gla_bf16x4*)(out + 16 * jb) = y;
      }
    }
  }
  if (MODE == 1) {
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) *(gla_f4*)(sp + (size_t)16 * jb * D + 16 * ib) = S[ib][jb];
    if (i16 == 0 && ch < d) *(gla_f4*)(a.chunk_loga + (size_t)unit * H * d + head * d + ch) = loga;
  }
}

static bool blocks_take(const GlaArgs& a, int dp) {
  return a.d <= 64 && a.d % 4 == 0 && a.dv == 128 && a.parts * dp == 64 && a.ld % 8 == 0
         && ((size_t)a.q | (size_t)a.k | (size_t)a.v | (size_t)a.g | (size_t)a.z | (size_t)a.z_bias | (size_t)a.out | (size_t)a.chunk_state | (size_t)a.chunk_loga) % 16 == 0;
}
#endif

template <typename T, typename TO, int DP, int MODE, int COLS>
static void launch_gla_mode(const GlaArgs& a, int units, int threads, size_t lds, hipStream_t s) {
  if constexpr (DP <= 32) {
    if (a.parts * DP == a.d && threads <= 512) {
      hipLaunchKernelGGL((gla_kernel<T, TO, DP, MODE, COLS, true>), dim3(units, a.H), dim3(threads), lds, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((gla_kernel<T, TO, DP, MODE, COLS, false>), dim3(units, a.H), dim3(threads), lds, s, a);
}

// A launch of MODE with ``cols`` columns of S a thread (1, 2 or 4; what DP allows is checked by the caller).
template <typename T, typename TO, int DP, int MODE>
static void launch_gla_cols(const GlaArgs& a, int units, int cols, int threads, size_t lds, hipStream_t s) {
  if constexpr (DP <= 16) { if (cols == 4) return launch_gla_mode<T, TO, DP, MODE, 4>(a, units, threads, lds, s); }
  if constexpr (DP <= 32) { if (cols == 2) return launch_gla_mode<T, TO, DP, MODE, 2>(a, units, threads, lds, s); }
  launch_gla_mode<T, TO, DP, MODE, 1>(a, units, threads, lds, s);
}

// The threads of gla_step_kernel for a head of these sizes, 0 where it does not take them.
static int step_threads(int dpad, int dv, int cols) {
  const int lanes = dpad / 4, threads = (lanes * ((dv + cols - 1) / cols) + WAVE - 1) / WAVE * WAVE;
  return lanes <= WAVE && threads <= STEP_THREADS ? threads : 0;
}

template <typename T, typename TO, int DP>
static int launch_gla(const GlaArgs& a, int T_rows, int R, int n_chunks, const int* req_chunk0, hipStream_t s) {
  if constexpr (sizeof(TO) == 2) {         // (in 32 bits a token's bits are the same alone and among others of its request: the walk's)
    const int cols = step_threads(a.parts * DP, a.dv, 4) > 0 ? 4 : 8, threads = n_chunks == 0 && T_rows <= R ? step_threads(a.parts * DP, a.dv, cols) : 0;
    if (threads > 0) {
      const size_t lds = (size_t)(4 * a.parts * DP + a.dv) * sizeof(float);
#define STEP(COLS, LOW) hipLaunchKernelGGL((gla_step_kernel<T, TO, COLS, LOW>), dim3(R, a.H), dim3(threads), lds, s, a, a.parts * DP / 4)
      if constexpr (!TIME_MIX && sizeof(T) == 2) {
        if (a.low) {
          if (cols == 4) STEP(4, true);
          else STEP(8, true);
          IFX_LAUNCH_CHECK();
        }
      }
      if (cols == 4) STEP(4, false);
      else STEP(8, false);
#undef STEP
      IFX_LAUNCH_CHECK();
    }
  }
  // A thread holds 1, 2 or 4 columns of S as its registers allow (4 for runs of 16 channels, 2 for 32): what it reads of a
  // token's q, k and decays from LDS then serves several columns.  Two where possible, more only where a head's columns would not fit a
  // workgroup otherwise.  us by one column / two: single tokens of 1, 16 and 64 requests in 32 bits, 16 heads of 64 x 128, 4.9, 8.2, 23.7 / 5.6, 9.0,
  // 23.4, in bfloat16 where gla_step_kernel does not take them, 4 heads of 128 x 256, 15.0, 17.1, 25.3 / 12.5, 15.1, 23.1; chunks that the
  // matrix cores do not take, 2,048 rows of 16 heads of 96 x 128, 493 / 382, but of 64 x 96 140 / 178; a prompt of 2,048 rows in 32 bits, one chain,
  // is longer by two: 16 heads of 64 x 128 1,639 / 2,732.  The first d threads also load, so a head of few values still gets a thread per key channel.
  IFX_REQUIRE(a.z, "gla_scan: the decays' second product is formed in steps of single tokens only (bfloat16, heads that gla_step_takes)");
  constexpr int MAX_COLS = DP <= 16 ? 4 : (DP <= 32 ? 2 : 1);
  const auto threads_for = [&](int cols) { return ((max((a.dv + cols - 1) / cols * a.parts, a.d) + WAVE - 1) / WAVE) * WAVE; };
  // (time mixing's heads have as few values as keys: with two columns a thread a head of 64 x 64 would be two waves)
  int cols_chunk = TIME_MIX && threads_for(1) <= 256 ? 1 : min(2, MAX_COLS);
  while (cols_chunk < MAX_COLS && threads_for(cols_chunk) > GLA_MAX_THREADS(DP)) cols_chunk *= 2;
  const int cols_walk = cols_chunk;
  IFX_REQUIRE(threads_for(cols_chunk) <= GLA_MAX_THREADS(DP), "gla_scan: %d threads a head with %d channels each (at most %d)",
              threads_for(cols_chunk), DP, GLA_MAX_THREADS(DP));
  const size_t lds = (size_t)STAGE * (4 * a.d + a.dv) * sizeof(float);
  if (n_chunks == 0) {
    launch_gla_cols<T, TO, DP, 0>(a, R, cols_walk, threads_for(cols_walk), lds, s);
    IFX_LAUNCH_CHECK();
  }
  bool blocks = false;
#if !TIME_MIX
  if constexpr (sizeof(T) == 2) blocks = blocks_take(a, DP);
  if (blocks) hipLaunchKernelGGL(gla_blocks_kernel<1>, dim3(n_chunks, a.H), dim3(256), 0, s, a);
#endif
  if (!blocks) launch_gla_cols<T, TO, DP, 1>(a, n_chunks, cols_chunk, threads_for(cols_chunk), lds, s);
  CombineArgs c{a.state, a.state_stride, a.state_offset, a.slots, req_chunk0, a.chunk_state, a.chunk_loga, a.H, a.d, a.dv, a.parts, DP};
  const size_t per = (size_t)a.H * a.dv * a.parts * DP;
  hipLaunchKernelGGL(gla_combine_kernel, dim3((unsigned)((per + 255) / 256), R), dim3(256), 0, s, c);
#if !TIME_MIX
  if (blocks) hipLaunchKernelGGL(gla_blocks_kernel<2>, dim3(n_chunks, a.H), dim3(256), 0, s, a);
#endif
  if (!blocks) launch_gla_cols<T, TO, DP, 2>(a, n_chunks, cols_chunk, threads_for(cols_chunk), lds, s);
  IFX_LAUNCH_CHECK();
}

// dp: channels a thread holds (16, 32, 64 or 128); parts: a power of two with parts * dp >= d; a head's columns, 1-4 a thread,
// times parts must fit a workgroup.
// z null: z = w2 low with low [T, rank] bfloat16, rows low_ld apart, both on 16 bytes, rank a multiple of 8 (see ifx_gla_step_takes).
extern "C" int ifx_gla_step_takes(int dpad, int dv) { return !TIME_MIX && step_threads(dpad, dv, 8) > 0 ? 1 : 0; }

extern "C" int ifx_gla_scan(const void* q, const void* k, const void* v, const void* g, int dtype, int out_dtype, int ld, const float* z,
                            const void* low, int low_ld, const void* w2, int rank, const float* z_bias, float inv_tau, float q_scale, float eps, const void* norm_w, int norm_dtype, const float* bonus,
                            float* state, long long state_stride, long long state_offset, const int* q_start, const int* q_len,
                            const int* slots, void* out, int T, int R, int H, int d, int dv, int dp, int parts,
                            int n_chunks, const int* chunk_req, const int* chunk_t0, const int* chunk_len,
                            const int* req_chunk0, float* chunk_state, float* chunk_loga, void* stream) {
  IFX_REQUIRE(T >= 0 && R >= 0 && H > 0 && d > 0 && dv > 0, "gla_scan: bad sizes T=%d R=%d H=%d d=%d dv=%d", T, R, H, d, dv);
  IFX_REQUIRE(parts > 0 && (parts & (parts - 1)) == 0 && parts <= WAVE && parts * dp >= d, "gla_scan: %d parts of %d channels for d=%d", parts, dp, d);
  IFX_REQUIRE(d <= 1024, "gla_scan: a head of %d key channels does not fit a workgroup", d);
  IFX_REQUIRE((state_offset % 4) == 0 && (state_stride % 4) == 0, "gla_scan: the state must lie at a multiple of 16 bytes");
  IFX_REQUIRE(state_stride >= state_offset + (long long)H * dv * parts * dp, "gla_scan: a state row of %lld floats is too short", state_stride);
  IFX_REQUIRE(n_chunks == 0 || (chunk_req && chunk_t0 && chunk_len && req_chunk0 && chunk_state && chunk_loga), "gla_scan: chunks without their lists");
  IFX_REQUIRE((size_t)STAGE * (4 * d + dv) * sizeof(float) <= 64 * 1024, "gla_scan: d=%d, dv=%d need more LDS than a workgroup has", d, dv);
  IFX_REQUIRE(!TIME_MIX || bonus, "time mixing needs the bonus per channel");
  IFX_REQUIRE((z == nullptr) == (low != nullptr) && (low != nullptr) == (w2 != nullptr), "gla_scan: the decays' logits, or what they are the product of");
  IFX_REQUIRE(!low || (rank > 0 && rank % 8 == 0 && low_ld >= rank && low_ld % 8 == 0 && (uintptr_t)low % 16 == 0 && (uintptr_t)w2 % 16 == 0),
              "gla_scan: a product of rank %d, rows %d apart (multiples of 8, on 16 bytes)", rank, low_ld);
  if (T == 0 || R == 0) return 0;
  GlaArgs a{q, k, v, g, ld, z, (const bf16_t*)low, (const bf16_t*)w2, low_ld, rank, z_bias, inv_tau, q_scale, eps, norm_w, norm_dtype, bonus, state,
            (size_t)state_stride, (size_t)state_offset, q_start, q_len, slots, out, H, d, dv, parts,
            chunk_req, chunk_t0, chunk_len, chunk_state, chunk_loga};
  hipStream_t s = (hipStream_t)stream;
#define GLA_CASE2(TY, TO, DPV) if (dp == DPV) return launch_gla<TY, TO, DPV>(a, T, R, n_chunks, req_chunk0, s);
#define GLA_CASE(TY, DPV) GLA_CASE2(TY, TY, DPV)
#if TIME_MIX
  if (dtype == DT_F32 && out_dtype == DT_BF16) { GLA_CASE2(float, bf16_t, 16) GLA_CASE2(float, bf16_t, 32) GLA_CASE2(float, bf16_t, 64) GLA_CASE2(float, bf16_t, 128) }
#endif
  if (dtype != out_dtype) IFX_FAIL("gla_scan: rows of type %d with an output of type %d", dtype, out_dtype);
  if (dtype == DT_F32) { GLA_CASE(float, 16) GLA_CASE(float, 32) GLA_CASE(float, 64) GLA_CASE(float, 128) }
  else if (dtype == DT_BF16) { GLA_CASE(bf16_t, 16) GLA_CASE(bf16_t, 32) GLA_CASE(bf16_t, 64) GLA_CASE(bf16_t, 128) }
  else IFX_FAIL("gla_scan: unknown dtype %d", dtype);
#undef GLA_CASE
#undef GLA_CASE2
  IFX_FAIL("gla_scan: %d channels a thread (16, 32, 64 or 128)", dp);
}
