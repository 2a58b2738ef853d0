// The gated delta rule: a recurrence per head whose state is a matrix S [d, dv] that is decayed by one number per token
// and corrected towards the token's value along the token's key.
//
// For a request's tokens t = 0, 1, ... and value head h (which reads query/key head h / (heads / kv_heads)):
//
//   q = unit(q_in) * d^(-1/2),  k = unit(k_in),  unit(x) = x / sqrt(sum(x^2) + 1e-6)
//   beta = sigmoid(b_in),  g = exp(-exp(A_log[h]) * softplus(a_in + dt_bias[h]))
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q          (the read-out sees the token's own write)
//   out = o / sqrt(mean(o^2) + eps) * w_norm * silu(gate_in)              (the norm over the head's dv values)
//
// q_in, k_in, v come from ``u`` [T, ldu] (the convolution's output: q heads, then k heads, then v heads), gate_in, b_in,
// a_in from ``rows`` [T, ldr] at the given columns; all of them in the activation type.  Unit norms, beta, the decay and
// its logarithms, S, every sum, the norm and the gate are float whatever that type is.
//
// A request's S lives in its state slot, float32, at ``state_offset`` floats into the slot's row, laid out
// [head][value column][d_pad] with d_pad = CH * KS >= d.  The columns of S never meet (column j is only ever read and
// written with v_j, u_j and o_j), so a head's columns are dealt to several workgroups of ``cols`` columns each, which
// spreads one request over many compute units.  In a workgroup thread (column j, run s) holds CH consecutive key channels
// of column j in registers; the KS threads of a column are neighbouring lanes and add their parts of S^T k and S^T q by
// butterfly shuffles (a fixed order).  Tokens are taken STAGE at a time: all threads load the stage's q, k and their
// columns of v into LDS (the next stage's are asked for before the walk and land in registers meanwhile), a few lanes per
// (token, vector) form the unit norms, a thread per token beta and the decay; everybody walks the stage's tokens and
// leaves o in LDS, from where it goes to ``o_raw`` [T, H dv] (float).  A second kernel, a wave per (token, head), norms and
// gates o.  The order of a token's operations does not depend on how a request's portions were cut, so its results are the same bits in
// every cutting into portions.  Tokens that come one to a step differ by their sums' order: in 32 bits their layout gives a thread of the walk more channels
// (differences of 1e-6); in bfloat16 they have a kernel of their own (delta_step_kernel), which does not round the convolution's output either.
#include "common.h"
#include "lane_sums.h"

IFX_DEFINE_LAST_ERROR()


struct DeltaArgs {
  const void* u;          // [T, ldu]: q (G d) | k (G d) | v (H dv)
  int ldu;
  const void* rows;       // [T, ldr]: the gate's columns from col_g, beta's from col_b, the decay's from col_a
  int ldr, col_g, col_b, col_a;
  const float* A_log;     // [H]
  const float* dt_bias;   // [H]
  const void* norm_w;     // [dv]
  int norm_dtype;
  float eps;
  float* state;           // [slots, state_stride]
  size_t state_stride, state_offset;
  const int* q_start; const int* q_len; const int* slots;     // [R]
  void* out;              // [T, H dv]
  float* o_raw;           // [T, H dv]: the read-outs before their norm and gate
  int T, H, G, d, dv, KS, cols;
};

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

#define STAGE 16
#define MAX_DPAD 256
#define MAX_COLS 128
#define MAX_PRE 16          // q and k elements of a stage a thread fetches at most (STAGE * d_pad / threads)
#define MAX_PRE_V 8         // ... and v elements (STAGE * columns / threads)

template <typename T, int CH>
__global__ __launch_bounds__(256) void delta_kernel(DeltaArgs a) {
  // LDS as the head's sizes need it (so that several workgroups share a compute unit): q and k of a stage [STAGE][dpad]
  // each, then its v and o [STAGE][cols] each
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float beta_s[STAGE + 1], g_s[STAGE + 1];      // (one more: the walk reads a token ahead, also behind the last)
  const int n_cb = (a.dv + a.cols - 1) / a.cols;
  const int h = blockIdx.x / n_cb, j0 = (blockIdx.x % n_cb) * a.cols, r = blockIdx.y;
  const int n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r];
  const int d = a.d, dv = a.dv, KS = a.KS, dpad = CH * KS;
  const int cols = min(a.cols, dv - j0);
  float* q_s = lds;
  float* k_s = lds + STAGE * dpad;
  float* v_s = lds + 2 * STAGE * dpad;
  float* o_s = v_s + STAGE * a.cols;
  const int g = h / (a.H / a.G);
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int wid = tid / WAVE, lane = tid % WAVE, nw = (nthr + WAVE - 1) / WAVE;
  const int jl = tid / KS, s = tid % KS;             // this thread's column (within the workgroup's) and its run of channels
  const bool owner = jl < cols;
  float* Sp = a.state + (size_t)a.slots[r] * a.state_stride + a.state_offset + ((size_t)h * dv + j0 + (owner ? jl : 0)) * dpad + s * CH;
  float S[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) S[i] = owner ? Sp[i] : 0.f;
  const T* u = (const T*)a.u;
  const T* rows = (const T*)a.rows;
  const float decay_rate = expf(a.A_log[h]), dt_b = a.dt_bias[h], q_mult = 1.0f / sqrtf((float)d);
  const LaneSteps col_steps = lane_steps(KS);
  const int NL = nthr >= 256 ? 8 : (nthr >= 128 ? 4 : 2);      // lanes to a (token, vector) pair of a stage's 2 STAGE unit norms
  // What a thread fetches of a stage: elements x = tid, tid + nthr, ... of the stage's (token, channel) pairs of q and of k
  // and of its (token, column) pairs of v.  STAGE * dpad and STAGE * cols are at most MAX_PRE * nthr.
  // (dpad is a power of two; the places of a thread's v elements are the same in every stage and found once)
  const int per_qk = (STAGE * dpad + nthr - 1) / nthr, per_v = (STAGE * cols + nthr - 1) / nthr;
  const int dshift = __ffs(dpad) - 1;
  // a thread's v elements of a stage are x = tid, tid + nthr, ...: (token, column) = (x / cols, x % cols), stepped from the
  // first by (nthr / cols, nthr % cols) with a carry, so that one division a thread is all there is
  const int v_tt0 = tid / cols, v_c0 = tid - v_tt0 * cols, v_dq = nthr / cols, v_dr = nthr - v_dq * cols;
  float pq[MAX_PRE], pk[MAX_PRE], pv[MAX_PRE_V], pb = 0.f, pg = 0.f;
  auto fetch = [&](int base) {
    const int cnt = min(STAGE, n - base);
#pragma unroll
    for (int e = 0; e < MAX_PRE; ++e) {
      if (e >= per_qk) break;
      const int x = tid + e * nthr, tt = x >> dshift, c = x & (dpad - 1);
      const bool in = tt < cnt && c < d;
      const size_t row = (size_t)(t0 + base + (in ? tt : 0)) * a.ldu;
      pq[e] = in ? to_f(u[row + (size_t)g * d + c]) : 0.f;
      pk[e] = in ? to_f(u[row + (size_t)(a.G + g) * d + c]) : 0.f;
    }
    int tt = v_tt0, c = v_c0;
#pragma unroll
    for (int e = 0; e < MAX_PRE_V; ++e) {
      if (e >= per_v) break;
      const bool in = tt < cnt;
      pv[e] = in ? to_f(u[(size_t)(t0 + base + tt) * a.ldu + (size_t)2 * a.G * d + (size_t)h * dv + j0 + c]) : 0.f;
      tt += v_dq; c += v_dr;
      if (c >= cols) { c -= cols; ++tt; }
    }
    if (tid < cnt) {
      const size_t row = (size_t)(t0 + base + tid) * a.ldr;
      pb = to_f(rows[row + a.col_b + h]);
      pg = to_f(rows[row + a.col_a + h]);
    }
  };
  fetch(0);
  for (int base = 0; base < n; base += STAGE) {
    const int cnt = min(STAGE, n - base);
    LDS_BARRIER();              // the last stage's walk is done with q_s, k_s, v_s, its write-out with o_s
#pragma unroll
    for (int e = 0; e < MAX_PRE; ++e) {
      if (e >= per_qk) break;
      const int x = tid + e * nthr;
      if (x < STAGE * dpad) { q_s[x] = pq[e]; k_s[x] = pk[e]; }
    }
    {
      int tt = v_tt0, c = v_c0;
#pragma unroll
      for (int e = 0; e < MAX_PRE_V; ++e) {
        if (e >= per_v) break;
        if (tt < STAGE) v_s[tt * a.cols + c] = pv[e];
        tt += v_dq; c += v_dr;
        if (c >= cols) { c -= cols; ++tt; }
      }
    }
    if (tid < cnt) {
      beta_s[tid] = 1.0f / (1.0f + expf(-pb));
      g_s[tid] = expf(-decay_rate * softplus_f(pg + dt_b));
    }
    LDS_BARRIER();
    if (base + STAGE < n) fetch(base + STAGE);          // the next stage's loads are on their way during the norms and the walk
    // unit norms: NL neighbouring lanes per (token, q or k), all pairs at once; the lanes' squares added by column_sum
    {
      const LaneSteps norm_steps = lane_steps(NL);
      const int pair = tid / NL, l = tid % NL;
      float* vec = ((pair & 1) ? k_s : q_s) + min(pair >> 1, STAGE - 1) * dpad;
      const bool mine = pair < 2 * cnt;
      float ss = 0.f;
      if (mine)
        for (int c = l; c < d; c += NL) ss = fmaf(vec[c], vec[c], ss);
      ss = column_sum(ss, norm_steps);
      if (mine) {
        const float f = ((pair & 1) ? 1.0f : q_mult) / sqrtf(ss + 1e-6f);
        for (int c = l; c < d; c += NL) vec[c] *= f;
      }
    }
    LDS_BARRIER();
    if (owner) {
      // a token's k, q, v, decay and beta are read from LDS while the token before it is worked on; the sums over a
      // thread's channels run in four chains that are added at the end (a fixed order)
      const float* kp = k_s + s * CH;          // this thread's channels of the stage's first token; a token further: + dpad
      const float* qp = q_s + s * CH;
      const float* vp = v_s + jl;
      float kn[CH], qn[CH], vn = vp[0], gn = g_s[0], bn = beta_s[0];
#pragma unroll
      for (int i = 0; i < CH; ++i) { kn[i] = kp[i]; qn[i] = qp[i]; }
#pragma unroll 2
      for (int tt = 0; tt < cnt; ++tt) {
        float kk[CH], qq[CH];
        const float gd = gn, bt = bn, vt = vn;
#pragma unroll
        for (int i = 0; i < CH; ++i) { kk[i] = kn[i]; qq[i] = qn[i]; }
        // the token after this one, also behind the stage's last, where what is read lies inside the workgroup's LDS all the
        // same (the row behind q's last is k's first, behind k's last v's first, behind v's last o's first) and is never used
        kp += dpad; qp += dpad; vp += a.cols;
        vn = vp[0]; gn = g_s[tt + 1]; bn = beta_s[tt + 1];
#pragma unroll
        for (int i = 0; i < CH; ++i) { kn[i] = kp[i]; qn[i] = qp[i]; }
        float p4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          S[i] *= gd;
          p4[i & 3] = fmaf(S[i], kk[i], p4[i & 3]);
        }
        const float pred = column_sum((p4[0] + p4[1]) + (p4[2] + p4[3]), col_steps);
        const float upd = bt * (vt - pred);
        float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          S[i] = fmaf(kk[i], upd, S[i]);
          o4[i & 3] = fmaf(S[i], qq[i], o4[i & 3]);
        }
        const float out = column_sum((o4[0] + o4[1]) + (o4[2] + o4[3]), col_steps);
        if (s == 0) o_s[tt * a.cols + jl] = out;
      }
    }
    LDS_BARRIER();
    for (int x = tid; x < cnt * cols; x += nthr)
      a.o_raw[((size_t)(t0 + base + x / cols) * a.H + h) * dv + j0 + x % cols] = o_s[(x / cols) * a.cols + x % cols];
  }
  if (owner) {
#pragma unroll
    for (int i = 0; i < CH; ++i) Sp[i] = S[i];
  }
}

// out[t, h, :] = o_raw[t, h, :] / sqrt(mean(o_raw[t, h, :]^2) + eps) * w * silu(gate[t, h, :]): a wave per (token, head)
template <typename T>
__global__ __launch_bounds__(256) void delta_finish_kernel(DeltaArgs a) {
  const size_t item = (size_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  const int lane = threadIdx.x % WAVE;
  if (item >= (size_t)a.T * a.H) return;
  const size_t t = item / a.H;
  const int h = (int)(item % a.H), dv = a.dv;
  const float* o = a.o_raw + item * dv;
  float ss = 0.f;
  for (int c = lane; c < dv; c += WAVE) ss = fmaf(o[c], o[c], ss);
  const float f = 1.0f / sqrtf(wave_sum(ss) / (float)dv + a.eps);
  const T* rows = (const T*)a.rows;
  for (int c = lane; c < dv; c += WAVE) {
    const float gt = to_f(rows[t * a.ldr + a.col_g + (size_t)h * dv + c]);
    ((T*)a.out)[item * dv + c] = from_f<T>(o[c] * f * load_dyn(a.norm_w, a.norm_dtype, c) * act_silu(gt));
  }
}

// Steps of single tokens in bfloat16 (a request's tokens one after the other where it has more): a workgroup takes a head of a request, so that the norm is
// there with the outputs, and with TAPS > 0 (heads with q and k of their own) the convolution before it, too.  A thread has four channels of COLS
// columns of S, the dpad / 4 threads of a column neighbours: a wave's load is 1 KB of contiguous memory.  The convolution is a channel a thread; its
// results and the gates meet in LDS, and every load goes out before any is used, without branches between them, so that what meets there is waited for
// while S is on its way.  Everything between the rows and the output is float.  Bound by its launch, a trip to memory and the arithmetic behind it, for
// many requests by S.  16 heads of 64 x 128, four taps, us in launches for the convolution, the walk and the norm / in one, at 1, 16, 32, 64
// requests: 13.0 / 5.2, 24.0 / 7.6, 37.8 / 10.1, 70.4 / 19.7 (67 MB of S at 64).  (32-bit steps stay with the walk.)
struct StepConv {
  const void* w;          // [2 G d + H dv][TAPS]
  int w_dtype;
  float* state;           // a slot's row begins with its last TAPS - 1 inputs of every channel
};
#define STEP_THREADS 512
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 step_bf16x4;
template <int TAPS, int COLS>
__global__ __launch_bounds__(STEP_THREADS) __attribute__((amdgpu_waves_per_eu(COLS == 8 ? 3 : 4))) void delta_step_kernel(DeltaArgs a, StepConv conv) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // q and k of a token [dpad] each, its values, in whose place its outputs [dv]
  __shared__ float gate_s[2];                                       // beta, decay
  const int h = blockIdx.x, r = blockIdx.y, n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r], d = a.d, dv = a.dv, KS = a.KS, dpad = 4 * KS, groups = blockDim.x / KS, g = h / (a.H / a.G);
  float *q_s = lds, *k_s = lds + dpad, *o_s = lds + 2 * dpad;
  const int tid = threadIdx.x, lane = tid % WAVE, s = tid % KS, j0 = tid / KS;      // column i of the thread: j0 + groups i
  const unsigned own = 4 * s, my_value = min(tid, dv - 1);
  const size_t slot = (size_t)a.slots[r] * a.state_stride;
  float* Sp = a.state + slot + a.state_offset + (size_t)h * dv * dpad;      // (the same for all threads: a thread's places are 32-bit offsets from it)
  static_assert(TAPS == 0 || TAPS == 4, "four taps, or no convolution");
  const int n_in = 2 * d + dv;                     // the head's channels: q, k, v
  const auto channel_of = [&](int i) { return i < d ? g * d + i : i < 2 * d ? a.G * d + g * d + (i - d) : 2 * a.G * d + h * dv + (i - 2 * d); };
  const auto place_of = [&](int i) { return i < d ? q_s + i : i < 2 * d ? k_s + (i - d) : o_s + (i - 2 * d); };
  const LaneSteps steps = lane_steps(KS);
  const float decay_rate = a.A_log[h], dt_b = a.dt_bias[h], q_mult = 1.0f / sqrtf((float)d);
  for (int t = t0; t < t0 + n; ++t) {
    const bf16_t *u = (const bf16_t*)a.u + (size_t)t * a.ldu, *row = (const bf16_t*)a.rows + (size_t)t * a.ldr;
    const bf16_t zb = row[a.col_b + h], za = row[a.col_a + h];
    const unsigned c0 = channel_of(min(tid, n_in - 1));
    const bf16_t x0 = u[c0];
    float4 wf = {};
    step_bf16x4 wh = {};
    float b0 = 0.f, b1 = 0.f, b2 = 0.f;
    if constexpr (TAPS > 0) {
      const float* st = conv.state + slot + c0 * 3;
      b0 = st[0]; b1 = st[1]; b2 = st[2];
      if (conv.w_dtype == DT_F32) wf = ((const float4*)conv.w)[c0];
      else wh = ((const step_bf16x4*)conv.w)[c0];
    }
    float4 S[COLS];      // (a token's own: where a request has several, a thread reads again what it has written)
#pragma unroll
    for (int i = 0; i < COLS; ++i) S[i] = *(const float4*)(Sp + (own + (unsigned)(min(j0 + groups * i, dv - 1) * dpad)));
    const bf16_t gate = row[a.col_g + h * dv + my_value];
    const float weight = load_dyn(a.norm_w, a.norm_dtype, my_value);
    // one input: the convolution over it and the three before it, the last three left in the state
    const auto put = [&](int i, unsigned c, float x, float last0, float last1, float last2, float4 w) {
      if constexpr (TAPS > 0) {
        float* st = conv.state + slot + c * 3;
        st[0] = last1; st[1] = last2; st[2] = x;
        x = act_silu(fmaf(w.w, x, fmaf(w.z, last2, fmaf(w.y, last1, w.x * last0))));
      }
      *place_of(i) = x;
    };
    const auto widened = [&](float4 f, step_bf16x4 h) { return conv.w_dtype == DT_F32 ? f : make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]); };
    if (tid < n_in) put(tid, c0, to_f(x0), b0, b1, b2, widened(wf, wh));
    for (int i = tid + blockDim.x; i < n_in; i += blockDim.x) {      // (a head of more channels than threads)
      const unsigned c = channel_of(i);
      if constexpr (TAPS > 0) {
        const float* st = conv.state + slot + c * 3;
        b0 = st[0]; b1 = st[1]; b2 = st[2];
        if (conv.w_dtype == DT_F32) wf = ((const float4*)conv.w)[c];
        else wh = ((const step_bf16x4*)conv.w)[c];
      }
      put(i, c, to_f(u[c]), b0, b1, b2, widened(wf, wh));
    }
    for (int c = d + tid; c < dpad; c += blockDim.x) { q_s[c] = 0.f; k_s[c] = 0.f; }
    if (tid == (int)blockDim.x - 1) {               // (a thread of the last wave, which has no channel as a rule)
      gate_s[0] = 1.0f / (1.0f + expf(-to_f(zb)));
      gate_s[1] = expf(-expf(decay_rate) * softplus_f(to_f(za) + dt_b));
    }
    LDS_BARRIER();
    const float beta = gate_s[0], decay = gate_s[1];
    float4 q = *(const float4*)(q_s + own), k = *(const float4*)(k_s + own);
    const float fq = q_mult / sqrtf(column_sum((q.x * q.x + q.y * q.y) + (q.z * q.z + q.w * q.w), steps) + 1e-6f);
    const float fk = 1.0f / sqrtf(column_sum((k.x * k.x + k.y * k.y) + (k.z * k.z + k.w * k.w), steps) + 1e-6f);
    q.x *= fq; q.y *= fq; q.z *= fq; q.w *= fq;
    k.x *= fk; k.y *= fk; k.z *= fk; k.w *= fk;
#pragma unroll
    for (int i = 0; i < COLS; ++i) {
      const int j = j0 + groups * i;
      S[i].x *= decay; S[i].y *= decay; S[i].z *= decay; S[i].w *= decay;
      const float upd = beta * (o_s[min(j, dv - 1)] - column_sum((S[i].x * k.x + S[i].y * k.y) + (S[i].z * k.z + S[i].w * k.w), steps));
      S[i].x = fmaf(k.x, upd, S[i].x);
      S[i].y = fmaf(k.y, upd, S[i].y);
      S[i].z = fmaf(k.z, upd, S[i].z);
      S[i].w = fmaf(k.w, upd, S[i].w);
      if (j < dv) *(float4*)(Sp + (own + (unsigned)(j * dpad))) = S[i];
      const float o = column_sum((S[i].x * q.x + S[i].y * q.y) + (S[i].z * q.z + S[i].w * q.w), steps);
      if (s == 0 && j < dv) o_s[j] = o;           // (a column's lanes are of one wave, and have read its value)
    }
    LDS_BARRIER();
    float ss = 0.f;
    for (int c = lane; c < dv; c += WAVE) ss = fmaf(o_s[c], o_s[c], ss);
    const float f = 1.0f / sqrtf(wave_sum(ss) / (float)dv + a.eps);
    bf16_t* out = (bf16_t*)a.out + ((size_t)t * a.H + h) * dv;
    if (tid < dv) out[tid] = (bf16_t)(o_s[tid] * f * weight * act_silu(to_f(gate)));
    for (int c = tid + blockDim.x; c < dv; c += blockDim.x)
      out[c] = (bf16_t)(o_s[c] * f * load_dyn(a.norm_w, a.norm_dtype, c) * act_silu(to_f(row[a.col_g + h * dv + c])));
    if (t + 1 < t0 + n) LDS_BARRIER();          // (the next token's q, k, gates and outputs overwrite what this one read)
  }
}

// The threads of delta_step_kernel for a head of these sizes, 0 where it does not take them.
static int step_threads(int dpad, int dv, int cols) {
  const int lanes = dpad / 4, threads = (lanes * ((dv + cols - 1) / cols) + WAVE - 1) / WAVE * WAVE;
  return lanes <= WAVE && threads <= STEP_THREADS ? threads : 0;
}
extern "C" int ifx_delta_step_takes(int dpad, int dv) { return dpad >= 4 && step_threads(dpad, dv, 8) > 0 ? 1 : 0; }

// ifx_delta_rule for steps of single tokens in bfloat16 (T <= R).  taps 4: u is the convolution's input, with conv_w [2 G d + H dv][4] (G == H), and
// a slot's row begins with its state; taps 0: u is its output.  dpad: a column of S.
extern "C" int ifx_delta_step(const void* u, int ldu, const void* conv_w, int conv_dtype, int taps, const void* rows, int ldr, int col_g, int col_b,
                              int col_a, const float* A_log, const float* dt_bias, const void* norm_w, int norm_dtype, float eps, float* state,
                              long long state_stride, long long state_offset, const int* q_start, const int* q_len, const int* slots, void* out,
                              int T, int R, int H, int G, int d, int dv, int dpad, void* stream) {
  IFX_REQUIRE(T >= 0 && R >= T && H > 0 && G > 0 && H % G == 0 && d > 0 && dv > 0, "delta_step: bad sizes T=%d R=%d H=%d G=%d d=%d dv=%d", T, R, H, G, d, dv);
  IFX_REQUIRE(dpad >= d && (dpad & (dpad - 1)) == 0 && ifx_delta_step_takes(dpad, dv), "delta_step: heads of %d (%d) x %d", d, dpad, dv);
  IFX_REQUIRE(taps == 0 || (taps == 4 && G == H && conv_w && state_offset >= (long long)3 * (2 * G * d + H * dv)), "delta_step: a convolution of %d taps (4, every head its own q and k)", taps);
  IFX_REQUIRE((uintptr_t)conv_w % 16 == 0, "delta_step: the convolution's weight must start on 16 bytes");
  IFX_REQUIRE(conv_dtype == DT_F32 || conv_dtype == DT_BF16, "delta_step: unknown weight dtype %d", conv_dtype);
  IFX_REQUIRE(ldu >= 2 * G * d + H * dv && col_g >= 0 && col_b >= 0 && col_a >= 0 && col_g + H * dv <= ldr && col_b + H <= ldr && col_a + H <= ldr, "delta_step: rows too narrow");
  IFX_REQUIRE(state_offset % 4 == 0 && state_stride % 4 == 0 && state_stride >= state_offset + (long long)H * dv * dpad, "delta_step: S must lie on 16 bytes within a row of %lld floats", state_stride);
  IFX_REQUIRE(R <= 65535, "delta_step: too many requests for one launch");
  if (R == 0 || T == 0) return 0;
  DeltaArgs a{u, ldu, rows, ldr, col_g, col_b, col_a, A_log, dt_bias, norm_w, norm_dtype, eps, state, (size_t)state_stride,
              (size_t)state_offset, q_start, q_len, slots, out, nullptr, T, H, G, d, dv, dpad / 4, 0};
  const StepConv conv{conv_w, conv_dtype, state};
  const int cols = step_threads(dpad, dv, 4) > 0 ? 4 : 8, threads = step_threads(dpad, dv, cols);
  const size_t lds_bytes = (size_t)(2 * dpad + dv) * sizeof(float);
  hipStream_t s = (hipStream_t)stream;
#define STEP(TAPS, COLS) hipLaunchKernelGGL((delta_step_kernel<TAPS, COLS>), dim3(H, R), dim3(threads), lds_bytes, s, a, conv)
  if (taps && cols == 4) STEP(4, 4);
  else if (taps) STEP(4, 8);
  else if (cols == 4) STEP(0, 4);
  else STEP(0, 8);
#undef STEP
  IFX_LAUNCH_CHECK();
}

extern "C" int ifx_delta_rule(const void* u, int ldu, const void* rows, int ldr, int col_g, int col_b, int col_a, int dtype,
                              const float* A_log, const float* dt_bias, const void* norm_w, int norm_dtype, float eps, float* state,
                              long long state_stride, long long state_offset, const int* q_start, const int* q_len, const int* slots,
                              void* out, float* o_raw, int T, int R, int H, int G, int d, int dv, int ch, int ks, int cols, void* stream) {
  IFX_REQUIRE(R >= 0 && H > 0 && G > 0 && H % G == 0 && d > 0 && dv > 0, "delta_rule: bad sizes R=%d H=%d G=%d d=%d dv=%d", R, H, G, d, dv);
  IFX_REQUIRE(ks > 0 && ks <= WAVE && (ks & (ks - 1)) == 0, "delta_rule: %d threads to a column (a power of two up to %d)", ks, WAVE);
  IFX_REQUIRE(ch * ks >= d && ch * ks <= MAX_DPAD, "delta_rule: %d x %d channels for heads of %d (at most %d)", ch, ks, d, MAX_DPAD);
  IFX_REQUIRE(cols > 0 && cols <= MAX_COLS && cols * ks <= 256, "delta_rule: %d columns x %d threads do not fit a workgroup of 256", cols, ks);
  IFX_REQUIRE(STAGE * ch * ks <= MAX_PRE * 64 * ((cols * ks + 63) / 64) && STAGE * cols <= MAX_PRE_V * 64 * ((cols * ks + 63) / 64),
              "delta_rule: a stage of %d x %d channels and %d columns is more than its %d threads fetch", STAGE, ch * ks, cols, cols * ks);
  IFX_REQUIRE(T >= 0 && o_raw, "delta_rule: the read-outs need a place");
  IFX_REQUIRE(ldu >= 2 * G * d + H * dv && col_g >= 0 && col_b >= 0 && col_a >= 0, "delta_rule: rows too narrow");
  IFX_REQUIRE(state_stride >= state_offset + (long long)H * dv * ch * ks, "delta_rule: a state row of %lld floats is too short", state_stride);
  IFX_REQUIRE(R <= 65535, "delta_rule: too many requests for one launch");
  if (R == 0) return 0;
  DeltaArgs a{u, ldu, rows, ldr, col_g, col_b, col_a, A_log, dt_bias, norm_w, norm_dtype, eps, state, (size_t)state_stride,
              (size_t)state_offset, q_start, q_len, slots, out, o_raw, T, H, G, d, dv, ks, cols};
  const int threads = (cols * ks + WAVE - 1) / WAVE * WAVE;
  const dim3 grid(H * ((dv + cols - 1) / cols), R);
  hipStream_t s = (hipStream_t)stream;
  const size_t lds_bytes = ((size_t)2 * STAGE * (ch * ks + cols) + ch * ks) * sizeof(float);      // (+ a row: the walk reads a token ahead)
#define LAUNCH(TY, C) hipLaunchKernelGGL((delta_kernel<TY, C>), grid, dim3(threads), lds_bytes, s, a)
#define BY_CH(TY)                                             \
  do {                                                        \
    if (ch == 4) LAUNCH(TY, 4);                               \
    else if (ch == 8) LAUNCH(TY, 8);                          \
    else if (ch == 16) LAUNCH(TY, 16);                        \
    else if (ch == 32) LAUNCH(TY, 32);                        \
    else if (ch == 64) LAUNCH(TY, 64);                        \
    else IFX_FAIL("delta_rule: %d channels a thread (4, 8, 16, 32 or 64)", ch); \
  } while (0)
  if (dtype == DT_F32) BY_CH(float);
  else if (dtype == DT_BF16) BY_CH(bf16_t);
  else IFX_FAIL("delta_rule: unknown dtype %d", dtype);
#undef BY_CH
#undef LAUNCH
  if (T > 0) {
    const unsigned blocks = (unsigned)(((size_t)T * H + 256 / WAVE - 1) / (256 / WAVE));
    if (dtype == DT_F32) hipLaunchKernelGGL(delta_finish_kernel<float>, dim3(blocks), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(delta_finish_kernel<bf16_t>, dim3(blocks), dim3(256), 0, s, a);
  }
  IFX_LAUNCH_CHECK();
}
