// Matrix memory with exponential gates: a recurrence per head whose state is a matrix S [d, dv] and a normaliser n [d], both
// decayed and written with one number per token and kept relative to exp(m), m the running maximum of the exponents.
//
// For a request's tokens t = 0, 1, ... and each head:
//
//   i = cap tanh((i_in + i_bias) / cap),  f = log sigmoid(cap tanh((f_in + f_bias) / cap))
//   m_t = max(f + m_(t-1), i),  m_(-1) = 0;  keep = exp(f + m_(t-1) - m_t),  write = exp(i - m_t)
//   S <- keep S + write k v^T;  n <- keep n + write k;  o = S^T q * q_scale / (max(|n . q * q_scale|, exp(-m_t)) + 1e-6)
//   out = o / sqrt(mean(o^2) + eps) * w_norm * sigmoid(gate_in)         (the norm over the head's dv values)
//
// q, k, v and gate_in are columns of projected rows [T, ld] (float or bfloat16), i_in and f_in columns of float rows.  Gates,
// m, S, n, every sum, the norm and the gate are float whatever those types are.
//
// The normaliser is one more column of S: column dv, whose value is 1 for every token.  A request's state is one float row:
// m [H, padded to a multiple of 4], then S laid out [head][column 0 .. dv][d_pad], d_pad = CH * KS >= d (padding stays zero).
// The columns of S never meet, so a head's columns are dealt to several workgroups of ``cols`` columns each.  In a workgroup
// thread (column, run) holds CH consecutive key channels of its column in registers; the KS threads of a column are
// neighbouring lanes and add their parts of S^T q in a fixed order.  Tokens are taken a stage of STAGE (fewer for wide heads) at a time: all threads load the
// stage's q, k and their columns of v into LDS, one wave forms the gates and the running maximum of the stage (the maximum
// as a scan over its lanes: m after a token is max(m + F, M) of the composed pairs (F, M)), everybody walks the tokens.  Read-outs
// go to ``o_raw`` [T, H, dv] and, of the normaliser's column, ``nq`` [T, H] (float); a second kernel, a wave per (token, head),
// divides, norms and gates them, and writes a request's last m into its state (the walk's workgroups all read the old one).
//
// Long portions in bfloat16 are cut into chunks of 64 tokens that run side by side on the matrix cores.  With F the sum of f
// from a chunk's start and m0 the maximum before the chunk, for tokens s <= t of a chunk
//   o_t = exp(F_t + m0 - m_t) S0^T q_t + sum_s exp(F_t - F_s + i_s - m_t) (q_t . k_s) v_s          (every exponent is <= 0)
//   S_end = exp(F_L + m0 - m_L) S0 + sum_s exp(F_L - F_s + i_s - m_L) k_s v_s^T
// in four launches: the gates and maxima of all tokens (exact for the whole portion, so nothing is ever rescaled), each chunk's
// own sum of outer products, the walk over a request's chunks that leaves S0 of every chunk, and the read-outs, which finish
// heads of up to CJ values themselves (the second kernel above does it for wider ones).  q, k and v are the projections' bfloat16 numbers as they are; what is float on the way into a product (S0,
// the weighted keys, the weighted scores) goes in as two bfloat16 numbers, the rounded one and the rest, so that nothing of
// the recurrence is rounded to 16 bits.  The normaliser's sums are plain float.
#include "common.h"
#include "lane_sums.h"
#include "chunk_tiles.h"

IFX_DEFINE_LAST_ERROR()

#define STAGE 16

struct MemoryArgs {
  const void* rows; int ld, q_col, k_col, v_col, g_col;
  const float* gates; int ldg, i_col, f_col;
  const float* i_bias; const float* f_bias; float cap, q_scale;
  const float* norm_w; float eps;              // [H dv]
  float* state; size_t state_stride; int s_off;
  const int* q_start; const int* q_len; const int* slots; const int* row_req;
  float* o_raw;        // [T, H, dv]
  float* nq;           // [T, H]: n . q * q_scale
  float* floor;        // [T, H]: exp(-m_t)
  float* m_end;        // [R, H], or null: the state's maxima are up to date
  void* out;           // [T, H dv]
  int T, R, H, d, dv, KS, cols, stage;      // stage: tokens taken at a time (at most STAGE)
};

__device__ __forceinline__ float log_sigmoid(float x) {      // -softplus(-x), without overflow
  return x >= 0.f ? -log1pf(expf(-x)) : x - log1pf(expf(x));
}
__device__ __forceinline__ float soft_cap(float x, float cap) { return cap * tanhf(x / cap); }

template <typename TI, int CH>
__global__ __launch_bounds__(256) void memory_walk_kernel(MemoryArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // q and k of a stage [STAGE][dpad] each, then its v [STAGE][cols]
  __shared__ float keep_s[STAGE], write_s[STAGE];
  const int n_cols = a.dv + 1, n_cb = (n_cols + a.cols - 1) / a.cols;
  const int h = blockIdx.x / n_cb, cb = blockIdx.x % n_cb, j0 = cb * a.cols, r = blockIdx.y;
  const int n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r], d = a.d, KS = a.KS, dpad = CH * KS;
  const int cols = min(a.cols, n_cols - j0);
  const int stage = a.stage;
  float* q_s = lds;
  float* k_s = lds + stage * dpad;
  float* v_s = lds + 2 * stage * dpad;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid % WAVE;
  const int jl = tid / KS, s = tid % KS;
  const bool owner = jl < cols;
  float* row = a.state + (size_t)a.slots[r] * a.state_stride;
  float* Sp = row + a.s_off + ((size_t)h * n_cols + j0 + (owner ? jl : 0)) * dpad + s * CH;
  float S[CH];
#pragma unroll
  for (int c = 0; c < CH; c += 4) {
    const float4 v = owner ? *(const float4*)(Sp + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    S[c] = v.x; S[c + 1] = v.y; S[c + 2] = v.z; S[c + 3] = v.w;
  }
  float m = row[h];                    // (kept by the first wave)
  const float ib = a.i_bias[h], fb = a.f_bias[h];
  const TI* rows = (const TI*)a.rows;
  const LaneSteps steps = lane_steps(KS);
  const int dshift = __ffs(dpad) - 1;
  for (int base = 0; base < n; base += stage) {
    const int cnt = min(stage, n - base);
    if (tid < WAVE) {
      // the stage's gates, a token a lane, and the running maximum as a scan of the pairs (F: sum of f, M: the best exponent)
      const bool in = lane < cnt;
      const size_t t = (size_t)(t0 + base + (in ? lane : 0));
      const float li = in ? soft_cap(a.gates[t * a.ldg + a.i_col + h] + ib, a.cap) : -INFINITY;
      const float lf = in ? log_sigmoid(soft_cap(a.gates[t * a.ldg + a.f_col + h] + fb, a.cap)) : 0.f;
      float F = lf, M = li;
#pragma unroll
      for (int o = 1; o < STAGE; o <<= 1) {
        const float Fp = __shfl_up(F, o, WAVE), Mp = __shfl_up(M, o, WAVE);
        if (lane >= o) { M = fmaxf(Mp + F, M); F += Fp; }
      }
      const float mt = fmaxf(m + F, M);
      const float up = __shfl_up(mt, 1, WAVE);
      const float before = lane == 0 ? m : up;
      if (in) {
        keep_s[lane] = expf(lf + before - mt);
        write_s[lane] = expf(li - mt);
        if (cb == 0) a.floor[t * a.H + h] = expf(-mt);
      }
      m = __shfl(mt, cnt - 1, WAVE);
    }
    for (int x = tid; x < cnt * dpad; x += nthr) {
      const int tt = x >> dshift, c = x & (dpad - 1);
      const size_t at = (size_t)(t0 + base + tt) * a.ld + (size_t)h * d + c;
      q_s[x] = c < d ? to_f(rows[at + a.q_col]) * a.q_scale : 0.f;
      k_s[x] = c < d ? to_f(rows[at + a.k_col]) : 0.f;
    }
    for (int x = tid; x < cnt * cols; x += nthr) {
      const int tt = x / cols, c = x - tt * cols;
      v_s[tt * a.cols + c] = j0 + c < a.dv ? to_f(rows[(size_t)(t0 + base + tt) * a.ld + a.v_col + (size_t)h * a.dv + j0 + c]) : 1.f;
    }
    __syncthreads();
    if (owner) {
      for (int tt = 0; tt < cnt; ++tt) {
        const float keep = keep_s[tt], wv = write_s[tt] * v_s[tt * a.cols + jl];
        const float* kp = k_s + tt * dpad + s * CH;
        const float* qp = q_s + tt * dpad + s * CH;
        float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          S[c] = fmaf(kp[c], wv, keep * S[c]);
          o4[c & 3] = fmaf(S[c], qp[c], o4[c & 3]);
        }
        const float o = column_sum((o4[0] + o4[1]) + (o4[2] + o4[3]), steps);
        const size_t item = (size_t)(t0 + base + tt) * a.H + h;
        if (s == 0) {
          if (j0 + jl < a.dv) a.o_raw[item * a.dv + j0 + jl] = o;
          else a.nq[item] = o;
        }
      }
    }
    __syncthreads();
  }
  if (owner) {
#pragma unroll
    for (int c = 0; c < CH; c += 4) *(float4*)(Sp + c) = make_float4(S[c], S[c + 1], S[c + 2], S[c + 3]);
  }
  if (cb == 0 && tid == 0) a.m_end[(size_t)r * a.H + h] = m;
}

// A wave per (token, head): o = o_raw / (max(|n . q|, exp(-m)) + 1e-6), its norm, the weight and the gate.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void memory_finish_kernel(MemoryArgs a) {
  const size_t item = (size_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  const int lane = threadIdx.x % WAVE;
  if (item >= (size_t)a.T * a.H) return;
  const size_t t = item / a.H;
  const int h = (int)(item % a.H), dv = a.dv;
  const float* o = a.o_raw + item * dv;
  const float inv_den = 1.0f / (fmaxf(fabsf(a.nq[item]), a.floor[item]) + 1e-6f);
  float ss = 0.f;
  for (int c = lane; c < dv; c += WAVE) { const float v = o[c] * inv_den; ss = fmaf(v, v, ss); }
  const float f = inv_den / sqrtf(wave_sum(ss) / (float)dv + a.eps);
  const TI* rows = (const TI*)a.rows;
  for (int c = lane; c < dv; c += WAVE) {
    const float g = to_f(rows[t * a.ld + a.g_col + (size_t)h * dv + c]);
    ((TO*)a.out)[item * dv + c] = from_f<TO>(o[c] * f * a.norm_w[(size_t)h * dv + c] / (1.0f + expf(-g)));
  }
  if (!a.m_end) return;
  const int r = a.row_req[t];
  if (lane == 0 && (int)t == a.q_start[r] + a.q_len[r] - 1)
    a.state[(size_t)a.slots[r] * a.state_stride + h] = a.m_end[(size_t)r * a.H + h];
}

// Steps of single tokens (a request's tokens one after the other where it has more): a workgroup takes all columns of a (request, head), so that the gates
// are formed once a head, the normaliser and the norm are there with the outputs, and nothing goes through memory to a second launch.  Bound by S,
// which is read and written once, and for few requests by a trip to memory and the arithmetic behind it.  A thread has V runs of four channels (two where
// a column has more than 256) of COLS columns, the threads of a column neighbours: a wave's load is 1 KB of contiguous memory; the normaliser's column
// is the first such threads' own.  q, k, v and the gates are formed once and meet in LDS; every load goes out before any is used, without branches
// between them, so that what meets there is waited for while S is on its way.  16 heads of 64 x 128, us with 16 channels of one column to a thread / 4
// columns / 8 columns, at 1, 16, 24, 32, 48 requests: 5.0 / 4.9, 7.3 / 7.3, 11.0 / 8.8, 12.0 / 9.7, 16.8 / 13.6, and at 64 22.3 / 18.1 / 16.9 (67 MB of S).
// A small head's columns are short waits one after the other, and two to a thread end sooner: us by four / two, 16 x 32 of 8 (request, head) pairs 4.7 / 4.3, of 16 x 128 and
// 160 5.4 / 5.1, 32 x 128 and 96 5.6 / 5.1, 32 x 32 and 896 (by eight) 6.9 / 5.5, 64 x 64 and 16 5.3 / 4.7, 128 x 32 and 160 6.0 / 5.3, but 64 x 128 and 64 5.4 / 5.6, and 656 12.9 / 16.5.
#define STEP_SMALL_HEAD 4096     // numbers of S up to which a thread takes two columns
#define STEP_MANY_HEADS 768      // (request, head) pairs beyond which eight columns, in four waves, are the better choice
template <typename TI, typename TO, int V, int COLS>
__global__ __launch_bounds__(1024) void memory_step_kernel(MemoryArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // q and k of a token [dpad] each, its values, in whose place its outputs [dv + 1]
  __shared__ float gate_s[3];                                       // keep, write, exp(-m)
  const int h = blockIdx.x, r = blockIdx.y, n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r], d = a.d, dv = a.dv, KS = a.KS, dpad = 4 * V * KS, groups = blockDim.x / KS;
  float *q_s = lds, *k_s = lds + dpad, *o_s = lds + 2 * dpad;
  const int tid = threadIdx.x, lane = tid % WAVE, s = tid % KS, j0 = tid / KS;      // column i of the thread: j0 + groups i
  float* row = a.state + (size_t)a.slots[r] * a.state_stride;
  float* Sp = row + a.s_off + (size_t)h * (dv + 1) * dpad;      // (the same for all threads: a thread's places are 32-bit offsets from it)
  const unsigned own = 4 * s, my_channel = min(tid, d - 1), my_value = min(tid, dv - 1);
  const LaneSteps steps = lane_steps(KS);
  float m = row[h];
  const float ib = a.i_bias[h], fb = a.f_bias[h];
  for (int t = t0; t < t0 + n; ++t) {
    const TI* x = (const TI*)a.rows + (size_t)t * a.ld;
    const TI *q_t = x + a.q_col + (size_t)h * d, *k_t = x + a.k_col + (size_t)h * d, *v_t = x + a.v_col + (size_t)h * dv, *g_t = x + a.g_col + (size_t)h * dv;
    const float* gates = a.gates + (size_t)t * a.ldg;
    const float zi = gates[a.i_col + h], zf = gates[a.f_col + h];
    const TI q0 = q_t[my_channel], k0 = k_t[my_channel], v0 = v_t[my_value];
    float4 S[COLS][V], N[V];      // (a token's own: where a request has several, a thread reads again what it has written)
#pragma unroll
    for (int i = 0; i < COLS; ++i)
#pragma unroll
      for (int u = 0; u < V; ++u) S[i][u] = *(const float4*)(Sp + (own + (unsigned)(min(j0 + groups * i, dv - 1) * dpad + 4 * KS * u)));
#pragma unroll
    for (int u = 0; u < V; ++u) N[u] = *(const float4*)(Sp + (own + (unsigned)(dv * dpad + 4 * KS * u)));
    const TI g = g_t[my_value];
    const float weight = a.norm_w[(size_t)h * dv + my_value];
    for (int c = tid; c < dpad; c += blockDim.x) {
      q_s[c] = c < d ? to_f(c == tid ? q0 : q_t[c]) * a.q_scale : 0.f;
      k_s[c] = c < d ? to_f(c == tid ? k0 : k_t[c]) : 0.f;
    }
    // (a column's value is read by its lanes, which are of one wave, before one of them writes the output in its place)
    if (tid < dv) o_s[tid] = to_f(v0);
    for (int c = tid + blockDim.x; c < dv; c += blockDim.x) o_s[c] = to_f(v_t[c]);
    const float li = soft_cap(zi + ib, a.cap), lf = log_sigmoid(soft_cap(zf + fb, a.cap)), mt = fmaxf(m + lf, li);
    if (tid < WAVE) {                  // (the first wave, which alone keeps m)
      if (lane == 0) { gate_s[0] = expf(lf + m - mt); gate_s[1] = expf(li - mt); gate_s[2] = expf(-mt); }
      m = mt;
    }
    LDS_BARRIER();
    const float keep = gate_s[0], write = gate_s[1], floor = gate_s[2];
    float4 q[V], k[V];
#pragma unroll
    for (int u = 0; u < V; ++u) { q[u] = *(const float4*)(q_s + own + 4 * KS * u); k[u] = *(const float4*)(k_s + own + 4 * KS * u); }
    auto column = [&](float4 (&S4)[V], float wv, unsigned at, bool held) {
      float o = 0.f;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        S4[u].x = fmaf(k[u].x, wv, keep * S4[u].x);
        S4[u].y = fmaf(k[u].y, wv, keep * S4[u].y);
        S4[u].z = fmaf(k[u].z, wv, keep * S4[u].z);
        S4[u].w = fmaf(k[u].w, wv, keep * S4[u].w);
        if (held) *(float4*)(Sp + (own + at + 4 * KS * u)) = S4[u];
        o += (S4[u].x * q[u].x + S4[u].y * q[u].y) + (S4[u].z * q[u].z + S4[u].w * q[u].w);
      }
      return column_sum(o, steps);
    };
#pragma unroll
    for (int i = 0; i < COLS; ++i) {
      const int j = j0 + groups * i;
      const float o = column(S[i], write * o_s[min(j, dv - 1)], (unsigned)(j * dpad), j < dv);
      if (s == 0 && j < dv) o_s[j] = o;
    }
    if (tid < WAVE) {                  // the normaliser's column, of value 1
      const float o = column(N, write, (unsigned)(dv * dpad), tid < KS);
      if (tid == 0) o_s[dv] = o;
    }
    LDS_BARRIER();
    const float inv_den = 1.0f / (fmaxf(fabsf(o_s[dv]), floor) + 1e-6f);      // (as memory_finish_kernel)
    float ss = 0.f;
    for (int c = lane; c < dv; c += WAVE) { const float w = o_s[c] * inv_den; ss = fmaf(w, w, ss); }
    const float f = inv_den / sqrtf(wave_sum(ss) / (float)dv + a.eps);
    TO* out = (TO*)a.out + ((size_t)t * a.H + h) * dv;
    if (tid < dv) out[tid] = from_f<TO>(o_s[tid] * f * weight / (1.0f + expf(-to_f(g))));
    for (int c = tid + blockDim.x; c < dv; c += blockDim.x)
      out[c] = from_f<TO>(o_s[c] * f * a.norm_w[(size_t)h * dv + c] / (1.0f + expf(-to_f(g_t[c]))));
    if (t + 1 < t0 + n) LDS_BARRIER();          // (the next token's q, k, gates and outputs overwrite what this one read)
  }
  if (tid == 0) row[h] = m;
}

// ---------------------------------------------------------------------------------------
struct ChunkArgs {
  MemoryArgs a;
  const int* chunk_req; const int* chunk_t0; const int* chunk_len; const int* req_chunk0;
  float* cum_f; float* log_i; float* m;        // [H, T]: sum of f from the token's chunk's start, i, the maximum after the token
  float* m0;           // [n_chunks, H]: the maximum before the chunk
  float* keep;         // [n_chunks, H]: exp(F_L + m0 - m_L)
  float* chunk_state;  // [n_chunks, H, dv + 1, dpad]
  int n_chunks, dpad;
};

// A workgroup per (request, head), a chunk a wave and a token a lane: the waves scan their chunks side by side, the chunks' sums
// meet in LDS, and every wave walks those before its own for the maximum its chunk starts from.
#define GATE_WAVES 16
__global__ __launch_bounds__(GATE_WAVES * WAVE) void memory_gates_kernel(ChunkArgs c) {
  const MemoryArgs& a = c.a;
  __shared__ float sum_f[2][GATE_WAVES], best[2][GATE_WAVES];      // two sets in turns: one barrier a round is enough
  const int h = blockIdx.x, r = blockIdx.y, lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  const int n = a.q_len[r];
  if (n <= 0) return;
  const int t0 = a.q_start[r], c0 = c.req_chunk0[r];
  float* m_state = a.state + (size_t)a.slots[r] * a.state_stride + h;
  float m = *m_state;                  // the maximum before the round's first chunk, the same in every wave
  const float ib = a.i_bias[h], fb = a.f_bias[h];
  for (int base = 0, round = 0; base < n; base += nw * CL, ++round) {
    const int at0 = base + wid * CL, cnt = min(CL, n - at0);        // (a wave behind the last chunk has none: cnt <= 0)
    const bool in = lane < cnt;
    const float* g = a.gates + (size_t)(t0 + (in ? at0 + lane : 0)) * a.ldg;
    const float li = in ? soft_cap(g[a.i_col + h] + ib, a.cap) : -INFINITY;
    const float lf = in ? log_sigmoid(soft_cap(g[a.f_col + h] + fb, a.cap)) : 0.f;
    float F = lf, M = li;
#pragma unroll
    for (int o = 1; o < CL; o <<= 1) {
      const float Fp = __shfl_up(F, o, WAVE), Mp = __shfl_up(M, o, WAVE);
      if (lane >= o) { M = fmaxf(Mp + F, M); F += Fp; }
    }
    float (&sf)[GATE_WAVES] = sum_f[round & 1], (&sb)[GATE_WAVES] = best[round & 1];
    if (lane == WAVE - 1) { sf[wid] = F; sb[wid] = M; }              // (lanes behind the chunk's end add nothing)
    __syncthreads();
    float m_here = m;
    for (int w = 0; w < nw; ++w) {
      if (w == wid) m_here = m;
      m = fmaxf(m + sf[w], sb[w]);                                   // (a wave without tokens: m + 0 against -inf)
    }
    if (cnt <= 0) continue;
    const float mt = fmaxf(m_here + F, M);
    if (in) {
      const size_t at = (size_t)h * a.T + t0 + at0 + lane;
      c.cum_f[at] = F; c.log_i[at] = li; c.m[at] = mt;
      a.floor[(size_t)(t0 + at0 + lane) * a.H + h] = expf(-mt);
    }
    if (lane == cnt - 1) {
      const size_t at = (size_t)(c0 + round * nw + wid) * a.H + h;
      c.m0[at] = m_here;
      c.keep[at] = expf(F + m_here - mt);
    }
  }
  if (threadIdx.x == 0) *m_state = m;
}

// A chunk's own sum: chunk_state[chunk][h][j][i] = sum_s w_s k_s[i] v_s[j], w_s = exp(F_L - F_s + i_s - m_L), for CJ columns and CI
// channels; the workgroups of the first columns form the normaliser's column too.
__global__ __launch_bounds__(256) void memory_chunk_sums_kernel(ChunkArgs c) {
  const MemoryArgs& a = c.a;
  __shared__ __attribute__((aligned(16))) bf16_t vt[CJ][CLP];
  __shared__ __attribute__((aligned(16))) bf16_t kh[CI][CLP];
  __shared__ __attribute__((aligned(16))) bf16_t kl[CI][CLP];
  __shared__ float wt[CL];
  const int n_jb = (a.dv + CJ - 1) / CJ;
  const int chunk = blockIdx.x, h = blockIdx.y, j0 = (blockIdx.z % n_jb) * CJ, i0 = (blockIdx.z / n_jb) * CI;
  const int t0 = c.chunk_t0[chunk], len = c.chunk_len[chunk], tid = threadIdx.x;
  if (tid < CL) {
    const float* F = c.cum_f + (size_t)h * a.T + t0;
    wt[tid] = tid < len ? expf(F[len - 1] - F[tid] + c.log_i[(size_t)h * a.T + t0 + tid] - c.m[(size_t)h * a.T + t0 + len - 1]) : 0.f;
  }
  stage_columns((const bf16_t*)a.rows, a.ld, a.v_col + h * a.dv, a.dv, j0, CJ, t0, len, vt);
  __syncthreads();
  const bf16_t* rows = (const bf16_t*)a.rows;
  for (int x = tid; x < (CL / 2) * (CI / 8); x += 256) {        // the keys, weighted, in two parts each
    const int p = x % (CL / 2), g = x / (CL / 2), s = 2 * p, i = i0 + 8 * g;
    const bf16_t* src = rows + (size_t)(t0 + s) * a.ld + a.k_col + h * a.d + i;
    const bf16x8 u = (s < len && i < a.d) ? *(const bf16x8*)src : zero8();
    const bf16x8 v = (s + 1 < len && i < a.d) ? *(const bf16x8*)(src + a.ld) : zero8();
    const float w0 = wt[s], w1 = wt[s + 1];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x0 = (float)u[e] * w0, x1 = (float)v[e] * w1;
      const bf16x2 hi = bf16x2{(__bf16)x0, (__bf16)x1};
      *(bf16x2*)&kh[8 * g + e][s] = hi;
      *(bf16x2*)&kl[8 * g + e][s] = bf16x2{(__bf16)(x0 - (float)hi[0]), (__bf16)(x1 - (float)hi[1])};
    }
  }
  __syncthreads();
  float* out = c.chunk_state + ((size_t)chunk * a.H + h) * (a.dv + 1) * c.dpad;
  if (j0 == 0 && tid < CI && i0 + tid < c.dpad) {
    float n = 0.f;
    for (int s = 0; s < CL; ++s) n += (float)kh[tid][s] + (float)kl[tid][s];
    out[(size_t)a.dv * c.dpad + i0 + tid] = n;
  }
  const int wave = tid / WAVE, lane = tid % WAVE, l32 = lane & 31, hi = lane >> 5;
  const int j = j0 + 32 * wave + l32;
  if (j0 + 32 * wave >= a.dv) return;
  floatx16 acc[CI / 32];
#pragma unroll
  for (int it = 0; it < CI / 32; ++it)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[it][e] = 0.f;
#pragma unroll
  for (int ks = 0; ks < CL / 16; ++ks) {
    const bf16x8 b = *(const bf16x8*)&vt[32 * wave + l32][16 * ks + 8 * hi];
#pragma unroll
    for (int it = 0; it < CI / 32; ++it) {
      const bf16x8 ah = *(const bf16x8*)&kh[32 * it + l32][16 * ks + 8 * hi], al = *(const bf16x8*)&kl[32 * it + l32][16 * ks + 8 * hi];
      acc[it] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, b, acc[it], 0, 0, 0);
      acc[it] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, b, acc[it], 0, 0, 0);
    }
  }
  if (j >= a.dv) return;
#pragma unroll
  for (int it = 0; it < CI / 32; ++it)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + 32 * it + 8 * q + 4 * hi;
      if (i < c.dpad) *(float4*)(out + (size_t)j * c.dpad + i) = make_float4(acc[it][4 * q], acc[it][4 * q + 1], acc[it][4 * q + 2], acc[it][4 * q + 3]);
    }
}

// Four numbers of a request's S a thread (see walk_chunks).
__global__ __launch_bounds__(WALK_THREADS) void memory_combine_kernel(ChunkArgs c) {
  const MemoryArgs& a = c.a;
  const size_t per = (size_t)a.H * (a.dv + 1) * c.dpad;
  const size_t e = ((size_t)blockIdx.x * WALK_THREADS + threadIdx.x) * 4;
  if (e >= per) return;
  const int r = blockIdx.y;
  const int h = (int)(e / ((size_t)(a.dv + 1) * c.dpad));
  walk_chunks((float4*)(a.state + (size_t)a.slots[r] * a.state_stride + a.s_off + e), c.chunk_state + e, per, c.req_chunk0[r],
              c.req_chunk0[r + 1], [&](int k) { return c.keep[(size_t)k * a.H + h]; });
}

// The read-outs of a chunk's tokens for CJ columns of a head.  FINISH (dv <= CJ): the head's norm, weight and gate as well, from
// the read-outs in LDS; else they go to o_raw and nq.
#define OTP (CJ + 4)         // a token's read-outs in LDS
template <typename TO, bool FINISH>
__global__ __launch_bounds__(256) void memory_chunk_out_kernel(ChunkArgs c) {
  const MemoryArgs& a = c.a;
  __shared__ __attribute__((aligned(16))) union {
    struct { bf16_t vt[CJ][CLP], ph[CL][CLP], pl[CL][CLP]; } w;
    float ot[CL][OTP];
  } pool;
  bf16_t (&vt)[CJ][CLP] = pool.w.vt;
  bf16_t (&ph)[CL][CLP] = pool.w.ph;
  bf16_t (&pl)[CL][CLP] = pool.w.pl;
  __shared__ float Fs[CL], is[CL], ms[CL], row_sum[2][CL], inv_den[CL];
  const int chunk = blockIdx.x, h = blockIdx.y, j0 = blockIdx.z * CJ;
  const int t0 = c.chunk_t0[chunk], len = c.chunk_len[chunk], tid = threadIdx.x, d = a.d;
  const int wave = tid / WAVE, lane = tid % WAVE, l32 = lane & 31, hi = lane >> 5;
  const bf16_t* rows = (const bf16_t*)a.rows;
  const bf16_t* qb = rows + (size_t)t0 * a.ld + a.q_col + h * d;
  const bf16_t* kb = rows + (size_t)t0 * a.ld + a.k_col + h * d;
  const float m0 = c.m0[(size_t)chunk * a.H + h];
  if (tid < CL) {
    const size_t at = (size_t)h * a.T + t0 + min(tid, len - 1);
    Fs[tid] = c.cum_f[at]; is[tid] = c.log_i[at]; ms[tid] = c.m[at];
  }
  stage_columns((const bf16_t*)a.rows, a.ld, a.v_col + h * a.dv, a.dv, j0, CJ, t0, len, vt);
  auto load_row = [&](const bf16_t* base, int row, int k) { return (row < len && k < d) ? *(const bf16x8*)(base + (size_t)row * a.ld + k) : zero8(); };
  // scores, transposed: wave (wt, ws) forms the 32 keys 32 ws ... against the 32 queries 32 wt ...
  const int wt = wave & 1, ws = wave >> 1;
  floatx16 sc;
#pragma unroll
  for (int e = 0; e < 16; ++e) sc[e] = 0.f;
  if (ws <= wt)          // (keys behind all of the tile's queries weigh nothing)
    for (int k = 8 * hi; k < d + 8 * hi; k += 16) {
      const bf16x8 kk = load_row(kb, 32 * ws + l32, k), qq = load_row(qb, 32 * wt + l32, k);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk, qq, sc, 0, 0, 0);
    }
  __syncthreads();
  {
    const int t = 32 * wt + l32;
    const float Ft = Fs[t], mt = ms[t];
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bf16x4 yh, yl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int s = 32 * ws + 8 * q + 4 * hi + e;
        const float p = (s <= t && t < len) ? sc[4 * q + e] * a.q_scale * expf(Ft - Fs[s] + is[s] - mt) : 0.f;
        sum += p;
        yh[e] = (__bf16)p;
        yl[e] = (__bf16)(p - (float)yh[e]);
      }
      *(bf16x4*)&ph[t][32 * ws + 8 * q + 4 * hi] = yh;
      *(bf16x4*)&pl[t][32 * ws + 8 * q + 4 * hi] = yl;
    }
    sum += __shfl_xor(sum, 32, WAVE);
    if (hi == 0) row_sum[ws][t] = sum;
  }
  __syncthreads();
  const float* S0 = c.chunk_state + ((size_t)chunk * a.H + h) * (a.dv + 1) * c.dpad;
  if (blockIdx.z == 0) {          // the normaliser: four threads a token
    const int t = tid >> 2, part = tid & 3;
    float nq = 0.f;
    if (t < len)
      for (int i = part; i < d; i += 4) nq = fmaf((float)qb[(size_t)t * a.ld + i], S0[(size_t)a.dv * c.dpad + i], nq);
    nq += __shfl_xor(nq, 1, WAVE);
    nq += __shfl_xor(nq, 2, WAVE);
    nq = nq * a.q_scale * expf(Fs[t] + m0 - ms[t]) + row_sum[0][t] + row_sum[1][t];
    if (FINISH) { if (part == 0) inv_den[t] = 1.0f / (fmaxf(fabsf(nq), expf(-ms[t])) + 1e-6f); }
    else if (part == 0 && t < len) a.nq[(size_t)(t0 + t) * a.H + h] = nq;
  }
  const int j = j0 + 32 * wave + l32;
  const bool mine = j0 + 32 * wave < a.dv;         // (the same for the whole wave)
  if (!FINISH && !mine) return;
  floatx16 acc[2];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[tt][e] = 0.f;
  // what the chunk starts from: S0's rows are asked for as floats and go in as two bfloat16 numbers
  const float* Srow = S0 + (size_t)min(j, a.dv - 1) * c.dpad;
  const int d_here = mine ? d : 0;
  for (int k = 8 * hi; k < d_here + 8 * hi; k += 16) {
    bf16x8 sh = zero8(), sl = zero8();
    if (k < d) {
      const float4 x = *(const float4*)(Srow + k), y = *(const float4*)(Srow + k + 4);
      const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) { sh[e] = (__bf16)f[e]; sl[e] = (__bf16)(f[e] - (float)sh[e]); }
    }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const bf16x8 qq = load_row(qb, 32 * tt + l32, k);
      acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sh, qq, acc[tt], 0, 0, 0);
      acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sl, qq, acc[tt], 0, 0, 0);
    }
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = 32 * tt + l32;
    const float f = a.q_scale * expf(Fs[t] + m0 - ms[t]);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[tt][e] *= f;
  }
#pragma unroll
  for (int ks = 0; ks < CL / 16; ++ks) {
    const bf16x8 v = *(const bf16x8*)&vt[32 * wave + l32][16 * ks + 8 * hi];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      if (16 * ks >= 32 * (tt + 1)) continue;        // (keys behind all of the tile's queries)
      const bf16x8 bh = *(const bf16x8*)&ph[32 * tt + l32][16 * ks + 8 * hi], bl = *(const bf16x8*)&pl[32 * tt + l32][16 * ks + 8 * hi];
      acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, bh, acc[tt], 0, 0, 0);
      acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, bl, acc[tt], 0, 0, 0);
    }
  }
  // acc[tt][e]: column j0 + 32 wave + 8 (e / 4) + 4 hi + e % 4 of token 32 tt + l32 (dv is a multiple of 8: runs of four are whole)
  if (FINISH) {
    __syncthreads();             // everyone is done with the columns and the weighted scores: the read-outs take their place
    if (mine)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(float4*)&pool.ot[32 * tt + l32][32 * wave + 8 * q + 4 * hi] =
              make_float4(acc[tt][4 * q], acc[tt][4 * q + 1], acc[tt][4 * q + 2], acc[tt][4 * q + 3]);
    __syncthreads();
    // four threads a token, each every fourth run of eight columns
    const int t = tid >> 2, part = tid & 3;
    const float* o = pool.ot[t];
    const float id = inv_den[t];
    float ss = 0.f;
    for (int g = 8 * part; g < a.dv; g += 32)
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float v = o[g + e] * id; ss = fmaf(v, v, ss); }
    ss += __shfl_xor(ss, 1, WAVE);
    ss += __shfl_xor(ss, 2, WAVE);
    if (t >= len) return;
    const float f = id / sqrtf(ss / (float)a.dv + a.eps);
    const size_t row = (size_t)(t0 + t);
    for (int g = 8 * part; g < a.dv; g += 32) {
      const bf16x8 gate = *(const bf16x8*)(rows + row * a.ld + a.g_col + (size_t)h * a.dv + g);
      const float* w = a.norm_w + (size_t)h * a.dv + g;
      TO* out = (TO*)a.out + (row * a.H + h) * a.dv + g;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = o[g + e] * f * w[e] / (1.0f + expf(-(float)gate[e]));
      if (sizeof(TO) == 2) {
        bf16x8 z;
#pragma unroll
        for (int e = 0; e < 8; ++e) z[e] = (__bf16)y[e];
        *(bf16x8*)out = z;
      } else {
        *(float4*)out = make_float4(y[0], y[1], y[2], y[3]);
        *(float4*)((float*)out + 4) = make_float4(y[4], y[5], y[6], y[7]);
      }
    }
    return;
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = 32 * tt + l32;
    if (t >= len) continue;
    float* o = a.o_raw + ((size_t)(t0 + t) * a.H + h) * a.dv;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int jj = j0 + 32 * wave + 8 * q + 4 * hi;
      if (jj < a.dv) *(float4*)(o + jj) = make_float4(acc[tt][4 * q], acc[tt][4 * q + 1], acc[tt][4 * q + 2], acc[tt][4 * q + 3]);
    }
  }
}

extern "C" int ifx_matrix_memory(const void* rows, int dtype, int ld, int q_col, int k_col, int v_col, int g_col, const float* gates, int ldg,
                                 int i_col, int f_col, const float* i_bias, const float* f_bias, float cap, float q_scale,
                                 const float* norm_w, float eps, float* state, long long state_stride, int s_off, const int* q_start,
                                 const int* q_len, const int* slots, const int* row_req, float* o_raw, float* nq, float* floor_, float* m_end,
                                 void* out, int out_dtype, int T, int R, int H, int d, int dv, int ch, int ks, int cols, int n_chunks,
                                 const int* chunk_req, const int* chunk_t0, const int* chunk_len, const int* req_chunk0, float* token_gates,
                                 float* chunk_gates, float* chunk_state, void* stream) {
  IFX_REQUIRE(T >= 0 && R >= 0 && H > 0 && d > 0 && dv > 0 && cap > 0.f, "matrix_memory: bad sizes T=%d R=%d H=%d d=%d dv=%d", T, R, H, d, dv);
  IFX_REQUIRE(ks > 0 && ks <= WAVE && (ks & (ks - 1)) == 0 && ch * ks >= d, "matrix_memory: %d threads of %d channels for heads of %d", ks, ch, d);
  IFX_REQUIRE(cols > 0 && cols * ks <= 256, "matrix_memory: %d columns x %d threads do not fit a workgroup of 256", cols, ks);
  IFX_REQUIRE(s_off >= H && s_off % 4 == 0 && state_stride % 4 == 0, "matrix_memory: S must lie at a multiple of 16 bytes behind the maxima");
  IFX_REQUIRE(state_stride >= s_off + (long long)H * (dv + 1) * ch * ks, "matrix_memory: a state row of %lld floats is too short", state_stride);
  IFX_REQUIRE(R <= 65535, "matrix_memory: too many requests for one launch");
  int stage = STAGE;
  while (stage > 4 && (size_t)stage * (2 * ch * ks + cols) * sizeof(float) > 60 * 1024) stage /= 2;
  const size_t lds = (size_t)stage * (2 * ch * ks + cols) * sizeof(float);
  IFX_REQUIRE(lds <= 60 * 1024, "matrix_memory: d=%d needs more LDS than a workgroup has", d);
  if (T == 0 || R == 0) return 0;
  MemoryArgs a{rows, ld, q_col, k_col, v_col, g_col, gates, ldg, i_col, f_col, i_bias, f_bias, cap, q_scale, norm_w, eps, state,
               (size_t)state_stride, s_off, q_start, q_len, slots, row_req, o_raw, nq, floor_, m_end, out, T, R, H, d, dv, ks, cols, stage};
  const dim3 grid(H * ((dv + cols) / cols), R);        // (dv + 1 columns)
  const int threads = (cols * ks + WAVE - 1) / WAVE * WAVE;
  const unsigned blocks = (unsigned)(((size_t)T * H + 256 / WAVE - 1) / (256 / WAVE));
  hipStream_t s = (hipStream_t)stream;
  if (n_chunks > 0) {
    IFX_REQUIRE(dtype == DT_BF16 && d % 8 == 0 && dv % 8 == 0 && ld % 8 == 0 && q_col % 8 == 0 && k_col % 8 == 0 && v_col % 8 == 0,
                "matrix_memory: chunks take bfloat16 rows whose heads (d=%d, dv=%d) and columns are multiples of 8", d, dv);
    IFX_REQUIRE(chunk_req && chunk_t0 && chunk_len && req_chunk0 && token_gates && chunk_gates && chunk_state, "matrix_memory: chunks without their lists");
    a.m_end = nullptr;           // (the gates' kernel writes the maxima back itself)
    const size_t HT = (size_t)H * T;
    const ChunkArgs c{a, chunk_req, chunk_t0, chunk_len, req_chunk0, token_gates, token_gates + HT, token_gates + 2 * HT, chunk_gates,
                      chunk_gates + (size_t)n_chunks * H, chunk_state, n_chunks, ch * ks};
    const int jb = (dv + CJ - 1) / CJ, ib = (ch * ks + CI - 1) / CI;
    const size_t per4 = (size_t)H * (dv + 1) * ch * ks / 4;
    const int gate_waves = min(GATE_WAVES, max(1, n_chunks - R + 1));        // (no request has more chunks than this)
    hipLaunchKernelGGL(memory_gates_kernel, dim3(H, R), dim3(gate_waves * WAVE), 0, s, c);
    hipLaunchKernelGGL(memory_chunk_sums_kernel, dim3(n_chunks, H, jb * ib), dim3(256), 0, s, c);
    hipLaunchKernelGGL(memory_combine_kernel, dim3((unsigned)((per4 + WALK_THREADS - 1) / WALK_THREADS), R), dim3(WALK_THREADS), 0, s, c);
    if (dv <= CJ && g_col % 8 == 0) {
      if (out_dtype == DT_BF16) hipLaunchKernelGGL((memory_chunk_out_kernel<bf16_t, true>), dim3(n_chunks, H, 1), dim3(256), 0, s, c);
      else hipLaunchKernelGGL((memory_chunk_out_kernel<float, true>), dim3(n_chunks, H, 1), dim3(256), 0, s, c);
      IFX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL((memory_chunk_out_kernel<float, false>), dim3(n_chunks, H, jb), dim3(256), 0, s, c);
    if (out_dtype == DT_BF16) hipLaunchKernelGGL((memory_finish_kernel<bf16_t, bf16_t>), dim3(blocks), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((memory_finish_kernel<bf16_t, float>), dim3(blocks), dim3(256), 0, s, a);
    IFX_LAUNCH_CHECK();
  }
  const int dpad = ch * ks, runs = dpad > 4 * WAVE ? 2 : 1, lanes = dpad / 4 / runs;
  const auto threads_of = [&](int cols_) { return (lanes * ((dv + cols_ - 1) / cols_) + WAVE - 1) / WAVE * WAVE; };
  const bool four = runs > 1 || (threads_of(4) <= 1024 && (long long)H * R <= STEP_MANY_HEADS) || threads_of(8) > 1024;
  const bool two = runs == 1 && dpad * dv <= STEP_SMALL_HEAD;
  const int step_threads = threads_of(two ? 2 : four ? 4 : 8);
  if (T <= R && lanes >= 4 && lanes <= WAVE && step_threads <= 1024) {
    a.KS = lanes;
    const size_t step_lds = (size_t)(2 * dpad + dv + 1) * sizeof(float);
    const dim3 step_grid(H, R);
#define STEP(TI, TO)                                                                                                             \
  do {                                                                                                                           \
    if (runs > 1) hipLaunchKernelGGL((memory_step_kernel<TI, TO, 2, 4>), step_grid, dim3(step_threads), step_lds, s, a);         \
    else if (two) hipLaunchKernelGGL((memory_step_kernel<TI, TO, 1, 2>), step_grid, dim3(step_threads), step_lds, s, a);         \
    else if (four) hipLaunchKernelGGL((memory_step_kernel<TI, TO, 1, 4>), step_grid, dim3(step_threads), step_lds, s, a);        \
    else hipLaunchKernelGGL((memory_step_kernel<TI, TO, 1, 8>), step_grid, dim3(step_threads), step_lds, s, a);                  \
  } while (0)
    if (dtype == DT_F32 && out_dtype == DT_F32) STEP(float, float);
    else if (dtype == DT_F32 && out_dtype == DT_BF16) STEP(float, bf16_t);
    else if (dtype == DT_BF16 && out_dtype == DT_BF16) STEP(bf16_t, bf16_t);
    else IFX_FAIL("matrix_memory: unsupported types rows=%d out=%d", dtype, out_dtype);
#undef STEP
    IFX_LAUNCH_CHECK();
  }
#define WALK(TY, C) hipLaunchKernelGGL((memory_walk_kernel<TY, C>), grid, dim3(threads), lds, s, a)
#define BY_CH(TY)                       \
  do {                                  \
    if (ch == 4) WALK(TY, 4);           \
    else if (ch == 8) WALK(TY, 8);      \
    else if (ch == 16) WALK(TY, 16);    \
    else if (ch == 32) WALK(TY, 32);    \
    else IFX_FAIL("matrix_memory: %d channels a thread (4, 8, 16 or 32)", ch); \
  } while (0)
  if (dtype == DT_F32) BY_CH(float);
  else if (dtype == DT_BF16) BY_CH(bf16_t);
  else IFX_FAIL("matrix_memory: unknown dtype %d", dtype);
#undef BY_CH
#undef WALK
#define FINISH(TI, TO) hipLaunchKernelGGL((memory_finish_kernel<TI, TO>), dim3(blocks), dim3(256), 0, s, a)
  if (dtype == DT_F32 && out_dtype == DT_F32) FINISH(float, float);
  else if (dtype == DT_F32 && out_dtype == DT_BF16) FINISH(float, bf16_t);
  else if (dtype == DT_BF16 && out_dtype == DT_BF16) FINISH(bf16_t, bf16_t);
  else IFX_FAIL("matrix_memory: unsupported types rows=%d out=%d", dtype, out_dtype);
#undef FINISH
  IFX_LAUNCH_CHECK();
}
