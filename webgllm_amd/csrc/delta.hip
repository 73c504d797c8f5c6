// Gated DeltaNet, the linear-attention layers of Qwen3.5 (the reference's
// Engine.linearAttend, src/engine.ts:6646-6825, and its lin* passes,
// src/gpu/kernels.ts:1544-1862; the math in src/delta-rule.ts:38-62).
//
// Per head h, with q^ and k^ the row's q and k over their L2 norms (q^ also
// over sqrt(dk)), beta = sigmoid(b) and a = exp(A softplus(a_in + dt_bias)):
//   d = beta (v - a S^T k^),  S <- a S + k^ d^T,  o = a S^T q^ + (q^.k^) d.
//
// `delta_rule_kernel` runs the gates, the q/k prep and the recurrence of a
// batch of rows in one launch (LIN_GATES + LIN_PREP + LIN_DELTA + LIN_STATE
// per token, or LIN_DELTA_FUSED at one). The columns of a head's state are
// independent given q^, k^ and the gates, so a workgroup takes one head and
// CB state columns (16 for short batches, 64 for long ones), and the 512 / CB
// threads of a column split its dk rows: each thread keeps its rows' state
// values in registers for the whole batch, so the state is read and written
// once a launch, whatever the row count. Per row, two barriers that wait on
// LDS only: one after q, k and the gates are in LDS, one after the partial
// S^T k^ and S^T q^ are; the next row's inputs load across them.
#include <type_traits>

#include "common.h"
#include "epilogue.h"

namespace wg {
namespace {

constexpr int DW = 8;        // waves a recurrence workgroup
constexpr int MAX_DK = 256;  // key dims a head (DW * 32 rows)
constexpr int MAX_CONV = 16; // convolution taps

struct DeltaArgs {
  const float *qkv;  // [M][ldq]: q (H dk) | k (H dk) | v (H dv)
  int ldq;
  const float *ba;  // [M][ldba]: b (H) | a (H)
  int ldba;
  const float *A, *dt;  // [H]
  int H, dk, dv, M;
  float *state;  // [H][dk][dv]
  float *snap;   // the state after row save_at, or null
  int save_at;
  float *out;  // [M][ldo]: H dv
  int ldo;
};


// A workgroup barrier that waits for this wave's LDS operations only: the
// next row's global loads, issued before it, stay in flight across it.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One row's inputs for this thread: q[t], k[t] (threads t < MAX_DK), v at
// this thread's column, b and a of the head (thread MAX_DK).
struct RowIn {
  float q, k, v, b, a;
};

__device__ inline RowIn load_row(const DeltaArgs &a, int m, int h, int j, bool col) {
  const float *row = a.qkv + (int64_t)m * a.ldq;
  const int t = threadIdx.x, K = a.H * a.dk;
  RowIn r{0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (t < a.dk) {
    r.q = row[h * a.dk + t];
    r.k = row[K + h * a.dk + t];
  } else if (t == MAX_DK) {
    const float *g = a.ba + (int64_t)m * a.ldba;
    r.b = g[h];
    r.a = g[a.H + h];
  }
  if (col) r.v = row[2 * K + h * a.dv + j];
  return r;
}

// CB state columns a workgroup, one a thread; the 512 / CB threads of a
// column split its dk rows, ROWS each.
template <int ROWS, int CB>
__global__ __launch_bounds__(64 * DW) void delta_rule_kernel(DeltaArgs a) {
  constexpr int RG = 64 * DW / CB;  // row groups
  static_assert(ROWS * RG <= MAX_DK, "rows a thread");
  // By row parity, so a row's writes never meet the previous row's reads.
  __shared__ float qn[2][MAX_DK], kn[2][MAX_DK];  // raw q, k (0 past dk)
  __shared__ float part[2][3][4];                 // sums of q^2, k^2, q k per wave
  __shared__ float gate[2][2];                    // beta, decay
  __shared__ float redk[2][DW][CB], redq[2][DW][CB];
  const int h = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = threadIdx.x % CB, rg = threadIdx.x / CB;
  const int j = blockIdx.x * CB + c;
  const bool col = j < a.dv;
  const int i0 = rg * ROWS;
  const float scale = 1.0f / sqrtf((float)a.dk);
  float *Sh = a.state + (int64_t)h * a.dk * a.dv;
  float s[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; r++)
    s[r] = col && i0 + r < a.dk ? Sh[(int64_t)(i0 + r) * a.dv + j] : 0.0f;
  RowIn in = load_row(a, 0, h, j, col);
  for (int m = 0; m < a.M; m++) {
    const int p = m & 1;
    const int t = threadIdx.x;
    if (t < MAX_DK) {  // waves 0-3: the head's q and k, their squares and products
      qn[p][t] = in.q;
      kn[p][t] = in.k;
      const float x0 = wave_sum(in.q * in.q), x1 = wave_sum(in.k * in.k);
      const float x2 = wave_sum(in.q * in.k);
      if (lane == 0) {
        part[p][0][w] = x0;
        part[p][1][w] = x1;
        part[p][2][w] = x2;
      }
    } else if (t == MAX_DK) {  // LIN_GATES for this head
      const float x = in.a + a.dt[h];
      const float softplus = fmaxf(x, 0.0f) + log1pf(expf(-fabsf(x)));
      gate[p][0] = 1.0f / (1.0f + expf(-in.b));
      gate[p][1] = expf(a.A[h] * softplus);
    }
    const float vj = in.v;
    if (m + 1 < a.M) in = load_row(a, m + 1, h, j, col);
    lds_barrier();
    const float sq = part[p][0][0] + part[p][0][1] + part[p][0][2] + part[p][0][3];
    const float sk = part[p][1][0] + part[p][1][1] + part[p][1][2] + part[p][1][3];
    const float sqk = part[p][2][0] + part[p][2][1] + part[p][2][2] + part[p][2][3];
    const float invq = scale / sqrtf(sq + 1e-6f), invk = 1.0f / sqrtf(sk + 1e-6f);
    float pk = 0.0f, pq = 0.0f;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      pk = fmaf(s[r], kn[p][i0 + r], pk);
      pq = fmaf(s[r], qn[p][i0 + r], pq);
    }
    if constexpr (CB < 64) {  // the wave's row groups of this column
      pk = group_reduce<CB>(pk, Plus());
      pq = group_reduce<CB>(pq, Plus());
    }
    if (lane < CB) {
      redk[p][w][c] = pk * invk;
      redq[p][w][c] = pq * invq;
    }
    lds_barrier();
    float kvs = 0.0f, qss = 0.0f;
#pragma unroll
    for (int u = 0; u < DW; u++) {
      kvs += redk[p][u][c];
      qss += redq[p][u][c];
    }
    const float beta = gate[p][0], decay = gate[p][1];
    const float d = beta * (vj - decay * kvs);
    if (rg == 0 && col)
      a.out[(int64_t)m * a.ldo + h * a.dv + j] = decay * qss + sqk * invq * invk * d;
#pragma unroll
    for (int r = 0; r < ROWS; r++) s[r] = fmaf(decay, s[r], kn[p][i0 + r] * invk * d);
    if (a.snap && m + 1 == a.save_at && col) {
      float *Sn = a.snap + (int64_t)h * a.dk * a.dv;
#pragma unroll
      for (int r = 0; r < ROWS; r++)
        if (i0 + r < a.dk) Sn[(int64_t)(i0 + r) * a.dv + j] = s[r];
    }
  }
  if (col) {
#pragma unroll
    for (int r = 0; r < ROWS; r++)
      if (i0 + r < a.dk) Sh[(int64_t)(i0 + r) * a.dv + j] = s[r];
  }
}

template <int CB>
void launch_delta_rule(const DeltaArgs &a, hipStream_t s) {
  constexpr int RG = 64 * DW / CB;
  const dim3 grid((a.dv + CB - 1) / CB, a.H);
  const int rows = (a.dk + RG - 1) / RG;
  if (rows <= 1 && RG <= MAX_DK)
    delta_rule_kernel<1, CB><<<grid, 64 * DW, 0, s>>>(a);
  else if (rows <= 2 && 2 * RG <= MAX_DK)
    delta_rule_kernel<(2 * RG <= MAX_DK ? 2 : 1), CB><<<grid, 64 * DW, 0, s>>>(a);
  else if (rows <= 4 && 4 * RG <= MAX_DK)
    delta_rule_kernel<(4 * RG <= MAX_DK ? 4 : 1), CB><<<grid, 64 * DW, 0, s>>>(a);
  else if (rows <= 8 && 8 * RG <= MAX_DK)
    delta_rule_kernel<(8 * RG <= MAX_DK ? 8 : 1), CB><<<grid, 64 * DW, 0, s>>>(a);
  else if (rows <= 16 && 16 * RG <= MAX_DK)
    delta_rule_kernel<(16 * RG <= MAX_DK ? 16 : 1), CB><<<grid, 64 * DW, 0, s>>>(a);
  else
    delta_rule_kernel<(32 * RG <= MAX_DK ? 32 : 1), CB><<<grid, 64 * DW, 0, s>>>(a);
}

// LIN_CONV + LIN_CONV_STATE: a thread per output (row, channel), then per
// state (row, channel).
__global__ __launch_bounds__(256) void delta_conv_kernel(const float *in, int ldi, int M, int C,
                                                         int W, const float *taps,
                                                         const float *state, float *state_out,
                                                         float *out, int ldo) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)(M + W - 1) * C) return;
  const int m = (int)(idx / C), c = (int)(idx % C);
  if (m < M) {
    float x[MAX_CONV];
    for (int k = 0; k < W; k++) {
      const int t = m - (W - 1) + k;
      x[k] = t >= 0 ? in[(int64_t)t * ldi + c] : state[(int64_t)(W - 1 + t) * C + c];
    }
    float acc = 0.0f;
    for (int k = 0; k < W; k++) acc = fmaf(taps[(int64_t)c * W + k], x[k], acc);
    out[(int64_t)m * ldo + c] = acc / (1.0f + expf(-acc));
  } else {
    const int i = m - M, t = M - (W - 1) + i;
    state_out[(int64_t)i * C + c] =
        t >= 0 ? in[(int64_t)t * ldi + c] : state[(int64_t)(M + i) * C + c];
  }
}

// The same of prompt batches: a thread takes 4 channels of CONV_ROWS rows,
// its window of rows loaded once into registers (11 16-byte loads for 8
// outputs). Bound by memory: 1500 x 6144 (74 MB in and out) took 54 us with
// a thread an output, 16 us now (4.6 TB/s). Channels and strides are multiples of 4,
// the arrays 16-byte aligned.
constexpr int CONV_ROWS = 8;
// Fewer outputs wait on memory round trips, which 32 times the threads hide
// better (a graph of them, us, a thread an output / 8 rows of 4: 24 rows of
// 6144 3.5 / 4.9, 41 3.9 / 4.6, 65 4.55 / 4.57, 98 5.7 / 4.7; 146 of 1024
// 3.4 / 4.4, 391 4.6 / 4.6, 781 6.7 / 4.8).
constexpr int CONV_ROWS_MIN = 400000;

template <int W>
__global__ __launch_bounds__(256) void delta_conv_rows_kernel(const float *in, int ldi, int M,
                                                              int C, const float *taps,
                                                              const float *state,
                                                              float *state_out, float *out,
                                                              int ldo) {
  const int c = 4 * (int)(blockIdx.x * 256 + threadIdx.x), m0 = (int)blockIdx.y * CONV_ROWS;
  if (c >= C) return;
  // row t of the stream: the state's rows come before row 0
  auto row = [&](int t) {
    return *reinterpret_cast<const float4 *>(t >= 0 ? in + (int64_t)t * ldi + c
                                                    : state + (int64_t)(W - 1 + t) * C + c);
  };
  float4 x[CONV_ROWS + W - 1];
#pragma unroll
  for (int k = 0; k < CONV_ROWS + W - 1; k++)
    x[k] = row(min(m0 - (W - 1) + k, M - 1));
  float w[4][W];
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int k = 0; k < W; k++) w[q][k] = taps[(int64_t)(c + q) * W + k];
#pragma unroll
  for (int r = 0; r < CONV_ROWS; r++) {
    if (m0 + r >= M) break;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < W; k++) {
      const float4 v = x[r + k];
      acc[0] = fmaf(w[0][k], v.x, acc[0]);
      acc[1] = fmaf(w[1][k], v.y, acc[1]);
      acc[2] = fmaf(w[2][k], v.z, acc[2]);
      acc[3] = fmaf(w[3][k], v.w, acc[3]);
    }
    float4 o;
    o.x = acc[0] / (1.0f + expf(-acc[0]));
    o.y = acc[1] / (1.0f + expf(-acc[1]));
    o.z = acc[2] / (1.0f + expf(-acc[2]));
    o.w = acc[3] / (1.0f + expf(-acc[3]));
    *reinterpret_cast<float4 *>(out + (int64_t)(m0 + r) * ldo + c) = o;
  }
  if (m0 + CONV_ROWS >= M) {  // the last rows' thread: the new state
#pragma unroll
    for (int i = 0; i < W - 1; i++)
      *reinterpret_cast<float4 *>(state_out + (int64_t)i * C + c) = row(M - (W - 1) + i);
  }
}

// LIN_NORM: a wave per (row, head), up to 4 values a lane.
__global__ __launch_bounds__(256) void delta_norm_kernel(const float *o, int ldo, int M, int H,
                                                         int dv, const float *z, int ldz,
                                                         const float *wt, float eps,
                                                         uint16_t *out16, int ldh) {
  const int lane = threadIdx.x & 63;
  const int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wv >= (int64_t)M * H) return;
  const int m = (int)(wv / H), h = (int)(wv % H);
  const float *oh = o + (int64_t)m * ldo + h * dv;
  const float *zh = z + (int64_t)m * ldz + h * dv;
  float x[4], ss = 0.0f;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int i = lane + 64 * u;
    x[u] = i < dv ? oh[i] : 0.0f;
    ss = fmaf(x[u], x[u], ss);
  }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)dv + eps);
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int i = lane + 64 * u;
    if (i < dv) {
      const float zz = zh[i];
      out16[(int64_t)m * ldh + h * dv + i] =
          half_bits(x[u] * inv * wt[i] * (zz / (1.0f + expf(-zz))));
    }
  }
}

// ---------------------------------------------------- the chunked form
//
// deltaChunked (src/delta-rule.ts:73-166; the reference's linCum, linGram,
// linSolve, linUW, linQO, linChunkOut and linChunkState passes): rows in
// chunks of CH (a first chunk of `first` rows, so that one ends at a
// snapshot), G the running sum of the log-decays within a chunk:
//   A[r][s] = beta_r e^{G_r - G_s} k^_r.k^_s (s < r), T = (I + A)^-1,
//   U = T diag(beta) V, W = T diag(beta e^G) K^, P[r][s] = e^{G_r - G_s} q^_r.k^_s,
//   Oi = P U, Q' = e^G Q^ - P W, K~_s = e^{G_last - G_s} k^_s;
// then from each chunk's starting state S: D = U - W S, O = Oi + Q' S,
// S <- e^{G_last} S + K~^T D. `delta_chunk_prep_kernel` does the first
// part for every (head, chunk) at once; `delta_chunk_chain_kernel` the
// state chain, a workgroup per (head, 16 state columns).
//
// Every product runs on v_mfma_f32_16x16x4_f32 (float32 operands and sums,
// twice the vector units' rate). A 16 x 16 x 16 product is 4 of them, step j
// contracting k = 4 c + j for the lane groups c = lane / 16: an A operand is
// then 4 consecutive floats of a row (one 16-byte read), and a result's 4
// registers (rows 4 c .. 4 c + 3 of column lane % 16) are the next product's
// B operand as they stand. So the solve, P U and P W stay in a wave's
// registers, and prep writes each matrix in the order the chain's lanes read
// it: a fragment (16 x 16, 4 floats a lane) is 1 KB in one load.

constexpr int CH = 64;        // rows a chunk
constexpr int CT = CH / 16;   // its row tiles
constexpr int CMAX = 128;     // key and value dims the chunked form takes
constexpr int KTM = CMAX / 16;
constexpr int RS = CMAX + 4;  // LDS row stride (floats) of the row tiles: rows 4 banks apart
constexpr int AS = CH + 4;    // LDS row stride of A and P
constexpr int TS = 20;        // LDS row stride of the inverted diagonal blocks
constexpr int CW = 8;         // waves a workgroup
constexpr size_t PREP_LDS = (2 * CH * RS + 2 * CH * AS + CH * TS + 4 * CH + 4) * sizeof(float);
typedef float f4v __attribute__((ext_vector_type(4)));

struct ChunkArgs {
  const float *qkv;
  int ldq;
  const float *ba;
  int ldba;
  const float *A, *dt;
  int H, dk, dv, M, first, nch;
  // fragments (256 floats) a (head, chunk): U, Oi [dv tile][row tile] as
  // results; -W, Q' [row tile][dk tile] and K~^T [dk tile][row tile] as A
  // operands; eg [H][nch]
  float *U, *W, *Oi, *Qp, *Kt, *eg;
  float *state, *snap;
  int save_at;
  float *out;
  int ldo;
};

__device__ inline void chunk_rows(const ChunkArgs &a, int c, int &c0, int &n) {
  c0 = c == 0 ? 0 : a.first + (c - 1) * CH;
  n = min(c == 0 ? a.first : CH, a.M - c0);
}

// c + (16 x 16 A) (16 x 16 B)
__device__ __forceinline__ f4v mma16(f4v a, f4v b, f4v c) {
#pragma unroll
  for (int j = 0; j < 4; j++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  return c;
}

// (16 x 16 lower triangular m) b. CAREFUL: a value of b that is not finite
// is kept from the rows before its own, which m's zeros there times it would
// make NaN: those rows come from b without such values.
template <bool CAREFUL>
__device__ __forceinline__ f4v mma16_lower(f4v m, f4v b) {
  const f4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f4v r = mma16(m, b, zero);
  if constexpr (CAREFUL) {
    const int row = 4 * ((threadIdx.x & 63) >> 4);
    int first = 16;  // this column's first row that is not finite
#pragma unroll
    for (int e = 3; e >= 0; e--)
      if (!isfinite(b[e])) {
        b[e] = 0.0f;
        first = row + e;
      }
    first = min(first, __shfl_xor(first, 16, 64));
    first = min(first, __shfl_xor(first, 32, 64));
    const f4v f = mma16(m, b, zero);
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (row + e < first) r[e] = f[e];
  }
  return r;
}

// Bound by its phases in turn (loads, norms, products, solve, products), which
// the one workgroup that 108 KB of LDS leave a compute unit does not overlap:
// its 1920 MFMA are 6.4 us of the SIMDs, and 1500 rows of 16 heads (384
// workgroups, two rounds) take 46 us, MFMA busy 21%. As vector code (one wave
// a SIMD, T by a serial forward substitution of 64 rows) they took 141 us.
__global__ __launch_bounds__(64 * CW) void delta_chunk_prep_kernel(ChunkArgs a) {
  extern __shared__ __align__(16) float sm[];
  float *sq = sm, *sk = sq + CH * RS;            // q^, k^ rows (0 past n, dims); then Q', -W
  float *sA = sk + CH * RS, *sP = sA + CH * AS;  // -A and P
  float *sT = sP + CH * AS;                      // (I + A_ii)^-1 of the diagonal blocks
  float *sG = sT + CH * TS, *sB = sG + CH, *sE = sB + CH, *sL = sE + CH;  // G, beta, e^G, e^(Gl-G)
  float *sF = sL + CH;  // whether a gate or key is not finite
  const int c = blockIdx.x, h = blockIdx.y, t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ln = lane & 15, lg = lane >> 4;
  int c0, n;
  chunk_rows(a, c, c0, n);
  const int K = a.H * a.dk, dk = a.dk, dv = a.dv;
  const int KT = (dk + 15) / 16, VT = (dv + 15) / 16;
  // every load issued before the first store: thread t takes column t % 128
  // of rows 4 u + t / 128; a wave its 16 value columns (rows and columns past
  // the chunk read its last, without a branch, and become 0)
  f4v x[CT];  // this wave's value columns: rows 16 i + 4 lg + e, column 16 wave + ln
  {
    const int i = t & (CMAX - 1), r0 = t >> 7;
    float rq[CH / 4], rk[CH / 4];
#pragma unroll
    for (int u = 0; u < CH / 4; u++) {
      const int r = 4 * u + r0;
      const float *row = a.qkv + (int64_t)(c0 + min(r, n - 1)) * a.ldq;
      rq[u] = row[h * dk + min(i, dk - 1)];
      rk[u] = row[K + h * dk + min(i, dk - 1)];
    }
    const int vj = 16 * wave + ln;
#pragma unroll
    for (int i2 = 0; i2 < CT; i2++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = 16 * i2 + 4 * lg + e;
        x[i2][e] = a.qkv[(int64_t)(c0 + min(r, n - 1)) * a.ldq + 2 * K + h * dv + min(vj, dv - 1)];
      }
#pragma unroll
    for (int u = 0; u < CH / 4; u++) {
      const bool in = 4 * u + r0 < n && i < dk;
      sq[(4 * u + r0) * RS + i] = in ? rq[u] : 0.0f;
      sk[(4 * u + r0) * RS + i] = in ? rk[u] : 0.0f;
    }
#pragma unroll
    for (int i2 = 0; i2 < CT; i2++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (16 * i2 + 4 * lg + e >= n || vj >= dv) x[i2][e] = 0.0f;
  }
  if (t < CH) {  // wave 0: the gates (LIN_GATES) and G by a shuffle scan (linCum)
    float beta = 0.0f, g = 0.0f;
    if (t < n) {
      const float *gb = a.ba + (int64_t)(c0 + t) * a.ldba;
      const float y = gb[a.H + h] + a.dt[h];
      beta = 1.0f / (1.0f + expf(-gb[h]));
      g = a.A[h] * (fmaxf(y, 0.0f) + log1pf(expf(-fabsf(y))));
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float y = __shfl_up(g, off, 64);
      if (lane >= off) g += y;
    }
    const float gl = __shfl(g, n - 1, 64), eg = expf(g);
    const bool bad = __ballot(!isfinite(beta) || !isfinite(g) || !isfinite(eg)) != 0;
    sB[t] = beta;
    sG[t] = g;
    sE[t] = eg;
    sL[t] = expf(gl - g);
    if (t == 0) {
      a.eg[h * a.nch + c] = expf(gl);
      *sF = bad ? 1.0f : 0.0f;
    }
  }
  lds_barrier();
  {  // LIN_PREP: eight threads a row
    const int r = t >> 3, part = t & 7;
    float ssq = 0.0f, ssk = 0.0f;
    for (int i = part; i < dk; i += 8) {
      ssq = fmaf(sq[r * RS + i], sq[r * RS + i], ssq);
      ssk = fmaf(sk[r * RS + i], sk[r * RS + i], ssk);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
      ssq += __shfl_xor(ssq, off, 64);
      ssk += __shfl_xor(ssk, off, 64);
    }
    const float invq = 1.0f / sqrtf((float)dk) / sqrtf(ssq + 1e-6f);
    const float invk = 1.0f / sqrtf(ssk + 1e-6f);
    if (part == 0 && !isfinite(ssk)) *sF = 1.0f;
    for (int i = part; i < dk; i += 8) {
      sq[r * RS + i] *= invq;
      sk[r * RS + i] *= invk;
    }
  }
  lds_barrier();
  // linGram: the lower triangle's 10 tiles of K^ K^T and of Q^ K^T
  for (int job = wave; job < CT * (CT + 1); job += CW) {
    const int pair = job >> 1, which = job & 1;
    const int ti = pair < 1 ? 0 : pair < 3 ? 1 : pair < 6 ? 2 : 3;
    const int tj = pair - ti * (ti + 1) / 2;
    const float *ra = (which ? sq : sk) + (16 * ti + ln) * RS + 4 * lg;
    const float *rb = sk + (16 * tj + ln) * RS + 4 * lg;
    f4v g[4] = {};  // four chains of sums: shorter, and so closer to exact
#pragma unroll
    for (int s = 0; s < KTM; s++) {
      if (s >= KT) break;
      g[s & 3] = mma16(*reinterpret_cast<const f4v *>(ra + 16 * s),
                       *reinterpret_cast<const f4v *>(rb + 16 * s), g[s & 3]);
    }
    const f4v dots = (g[0] + g[1]) + (g[2] + g[3]);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 16 * ti + 4 * lg + e, s = 16 * tj + ln;
      const float d = dots[e];
      const bool ok = r < n && s <= r;
      const float ex = ok ? expf(sG[r] - sG[s]) : 0.0f;
      if (which) sP[r * AS + s] = ok ? ex * d : 0.0f;
      else sA[r * AS + s] = ok && s < r ? -(sB[r] * ex * d) : 0.0f;
    }
  }
  // K~^T as A operands: fragment (dk tile, row tile s), lane rows 16 s + 4 lg ..
  const int64_t hc = (int64_t)h * a.nch + c;
  if (wave < KT) {
#pragma unroll
    for (int s = 0; s < CT; s++) {
      f4v v;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = 16 * s + 4 * lg + e;
        v[e] = sL[r] * sk[r * RS + 16 * wave + ln];
      }
      *reinterpret_cast<f4v *>(a.Kt + ((hc * KT + wave) * CT + s) * 256 + 4 * lane) = v;
    }
  }
  lds_barrier();
  if (wave < CT && lane < 16) {  // linSolve: (I + A_ii)^-1, forward substitution, lane = column
    const float *Ai = sA + 16 * wave * AS + 16 * wave;  // (holds -A)
    float Tc[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      float acc[2] = {lane == r ? 1.0f : 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < r; s++) acc[s & 1] = fmaf(Ai[r * AS + s], Tc[s], acc[s & 1]);
      Tc[r] = acc[0] + acc[1];
    }
#pragma unroll
    for (int r = 0; r < 16; r++) sT[(16 * wave + r) * TS + lane] = Tc[r];
  }
  lds_barrier();
  // linUW by blocks: X_i = T_ii (R_i - sum_j<i A_ij X_j), this wave's value
  // columns (R = beta V) and key columns (R = beta e^G K^); then linQO: Oi =
  // P U, Q' = e^G Q^ + P (-W).
  const f4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f4v y[CT], qp[CT], o[CT], off = zero;
  auto solve = [&](auto careful) {
    constexpr bool CAREFUL = decltype(careful)::value;
#pragma unroll
    for (int i = 0; i < CT; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = 16 * i + 4 * lg + e;
        const float b = sB[r], ex = sE[r];
        x[i][e] *= b;
        y[i][e] = sk[r * RS + 16 * wave + ln] * (b * ex);
        qp[i][e] = sq[r * RS + 16 * wave + ln] * ex;
        if constexpr (!CAREFUL) off[e] = fmaf(x[i][e], 0.0f, off[e]);
      }
#pragma unroll
    for (int i = 0; i < CT; i++) {
#pragma unroll
      for (int j = 0; j < i; j++) {  // (each block's sum by itself, then added)
        const f4v m = *reinterpret_cast<const f4v *>(sA + (16 * i + ln) * AS + 16 * j + 4 * lg);
        x[i] += mma16(m, x[j], zero);
        y[i] += mma16(m, y[j], zero);
      }
      const f4v m = *reinterpret_cast<const f4v *>(sT + (16 * i + ln) * TS + 4 * lg);
      x[i] = mma16_lower<CAREFUL>(m, x[i]);
      y[i] = mma16_lower<CAREFUL>(m, y[i]);
    }
#pragma unroll
    for (int i = 0; i < CT; i++) y[i] = -y[i];
#pragma unroll
    for (int i = 0; i < CT; i++) {
      o[i] = zero;
#pragma unroll
      for (int j = 0; j <= i; j++) {
        const f4v m = *reinterpret_cast<const f4v *>(sP + (16 * i + ln) * AS + 16 * j + 4 * lg);
        o[i] += j < i ? mma16(m, x[j], zero) : mma16_lower<CAREFUL>(m, x[j]);
        qp[i] += j < i ? mma16(m, y[j], zero) : mma16_lower<CAREFUL>(m, y[j]);
      }
    }
  };
  solve(std::false_type{});
  // Where a value (off is NaN), a key or a gate is not finite: again, with the
  // rows before it kept from it.
  if (__builtin_expect(__ballot((off[0] + off[1]) + (off[2] + off[3]) + *sF != 0.0f) != 0, 0)) {
    // (none of the first loads' addresses and masks kept for these)
    const float *v = a.qkv + (int64_t)c0 * a.ldq + 2 * K + h * dv + 16 * wave + ln;
    int rows = 16 * wave + ln < dv ? n : 0;
    asm volatile("" : "+v"(v), "+v"(rows));
#pragma unroll
    for (int i = 0; i < CT; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = 16 * i + 4 * lg + e;
        x[i][e] = r < rows ? v[(int64_t)r * a.ldq] : 0.0f;
      }
    solve(std::true_type{});
  }
  if (wave < VT) {
#pragma unroll
    for (int i = 0; i < CT; i++) {
      const int64_t at = ((hc * VT + wave) * CT + i) * 256 + 4 * lane;
      *reinterpret_cast<f4v *>(a.U + at) = x[i];
      *reinterpret_cast<f4v *>(a.Oi + at) = o[i];
    }
  }
  lds_barrier();  // every read of q^ and k^ is done: Q' and -W take their places
#pragma unroll
  for (int i = 0; i < CT; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int at = (16 * i + 4 * lg + e) * RS + 16 * wave + ln;
      sk[at] = y[i][e];
      sq[at] = qp[i][e];
    }
  lds_barrier();
  if (wave < KT) {
#pragma unroll
    for (int i = 0; i < CT; i++) {
      const int from = (16 * i + ln) * RS + 16 * wave + 4 * lg;
      const int64_t at = ((hc * CT + i) * KT + wave) * 256 + 4 * lane;
      *reinterpret_cast<f4v *>(a.W + at) = *reinterpret_cast<const f4v *>(sk + from);
      *reinterpret_cast<f4v *>(a.Qp + at) = *reinterpret_cast<const f4v *>(sq + from);
    }
  }
}

// A chunk's fragments for one chain wave: its row tile of -W and U (waves 0
// to 3) or of Q' and Oi (4 to 7), its dk tile of K~^T, the decay.
struct ChainIn {
  f4v a[KTM], k[CT], u;
  float e;
};

// A workgroup per (head, 16 state columns): waves 0 to 3 a row tile of D
// each, 4 to 7 one of O, then every wave its 16 state rows. The state and D
// pass between the waves through LDS as fragments; the memory's come one
// chunk ahead. Bound by the chain of a chunk: 384 MFMA (1.3 us of 4 SIMDs) and
// two exchanges in 2.8 us, on one compute unit in two at 16 heads of 128 (MFMA
// busy 23% of them all, 46% of those in use). As vector code over LDS tiles a
// chunk took 7.6 us, 1500 rows 184 us; this takes 66 us.
__global__ __launch_bounds__(64 * CW) void delta_chunk_chain_kernel(ChunkArgs a) {
  __shared__ __align__(16) float sS[2][KTM][256], sD[CT][256];
  // blockIdx.x is the head: the workgroups of one head (consecutive in
  // blockIdx.y, H apart in launch order) land on one XCD, whose L2 then
  // serves the head's fragments to all of them.
  const int h = blockIdx.x, vt = blockIdx.y, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, lg = lane >> 4, jj = 16 * vt + ln;
  const int dk = a.dk, dv = a.dv, KT = (dk + 15) / 16, VT = (dv + 15) / 16;
  const bool col = jj < dv, low = wave < CT;
  const int tile = low ? wave : wave - CT;
  float *Sh = a.state + (int64_t)h * dk * dv + jj;
  f4v S;  // state rows 16 wave + 4 lg + e, column jj
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int i = 16 * wave + 4 * lg + e;
    S[e] = col && i < dk ? Sh[(int64_t)i * dv] : 0.0f;
  }
  *reinterpret_cast<f4v *>(&sS[0][wave][4 * lane]) = S;
  const float *A0 = low ? a.W : a.Qp, *U0 = low ? a.U : a.Oi;
  auto fetch = [&](ChainIn &f, int c) {
    const int64_t hc = (int64_t)h * a.nch + c;
    const float *pa = A0 + (hc * CT + tile) * KT * 256 + 4 * lane;
    const float *pk = a.Kt + (hc * KT + min(wave, KT - 1)) * CT * 256 + 4 * lane;
#pragma unroll
    for (int s = 0; s < KTM; s++)  // (tiles past dk: the last again, unused)
      f.a[s] = *reinterpret_cast<const f4v *>(pa + min(s, KT - 1) * 256);
    f.u = *reinterpret_cast<const f4v *>(U0 + ((hc * VT + vt) * CT + tile) * 256 + 4 * lane);
#pragma unroll
    for (int s = 0; s < CT; s++) f.k[s] = *reinterpret_cast<const f4v *>(pk + s * 256);
    f.e = a.eg[hc];
  };
  auto chunk = [&](const ChainIn &f, ChainIn &next, int c) {
    int c0, n;
    chunk_rows(a, c, c0, n);
    const int p = c & 1;
    fetch(next, min(c + 1, a.nch - 1));  // in flight while this chunk computes
    // linChunkOut: D = U - W S, O = Oi + Q' S
    f4v g[4] = {};  // four chains of sums: shorter, and so closer to exact
#pragma unroll
    for (int s = 0; s < KTM; s++) {
      if (s >= KT) break;
      const f4v b = *reinterpret_cast<const f4v *>(&sS[p][s][4 * lane]);
      g[s & 3] = mma16(f.a[s], b, g[s & 3]);
    }
    const f4v r0 = f.u + ((g[0] + g[1]) + (g[2] + g[3]));
    if (low) *reinterpret_cast<f4v *>(&sD[tile][4 * lane]) = r0;
    lds_barrier();
    // linChunkState: S <- e^{G_last} S + K~^T D
    f4v u[2] = {};
#pragma unroll
    for (int s = 0; s < CT; s++)
      u[s & 1] = mma16(f.k[s], *reinterpret_cast<const f4v *>(&sD[s][4 * lane]), u[s & 1]);
#pragma unroll
    for (int e = 0; e < 4; e++) S[e] = fmaf(f.e, S[e], u[0][e] + u[1][e]);
    if (wave >= KT) S = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    *reinterpret_cast<f4v *>(&sS[p ^ 1][wave][4 * lane]) = S;
    if (!low && col) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = 16 * tile + 4 * lg + e;
        if (r < n) a.out[(int64_t)(c0 + r) * a.ldo + h * dv + jj] = r0[e];
      }
    }
    if (a.snap && c0 + n == a.save_at && col) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i = 16 * wave + 4 * lg + e;
        if (i < dk) a.snap[(int64_t)h * dk * dv + (int64_t)i * dv + jj] = S[e];
      }
    }
    lds_barrier();
  };
  ChainIn f0, f1;
  fetch(f0, 0);
  lds_barrier();
  for (int c = 0; c < a.nch; c += 2) {
    chunk(f0, f1, c);
    if (c + 1 < a.nch) chunk(f1, f0, c + 1);
  }
  if (col) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = 16 * wave + 4 * lg + e;
      if (i < dk) Sh[(int64_t)i * dv] = S[e];
    }
  }
}

// Chunks of a batch of M rows whose first chunk has `first` rows.
inline int chunk_count(int M, int first) { return M <= first ? 1 : 1 + (M - first + CH - 1) / CH; }

// A chunk's fragments of `dim` columns, in floats.
inline size_t fragment_floats(int dim) { return (size_t)((dim + 15) / 16) * CT * 256; }

// The first chunk's rows: shorter, so that a chunk ends at save_at
// (Engine.recurrenceChunks' rule), else CH.
inline int first_rows(int save_at) { return save_at > 0 && save_at % CH ? save_at % CH : CH; }

}  // namespace
}  // namespace wg

using namespace wg;

extern "C" {

int wg_delta_rule(const float *qkv, int32_t M, int32_t ldq, const float *ba, int32_t ldba,
                  const float *A, const float *dt_bias, const wg_delta_shape *shape,
                  float *state, float *snapshot, int32_t save_at, float *out, int32_t ldo,
                  void *stream) {
  WG_REQUIRE(qkv && ba && A && dt_bias && shape && state && out && M >= 1,
             "wg_delta_rule: bad arguments");
  const int H = shape->heads, dk = shape->key_dim, dv = shape->value_dim;
  WG_REQUIRE(H >= 1 && dk >= 1 && dk <= MAX_DK && dv >= 1,
             "wg_delta_rule: %d heads of %d key and %d value dims (key dims 1 to %d)", H, dk,
             dv, MAX_DK);
  WG_REQUIRE(ldq >= 2 * H * dk + H * dv && ldba >= 2 * H && ldo >= H * dv,
             "wg_delta_rule: row strides too short for the heads");
  WG_REQUIRE(save_at >= 0 && save_at <= M && (save_at == 0 || snapshot),
             "wg_delta_rule: save_at %d of %d rows needs a snapshot buffer", save_at, M);
  const size_t state_bytes = (size_t)H * dk * dv * sizeof(float);
  WG_REQUIRE(!snapshot || !overlaps(snapshot, state_bytes, state, state_bytes),
             "wg_delta_rule: the snapshot overlaps the state");
  DeltaArgs a{qkv, ldq, ba, ldba, A, dt_bias, H, dk, dv, M, state, snapshot, save_at, out, ldo};
  // Short batches: 16 columns a workgroup (128 workgroups at 16 heads of
  // 128), so more CUs read the state; long ones: 64 (fewer shuffles a row).
  if (M <= tuning("delta_narrow_rows"))
    launch_delta_rule<16>(a, as_stream(stream));
  else
    launch_delta_rule<64>(a, as_stream(stream));
  return launched("wg_delta_rule");
}

size_t wg_delta_chunk_scratch_bytes(int32_t M, const wg_delta_shape *shape, int32_t save_at) {
  if (!shape || M < 1) return 0;
  const size_t nch = (size_t)chunk_count(M, first_rows(save_at));
  return sizeof(float) * (shape->heads * nch * (fragment_floats(shape->value_dim) * 2 +
                                                fragment_floats(shape->key_dim) * 3) +
                          shape->heads * nch);
}

int wg_delta_rule_chunked(const float *qkv, int32_t M, int32_t ldq, const float *ba,
                          int32_t ldba, const float *A, const float *dt_bias,
                          const wg_delta_shape *shape, float *state, float *snapshot,
                          int32_t save_at, float *out, int32_t ldo, void *scratch,
                          size_t scratch_bytes, void *stream) {
  WG_REQUIRE(qkv && ba && A && dt_bias && shape && state && out && scratch && M >= 1,
             "wg_delta_rule_chunked: bad arguments");
  const int H = shape->heads, dk = shape->key_dim, dv = shape->value_dim;
  WG_REQUIRE(H >= 1 && dk >= 4 && dk <= CMAX && dk % 4 == 0 && dv >= 1 && dv <= CMAX,
             "wg_delta_rule_chunked: %d key and %d value dims (key dims a multiple of 4, "
             "both at most %d)", dk, dv, CMAX);
  WG_REQUIRE(ldq >= 2 * H * dk + H * dv && ldba >= 2 * H && ldo >= H * dv,
             "wg_delta_rule_chunked: row strides too short for the heads");
  WG_REQUIRE(save_at >= 0 && save_at <= M && (save_at == 0 || snapshot),
             "wg_delta_rule_chunked: save_at %d of %d rows needs a snapshot buffer", save_at, M);
  const size_t state_bytes = (size_t)H * dk * dv * sizeof(float);
  WG_REQUIRE(!snapshot || !overlaps(snapshot, state_bytes, state, state_bytes),
             "wg_delta_rule_chunked: the snapshot overlaps the state");
  const size_t need = wg_delta_chunk_scratch_bytes(M, shape, save_at);
  WG_REQUIRE(scratch_bytes >= need, "wg_delta_rule_chunked: scratch of %zu bytes, %zu needed",
             scratch_bytes, need);
  WG_REQUIRE(((uintptr_t)scratch & 15) == 0, "wg_delta_rule_chunked: scratch not 16-byte aligned");
  int rc = raise_lds((const void *)delta_chunk_prep_kernel, (int)PREP_LDS);
  if (rc) return rc;
  const int first = first_rows(save_at), nch = chunk_count(M, first);
  const size_t fv = (size_t)H * nch * fragment_floats(dv), fk = (size_t)H * nch * fragment_floats(dk);
  float *f = static_cast<float *>(scratch);
  ChunkArgs a{qkv, ldq, ba, ldba, A, dt_bias, H, dk, dv, M, first, nch,
              f, f + 2 * fv, f + fv, f + 2 * fv + fk, f + 2 * fv + 2 * fk, f + 2 * fv + 3 * fk,
              state, snapshot, save_at, out, ldo};
  hipStream_t s = as_stream(stream);
  delta_chunk_prep_kernel<<<dim3(nch, H), 64 * CW, PREP_LDS, s>>>(a);
  rc = launched("wg_delta_rule_chunked");
  if (rc) return rc;
  delta_chunk_chain_kernel<<<dim3(H, (dv + 15) / 16), 64 * CW, 0, s>>>(a);
  return launched("wg_delta_rule_chunked");
}

int wg_delta_conv(const float *in, int32_t M, int32_t ldi, int32_t C, int32_t W,
                  const float *taps, const float *state, float *state_out, float *out,
                  int32_t ldo, void *stream) {
  WG_REQUIRE(in && taps && out && M >= 1 && C >= 1 && W >= 1 && W <= MAX_CONV,
             "wg_delta_conv: bad arguments (%d taps, 1 to %d)", W, MAX_CONV);
  WG_REQUIRE(ldi >= C && ldo >= C, "wg_delta_conv: row strides shorter than %d channels", C);
  const size_t sb = (size_t)(W - 1) * C * sizeof(float);
  WG_REQUIRE(W == 1 || (state && state_out && !overlaps(state, sb, state_out, sb)),
             "wg_delta_conv: %d taps need a state and a separate state_out", W);
  const uintptr_t ptrs = (uintptr_t)in | (uintptr_t)out | (uintptr_t)state | (uintptr_t)state_out;
  if (M >= CONV_ROWS && (int64_t)M * C >= CONV_ROWS_MIN && W >= 2 && W <= 4 && C % 4 == 0 &&
      ldi % 4 == 0 && ldo % 4 == 0 && (ptrs & 15) == 0 &&
      (M + CONV_ROWS - 1) / CONV_ROWS <= 65535) {
    auto kernel = W == 2 ? delta_conv_rows_kernel<2>
                         : W == 3 ? delta_conv_rows_kernel<3> : delta_conv_rows_kernel<4>;
    kernel<<<dim3((C / 4 + 255) / 256, (M + CONV_ROWS - 1) / CONV_ROWS), 256, 0,
             as_stream(stream)>>>(in, ldi, M, C, taps, state, state_out, out, ldo);
    return launched("wg_delta_conv");
  }
  const int64_t n = (int64_t)(M + W - 1) * C;
  delta_conv_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(
      in, ldi, M, C, W, taps, state, state_out, out, ldo);
  return launched("wg_delta_conv");
}

int wg_delta_norm(const float *o, int32_t M, int32_t ldo, const wg_delta_shape *shape,
                  const float *z, int32_t ldz, const float *weight, float eps, uint16_t *out16,
                  int32_t ldh, void *stream) {
  WG_REQUIRE(o && shape && z && weight && out16 && M >= 1, "wg_delta_norm: bad arguments");
  const int H = shape->heads, dv = shape->value_dim;
  WG_REQUIRE(H >= 1 && dv >= 1 && dv <= 256, "wg_delta_norm: %d value dims (1 to 256)", dv);
  WG_REQUIRE(ldo >= H * dv && ldz >= H * dv && ldh >= H * dv,
             "wg_delta_norm: row strides shorter than %d", H * dv);
  const int64_t waves = (int64_t)M * H;
  delta_norm_kernel<<<(unsigned)((waves + 3) / 4), 256, 0, as_stream(stream)>>>(
      o, ldo, M, H, dv, z, ldz, weight, eps, out16, ldh);
  return launched("wg_delta_norm");
}

}  // extern "C"
