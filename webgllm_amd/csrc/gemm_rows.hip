// The many-row product of a matrix too narrow for the prefill GEMM's tiles
// (a linear attention block's b|a projection, 2 H rows): C[m][n] = sum_k
// A[m][k] W[n][k] with the GEMV's exact products, for any number of rows.
//
// Bound by latency: 1500 rows of a 32 x 2048 matrix are 6 MB of
// activations and 0.2 GFLOP. As GEMVs of 8 rows they were 188 launches (4.3
// us each on the device, 8 with the host's share); one launch takes 8 us:
//  - a workgroup owns 16 rows x 32 columns and its waves split K between
//    them, each on its own: activations and weights go from memory straight
//    to the operand registers of v_mfma_f32_16x16x32_f16, two steps of 64
//    weights in flight under the third, and no wave waits for another until
//    the end;
//  - one MFMA is one 32-weight block of 16 columns, its weights q - z exact
//    halves: exact products, whose float32 sum the block's scale multiplies;
//  - the waves' sums meet in LDS once, in the waves' order.
// An operand: lane (n = lane % 16, c = lane / 16) holds activations 8 c ..
// 8 c + 7 of the block's 32 in row n, and the same 8 weights of column n:
// the low (c < 2) or high nibbles of the block row's bytes 8 (c % 2) ..;
// of an 8-bit block its bytes 8 c ...
#include "common.h"
#include "dot.h"
#include "gemm_core.h"

namespace wg {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int ROWS_WAVES = 8;            // most waves a workgroup
constexpr int BM = 16, CT = 2, BN = 16 * CT;
constexpr int LDW = BN + 4;              // LDS row stride: 4 rows apart is 16 banks
constexpr int DEPTH = 3;                 // steps held: two in flight under the third

// 8 weights of a block (two dwords of nibble bytes, or of code bytes) as
// halves q - z: 1024 + q (or 1024 + 128 + q) under a 0x64 exponent byte less
// its offset, exact.
template <int ZK>
__device__ inline half8 weights8(uint2 q, uint32_t shift, float zero) {
  const _Float16 off = ZK == Q8 ? (_Float16)1152.0f : (_Float16)(1024.0f + zero);
  const half2v off2 = {off, off};
  const uint32_t k64 = 0x64646464u;
  u4v o;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t b = i ? q.y : q.x;
    const uint32_t w = ZK == Q8 ? b ^ 0x80808080u : (b >> shift) & 0x0f0f0f0fu;
    o[2 * i] = __builtin_bit_cast(
        uint32_t, as_h2(__builtin_amdgcn_perm(k64, w, 0x04010400u)) - off2);
    o[2 * i + 1] = __builtin_bit_cast(
        uint32_t, as_h2(__builtin_amdgcn_perm(k64, w, 0x04030402u)) - off2);
  }
  return __builtin_bit_cast(half8, o);
}

// One step's operands: two blocks of 32.
struct Operands {
  uint4 a[2];
  uint2 q[2][CT];
  uint16_t s[2][CT];
  uint8_t z[2][CT];
};

template <int ZK>
__global__ __launch_bounds__(64 * ROWS_WAVES) void gemm_rows_kernel(
    const uint8_t *__restrict__ quants, const uint16_t *__restrict__ scales,
    const uint8_t *__restrict__ zeros, const uint8_t *__restrict__ A, int lda,
    float *__restrict__ C, int ldc, int M, int N, int B, int tiles_m) {
  __shared__ __align__(16) float red[ROWS_WAVES][BM][LDW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int n = lane & 15, c = lane >> 4;
  const int m0 = (int)(blockIdx.x % tiles_m) * BM, n0 = (int)(blockIdx.x / tiles_m) * BN;
  // this lane's pieces at block 0 (rows and columns past the matrix read its
  // last one; their sums are not stored)
  const uint32_t off_a =
      ((uint32_t)min(m0 + n, M - 1) * (uint32_t)lda + 8u * c) * 2u;
  uint32_t row0[CT], off_q[CT];
#pragma unroll
  for (int u = 0; u < CT; u++) {
    const uint32_t col = (uint32_t)min(n0 + 16 * u + n, N - 1);
    row0[u] = (col >> 2) * (uint32_t)B * 4u + (col & 3u);
    off_q[u] = ZK == Q8 ? row0[u] * 32u + 8u * c : row0[u] * 16u + 8u * (c & 1);
  }
  const uint32_t shift = 4u * (c >> 1);
  auto load = [&](Operands &o, int u2) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint32_t b = (uint32_t)min(2 * u2 + j, B - 1);
#pragma unroll
      for (int u = 0; u < CT; u++) {
        o.q[j][u] = *reinterpret_cast<const uint2 *>(
            quants + (size_t)(off_q[u] + b * (ZK == Q8 ? 128u : 64u)));
        o.s[j][u] = scales[row0[u] + 4u * b];
        if constexpr (ZK == WG_ZERO_U8) o.z[j][u] = zeros[row0[u] + 4u * b];
      }
      o.a[j] = *reinterpret_cast<const uint4 *>(A + (size_t)(off_a + b * 64u));
    }
  };
  f4v acc[CT];
#pragma unroll
  for (int u = 0; u < CT; u++) acc[u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
  auto block = [&](const Operands &o, int j) {
#pragma unroll
    for (int u = 0; u < CT; u++) {
      float zero = 8.0f;
      if constexpr (ZK == WG_ZERO_U8) zero = (float)o.z[j][u];
      const f4v d = __builtin_amdgcn_mfma_f32_16x16x32_f16(
          __builtin_bit_cast(half8, o.a[j]), weights8<ZK>(o.q[j][u], shift, zero),
          f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
      const float s = (float)__builtin_bit_cast(_Float16, o.s[j][u]);
#pragma unroll
      for (int i = 0; i < 4; i++) acc[u][i] = fmaf(s, d[i], acc[u][i]);
    }
  };

  const int U = (B + 1) / 2;  // steps of two blocks; this wave's run of them
  const int u0 = U * wave / waves, u1 = U * (wave + 1) / waves;
  if (u0 < u1) {
    Operands st[DEPTH];
    // (steps past the run load its last one again: the loads stay
    // unconditional, so the waits count exactly)
#pragma unroll
    for (int i = 0; i < DEPTH - 1; i++) load(st[i], min(u0 + i, u1 - 1));
    for (int u = u0; u < u1; u += DEPTH) {
#pragma unroll
      for (int i = 0; i < DEPTH; i++) {
        if (u + i >= u1) break;
        load(st[(i + DEPTH - 1) % DEPTH], min(u + i + DEPTH - 1, u1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        block(st[i], 0);
        if (2 * (u + i) + 1 < B) block(st[i], 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // D[i] of lane (n, c): row 4 c + i, column n.
#pragma unroll
  for (int u = 0; u < CT; u++)
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave][4 * c + i][16 * u + n] = acc[u][i];
  __syncthreads();
  for (int e = tid; e < BM * BN / 4; e += blockDim.x) {
    const int r = e / (BN / 4), cq = (e % (BN / 4)) * 4;
    const int m = m0 + r, col = n0 + cq;
    if (m >= M || col >= N) continue;  // (N: a multiple of 4)
    f4v v = *reinterpret_cast<const f4v *>(&red[0][r][cq]);
    for (int w = 1; w < waves; w++) v += *reinterpret_cast<const f4v *>(&red[w][r][cq]);
#pragma unroll
    for (int i = 0; i < 4; i++) C[(int64_t)m * ldc + col + i] = v[i];
  }
}

template <int ZK>
int launch_rows(const wg_q4_matrix *w, const uint16_t *A, int M, int lda, float *C, int ldc,
                hipStream_t s) {
  const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((w->N + BN - 1) / BN);
  // 8 waves a compute unit, each of 2 steps or more
  const int B = w->K / 32, steps = (B + 1) / 2, cus = persistent_grid(1 << 30, 1);
  int waves = 1;
  while (waves < ROWS_WAVES && (int64_t)tiles * waves < 8 * cus && steps >= 4 * waves) waves *= 2;
  gemm_rows_kernel<ZK><<<tiles, waves * 64, 0, s>>>(
      (const uint8_t *)w->quants, (const uint16_t *)w->scales, (const uint8_t *)w->zeros,
      (const uint8_t *)A, lda, C, ldc, M, w->N, B, tiles_m);
  return launched("wg_q4_gemm_rows");
}

}  // namespace
}  // namespace wg

using namespace wg;

extern "C" {

int wg_q4_gemm_rows(const wg_q4_matrix *w, const uint16_t *A, int32_t M, int32_t lda, float *C,
                    int32_t ldc, void *stream) {
  int rc = check_matrix(w, "wg_q4_gemm_rows");
  if (rc) return rc;
  WG_REQUIRE(A && C && M >= 1, "wg_q4_gemm_rows: bad arguments");
  WG_REQUIRE(lda >= w->K && lda % 8 == 0 && ((uintptr_t)A & 15) == 0,
             "wg_q4_gemm_rows: activations need a 16-byte aligned stride >= K");
  WG_REQUIRE(((uintptr_t)w->quants & 7) == 0, "wg_q4_gemm_rows: quants not 8-byte aligned");
  WG_REQUIRE(ldc >= w->N, "wg_q4_gemm_rows: ldc %d < N %d", ldc, w->N);
  WG_REQUIRE((int64_t)M * lda * 2 < ((int64_t)1 << 31) && (int64_t)w->N * w->K < ((int64_t)1 << 32),
             "wg_q4_gemm_rows: %d x %d activations or a %d x %d matrix past 2 GiB", M, lda, w->N,
             w->K);
  WG_REQUIRE(!overlaps(A, (size_t)M * lda * 2, C, (size_t)M * ldc * 4),
             "wg_q4_gemm_rows: activations and output overlap");
  hipStream_t s = as_stream(stream);
  if (w->layout == WG_LAYOUT_Q8) return launch_rows<Q8>(w, A, M, lda, C, ldc, s);
  if (w->layout == WG_LAYOUT_ROWGROUP && w->zero == WG_ZERO_8)
    return launch_rows<WG_ZERO_8>(w, A, M, lda, C, ldc, s);
  if (w->layout == WG_LAYOUT_ROWGROUP && w->zero == WG_ZERO_U8)
    return launch_rows<WG_ZERO_U8>(w, A, M, lda, C, ldc, s);
  return fail(WG_ERR_UNSUPPORTED,
              "wg_q4_gemm_rows: reads 8-bit and integer-zero-point 4-bit row-group matrices");
}

}  // extern "C"
