// Sampling candidates on the GPU (the reference's PENALIZED + CHUNK_MAX,
// CHUNK_RANK, CHUNK_BY_RANK and CHUNK_GATHER, src/gpu/kernels.ts:3085-3163,
// :3265-3323, run by Engine.pick, src/engine.ts:8352-8473): the logits of
// the `count` 256-token chunks with the largest penalized logit, so the
// host reads back count x 1 KB a row instead of the vocabulary, and samples
// from them (for top-k with k <= count they hold the k largest: each lies
// in a chunk whose maximum is among the k largest).
//
// Stage 1 (`chunk_max_kernel`): a wave per (row, chunk) reads the chunk's
// 256 logits and mask bytes (4 a lane), penalizes each and
// reduces the maximum. Stage 2 (`chunk_rank_gather_kernel`): a wave per
// (row, chunk) ranks its chunk by maximum (larger first, ties to the lower
// index: the order the reference's ranks give) and writes the first
// `count` chunks' penalized logits.
#include "common.h"
#include "dot.h"

namespace wg {
namespace {

constexpr int CHUNK = 256;
constexpr int MAX_SEEN = 16;
constexpr int MAX_TOTAL = 2048;  // chunks a row (vocabularies up to 524,288)

struct Penalty {
  const uint8_t *mask;      // [V]: 0 unseen, 1 prompt, 2 never draw, 3 written
  const int32_t *seen;      // [n_seen][4]: token, state, first row, end row
  int n_seen, row0;
  float penalty, presence;
  const uint32_t *allowed;  // [allowed_rows][ld_allowed] bit per token, or NULL
  int allowed_rows, ld_allowed;
};

// penalized (src/gpu/kernels.ts:3102-3122): token id's logit v (its mask
// byte m) for batch row r, or -1e30 when it may not be drawn.
__device__ inline float penalized(float v, int id, int r, const Penalty &p, int V, int m) {
  if (id >= V) return -1e30f;  // past the vocabulary in the last chunk
  if (p.allowed) {
    const int row = p.allowed_rows == 1 ? 0 : r;
    if (row >= p.allowed_rows) return -1e30f;
    const uint32_t bits = p.allowed[(int64_t)row * p.ld_allowed + (id >> 5)];
    if (!((bits >> (id & 31)) & 1u)) return -1e30f;
  }
  if (m == 2) return -1e30f;
  int state = m;
  for (int k = 0; k < p.n_seen; k++) {
    const int *s = p.seen + 4 * k;
    if (s[0] == id && r >= s[2] && r < s[3]) state = s[1];
  }
  if (state == 1 || state == 3) {
    v = v < 0.0f ? v * p.penalty : v / p.penalty;
    v -= p.presence;
  }
  return v;
}

__global__ __launch_bounds__(256) void chunk_max_kernel(const float *logits, int M, int V,
                                                        int ld, Penalty p, int total,
                                                        float *maxima) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (row, chunk)
  if (w >= (int64_t)M * total) return;
  const int r = (int)(w / total), c = (int)(w % total);
  const float *row = logits + (int64_t)r * ld;
  float mx = -1e30f;
  float v[4];
  int m[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int id = c * CHUNK + 4 * lane + i;
    v[i] = id < V ? row[id] : 0.0f;
    m[i] = id < V && p.mask ? p.mask[id] : 0;
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
    mx = fmaxf(mx, penalized(v[i], c * CHUNK + 4 * lane + i, r + p.row0, p, V, m[i]));
  mx = wave_max(mx);
  if (lane == 0) maxima[w] = mx;
}

// CHUNK_RANK + CHUNK_BY_RANK + CHUNK_GATHER: a wave per (row, chunk) counts
// the chunks ahead of its own (a larger maximum, or an equal one at a lower
// index: the reference's order), which is its rank, and where that is below
// `count` writes the chunk's id and penalized logits there. Every rank
// belongs to one chunk, so every output is written once. Bound by latency:
// the chunk's logits load while the rank is counted (64 maxima a step), one
// memory round trip for both. For 128,256 logits and 64 chunks a bitonic
// sort in one workgroup and a gather launch took 11.9 + 2.7 us; this takes
// 4.6 us.
__global__ __launch_bounds__(256) void chunk_rank_gather_kernel(const float *logits, int M, int V,
                                                               int ld, Penalty p, int total,
                                                               const float *maxima, int count,
                                                               int32_t *chunks_out,
                                                               float *cand_out) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (row, chunk)
  if (w >= (int64_t)M * total) return;
  const int r = (int)(w / total), c = (int)(w % total);
  const float *row = logits + (int64_t)r * ld;
  float v[4];
  int m[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int id = c * CHUNK + 64 * i + lane;
    v[i] = id < V ? row[id] : 0.0f;
    m[i] = id < V && p.mask ? p.mask[id] : 0;
  }
  const float *mr = maxima + (int64_t)r * total;
  const float mine = mr[c];
  int rank = 0;
  for (int o = 0; o < total; o += 64) {
    const int k = o + lane;
    const float x = k < total ? mr[k] : -INFINITY;
    rank += __popcll(__ballot(k < total && (x > mine || (x == mine && k < c))));
  }
  if (rank >= count) return;  // (wave-uniform)
  if (lane == 0) chunks_out[(int64_t)r * count + rank] = c;
  float *o = cand_out + ((int64_t)r * count + rank) * CHUNK;
#pragma unroll
  for (int i = 0; i < 4; i++)
    o[64 * i + lane] = penalized(v[i], c * CHUNK + 64 * i + lane, r + p.row0, p, V, m[i]);
}

}  // namespace
}  // namespace wg

using namespace wg;

extern "C" {

size_t wg_pick_scratch_bytes(int32_t M, int32_t V) {
  return (size_t)M * ((V + CHUNK - 1) / CHUNK) * sizeof(float);
}

int wg_pick_candidates(const float *logits, int32_t M, int32_t V, int32_t ld,
                       const uint8_t *mask, const int32_t *seen_rows, int32_t n_seen,
                       int32_t row0, float penalty, float presence_penalty,
                       const uint32_t *allowed, int32_t allowed_rows, int32_t ld_allowed,
                       int32_t count, int32_t *chunks_out, float *candidates, void *scratch,
                       size_t scratch_bytes, void *stream) {
  WG_REQUIRE(logits && chunks_out && candidates && scratch && M >= 1 && V >= 1 && ld >= V,
             "wg_pick_candidates: bad arguments");
  const int total = (V + CHUNK - 1) / CHUNK;
  WG_REQUIRE(total <= MAX_TOTAL, "wg_pick_candidates: %d chunks a row (at most %d)", total,
             MAX_TOTAL);
  WG_REQUIRE(count >= 1 && count <= 64 && count <= total,
             "wg_pick_candidates: %d chunks asked of %d (1 to 64)", count, total);
  WG_REQUIRE(n_seen >= 0 && n_seen <= MAX_SEEN && (n_seen == 0 || seen_rows),
             "wg_pick_candidates: %d seen rows (at most %d)", n_seen, MAX_SEEN);
  WG_REQUIRE(penalty > 0.0f, "wg_pick_candidates: the repetition penalty must be positive");
  WG_REQUIRE(!allowed || (allowed_rows >= 1 && ld_allowed >= (V + 31) / 32),
             "wg_pick_candidates: the allowed-token bitmap needs rows and %d words a row",
             (V + 31) / 32);
  WG_REQUIRE(scratch_bytes >= wg_pick_scratch_bytes(M, V),
             "wg_pick_candidates: scratch of %zu bytes, %zu needed", scratch_bytes,
             wg_pick_scratch_bytes(M, V));
  Penalty p{mask, seen_rows, n_seen, row0, penalty, presence_penalty, allowed, allowed_rows,
            ld_allowed};
  hipStream_t s = as_stream(stream);
  const int64_t waves = (int64_t)M * total;
  float *maxima = static_cast<float *>(scratch);
  chunk_max_kernel<<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(logits, M, V, ld, p, total,
                                                               maxima);
  int rc = launched("wg_pick_candidates");
  if (rc) return rc;
  chunk_rank_gather_kernel<<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(
      logits, M, V, ld, p, total, maxima, count, chunks_out, candidates);
  return launched("wg_pick_candidates");
}

}  // extern "C"
