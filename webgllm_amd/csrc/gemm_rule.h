// Which tile and how many K splits a prefill GEMM (gemm.hip) takes: host
// arithmetic on sizes alone.
#pragma once

#include <cstdint>

#include "../../include/webgllm_hip.h"
#include "gemm_core.h"

namespace wg {

// K splits that meet through memory, doubled (up to 4) while the workgroups
// stay within `room` and every split keeps at least `stages` steps of 64.
inline int gemm_k_splits(int64_t tiles, int steps, int stages, int64_t room) {
  int ks = 1;
  while (ks < 4 && tiles * ks * 2 <= room && steps % (2 * ks) == 0 && steps / (2 * ks) >= stages)
    ks *= 2;
  return ks;
}

// The tile of an M x N x K product of weight form zk on `cus` compute units:
// 0 64 x 64, 1 64 x 128, 2 128 x 128, 3 128 x 256; wave groups 4 64 x 128
// (2 of them), 5 64 x 64 (4), 6 32 x 32 (8), 7 32 x 64 (4), 8 128 x 128 (2).
// residual: whether a residual is added, which the last wave group alone
// reads; groups: whether wave groups may be taken; splits: whether 0 to 3 may
// split K between workgroups (not while a stream is captured).
//
// Every line was measured on a grid of 9 to 2048 rows, 256 to 28672 columns
// and 64 to 14336 deep, all four weight forms, with and without a residual,
// eager launches over several matrices; "/" stands between this tile and the
// one on the line's other side, in microseconds.
inline int gemm_tile_for(int zk, int M, int N, int K, int cus, bool residual, bool groups,
                         bool splits) {
  const int64_t m32 = (M + 31) / 32, m64 = (M + 63) / 64, m128 = (M + 127) / 128;
  // Wave groups: the smallest tile whose workgroups all run at once, so that
  // no weight waits for a second round and no sum goes through memory (131
  // rows of 896 -> 1152 6.8 / 12.5 (6), 4864 -> 896 12.4 / 23.9 (6); 45 rows,
  // 8-bit, 2048 -> 16384 13.6 / 20.2 (5); 512 rows of 4096 -> 4096 25.5 /
  // 31.7 (4)). Past those workgroups they are slower (512 rows of 896 -> 9728
  // 28.9 / 22.7). Past 8192 deep, where the loop outweighs the splits'
  // meeting, only 32 x 32 is faster (45 rows of 14336 -> 4096 32.9 / 45.0).
  // Under 256 deep (4 steps) their groups have a step or none each (45 rows ->
  // 1152, Q4_0: 64 deep 4.8 / 4.3, 256 deep 4.7 / 5.3, 512 deep 4.6 / 7.3).
  if (groups && K >= 256) {
    const bool shallow = K <= 8192;
    if (m32 * (N / 32) <= cus) return 6;
    if (shallow && m32 * (N / 64) <= cus) return 7;
    // One 64 x 64 a compute unit against two 32 x 64 (300 rows of 4096 ->
    // 3072, half zero points, 19.4 / 22.4; 400 of 8192 -> 2048, Q4_0, 26.1 /
    // 29.5), but for the shallowest (Q4_0 at 768 2% slower in the mean) and,
    // where two waves would wait for 64 x 64 values of a residual, the 4-bit
    // forms (700 rows of 4608 -> 1024, Q4_0, 24.4 / 22.8; 2048 -> 768 1.5
    // times) up to 6144 deep for half zero points, 2% in the mean, and at any
    // depth for the others. Up to 64 rows a residual is too little to matter
    // (45 rows of 5632 -> 9216, half zero points, 8% faster than two). Byte
    // zero points gain on neither past 6144 deep, 7168 with a residual (33
    // rows of 8192 -> 9728 28.3 / 25.4 on the split 64 x 128).
    if (shallow && m64 * (N / 64) <= cus) {
      const bool waits = residual && m64 > 1;
      if (splits && zk == WG_ZERO_U8 && K > (waits ? 7168 : 6144)) return N % 128 ? 0 : 1;
      if (zk == Q8 || (waits ? zk == WG_ZERO_F16 && K > 6144 : K >= 1024)) return 5;
    }
    // Two 32 x 64 a compute unit (their rings leave room, an 8-bit one's but
    // just: from 2048 deep, past it with a residual, 65 rows of 2048 -> 9216
    // 21.9 / 18.6): 131 rows of 4096 -> 6144 17.0 / 21.4, 8192 ->
    // 6144 30.5 / 36.3.
    if (shallow && m32 * (N / 64) <= 2 * cus && (zk != Q8 || K >= (residual ? 2560 : 2048)))
      return 7;
    // 64 x 128 in two groups, up to where the splits of one group catch up:
    // Q4_0 first, whose dequant is cheapest (100 rows of 8192 -> 9728 41.4 /
    // 36.4), half zero points last (131 of 8192 -> 9728 56.0 / 58.7, 1500 of
    // 8192 -> 896 55.9 / 46.6 on 128 x 128). A residual costs the splits of
    // 128 x 128 more (1500 rows of 8192 -> 1024, half zero points, 4% in the
    // mean against 14%).
    if (shallow && N % 128 == 0 && m64 * (N / 128) <= cus) {
      const bool few = M < 512;
      const int deep = zk == WG_ZERO_8     ? (!residual ? 3072 : few ? 4096 : 5632)
                       : zk == WG_ZERO_U8  ? 4096
                       : zk == WG_ZERO_F16 ? (few || residual ? 8192 : 4096)
                       : few               ? 7168
                                           : (residual ? 8192 : 6144);
      if (!splits || K <= deep) return 4;
      // (Q4_0, 1024 rows of 8192 -> 1152: 64 x 128 36.9, 128 x 128 39.8)
      if (zk == WG_ZERO_8 || zk == WG_ZERO_U8) return 1;
    }
  }
  if (N % 128) return 0;
  // Each weight is dequantized once per tile, so taller tiles (more rows a
  // wave) spend fewer vector instructions per MFMA: 128 x 256 where its
  // tiles cover most compute units, else 128 x 128 from 512 rows, else 64 x
  // 128; splitting K makes up the workgroups that few tiles leave short.
  const int64_t t1 = m64 * (N / 128), t2 = m128 * (N / 128);
  if (N % 256 == 0 && m128 * (N / 256) * 4 >= (int64_t)cus * 3) return 3;
  // 128 x 128 tiles that run at most one a compute unit leave its SIMDs a
  // wave each: two wave groups a tile (8: 100 rows of 4096 -> 28672 44.5 /
  // 57.2, 512 of 4096 -> 6144 55.5 / 60.4, 1500 of 8192 -> 2048 78.5 / 85.0),
  // or up to 2048 deep, where the groups' own loops are short, 64 x 128
  // (1500 of 2048 -> 2048 32.0 / 42.6, 512 of 2048 -> 8192 33.3 / 43.4, Q4_0;
  // half zero points, whose dequant costs most, to 1536 without a residual:
  // 2048 of 2048 -> 1152 30.6 / 28.7). Below 512 rows only half zero points
  // pay for 8 (200 rows of 4096 -> 14336, Q4_0: 50.9 / 46.4 on 64 x 128).
  if (K >= 256 && K <= (zk == WG_ZERO_F16 && !residual ? 1536 : 2048) && t2 <= cus) return 1;
  if (groups && K > 2048 && K <= 8192 && t2 <= cus && 4 * t2 >= 3 * (int64_t)cus &&
      (M >= 512 || zk == WG_ZERO_F16))
    return 8;
  // Past 8192 deep 128 rows pay below 512 where they alone leave room for
  // another split, and only for the forms whose dequant costs most (300 rows
  // of 14336 -> 4096: half zero points 72.2 / 93.4, 8-bit 67.3 / 74.1, byte
  // zero points 63.9 / 65.5, Q4_0 61.9 / 59.9; -> 2048, both split 4 ways,
  // 8-bit 49.4 / 44.5). A residual costs the taller tile's waves more: then
  // only half zero points, and 8-bit where 64 rows need a second round (400
  // of 8448 -> 4096, 8-bit, 68.9 / 60.6; -> 5120 85.5 / 88.4). Unsplit, half zero points pay where only 64 rows need
  // a second round (300 of 8448 -> 9728 98.7 / 108.8).
  if (K > 8192 && M > 256 && M < 512 && zk != WG_ZERO_8 && (zk != WG_ZERO_U8 || K > 11008)) {
    const int64_t room = 2 * (int64_t)cus;
    const bool pays = zk == WG_ZERO_F16 || !residual || (zk == Q8 && t1 > cus);
    if (splits ? pays && gemm_k_splits(t2, K / 64, 3, room) > gemm_k_splits(t1, K / 64, 4, room)
               : zk == WG_ZERO_F16 && t1 > cus && t2 <= cus)
      return 2;
  }
  return M >= 512 ? 2 : 1;
}

}  // namespace wg
