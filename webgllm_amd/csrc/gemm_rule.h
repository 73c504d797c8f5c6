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
// groups: whether wave groups may be taken.
inline int gemm_tile_for(int zk, int M, int N, int K, int cus, bool groups) {
  // The smallest tile whose workgroups all run at once (7's rings leave room
  // for two a compute unit but for 8-bit weights), so that no weight waits
  // for a second round and no sum goes through memory. Microseconds, with
  // groups / the forms below: 131 rows of 896 -> 1152 6.8 / 12.5 (6), 896 ->
  // 9728 10.7 / 15.0 (4), 4864 -> 896 12.4 / 23.9 (6); 45 rows, 8-bit, 2048
  // -> 16384 13.6 / 20.2 (5), 8192 -> 2048 15.8 / 23.0 (6); 512 rows of 2048
  // -> 2048 13.4 / 28.8 (7), 4096 -> 4096 40.7 / 51.4 (4). Past those
  // workgroups they are slower (512 rows of 896 -> 9728 28.9 / 22.7), and
  // past 8192 deep, where the loop outweighs the splits' meeting, no faster
  // (131 rows of 14336 -> 4096 63 / 60; 6, with 45 rows, 32.9 / 45.0). Rows
  // under 768 deep (12 steps) keep the forms below too: the groups would save
  // them 4 of 8 to 10 us, but models that narrow are tests', whose greedy
  // picks follow the order of the sums.
  if (groups && K >= 768) {
    const int64_t m32 = (M + 31) / 32, m64 = (M + 63) / 64;
    const bool shallow = K <= 8192;
    if (m32 * (N / 32) <= cus) return 6;
    if (shallow && m32 * (N / 64) <= (zk == Q8 ? 1 : 2) * cus) return 7;
    if (shallow && m64 * (N / 64) <= cus) return 5;
    if (shallow && N % 128 == 0 && m64 * (N / 128) <= cus) return 4;
  }
  if (N % 128) return 0;
  // Each weight is dequantized once per tile, so taller tiles (more rows a
  // wave) spend fewer vector instructions per MFMA: 128 x 256 where its
  // tiles cover most compute units, else 128 x 128 from 512 rows, else 64 x
  // 128; splitting K makes up the workgroups that few tiles leave short.
  const int64_t m128 = (M + 127) / 128, t2 = m128 * (N / 128);
  if (N % 256 == 0 && m128 * (N / 256) * 4 >= (int64_t)cus * 3) return 3;
  // 128 x 128 tiles that run at most one a compute unit leave its SIMDs a
  // wave each: two wave groups a tile (8), or up to 2048 deep, where the
  // groups' own loops are short, the smaller tiles. Microseconds, 128 x 128
  // / this: 100 rows of 4096 -> 28672 57.2 (64 x 128) / 44.5 (8), 512 of
  // 4096 -> 6144 60.4 / 55.5 (8), 1500 of 8192 -> 2048 85.0 / 78.5 (8), 1500
  // of 2048 -> 2048 42.6 / 32.0 (64 x 128), 512 of 2048 -> 8192 43.4 / 33.3
  // (64 x 128). Below 512 rows only half zero points, whose dequant costs
  // most, pay for the taller tile (200 rows of 4096 -> 14336, Q4_0: 46.4 on
  // 64 x 128 against 50.9). Past 8192 deep 128 rows pay from 257 on (300 of 14336 ->
  // 4096: 87.9 against 100.4 on 64 x 128; 192: 65.5 against 60.4).
  if (K >= 768 && K <= 2048 && t2 <= cus) return 1;
  if (groups && K > 2048 && K <= 8192 && t2 <= cus && 4 * t2 >= 3 * (int64_t)cus &&
      (M >= 512 || zk == WG_ZERO_F16))
    return 8;
  return M >= (K > 8192 ? 257 : 512) ? 2 : 1;
}

}  // namespace wg
