// mc_cols_form.h -- the form of k_pair_cols_r (mc_cols.hip) that a transform
// size and peak box take, with its waves and LDS.  Host code without HIP, so
// that a CPU test can walk every size and box.
#pragma once
#include <stddef.h>

#include <initializer_list>

namespace mc {

constexpr size_t COLS_LDS_MAX = 160 * 1024;  // LDS of a CU, and the most of one workgroup

inline int cols_r_waves(int n, int R0) { return (n / R0 + 63) / 64; }

// LDS of a workgroup: per wave its exchange block and two buffers of the sums.
inline size_t cols_r_lds(int n, int R0, int tiles) {
  return (size_t)cols_r_waves(n, R0) * ((R0 > 8 ? 8192 : 66 * 64) + tiles * 2048);
}

// The radix of k_pair_cols_r at size n and the tiles of eight groups that the
// box needs: the largest divisor whose tiles, waves and LDS the kernel holds (its
// work per element falls with R0); 0: none, the chirp-z pass.  The LDS excludes
// three tiles at 16 waves alone: 165888 bytes (radix 6, n from 5766, boxes above
// 96; radix 8, n from 7688, boxes above 128).
inline int cols_radix(int n, int box, int* tiles) {
  for (int R0 : {16, 14, 12, 10, 8, 6}) {
    const int t = (box + 8 * R0 - 1) / (8 * R0);
    if (n % R0 || t > (R0 > 8 ? 2 : 3) || cols_r_waves(n, R0) > (t == 1 || R0 <= 8 ? 16 : 8) ||
        cols_r_lds(n, R0, t) > COLS_LDS_MAX)
      continue;
    *tiles = t;
    return R0;
  }
  return 0;
}

}  // namespace mc
