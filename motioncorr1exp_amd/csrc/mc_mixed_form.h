// mc_mixed_form.h -- factors of the mixed-factor transforms (mc_mixed.hip) and the
// choice between them and the chirp-z transform (mc_czt.hip) by the length and the
// transforms of a launch.  Host code without HIP, so that a CPU test can walk them.
#pragma once
#include <algorithm>

namespace mc {

// Length of the cyclic convolutions of a chirp-z transform: `need` or more.
inline int czt_len(int need) {
  int M = 64;
  while (M < need) M <<= 1;
  return M;
}

// Estimated clocks per element and SIMD of a level (issue of the vector ALU and
// the matrix unit; measured sums of the parts).
inline double mix_cost(int F) {
  constexpr double regs[17] = {0, 0, 11, 14, 13, 17, 16, 19, 16, 20, 19, 24, 18, 27, 21, 21, 18};
  if (F <= 16) return regs[F] * 4 / 64;
  const int mt = (F / 2 + 16) / 16, ks = (F / 2 + 4) / 4;
  return (mt * ks * 128 + ks * 88 + mt * 400) / (16.0 * F);
}

// Cheapest factors of N in 2..127, two to four, ascending; 0: none.
struct MixSearch {
  double best = 1e30;
  int m = 0, f[4], F[4];
  void walk(int rest, int lo, int i, double c) {
    if (c >= best) return;
    if (rest == 1) {
      if (i < 2) return;
      best = c;
      m = i;
      std::copy(f, f + i, F);
      return;
    }
    if (i == 4) return;
    for (int x = lo; x <= 127 && x <= rest; x++) {
      if (rest % x) continue;
      f[i] = x;
      walk(rest / x, x, i + 1, c + mix_cost(x));
    }
  }
};
inline int mix_factors(int N, int* F) {
  MixSearch s;
  s.walk(N, 2, 0, 0.0);
  std::copy(s.F, s.F + s.m, F);
  return s.m;
}

// Whether `items` transforms of length N in one launch run in mixed factors; the
// others are chirp-z.  A large factor F is a serial chain of matrix instructions
// (F = 127: 256 of them, 3.4 us), and a short transform has few columns N/F to
// fill the waves with.  So a launch that does not fill the chip takes as long as
// the chirp-z transform of two short power-of-two convolutions or longer: one
// 254 x 254 image, columns 10.9 us against 5.0; 762, rows and columns 15.0 and 13.0
// against 9.8 and 10.2; 508, 13.7 and 11.6 against 6.6 and 7.2.  The convolution
// of twice the length doubles its time, so the factor at which the chain is the
// longer of the two grows with its length M: 17 up to M = 512, 41 at 1024, 97 at
// 2048 (1010 = 101 x 10, columns 12.8 against 11.4; 890 = 89 x 10, 10.7 against
// 11.0), none above (1090 = 109 x 10: the whole transform 52 us against 61).  It
// fills the chip at about 1400, 2000, 1600 and 800 transforms of M = 256, 512, 1024
// and 2048, from where on its time steps up (24 frames of 762: stage 1 224 us
// against 163).  At M = 512 a factor of 97 or more is slower at
// any count (254, 32 frames: 18.5 against 15.0).  Factors up to 16 are the slower of
// the two only at M = 512, up to 1000 transforms and forward (rows of 416 x 416
// images, 16 x 13: one 7.4 us against 6.4, eight 9.3 against 15.8; back, within 0.5
// us of each other).
inline bool mix_use(int N, long long items, bool forward) {
  int F[4];
  const int m = mix_factors(N, F);
  if (!m) return false;
  const int big = F[m - 1], M = czt_len(2 * N - 1);
  if (M == 512 && forward && items <= 1000) return false;
  if (big <= 16 || M > 2048) return true;
  if (M <= 256) return big < 97 && items > 1400;
  if (M == 512) return big < 97 && items > 2000;
  if (M == 1024) return big < 41 || items > 1600;
  return big < 97 || items > 800;
}

}  // namespace mc
