// mc_peak.hip -- integer peak and 1/32-pixel Fourier-interpolated peak of
// each box map, in FP64.
//
// Reference FindShift (cufunc.cu:396-497):
//  1. first maximum of the box in row-major order, excluding
//     |c - box/2| <= w && |r - box/2| <= w (w = -nps - 1 ... default -1);
//  2. 16 x 16 window at o = clamp(peak - 8, 0, box - 16), real FFT
//     (func.cpp:10-15), cosine mask 0.5 + 0.5 cos(pi r/8) for
//     r = floor(sqrt(kx^2 + ky'^2)) < 8, else 0 (func.cpp:348-370);
//  3. zero-pad to 512 x 512 (rows 0..7 and 504..511, columns 0..8) and
//     C2R (func.cpp:18-23);
//  4. first strict maximum over the 512 x 512 map starting from U[0], with
//     the exclusion scaled by 32; shift = o + p/32 - box/2, cc = U/(n^2 256).
// The 512 x 512 map is evaluated exactly from the 16 x 9 masked spectrum:
//  U[q][p] = Re sum_{kx=0}^{8} a_kx e^{2 pi i kx p/512}
//                sum_{ky} G[ky][kx] e^{2 pi i ky' q/512},
// a_0 = 1, a_kx = 2 (the C2R row weight), ky' = ky (ky < 8) or ky - 16.
#include <hip/hip_runtime.h>

#include "mc_device.h"
#include "mc_kernels.h"

namespace mc {

struct ValIdx {
  double v;
  int i;
};

// max value, ties -> smaller index (row-major first maximum)
MC_DEV ValIdx better(ValIdx a, ValIdx b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

// Result of pair p from the first strict maximum (v, i) over the map points
// other than U[0]: the sequential search starts from U[0] with a strict '>'
// (cufunc.cu:460-476); shift = o + p/32 - box/2, cc = U/(n^2 256).
MC_DEV void peak_result(int p, double v, int i, double u0, int offx, int offy, int box, int n,
                        double* __restrict__ out) {
  double bv = u0;
  int sxp = 0, syp = 0;
  if (i != 0x7fffffff && v > u0) {
    bv = v;
    sxp = i % 512;
    syp = i / 512;
  }
  out[3 * p + 0] = offx + sxp / 32.0 - box / 2;
  out[3 * p + 1] = offy + syp / 32.0 - box / 2;
  out[3 * p + 2] = bv / n / n / 16 / 16;
}

MC_DEV ValIdx wave_first_max(ValIdx b) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) b = better(b, ValIdx{__shfl_xor(b.v, o), __shfl_xor(b.i, o)});
  return b;
}

// One workgroup per pair, 512 threads.
//
// What bounds it is FP64 issue: all 512 x 512 points cost 16 multiply-adds and
// six instructions of comparison each, 107 us for 253 pairs (one workgroup per
// CU), and for few pairs the serial chain of the steps before.  Only the first
// maximum is wanted, so the points are searched in 64 x 64 cells of 8 x 8: with
// T, Tx and Ty at the cell's centre, no point of the cell exceeds
//   T + h (|Tx| + |Ty|) + h^2/2 sum |A| (|kx| + |ky|)^2,   h = 4 steps,
// the Taylor bound of the trigonometric sum with coefficients A.  Cells whose
// bound lies below the largest T found at an admitted centre hold no maximum;
// the points of the others (10 to 40 of the 4096 cells for box maps with a
// peak, up to 100 for noise) are evaluated as in the full search, so the
// result is the same bit for bit.  1e-10 sum |A| covers the rounding of T and
// of the points (about 1e-14).  A map whose points are all zero (a blank frame) or
// NaN is answered from the bound's sum alone.  A constant map keeps all cells: the
// points are then evaluated in whole rows, with factors from registers, 100 us
// against 320 cell by cell (15 maps; the line between the two lies at a quarter of
// the cells, where both take about as long).
// 96 x 96 maps: 22 us up to 256 pairs, 37 to 46 for noise; the full search took
// 51 (40 pairs, four workgroups each and a launch to combine them), 70 (105)
// and 106 (253).  What is left is latency: one wave issues an instruction in
// about 6 clocks and no step has work for more than two waves per SIMD.
constexpr int PEAK_NT = 512, PEAK_CELL = 8, PEAK_NCELL = 512 / PEAK_CELL;
constexpr int PEAK_ROWS = 14;  // cell rows whose row sums are held at a time
constexpr int PEAK_FULL = 1024;  // with more cells kept, all points in whole rows

__global__ __launch_bounds__(PEAK_NT) void k_find_peaks(const float* __restrict__ boxmaps, int box,
                                                        int n, int wnoise, double* __restrict__ out) {
  constexpr int NT = PEAK_NT, NW = NT / 64;
  __shared__ double2 t512[512 + 64];  // entry e at e + e/8: no stride of 8 in one bank
  __shared__ __align__(16) float sub[256];
  __shared__ __align__(256) double tab[2][16];  // cos, -sin of 2 pi e/16
  __shared__ double2 G[16][9];
  __shared__ double2 Hs[PEAK_ROWS * PEAK_CELL * 9];  // row sums; the centre rows' [64][9] before
  __shared__ double2 Hy[PEAK_NCELL * 9];
  __shared__ double rv[NW], rs[NW];
  __shared__ int ri[NW];
  __shared__ unsigned long long keep[PEAK_NCELL];
  __shared__ double u0s;
  static_assert(PEAK_ROWS * PEAK_CELL >= PEAK_NCELL, "the centre rows share Hs");
  static_assert(NW == PEAK_CELL && PEAK_NCELL == 64, "waves are a cell's rows, a ballot a row of cells");
  const int p = blockIdx.x;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const float* bm = boxmaps + (size_t)p * box * box;
  auto tw = [&](int e) {  // e^{2 pi i e/512}
    e &= 511;
    return t512[e + (e >> 3)];
  };
  {
    double s, c;
    sincospi((double)tid / 256.0, &s, &c);
    t512[tid + (tid >> 3)] = make_double2(c, s);
    if (tid % 32 == 0) {
      tab[0][tid / 32] = c;
      tab[1][tid / 32] = -s;
    }
  }
  // 1. integer peak (cufunc.cu:409-424); 18 loads in flight
  {
    float bv = -1e9f;
    int bi = 0x7fffffff;
    const int dr = NT / box, dc = NT - dr * box, nb = box * box;
    int r = tid / box, c = tid - r * box;
    for (int i0 = tid; i0 < nb; i0 += 18 * NT) {
      float v[18];
#pragma unroll
      for (int e = 0; e < 18; e++) v[e] = bm[min(i0 + e * NT, nb - 1)];
#pragma unroll
      for (int e = 0; e < 18; e++) {
        const int i = i0 + e * NT;
        // selects, no branches: integer products of the conditions
        const int ex = int(abs(c - box / 2) <= wnoise) & int(abs(r - box / 2) <= wnoise);
        const int up = int(i < nb) & (ex ^ 1) & int(v[e] > bv);
        bv = up ? v[e] : bv;
        bi = up ? i : bi;
        c += dc;
        const int wrap = c >= box;
        c -= wrap ? box : 0;
        r += dr + wrap;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float v = __shfl_xor(bv, o);
      const int i = __shfl_xor(bi, o);
      if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
      }
    }
    if (l == 0) {
      rv[w] = bv;
      ri[w] = bi;
    }
  }
  __syncthreads();
  ValIdx pk = {rv[0], ri[0]};
#pragma unroll
  for (int x = 1; x < NW; x++) pk = better(pk, ValIdx{rv[x], ri[x]});
  int offx = -8, offy = -8;  // no candidate: the reference keeps (0, 0)
  if (pk.i != 0x7fffffff) {
    offx = pk.i % box - 8;
    offy = pk.i / box - 8;
  }
  if (offx + 16 > box) offx = box - 16;  // cufunc.cu:430-435
  else if (offx < 0) offx = 0;
  if (offy + 16 > box) offy = box - 16;
  else if (offy < 0) offy = 0;
  offx = __builtin_amdgcn_readfirstlane(offx);
  offy = __builtin_amdgcn_readfirstlane(offy);
  if (tid < 256) sub[tid] = bm[(size_t)(offy + tid / 16) * box + offx + tid % 16];
  __syncthreads();
  // 2. 16 x 16 R2C (forward) and cosine mask, times the C2R row weight.  A
  // thread sums the real or the imaginary part of ky and of ky + 8, whose
  // factors differ by (-1)^y.
  if (tid < 144) {
    const int part = tid >= 72, o = tid - 72 * part, ky = o / 9, kx = o - 9 * ky;
    int ex[16];
#pragma unroll
    for (int x = 0; x < 16; x++) ex[x] = 8 * kx * x;
    double s0 = 0, s1 = 0;
#pragma unroll 2
    for (int y = 0; y < 16; y++) {
      const int ey = 8 * ky * y;
#pragma unroll
      for (int x = 0; x < 16; x++) {
        unsigned a = (ey + ex[x]) & 127 | part * 128;
        asm("" : "+v"(a));  // keeps the table's address out of the sum
        const double t = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(tab) + a);
        const double v = (double)sub[16 * y + x];
        s0 = fma(v, t, s0);
        s1 = fma(v, (y & 1) ? -t : t, s1);
      }
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int yy = e ? ky - 8 : ky;
      // floor(sqrt(kx^2 + yy^2)), up to 8; cos(pi r/8) is the table's
      int rr = 0;
#pragma unroll
      for (int i = 1; i <= 8; i++) rr += kx * kx + yy * yy >= i * i;
      double m = rr < 8 ? tab[0][rr] / 2 + 0.5 : 0.0;
      if (kx > 0) m *= 2.0;
      double2& g = G[ky + 8 * e][kx];
      (part ? g.y : g.x) = (e ? s1 : s0) * m;
    }
  }
  __syncthreads();
  // 3. the bound's constant term, and T, Tx, Ty at the cell centres (8 R, 8 C):
  // row sums of the centre rows, then a thread takes the columns C = l % 16 + 16 k,
  // k < 4, whose factors differ by i^(kx k), in the rows R = 4 w + 32 j + l / 16
  {
    double s = 0.0;
    constexpr double h = PEAK_CELL / 2 * 2 * 3.14159265358979323846 / 512;
    if (tid < 144) {
      const int ky = tid / 9, kx = tid - 9 * ky, yy = ky < 8 ? ky : 16 - ky;
      const double k = (kx + yy) * h;
      s = (fabs(G[ky][kx].x) + fabs(G[ky][kx].y)) * (0.5 * k * k + 1e-10);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (l == 0) rs[w] = s;
  }
  // (rows R and R + 32, whose factors differ by (-1)^yy, per thread)
  if (tid < PEAK_NCELL / 2 * 9) {
    const int q = PEAK_CELL * (tid / 9), kx = tid % 9;
    double2 h[2] = {}, d[2] = {};
#pragma unroll
    for (int ky = 0; ky < 16; ky++) {
      const int yy = ky < 8 ? ky : ky - 16;
      const double2 t = tw(yy * q), g = G[ky][kx];
      const double2 v = make_double2(g.x * t.x - g.y * t.y, g.x * t.y + g.y * t.x);
      double2& a = h[ky & 1];
      double2& b = d[ky & 1];
      a.x += v.x;
      a.y += v.y;
      b.x -= yy * v.y;
      b.y += yy * v.x;
    }
    constexpr int up = PEAK_NCELL / 2 * 9;
    Hs[tid] = make_double2(h[0].x + h[1].x, h[0].y + h[1].y);
    Hs[tid + up] = make_double2(h[0].x - h[1].x, h[0].y - h[1].y);
    Hy[tid] = make_double2(d[0].x + d[1].x, d[0].y + d[1].y);
    Hy[tid + up] = make_double2(d[0].x - d[1].x, d[0].y - d[1].y);
  }
  __syncthreads();
  const int scale = 32;
  const int wns = scale * wnoise;
  const int ox = (box / 2 - offx) * scale, oy = (box / 2 - offy) * scale;
  const double b2 = rs[0] + rs[1] + rs[2];
  if (!(b2 > 0)) {  // every point is zero (b2 too), or NaN
    if (tid == 0) peak_result(p, 0.0, 0x7fffffff, b2, offx, offy, box, n, out);
    return;
  }
  double bound[2][4], m0 = -1e300;
  {
    constexpr double h = PEAK_CELL / 2 * 2 * 3.14159265358979323846 / 512;
    const int c0 = PEAK_CELL * (l & 15);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int R = 4 * w + 32 * j + (l >> 4), q = PEAK_CELL * R;
      // sums of the terms kx = m mod 4 (complex: T and Tx take both parts)
      double2 S[4] = {}, X[4] = {}, Y[4] = {};
      S[0].x = Hs[R * 9].x;
      Y[0].x = Hy[R * 9].x;
#pragma unroll
      for (int kx = 1; kx < 9; kx++) {
        const double2 t = tw(kx * c0), a = Hs[R * 9 + kx], d = Hy[R * 9 + kx];
        const double2 v = make_double2(a.x * t.x - a.y * t.y, a.x * t.y + a.y * t.x);
        const int m = kx & 3;
        S[m].x += v.x;
        S[m].y += v.y;
        X[m].x -= kx * v.y;
        X[m].y += kx * v.x;
        Y[m].x += d.x * t.x - d.y * t.y;
        Y[m].y += d.x * t.y + d.y * t.x;
      }
      // Re sum_m i^(m k) z[m]
      auto at = [](const double2* z, int k) {
        const double e = (k & 1) ? z[0].x - z[2].x : z[0].x + z[2].x;
        return k == 0 ? e + (z[1].x + z[3].x) : k == 1 ? e - (z[1].y - z[3].y)
             : k == 2 ? e - (z[1].x + z[3].x) : e + (z[1].y - z[3].y);
      };
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const double T = at(S, k);
        bound[j][k] = T + h * (fabs(at(X, k)) + fabs(at(Y, k))) + b2;
        if (!(abs(q - oy) <= wns && abs(c0 + 128 * k - ox) <= wns) && T > m0) m0 = T;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m0 = fmax(m0, __shfl_xor(m0, o));
    if (l == 0) rv[w] = m0;
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < NW; x++) m0 = fmax(m0, rv[x]);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    unsigned long long b[4];
#pragma unroll
    for (int k = 0; k < 4; k++) b[k] = __ballot(!(bound[j][k] < m0));
    if (l < 4) {
      const int R = 4 * w + 32 * j + l;
      unsigned long long k = 0;
#pragma unroll
      for (int x = 0; x < 4; x++) k |= (b[x] >> (16 * l) & 0xffff) << (16 * x);
      // cell (0, 0) is always kept: the search starts from U[0]
      keep[R] = R == 0 ? k | 1 : k;
    }
  }
  __syncthreads();
  // 4. exact evaluation of the kept cells, first maximum
  ValIdx bb = {-1e300, 0x7fffffff};
  auto row_sum = [&](int q, int kx) {
    double2 h = make_double2(0.0, 0.0);
#pragma unroll
    for (int ky = 0; ky < 16; ky++) {
      const int yy = ky < 8 ? ky : ky - 16;
      const double2 t = tw(yy * q);
      const double2 g = G[ky][kx];
      h.x += g.x * t.x - g.y * t.y;
      h.y += g.x * t.y + g.y * t.x;
    }
    return h;
  };
  unsigned long long rows = __ballot(keep[l] != 0);
  int kept = 0;
  if (rows == ~0ull) {
    kept = __popcll(keep[l]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kept += __shfl_xor(kept, o);
  }
  if (kept > PEAK_FULL) rows = 0;  // all points, below
  while (rows) {
    // the next (up to PEAK_ROWS) cell rows: row sums, then wave w takes row w of
    // each cell and 64 lanes the points of eight cells
    unsigned long long todo = rows;
    int nr = 0;
    for (; nr < PEAK_ROWS && rows; nr++) rows &= rows - 1;
    for (int i = tid; i < nr * PEAK_CELL * 9; i += NT) {
      const int s = i / (PEAK_CELL * 9), e = i - s * (PEAK_CELL * 9), dq = e / 9, kx = e - 9 * dq;
      unsigned long long t = todo;
      for (int x = 0; x < s; x++) t &= t - 1;
      Hs[i] = row_sum(PEAK_CELL * (__ffsll((long long)t) - 1) - PEAK_CELL / 2 + dq, kx);
    }
    __syncthreads();
    for (int s = 0; s < nr; s++, todo &= todo - 1) {
      const int R = __ffsll((long long)todo) - 1;
      const int q = (PEAK_CELL * R - PEAK_CELL / 2 + w) & 511;
      double2 hq[9];
#pragma unroll
      for (int kx = 0; kx < 9; kx++) hq[kx] = Hs[(s * PEAK_CELL + w) * 9 + kx];
      for (unsigned long long k = keep[R]; k;) {
        unsigned long long mine = k;
#pragma unroll
        for (int x = 0; x < 8; x++) {
          if (x < l / PEAK_CELL) mine &= mine - 1;
          k &= k - 1;
        }
        if (!mine) continue;
        const int C = __ffsll((long long)mine) - 1;
        const int pp = (PEAK_CELL * C - PEAK_CELL / 2 + l % PEAK_CELL) & 511;
        double u = hq[0].x;
#pragma unroll
        for (int kx = 1; kx < 9; kx++) {
          const double2 t = tw(kx * pp);
          u += hq[kx].x * t.x - hq[kx].y * t.y;
        }
        if (q == 0 && pp == 0) u0s = u;
        if (abs(q - oy) <= wns && abs(pp - ox) <= wns) continue;
        // rows and cells wrap round: the points come in no particular order
        if (u > bb.v || (u == bb.v && q * 512 + pp < bb.i)) bb = ValIdx{u, q * 512 + pp};
      }
    }
    __syncthreads();
  }
  if (kept > PEAK_FULL) {
    // A thread takes the columns c0 + 128 j, whose factors stay in registers, in
    // the rows q = tid / 128 mod 4.  (After the loop above: before it, this block
    // cost the loop 2 us, 35 to 37 on 15 maps of noise.)
    constexpr int NC = 4, QC = 56;  // a row sum per thread
    static_assert(QC * 9 <= NT && QC <= PEAK_ROWS * PEAK_CELL && NT == NC * 128, "sums, rows of Hs, classes");
    const int c0 = tid & 127;
    double2 wc[NC][8];
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int kx = 1; kx < 9; kx++) wc[j][kx - 1] = tw(kx * (c0 + 128 * j));
    for (int q0 = 0; q0 < 512; q0 += QC) {
      if (tid < QC * 9) Hs[tid] = row_sum(q0 + tid / 9, tid % 9);
      __syncthreads();
      for (int qi = w >> 1; qi < min(QC, 512 - q0); qi += NC) {
        const int q = q0 + qi;
        const bool rowex = abs(q - oy) <= wns;
        double2 hq[9];
#pragma unroll
        for (int kx = 0; kx < 9; kx++) hq[kx] = Hs[qi * 9 + kx];
#pragma unroll
        for (int j = 0; j < NC; j++) {
          const int pp = c0 + 128 * j;
          double u = hq[0].x;
#pragma unroll
          for (int kx = 1; kx < 9; kx++) u += hq[kx].x * wc[j][kx - 1].x - hq[kx].y * wc[j][kx - 1].y;
          if (q == 0 && pp == 0) u0s = u;
          // a thread's points come in row-major order
          if (!(rowex && abs(pp - ox) <= wns) && u > bb.v) bb = ValIdx{u, q * 512 + pp};
        }
      }
      __syncthreads();
    }
  }
  bb = wave_first_max(bb);
  if (l == 0) {
    rs[w] = bb.v;
    ri[w] = bb.i;
  }
  __syncthreads();
  if (tid == 0) {
    bb = ValIdx{rs[0], ri[0]};
#pragma unroll
    for (int x = 1; x < NW; x++) bb = better(bb, ValIdx{rs[x], ri[x]});
    peak_result(p, bb.v, bb.i, u0s, offx, offy, box, n, out);
  }
}

hipError_t launch_find_peaks(const float* boxmaps, int npairs, int box, int n, int wnoise,
                             double* out, hipStream_t st) {
  if (npairs <= 0) return hipSuccess;
  if (box < 16) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_find_peaks, dim3(npairs), dim3(PEAK_NT), 0, st, boxmaps, box, n, wnoise, out);
  return hipGetLastError();
}

}  // namespace mc
