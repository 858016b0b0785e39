// mc_cols.hip -- FP32 column pass of the pair stage: per (pair, kx) the
// weighted cross power X[ky] = F_a[ky] conj(F_b[ky]) wx wy[ky] and the rows of
// its column inverse that the peak box needs,
//   T[r] = sum_ky X[ky] e^{2 pi i ky (ori + r)/n},  r < box, ori = (n - box)/2
// (cuShiftCC cufunc.cu:343-361, the column half of the C2R at DFAlign.cu:897,
// 1008, and FindShift's read-out of the central box, cufunc.cu:398-407).
//
// What bounds the pass is vector-ALU issue and the delivery of the two columns
// out of L2 (64 KB per item at n = 4096, 34 GB for 253 pairs).  So:
//  - columns are read with 16-byte loads (8-byte loads are held to half the
//    L1 rate, which alone took 1.7 ms of a 3.1 ms pass at 3838x3710x40 padded
//    to 4096): a lane loads two neighbouring elements of one row for the lower
//    or the upper half of the rows, and v_permlane32_swap turns that into one
//    element of every row;
//  - each wave transforms its own share of an item and exchanges through its
//    own LDS block, ordered within the wave; one workgroup barrier per item,
//    before the partial T columns of the waves are added;
//  - the contraction that follows runs on FP32 matrix instructions, which
//    retire twice the multiply-adds of the (unpacked) vector ALU per cycle.
//    They share its issue: the two do not overlap (594 issue slots per wave
//    and item measured 2376 clocks), so they only pay where they replace
//    products one for one.
//
// Persistent launches: a grid of the resident workgroups, a multiple of 8;
// workgroup b runs on XCD b % 8 and walks the kx-major items of that XCD's
// range, so that the frame columns of one kx are reused out of its L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "mc_cols_form.h"
#include "mc_device.h"
#include "mc_kernels.h"

namespace mc {

typedef float v4f __attribute__((ext_vector_type(4)));

// n a multiple of 128, box <= 256.  ky = a + A (j + 4 r), A = n/64, j < 4,
// r < 16.  Per (a, j) a 16-point DFT over r in registers; times
// e^{2 pi i k (a + A j)/n}, which holds the twiddles of both later steps; per
// (a, k) a 4-point DFT over j, giving Y_a[q] e^{2 pi i a k/n} with q the output
// residue; then with the rows R = base + 16 g + k, base = n/2 - 64 SETS (a
// multiple of 64), g < 8 SETS, which contain every box up to 128 SETS,
//   T[R] = sum_a e^{2 pi i a (base + 16 g)/n} (Y_a[g mod 4] e^{2 pi i a k/n}),
// on v_mfma_f32_4x4x1 (16 blocks): block = (a mod 4, k / 4), columns k mod 4,
// rows (re, im) of the factors of the groups q and q + 4.  The real and the
// imaginary part of Y are multiplied by the same rows (D1, D2) and combined at
// the end, which needs no second set of factors.  A wave takes up to 16 a of
// all four j (64 lanes); the lanes' sums are added with lane swaps.
// NG = 6 stores only the groups 1..6 (box <= 96), NG = 8 all; NG = 16 takes a
// second set of factors for the groups 8..15 (128 < box <= 256).
// 128 VGPRs, 4 waves per SIMD (at 3 the pass takes 2.78 ms against 2.55).
// 4096, 253 pairs: 2.5 ms; the two-stage 16 x 8 pass
// with LDS combine that it replaces took 3.1.  2048, 153 pairs: 0.37 against
// 0.47 and, untuned, 0.78.  Two pairs of one first operand per load of that
// operand saved 6% of the issue and 25% of the loads and gave 2%: dropped.
// Boxes above 128, 15 pairs: 4096, box 200: 0.24 ms against 0.25 for the
// 256-point form of the former pass and 0.28 for k_pair_cols_r<16, 2>; 2048,
// box 256: 67 us against 69 and 78.
template <int NG>
__global__ __launch_bounds__(512, NG > 8 ? 3 : 4) void k_pair_cols64(
    const float2* __restrict__ spectra, size_t spec_stride, const int2* __restrict__ pairs,
    int npairs, const float* __restrict__ wxy, int n, int box, float2* __restrict__ tbuf,
    const float2* __restrict__ tw, int kxb, int nkx) {
  extern __shared__ float4 cols_lds[];
  constexpr int SETS = (NG + 7) / 8, NR = 128 * SETS;  // factor sets, rows R
  const int A = n / 64, nw = (A + 15) / 16, H = n / 2 + 1;
  const int AC = ((A + nw - 1) / nw + 1) / 2 * 2;  // a's per wave, even, <= 16
  const int tid = threadIdx.x, nt = nw * 64;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  // loads: lane (h, j, ap) takes a = a0, a0 + 1 in the rows r = s + 8 h; after
  // the swap it holds a = a0 + h in all 16 rows
  const int h = l >> 5, ap = l & 7, j = (l >> 3) & 3;
  const int a0 = w * AC + 2 * ap;
  const bool act = 2 * ap < AC && a0 < A;
  const int voff = act ? 8 * (a0 + A * j + 32 * A * h) : n * 8;  // past the end: reads zero
  const int xi = act ? a0 + h + A * j : 0;
  const int base = n / 2 - 64 * SETS, ori = (n - box) / 2;
  float wy[16];
#pragma unroll
  for (int r = 0; r < 16; r++) wy[r] = wxy[H + xi + 4 * A * r];
  float2 tk[16];
#pragma unroll
  for (int k = 1; k < 16; k++) tk[k] = tw[k * xi];
  // matrix rows m = l % 4: (re, im) of the factor of group q + 4 (m / 2) at
  // a = (l / 16) + 4 t of this wave; q >= 4: the second set, groups 8 on
  float P[4][4 * SETS];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int q = 0; q < 4 * SETS; q++) {
      const int ac = (l >> 4) + 4 * t, a = w * AC + ac, g = (q & 3) + 8 * (q >> 2) + 4 * ((l & 3) >> 1);
      const float2 f = ac < AC && a < A ? tw[a * (base + 16 * g) % n] : make_float2(0.f, 0.f);
      P[t][q] = (l & 1) ? f.y : f.x;
    }
  // exchange block of the wave: row j * 16 + a (16 k, 128 bytes), 16-byte
  // slots permuted by a / 2: conflict-free writes by (j, ap) and reads by k
  const int zb = w * 8192 + (j * 16 + 2 * ap + h) * 128 + ap * 16;
  const int k = l & 15, al = l >> 4;
  const int rd = w * 8192 + al * 128 + (((k >> 1) ^ (al >> 1)) << 4) + (k & 1) * 8;
  float* red = reinterpret_cast<float*>(cols_lds + nw * 512);  // [2][nw][NR] complex
  const int xcd = blockIdx.x % 8, lid = blockIdx.x / 8, nper = gridDim.x / 8;
  const long long items = (long long)npairs * nkx;
  const int i1 = (int)(items * (xcd + 1) / 8);
  int it = (int)(items * xcd / 8) + lid;
  if (it >= i1) return;
  int kx = it / npairs, p = it - kx * npairs;
  const int dkx = nper / npairs, dp = nper - dkx * npairs;
  for (int par = 0;; par ^= nw * 2 * NR) {
    const int2 pr = pairs[p];
    const auto qa = buf_rsrc(spectra + (size_t)pr.x * spec_stride + (size_t)(kxb + kx) * n, n * 8);
    const auto qb = buf_rsrc(spectra + (size_t)pr.y * spec_stride + (size_t)(kxb + kx) * n, n * 8);
    float4 ra[8], rb[8];
    float2 v[16];
    auto load = [&](int s) {
      ra[s] = buf_ld4(qa, voff, 32 * A * s);
      rb[s] = buf_ld4(qb, voff, 32 * A * s);
    };
    // Seven of the eight row pairs are loaded ahead, in order, and the eighth
    // when the first has been used: eight put the loop over its 128 registers,
    // and any spill in it costs more than its own loads (2.47 ms without, 2.65
    // with 3 to 12 registers spilled, 3.2 with 9 or more in the product).
    constexpr int D = 7;
#pragma unroll
    for (int s = 0; s < D; s++) {
      load(s);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < 8; s++) {
      v[s] = cmulc(make_float2(ra[s].x, ra[s].y), make_float2(rb[s].x, rb[s].y));
      v[s + 8] = cmulc(make_float2(ra[s].z, ra[s].w), make_float2(rb[s].z, rb[s].w));
      swap32(v[s].x, v[s + 8].x);
      swap32(v[s].y, v[s + 8].y);
      if (s + D < 8) load(s + D);
      __builtin_amdgcn_sched_barrier(0);
    }
    dft16w<1>(v, wy);
#pragma unroll
    for (int e = 1; e < 16; e++) v[e] = cmul(v[e], tk[e]);
    // the slot addresses are recomputed per item (an opaque copy): held, they
    // would push constants of the loop out of the 128 registers
    int za = zb;
    asm volatile("" : "+v"(za));
#pragma unroll
    for (int e = 0; e < 8; e++)
      *reinterpret_cast<float4*>(reinterpret_cast<char*>(cols_lds) + (za ^ (16 * e))) =
          make_float4(v[2 * e].x, v[2 * e].y, v[2 * e + 1].x, v[2 * e + 1].y);
    wave_fence();
    v4f D1[4 * SETS], D2[4 * SETS];
#pragma unroll
    for (int q = 0; q < 4 * SETS; q++) D1[q] = D2[q] = v4f{0.f, 0.f, 0.f, 0.f};
    int ra0 = rd;
    asm volatile("" : "+v"(ra0));
#pragma unroll
    for (int t = 0; t < 4; t++) {
      float2 u[4];
#pragma unroll
      for (int jj = 0; jj < 4; jj++)
        u[jj] = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(cols_lds) +
                                                 (ra0 ^ (t << 5)) + 512 * t + jj * 2048);
      dft4<1>(u);
#pragma unroll
      for (int q = 0; q < 4 * SETS; q++) {
        D1[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(P[t][q], u[q & 3].x, D1[q], 0, 0, 0);
        D2[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(P[t][q], u[q & 3].y, D2[q], 0, 0, 0);
      }
    }
    wave_fence();
    // add the four a mod 4: lanes l < 32 end with the real parts, the others
    // with the imaginary ones; even rows of 16 lanes with group g, odd g + 1
    constexpr int G0 = (8 * SETS - NG) / 2;
    float S[8 * SETS];
#pragma unroll
    for (int g = G0; g < 8 * SETS - G0; g++) {
      const int q = (g & 3) + 4 * (g >> 3), m = 2 * ((g >> 2) & 1);
      float re = D1[q][m] - D2[q][m + 1], im = D1[q][m + 1] + D2[q][m];
      swap32(re, im);
      S[g] = re + im;
    }
    int lt;  // the lane, made again per item: one register less in the loop
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lt));
    float* rw = red + par + w * 2 * NR + (lt & 31) * 2 + (lt >> 5);
#pragma unroll
    for (int g = G0; g < 8 * SETS - G0; g += 2) {
      swap16(S[g], S[g + 1]);
      rw[g * 32] = S[g] + S[g + 1];
    }
    if (nw > 1) lds_barrier();
    else wave_fence();
    // the next item writes the other half of red: one barrier per item
    const float wx = wxy[kxb + kx];
    const float2* rp = reinterpret_cast<const float2*>(red + par);
    const auto qt = buf_rsrc(tbuf + ((size_t)p * H + kxb + kx) * box, box * 8);
    for (int r = w * 64 + lt; r < box; r += nt) {
      float2 s = rp[r + ori - base];
      for (int x = 1; x < nw; x++) s = cadd(s, rp[x * NR + r + ori - base]);
      buf_st2(qt, 8 * r, cscale(s, wx));
    }
    it += nper;
    if (it >= i1) break;
    kx += dkx;
    p += dp;
    if (p >= npairs) {
      p -= npairs;
      kx++;
    }
  }
}

// Any other even n = R0 A, R0 a divisor of n out of 16, 14, 12, 10, 8 and 6.
// ky = xi + A r, r < R0: per xi an R0-point DFT over r in registers, times
// e^{2 pi i xi kappa/n}, giving z_xi[kappa]; then with the rows
// ori + r' = base + R0 g + kappa (base: the multiple of R0 at or below ori; the
// columns kappa < c = ori - base take the next group, by a factor
// e^{2 pi i xi R0/n} folded into their twiddle)
//   T = sum_xi f_g(xi) z_xi[kappa],  f_g(xi) = e^{2 pi i xi (base + R0 g)/n},
// on v_mfma_f32_16x16x4: rows (g, re | im), eight groups per tile, columns
// kappa, four xi per instruction.  The real and imaginary parts of z are
// multiplied by the same rows and combined at the end.  R0 <= 8 fills the 16
// columns with two sets of xi (lanes l and l + 32, xi and xi + 1), whose sums
// differ by one factor per group.
// The contraction costs 8 n box/R0 multiply-adds per item on units twice as
// fast as the vector ALU; the chirp-z pass it replaces takes two transforms of
// the next power of two above n + box: 1854, box 96, 78 pairs: 0.36 ms against
// 0.83; 3710, 253 pairs: 3.9 against 5.0 for its decimated pass (53 FFTs of 70
// points with five barriers per item); 4092, 55 pairs: 0.99 against 1.20.
// 105 pairs: 3696 (R0 = 16) 1.17 ms, 3710 (R0 = 14) 1.63; the radix and the columns
// of 3710 that do not start on 64 bytes were not measured apart.
template <int R0, int TILES>
__global__ __launch_bounds__(TILES == 1 || R0 <= 8 ? 1024 : 512, TILES == 1 || R0 <= 8 ? 4 : 3) void k_pair_cols_r(
    const float2* __restrict__ spectra, size_t spec_stride, const int2* __restrict__ pairs,
    int npairs, const float* __restrict__ wxy, int n, int box, float2* __restrict__ tbuf,
    const float2* __restrict__ tw, int kxb, int nkx) {
  extern __shared__ float4 cols_lds[];
  constexpr int KP = R0 > 8 ? 16 : 8;   // columns of the exchange rows
  constexpr int NH = 16 / KP;           // xi sets side by side
  constexpr int NR = 16 / NH;           // rounds of 4 NH xi
  constexpr int ZB = KP == 16 ? 8192 : 66 * 64;  // exchange bytes per wave
  constexpr int S = R0 / 2;
  const int A = n / R0, nw = (A + 63) / 64, H = n / 2 + 1, nt = nw * 64;
  const int LC = ((A + nw - 1) / nw + 1) / 2 * 2;  // xi per wave, even, <= 64
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  // loads: lane (h, i) takes xi = x0, x0 + 1 in the rows r = s + S h; after the
  // swap it holds xi = x0 + h in all rows.  An odd A's last pair starts one
  // element early: its first element belongs to the pair before and gets
  // weight zero.
  const int h = l >> 5, i = l & 31;
  auto pair_start = [&](int ii) {
    const int x = w * LC + 2 * ii;
    return 2 * ii >= LC || x >= A ? -1 : (x == A - 1 ? x - 1 : x);
  };
  const int x0 = pair_start(i);
  const bool own = x0 >= 0, twice = own && x0 != w * LC + 2 * i;
  const int voff = own ? 8 * (x0 + S * A * h) : n * 8;  // past the end: reads zero
  const int xi = own ? x0 + h : 0;
  const int ori = (n - box) / 2, c = ori % R0, base = ori - c, G = (box + R0 - 1) / R0;
  float wy[R0];
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int e = 0; e < 2; e++)
      wy[s + S * e] = own && !(twice && e == 0) ? wxy[H + x0 + e + A * (s + S * h)] : 0.f;
  float2 tk[R0];
#pragma unroll
  for (int k = 0; k < R0; k++) {
    const int e = xi * (k + (k < c ? R0 : 0));  // below 2 n
    tk[k] = tw[e < n ? e : e - n];
  }
  // matrix rows m = l % 16: (re, im) of group 8 tile + m / 2 at the xi of
  // exchange row 4 q + l / 16
  float P[NR][TILES];
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const int row = 4 * q + (l >> 4), xs = pair_start(row & 31);
    const unsigned x = xs < 0 ? 0 : xs + (row >> 5);
#pragma unroll
    for (int t = 0; t < TILES; t++) {
      const int g = 8 * t + ((l & 15) >> 1);
      // x < 1024 and n < 2^15: the product fits 32 bits
      const float2 f = g < G ? tw[x * (unsigned)(base + R0 * g) % (unsigned)n] : make_float2(0.f, 0.f);
      P[q][t] = (l & 1) ? f.y : f.x;
    }
  }
  const int kl = l & (KP - 1), hf = (l >> 3) & (NH - 1), al = l >> 4;
  // the second set's factor e^{2 pi i (base + R0 g)/n} for this lane's groups
  float2 cf[TILES][2];
#pragma unroll
  for (int t = 0; t < TILES; t++)
#pragma unroll
    for (int e = 0; e < 2; e++)
      cf[t][e] = hf ? tw[(base + R0 * (8 * t + 2 * al + e)) % n] : make_float2(1.f, 0.f);
  // exchange row l (lane order), 16-byte slots permuted: by l mod 8 (KP = 16),
  // by (l / 4) mod 4 with the second 32 rows two rows further (KP = 8)
  const int zb = w * ZB + (KP == 16 ? l * 128 + (l & 7) * 16 : (l + 2 * h) * 64 + ((l >> 2) & 3) * 16);
  const int rd = KP == 16 ? w * ZB + al * 128 + (((kl >> 1) ^ al) << 4) + (kl & 1) * 8
                          : w * ZB + (al + 34 * hf) * 64 + ((kl >> 1) << 4) + (kl & 1) * 8;
  float4* red = reinterpret_cast<float4*>(reinterpret_cast<char*>(cols_lds) + nw * ZB);
  const int xcd = blockIdx.x % 8, lid = blockIdx.x / 8, nper = gridDim.x / 8;
  const long long items = (long long)npairs * nkx;
  const int i1 = (int)(items * (xcd + 1) / 8);
  int it = (int)(items * xcd / 8) + lid;
  if (it >= i1) return;
  int kx = it / npairs, p = it - kx * npairs;
  const int dkx = nper / npairs, dp = nper - dkx * npairs;
  for (int par = 0;; par ^= nw * TILES * 64) {
    const int2 pr = pairs[p];
    const auto qa = buf_rsrc(spectra + (size_t)pr.x * spec_stride + (size_t)(kxb + kx) * n, n * 8);
    const auto qb = buf_rsrc(spectra + (size_t)pr.y * spec_stride + (size_t)(kxb + kx) * n, n * 8);
    float4 ra[S], rb[S];
    float2 v[R0];
    auto load = [&](int s) {
      ra[s] = buf_ld4(qa, voff, 8 * A * s);
      rb[s] = buf_ld4(qb, voff, 8 * A * s);
    };
    constexpr int D = S < 7 ? S : 7;  // as in k_pair_cols64
#pragma unroll
    for (int s = 0; s < D; s++) {
      load(s);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < S; s++) {
      v[s] = cscale(cmulc(make_float2(ra[s].x, ra[s].y), make_float2(rb[s].x, rb[s].y)), wy[s]);
      v[s + S] = cscale(cmulc(make_float2(ra[s].z, ra[s].w), make_float2(rb[s].z, rb[s].w)), wy[s + S]);
      swap32(v[s].x, v[s + S].x);
      swap32(v[s].y, v[s + S].y);
      if (s + D < S) load(s + D);
      __builtin_amdgcn_sched_barrier(0);
    }
    dft<R0, 1>(v);
#pragma unroll
    for (int k = 0; k < R0; k++) v[k] = cmul(v[k], tk[k]);
    int za = zb;
    asm volatile("" : "+v"(za));
#pragma unroll
    for (int e = 0; e < R0 / 2; e++)
      *reinterpret_cast<float4*>(reinterpret_cast<char*>(cols_lds) + (za ^ (16 * e))) =
          make_float4(v[2 * e].x, v[2 * e].y, v[2 * e + 1].x, v[2 * e + 1].y);
    wave_fence();
    v4f D1[TILES], D2[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++) D1[t] = D2[t] = v4f{0.f, 0.f, 0.f, 0.f};
    int ra0 = rd;
    asm volatile("" : "+v"(ra0));
#pragma unroll
    for (int q = 0; q < NR; q++) {
      // rounds whose rows hold no xi of any wave are skipped
      if (2 * ((4 * q) & 31) >= LC) continue;
      const int ad = KP == 16 ? (ra0 ^ ((q & 1) << 6)) + 512 * q : (ra0 ^ ((q & 3) << 4)) + 256 * q;
      const float2 u = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(cols_lds) + ad);
#pragma unroll
      for (int t = 0; t < TILES; t++) {
        D1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(P[q][t], u.x, D1[t], 0, 0, 0);
        D2[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(P[q][t], u.y, D2[t], 0, 0, 0);
      }
    }
    wave_fence();
    int lt;  // the lane, made again per item: one register less in the loop
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lt));
#pragma unroll
    for (int t = 0; t < TILES; t++) {
      float2 a = make_float2(D1[t][0] - D2[t][1], D1[t][1] + D2[t][0]);
      float2 b = make_float2(D1[t][2] - D2[t][3], D1[t][3] + D2[t][2]);
      if constexpr (NH == 2) {
        a = cmul(a, cf[t][0]);
        b = cmul(b, cf[t][1]);
      }
      red[par + (w * TILES + t) * 64 + lt] = make_float4(a.x, a.y, b.x, b.y);
    }
    if (nw > 1) lds_barrier();
    else wave_fence();
    const float wx = wxy[kxb + kx];
    const float2* rp = reinterpret_cast<const float2*>(red + par);
    const auto qt = buf_rsrc(tbuf + ((size_t)p * H + kxb + kx) * box, box * 8);
    for (int r = w * 64 + lt; r < box; r += nt) {
      const int g = r / R0, kk = r - g * R0 + c, k = kk < R0 ? kk : kk - R0;
      const int o = ((g >> 3) * 64 + ((g & 7) >> 1) * 16 + k) * 2 + (g & 1);
      float2 s = make_float2(0.f, 0.f);
      for (int x = 0; x < nw; x++)
#pragma unroll
        for (int e = 0; e < NH; e++) s = cadd(s, rp[x * (TILES * 128) + o + 16 * e]);
      buf_st2(qt, 8 * r, cscale(s, wx));
    }
    it += nper;
    if (it >= i1) break;
    kx += dkx;
    p += dp;
    if (p >= npairs) {
      p -= npairs;
      kx++;
    }
  }
}

// Resident workgroups of a persistent launch of nw waves with dynamic LDS, asked
// once per kernel, device and workgroup size.  The kernel's LDS limit is always
// set to the most that any size needs: a call with fewer waves does not lower it
// for a grid that is in the cache.
template <class K>
static hipError_t cols_grid(K kernel, int nw, size_t lds, std::atomic<int> (&cache)[16][17], int* grid) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::atomic<int>& c = cache[dev >= 0 && dev < 16 ? dev : 0][nw];
  *grid = c.load(std::memory_order_relaxed);
  if (*grid > 0) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)COLS_LDS_MAX);
  if (e != hipSuccess) return e;
  *grid = persistent_grid(kernel, nw * 64, lds);
  c.store(*grid, std::memory_order_relaxed);
  return hipSuccess;
}

// kx segments of a persistent column-pass launch: about 128 items per
// workgroup each, at most 8.  Within one launch the workgroups of an XCD
// drift apart as they go, and the frame columns of the kx values in flight
// outgrow its L2; a new launch lines them up again (3838x3710x40: 2.90 ms in
// one launch, 2.64 in four, measured on the 16-point form).
int col_segments(int npairs, int H, int grid) {
  const long long per_wg = (long long)npairs * H / std::max(1, grid);
  return (int)std::max(1LL, std::min(8LL, (per_wg + 64) / 128));
}

template <class K, class F>
static hipError_t cols_launches(K kernel, int nw, size_t lds, std::atomic<int> (&cache)[16][17],
                                int npairs, int H, F&& launch) {
  int grid = 0;
  const hipError_t e = cols_grid(kernel, nw, lds, cache, &grid);
  if (e != hipSuccess) return e;
  const int S = col_segments(npairs, H, grid);
  for (int s = 0; s < S; s++) {
    const int kxb = H * s / S, nkx = H * (s + 1) / S - kxb;
    // no more workgroups than items
    const long long items = ((long long)npairs * nkx + 7) / 8 * 8;
    launch((int)std::min<long long>(grid, items), kxb, nkx);
  }
  return hipGetLastError();
}

template <int NG>
static hipError_t cols64(const float2* spectra, size_t spec_stride, const int2* pairs, int npairs,
                         const float* wxy, int n, int box, float2* tbuf, const float2* tw,
                         hipStream_t st) {
  static std::atomic<int> cache[16][17];
  const int nw = (n / 64 + 15) / 16;
  const size_t lds = (size_t)nw * (8192 + (NG > 8 ? 4096 : 2048));
  return cols_launches(k_pair_cols64<NG>, nw, lds, cache, npairs, n / 2 + 1,
                       [&](int grid, int kxb, int nkx) {
                         hipLaunchKernelGGL(k_pair_cols64<NG>, dim3(grid), dim3(nw * 64), lds, st,
                                            spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf,
                                            tw, kxb, nkx);
                       });
}

template <int R0, int TILES>
static hipError_t cols_r(const float2* spectra, size_t spec_stride, const int2* pairs, int npairs,
                         const float* wxy, int n, int box, float2* tbuf, const float2* tw,
                         hipStream_t st) {
  static std::atomic<int> cache[16][17];
  const int nw = cols_r_waves(n, R0);
  const size_t lds = cols_r_lds(n, R0, TILES);
  return cols_launches(k_pair_cols_r<R0, TILES>, nw, lds, cache, npairs, n / 2 + 1,
                       [&](int grid, int kxb, int nkx) {
                         hipLaunchKernelGGL((k_pair_cols_r<R0, TILES>), dim3(grid), dim3(nw * 64), lds,
                                            st, spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf,
                                            tw, kxb, nkx);
                       });
}

hipError_t launch_pair_cols_fp32(const float2* spectra, size_t spec_stride, const int2* pairs,
                                 int npairs, const float* wxy, int n, int box, float2* tbuf,
                                 hipStream_t st) {
  const float2* tw = twiddles(n);
  if (!tw) return hipErrorOutOfMemory;
  if (n % 128 == 0 && box <= 256) {
    if (box <= 96) return cols64<6>(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, tw, st);
    if (box > 128)
      return cols64<16>(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, tw, st);
    return cols64<8>(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, tw, st);
  }
  int tiles = 0;
  const int R0 = cols_radix(n, box, &tiles);
  switch (R0 * 4 + tiles) {
#define MC_COLS_R(R, T) \
  case R * 4 + T: return cols_r<R, T>(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, tw, st);
    MC_COLS_R(16, 1) MC_COLS_R(16, 2) MC_COLS_R(14, 1) MC_COLS_R(14, 2) MC_COLS_R(12, 1)
    MC_COLS_R(12, 2) MC_COLS_R(10, 1) MC_COLS_R(10, 2) MC_COLS_R(8, 1) MC_COLS_R(8, 2)
    MC_COLS_R(8, 3) MC_COLS_R(6, 1) MC_COLS_R(6, 2) MC_COLS_R(6, 3)
#undef MC_COLS_R
    default: break;
  }
  return launch_pair_cols_czt(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, st);
}

}  // namespace mc
