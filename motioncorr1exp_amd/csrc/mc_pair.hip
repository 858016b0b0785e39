// mc_pair.hip -- B-factor-weighted cross-power of frame pairs and the pruned
// inverse that produces only the box x box window of each correlation map.
//
// Reference: cuShiftCC (cufunc.cu:343-361, called with sx = sy = 0 at
// DFAlign.cu:894,1006) forms dfft <- dsum * conj(dfft) * z / sizec with
// z = (-1)^{x+y'} exp(-B (x^2+y'^2)/(2 n^2)) (MkPosList, cufunc.cu:309-341);
// a full n x n C2R follows (DFAlign.cu:897,1008) and only the central box is
// read back (FindShift, cufunc.cu:398-407).  Here the product, the weight
// and the inverse restricted to the box are fused:
//
//  column pass : T[r], the column inverse at the box rows R_r = (n-box)/2 + r
//    of the product formed on the fly from the two spectra columns (mc_cols.hip).
//  row pass    : C[r][c] = sum_kx a_kx Re(T[kx][r] e^{2 pi i kx R_c/n}) with
//    a_0 = a_{n/2} = 1, a_kx = 2 (the C2R row transform with the DC/Nyquist
//    projection): a real GEMM with K = 2(n/2+1) on the matrix cores.
#include <hip/hip_runtime.h>

#include <atomic>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "mc_device.h"
#include "mc_kernels.h"

namespace mc {

typedef float v4f __attribute__((ext_vector_type(4)));

// MFMA operand and accumulator vectors
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// ----------------------------------------------- MFMA FP16 hi/lo form
// The pruned inverse of a column (T of mc_cols.hip), decimated ky = a + A b
// (A = n/128) into 128-point transforms and a combine, with their first DFT
// stage (16 points, stride 8A in ky) run on the matrix cores.  With
// ky = c + 8A b1 (c in [0, 8A), b1 in [0, 16)) the stage is the complex
// product Z[k1][c] = sum_b1 e^{2 pi i b1 k1/16} X[c + 8A b1], i.e. the real
// product [Zr; Zi] = [[C, -S], [S, C]] [Xr; Xi] with K = 32, on 32-column
// blocks of c.  Operands are split into FP16 pairs x = hi + lo (hi =
// fp16(x), lo = fp16(x - hi)) and multiplied as hi*hi + hi*lo + lo*hi with
// FP32 accumulation (v_mfma_f32_32x32x8f16): relative error about 2^-21 per
// product.  Each column of X is scaled by a power of two that puts its
// largest component in [2^13, 2^14) before the split and unscaled after,
// so the FP16 range never clips.  Stage 2 (radix 8 with twiddles) and the
// combine run on the vector ALUs in FP32 as in the plain form.
// Lane layout (32x32x8 f16): lane l feeds A[l % 32][4 (l / 32) + t] and
// B[4 (l / 32) + t][l % 32], t = 0..3; accumulator v of lane l is
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].
MC_DEV void split_hilo(float x, _Float16& hi, _Float16& lo) {
  hi = (_Float16)x;
  lo = (_Float16)(x - (float)hi);
}

template <int N, int SP>
__global__ __launch_bounds__(256) void k_pair_cols_mfma(const float2* __restrict__ spectra,
                                                        size_t spec_stride,
                                                        const int2* __restrict__ pairs,
                                                        int npairs,
                                                        const float* __restrict__ wxy, int box,
                                                        float2* __restrict__ tbuf,
                                                        const float2* __restrict__ tw,
                                                        int kxb, int nkx) {
  constexpr int NT = 256;
  constexpr int M = 128;
  constexpr int A = N / M;
  constexpr int H = N / 2 + 1;
  constexpr int PB = 4;
  constexpr int TS = lds_len<PB>(M) | 1;
  constexpr int CB = 8 * A / 32;       // 32-column blocks of c (block cb -> wave cb % 4)
  constexpr int CBW = (CB + 3) / 4;    // blocks per wave (at most)
  constexpr int NB1 = A * 16;
  constexpr int P1 = (NB1 + NT - 1) / NT;
  constexpr int AS = A / SP;
  static_assert(CB >= 1 && (8 * A) % 32 == 0 && A % SP == 0, "shape");
  __shared__ float2 buf[A * TS];
  const int tid = threadIdx.x;
  const int wv = tid / 64, l = tid % 64, li = l % 32, lh = l / 32;
  // DFT-16 matrix fragments (rows (k1, re|im), columns (b1, re|im)), hi/lo
  v4h dh[4], dl[4];
  {
    const int i = li;
    const int k1 = i & 15;
    const bool im_row = i >= 16;
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int kg = 8 * ks + 4 * lh + t;
        const int b1 = kg & 15;
        const bool im_col = kg >= 16;
        const float2 e = tw[((b1 * k1) & 15) * (N / 16)];  // (cos, sin)(2 pi b1 k1/16)
        float v;
        if (!im_row) v = im_col ? -e.y : e.x;
        else v = im_col ? e.x : e.y;
        _Float16 h, lo;
        split_hilo(v, h, lo);
        dh[ks][t] = h;
        dl[ks][t] = lo;
      }
  }
  // per-lane ky weights: column c = 32 (wv + 4 u) + li, rows b1 = 4 lh + t
  // and 8 + 4 lh + t
  float wy[CBW][8];
#pragma unroll
  for (int u = 0; u < CBW; u++) {
    const int cb = wv + 4 * u;
    const int c = 32 * (cb < CB ? cb : 0) + li;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const int b1 = (t < 4 ? 0 : 8) + 4 * lh + (t & 3);
      wy[u][t] = wxy[H + c + 8 * A * b1];
    }
  }
  float2 t1[8];
#pragma unroll
  for (int r = 0; r < 8; r++) t1[r] = tw[((tid % 16) * r * (N / M)) % N];
  const int ori = (N - box) / 2;
  const int cr = tid / SP, ch = tid % SP;
  const bool cact = cr < box;
  const int R = ori + (cact ? cr : 0);
  const int Rm = R & (M - 1);
  float2 ctw[AS];
#pragma unroll
  for (int i = 0; i < AS; i++) ctw[i] = tw[((i * SP + ch) * R) % N];
  const int xcd = blockIdx.x % 8, lid = blockIdx.x / 8, nper = gridDim.x / 8;
  const long long items = (long long)npairs * nkx;
  const long long i0 = items * xcd / 8, i1 = items * (xcd + 1) / 8;
  for (long long it = i0 + lid; it < i1; it += nper) {
    const int kx = kxb + (int)(it / npairs), p = (int)(it % npairs);
    const int2 pr = pairs[p];
    const float2* sa = spectra + (size_t)pr.x * spec_stride + (size_t)kx * N;
    const float2* sb = spectra + (size_t)pr.y * spec_stride + (size_t)kx * N;
    const float wx = wxy[kx];
#pragma unroll
    for (int u = 0; u < CBW; u++) {
      const int cb = wv + 4 * u;
      if (cb >= CB) continue;  // uniform per wave
      const int c = 32 * cb + li;
      float2 x[8];
      float m = 0.f;
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const int b1 = (t < 4 ? 0 : 8) + 4 * lh + (t & 3);
        const int e = c + 8 * A * b1;
        x[t] = cscale(cmulc(sa[e], sb[e]), wx * wy[u][t]);
        m = fmaxf(m, fmaxf(fabsf(x[t].x), fabsf(x[t].y)));
      }
      m = fmaxf(m, __shfl_xor(m, 32));
      int ex = 0;
      (void)frexpf(m, &ex);
      const int sh = m > 0.f ? 14 - ex : 0;
      v4h bh[4], bl[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        _Float16 h, lo;
        split_hilo(ldexpf(x[t].x, sh), h, lo);      // ks 0: Re, b1 = 4 lh + t
        bh[0][t] = h; bl[0][t] = lo;
        split_hilo(ldexpf(x[t + 4].x, sh), h, lo);  // ks 1: Re, b1 = 8 + 4 lh + t
        bh[1][t] = h; bl[1][t] = lo;
        split_hilo(ldexpf(x[t].y, sh), h, lo);      // ks 2: Im
        bh[2][t] = h; bl[2][t] = lo;
        split_hilo(ldexpf(x[t + 4].y, sh), h, lo);  // ks 3: Im
        bh[3][t] = h; bl[3][t] = lo;
      }
      v16f acc;
#pragma unroll
      for (int v = 0; v < 16; v++) acc[v] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        acc = __builtin_amdgcn_mfma_f32_32x32x8f16(dh[ks], bl[ks], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x8f16(dl[ks], bh[ks], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x8f16(dh[ks], bh[ks], acc, 0, 0, 0);
      }
      // rows 8 (v/4) + 4 lh + v%4: Re of k1 for v < 8, Im of the same k1 at v + 8
      const int a = c % A, j = c / A;
#pragma unroll
      for (int v = 0; v < 8; v++) {
        const int k1 = 8 * (v / 4) + 4 * lh + (v % 4);
        buf[a * TS + lix<PB>(16 * j + k1)] = make_float2(ldexpf(acc[v], -sh), ldexpf(acc[v + 8], -sh));
      }
    }
    __syncthreads();
    // ---- stage 1 in place (radix 8, Ns = 16), FP32
#pragma unroll
    for (int pp = 0; pp < P1; pp++) {
      const int q = tid + pp * NT;
      if (NB1 % NT == 0 || q < NB1) {
        const int a = q / 16, j = q % 16;
        float2 v[8];
#pragma unroll
        for (int r = 0; r < 8; r++) v[r] = buf[a * TS + lix<PB>(j + 16 * r)];
#pragma unroll
        for (int r = 1; r < 8; r++) v[r] = cmul(v[r], t1[r]);
        dft8<1>(v);
#pragma unroll
        for (int r = 0; r < 8; r++) buf[a * TS + lix<PB>(j + 16 * r)] = v[r];
      }
    }
    __syncthreads();
    // ---- combine T[R] = sum_a e^{2 pi i a R/N} Y_a[R mod M]
    float2 acc = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < AS; i++) acc = cadd(acc, cmul(ctw[i], buf[(i * SP + ch) * TS + lix<PB>(Rm)]));
#pragma unroll
    for (int o = 1; o < SP; o <<= 1) {
      acc.x += __shfl_xor(acc.x, o);
      acc.y += __shfl_xor(acc.y, o);
    }
    if (cact && ch == 0) tbuf[((size_t)p * H + kx) * box + cr] = acc;
    __syncthreads();  // buf is rewritten by the next item's stage 0
  }
}

// Row pass: per pair the box map is the real product C = A B with
// A[r][(kx, 0|1)] = a_kx (Re, Im) T[kx][r] and B[(kx, 0|1)][c] = (cos, -sin)(2 pi
// kx R_c/n), K = 2(n/2+1) (the row half of the C2R at DFAlign.cu:897 restricted to
// FindShift's box, cufunc.cu:398-407), on FP32 matrix instructions, whose rate
// bounds it.  So it is computed as the even and odd parts about the box's
// centre: with T' = T e^{2 pi i kx c/n}, c = ori + (box - 1)/2, the columns c +- x
// (x = i + 1/2, of an odd box x = i) are
//   E_x -+ O_x,  E_x = sum a_kx Re T' cos(2 pi kx x/n),  O_x = sum a_kx Im T' sin(..),
// half the multiply-adds.  v_mfma_f32_16x16x4: rows r, columns i, four bins per
// instruction; lane l holds T[kx + l / 16][16 i + l % 16] and the factors of its
// bin, D steps ahead in registers, and keeps all 2 MR NC blocks.  No LDS in the
// main loop.  Rows of A past the box repeat the last box row; their outputs are
// never stored.  A workgroup takes 16 MR rows (blockIdx.z).
// The bins of a pair are split over ks workgroups and over the NW waves of each.
// The NW partial maps are summed in LDS, 16 bytes per lane; workgroup s writes
// partial map s of its pair and k_sum_parts adds them.  Bin 0 is added last and
// the partial maps from the highest bins down: the terms grow that way (B-factor
// weight, and the mean of the image in bin 0 is the largest of all), so the
// rounding of the partial sums is that of the correlation itself and not that of
// its constant offset.
// Box 96: 512, 21 pairs 18 us; 1854, 66 pairs 29; 2048, 15 pairs 23, 55 pairs 27;
// 4096, 91 pairs 67.  The product over all columns (32x32x2, 128 bins per wave)
// took 58, 111, 79, 82 and 140; forms staged through LDS or in FP16 pieces more.
template <int MR, int NC, int NW, int D>
__global__ __launch_bounds__(NW * 64, (8 / NW > 1 ? 8 / NW : 1)) void k_pair_rows_stream(
    const float2* __restrict__ tbuf, int n, int box, int ks, float* __restrict__ out,
    const float2* __restrict__ ef, const float2* __restrict__ ph) {
  constexpr int W = 16 * NC;
  const int p = blockIdx.x, s = blockIdx.y, r0 = 16 * MR * blockIdx.z;
  const int H = n / 2 + 1;
  const int wv = threadIdx.x / 64, l = threadIdx.x % 64, li = l % 16, lk = l / 16;
  const int nsub = ks * NW, sub = s * NW + wv;
  const int k0 = (int)((long long)H * sub / nsub), k1 = (int)((long long)H * (sub + 1) / nsub);
  const int kb = k0 > 0 ? k0 : 1;  // bin 0 comes last
  const float2* T = tbuf + (size_t)p * H * box;
  int roff[MR];
#pragma unroll
  for (int i = 0; i < MR; i++) roff[i] = min(r0 + 16 * i + li, box - 1);
  v4f e[MR][NC], o[MR][NC];
#pragma unroll
  for (int i = 0; i < MR; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) e[i][j] = o[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  float2 a[D][MR], b[D][NC], f[D];
  // operands of the bins kx + lk (at most n/2) into slot d; bins at or past
  // `end` get the factor zero
  auto load = [&](int d, int kx, int end) {
    const int kc = min(kx + lk, H - 1);
    const float2* tr = T + (size_t)kc * box;
    const float2* er = ef + (size_t)kc * W + li;
#pragma unroll
    for (int i = 0; i < MR; i++) a[d][i] = tr[roff[i]];
#pragma unroll
    for (int j = 0; j < NC; j++) b[d][j] = er[16 * j];
    f[d] = ph[kx + lk < end ? kc : H];
  };
  auto mul = [&](int d) {
#pragma unroll
    for (int i = 0; i < MR; i++) {
      const float2 t = cmul(a[d][i], f[d]);
#pragma unroll
      for (int j = 0; j < NC; j++) {
        e[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.x, b[d][j].x, e[i][j], 0, 0, 0);
        o[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.y, b[d][j].y, o[i][j], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d, kb + 4 * d, k1);
  const int steps = (k1 - kb + 3) / 4, nfull = steps / D, rem = steps % D;
  for (int it = 0; it < nfull; it++) {
    const int kn = kb + (it + 1) * 4 * D;
#pragma unroll
    for (int d = 0; d < D; d++) {
      mul(d);
      load(d, kn + 4 * d, k1);
      // keeps each step's loads in that step, D steps ahead of their use: the
      // memory clobber stops them sinking into the next iteration, the
      // scheduling barrier stops the MFMAs of later steps moving above them
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < rem) mul(d);
  if (k0 == 0) {
    load(0, 0, 1);
    mul(0);
  }
  // ordered sum of the NW wave maps, high bins first: blocks [E | O][i][j] of
  // 64 lanes x 4
  __shared__ float4 red[2 * MR * NC][64];
  for (int w = NW - 1; w >= 0; w--) {
    if (wv == w) {
#pragma unroll
      for (int i = 0; i < MR; i++)
#pragma unroll
        for (int j = 0; j < NC; j++)
#pragma unroll
          for (int q = 0; q < 2; q++) {
            const v4f v = q ? o[i][j] : e[i][j];
            float4& r = red[(q * MR + i) * NC + j][l];
            float4 x = make_float4(v[0], v[1], v[2], v[3]);
            if (w < NW - 1) {
              const float4 y = r;
              x = make_float4(y.x + x.x, y.y + x.y, y.z + x.z, y.w + x.w);
            }
            r = x;
          }
    }
    __syncthreads();
  }
  // columns c + x: E - O, c - x: E + O
  float* om = out + ((size_t)p * ks + s) * box * box;
  const int half = (box + 1) / 2;
  for (int t = wv; t < MR * NC; t += NW) {
    const float4 x = red[t][l], y = red[MR * NC + t][l];
    const int i = t / NC, c = 16 * (t - i * NC) + li;
    const float E[4] = {x.x, x.y, x.z, x.w}, O[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = r0 + 16 * i + 4 * lk + v;
      if (r < box && c < half) {
        om[(size_t)r * box + box - half + c] = E[v] - O[v];
        om[(size_t)r * box + half - 1 - c] = E[v] + O[v];
      }
    }
  }
}

// out[p][e] = sum_{s < ks} part[p][s][e] (e < m), added from the last s to 0.
__global__ __launch_bounds__(256) void k_sum_parts(const float* __restrict__ part, int ks, int m,
                                                   long long total, float* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const long long p = i / m, e = i % m;
  const float* q = part + p * ks * m + e;
  float v = q[(size_t)(ks - 1) * m];
  for (int s = ks - 2; s >= 0; s--) v += q[(size_t)s * m];
  out[i] = v;
}

// Weight table: wxy[kx] = (-1)^kx exp(m kx^2), kx in [0, n/2]; wxy[n/2+1+ky]
// = (-1)^{y'} exp(m y'^2) / sizec, so z/sizec = wxy[kx] * wxy[n/2+1+ky] with
// m = -0.5 B/n^2 as in MkPosList (cufunc.cu:309-341).
static const float* weights(int n, float bfactor) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, float>, float*> cache;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_tuple(dev, n, bfactor);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  const int H = n / 2 + 1;
  const double m = -0.5 * (double)bfactor / n / n;
  const double sizec = (double)H * n;
  std::vector<float> h(H + n);
  for (int kx = 0; kx < H; kx++) h[kx] = (float)((kx & 1 ? -1.0 : 1.0) * std::exp(m * kx * kx));
  for (int ky = 0; ky < n; ky++) {
    const int yy = ky < n / 2 ? ky : ky - n;
    h[H + ky] = (float)(((yy & 1) ? -1.0 : 1.0) * std::exp(m * (double)yy * yy) / sizec);
  }
  float* d = nullptr;
  if (hipMalloc(&d, sizeof(float) * h.size()) != hipSuccess) return nullptr;
  if (hipMemcpy(d, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(d);
    return nullptr;
  }
  cache[key] = d;
  return d;
}

// Tables of k_pair_rows_stream: per bin kx W columns of a_kx
// (cos, sin)(2 pi kx x_i/n), x_i = i + 1/2 (of an odd box i), a_0 = a_{n/2} = 1,
// a_kx = 2 otherwise, zeros past the half box; then e^{2 pi i kx c/n}, c = ori +
// (box - 1)/2, and a zero.
static const float2* row_twiddles_stream(int n, int box, int W) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int>, float2*> cache;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_tuple(dev, n, box);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  const int H = n / 2 + 1, ori = (n - box) / 2, half = (box + 1) / 2;
  std::vector<float2> h((size_t)H * W + H + 1, make_float2(0.f, 0.f));
  const double u = M_PI / n;  // angles in units of pi/n, reduced mod 2 n
  for (int kx = 0; kx < H; kx++) {
    const float al = (kx == 0 || 2 * kx == n) ? 1.f : 2.f;
    for (int i = 0; i < half; i++) {
      const double a = u * (double)(((long long)kx * (2 * i + (box % 2 ? 0 : 1))) % (2 * n));
      h[(size_t)kx * W + i] = make_float2(al * (float)cos(a), al * (float)sin(a));
    }
    const double c = u * (double)(((long long)kx * (2 * ori + box - 1)) % (2 * n));
    h[(size_t)H * W + kx] = make_float2((float)cos(c), (float)sin(c));
  }
  float2* d = nullptr;
  if (hipMalloc(&d, sizeof(float2) * h.size()) != hipSuccess) return nullptr;
  if (hipMemcpy(d, h.data(), sizeof(float2) * h.size(), hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(d);
    return nullptr;
  }
  cache[key] = d;
  return d;
}

// Waves per workgroup of the row pass; two workgroups share a CU.
constexpr int ROWS_NW = 4;

// K splits of the row pass: ks = clamp((n/2+1)/256, 2, 8), so that a wave walks
// about 64 bins (128: 2048, 15 pairs 33 us against 23; 32: 4096, 91 pairs the
// same).  The split fixes the order in which the FP32 partial products of a box
// map are added, so it depends on the transform size alone: a pair gives the
// same map whatever the number of pairs in the launch (one movie or a batch, a
// full pair set or an align-to-sum round) and whatever the device's CU count.
static int pair_rows_splits(int n) { return std::max(2, std::min(8, (n / 2 + 1) / 256)); }

size_t pair_rows_part_elems(int npairs, int n, int box) {
  return (size_t)npairs * pair_rows_splits(n) * box * box;
}

template <int N, int SP>
static hipError_t pair_cols_mfma(const float2* spectra, size_t spec_stride, const int2* pairs,
                                 int npairs, const float* wxy, int box, float2* tbuf,
                                 hipStream_t st) {
  const float2* tw = twiddles(N);
  if (!tw) return hipErrorOutOfMemory;
  static const int g = persistent_grid(k_pair_cols_mfma<N, SP>, 256);
  const int H = N / 2 + 1;
  const int S = col_segments(npairs, H, g);
  for (int sgi = 0; sgi < S; sgi++) {
    const int kxb = H * sgi / S, nkx = H * (sgi + 1) / S - kxb;
    hipLaunchKernelGGL((k_pair_cols_mfma<N, SP>), dim3(g), dim3(256), 0, st, spectra, spec_stride,
                       pairs, npairs, wxy, box, tbuf, tw, kxb, nkx);
  }
  return hipGetLastError();
}

bool pair_form_supported(int precision, int n, int box) {
  if (precision == 0) return box >= 1 && box <= n && box <= 256 && n >= 64 && n <= 8192 && n % 2 == 0;
  // the hi/lo column kernel needs 32-column blocks of 8 n/128 columns
  if (precision == 1) return n >= 512 && n <= 8192 && n % 512 == 0 && box >= 1 && box <= 96;
  return false;
}

hipError_t launch_pair_cols(const float2* spectra, size_t spec_stride, const int2* pairs,
                            int npairs, int n, float bfactor, int box, float2* tbuf,
                            int precision, hipStream_t st) {
  if (npairs <= 0) return hipSuccess;
  if (!pair_form_supported(precision, n, box)) return hipErrorInvalidValue;
  const float* wxy = weights(n, bfactor);
  if (!wxy) return hipErrorOutOfMemory;
  if (precision == 1) {
    switch (n) {
#define MC_COLS_MFMA(NN) \
  case NN: return box <= 64 ? pair_cols_mfma<NN, 4>(spectra, spec_stride, pairs, npairs, wxy, box, tbuf, st) \
                            : pair_cols_mfma<NN, 2>(spectra, spec_stride, pairs, npairs, wxy, box, tbuf, st);
      MC_COLS_MFMA(512) MC_COLS_MFMA(1024) MC_COLS_MFMA(2048) MC_COLS_MFMA(4096) MC_COLS_MFMA(8192)
      MC_COLS_MFMA(1536) MC_COLS_MFMA(3072) MC_COLS_MFMA(6144) MC_COLS_MFMA(2560)
      MC_COLS_MFMA(5120)
#undef MC_COLS_MFMA
      default: return hipErrorInvalidValue;
    }
  }
  return launch_pair_cols_fp32(spectra, spec_stride, pairs, npairs, wxy, n, box, tbuf, st);
}

template <int MR, int NC, int D>
static hipError_t pair_rows(const float2* tbuf, int npairs, int n, int box, float* part,
                            hipStream_t st) {
  constexpr int W = 16 * NC;
  const float2* ef = row_twiddles_stream(n, box, W);
  if (!ef) return hipErrorOutOfMemory;
  const int ks = pair_rows_splits(n);
  hipLaunchKernelGGL((k_pair_rows_stream<MR, NC, ROWS_NW, D>),
                     dim3(npairs, ks, (box + 16 * MR - 1) / (16 * MR)), dim3(ROWS_NW * 64), 0, st, tbuf,
                     n, box, ks, part, ef, ef + (size_t)(n / 2 + 1) * W);
  return hipGetLastError();
}

// Tiles by the box: all rows up to 96; above, as many rows per workgroup as leave
// the accumulators of its columns in registers (box 200, 4096, 15 pairs: 65 us
// against 2.9 ms on the vector ALU).
hipError_t launch_pair_rows(const float2* tbuf, int npairs, int n, int box, float* boxmaps,
                            float* part, hipStream_t st) {
  if (npairs <= 0) return hipSuccess;
  if (!pair_form_supported(0, n, box) || !part) return hipErrorInvalidValue;
  hipError_t e;
  if (box <= 32) e = pair_rows<2, 1, 6>(tbuf, npairs, n, box, part, st);
  else if (box <= 64) e = pair_rows<4, 2, 4>(tbuf, npairs, n, box, part, st);
  else if (box <= 96) e = pair_rows<6, 3, 3>(tbuf, npairs, n, box, part, st);
  else if (box <= 128) e = pair_rows<4, 4, 3>(tbuf, npairs, n, box, part, st);
  else if (box <= 192) e = pair_rows<3, 6, 3>(tbuf, npairs, n, box, part, st);
  else e = pair_rows<2, 8, 3>(tbuf, npairs, n, box, part, st);
  if (e != hipSuccess) return e;
  const long long total = (long long)npairs * box * box;
  hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, part,
                     pair_rows_splits(n), box * box, total, boxmaps);
  return hipGetLastError();
}

}  // namespace mc
