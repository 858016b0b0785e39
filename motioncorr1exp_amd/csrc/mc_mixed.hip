// mc_mixed.hip -- stage-1 and sum-image transforms at sizes without a
// power-of-two-like plan (cufftPlan2d of any size, DFAlign.cu:586-640,
// 1284-1290): N = F_0 F_1 .. F_(m-1), 2 <= m <= 4, each factor 2..16 or, for
// the larger primes, up to 127 (the 3710 crop of a K2 frame is 53 x 7 x 10,
// 4092 is 31 x 11 x 12, 1854 is 103 x 3 x 6, 7420 is 53 x 10 x 14).
//
// In place in LDS, level by level: with S_i = N/(F_0 .. F_i) and element
// b S_i + a of a sub-transform of length F_i S_i,
//   y[k S_i + a] = w_(F_i S_i)^(a k) sum_b x[b S_i + a] w_(F_i)^(b k),
// and output k_0 + F_0 (k_1 + F_1 (k_2 + ..)) ends at k_0 S_0 + k_1 S_1 + ..
// Factors up to 16 are butterflies in registers, one column a per lane.  A
// larger one is two dense products on FP32 matrix instructions
// (v_mfma_f32_16x16x4): with s_b = x_b + x_(L-b), d_b = x_b - x_(L-b),
//   U = sum_(b <= L/2) cos(2 pi b k/L) s_b,  V = sum_(b <= L/2) sin(..) d_b,
//   y_k = U -+ i V,  y_(L-k) = U +- i V,  k <= L/2,
// rows k, columns 16 DFTs, real and imaginary parts by separate instructions
// that share the coefficients.
//
// What bounds them is issue: a level of a register radix costs about 1.2 clocks
// per element and SIMD, the 53-point matrix level 3.9 (54% of it in the matrix
// unit), loads, unpacking and stores about 4.  Measured per launch, rows and
// columns: 7420 to 3710 (one frame, 8 bit with gain) 168 and 78 us against 366 and
// 256 by the chirp-z convolutions of twice the next power of two; 1854 (13
// frames) 203 and 159 against 341 and 369; 3710 (three frames, gain) 161 and 122
// against 558 and 149 by 53-point direct sums with Stockham transforms of 35 and
// 70 points, whose lanes read the frame, dark and gain pixel by pixel; 4092 (three
// frames) 152 and 123 against 162 and 155.  Two dense levels (53 x 70) took 225
// and 205.  FP64 error: 1.0e-7 to 1.6e-7 of the norm against 1.2e-7 to 2.6e-7.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "mc_device.h"
#include "mc_frames.h"
#include "mc_kernels.h"
#include "mc_mixed_form.h"

namespace mc {

typedef float v4f __attribute__((ext_vector_type(4)));

// A level: factor F, stride S and in LDS elements Sp, nc = N/F columns; mt row
// tiles and ks steps of four terms of a matrix level (mt = 0: registers) with
// e^{2 pi i e/F} at LDS element co; tw: e^{-2 pi i a k/(F S)} at k S + a.
// mF: 2^20/F rounded up; mS, mC: 2^32/S, 2^32/nc rounded up.
struct MixLevel {
  int F, S, Sp, nc, mt, ks, co;
  unsigned mF, mS, mC;
  const float2 *tw, *cs;
};
// R = 1 << lr items of N elements side by side in LDS, item r at r IS, element
// x at x + x/F_(m-1) if the last factor is even and above 4 (pd): the last level
// reads columns of F_(m-1) consecutive elements at odd distances.
struct MixPlan {
  int N, m, pd, IS, lr;
  int dump;     // LDS element that lanes without a result write
  int nt, lds;  // threads per workgroup, LDS bytes
  unsigned mLast;  // mF of the last level
  MixLevel l[4];
};

// Level i by constant indexes: a variable one would put the plan into scratch.
MC_DEV MixLevel mix_lv(const MixPlan& d, int i) {
  return i == 0 ? d.l[0] : i == 1 ? d.l[1] : i == 2 ? d.l[2] : d.l[3];
}

MC_DEV int mix_pos(const MixPlan& d, int x) {  // input element x
  return d.pd ? x + (int)(__umul24(x, d.mLast) >> 20) : x;
}
// LDS element of output k, and of output k's first digits: levels 0 .. m - 2
MC_DEV int mix_at(const MixPlan& d, int k) {
  int p = 0;
#pragma unroll
  for (int i = 0; i < 3; i++)
    if (i < d.m - 1) {
      const int q = (int)(__umul24(k, d.l[i].mF) >> 20);
      p += (k - q * d.l[i].F) * d.l[i].Sp;
      k = q;
    }
  return p + k;
}

// DFT of length L of this lane's column (element b at x[base + str b]) for the
// first 16 MT outputs k <= L/2 and their mirrors L - k, cs[e] = (cos, sin) of
// 2 pi e/L.  out(k[8], ok[8], v[8]) per tile (k = 0 where not ok), after all
// reads of the column.
template <int MT, int SIGN, class Out>
MC_DEV void dense_tile(const float2* x, int base, int str, int L, int ks, unsigned mF,
                       const float2* cs, Out&& out) {
  int l = threadIdx.x & 63;
  // opaque: the compiler would compute the addresses of all tiles of all forms
  // once, before the loops, and spill them
  asm volatile("" : "+v"(l));
  const int kk = l >> 4;
  v4f ur[MT], ui[MT], vr[MT], vi[MT];
  // The coefficient of (k, b) is entry b k mod L.  From the last term to the
  // first: x_0, which may be a spectrum's mean, is added last (the inverse at
  // 762 = 6 x 127 is 1.8e-7 off FP64, 2.7e-7 the other way round).
  int idx[MT], adv[MT];
#pragma unroll
  for (int t = 0; t < MT; t++) {
    ur[t] = ui[t] = vr[t] = vi[t] = v4f{0.f, 0.f, 0.f, 0.f};
    const int k = 16 * t + (l & 15), e = (4 * ks - 4 + kk) * k, f = 4 * k;  // below 2^20/L
    idx[t] = e - (int)(__umul24(e, mF) >> 20) * L;
    adv[t] = f - (int)(__umul24(f, mF) >> 20) * L;
  }
  int p = base + str * (4 * ks - 4 + kk), q = base + str * (L - (4 * ks - 4 + kk));
  for (int i = ks - 1; i >= 0; i--) {
    const int b = 4 * i + kk;
    // x_0 and, of an even L, x_{L/2} have no partner; terms past L/2 are none
    // (their addresses stay in the column: L >= 7)
    float2 f = x[p], h = x[b == 0 ? p : q];
    float2 c[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
      c[t] = cs[idx[t]];
      const unsigned n = idx[t] - adv[t];
      idx[t] = (int)min(n, n + (unsigned)L);
    }
    p -= 4 * str;
    q += 4 * str;
    const bool in = 2 * b <= L, pair = b > 0 && 2 * b < L;
    f = in ? f : make_float2(0.f, 0.f);
    h = pair ? h : make_float2(0.f, 0.f);
    const float2 s = cadd(f, h), e = csub(f, h);
#pragma unroll
    for (int t = 0; t < MT; t++) {
      ur[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[t].x, s.x, ur[t], 0, 0, 0);
      ui[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[t].x, s.y, ui[t], 0, 0, 0);
      vr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[t].y, e.x, vr[t], 0, 0, 0);
      vi[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c[t].y, e.y, vi[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < MT; t++) {
    int k[8];
    bool ok[8];
    float2 v[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int m = 16 * t + 4 * kk + e;
      const float2 u = make_float2(ur[t][e], ui[t][e]);
      const float2 w = SIGN < 0 ? make_float2(vi[t][e], -vr[t][e]) : make_float2(-vi[t][e], vr[t][e]);
      ok[e] = 2 * m <= L;
      ok[e + 4] = m > 0 && 2 * m < L;
      k[e] = ok[e] ? m : 0;
      k[e + 4] = ok[e + 4] ? L - m : 0;
      v[e] = cadd(u, w);
      v[e + 4] = csub(u, w);
    }
    out(k, ok, v);
    __builtin_amdgcn_sched_barrier(0);  // bounds the addresses held at a time
  }
}

template <int SIGN, class Out>
MC_DEV void dense_tile_any(int mt, const float2* x, int base, int str, int L, int ks, unsigned mF,
                           const float2* cs, Out&& out) {
  switch (mt) {
    case 1: dense_tile<1, SIGN>(x, base, str, L, ks, mF, cs, out); break;
    case 2: dense_tile<2, SIGN>(x, base, str, L, ks, mF, cs, out); break;
    case 3: dense_tile<3, SIGN>(x, base, str, L, ks, mF, cs, out); break;
    default: dense_tile<4, SIGN>(x, base, str, L, ks, mF, cs, out); break;
  }
}

template <int R, int SIGN> MC_DEV void mix_dft(float2 (&v)[R]) {
  if constexpr (R == 9 || R == 13) {
    float2 y[R];
    odd_dft<R, SIGN>(v, [&](int k, float2 z) { y[k] = z; });
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = y[k];
  } else if constexpr (R == 15) {
    dft_pfa<3, 5, SIGN>(v);
  } else {
    dft<R, SIGN>(v);
  }
}

// Column c of a level: its item, LDS base, and the offset a (inner levels) or
// the output index of element 0 (last level).
struct MixCol {
  int r, base, a;
};
template <bool LAST> MC_DEV MixCol mix_col(const MixPlan& d, const MixLevel& v, int c) {
  MixCol o;
  o.r = (int)__umulhi((unsigned)c, v.mC);
  c -= o.r * v.nc;
  o.base = o.r * d.IS;
  if (LAST) {  // lanes over the output index: whole lines where it is stored
    o.a = c;
    o.base += mix_at(d, c);
  } else {
    const int p = v.S > 1 ? (int)__umulhi((unsigned)c, v.mS) : c;
    o.a = c - p * v.S;
    o.base += p * v.F * v.Sp + mix_pos(d, o.a);
  }
  return o;
}

// Register level of radix R.  Inner levels multiply by the factors and write
// back; the last hands out(true, item, k, LDS element, value) the outputs k.
template <int R, int SIGN, bool LAST, class Out>
MC_DEV void mix_radix(float2* buf, const MixPlan& d, const MixLevel& lv, int total, Out&& out) {
  const int S = lv.S, Sp = lv.Sp;
  const __amdgpu_buffer_rsrc_t tw = buf_rsrc(lv.tw, LAST ? 0 : R * S * 8);
#pragma unroll 1
  for (int c = threadIdx.x; c < total; c += blockDim.x) {
    const MixCol o = mix_col<LAST>(d, lv, c);
    float2 v[R], t[R];
    if (!LAST)
#pragma unroll
      for (int k = 1; k < R; k++) t[k] = buf_ld2(tw, 8 * o.a, 8 * k * S);
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = buf[o.base + k * Sp];
    mix_dft<R, SIGN>(v);
    if (LAST) {
#pragma unroll
      for (int k = 0; k < R; k++) out(true, o.r, o.a + k * lv.nc, o.base + k, v[k]);
    } else {
      buf[o.base] = v[0];
#pragma unroll
      for (int k = 1; k < R; k++)
        buf[o.base + k * Sp] = SIGN < 0 ? cmul(v[k], t[k]) : cmulc(v[k], t[k]);
    }
  }
}

// Matrix level: 16 columns per wave at a time.
template <int SIGN, bool LAST, class Out>
MC_DEV void mix_dense(float2* buf, const MixPlan& d, const MixLevel& lv, int total, Out&& out) {
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6, l15 = threadIdx.x & 15;
  const int F = lv.F, S = lv.S, Sp = lv.Sp;
  const __amdgpu_buffer_rsrc_t tw = buf_rsrc(lv.tw, LAST ? 0 : F * S * 8);
#pragma unroll 1
  for (int c0 = 16 * w; c0 < total; c0 += 16 * nw) {
    // lanes past the last column repeat it (same wave) and store nothing
    const bool own = c0 + l15 < total;
    const MixCol o = mix_col<LAST>(d, lv, own ? c0 + l15 : total - 1);
    dense_tile_any<SIGN>(
        lv.mt, buf, o.base, Sp, F, lv.ks, lv.mF, buf + lv.co,
        [&](const int (&k)[8], const bool (&ok)[8], const float2 (&v)[8]) {
          if (LAST) {
#pragma unroll
            for (int e = 0; e < 8; e++)
              out(ok[e] && own, o.r, o.a + k[e] * lv.nc, ok[e] && own ? o.base + k[e] : d.dump, v[e]);
          } else {
            float2 t[8];
#pragma unroll
            for (int e = 0; e < 8; e++) t[e] = buf_ld2(tw, 8 * (o.a + k[e] * S), 0);
#pragma unroll
            for (int e = 0; e < 8; e++)
              buf[ok[e] && own ? o.base + k[e] * Sp : d.dump] =
                  SIGN < 0 ? cmul(v[e], t[e]) : cmulc(v[e], t[e]);
          }
        });
  }
}

template <int SIGN, bool LAST, class Out>
MC_DEV void mix_level(float2* buf, const MixPlan& d, int i, int nr, Out&& out) {
  const MixLevel lv = mix_lv(d, i);
  const int total = nr * lv.nc;
  if (lv.mt) {
    mix_dense<SIGN, LAST>(buf, d, lv, total, out);
    return;
  }
  switch (lv.F) {
#define MC_MIX(R) case R: mix_radix<R, SIGN, LAST>(buf, d, lv, total, out); break;
    MC_MIX(2) MC_MIX(3) MC_MIX(4) MC_MIX(5) MC_MIX(6) MC_MIX(7) MC_MIX(8) MC_MIX(9) MC_MIX(10)
    MC_MIX(11) MC_MIX(12) MC_MIX(13) MC_MIX(14) MC_MIX(15) MC_MIX(16)
#undef MC_MIX
  }
}

// The dense levels' tables, behind the items: read before mix_transform's barrier.
MC_DEV void mix_load_tables(float2* buf, const MixPlan& d) {
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i < d.m && d.l[i].mt)
      for (int e = threadIdx.x; e < d.l[i].F; e += blockDim.x) buf[d.l[i].co + e] = d.l[i].cs[e];
}

// All levels on the first nr items; out(ok, item, k, LDS element of output k,
// value) of the last.  The caller has a barrier before and, if it reads LDS, after.
template <int SIGN, class Out>
MC_DEV void mix_transform(float2* buf, const MixPlan& d, int nr, Out&& out) {
#pragma unroll 1
  for (int i = 0; i < d.m - 1; i++) {
    mix_level<SIGN, false>(buf, d, i, nr, [](bool, int, int, int, float2) {});
    __syncthreads();
  }
  mix_level<SIGN, true>(buf, d, d.m - 1, nr, out);
}

// ------------------------------------------------------------ stage-1 rows
// Pixels x .. x + 3 of canvas row y, all inside the data region, no stretch.
// One load each of frame, dark and gain, at any alignment.
template <int DT>
struct Px4 {
  typedef typename Elem<DT>::T T;
  T v[4];
  float d[4], g[4];
  MC_DEV void load(const R2CGeom& q, const char* fbase, int x, int y) {
    const size_t X = q.offx + x, Y = q.offy + y;
    __builtin_memcpy(v, reinterpret_cast<const T*>(fbase + Y * q.row_pitch) + X, sizeof v);
    if (q.dark) __builtin_memcpy(d, q.dark + Y * q.nx + X, sizeof d);
    if (q.gain) __builtin_memcpy(g, q.gain + Y * q.nx + X, sizeof g);
  }
  MC_DEV float at(const R2CGeom& q, int e) const {
    return correct(q, (float)v[e], q.dark ? d[e] : 0.f, q.gain ? g[e] : 1.f);
  }
};

template <int DT>
MC_DEV void mix_load_rows(const R2CGeom& g, const MixPlan& d, const char* fbase, int y0, int nr,
                          float2* buf) {
  const int tr = blockDim.x >> d.lr, r = threadIdx.x / tr, t = threadIdx.x - r * tr, N = d.N;
  if (r >= nr) return;
  const bool stretch = g.xs < 1.f || g.ys < 1.f;
  const int full = stretch ? 0 : g.w / 4;  // groups of four pixels inside the region
  float2* b = buf + r * d.IS;
  constexpr int U = 4;
  for (int i0 = t; i0 < full; i0 += U * tr) {
    Px4<DT> v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u].load(g, fbase, 4 * min(i0 + u * tr, full - 1), y0 + r);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int m = 2 * min(i0 + u * tr, full - 1);
      b[mix_pos(d, m)] = make_float2(v[u].at(g, 0), v[u].at(g, 1));
      b[mix_pos(d, m + 1)] = make_float2(v[u].at(g, 2), v[u].at(g, 3));
    }
  }
  const bool corr = g.dark || g.gain || stretch;
  for (int m = 2 * full + t; m < N; m += tr)
    b[mix_pos(d, m)] = make_float2(row_px<DT>(g, fbase, corr, 2 * m, y0 + r),
                                   row_px<DT>(g, fbase, corr, 2 * m + 1, y0 + r));
}

// Rows y0 .. of one frame: the row packed into N = nu/2 complex values, the
// DFT, and the unpack to the kept bins kx < nkx, RT[kx/4][y][kx%4].
__global__ __launch_bounds__(512, 4) void k_r2c_rows_mix(R2CGeom g, MixPlan d, int f0, int nkx,
                                                           float2* __restrict__ rt, size_t rt_fstride,
                                                           float* __restrict__ rowsum,
                                                           const float2* __restrict__ twnu) {
  extern __shared__ float4 mix_lds[];
  float2* buf = reinterpret_cast<float2*>(mix_lds);
  mix_load_tables(buf, d);
  const int NT = blockDim.x, R = 1 << d.lr, N = d.N, NU = 2 * N;
  const int ng = (g.h + R - 1) >> d.lr;
  const int L = xcd_remap(blockIdx.x, gridDim.x), f = L / ng, y0 = (L - f * ng) << d.lr;
  const int nr = min(R, g.h - y0);
  const char* fbase = g.src + (size_t)(f0 + f) * g.frame_pitch;
  switch (g.dtype) {
#define MC_LR(D) case D: mix_load_rows<D>(g, d, fbase, y0, nr, buf); break;
    MC_LR(DT_INT8) MC_LR(DT_UINT8) MC_LR(DT_INT16) MC_LR(DT_UINT16) MC_LR(DT_FLOAT32)
#undef MC_LR
  }
  __syncthreads();
  mix_transform<-1>(buf, d, nr, [&](bool, int, int, int at, float2 v) { buf[at] = v; });
  __syncthreads();
  // X[k] = E + e^{-2 pi i k/NU} O with E, O from Z[k], Z[N - k], which give
  // X[N - k] too; lanes over four bins, then the rows: whole lines of RT
  float2* out = rt + (size_t)f * rt_fstride;
  const int nk = min(nkx - 1, N / 2) + 1;
  for (int i = threadIdx.x; i < ((nk + 3) >> 2) << (2 + d.lr); i += NT) {
    const int r = (i >> 2) & (R - 1), k = ((i >> (2 + d.lr)) << 2) + (i & 3);
    if (r >= nr || k >= nk) continue;
    const float2* b = buf + r * d.IS;
    const float2 zk = b[mix_at(d, k)], zc = cconj(b[mix_at(d, k ? N - k : 0)]);
    const float2 E = cscale(cadd(zk, zc), 0.5f);
    const float2 D = csub(zk, zc);
    const float2 O = make_float2(0.5f * D.y, -0.5f * D.x);
    const float2 X = cadd(E, cmul(cconj(twnu[k]), O));
    float2* o = out + (size_t)(y0 + r) * 4;
    o[(size_t)(k >> 2) * NU * 4 + (k & 3)] = X;
    if (k == 0 && rowsum) rowsum[(size_t)f * NU + y0 + r] = X.x;
    const int m = N - k;
    if (m < nkx && m != k) {
      const float2 Y = k ? cadd(cconj(E), cmul(cconj(twnu[m]), make_float2(O.x, -O.y))) : csub(E, O);
      o[(size_t)(m >> 2) * NU * 4 + (m & 3)] = Y;
    }
  }
}

// --------------------------------------------------------- stage-1 columns
// Columns kx0 .. of one frame: rows [0, h) of the row pass (the rest of the
// canvas zero, or the fill times the spectrum P of the fill mask), the DFT, and
// the rows of the Fourier crop to n.
__global__ __launch_bounds__(512, 4) void k_c2c_cols_mix(const float2* __restrict__ rt,
                                                           size_t rt_fstride, MixPlan d, int nkx,
                                                           int h_data, const float* __restrict__ fill,
                                                           const float2* __restrict__ padP, int n,
                                                           float2* __restrict__ spec,
                                                           size_t spec_stride) {
  extern __shared__ float4 mix_lds[];
  float2* buf = reinterpret_cast<float2*>(mix_lds);
  mix_load_tables(buf, d);
  const int NT = blockDim.x, R = 1 << d.lr, N = d.N;
  const int ng = (nkx + R - 1) >> d.lr;
  const int L = xcd_remap(blockIdx.x, gridDim.x), f = L / ng, kx0 = (L - f * ng) << d.lr;
  const int nr = min(R, nkx - kx0);
  const float2* src = rt + (size_t)f * rt_fstride + (size_t)(kx0 >> 2) * N * 4 + (kx0 & 3);
  const float fv = fill ? fill[f] : 0.f;
  constexpr int U = 8;
  if (R > 1) {  // two columns per load (the scratch holds whole groups of four)
    const int lh = d.lr - 1, total = h_data << lh;
    for (int i0 = threadIdx.x; i0 < total; i0 += U * NT) {
      float4 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int i = min(i0 + u * NT, total - 1), y = i >> lh, c = 2 * (i - (y << lh));
        v[u] = *reinterpret_cast<const float4*>(src + (size_t)y * 4 + c);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int i = min(i0 + u * NT, total - 1), y = i >> lh, c = 2 * (i - (y << lh));
        float2* b = buf + c * d.IS + mix_pos(d, y);
        b[0] = make_float2(v[u].x, v[u].y);
        b[d.IS] = make_float2(v[u].z, v[u].w);
      }
    }
  } else {
    for (int i0 = threadIdx.x; i0 < h_data; i0 += U * NT) {
      float2 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = src[(size_t)min(i0 + u * NT, h_data - 1) * 4];
#pragma unroll
      for (int u = 0; u < U; u++) buf[mix_pos(d, min(i0 + u * NT, h_data - 1))] = v[u];
    }
  }
  if (fill || h_data < N) {
    for (int r = 0; r < nr; r++)
      for (int y = h_data + threadIdx.x; y < N; y += NT)
        buf[r * d.IS + mix_pos(d, y)] = make_float2(kx0 + r == 0 ? fv * (float)N : 0.f, 0.f);
    if (fill) {
      __syncthreads();
      for (int r = 0; r < nr; r++) {
        const float2 P = cscale(padP[kx0 + r], fv);
        for (int y = threadIdx.x; y < h_data; y += NT) {
          float2* b = buf + r * d.IS + mix_pos(d, y);
          *b = cadd(*b, P);
        }
      }
    }
  }
  __syncthreads();
  // stores past the buffer's end are dropped: the outputs that are not kept
  const auto dst = buf_rsrc(spec + (size_t)f * spec_stride + (size_t)kx0 * n, nr * n * 8);
  mix_transform<-1>(buf, d, nr, [&](bool ok, int r, int k, int, float2 v) {
    const int o = k < n / 2 ? k : k - (N - n);
    ok = ok && (k < n / 2 || k >= N - n / 2);
    buf_st2(dst, ok ? 8 * (r * n + o) : nr * n * 8, v);
  });
}

// ----------------------------------------------- sum image: columns and rows
__global__ __launch_bounds__(512, 4) void k_cols_inv_mix(const float2* __restrict__ spec,
                                                           MixPlan d, float2* __restrict__ tmp) {
  extern __shared__ float4 mix_lds[];
  float2* buf = reinterpret_cast<float2*>(mix_lds);
  mix_load_tables(buf, d);
  const int NT = blockDim.x, R = 1 << d.lr, N = d.N, nkx = N / 2 + 1;
  const int kx0 = xcd_remap(blockIdx.x, gridDim.x) << d.lr, nr = min(R, nkx - kx0);
  for (int r = 0; r < nr; r++)
    for (int i = threadIdx.x; i < N; i += NT)
      buf[r * d.IS + mix_pos(d, i)] = spec[(size_t)(kx0 + r) * N + i];
  __syncthreads();
  mix_transform<1>(buf, d, nr, [&](bool, int, int, int at, float2 v) { buf[at] = v; });
  __syncthreads();
  float2* dst = tmp + (size_t)(kx0 >> 2) * N * 4 + (kx0 & 3);
  for (int i = threadIdx.x; i < N << d.lr; i += NT) {
    const int y = i >> d.lr, r = i & (R - 1);
    if (r < nr) dst[(size_t)y * 4 + r] = buf[r * d.IS + mix_at(d, y)];
  }
}

// Z[k] = (X[k] + conj X[N-k]) + i e^{+2 pi i k/2N} (X[k] - conj X[N-k]), the
// inverse DFT of length N = n/2, x *= scale.
__global__ __launch_bounds__(512, 4) void k_c2r_rows_mix(const float2* __restrict__ tmp, MixPlan d,
                                                           float scale, float* __restrict__ img,
                                                           size_t pitch,
                                                           const float2* __restrict__ twn) {
  extern __shared__ float4 mix_lds[];
  float2* buf = reinterpret_cast<float2*>(mix_lds);
  mix_load_tables(buf, d);
  const int NT = blockDim.x, R = 1 << d.lr, N = d.N, n = 2 * N;
  const int y0 = xcd_remap(blockIdx.x, gridDim.x) << d.lr, nr = min(R, n - y0);
  const int nyq = d.IS - 1;  // X[N], after the item's last element
  for (int i = threadIdx.x; i < ((N + 4) >> 2) * 4 * R; i += NT) {
    const int r = (i >> 2) & (R - 1), k = ((i >> (2 + d.lr)) << 2) + (i & 3);
    if (r >= nr || k > N) continue;
    float2 v = tmp[((size_t)(k >> 2) * n + y0 + r) * 4 + (k & 3)];
    if (k == 0 || k == N) v.y = 0.f;
    buf[r * d.IS + (k < N ? mix_pos(d, k) : nyq)] = v;
  }
  __syncthreads();
  for (int r = 0; r < nr; r++)
    for (int k = threadIdx.x; k <= N / 2; k += NT) {
      float2* pk = buf + r * d.IS + mix_pos(d, k);
      float2* pm = buf + r * d.IS + (k ? mix_pos(d, N - k) : nyq);
      const float2 a = *pk, b = *pm;
      *pk = cadd(cadd(a, cconj(b)), mul_si<1>(cmul(twn[k], csub(a, cconj(b)))));
      if (k != 0 && k != N - k)
        *pm = cadd(cadd(b, cconj(a)), mul_si<1>(cmul(twn[N - k], csub(b, cconj(a)))));
    }
  __syncthreads();
  mix_transform<1>(buf, d, nr, [&](bool, int, int, int at, float2 v) { buf[at] = v; });
  __syncthreads();
  for (int r = 0; r < nr; r++) {
    float2* row = reinterpret_cast<float2*>(img + (size_t)(y0 + r) * pitch);
    for (int m = threadIdx.x; m < N; m += NT) row[m] = cscale(buf[r * d.IS + mix_at(d, m)], scale);
  }
}

// ---------------------------------------------------------------- host part
// Plan of a transform of N elements for `items` of them.  The largest factor
// goes first (its factors w_N are the long table), an even one last (padded to
// odd distances), so that an odd product between them keeps the last level's
// columns in distinct banks.  Items per workgroup: up to 40 KB with four waves,
// or 80 KB with eight above N = 1900 (1854: rows and columns 203 and 159 us
// with the first, 240 and 169 with the second; 4092: 161 and 133, 152 and 123;
// other sizes of the workgroup leave the CU with fewer than 16 waves: 30 to 50%
// slower), fewer items if that leaves less than two workgroups per CU.
static bool mix_plan(int N, long long items, MixPlan* d) {
  int F[4];
  const int m = mix_factors(N, F);  // ascending
  if (!m) return false;
  std::reverse(F, F + m);
  for (int i = 1; i + 1 < m; i++)
    if (F[i] % 2 == 0 && F[m - 1] % 2) std::swap(F[i], F[m - 1]);
  *d = MixPlan{};
  d->N = N;
  d->m = m;
  d->pd = F[m - 1] % 2 == 0 && F[m - 1] >= 6;  // at most 7/6 of the space
  int S = N;
  for (int i = 0; i < m; i++) {
    S /= F[i];
    MixLevel& v = d->l[i];
    v.F = F[i];
    v.S = S;
    v.Sp = i == m - 1 ? 1 : S / F[m - 1] * (F[m - 1] + d->pd);
    v.nc = N / F[i];
    v.mF = ((1u << 20) + F[i] - 1) / F[i];
    v.mS = S > 1 ? (unsigned)(((1ull << 32) + S - 1) / S) : 0;
    v.mC = (unsigned)(((1ull << 32) + v.nc - 1) / v.nc);
    if (i < m - 1 && !(v.tw = qp_twiddles(S, F[i]))) return false;
  }
  d->mLast = d->l[m - 1].mF;
  d->IS = N / F[m - 1] * (F[m - 1] + d->pd) + 1;
  int coef = 0;
  for (int i = 0; i < m; i++)
    if (F[i] > 16) coef += F[i];
  const int cap = N > 1900 ? 80 : 40;
  d->lr = 2;
  while (d->lr > 0 && (((size_t)d->IS << d->lr) + 1 + coef > cap * 1024 / 8 || items >> d->lr < 512))
    d->lr--;
  d->dump = d->IS << d->lr;
  int at = d->dump + 1;
  for (int i = 0; i < m; i++)
    if (F[i] > 16) {
      MixLevel& v = d->l[i];
      v.mt = (F[i] / 2 + 16) / 16;
      v.ks = (F[i] / 2 + 4) / 4;
      v.co = at;
      at += F[i];
      if (!(v.cs = twiddles(F[i]))) return false;
    }
  d->lds = at * 8;
  d->nt = N > 1900 ? 512 : 256;
  return true;
}

template <class K, class... Args>
static hipError_t mix_launch(K kernel, const MixPlan& d, int groups, hipStream_t st, Args... args) {
  if (d.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(groups), dim3(d.nt), d.lds, st, args...);
  return hipGetLastError();
}
static int mix_groups(const MixPlan& d, int items) { return (items + (1 << d.lr) - 1) >> d.lr; }

hipError_t launch_rows_mix(const R2CGeom& g, int f0, int nframes, int nkx, float2* rt,
                           size_t rt_fstride, float* rowsum, hipStream_t st) {
  MixPlan d;
  const float2* twnu = twiddles(g.nu);
  if (!mix_plan(g.nu / 2, (long long)g.h * nframes, &d) || !twnu) return hipErrorOutOfMemory;
  return mix_launch(k_r2c_rows_mix, d, mix_groups(d, g.h) * nframes, st, g, d, f0, nkx, rt, rt_fstride,
                    rowsum, twnu);
}

hipError_t launch_cols_mix(const R2CGeom& g, int nframes, int nkx, const float2* rt,
                           size_t rt_fstride, const float* fill, const float2* padP,
                           float2* spectra, size_t spec_stride, hipStream_t st) {
  MixPlan d;
  if (!mix_plan(g.nu, (long long)nkx * nframes, &d)) return hipErrorOutOfMemory;
  return mix_launch(k_c2c_cols_mix, d, mix_groups(d, nkx) * nframes, st, rt, rt_fstride, d, nkx, g.h,
                    fill, padP, g.n, spectra, spec_stride);
}

hipError_t launch_cols_inv_mix(const float2* spec, int n, float2* tmp, hipStream_t st) {
  MixPlan d;
  if (!mix_plan(n, n / 2 + 1, &d)) return hipErrorOutOfMemory;
  return mix_launch(k_cols_inv_mix, d, mix_groups(d, n / 2 + 1), st, spec, d, tmp);
}

hipError_t launch_c2r_rows_mix(const float2* tmp, int n, float scale, float* img, size_t pitch,
                               hipStream_t st) {
  MixPlan d;
  const float2* twn = twiddles(n);
  if (!mix_plan(n / 2, n, &d) || !twn) return hipErrorOutOfMemory;
  return mix_launch(k_c2r_rows_mix, d, mix_groups(d, n), st, tmp, d, scale, img, pitch, twn);
}

}  // namespace mc
