// mc_sum.hip -- Fourier phase-shift-and-sum of a stack of spectra.
//
// Reference: cuShift (cufunc.cu:372-394) multiplies a frame spectrum by
// e^{i (shx x + shy y')}, shx = sx 2 pi/n, and cuAdd (cufunc.cu:243-252)
// accumulates it into the sum (iteration sums DFAlign.cu:974-989, final sum
// DFAlign.cu:1143-1267).  One pass here reads every frame once and writes
// the sum once: the F shifted spectra are never materialised.  The phase
// (sx kx + sy ky')/n is reduced to [0, 1) in FP64 before the FP32 sincospi,
// so its error does not grow with the shift or the frequency.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mc_device.h"
#include "mc_kernels.h"

namespace mc {

// Element e (kx, yy) of the frames f0 .. f0 + U - 1 times its phase factor.
// All loads are issued together, whatever the shifts are: a test before each
// would make the load wait for the shift (2048, 24 frames: 84 us with the tests,
// 78 without).  NaN: frame not summed, value zero.  y2 is the imaginary part
// with the other of its two products rounded.
template <int U>
MC_DEV void rotate_frames(const float2* __restrict__ spectra, size_t spec_stride,
                          const double2* __restrict__ shifts, int f0, size_t e, int kx, int yy,
                          double inv_n, float2 (&g)[U], float (&y2)[U]) {
  double2 s[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    g[u] = spectra[(size_t)(f0 + u) * spec_stride + e];
    s[u] = shifts[f0 + u];
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    // contractions written out: sum and gradient keep their rounding wherever
    // this is compiled into
    double w = fma(s[u].x, (double)kx, s[u].y * yy);
    w = fma(inv_n, w, -floor(inv_n * w));
    float sn, cs;
    sincospif(2.0f * (float)w, &sn, &cs);
    const float2 v = g[u];
    const bool in = s[u].x == s[u].x;
    g[u].x = in ? fmaf(v.x, cs, -(v.y * sn)) : 0.f;
    g[u].y = in ? fmaf(v.y, cs, v.x * sn) : 0.f;
    y2[u] = in ? fmaf(v.x, sn, v.y * cs) : 0.f;
  }
}
// use(f, value, y2) for all frames in order: groups of eight, of four, single ones
template <class F>
MC_DEV void rotate_all(const float2* __restrict__ spectra, size_t spec_stride,
                       const double2* __restrict__ shifts, int nframes, size_t e, int kx, int yy,
                       double inv_n, F&& use) {
  int f = 0;
  for (; f + 8 <= nframes; f += 8) {
    float2 g[8];
    float y2[8];
    rotate_frames<8>(spectra, spec_stride, shifts, f, e, kx, yy, inv_n, g, y2);
#pragma unroll
    for (int u = 0; u < 8; u++) use(f + u, g[u], y2[u]);
  }
  if (f + 4 <= nframes) {
    float2 g[4];
    float y2[4];
    rotate_frames<4>(spectra, spec_stride, shifts, f, e, kx, yy, inv_n, g, y2);
#pragma unroll
    for (int u = 0; u < 4; u++) use(f + u, g[u], y2[u]);
    f += 4;
  }
  for (; f < nframes; f++) {
    float2 g[1];
    float y2[1];
    rotate_frames<1>(spectra, spec_stride, shifts, f, e, kx, yy, inv_n, g, y2);
    use(f, g[0], y2[0]);
  }
}

__global__ __launch_bounds__(256) void k_shift_sum(const float2* __restrict__ spectra,
                                                   size_t spec_stride, int nframes, int n,
                                                   const double2* __restrict__ shifts,
                                                   float2* __restrict__ sum,
                                                   float2* __restrict__ sum2, int f2_last) {
  const size_t total = (size_t)(n / 2 + 1) * n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  const int kx = (int)(e / n), ky = (int)(e % n);
  const int yy = ky < n / 2 ? ky : ky - n;
  float2 acc = make_float2(0.f, 0.f), acc2 = make_float2(0.f, 0.f);
  rotate_all(spectra, spec_stride, shifts, nframes, e, kx, yy, 1.0 / n, [&](int f, float2 t, float) {
    acc = cadd(acc, t);
    if (sum2 && f <= f2_last) acc2 = cadd(acc2, t);
  });
  sum[e] = acc;
  if (sum2) sum2[e] = acc2;
}

hipError_t launch_shift_sum(const float2* spectra, size_t spec_stride, int nframes, int n,
                            const double2* shifts, float2* sum, float2* sum2, int f2_last,
                            hipStream_t st) {
  const size_t total = (size_t)(n / 2 + 1) * n;
  hipLaunchKernelGGL(k_shift_sum, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     spectra, spec_stride, nframes, n, shifts, sum, sum2, f2_last);
  return hipGetLastError();
}

// Several sums in one launch (one per blockIdx.y): job j = (first slot,
// frame count, first shift, destination slot) sums its frames into its
// destination slot of the same spectrum array.  Destination slots are
// disjoint from every job's frame slots.
__global__ __launch_bounds__(256) void k_shift_sum_multi(float2* spectra, size_t spec_stride,
                                                         int n, const int4* __restrict__ jobs,
                                                         const double2* __restrict__ shifts) {
  const size_t total = (size_t)(n / 2 + 1) * n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  const int4 jb = jobs[blockIdx.y];
  const int kx = (int)(e / n), ky = (int)(e % n);
  const int yy = ky < n / 2 ? ky : ky - n;
  float2 acc = make_float2(0.f, 0.f);
  rotate_all(spectra + (size_t)jb.x * spec_stride, spec_stride, shifts + jb.z, jb.y, e, kx, yy,
             1.0 / n, [&](int, float2 t, float) { acc = cadd(acc, t); });
  spectra[(size_t)jb.w * spec_stride + e] = acc;
}

hipError_t launch_shift_sum_multi(float2* spectra, size_t spec_stride, int n, const int4* jobs,
                                  int njobs, const double2* shifts, hipStream_t st) {
  if (njobs <= 0) return hipSuccess;
  if (njobs > 65535) return hipErrorInvalidValue;
  const size_t total = (size_t)(n / 2 + 1) * n;
  hipLaunchKernelGGL(k_shift_sum_multi, dim3((unsigned)((total + 255) / 256), (unsigned)njobs),
                     dim3(256), 0, st, spectra, spec_stride, n, jobs, shifts);
  return hipGetLastError();
}

// Even/odd half sums of `count` consecutive spectra in one pass (the halves
// of the FSC table): frame f adds to h0 when f is even, else to h1, after its
// phase shift (shifts == nullptr: unshifted; a NaN shift skips the frame).
// Each half accumulates in frame order (DFAlign.cu:808-812 raw halves,
// 1143-1243 aligned halves).  count == 0 writes zeros.
__global__ __launch_bounds__(256) void k_half_sums(const float2* __restrict__ spectra,
                                                   size_t spec_stride, int count, int n,
                                                   const double2* __restrict__ shifts,
                                                   float2* __restrict__ h0,
                                                   float2* __restrict__ h1) {
  const size_t total = (size_t)(n / 2 + 1) * n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  const int kx = (int)(e / n), ky = (int)(e % n);
  const int yy = ky < n / 2 ? ky : ky - n;
  const double inv_n = 1.0 / n;
  float2 acc[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
  constexpr int U = 8;
  for (int f0 = 0; f0 < count; f0 += U) {
    float2 v[U];
    double2 sh[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      sh[u] = f0 + u >= count ? make_double2(NAN, NAN)
                              : (shifts ? shifts[f0 + u] : make_double2(0.0, 0.0));
      v[u] = sh[u].x == sh[u].x ? spectra[(size_t)(f0 + u) * spec_stride + e]
                                : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const double2 s = sh[u];
      if (s.x != s.x) continue;
      float2 t = v[u];
      if (shifts) {
        double w = (s.x * kx + s.y * yy) * inv_n;
        w -= floor(w);
        float sn, cs;
        sincospif(2.0f * (float)w, &sn, &cs);
        t = cmul(t, make_float2(cs, sn));
      }
      acc[(f0 + u) & 1] = cadd(acc[(f0 + u) & 1], t);
    }
  }
  h0[e] = acc[0];
  h1[e] = acc[1];
}

hipError_t launch_half_sums(const float2* spectra, size_t spec_stride, int count, int n,
                            const double2* shifts, float2* h0, float2* h1, hipStream_t st) {
  const size_t total = (size_t)(n / 2 + 1) * n;
  hipLaunchKernelGGL(k_half_sums, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     spectra, spec_stride, count, n, shifts, h0, h1);
  return hipGetLastError();
}

// ------------------------------------------------- FSC shells (DFAlign.cu:212-297)
// Element (kx, y) of the half spectrum (y = ky for ky < n/2, else ky - n,
// cufunc.cu:309-340) with r = sqrtf(kx^2 + y^2) in float belongs to shell
// int(r / step) unless int(r) <= 0 or r >= n/2+1, on side 0 (parallel to the
// drift direction d) when float(|kx dx + y dy| / r) > float(cos(pi/4)), else
// side 1.  Per (shell, side) the sums of Re(a conj b), |a|^2 and |b|^2 are
// taken in FP64.
//
// The float square root and division are rounded to nearest exactly
// (sqrt_rn, div_rn), so shell membership is the reference's whatever the
// compiler's lowering of sqrtf and '/'.

// Side of (kx, y): FP64 products, sum and quotient each rounded once as in
// the reference's host code (no fused multiply-add).
__device__ inline int fsc_side(int kx, int y, float r, double dx, double dy) {
#pragma clang fp contract(off)
  const double p = (double)kx * dx;
  const double q = (double)y * dy;
  const float angle = (float)(fabs(p + q) / (double)r);
  return angle > (float)0.70710678118654752440 ? 0 : 1;
}

// Block-partial shell sums.  Each wave takes chunks of 64 consecutive
// elements (chunk c goes to wave c mod (waves of the grid)), groups the
// lanes of a chunk by (shell, side) and adds each group's wave-reduced sums
// into its own LDS table in program order; the block's tables are then added
// in wave order.  The result depends only on n and the grid, not on timing.
// padded = 1: row-major [ky][kx] layout (pitch n/2+1), else [kx][ky].
constexpr int FSC_NW = 4;

__global__ __launch_bounds__(FSC_NW * 64) void k_fsc_partial(const float2* __restrict__ a,
                                                            const float2* __restrict__ b, int n,
                                                            int padded, int step, int nbox,
                                                            double dx, double dy,
                                                            double* __restrict__ part) {
  extern __shared__ double fsc_acc[];  // [FSC_NW][nbox][2][3]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int H = n / 2 + 1, total = H * n, nchunk = (total + 63) / 64;
  const int nk = nbox * 6;
  for (int i = threadIdx.x; i < FSC_NW * nk; i += FSC_NW * 64) fsc_acc[i] = 0.0;
  __syncthreads();
  double* my = fsc_acc + w * nk;
  for (int c = blockIdx.x * FSC_NW + w; c < nchunk; c += gridDim.x * FSC_NW) {
    const int e = c * 64 + lane;
    int key = -1;
    double sab = 0.0, saa = 0.0, sbb = 0.0;
    if (e < total) {
      int kx, ky;
      if (padded) {
        ky = e / H;
        kx = e - ky * H;
      } else {
        kx = e / n;
        ky = e - kx * n;
      }
      const int y = ky < n / 2 ? ky : ky - n;
      const int q = kx * kx + y * y;
      if (q > 0) {
        const float r = sqrt_rn((float)q);
        if ((int)r > 0 && r < (float)H) {
          const int id = min((int)div_rn(r, (float)step), nbox - 1);  // r < H keeps id < nbox
          key = 2 * id + fsc_side(kx, y, r, dx, dy);
          const float2 va = a[e], vb = b[e];
          sab = (double)va.x * vb.x + (double)va.y * vb.y;
          saa = (double)va.x * va.x + (double)va.y * va.y;
          sbb = (double)vb.x * vb.x + (double)vb.y * vb.y;
        }
      }
    }
    unsigned long long rem = __ballot(key >= 0);
    while (rem) {
      const int k = __shfl(key, __ffsll((unsigned long long)rem) - 1);
      const bool mine = key == k;
      double t0 = mine ? sab : 0.0, t1 = mine ? saa : 0.0, t2 = mine ? sbb : 0.0;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        t0 += __shfl_xor(t0, o);
        t1 += __shfl_xor(t1, o);
        t2 += __shfl_xor(t2, o);
      }
      if (lane == 0) {
        my[3 * k] += t0;
        my[3 * k + 1] += t1;
        my[3 * k + 2] += t2;
      }
      rem &= ~__ballot(mine);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nk; i += FSC_NW * 64) {
    double s = 0.0;
#pragma unroll
    for (int v = 0; v < FSC_NW; v++) s += fsc_acc[v * nk + i];
    part[(size_t)blockIdx.x * nk + i] = s;
  }
}

__global__ __launch_bounds__(256) void k_fsc_final(const double* __restrict__ part, int nblocks,
                                                   int nk, double* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nk) return;
  double s = 0.0;
  for (int b = 0; b < nblocks; b++) s += part[(size_t)b * nk + i];
  out[i] = s;
}

int fsc_bins(int n, int* step) {
  int st = n / 400;  // DFAlign.cu:214 (n < 400 would divide by zero there)
  if (st < 1) st = 1;
  if (step) *step = st;
  return (n / 2 + 1) / st + 1;  // DFAlign.cu:218
}

int fsc_grid(int n) {
  const long long nchunk = ((long long)(n / 2 + 1) * n + 63) / 64;
  return (int)std::max(1LL, std::min(512LL, nchunk / 64));
}

hipError_t launch_fsc_sums(const float2* a, const float2* b, int n, int padded, double dx,
                           double dy, double* part, double* sums, hipStream_t st) {
  int step;
  const int nbox = fsc_bins(n, &step);
  const int nk = nbox * 6, G = fsc_grid(n);
  const size_t lds = sizeof(double) * FSC_NW * nk;
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_fsc_partial, dim3(G), dim3(FSC_NW * 64), lds, st, a, b, n, padded, step,
                     nbox, dx, dy, part);
  hipLaunchKernelGGL(k_fsc_final, dim3((nk + 255) / 256), dim3(256), 0, st, part, G, nk, sums);
  return hipGetLastError();
}

// ------------------------------------------------ sharpness and its adjoint
// J(s) = sum_k w(k) |S(k)|^2 with S = sum_f F_f e^{i phi_f}, phi_f(k) =
// 2 pi (s_fx kx + s_fy ky')/n, w = exp(-B|k|^2/(2n^2)) * a_kx (a = 1 at DC and
// Nyquist columns, 2 otherwise: the half-plane counts both halves).
// dJ/ds_fx = -2 sum_k w (2 pi kx/n) Im(conj(S) F_f e^{i phi_f}); same for y.
//
// The phase factors bound it: sincospif and the FP64 phase are 40 of about 60
// instructions per element and frame, so each is formed once.  Per tile of NT
// elements a thread rotates its element of every frame, in frame order as
// k_shift_sum, keeps the rotated values in LDS and has S at the end; then a
// thread takes the frames (f, f + FH) over part of the tile's elements, so
// that an element's S, weight and indexes are read once for two frames and the
// per-frame sums need no reduction until the end.  Frames are read once.
// LDS entry (f, e) lies at f NT + (e + f) mod NT: both phases without bank
// conflicts.
// 2048, 24 frames: 132 us for sum, J and gradient with the closing sum; the
// sum (84 us), a second pass over frames and sum (125) and a closing sum in
// one wave (77) before.
// SUM = false: S was formed before and is read; the frames are split over
// blockIdx.y (more frames than the LDS holds for a useful number of waves).
template <int NT, bool SUM>
__global__ __launch_bounds__(NT) void k_sharp(const float2* __restrict__ spectra, size_t spec_stride,
                                              int nframes, int FB, int n,
                                              const double2* __restrict__ shifts,
                                              float2* __restrict__ S, const float* __restrict__ wk,
                                              double2* __restrict__ part) {
  extern __shared__ float4 sharp_lds[];
  float4* rec = sharp_lds;  // [NT] S, weight, kx | ky' << 16
  float2* G = reinterpret_cast<float2*>(sharp_lds + NT);  // [FB][NT]
  const int H = n / 2 + 1, t = threadIdx.x;
  const long long total = (long long)H * n;
  const int c = blockIdx.x, nchunks = gridDim.x;
  const int e0 = (int)(total * c / nchunks), e1 = (int)(total * (c + 1) / nchunks);
  const int fb = blockIdx.y * FB, nf = min(FB, nframes - fb);
  const double inv_n = 1.0 / n;
  const int FH = (nf + 1) / 2, P = NT / FH;
  const int fa = t % FH, fz = fa + FH < nf ? fa + FH : fa, ep = t / FH;
  double J = 0, ax = 0, ay = 0, zx = 0, zy = 0;
  for (int et = e0; et < e1; et += NT) {
    const int e = min(et + t, e1 - 1);
    const int kx = e / n, ky = e - kx * n;
    const int yy = ky < n / 2 ? ky : ky - n;
    const float w = wk[kx] * wk[H + ky] * (et + t < e1 ? 1.f : 0.f);
    float2 acc = make_float2(0.f, 0.f);
    rotate_all(spectra + (size_t)fb * spec_stride, spec_stride, shifts + fb, nf, e, kx, yy, inv_n,
               [&](int f, float2 g, float y2) {
                 // sum and gradient round the product as their former passes did
                 acc = cadd(acc, g);
                 G[f * NT + (t + f < NT ? t + f : t + f - NT)] = make_float2(g.x, y2);
               });
    if (SUM) {
      if (et + t < e1) S[e] = acc;
    } else {
      acc = S[e];
    }
    rec[t] = make_float4(acc.x, acc.y, w, __int_as_float(kx | yy * 65536));
    J += (double)w * ((double)acc.x * acc.x + (double)acc.y * acc.y);
    __syncthreads();
    if (ep < P) {
#pragma unroll 4
      for (int x = ep; x < NT; x += P) {
        const float4 r = rec[x];
        const int k = __float_as_int(r.w);
        const double dkx = k & 0xffff, dyy = k >> 16, sx = r.x, sy = r.y, dw = r.z;
        const int ra = x + fa < NT ? x + fa : x + fa - NT, rz = x + fz < NT ? x + fz : x + fz - NT;
        const float2 ga = G[fa * NT + ra], gz = G[fz * NT + rz];
        const double ta = dw * (sx * ga.y - sy * ga.x);  // w Im(conj(S) G)
        const double tz = dw * (sx * gz.y - sy * gz.x);
        ax += ta * dkx;
        ay += ta * dyy;
        zx += tz * dkx;
        zy += tz * dyy;
      }
    }
    __syncthreads();
  }
  double2* red = reinterpret_cast<double2*>(G);  // [P][nf], at most 2 NT
  double* rj = reinterpret_cast<double*>(rec);
  if (ep < P) {
    if (fa + FH < nf) red[ep * nf + fa + FH] = make_double2(zx, zy);
    red[ep * nf + fa] = make_double2(ax, ay);
  }
  rj[t] = J;
  __syncthreads();
  const double m = -2.0 * (2.0 * M_PI * inv_n);
  double2* out = part + (size_t)c * (nframes + 1);
  for (int f = t; f < nf; f += NT) {
    double x = 0, y = 0;
    for (int q = 0; q < P; q++) {
      const double2 v = red[q * nf + f];
      x += v.x;
      y += v.y;
    }
    const double sx = shifts[fb + f].x;
    out[fb + f] = sx == sx ? make_double2(m * x, m * y) : make_double2(0.0, 0.0);
  }
  if (blockIdx.y == 0 && t < 64) {
    double x = 0;
    for (int q = t; q < NT; q += 64) x += rj[q];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    if (t == 0) out[nframes] = make_double2(x, 0.0);
  }
}

// Sums the chunk partials in a fixed order, one workgroup per output:
// out[f] = (gx, gy), out[F] = (J, 0).
__global__ __launch_bounds__(256) void k_sharp_final(const double2* __restrict__ part, int nchunks,
                                                     int nframes, double2* __restrict__ out) {
  __shared__ double2 red[4];
  const int f = blockIdx.x, t = threadIdx.x;
  double x = 0, y = 0;
  for (int c = t; c < nchunks; c += 256) {
    const double2 v = part[(size_t)c * (nframes + 1) + f];
    x += v.x;
    y += v.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    x += __shfl_xor(x, o);
    y += __shfl_xor(y, o);
  }
  if ((t & 63) == 0) red[t >> 6] = make_double2(x, y);
  __syncthreads();
  if (t == 0)
    out[f] = make_double2(red[0].x + red[1].x + red[2].x + red[3].x,
                          red[0].y + red[1].y + red[2].y + red[3].y);
}

// Tiles: as many threads as leave the LDS room for two workgroups per CU, the
// grid as many workgroups as the CUs then hold (at most four each) and no
// shorter chunks than a tile.  The rotated values of all frames of a tile limit
// the waves per CU (12 at 24 frames, 4 at 64), so up to 64 frames the sum is
// formed in the same pass (2048: 40 frames 285 us, 64 frames 599) and above by
// a pass of its own, then 24 frames at a time (64: 630, 80: 755).  The two
// passes that this replaces took 448, 668 and 859.
struct SharpPlan {
  bool fused;
  int nb, FB, NT, lds, nchunks;
};
static SharpPlan sharp_plan(int nframes, int n) {
  SharpPlan p;
  p.fused = nframes <= 64;
  p.nb = p.fused ? 1 : (nframes + 23) / 24;
  p.FB = (nframes + p.nb - 1) / p.nb;
  p.NT = p.FB <= 38 ? 256 : p.FB <= 51 ? 192 : 128;
  p.lds = p.NT * (std::max(p.FB, 4) * 8 + 16);  // the closing sums take 32 bytes per thread
  const long long tiles = ((long long)(n / 2 + 1) * n + p.NT - 1) / p.NT;
  p.nchunks = (int)std::min<long long>(tiles, 256 * std::min(4, 160 * 1024 / p.lds));
  return p;
}
size_t sharp_part_elems(int nframes, int n) {
  return (size_t)sharp_plan(nframes, n).nchunks * (nframes + 1);
}

template <int NT, bool SUM>
static hipError_t sharp_launch(const SharpPlan& p, const float2* spectra, size_t spec_stride,
                               int nframes, int n, const double2* shifts, float2* S,
                               const float* wk, double2* part, hipStream_t st) {
  // the same limit at every call: a smaller launch of another thread does not
  // lower it between this call and its launch
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_sharp<NT, SUM>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_sharp<NT, SUM>), dim3(p.nchunks, p.nb), dim3(NT), p.lds, st, spectra,
                     spec_stride, nframes, p.FB, n, shifts, S, wk, part);
  return hipGetLastError();
}

hipError_t launch_sharpness(const float2* spectra, size_t spec_stride, int nframes, int n,
                            const double2* shifts, float2* S, const float* wk, double2* part,
                            double2* out, hipStream_t st) {
  const SharpPlan p = sharp_plan(nframes, n);
  hipError_t e = hipSuccess;
  if (!p.fused) {
    e = launch_shift_sum(spectra, spec_stride, nframes, n, shifts, S, nullptr, -1, st);
    if (e != hipSuccess) return e;
    e = sharp_launch<256, false>(p, spectra, spec_stride, nframes, n, shifts, S, wk, part, st);
  } else if (p.NT == 256) {
    e = sharp_launch<256, true>(p, spectra, spec_stride, nframes, n, shifts, S, wk, part, st);
  } else if (p.NT == 192) {
    e = sharp_launch<192, true>(p, spectra, spec_stride, nframes, n, shifts, S, wk, part, st);
  } else {
    e = sharp_launch<128, true>(p, spectra, spec_stride, nframes, n, shifts, S, wk, part, st);
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_sharp_final, dim3(nframes + 1), dim3(256), 0, st, part, p.nchunks, nframes,
                     out);
  return hipGetLastError();
}

// ------------------------------------------- elementwise (cufunc.cu:243-263)
__global__ void k_add(float* __restrict__ dst, const float* __restrict__ src, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] += src[i];
}
__global__ void k_scale(float* __restrict__ dst, float s, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] *= s;
}

hipError_t launch_add(float* dst, const float* src, size_t n, hipStream_t st) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(k_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dst, src, n);
  return hipGetLastError();
}
hipError_t launch_scale(float* dst, float s, size_t n, hipStream_t st) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(k_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dst, s, n);
  return hipGetLastError();
}

}  // namespace mc
