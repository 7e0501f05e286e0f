/*
 * fmb_device.h -- device-side helpers shared by the gfx950 kernels:
 * complex arithmetic on (re, im) pairs of the compute type, launch checks,
 * FP64 special functions (spherical Bessel, normalised Legendre, R_n^m and
 * its normal derivative) used by operator generation and the bases.
 */
#ifndef FMB_DEVICE_H
#define FMB_DEVICE_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>

#include "fmb_hip.h"

#define FMB_HIP_CHECK(call)                                                    \
  do {                                                                         \
    hipError_t e_ = (call);                                                    \
    if (e_ != hipSuccess)                                                      \
      return fmb_set_error(FMB_ERR_HIP, "%s:%d: %s", __FILE__, __LINE__,       \
                           hipGetErrorString(e_));                             \
  } while (0)

#define FMB_LAUNCH_CHECK() FMB_HIP_CHECK(hipGetLastError())

/* Block i of n with each of the 8 XCDs (workgroups go round them in turn)
 * taking a contiguous range: neighbours share an L2. */
__device__ __forceinline__ int xcd_block(int i, int n) {
  const int x = i & 7, q = n >> 3, r = n & 7;
  return x * q + min(x, r) + (i >> 3);
}

template <typename T> struct cplx {
  T re, im;
};

template <typename T>
__device__ __forceinline__ cplx<T> cmk(T r, T i) {
  cplx<T> z;
  z.re = r;
  z.im = i;
  return z;
}
template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) {
  return cmk<T>(a.re + b.re, a.im + b.im);
}
template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return cmk<T>(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
/* a += b*c */
template <typename T>
__device__ __forceinline__ void cfma(cplx<T> &a, cplx<T> b, cplx<T> c) {
  a.re = fma(b.re, c.re, a.re);
  a.re = fma(-b.im, c.im, a.re);
  a.im = fma(b.re, c.im, a.im);
  a.im = fma(b.im, c.re, a.im);
}
/* a += h*c, h real */
template <typename T>
__device__ __forceinline__ void rfma(cplx<T> &a, T h, cplx<T> c) {
  a.re = fma(h, c.re, a.re);
  a.im = fma(h, c.im, a.im);
}

/* a += v with hardware float atomics (-munsafe-fp-atomics) */
template <typename T>
__device__ __forceinline__ void atomic_add_c(cplx<T> *dst, cplx<T> v) {
  unsafeAtomicAdd(&dst->re, v.re);
  unsafeAtomicAdd(&dst->im, v.im);
}

/* n with n^2 <= f < (n+1)^2: the degree of coefficient index f = n^2+n+m.
 * For 0 <= f < 2^22 the float square root is within one of n, so one
 * correction each way makes it exact (no data-dependent loop). */
__device__ __forceinline__ int isqrt_fix(int f) {
  int n = (int)sqrtf((float)f);
  n -= n * n > f;
  n += (n + 1) * (n + 1) <= f;
  return n;
}

/* one M2L offset: polar-angle table index, distance class, azimuth phi */
struct OffInfo {
  int beta, dist;
  double phi;
};

/* Morton keys: x is the most significant bit of each octal digit, coarse
 * levels most significant (octree.c:132-142). */
__device__ __forceinline__ int interleave3(int tx, int ty, int tz, int l) {
  int key = 0;
  for (int i = l - 1; i >= 0; i--)
    key = key * 8 + 4 * ((tx >> i) & 1) + 2 * ((ty >> i) & 1) + ((tz >> i) & 1);
  return key;
}

__device__ __forceinline__ void deinterleave3(int key, int l, int &tx, int &ty,
                                              int &tz) {
  int x = 0, y = 0, z = 0;
  for (int i = 0; i < l; i++) {
    int d = (key >> (3 * i)) & 7;
    x |= ((d >> 2) & 1) << i;
    y |= ((d >> 1) & 1) << i;
    z |= (d & 1) << i;
  }
  tx = x;
  ty = y;
  tz = z;
}

static inline __host__ __device__ int rot_off(int n) {
  return n * (4 * n * n - 1) / 3;
}
static inline __host__ __device__ int coax_size(int p) {
  return p * (2 * p * p + 3 * p + 1) / 6;
}
static inline __host__ __device__ int coax_blk(int p, int m) {
  int a = m < 0 ? -m : m;
  return a * (2 * a * a - (3 + 6 * p) * a + 1 + 6 * (p + p * p)) / 6;
}

/* translation.cu:189-212 in FP64 */
__device__ __forceinline__ double acoef(int n, int m) {
  int am = m < 0 ? -m : m;
  if (n < am) return 0.0;
  double nf = n, mf = m;
  return sqrt((nf + 1 + mf) * (nf + 1 - mf) / ((2 * nf + 1) * (2 * nf + 3)));
}
__device__ __forceinline__ double bcoef(int n, int m) {
  double nf = n, mf = m;
  if (m >= 0 && n >= m)
    return sqrt((nf - mf - 1) * (nf - mf) / ((2 * nf - 1) * (2 * nf + 1)));
  if (-n <= m && m < 0)
    return -sqrt((nf - mf - 1) * (nf - mf) / ((2 * nf - 1) * (2 * nf + 1)));
  return 0.0;
}

/* j_n(x), n = 0..nmax: Miller downward recurrence normalised by
 * sum (2n+1) j_n^2 = 1; serial (one lane). */
__device__ inline void dev_sph_jn(int nmax, double x, double *j) {
  if (x == 0.0) {
    j[0] = 1.0;
    for (int n = 1; n <= nmax; n++) j[n] = 0.0;
    return;
  }
  int nk = nmax < 1 ? 1 : nmax;
  double ax = fabs(x);
  double top = nk > ax ? (double)nk : ax;
  int nst = (int)ceil(top) + 40 + (int)ceil(6.0 * cbrt(top));
  const double ix = 1.0 / x;
  double fp1 = 0.0, fc = 1.0, sum = 0.0, f0 = 0.0, f1 = 0.0;
  for (int n = nst; n >= 0; n--) {
    if (n <= nmax) j[n] = fc;
    if (n == 0) f0 = fc;
    if (n == 1) f1 = fc;
    sum += (2.0 * n + 1.0) * fc * fc;
    if (n == 0) break;
    double fm1 = (2.0 * n + 1.0) * ix * fc - fp1;
    fp1 = fc;
    fc = fm1;
    if (fabs(fc) > 1e100) {
      const double s = 1e-100;
      fc *= s;
      fp1 *= s;
      sum *= s * s;
      if (n <= 1) f1 *= s;
      for (int q = (n - 1 > nmax ? nmax + 1 : n); q <= nmax; q++) j[q] *= s;
    }
  }
  double c = 1.0 / sqrt(sum);
  double sx, cx;
  sincos(x, &sx, &cx);
  double j0 = sx / x, j1 = sx / (x * x) - cx / x;
  bool neg = (fabs(j0) >= fabs(j1)) ? ((j0 < 0) != (f0 < 0))
                                    : ((j1 < 0) != (f1 < 0));
  if (neg) c = -c;
  for (int n = 0; n <= nmax; n++) j[n] *= c;
}

/* y_n(x) by upward recurrence */
__device__ inline void dev_sph_yn(int nmax, double x, double *y) {
  double sx, cx;
  sincos(x, &sx, &cx);
  y[0] = -cx / x;
  if (nmax == 0) return;
  y[1] = -cx / (x * x) - sx / x;
  for (int n = 1; n < nmax; n++) y[n + 1] = (2.0 * n + 1.0) / x * y[n] - y[n - 1];
}

/* Regular panel integrals at point x (normal nx) over triangle tri (9
 * doubles, normal ny, area) with the rule quad (nq x {b0, b1, b2, w}):
 * out = [S = int G, K = int dG/dn_y, K' = int dG/dn_x, T = int d2G/dn_x dn_y],
 * G = e^{ikr} / (4 pi r), r = |x - y| (integral.cu:72-78, 391-415, 602-622). */
__device__ inline void panel_sum(double k, const double *x, const double *nx,
                          const double *tri, const double *ny, double area,
                          const double *quad, int nq, double2 out[4]) {
  for (int i = 0; i < 4; i++) out[i] = make_double2(0, 0);
  for (int q = 0; q < nq; q++) {
    const double *qq = quad + 4 * q;
    double y[3], d[3];
    for (int a = 0; a < 3; a++) {
      y[a] = qq[0] * tri[a] + qq[1] * tri[3 + a] + qq[2] * tri[6 + a];
      d[a] = x[a] - y[a];
    }
    double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    double s, c;
    sincos(k * r, &s, &c);
    double w = qq[3] * area;
    // one division a point (81,920 panels at 32 points: 120 us, 142 with six)
    double ir = 1.0 / r;
    double g0 = (1.0 / (4.0 * M_PI)) * ir;
    double gr = c * g0, gi = s * g0;
    double rnx = (d[0] * nx[0] + d[1] * nx[1] + d[2] * nx[2]) * ir;
    double rny = -(d[0] * ny[0] + d[1] * ny[1] + d[2] * ny[2]) * ir;
    // gp = g (-1/r + i k)
    double gpr = -gr * ir - k * gi, gpi = -gi * ir + k * gr;
    double nn = nx[0] * ny[0] + nx[1] * ny[1] + nx[2] * ny[2];
    // d2G = e/(4 pi r^3) [ (3 - k^2 r^2 - 3ikr) rnx rny + (1 - ikr) nn ]
    double ar = (3.0 - k * k * r * r) * rnx * rny + nn;
    double ai = -3.0 * k * r * rnx * rny - k * r * nn;
    double h0 = g0 * ir * ir;
    double hr = h0 * (c * ar - s * ai), hi = h0 * (c * ai + s * ar);
    out[0].x += w * gr;
    out[0].y += w * gi;
    out[1].x += w * gpr * rny;
    out[1].y += w * gpi * rny;
    out[2].x += w * gpr * rnx;
    out[2].y += w * gpi * rnx;
    out[3].x += w * hr;
    out[3].y += w * hi;
  }
}

/* Self-panel integrals at the centroid c of a flat triangle (9 doubles) as
 * contour integrals over its three edges (integral.cu:202-249, 666-751):
 *   S = (1/4pi) oint (e^{ik rho}-1)/(ik) dtheta
 *   T = -(1/4pi) [ oint (e^{ik rho}-1)/rho dtheta + oint dtheta/rho - 2 pi i k ]
 * with nedge Gauss points per edge (edge: {x, w} pairs on [-1,1]).  By a
 * whole wavefront, one point a lane, the result in every lane: by one lane
 * while 63 wait, the 72 points of a panel took longer than its row of near
 * entries. */
__device__ __forceinline__ double wave_all_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ inline void self_terms(double k, const double *tri, const double *c,
                           const double *edge, int nedge, int lane, double2 &S,
                           double2 &T) {
  double sSr = 0, sSi = 0, sTr = 0, sTi = 0;
  for (int i = lane; i < 3 * nedge; i += 64) {
    const int e = i / nedge, q = i - e * nedge;
    double P[3], Q[3], ev[3], L = 0;
    for (int a = 0; a < 3; a++) {
      P[a] = e == 0 ? tri[a] : e == 1 ? tri[3 + a] : tri[6 + a];
      Q[a] = e == 0 ? tri[3 + a] : e == 1 ? tri[6 + a] : tri[a];
      ev[a] = Q[a] - P[a];
      L += ev[a] * ev[a];
    }
    L = sqrt(L);
    double tp = 0;
    for (int a = 0; a < 3; a++) {
      ev[a] /= L;
      tp += (c[a] - P[a]) * ev[a];
    }
    double h = 0;
    for (int a = 0; a < 3; a++) {
      double f = P[a] + tp * ev[a] - c[a];
      h += f * f;
    }
    h = sqrt(h);
    double thP = atan2(-tp, h), thQ = atan2(L - tp, h);
    if (q == 0) sTr += (sin(thQ) - sin(thP)) / h;
    double half = 0.5 * (thQ - thP), mid = 0.5 * (thQ + thP);
    double th = mid + half * edge[2 * q];
    double rho = h / cos(th);
    double w = half * edge[2 * q + 1];
    double s2, c2;
    sincos(0.5 * k * rho, &s2, &c2);
    // gs = 2 sin(k rho/2) e^{i k rho/2} / k
    double gr, gi;
    if (k == 0.0) {
      gr = rho;
      gi = 0;
    } else {
      gr = 2.0 * s2 * c2 / k;
      gi = 2.0 * s2 * s2 / k;
    }
    sSr += w * gr;
    sSi += w * gi;
    // i k gs / rho
    sTr += w * (-k * gi / rho);
    sTi += w * (k * gr / rho);
  }
  sSr = wave_all_sum(sSr);
  sSi = wave_all_sum(sSi);
  sTr = wave_all_sum(sTr);
  sTi = wave_all_sum(sTi);
  const double f = 1.0 / (4.0 * M_PI);
  S = make_double2(f * sSr, f * sSi);
  T = make_double2(-f * sTr, -f * (sTi - 2.0 * M_PI * k));
}

/* ---- spherical basis tables (P2M / L2P bases, shape sensitivities) ---- */

/* degree and order of entry f of a table of n = 0, 1, ..., m = 0 .. n */
__device__ __forceinline__ int tri_idx(int n, int m) { return n * (n + 1) / 2 + m; }
__device__ __forceinline__ void tri_nm(int f, int &n, int &m) {
  n = (int)((sqrtf(8.0f * f + 1.0f) - 1.0f) * 0.5f);
  n -= tri_idx(n, 0) > f;
  n += tri_idx(n + 1, 0) <= f;
  m = f - tri_idx(n, 0);
}

/* R_n^m(v), n <= nm, m >= 0 (R_n^{-m} is its conjugate), of one wavefront's
 * points in LDS: Rs the sum over the points with weights, R1 one more point.
 * The points' serial parts (the Bessel recurrence, its 70 steps the longest
 * chain here) run side by side, a point a lane; then a lane runs column m of
 * the Legendre functions up for one point, 1, 2 or 4 points at a time by the
 * order.  With a point after the other and one lane at the recurrences of
 * each, a table cost 20,000 cycles. */
constexpr int kRPts = 16; /* points of a pass */
struct r_lds {
  double2 *Rs, *R1, *leg; /* nt entries each; leg: recurrence factors      */
  double2 *part;          /* further sums, a table each                    */
  double *pt, *jn;        /* cos, sin, azimuth, weight; j_n of each point  */
};
static inline __host__ __device__ int r_slots(int nm) { return nm < 16 ? 4 : nm < 32 ? 2 : 1; }
static inline __host__ __device__ size_t r_lds_bytes(int nm, int one) {
  const size_t nt = (size_t)(nm + 1) * (nm + 2) / 2;
  return 16 * nt * (1 + r_slots(nm) + (one ? 1 : 0)) + 8 * (size_t)kRPts * (nm + 5);
}
__device__ __forceinline__ r_lds r_lds_at(void *p, int nm, int one) {
  const int nt = (nm + 1) * (nm + 2) / 2;
  r_lds t;
  t.leg = (double2 *)p;
  t.Rs = t.leg + nt;
  t.part = t.Rs + nt;
  t.R1 = t.part + (r_slots(nm) - 1) * nt;
  t.pt = (double *)(t.R1 + (one ? nt : 0));
  t.jn = t.pt + 4 * kRPts;
  return t;
}

/* np points with weights (point(q, v, w)), then, with one set, point np for
 * R1; np >= 1 */
template <typename F>
__device__ inline void r_tables(int nm, double k, int np, int one, F point, const r_lds &t) {
  const int lane = threadIdx.x, nt = (nm + 1) * (nm + 2) / 2;
  for (int f = lane; f < nt; f += 64) {
    int n, m;
    tri_nm(f, n, m);
    double a, b = 0.0;
    if (n == m) { /* P_m^m = a sin^m */
      a = 1.0 / (4.0 * M_PI);
      for (int i = 1; i <= m; i++) a *= (2.0 * i + 1.0) / (2.0 * i);
      a = sqrt(a);
    } else { /* P_n^m = a (cos P_{n-1}^m - b P_{n-2}^m) */
      a = sqrt((4.0 * n * n - 1.0) / ((double)n * n - (double)m * m));
      if (n > m + 1)
        b = sqrt((((double)(n - 1) * (n - 1)) - (double)m * m) /
                 (4.0 * (n - 1) * (n - 1) - 1.0));
    }
    t.leg[f] = make_double2(a, b);
  }
  const int slots = r_slots(nm), wd = 64 / slots, slot = lane / wd, lm = lane % wd;
  double2 *Rp = slot ? t.part + (slot - 1) * nt : t.Rs;
  const int all = np + (one ? 1 : 0);
  for (int q0 = 0; q0 < all; q0 += kRPts) {
    const int nq = min(kRPts, all - q0);
    __syncthreads();
    if (lane < nq) {
      double v[3], w;
      point(q0 + lane, v, w);
      double rho2 = v[0] * v[0] + v[1] * v[1];
      double r = sqrt(rho2 + v[2] * v[2]);
      double ct = 1.0, st = 0.0, phi = 0.0;
      if (r > 0) {
        ct = v[2] / r;
        st = sqrt(rho2) / r;
        phi = atan2(v[1], v[0]);
      }
      double *pt = t.pt + 4 * lane;
      pt[0] = ct;
      pt[1] = st;
      pt[2] = phi;
      pt[3] = w;
      dev_sph_jn(nm, k * r, t.jn + lane * (nm + 1));
    }
    __syncthreads();
    for (int i = slot; i < nq; i += slots) {
      const int q = q0 + i;
      const double ct = t.pt[4 * i], st = t.pt[4 * i + 1], phi = t.pt[4 * i + 2];
      const double w = q < np ? t.pt[4 * i + 3] : 1.0;
      const double *jn = t.jn + i * (nm + 1);
      double2 *R = q < np ? Rp : t.R1;
      const bool add = q < np && q >= slots;
      for (int m = lm; m <= nm; m += wd) {
        double pw = 1.0, base = st;
        for (int e = m; e > 0; e >>= 1) {
          if (e & 1) pw *= base;
          base *= base;
        }
        double s, c;
        sincos(m * phi, &s, &c);
        c *= w;
        s *= w;
        double p1 = t.leg[tri_idx(m, m)].x * pw, p2 = 0.0;
        for (int n = m; n <= nm; n++) {
          const int f = tri_idx(n, m);
          if (n > m) {
            const double2 ab = t.leg[f];
            const double pv = ab.x * (ct * p1 - ab.y * p2);
            p2 = p1;
            p1 = pv;
          }
          const double a = jn[n] * p1;
          double2 v = make_double2(a * c, a * s);
          if (add) {
            v.x += R[f].x;
            v.y += R[f].y;
          }
          R[f] = v;
        }
      }
    }
  }
  __syncthreads();
  const int ns = min(slots, np);
  if (ns > 1) {
    for (int f = lane; f < nt; f += 64) {
      double2 v = t.Rs[f];
      for (int s = 1; s < ns; s++) {
        v.x += t.part[(s - 1) * nt + f].x;
        v.y += t.part[(s - 1) * nt + f].y;
      }
      t.Rs[f] = v;
    }
    __syncthreads();
  }
}

/* dR_n^m/dn, m >= 0, of a table of m >= 0 (integral.cu:284-331); f: its
 * factors, which depend on n and m only */
struct dr_fac {
  double f0, f1, f2, f3, f4, f5;
};
__device__ __forceinline__ dr_fac dr_factors(int n, int m) {
  dr_fac f;
  f.f0 = bcoef(n + 1, -m - 1);
  f.f1 = bcoef(n, m);
  f.f2 = bcoef(n + 1, m - 1);
  f.f3 = bcoef(n, -m);
  f.f4 = acoef(n - 1, m);
  f.f5 = acoef(n, m);
  return f;
}
__device__ __forceinline__ double2 r_get(const double2 *R, int n, int m) {
  if (m > n || n < 0) return make_double2(0.0, 0.0);
  if (m >= 0) return R[tri_idx(n, m)];
  if (-m > n) return make_double2(0.0, 0.0);
  const double2 v = R[tri_idx(n, -m)];
  return make_double2(v.x, -v.y);
}
__device__ __forceinline__ double2 dRdn(const double2 *R, int n, int m, const dr_fac &f,
                                        double k, const double *nr) {
  double2 a1 = r_get(R, n + 1, m + 1), a2 = r_get(R, n - 1, m + 1);
  double2 b1 = r_get(R, n + 1, m - 1), b2 = r_get(R, n - 1, m - 1);
  double2 c1 = r_get(R, n - 1, m), c2 = r_get(R, n + 1, m);
  double t0r = f.f0 * a1.x - f.f1 * a2.x, t0i = f.f0 * a1.y - f.f1 * a2.y;
  double t1r = f.f2 * b1.x - f.f3 * b2.x, t1i = f.f2 * b1.y - f.f3 * b2.y;
  double t2r = f.f4 * c1.x - f.f5 * c2.x, t2i = f.f4 * c1.y - f.f5 * c2.y;
  double hx = 0.5 * k * nr[0], hy = 0.5 * k * nr[1], kz = k * nr[2];
  return make_double2(hx * t0r + hy * t0i + hx * t1r - hy * t1i + kz * t2r,
                      hx * t0i - hy * t0r + hx * t1i + hy * t1r + kz * t2i);
}

#endif
