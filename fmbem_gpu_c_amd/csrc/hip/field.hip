// field.hip -- pressure at field points off the surface from a surface
// solution, by the exterior representation formula
//   p(y) = p_inc(y) + sum_j x_j int_j (dG/dn_y - sigma_j G) dS_y
// with the same kernels, signs and panel rules as the collocation entries
// (near.hip): the refined rule when |y - c_j| < ratio * radius_j.  The
// reference has no field evaluation.  One workgroup per field point reduces
// over all panels in FP64 (for few points, over one slice of them, the
// slices summed in order by k_field_sum); R right-hand sides per pass.
//
// Its transpose, for adjoint objectives: given weights u[r][q] at the field
// points, per element j (caller order)
//   kt[r][j] = sum_q u[r][q] int_j (dG/dn_y - sigma_j G)(y_q, y) dS_y
//   st[r][j] = sum_q u[r][q] int_j G(y_q, y) dS_y
// one thread per element, R right-hand sides per pass.
//
// Through the tree (k_field_box, k_field_tree): the multipole expansions M
// of the upward pass stand in for the panels of every box well separated
// from the point (a treecode with the separation of the M2L lists), the
// panels next to the point are summed directly with the rule above.  The
// coarse levels, whose orders are high, run box-major over chunks of points
// in Morton order; the finer levels per point.
#include <hipcub/hipcub.hpp>

#include "fmb_device.h"

namespace {

constexpr int kT = 256, kR = 8;
constexpr int kFieldSlicePts = 1024; // below this many point groups k_field slices the panels

// R right-hand sides at P field points a workgroup: a thread takes a panel for
// all P, so that its 136 bytes, strided over the lanes, are read once for them
// and the points' chains run beside each other.  81,920 panels at 32 points
// with one right-hand side: 120 us at P = 1, 87 at 4.  The refined rule
// has a loop of its own, so that its registers do not cost the plain one a
// workgroup a CU: two right-hand sides at 1,000 points, 20,480 panels, 757 us
// in one loop (181 VGPRs), 655 in two (147).
template <int P, int R>
__global__ void __launch_bounds__(kT, P > 1 ? 2 : R > 1 ? 3 : 4)
    k_field(const double *__restrict__ pts, int npts, const double *__restrict__ tri,
            const double *__restrict__ geo, const int *__restrict__ perm, int N,
            double k, const double2 *__restrict__ robin,
            const double *__restrict__ quad, int nq, const double *__restrict__ quadn,
            int nqn, double ratio, const double2 *__restrict__ x, int nrhs, int r0,
            const double *__restrict__ dirs, double2 *__restrict__ out,
            double2 *__restrict__ part) {
  __shared__ double2 red[kT / 64][P * R];
  const int q0 = blockIdx.x * P, nsl = gridDim.y;
  const double nz[3] = {0.0, 0.0, 0.0};
  const int nr = min(R, nrhs - r0);
  double y[P][3];
  double2 acc[P][R];
#pragma unroll
  for (int i = 0; i < P; i++) {
    const int q = min(q0 + i, npts - 1);  // (points beyond the last repeat it)
    for (int a = 0; a < 3; a++) y[i][a] = pts[3 * (size_t)q + a];
#pragma unroll
    for (int r = 0; r < R; r++) acc[i][r] = make_double2(0.0, 0.0);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // a panel's integrals S, K at point i, Robin coefficient sg, times its values val(r)
  auto add = [&](int i, const double2 &S, const double2 &K, const double2 &sg, auto val) {
    double2 g = K;
    if (robin) {
      g.x -= sg.x * S.x - sg.y * S.y;
      g.y -= sg.x * S.y + sg.y * S.x;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (r < nr) {
        const double2 v = val(r);
        acc[i][r].x += g.x * v.x - g.y * v.y;
        acc[i][r].y += g.x * v.y + g.y * v.x;
      }
    }
  };
  auto coeff = [&](int j) { return robin ? robin[j] : make_double2(0.0, 0.0); };
  auto values = [&](int j) {
    return [=, c = perm[j]](int r) { return x[(size_t)(r0 + r) * N + c]; };
  };
  const double lim2 = ratio * ratio;
  auto is_close = [&](int i, const double *g) {
    const double dx = y[i][0] - g[0], dy = y[i][1] - g[1], dz = y[i][2] - g[2];
    return dx * dx + dy * dy + dz * dz < lim2 * g[7] * g[7];
  };
  // panels of the refined rule, a point of the rule a lane (128 points next to a
  // surface of 1,280 panels: 90 us with the rule by the lane of the panel, one
  // point a workgroup; 137 with four points, one after the other; 66 now)
  auto refined = [&](int i, int j0, unsigned long long near) {
    for (; near; near &= near - 1) {
      const int j = j0 + __ffsll(near) - 1;
      const double *gj = geo + 8 * (size_t)j;
      for (int q = lane; q < nqn; q += 64) {
        double2 o[4];
        panel_sum(k, y[i], nz, tri + 9 * (size_t)j, gj + 3, gj[6], quadn + 4 * q, 1, o);
        add(i, o[0], o[1], coeff(j), values(j));
      }
    }
  };
  const int first = blockIdx.y * kT + 64 * w;  // the wave's first panel
  static_assert(P == 1 || R == 1, "v is the one right-hand side of several points");
  bool met = false;
  for (int j = first + lane; j < N; j += nsl * kT) {
    if constexpr (P == 1) {
      const double *gj = geo + 8 * (size_t)j;
      if (is_close(0, gj)) {
        met = true;
      } else {
        double2 o[4];
        panel_sum(k, y[0], nz, tri + 9 * (size_t)j, gj + 3, gj[6], quad, nq, o);
        add(0, o[0], o[1], coeff(j), values(j));
      }
    } else {
      const double *gj = geo + 8 * (size_t)j, *tr = tri + 9 * (size_t)j;
      double t[9], g8[8];
      for (int a = 0; a < 9; a++) t[a] = tr[a];
      for (int a = 0; a < 8; a++) g8[a] = gj[a];
      bool close[P];
      double2 S[P], K[P];  // int G, int dG/dn_y
#pragma unroll
      for (int i = 0; i < P; i++) {
        close[i] = is_close(i, g8);
        S[i] = K[i] = make_double2(0.0, 0.0);
      }
      for (int q = 0; q < nq; q++) {  // (panel_sum's S and K)
        const double *qq = quad + 4 * q;
        const double wt = qq[3] * g8[6];
        double z[3];
        for (int a = 0; a < 3; a++) z[a] = qq[0] * t[a] + qq[1] * t[3 + a] + qq[2] * t[6 + a];
#pragma unroll
        for (int i = 0; i < P; i++) {
          const double d0 = y[i][0] - z[0], d1 = y[i][1] - z[1], d2 = y[i][2] - z[2];
          const double r = sqrt(d0 * d0 + d1 * d1 + d2 * d2), ir = 1.0 / r;
          double sn, cs;
          sincos(k * r, &sn, &cs);
          const double g0 = (1.0 / (4.0 * M_PI)) * ir, gr = cs * g0, gi = sn * g0;
          const double wn = -wt * ((d0 * g8[3] + d1 * g8[4] + d2 * g8[5]) * ir);
          const double gpr = -gr * ir - k * gi, gpi = -gi * ir + k * gr;
          S[i].x += wt * gr;
          S[i].y += wt * gi;
          K[i].x += wn * gpr;
          K[i].y += wn * gpi;
        }
      }
      const double2 sg = coeff(j), v = values(j)(0);
#pragma unroll
      for (int i = 0; i < P; i++) {
        met |= close[i];
        if (!close[i]) add(i, S[i], K[i], sg, [&](int) { return v; });
      }
    }
  }
  if (__any(met))  // the refined rule
    for (int j0 = first; j0 < N; j0 += nsl * kT) {
      const int j = j0 + lane;
#pragma unroll
      for (int i = 0; i < P; i++)
        refined(i, j0, __ballot(j < N && is_close(i, geo + 8 * (size_t)min(j, N - 1))));
    }
#pragma unroll
  for (int i = 0; i < P; i++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const double re = wave_all_sum(acc[i][r].x), im = wave_all_sum(acc[i][r].y);
      if (lane == 0) red[w][i * R + r] = make_double2(re, im);
    }
  __syncthreads();
  if (threadIdx.x < P * R) {
    const int r = threadIdx.x % R, q = q0 + threadIdx.x / R;
    if (r >= nr || q >= npts) return;
    double2 s = make_double2(0.0, 0.0);
    for (int i = 0; i < kT / 64; i++) {
      s.x += red[i][threadIdx.x].x;
      s.y += red[i][threadIdx.x].y;
    }
    if (part) {
      part[((size_t)blockIdx.y * kR + r) * npts + q] = s;
      return;
    }
    if (dirs) {
      const double *d = dirs + 3 * (r0 + r), *yq = pts + 3 * (size_t)q;
      double sn, cs;
      sincos(k * (d[0] * yq[0] + d[1] * yq[1] + d[2] * yq[2]), &sn, &cs);
      s.x += cs;
      s.y += sn;
    }
    out[(size_t)(r0 + r) * npts + q] = s;
  }
}

// The panel slices of k_field summed in a fixed order, plus the incident
// waves: one wavefront per (point, right-hand side).
__global__ void __launch_bounds__(kT)
    k_field_sum(const double2 *__restrict__ part, int nsl, const double *__restrict__ pts,
                int npts, double k, int nrhs, int r0, const double *__restrict__ dirs,
                double2 *__restrict__ out) {
  const int i = (blockIdx.x * kT + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  const int nr = min(kR, nrhs - r0);
  if (i >= npts * nr) return;
  const int r = i / npts, q = i % npts;
  double2 s = make_double2(0.0, 0.0);
  for (int sl = lane; sl < nsl; sl += 64) {
    const double2 v = part[((size_t)sl * kR + r) * npts + q];
    s.x += v.x;
    s.y += v.y;
  }
  s.x = wave_all_sum(s.x);
  s.y = wave_all_sum(s.y);
  if (lane != 0) return;
  if (dirs) {
    const double *d = dirs + 3 * (r0 + r);
    double sn, cs;
    sincos(k * (d[0] * pts[3 * q] + d[1] * pts[3 * q + 1] + d[2] * pts[3 * q + 2]), &sn, &cs);
    s.x += cs;
    s.y += sn;
  }
  out[(size_t)(r0 + r) * npts + q] = s;
}

__global__ void __launch_bounds__(kT)
    k_field_t(const double *__restrict__ pts, int npts, const double *__restrict__ tri,
              const double *__restrict__ geo, const int *__restrict__ perm, int N,
              double k, const double2 *__restrict__ robin,
              const double *__restrict__ quad, int nq, const double *__restrict__ quadn,
              int nqn, double ratio, const double2 *__restrict__ u, int nrhs, int r0,
              double2 *__restrict__ kt, double2 *__restrict__ st) {
  const int j = blockIdx.x * kT + threadIdx.x;
  if (j >= N) return;
  const int nr = min(kR, nrhs - r0);
  const double *gj = geo + 8 * (size_t)j;
  const double nz[3] = {0.0, 0.0, 0.0};
  const double2 sg = robin ? robin[j] : make_double2(0.0, 0.0);
  double2 ak[kR], as[kR];
#pragma unroll
  for (int r = 0; r < kR; r++) ak[r] = as[r] = make_double2(0.0, 0.0);
  for (int q = 0; q < npts; q++) {
    const double y[3] = {pts[3 * q], pts[3 * q + 1], pts[3 * q + 2]};
    const double dx = y[0] - gj[0], dy = y[1] - gj[1], dz = y[2] - gj[2];
    const bool close = dx * dx + dy * dy + dz * dz < ratio * ratio * gj[7] * gj[7];
    double2 o[4];
    panel_sum(k, y, nz, tri + 9 * (size_t)j, gj + 3, gj[6], close ? quadn : quad,
              close ? nqn : nq, o);
    const double2 g = make_double2(o[1].x - (sg.x * o[0].x - sg.y * o[0].y),
                                   o[1].y - (sg.x * o[0].y + sg.y * o[0].x));
#pragma unroll
    for (int r = 0; r < kR; r++) {
      if (r < nr) {
        const double2 w = u[(size_t)(r0 + r) * npts + q];
        ak[r].x += g.x * w.x - g.y * w.y;
        ak[r].y += g.x * w.y + g.y * w.x;
        as[r].x += o[0].x * w.x - o[0].y * w.y;
        as[r].y += o[0].x * w.y + o[0].y * w.x;
      }
    }
  }
  const int c = perm[j];
#pragma unroll
  for (int r = 0; r < kR; r++) {
    if (r < nr) {
      kt[(size_t)(r0 + r) * N + c] = ak[r];
      st[(size_t)(r0 + r) * N + c] = as[r];
    }
  }
}

// ---------------------------------------------------------------- treecode

constexpr int kCand = 256; // candidates of one level: <= 64 at level 2, <= 27*8 below
constexpr int kFieldChunk = 32768; // points per pass of the box-major sums
constexpr int kBoxMinP = 24;        // box-major from level 2 down while orders reach this
constexpr int kBoxMaxBoxes = 32768; // and the level has at most this many boxes

struct TreeLevels {
  int L;
  int p[FMB_MAXLEV], nbox[FMB_MAXLEV];
  const int *keys[FMB_MAXLEV];
  const int *cstart[FMB_MAXLEV];
  const double *scale[FMB_MAXLEV];
  const double2 *M[FMB_MAXLEV];
  double D, pmin[3];
};

__device__ __forceinline__ double2 cmul2(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Pressure at field point blockIdx.x through the tree, right-hand sides
// r0 .. r0+kR-1 of the nrhs the upward pass ran on.  Per level l, wave 0
// sorts the level's candidate boxes: a box whose level-l index differs by
// 2 or more in some coordinate from the index of the level-l box holding
// the point adds its expansion, -sum_{n<p} w_n Mt_n^m S_n^m(y - c) (Mt the
// stored coefficients M / w_n; the P2M basis expands -dG/dn + sigma G, the
// negative of the field kernel); a box next to it passes its children on;
// at the leaf level its panels are summed directly.  Levels up to lb were
// summed box-major by k_field_box into boxsum, read back here; below lb
// groups of 16, 32 or 64 lanes (by the level's order) take one box each,
// and lane m of a group runs column m of S_n^m up in n: the normalised
// Legendre recurrence P_n^m = a (cos(theta) P_{n-1}^m - b P_{n-2}^m) from
// the table leg (a, b per (n, m)) and dg[m] sin(theta)^m, and h_n by the
// upward recurrence h_{n+1} = (2n+1)/x h_n - h_{n-1}, dominated by y_n
// wherever the two recurrences part.  The workgroup's sums are reduced in a
// fixed order; the result goes to the caller's index qperm[q].
__global__ void __launch_bounds__(kT)
    k_field_tree(TreeLevels tl, const double2 *__restrict__ leg,
                 const double *__restrict__ dg, const double *__restrict__ pts,
                 const double *__restrict__ tri, const double *__restrict__ geo,
                 const int *__restrict__ perm, const int *__restrict__ bstart, int N,
                 double k, const double2 *__restrict__ robin,
                 const double *__restrict__ quad, int nq, const double *__restrict__ quadn,
                 int nqn, double ratio, const double2 *__restrict__ x, int nrhs, int r0,
                 const double *__restrict__ dirs, int npts, double2 *__restrict__ out,
                 int ostride, const int *__restrict__ qperm, int lb,
                 const double2 *__restrict__ boxsum) {
  __shared__ int cand[2][kCand];
  __shared__ int farl[kCand];
  __shared__ int nearl[32];
  __shared__ int cnt[3];
  __shared__ double2 red[kT / 64][kR];
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const double y[3] = {pts[3 * q], pts[3 * q + 1], pts[3 * q + 2]};
  double u[3];
  for (int a = 0; a < 3; a++) u[a] = (y[a] - tl.pmin[a]) / tl.D;
  const int nr = min(kR, nrhs - r0);
  double2 acc[kR];
#pragma unroll
  for (int r = 0; r < kR; r++) acc[r] = make_double2(0.0, 0.0);
  const int L = tl.L;
  const int nb2 = min(tl.nbox[2], 64);
  if (tid == 0) cnt[0] = nb2;
  if (tid < nb2) cand[0][tid] = tid;
  __syncthreads();
  int cur = 0;
  for (int l = 2; l <= L; l++) {
    const int nc = cnt[0];
    if (nc == 0) break;
    const double sc = ldexp(1.0, l);
    const double ty[3] = {floor(u[0] * sc), floor(u[1] * sc), floor(u[2] * sc)};
    __syncthreads();  // cnt[0] read by every thread before wave 0 rewrites it
    if (w == 0) {
      int nfar = 0, nnext = 0, nnear = 0;
      const unsigned long long lt = (1ull << lane) - 1ull;
      for (int i0 = 0; i0 < nc; i0 += 64) {
        const int i = i0 + lane;
        const bool valid = i < nc;
        const int b = valid ? cand[cur][i] : 0;
        bool far = false;
        if (valid) {
          int tx, tyy, tz;
          deinterleave3(tl.keys[l][b], l, tx, tyy, tz);
          const double sep = fmax(fabs(tx - ty[0]), fmax(fabs(tyy - ty[1]), fabs(tz - ty[2])));
          far = sep >= 2.0;
        }
        const bool nb = valid && !far;
        const unsigned long long fm = __ballot(far);
        if (far) {
          const int o = nfar + __popcll(fm & lt);
          if (o < kCand) farl[o] = b;
        }
        nfar += __popcll(fm);
        if (l < L) {
          const int c0 = nb ? tl.cstart[l][b] : 0, c1 = nb ? tl.cstart[l][b + 1] : 0;
          const int c = c1 - c0;
          int s = c;
          for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(s, o, 64);
            if (lane >= o) s += v;
          }
          const int base = nnext + s - c;
          for (int j = 0; j < c; j++)
            if (base + j < kCand) cand[cur ^ 1][base + j] = c0 + j;
          nnext += __shfl(s, 63, 64);
        } else {
          const unsigned long long nm = __ballot(nb);
          if (nb) {
            const int o = nnear + __popcll(nm & lt);
            if (o < 32) nearl[o] = b;
          }
          nnear += __popcll(nm);
        }
      }
      if (lane == 0) {
        cnt[0] = min(nnext, kCand);
        cnt[1] = min(nfar, kCand);
        cnt[2] = min(nnear, 32);
      }
    }
    __syncthreads();
    // expansions of the well-separated boxes (levels up to lb: summed
    // box-major by k_field_box into boxsum)
    const int p = tl.p[l], ps = p * p;
    const int G = p <= 16 ? 16 : (p <= 32 ? 32 : 64);
    const int gpw = 64 / G, ng = (kT / 64) * gpw;
    const int g = w * gpw + lane / G, lm = lane % G;
    const double *wsc = tl.scale[l];
    const double h = tl.D / sc;
    for (int i = g; l > lb && i < cnt[1]; i += ng) {
      const int b = farl[i];
      int tx, tyy, tz;
      deinterleave3(tl.keys[l][b], l, tx, tyy, tz);
      const double v0 = y[0] - (tl.pmin[0] + (tx + 0.5) * h);
      const double v1 = y[1] - (tl.pmin[1] + (tyy + 0.5) * h);
      const double v2 = y[2] - (tl.pmin[2] + (tz + 0.5) * h);
      const double rho = sqrt(v0 * v0 + v1 * v1), r = sqrt(rho * rho + v2 * v2);
      const double ct = v2 / r, st = rho / r, phi = atan2(v1, v0);
      const double kr = k * r, ikr = 1.0 / kr;
      double sx, cx;
      sincos(kr, &sx, &cx);
      // h_0 = -i e^{ix}/x, h_1 = -e^{ix}(x + i)/x^2
      const double2 h0 = make_double2(sx * ikr, -cx * ikr);
      const double2 h1 = make_double2((sx - cx * kr) * ikr * ikr, -(sx * kr + cx) * ikr * ikr);
      const double2 *Mb = tl.M[l] + ((size_t)b * nrhs + r0) * ps;
      for (int m = lm; m < p; m += G) {
        double stm = 1.0, base = st;
        for (int e = m; e > 0; e >>= 1) {
          if (e & 1) stm *= base;
          base *= base;
        }
        double P = dg[m] * stm, Pp = 0.0;
        double sm, cm;
        sincos(m * phi, &sm, &cm);
        const double2 ep = make_double2(cm, sm), em = make_double2(cm, -sm);
        double2 hc = h0, hp = make_double2(0.0, 0.0);
        for (int n = 0; n < p; n++) {
          if (n >= m) {
            if (n > m) {
              const double2 ab = leg[n * (n + 1) / 2 + m];
              const double Pn = ab.x * (ct * P - ab.y * Pp);
              Pp = P;
              P = Pn;
            }
            const double f = wsc[n] * P;
            const double2 t = make_double2(f * hc.x, f * hc.y);
            const int fp = n * n + n + m, fm = n * n + n - m;
#pragma unroll
            for (int rr = 0; rr < kR; rr++) {
              if (rr < nr) {
                double2 z = cmul2(Mb[(size_t)rr * ps + fp], ep);
                if (m > 0) {
                  const double2 zm = cmul2(Mb[(size_t)rr * ps + fm], em);
                  z.x += zm.x;
                  z.y += zm.y;
                }
                const double2 tz = cmul2(t, z);
                acc[rr].x -= tz.x;
                acc[rr].y -= tz.y;
              }
            }
          }
          if (n == 0) {
            hp = hc;
            hc = h1;
          } else {
            const double c = (2.0 * n + 1.0) * ikr;
            const double2 hn = make_double2(c * hc.x - hp.x, c * hc.y - hp.y);
            hp = hc;
            hc = hn;
          }
        }
      }
    }
    if (l == L) {
      // panels of the leaf boxes next to the point
      const double nz[3] = {0.0, 0.0, 0.0};
      for (int i = 0; i < cnt[2]; i++) {
        const int b = nearl[i];
        for (int j = bstart[b] + tid; j < bstart[b + 1]; j += kT) {
          const double *gj = geo + 8 * (size_t)j;
          const double dx = y[0] - gj[0], dy = y[1] - gj[1], dz = y[2] - gj[2];
          const bool close = dx * dx + dy * dy + dz * dz < ratio * ratio * gj[7] * gj[7];
          double2 o[4];
          panel_sum(k, y, nz, tri + 9 * (size_t)j, gj + 3, gj[6], close ? quadn : quad,
                    close ? nqn : nq, o);
          double2 gg = o[1];
          if (robin) {
            const double2 sg = robin[j];
            gg.x -= sg.x * o[0].x - sg.y * o[0].y;
            gg.y -= sg.x * o[0].y + sg.y * o[0].x;
          }
          const int c = perm[j];
#pragma unroll
          for (int rr = 0; rr < kR; rr++) {
            if (rr < nr) {
              const double2 v = x[(size_t)(r0 + rr) * N + c];
              acc[rr].x += gg.x * v.x - gg.y * v.y;
              acc[rr].y += gg.x * v.y + gg.y * v.x;
            }
          }
        }
      }
    }
    cur ^= 1;
    __syncthreads();  // farl, nearl and cnt are rewritten by the next level
  }
  if (tid == 0) {
#pragma unroll
    for (int rr = 0; rr < kR; rr++) {
      if (rr < nr) {
        const double2 v = boxsum[(size_t)rr * npts + q];
        acc[rr].x += v.x;
        acc[rr].y += v.y;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kR; r++) {
    double re = acc[r].x, im = acc[r].y;
    for (int o = 32; o > 0; o >>= 1) {
      re += __shfl_down(re, o, 64);
      im += __shfl_down(im, o, 64);
    }
    if (lane == 0) red[w][r] = make_double2(re, im);
  }
  __syncthreads();
  if (tid < nr) {
    const int r = tid;
    double2 s = make_double2(0.0, 0.0);
    for (int i = 0; i < kT / 64; i++) {
      s.x += red[i][r].x;
      s.y += red[i][r].y;
    }
    if (dirs) {
      const double *d = dirs + 3 * (r0 + r);
      double sn, cs;
      sincos(k * (d[0] * y[0] + d[1] * y[1] + d[2] * y[2]), &sn, &cs);
      s.x += cs;
      s.y += sn;
    }
    out[(size_t)(r0 + r) * ostride + qperm[q]] = s;
  }
}

// The expansions of level l box-major: wavefront w evaluates box w / nchunk of
// level l at the 64 points of chunk w % nchunk (the points come sorted in
// Morton order, so a chunk is compact), one point per lane, for the points the
// traversal of k_field_tree meets the box at: the box is well separated from
// the point at level l (indices 2 or more apart) and its parent is next to the
// point at level l - 1 (no condition at level 2; the parent's ancestors then
// lie next to the point too).  boxsum[r * npts + q] += -sum w_n Mt_n^m
// S_n^m(y_q - c) for right-hand sides r0 + r, r < nr <= NR, by FP64 atomic adds
// (the order of the boxes' contributions is not fixed).
//
// Bound by FP64 issue.  A lane runs CB columns m0 .. of S_n^m up in n beside
// each other, which share h_n and its weight and hide each other's chains: 13
// operations a coefficient pair and 5 a step; the azimuth factors, the same
// down a column, enter at its end.  The coefficients and the recurrence's
// factors are the same for all lanes and come through scalar loads: from LDS
// they would take as long as the arithmetic.  The state of h_n where the next
// columns start is kept on the way.  Levels 2 to 4 of 81,920 triangles (orders
// 47, 33, 25) at 16,384 points take 1.36 ms; 3.76 by single columns from LDS
// with h_n run up from n = 0 for each.
template <int CB, int NR>
__global__ void __launch_bounds__(64)
    k_field_box(const int *__restrict__ keys, int l, int p, double D, double p0, double p1,
                double p2, const double *__restrict__ wsc, const double2 *__restrict__ M,
                const double2 *__restrict__ leg, const double *__restrict__ dg,
                const double *__restrict__ pts, int npts, int nchunk, double k, int nrhs, int r0,
                int nr, double2 *__restrict__ boxsum) {
  // (grid y: groups of NR right-hand sides)
  r0 += NR * blockIdx.y;
  nr = min(NR, nr - NR * (int)blockIdx.y);
  boxsum += (size_t)NR * blockIdx.y * npts;
  const int b = blockIdx.x / nchunk, q = (blockIdx.x % nchunk) * 64 + threadIdx.x;
  int tx, tyy, tz;
  deinterleave3(keys[b], l, tx, tyy, tz);
  const double sc = ldexp(1.0, l);
  const double pmin[3] = {p0, p1, p2};
  double y[3] = {0.0, 0.0, 0.0};
  bool active = false;
  if (q < npts) {
    for (int a = 0; a < 3; a++) y[a] = pts[3 * q + a];
    const int t3[3] = {tx, tyy, tz};
    double sep = 0.0, psep = 0.0;
    for (int a = 0; a < 3; a++) {
      const double u = (y[a] - pmin[a]) / D;
      sep = fmax(sep, fabs(t3[a] - floor(u * sc)));
      psep = fmax(psep, fabs((t3[a] >> 1) - floor(u * (0.5 * sc))));
    }
    active = sep >= 2.0 && (l == 2 || psep <= 1.0);
  }
  if (!__any(active)) return;
  const double h = D / sc;
  const double v0 = y[0] - (p0 + (tx + 0.5) * h);
  const double v1 = y[1] - (p1 + (tyy + 0.5) * h);
  const double v2 = y[2] - (p2 + (tz + 0.5) * h);
  const double rho = sqrt(v0 * v0 + v1 * v1), r = sqrt(rho * rho + v2 * v2);
  // inactive lanes run the same steps on a harmless point and add nothing
  const double ct = active ? v2 / r : 1.0, st = active ? rho / r : 0.0;
  const double phi = active ? atan2(v1, v0) : 0.0;
  const double kr = active ? k * r : 1.0, ikr = 1.0 / kr;
  double sx, cx, s1, c1;
  sincos(kr, &sx, &cx);
  sincos(phi, &s1, &c1);
  const double2 e1 = make_double2(c1, s1);
  // h_m and h_{m-1} of the first column: h_0 = -i e^{ix}/x, h_{-1} = e^{ix}/x
  double2 hc0 = make_double2(sx * ikr, -cx * ikr), hp0 = make_double2(cx * ikr, sx * ikr);
  const double2 *Mb[NR];
  double2 acc[NR];
#pragma unroll
  for (int i = 0; i < NR; i++) {
    Mb[i] = M + ((size_t)b * nrhs + r0 + min(i, nr - 1)) * (size_t)(p * p);
    acc[i] = make_double2(0.0, 0.0);
  }
  double stm = 1.0;
  for (int m0 = 0; m0 < p; m0 += CB) {
    double P[CB], Pp[CB], first[CB];
    double2 ap[CB][NR], am[CB][NR];
#pragma unroll
    for (int c = 0; c < CB; c++) {
      first[c] = m0 + c < p ? dg[m0 + c] * stm : 0.0;
      stm *= st;
      P[c] = Pp[c] = 0.0;
#pragma unroll
      for (int i = 0; i < NR; i++) ap[c][i] = am[c][i] = make_double2(0.0, 0.0);
    }
    double2 hc = hc0, hp = hp0;
    // column c at degree n; j: n - m0 within the first CB degrees, else CB
    auto step = [&](int n, int j) {
      const double w = wsc[n];
      const double2 t = make_double2(w * hc.x, w * hc.y);
      const int f0 = n * n + n;
#pragma unroll
      for (int c = 0; c < CB; c++) {
        if (c > j) break;
        const int m = m0 + c;
        if (c == j) {
          P[c] = first[c];
        } else {
          const double2 ab = leg[n * (n + 1) / 2 + m];
          const double Pn = ab.x * (ct * P[c] - ab.y * Pp[c]);
          Pp[c] = P[c];
          P[c] = Pn;
        }
        const double2 u = make_double2(t.x * P[c], t.y * P[c]);
#pragma unroll
        for (int i = 0; i < NR; i++) {
          const double2 a = Mb[i][f0 + m], d = Mb[i][f0 - m];
          ap[c][i].x = fma(u.x, a.x, ap[c][i].x);
          ap[c][i].x = fma(-u.y, a.y, ap[c][i].x);
          ap[c][i].y = fma(u.x, a.y, ap[c][i].y);
          ap[c][i].y = fma(u.y, a.x, ap[c][i].y);
          am[c][i].x = fma(u.x, d.x, am[c][i].x);
          am[c][i].x = fma(-u.y, d.y, am[c][i].x);
          am[c][i].y = fma(u.x, d.y, am[c][i].y);
          am[c][i].y = fma(u.y, d.x, am[c][i].y);
        }
      }
      const double g = (2.0 * n + 1.0) * ikr;
      const double2 hn = make_double2(g * hc.x - hp.x, g * hc.y - hp.y);
      hp = hc;
      hc = hn;
    };
#pragma unroll
    for (int j = 0; j < CB; j++)
      if (m0 + j < p) step(m0 + j, j);
    hc0 = hc;
    hp0 = hp;
    for (int n = m0 + CB; n < p; n++) step(n, CB);
    double sm, cm;
    sincos(m0 * phi, &sm, &cm);
    double2 ep = make_double2(cm, sm);
#pragma unroll
    for (int c = 0; c < CB; c++) {
      if (m0 + c >= p) break;
      const double2 em = make_double2(ep.x, -ep.y);
#pragma unroll
      for (int i = 0; i < NR; i++) {
        double2 z = cmul2(ap[c][i], ep);
        if (m0 + c > 0) {
          const double2 zm = cmul2(am[c][i], em);
          z.x += zm.x;
          z.y += zm.y;
        }
        acc[i].x -= z.x;
        acc[i].y -= z.y;
      }
      ep = cmul2(ep, e1);
    }
  }
  if (active) {
#pragma unroll
    for (int i = 0; i < NR; i++) {
      if (i < nr) {
        atomicAdd(&boxsum[(size_t)i * npts + q].x, acc[i].x);
        atomicAdd(&boxsum[(size_t)i * npts + q].y, acc[i].y);
      }
    }
  }
}

// Order of the field points: Morton keys on a grid of 1/1024 of the cube over
// three cube widths (points beyond clamp to its faces), so that the wavefronts
// of the box-major levels take compact groups of points.
__global__ void k_field_keys(const double *__restrict__ pts, int npts, double D, double p0,
                             double p1, double p2, unsigned long long *__restrict__ key,
                             int *__restrict__ idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npts) return;
  const double pmin[3] = {p0, p1, p2};
  unsigned g[3];
  for (int c = 0; c < 3; c++) {
    const double v = floor((pts[3 * (size_t)i + c] - pmin[c]) / D * 1024.0) + 1024.0;
    g[c] = v < 0.0 ? 0u : (v > 3071.0 ? 3071u : (unsigned)v);
  }
  unsigned long long z = 0;
  for (int b = 11; b >= 0; b--)
    z = z * 8 + 4 * ((g[0] >> b) & 1) + 2 * ((g[1] >> b) & 1) + ((g[2] >> b) & 1);
  key[i] = z;
  idx[i] = i;
}

__global__ void k_field_points(const double *__restrict__ pts, const int *__restrict__ idx,
                               int npts, double *__restrict__ out) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 3 * (size_t)npts) out[t] = pts[3 * (size_t)idx[t / 3] + t % 3];
}

// normalised Legendre recurrence: (a, b) per (n, m < n), then P_m^m / sin^m
__global__ void k_field_leg(int pmax, double2 *__restrict__ leg, double *__restrict__ dg) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= tri_idx(pmax, 0)) return;
  int n, m;
  tri_nm(f, n, m);
  if (n == m) {
    double a = 1.0 / (4.0 * M_PI);
    for (int i = 1; i <= m; i++) a *= (2.0 * i + 1.0) / (2.0 * i);
    dg[m] = sqrt(a);
    return;
  }
  double b = 0.0;
  if (n > m + 1)
    b = sqrt(((double)(n - 1) * (n - 1) - (double)m * m) / (4.0 * (n - 1) * (n - 1) - 1.0));
  leg[f] = make_double2(sqrt((4.0 * n * n - 1.0) / ((double)n * n - (double)m * m)), b);
}

template <int CB, int NR>
void launch_box(const fmb_plan *pl, const fmb_opset *o, int l, const double2 *leg,
                const double *dg, const double *pts, int npts, int nrhs, int r0, int nr,
                double2 *boxsum, hipStream_t st) {
  const fmb_tree *t = pl->tree;
  const int nchunk = (npts + 63) / 64;
  hipLaunchKernelGGL((k_field_box<CB, NR>), dim3(nchunk * t->nbox[l], (nr + NR - 1) / NR),
                     dim3(64), 0, st,
                     t->d_keys[l], l, pl->p[l], t->D, t->pmin[0], t->pmin[1], t->pmin[2],
                     pl->d_scale[l], (const double2 *)o->d_M[l], leg, dg, pts, npts, nchunk,
                     pl->k, nrhs, r0, nr, boxsum);
}

}  // namespace

extern "C" int fmbh_field_t(const fmb_plan *pl, const fmb_c64 *u, int nrhs,
                            const double *d_pts, int npts, fmb_c64 *kt, fmb_c64 *st,
                            void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t s = (hipStream_t)stream;
  const int N = t->nelem;
  for (int r0 = 0; r0 < nrhs; r0 += kR) {
    hipLaunchKernelGGL(k_field_t, dim3((N + kT - 1) / kT), dim3(kT), 0, s, d_pts, npts,
                       t->d_tri, t->d_geo, t->d_perm, N, pl->k,
                       (const double2 *)pl->d_robin, pl->d_quad, pl->nq, pl->d_quadn,
                       pl->nqn, pl->prm.near_ratio, (const double2 *)u, nrhs, r0,
                       (double2 *)kt, (double2 *)st);
    FMB_LAUNCH_CHECK();
  }
  return FMB_OK;
}

extern "C" int fmbh_field(const fmb_plan *pl, const fmb_c64 *x, int nrhs,
                          const double *d_pts, int npts, const double *d_dirs,
                          fmb_c64 *out, void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  // one right-hand side: four points a workgroup; few points: their panels in
  // slices over several workgroups, so that the launch fills the device; the
  // slices are summed in order.  (81,920 panels at 32 points, 32 / 64 / 128
  // slices: 149 / 133 / 130 us a call; at 1,280 to 81,920 panels and 4 to 6,000
  // points 0.60 to 0.96 of the time of one point a workgroup in 32 slices.)
  const int P = nrhs == 1 && npts >= 4 ? 4 : 1, ng = (npts + P - 1) / P;
  const int nsl = ng >= kFieldSlicePts
                      ? 1
                      : min(P == 4 ? 128 : 32, (2 * kFieldSlicePts + ng - 1) / ng);
  double2 *d_part = NULL;
  int rc = FMB_OK;
  if (nsl > 1 && (rc = fmbh_malloc((void **)&d_part, sizeof(double2) * (size_t)nsl * kR * npts)))
    return rc;
  for (int r0 = 0; r0 < nrhs && !rc; r0 += kR) {
    hipLaunchKernelGGL((P == 4 ? k_field<4, 1> : nrhs == 1 ? k_field<1, 1> : k_field<1, kR>),
                       dim3(ng, nsl), dim3(kT), 0, st, d_pts, npts, t->d_tri, t->d_geo, t->d_perm,
                       t->nelem, pl->k, (const double2 *)pl->d_robin, pl->d_quad, pl->nq,
                       pl->d_quadn, pl->nqn, pl->prm.near_ratio, (const double2 *)x, nrhs, r0,
                       d_dirs, (double2 *)out, d_part);
    if (nsl > 1) {
      const int nr = nrhs - r0 < kR ? nrhs - r0 : kR;
      hipLaunchKernelGGL(k_field_sum, dim3((npts * nr + 3) / 4), dim3(kT), 0, st, d_part, nsl,
                         d_pts, npts, pl->k, nrhs, r0, d_dirs, (double2 *)out);
    }
    if (hipGetLastError() != hipSuccess) rc = fmb_set_error(FMB_ERR_HIP, "k_field launch");
  }
  if (d_part) {
    // the slices are freed only after the launches that read them
    if (hipStreamSynchronize(st) != hipSuccess && !rc)
      rc = fmb_set_error(FMB_ERR_HIP, "k_field");
    fmbh_free(d_part);
  }
  return rc;
}

// Treecode field of one upward pass: x, dirs and out start at the pass's
// first right-hand side; the opset op holds its multipole expansions.
// d_pts holds the points in Morton order, d_qperm[i] the caller's index of
// sorted point i (out is in caller order).
extern "C" int fmbh_field_tree(const fmb_plan *pl, int op, const fmb_c64 *x, int nrhs,
                               const double *d_pts, const int *d_qperm, int npts,
                               const double *d_dirs, fmb_c64 *out, void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  const fmb_opset *o = &pl->ops[op];
  if (o->prec != FMB_FP64)
    return fmb_set_error(FMB_ERR_ARG, "field through the tree: FP64 expansions only");
  if (t->lmax < 2 || t->nbox[2] > 64)
    return fmb_set_error(FMB_ERR_ARG, "field through the tree: no level-2 boxes");
  for (int l = 2; l <= t->lmax; l++)
    if (pl->p[l] > 256)
      return fmb_set_error(FMB_ERR_RANGE, "field through the tree: order %d", pl->p[l]);
  TreeLevels tl = {};
  tl.L = t->lmax;
  tl.D = t->D;
  for (int a = 0; a < 3; a++) tl.pmin[a] = t->pmin[a];
  int pmax = 0;
  for (int l = 2; l <= t->lmax; l++) {
    tl.p[l] = pl->p[l];
    tl.nbox[l] = t->nbox[l];
    tl.keys[l] = t->d_keys[l];
    tl.cstart[l] = l < t->lmax ? t->d_cstart[l] : NULL;
    tl.scale[l] = pl->d_scale[l];
    tl.M[l] = (const double2 *)o->d_M[l];
    pmax = pl->p[l] > pmax ? pl->p[l] : pmax;
  }
  const int ntri = pmax * (pmax + 1) / 2;
  double *d_tab = NULL;
  int rc = fmbh_malloc((void **)&d_tab, sizeof(double) * (2 * (size_t)ntri + pmax));
  if (rc) return rc;
  double2 *leg = (double2 *)d_tab;
  double *dg = d_tab + 2 * ntri;
  hipLaunchKernelGGL(k_field_leg, dim3((ntri + 63) / 64), dim3(64), 0, st, pmax, leg, dg);
  // levels 2 .. lb box-major (orders of kBoxMinP and above), the rest per
  // point; the box-major sums of one chunk of points: [kR][chunk]
  int lb = 2;
  while (lb < t->lmax && pl->p[lb + 1] >= kBoxMinP && t->nbox[lb + 1] <= kBoxMaxBoxes) lb++;
  const int chunk = npts < kFieldChunk ? npts : kFieldChunk;
  double2 *d_box = NULL;
  if (!rc) rc = fmbh_malloc((void **)&d_box, sizeof(double2) * (size_t)kR * chunk);
  for (int q0 = 0; q0 < npts && !rc; q0 += chunk) {
    const int nq0 = npts - q0 < chunk ? npts - q0 : chunk;
    for (int r0 = 0; r0 < nrhs && !rc; r0 += kR) {
      const int nr = nrhs - r0 < kR ? nrhs - r0 : kR;
      if ((rc = fmbh_memset(d_box, 0, sizeof(double2) * (size_t)kR * nq0, stream))) break;
      // one column group and several right-hand sides share the registers; two
      // groups of one form go into one launch (at 64 points a launch is a single
      // round: eight right-hand sides, 20,480 triangles, 1.60 ms a call with two
      // launches a level, 1.19 with one)
      for (int l = 2; l <= lb; l++)
        for (int q = 0, nb; q < nr; q += nb) {
          nb = nr - q >= 7 || nr - q < 4 ? nr - q : 4;
          auto launch = nb == 1 ? launch_box<4, 1> : nb == 2 ? launch_box<2, 2> : launch_box<1, 4>;
          launch(pl, o, l, leg, dg, d_pts + 3 * (size_t)q0, nq0, nrhs, r0 + q, nb,
                 d_box + (size_t)q * nq0, st);
        }
      hipLaunchKernelGGL(k_field_tree, dim3(nq0), dim3(kT), 0, st, tl,
                         (const double2 *)leg, dg, d_pts + 3 * (size_t)q0,
                         t->d_tri, t->d_geo, t->d_perm, t->d_box_start, t->nelem, pl->k,
                         (const double2 *)pl->d_robin, pl->d_quad, pl->nq, pl->d_quadn,
                         pl->nqn, pl->prm.near_ratio, (const double2 *)x, nrhs, r0,
                         d_dirs, nq0, (double2 *)out, npts, d_qperm + q0, lb, d_box);
      if (hipGetLastError() != hipSuccess)
        rc = fmb_set_error(FMB_ERR_HIP, "k_field_tree launch");
    }
  }
  // the tables are freed only after the launches that read them
  if (hipStreamSynchronize(st) != hipSuccess && !rc)
    rc = fmb_set_error(FMB_ERR_HIP, "k_field_tree");
  fmbh_free(d_tab);
  fmbh_free(d_box);
  return rc;
}

// Morton order of npts points (device, caller order): sorted points and the
// caller's index of each, in memory of the caller (fmbh_field_order_bytes).
extern "C" size_t fmbh_field_order_bytes(int npts) {
  size_t tb = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (unsigned long long *)nullptr,
                                         (unsigned long long *)nullptr, (int *)nullptr,
                                         (int *)nullptr, npts, 0, 36) != hipSuccess)
    return 0;
  const size_t n = ((size_t)npts + 1) & ~(size_t)1;
  return 16 * n + 4 * n + tb + 256;
}

extern "C" int fmbh_field_order(const fmb_tree *t, const double *d_pts, int npts, double *d_spts,
                                int *d_qperm, void *work, size_t bytes, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  const size_t n = ((size_t)npts + 1) & ~(size_t)1;
  unsigned long long *key = (unsigned long long *)work, *key2 = key + n;
  int *idx = (int *)(key2 + n);
  void *tmp = (void *)(((size_t)(idx + n) + 255) & ~(size_t)255);
  size_t tb = (char *)work + bytes - (char *)tmp;
  hipLaunchKernelGGL(k_field_keys, dim3((npts + 255) / 256), dim3(256), 0, st, d_pts, npts, t->D,
                     t->pmin[0], t->pmin[1], t->pmin[2], key, idx);
  FMB_LAUNCH_CHECK();
  FMB_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, key, key2, idx, d_qperm, npts, 0, 36,
                                                   st));
  hipLaunchKernelGGL(k_field_points, dim3((unsigned)((3 * (size_t)npts + 255) / 256)), dim3(256),
                     0, st, d_pts, d_qperm, npts, d_spts);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}
