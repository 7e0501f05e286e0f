// near.hip -- near-field blocks of the Burton-Miller operator and the fused
// L2P + near-field product.
//
// For a leaf box b the block holds rows = elements of b, columns = elements
// of the boxes in b's 27-box neighbourhood (the reference's I2 set,
// octree.c:497-505), row-major, in Morton element order.  Entries
//   A_ij = -K_ij - alpha T_ij + sigma_j (S_ij + alpha K'_ij)        (i != j)
//   A_ii = 1/2 + alpha sigma_i/2 - alpha T_ii + sigma_i S_ii
// with the kernels of integral.cu:72-78, 391-415, 602-622 integrated by the
// far rule (integral.cu:80-139 style panel rules), a refined rule when
// |x_i - c_j| < ratio * circumradius_j, and the centroid self terms as
// contour integrals over the three edges (integral.cu:202-249, 666-751):
//   S_ii = (1/4pi) oint (e^{ik rho}-1)/(ik) dtheta
//   T_ii = -(1/4pi) [ oint (e^{ik rho}-1)/rho dtheta + oint dtheta/rho - 2 pi i k ]
// (K_ii = K'_ii = 0 on a flat panel).  Evaluated in FP64, stored in the
// compute precision.  With dsig set the blocks hold dA_ij/dsigma_j instead:
// S_ij + alpha K'_ij (i != j) and alpha/2 + S_ii.
#include <hipcub/hipcub.hpp>

#include "fmb_device.h"

namespace {

__global__ void k_near_sizes(const int *bstart, const int *nstart,
                             const int *nbox, int nb, int *ncol,
                             unsigned long long *bsz) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  int c = 0;
  for (int q = nstart[b]; q < nstart[b + 1]; q++) {
    int o = nbox[q];
    c += bstart[o + 1] - bstart[o];
  }
  ncol[b] = c;
  bsz[b] = (unsigned long long)(bstart[b + 1] - bstart[b]) * c;
}

__device__ __forceinline__ double2 cm(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

template <typename T>
__global__ void __launch_bounds__(256)
    k_near_assemble(const int *__restrict__ bstart, const int *__restrict__ nstart,
                    const int *__restrict__ nbox, const int *__restrict__ ncols,
                    const unsigned long long *__restrict__ boff,
                    const double *__restrict__ tri, const double *__restrict__ geo,
                    double k, double alre, double alim,
                    const double2 *__restrict__ robin,
                    const double *__restrict__ quad, int nq,
                    const double *__restrict__ quadn, int nqn, double ratio,
                    const double *__restrict__ edge, int nedge, T *__restrict__ A,
                    int dsig) {
  __shared__ int cpre[28], cbox[27];
  __shared__ int ncb;
  int b = blockIdx.x;
  if (threadIdx.x == 0) {
    int acc = 0, q0 = nstart[b], q1 = nstart[b + 1];
    ncb = q1 - q0;
    for (int q = q0; q < q1; q++) {
      cpre[q - q0] = acc;
      cbox[q - q0] = nbox[q];
      int o = nbox[q];
      acc += bstart[o + 1] - bstart[o];
    }
    cpre[q1 - q0] = acc;
  }
  __syncthreads();
  int r0 = bstart[b], nr = bstart[b + 1] - r0, nc = ncols[b];
  double2 alpha = make_double2(alre, alim);
  unsigned long long base = boff[b];
  const int lane = threadIdx.x & 63;
  // entry (i, j) of the panel integrals o
  auto entry = [&](const double2 *o, int j) {
    double2 sj = robin ? robin[j] : make_double2(0, 0);
    double2 aT = cm(alpha, o[3]), aKp = cm(alpha, o[2]);
    double2 t = make_double2(o[0].x + aKp.x, o[0].y + aKp.y);
    double2 st = cm(sj, t);
    return dsig ? t : make_double2(-o[1].x - aT.x + st.x, -o[1].y - aT.y + st.y);
  };
  for (int e0 = threadIdx.x - lane; e0 < nr * nc; e0 += blockDim.x) {
    const int e = e0 + lane;
    int i = r0, j = r0;
    if (e < nr * nc) {
      int r = e / nc, cc = e % nc;
      int q = 0;
      while (q + 1 < ncb && cpre[q + 1] <= cc) q++;
      i = r0 + r;
      j = bstart[cbox[q]] + (cc - cpre[q]);
    }
    const double *gi = geo + 8 * (size_t)i, *gj = geo + 8 * (size_t)j;
    double dx = gi[0] - gj[0], dy = gi[1] - gj[1], dz = gi[2] - gj[2];
    const bool close = i != j && dx * dx + dy * dy + dz * dz < ratio * ratio * gj[7] * gj[7];
    double2 o[4], v = make_double2(0, 0);
    if (i != j && !close) {
      panel_sum(k, gi, gi + 3, tri + 9 * (size_t)j, gj + 3, gj[6], quad, nq, o);
      v = entry(o, j);
    }
    // entries of the refined rule, a point a lane: 10,580 triangles, 980 us with
    // these 64 points and the self terms by single lanes while the others
    // wait, 330 with the self terms spread, 190 with both
    for (unsigned long long mk = __ballot(close); mk; mk &= mk - 1) {
      const int src = __ffsll(mk) - 1, ii = __shfl(i, src, 64), jj = __shfl(j, src, 64);
      const double *hi = geo + 8 * (size_t)ii, *hj = geo + 8 * (size_t)jj;
      double2 w = make_double2(0, 0);
      for (int q = lane; q < nqn; q += 64) {
        panel_sum(k, hi, hi + 3, tri + 9 * (size_t)jj, hj + 3, hj[6], quadn + 4 * q, 1, o);
        const double2 u = entry(o, jj);
        w.x += u.x;
        w.y += u.y;
      }
      w.x = wave_all_sum(w.x);
      w.y = wave_all_sum(w.y);
      if (lane == src) v = w;
    }
    if (i != j) {
      A[2 * (base + e)] = (T)v.x;
      A[2 * (base + e) + 1] = (T)v.y;
    }
  }
  // the diagonal, an entry a wavefront
  int cs = 0;
  while (cs + 1 < ncb && cbox[cs] != b) cs++;
  for (int r = threadIdx.x >> 6; r < nr; r += blockDim.x >> 6) {
    const int j = r0 + r;
    const double2 sj = robin ? robin[j] : make_double2(0, 0);
    double2 S, Tt, v;
    self_terms(k, tri + 9 * (size_t)j, geo + 8 * (size_t)j, edge, nedge, lane, S, Tt);
    double2 aT = cm(alpha, Tt), sS = cm(sj, S), as = cm(alpha, sj);
    if (dsig)
      v = make_double2(0.5 * alpha.x + S.x, 0.5 * alpha.y + S.y);
    else
      v = make_double2(0.5 + 0.5 * as.x - aT.x + sS.x, 0.5 * as.y - aT.y + sS.y);
    if (lane == 0) {
      const unsigned long long e = base + (unsigned long long)r * nc + cpre[cs] + r;
      A[2 * e] = (T)v.x;
      A[2 * e + 1] = (T)v.y;
    }
  }
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// L2P + near: one block per leaf box, one wavefront per (row, RC right-hand
// sides) job, the result in the caller's order.  The neighbourhood is read a box a lane and
// its columns listed by all threads (by one thread, with a launch of its own
// for the caller's order, 14 us of a 1,280-triangle product, 9 now); with
// several right-hand sides a row is read once for four (60,500 triangles, 64
// right-hand sides, FP32: 1.93 -> 1.74 ms).  Neighbouring boxes share an XCD,
// since they read the same elements and write to the same cache lines.
template <typename T, int RC>
__global__ void __launch_bounds__(256)
    k_l2p_near(const int *__restrict__ bstart, const int *__restrict__ nstart,
               const int *__restrict__ nbox, const int *__restrict__ ncols,
               const unsigned long long *__restrict__ boff,
               const cplx<T> *__restrict__ A, const cplx<T> *__restrict__ E,
               const cplx<T> *__restrict__ Lc, const cplx<T> *__restrict__ xs,
               const int *__restrict__ perm, double2 *__restrict__ y, int N, int ps, int nrhs,
               int parts) {
  extern __shared__ int colj[];
  __shared__ int cpre[28], cfirst[27];
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int r0 = bstart[b], nr = bstart[b + 1] - r0, nc = ncols[b];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int q0 = nstart[b], ncb = nstart[b + 1] - q0;
  if (wave == 0) {
    int f = 0, cnt = 0;
    if (lane < ncb) {
      const int o = nbox[q0 + lane];
      f = bstart[o];
      cnt = bstart[o + 1] - f;
    }
    int pre = cnt;
    for (int o = 1; o < 32; o <<= 1) {
      const int v = __shfl_up(pre, o, 64);
      if (lane >= o) pre += v;
    }
    if (lane < ncb) {
      cfirst[lane] = f;
      cpre[lane + 1] = pre;
    }
    if (lane == 0) cpre[0] = 0;
  }
  __syncthreads();
  for (int c = threadIdx.x; c < nc; c += blockDim.x) {
    int q = 0;
    while (q + 1 < ncb && cpre[q + 1] <= c) q++;
    colj[c] = cfirst[q] + (c - cpre[q]);
  }
  __syncthreads();
  const cplx<T> *Ab = A + boff[b];
  const int ng = (nrhs + RC - 1) / RC;
  for (int job = wave; job < nr * ng; job += (blockDim.x >> 6)) {
    const int r = job % nr, h0 = job / nr * RC, i = r0 + r, to = perm[i];
    T sr[RC], si[RC];
    const cplx<T> *x[RC], *l[RC];
#pragma unroll
    for (int h = 0; h < RC; h++) {
      // (right-hand sides beyond the last repeat it: no branch between loads)
      const int rh = min(h0 + h, nrhs - 1);
      sr[h] = si[h] = 0;
      x[h] = xs + (size_t)rh * N;
      l[h] = Lc + ((size_t)b * nrhs + rh) * ps;
    }
    const cplx<T> *arow = Ab + (size_t)r * nc;
#pragma unroll 2
    for (int c = (parts & 1) ? lane : nc; c < nc; c += 64) {
      const cplx<T> a = arow[c];
      const int j = colj[c];
#pragma unroll
      for (int h = 0; h < RC; h++) {
        const cplx<T> v = x[h][j];
        sr[h] += a.re * v.re - a.im * v.im;
        si[h] += a.re * v.im + a.im * v.re;
      }
    }
    const cplx<T> *e = E + (size_t)i * ps;
#pragma unroll 4
    for (int f = (parts & 2) ? lane : ps; f < ps; f += 64) {
      const cplx<T> a = e[f];
#pragma unroll
      for (int h = 0; h < RC; h++) {
        const cplx<T> v = l[h][f];
        sr[h] += a.re * v.re - a.im * v.im;
        si[h] += a.re * v.im + a.im * v.re;
      }
    }
#pragma unroll
    for (int h = 0; h < RC; h++) {
      if (h0 + h >= nrhs) break;
      const T vr = wave_sum(sr[h]), vi = wave_sum(si[h]);
      if (lane == 0)
        y[(size_t)(h0 + h) * N + to] = make_double2((double)vr, (double)vi);
    }
  }
}

// Transposed near field + transposed P2M: one block per leaf box c, one
// wavefront per (element j of c, right-hand side) job, the result in the
// caller's order.  Column j of A lies in the blocks of the boxes b of c's
// neighbourhood (neighbourhoods are symmetric), at the columns where b's
// block lists box c: found by eight threads a box (by one thread for all,
// 29 us at 5,120 triangles, 19 now).  Far part:
// sum_f B[j][f] (-1)^n M'[c][r][f], the transposed pass's coefficients being
// kept multiplied by (-1)^n.
template <typename T, int RC>
__global__ void __launch_bounds__(256)
    k_near_t(const int *__restrict__ bstart, const int *__restrict__ nstart,
             const int *__restrict__ nbox, const int *__restrict__ ncols,
             const unsigned long long *__restrict__ boff,
             const cplx<T> *__restrict__ A, const cplx<T> *__restrict__ B,
             const cplx<T> *__restrict__ Mc, const cplx<T> *__restrict__ xs,
             const int *__restrict__ perm, double2 *__restrict__ y, int N, int ps, int nrhs,
             int parts) {
  __shared__ int nb_first[32], nb_row0[33], nb_col[32], nb_nc[32];
  __shared__ unsigned long long nb_off[32];
  const int c = xcd_block(blockIdx.x, gridDim.x);
  const int e0 = bstart[c], nj = bstart[c + 1] - e0;
  const int q0 = nstart[c], nnb = nstart[c + 1] - q0;
  {
    const int q = threadIdx.x >> 3, sub = threadIdx.x & 7;
    int cnt[4] = {0, 0, 0, 0}, pos = 32, b = -1;
    if (q < nnb) {
      b = nbox[q0 + q];
      const int s0 = nstart[b], s1 = nstart[b + 1];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int s = s0 + sub + 8 * i;
        if (s < s1) {
          const int o = nbox[s];
          cnt[i] = bstart[o + 1] - bstart[o];
          if (o == c) pos = sub + 8 * i;
        }
      }
    }
    for (int o = 1; o < 8; o <<= 1) pos = min(pos, __shfl_xor(pos, o, 64));
    int co = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) co += sub + 8 * i < pos ? cnt[i] : 0;
    for (int o = 1; o < 8; o <<= 1) co += __shfl_xor(co, o, 64);
    if (sub == 0) {
      nb_row0[q + 1] = 0;
      if (b >= 0 && pos < 32) {
        nb_first[q] = bstart[b];
        nb_row0[q + 1] = bstart[b + 1] - bstart[b];
        nb_col[q] = co;
        nb_nc[q] = ncols[b];
        nb_off[q] = boff[b];
      }
    }
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave == 0) {
    int pre = lane < 32 ? nb_row0[lane + 1] : 0;
    for (int o = 1; o < 32; o <<= 1) {
      const int v = __shfl_up(pre, o, 64);
      if (lane >= o) pre += v;
    }
    if (lane < 32) nb_row0[lane + 1] = pre;
    if (lane == 0) nb_row0[0] = 0;
  }
  __syncthreads();
  const int R = nb_row0[nnb], ng = (nrhs + RC - 1) / RC;
  for (int job = wave; job < nj * ng; job += (blockDim.x >> 6)) {
    const int jj = job % nj, h0 = job / nj * RC, j = e0 + jj, to = perm[j];
    T sr[RC], si[RC];
    const cplx<T> *x[RC], *l[RC];
#pragma unroll
    for (int h = 0; h < RC; h++) {
      const int rh = min(h0 + h, nrhs - 1);
      sr[h] = si[h] = 0;
      x[h] = xs + (size_t)rh * N;
      l[h] = Mc + ((size_t)c * nrhs + rh) * ps;
    }
    for (int u = (parts & 1) ? lane : R; u < R; u += 64) {
      int q = 0;
      while (q + 1 < nnb && nb_row0[q + 1] <= u) q++;
      const int r = u - nb_row0[q];
      const cplx<T> a = A[nb_off[q] + (size_t)r * nb_nc[q] + nb_col[q] + jj];
      const int i = nb_first[q] + r;
#pragma unroll
      for (int h = 0; h < RC; h++) {
        const cplx<T> v = x[h][i];
        sr[h] += a.re * v.re - a.im * v.im;
        si[h] += a.re * v.im + a.im * v.re;
      }
    }
    const cplx<T> *e = B + (size_t)j * ps;
#pragma unroll 4
    for (int f = (parts & 2) ? lane : ps; f < ps; f += 64) {
      cplx<T> a = e[f];
      if (isqrt_fix(f) & 1) a = cmk<T>(-a.re, -a.im);
#pragma unroll
      for (int h = 0; h < RC; h++) {
        const cplx<T> v = l[h][f];
        sr[h] += a.re * v.re - a.im * v.im;
        si[h] += a.re * v.im + a.im * v.re;
      }
    }
#pragma unroll
    for (int h = 0; h < RC; h++) {
      if (h0 + h >= nrhs) break;
      const T vr = wave_sum(sr[h]), vi = wave_sum(si[h]);
      if (lane == 0)
        y[(size_t)(h0 + h) * N + to] = make_double2((double)vr, (double)vi);
    }
  }
}

inline int nblk(size_t n, int b = 256) { return (int)((n + b - 1) / b); }

}  // namespace

extern "C" int fmbh_near_layout(fmb_plan *pl, void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  int L = t->lmax, nb = t->nbox[L];
  unsigned long long *bsz;
  int rc = fmbh_malloc((void **)&pl->d_near_ncol, sizeof(int) * nb);
  if (!rc) rc = fmbh_malloc((void **)&bsz, sizeof(unsigned long long) * (nb + 1));
  if (!rc)
    rc = fmbh_malloc((void **)&pl->d_near_off,
                     sizeof(unsigned long long) * (nb + 1));
  if (rc) return rc;
  FMB_HIP_CHECK(hipMemsetAsync(bsz, 0, sizeof(unsigned long long) * (nb + 1), st));
  hipLaunchKernelGGL(k_near_sizes, dim3(nblk(nb)), dim3(256), 0, st,
                     t->d_box_start, t->d_near_start, t->d_near_box, nb,
                     pl->d_near_ncol, bsz);
  FMB_LAUNCH_CHECK();
  size_t tb = 0;
  unsigned long long *off = (unsigned long long *)pl->d_near_off;
  FMB_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, bsz, off, nb + 1, st));
  void *tmp;
  if ((rc = fmbh_malloc(&tmp, tb))) return rc;
  FMB_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, tb, bsz, off, nb + 1, st));
  unsigned long long tot;
  if ((rc = fmbh_d2h(&tot, off + nb, sizeof(tot), stream))) return rc;
  pl->near_total = (size_t)tot;
  int *h = (int *)malloc(sizeof(int) * nb);
  rc = fmbh_d2h(h, pl->d_near_ncol, sizeof(int) * nb, stream);
  int mx = 0;
  for (int b = 0; b < nb; b++)
    if (h[b] > mx) mx = h[b];
  free(h);
  pl->near_max_ncol = mx;
  fmbh_free(tmp);
  fmbh_free(bsz);
  if (mx > 16384)
    return fmb_set_error(FMB_ERR_RANGE,
                         "near-field neighbourhood of %d elements exceeds 16384; "
                         "use a deeper tree",
                         mx);
  return rc;
}

static int launch_near(fmb_plan *pl, int op, const fmb_c64 *robin, void *out,
                       int dsig, void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  int L = t->lmax, nb = t->nbox[L];
  fmb_opset *o = &pl->ops[op];
  const unsigned long long *off = (const unsigned long long *)pl->d_near_off;
  if (o->prec == FMB_FP64)
    hipLaunchKernelGGL(k_near_assemble<double>, dim3(nb), dim3(256), 0, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, t->d_tri, t->d_geo, pl->k,
                       pl->alpha_re, pl->alpha_im, (const double2 *)robin,
                       pl->d_quad, pl->nq, pl->d_quadn, pl->nqn,
                       pl->prm.near_ratio, pl->d_edge, pl->prm.nedge,
                       (double *)out, dsig);
  else
    hipLaunchKernelGGL(k_near_assemble<float>, dim3(nb), dim3(256), 0, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, t->d_tri, t->d_geo, pl->k,
                       pl->alpha_re, pl->alpha_im, (const double2 *)robin,
                       pl->d_quad, pl->nq, pl->d_quadn, pl->nqn,
                       pl->prm.near_ratio, pl->d_edge, pl->prm.nedge,
                       (float *)out, dsig);
  FMB_LAUNCH_CHECK();
  FMB_HIP_CHECK(hipStreamSynchronize(st));
  return FMB_OK;
}

extern "C" int fmbh_near_assemble(fmb_plan *pl, int op, const fmb_c64 *robin,
                                  void *stream) {
  return launch_near(pl, op, robin, pl->ops[op].d_near, 0, stream);
}

extern "C" int fmbh_near_dsigma(fmb_plan *pl, int op, void *out, void *stream) {
  return launch_near(pl, op, NULL, out, 1, stream);
}

extern "C" int fmbh_l2p_near(const fmb_plan *pl, int op, fmb_c64 *y, int nrhs, int parts,
                             void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  int L = t->lmax, nb = t->nbox[L], pL = pl->p[L];
  const fmb_opset *o = &pl->ops[op];
  size_t lds = sizeof(int) * (size_t)(pl->near_max_ncol > 0 ? pl->near_max_ncol : 1);
  const unsigned long long *off = (const unsigned long long *)pl->d_near_off;
  if (o->prec == FMB_FP64)
    hipLaunchKernelGGL((nrhs == 1   ? k_l2p_near<double, 1>
                        : nrhs == 2 ? k_l2p_near<double, 2>
                                    : k_l2p_near<double, 4>),
                       dim3(nb), dim3(256), lds, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, (const cplx<double> *)o->d_near,
                       (const cplx<double> *)o->d_L2P,
                       (const cplx<double> *)o->d_L[L],
                       (const cplx<double> *)o->d_xs, t->d_perm, (double2 *)y,
                       t->nelem, pL * pL, nrhs, parts);
  else
    hipLaunchKernelGGL((nrhs == 1   ? k_l2p_near<float, 1>
                        : nrhs == 2 ? k_l2p_near<float, 2>
                                    : k_l2p_near<float, 4>),
                       dim3(nb), dim3(256), lds, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, (const cplx<float> *)o->d_near,
                       (const cplx<float> *)o->d_L2P,
                       (const cplx<float> *)o->d_L[L],
                       (const cplx<float> *)o->d_xs, t->d_perm, (double2 *)y,
                       t->nelem, pL * pL, nrhs, parts);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_near_t(const fmb_plan *pl, int op, const void *near, const void *basis,
                           fmb_c64 *y, int nrhs, int parts, void *stream) {
  const fmb_tree *t = pl->tree;
  hipStream_t st = (hipStream_t)stream;
  int L = t->lmax, nb = t->nbox[L], pL = pl->p[L];
  const fmb_opset *o = &pl->ops[op];
  const void *A = near ? near : o->d_near;
  const void *B = basis ? basis : o->d_P2M;
  const unsigned long long *off = (const unsigned long long *)pl->d_near_off;
  if (o->prec == FMB_FP64)
    hipLaunchKernelGGL((nrhs == 1   ? k_near_t<double, 1>
                        : nrhs == 2 ? k_near_t<double, 2>
                                    : k_near_t<double, 4>),
                       dim3(nb), dim3(256), 0, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, (const cplx<double> *)A,
                       (const cplx<double> *)B, (const cplx<double> *)o->d_M[L],
                       (const cplx<double> *)o->d_xs, t->d_perm, (double2 *)y,
                       t->nelem, pL * pL, nrhs, parts);
  else
    hipLaunchKernelGGL((nrhs == 1   ? k_near_t<float, 1>
                        : nrhs == 2 ? k_near_t<float, 2>
                                    : k_near_t<float, 4>),
                       dim3(nb), dim3(256), 0, st,
                       t->d_box_start, t->d_near_start, t->d_near_box,
                       pl->d_near_ncol, off, (const cplx<float> *)A,
                       (const cplx<float> *)B, (const cplx<float> *)o->d_M[L],
                       (const cplx<float> *)o->d_xs, t->d_perm, (double2 *)y,
                       t->nelem, pL * pL, nrhs, parts);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}
