// basis.hip -- per-element P2M and L2P bases, evaluated once per plan in FP64
// and stored scaled in the compute precision.
//
//   P2M_j[n,m] = ik sum_q w_q A_j [ -dR_n^{-m}/dn_j + sigma_j R_n^{-m} ](y_q - c)
//                / w_n                    (bottomLevelCoeff_L, integral.cu:821-836,
//                                          triElemIntegral_R / _pRpn, 251-365)
//   L2P_i[n,m] = [ R_n^m + alpha dR_n^m/dn_i ](x_i - c) / w_n
// c is the leaf-box centre; dR/dn follows dirDev_R (integral.cu:284-331).
// With dsig set the kernel writes dP2M_j/dsigma_j = ik sum_q w_q A_j R_n^{-m}
// / w_n instead (and no L2P), the column factor of the sigma derivative.
// One wavefront per element.  Its time is the FP64 chain of the R tables
// (fmb_device.h), so the points run side by side and dR/dn, six square roots
// an entry, is taken once of their sum: order 14, 10,580 triangles, 1.14 ms
// before and 0.13 now.
#include "fmb_device.h"

namespace {

constexpr int WG = 64;

template <typename T>
__global__ void __launch_bounds__(WG)
    k_bases(int N, int pL, double k, double alre, double alim,
            const double *__restrict__ tri, const double *__restrict__ geo,
            const int *__restrict__ ebox, const int *__restrict__ keys, int L,
            double D, double p0, double p1, double p2,
            const double2 *__restrict__ robin, const double *__restrict__ quad,
            int nq, const double *__restrict__ wsc, T *__restrict__ P2M,
            T *__restrict__ L2P, int dsig) {
  extern __shared__ double2 sm[];
  const int nm = pL;  // R needed up to degree pL for the derivative of degree pL-1
  const int ps = pL * pL;
  const r_lds tb = r_lds_at(sm, nm, L2P != nullptr);
  int j = blockIdx.x;
  int lane = threadIdx.x;
  // leaf-box centre
  int key = keys[ebox[j]];
  int tx = 0, ty = 0, tz = 0;
  for (int i = 0; i < L; i++) {
    int d = (key >> (3 * i)) & 7;
    tx |= ((d >> 2) & 1) << i;
    ty |= ((d >> 1) & 1) << i;
    tz |= (d & 1) << i;
  }
  double h = ldexp(1.0, -L);
  double c[3] = {D * (h * tx + 0.5 * h) + p0, D * (h * ty + 0.5 * h) + p1,
                 D * (h * tz + 0.5 * h) + p2};
  const double *tr = tri + 9 * (size_t)j;
  const double *g = geo + 8 * (size_t)j;
  double nr[3] = {g[3], g[4], g[5]};
  double area = g[6];
  double2 sg = robin ? robin[j] : make_double2(0.0, 0.0);
  // the sum over the panel's points comes first: dR/dn is linear in R and the normal is one
  r_tables(nm, k, nq, L2P != nullptr,
           [&](int q, double *v, double &w) {
             const double *qq = quad + 4 * q;
             for (int a = 0; a < 3; a++)
               v[a] = (q < nq ? qq[0] * tr[a] + qq[1] * tr[3 + a] + qq[2] * tr[6 + a] : g[a]) -
                      c[a];
             w = q < nq ? qq[3] * area : 1.0;
           },
           tb);
  // (n, m) and (n, -m) together: R_n^{-m} and its derivative are the conjugates
  for (int f = lane; f < pL * (pL + 1) / 2; f += WG) {
    int n, m;
    tri_nm(f, n, m);
    const dr_fac fc = dr_factors(n, m);
    const double s = 1.0 / wsc[n];
    {
      const double2 R = tb.Rs[f], dR = dRdn(tb.Rs, n, m, fc, k, nr);
#pragma unroll
      for (int sg2 = 0; sg2 < 2; sg2++) {  // order -m takes R_n^m, order m its conjugate
        if (sg2 && m == 0) break;
        const double u = sg2 ? -1.0 : 1.0, Ry = u * R.y, dy = u * dR.y;
        // val = -dR + sigma R (dsig: R) ; P2M = i k val
        const double vr = dsig ? R.x : -dR.x + sg.x * R.x - sg.y * Ry;
        const double vi = dsig ? Ry : -dy + sg.x * Ry + sg.y * R.x;
        const size_t o = 2 * ((size_t)j * ps + n * n + n - (sg2 ? -m : m));
        P2M[o] = (T)(-k * vi * s);
        P2M[o + 1] = (T)(k * vr * s);
      }
    }
    if (L2P) {
      const double2 R = tb.R1[f], dR = dRdn(tb.R1, n, m, fc, k, nr);
#pragma unroll
      for (int sg2 = 0; sg2 < 2; sg2++) {
        if (sg2 && m == 0) break;
        const double u = sg2 ? -1.0 : 1.0, Ry = u * R.y, dy = u * dR.y;
        const size_t o = 2 * ((size_t)j * ps + n * n + n + (sg2 ? -m : m));
        L2P[o] = (T)((R.x + alre * dR.x - alim * dy) * s);
        L2P[o + 1] = (T)((Ry + alre * dy + alim * dR.x) * s);
      }
    }
  }
}

}  // namespace

static int launch_bases(fmb_plan *pl, int op, const fmb_c64 *robin, void *P2M,
                        void *L2P, int dsig, void *stream) {
  const fmb_tree *t = pl->tree;
  int L = t->lmax, pL = pl->p[L];
  const size_t lds = r_lds_bytes(pL, L2P != NULL);
  if (pL > 66)
    return fmb_set_error(FMB_ERR_RANGE, "leaf order %d too large for bases",
                         pL);
  hipStream_t st = (hipStream_t)stream;
  fmb_opset *o = &pl->ops[op];
  if (o->prec == FMB_FP64) {
    auto kern = k_bases<double>;
    if (lds > 64 * 1024)
      FMB_HIP_CHECK(hipFuncSetAttribute(
          (const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
          160 * 1024));
    hipLaunchKernelGGL(kern, dim3(t->nelem), dim3(WG), lds, st, t->nelem, pL,
                       pl->k, pl->alpha_re, pl->alpha_im, t->d_tri, t->d_geo,
                       t->d_elem_box, t->d_keys[L], L, t->D, t->pmin[0],
                       t->pmin[1], t->pmin[2], (const double2 *)robin,
                       pl->d_quad, pl->nq, pl->d_scale[L], (double *)P2M,
                       (double *)L2P, dsig);
  } else {
    auto kern = k_bases<float>;
    if (lds > 64 * 1024)
      FMB_HIP_CHECK(hipFuncSetAttribute(
          (const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
          160 * 1024));
    hipLaunchKernelGGL(kern, dim3(t->nelem), dim3(WG), lds, st, t->nelem, pL,
                       pl->k, pl->alpha_re, pl->alpha_im, t->d_tri, t->d_geo,
                       t->d_elem_box, t->d_keys[L], L, t->D, t->pmin[0],
                       t->pmin[1], t->pmin[2], (const double2 *)robin,
                       pl->d_quad, pl->nq, pl->d_scale[L], (float *)P2M,
                       (float *)L2P, dsig);
  }
  FMB_LAUNCH_CHECK();
  FMB_HIP_CHECK(hipStreamSynchronize(st));
  return FMB_OK;
}

extern "C" int fmbh_bases(fmb_plan *pl, int op, const fmb_c64 *robin,
                          void *stream) {
  return launch_bases(pl, op, robin, pl->ops[op].d_P2M, pl->ops[op].d_L2P, 0, stream);
}

extern "C" int fmbh_bases_dsigma(fmb_plan *pl, int op, void *out, void *stream) {
  return launch_bases(pl, op, NULL, out, NULL, 1, stream);
}
