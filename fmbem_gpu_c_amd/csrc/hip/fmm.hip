// fmm.hip -- the FMM pass on gfx950: its start (caller to Morton element
// order, P2M, cleared sums) and the VALU translations M2M ("SS"), M2L ("SR"),
// L2L ("RR").
//
// Translations are rotate-coaxial-rotate (translation.cu:1711-1808,
// 3461-3759): with t = (|t|, theta, phi),
//   a_n^m  = e^{i m phi} x_n^m                     (rotation alpha = phi)
//   b_n^m' = sum_m H_n^{m' m}(theta) a_n^m          (beta = theta, gamma = 0)
//   c_n'^m = sum_n C^{|m|}_{n' n}(|t|) b_n^m        (coaxial block |m|)
//   y_n^m' = e^{-i m' phi} sum_m H_n^{m' m}(theta) c_n^m   (0, theta, phi)
// on n-dependent scaled coefficients (M~ = M / w_n, L~ = w_n L) so that FP32
// operators stay inside the float range.  One translation job (box pair x
// right-hand side) runs on one workgroup of GS lanes: the vector is staged in
// LDS, each lane owns R outputs in registers between the three stages, and
// the rotation / coaxial matrices are read with lanes along rows of the
// column-major reference layouts (coalesced).  M2L jobs are grouped by offset
// (one H, one coaxial matrix per workgroup chunk) and accumulate into the
// target with hardware float atomics.
#include "fmb_device.h"

namespace {

// One rotate-coaxial-rotate translation of vector x (order pin) to order
// pout.  H: rotation blocks for theta (prefix layout), C: coaxial matrix at
// order P >= pin, pout (|m|-block layout), mtab: m-major enumeration of the
// pout^2 outputs (natural indices).  buf: LDS, max(pin,pout)^2 entries;
// ph: LDS, max(pin,pout) entries e^{i m phi}.  Leaves out[r] = output with
// natural index lane + GS*r.
template <typename T, int GS, int R>
__device__ __forceinline__ void rcr_job(const T *__restrict__ H,
                                        const cplx<T> *__restrict__ C, int P,
                                        int pin, int pout,
                                        const cplx<T> *__restrict__ x,
                                        const int *__restrict__ mtab,
                                        cplx<T> *buf, const cplx<T> *ph,
                                        cplx<T> out[R]) {
  const int lane = threadIdx.x;
  const int nin = pin * pin, nout = pout * pout;
  // 1. stage with forward phase e^{i m phi}
  for (int f = lane; f < nin; f += GS) {
    int n = isqrt_fix(f), m = f - n * n - n;
    cplx<T> e = ph[m < 0 ? -m : m];
    if (m < 0) e.im = -e.im;
    buf[f] = cmul(x[f], e);
  }
  __syncthreads();
  // 2. forward rotation, block n: b^{m'} = sum_m H^{m' m} a^m
#pragma unroll
  for (int r = 0; r < R; r++) {
    int f = lane + GS * r;
    cplx<T> s = cmk<T>(0, 0);
    if (f < nin) {
      int n = isqrt_fix(f), mp = f - n * n - n, ld = 2 * n + 1;
      const T *h = H + rot_off(n) + (mp + n);
      const cplx<T> *a = buf + n * n;
      for (int m = 0; m < ld; m++) rfma(s, h[m * ld], a[m]);
    }
    out[r] = s;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; r++) {
    int f = lane + GS * r;
    if (f < nin) buf[f] = out[r];
  }
  __syncthreads();
  // 3. coaxial, m-major outputs: c_{n'}^m = sum_{n>=|m|} C^{|m|}(n', n) b_n^m
#pragma unroll
  for (int r = 0; r < R; r++) {
    int g = lane + GS * r;
    cplx<T> s = cmk<T>(0, 0);
    if (g < nout) {
      int nat = mtab[g];
      int np = isqrt_fix(nat), m = nat - np * np - np, am = m < 0 ? -m : m;
      int ld = P - am;
      const cplx<T> *c = C + coax_blk(P, am) + (np - am);
      for (int n = am; n < pin; n++) cfma(s, c[(n - am) * ld], buf[n * n + n + m]);
    }
    out[r] = s;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; r++) {
    int g = lane + GS * r;
    if (g < nout) buf[mtab[g]] = out[r];
  }
  __syncthreads();
  // 4. back rotation with output phase e^{-i m' phi}
#pragma unroll
  for (int r = 0; r < R; r++) {
    int f = lane + GS * r;
    cplx<T> s = cmk<T>(0, 0);
    if (f < nout) {
      int n = isqrt_fix(f), mp = f - n * n - n, ld = 2 * n + 1;
      const T *h = H + rot_off(n) + (mp + n);
      const cplx<T> *a = buf + n * n;
      for (int m = 0; m < ld; m++) rfma(s, h[m * ld], a[m]);
      cplx<T> e = ph[mp < 0 ? -mp : mp];
      if (mp > 0) e.im = -e.im;
      s = cmul(s, e);
    }
    out[r] = s;
  }
  __syncthreads();
}

template <typename T>
__device__ __forceinline__ void fill_phase(cplx<T> *ph, int np_, double phi) {
  for (int m = threadIdx.x; m < np_; m += blockDim.x) {
    double s, c;
    sincos(m * phi, &s, &c);
    ph[m] = cmk<T>((T)c, (T)s);
  }
}

// M2L: blocks take chunks (offset, first pair, last pair) of one offset bucket
template <typename T, int GS, int R>
__global__ void __launch_bounds__(GS)
    k_m2l(const int4 *__restrict__ chunks, const OffInfo *__restrict__ info,
          const int *__restrict__ ptgt, const int *__restrict__ psrc,
          const T *__restrict__ Hall, size_t hstride,
          const cplx<T> *__restrict__ Call, size_t cstride, int p,
          const int *__restrict__ mtab, const cplx<T> *__restrict__ Min,
          cplx<T> *__restrict__ Lout, int nrhs) {
  extern __shared__ unsigned char smem[];
  cplx<T> *buf = (cplx<T> *)smem;
  cplx<T> *ph = buf + p * p;
  int4 ch = chunks[blockIdx.x];
  OffInfo oi = info[ch.x];
  const T *H = Hall + hstride * oi.beta;
  const cplx<T> *C = Call + cstride * oi.dist;
  fill_phase<T>(ph, p, oi.phi);
  __syncthreads();
  const int ps = p * p;
  cplx<T> out[R];
  for (int q = ch.y; q < ch.z; q++) {
    int tg = ptgt[q], sr = psrc[q];
    for (int r = 0; r < nrhs; r++) {
      rcr_job<T, GS, R>(H, C, p, p, p, Min + ((size_t)sr * nrhs + r) * ps, mtab,
                        buf, ph, out);
      cplx<T> *dst = Lout + ((size_t)tg * nrhs + r) * ps;
#pragma unroll
      for (int k = 0; k < R; k++) {
        int f = threadIdx.x + GS * k;
        if (f < ps) atomic_add_c(dst + f, out[k]);
      }
    }
  }
}

// M2M: one block per parent, children of level l -> parent at level l-1
template <typename T, int GS, int R>
__global__ void __launch_bounds__(GS)
    k_m2m(const int *__restrict__ cstart, const int *__restrict__ ckeys,
          const int *__restrict__ obeta, const double *__restrict__ ophi,
          const T *__restrict__ Hall, size_t hstride,
          const cplx<T> *__restrict__ C, int P, int pc, int pp,
          const int *__restrict__ mtab, const cplx<T> *__restrict__ Mc,
          cplx<T> *__restrict__ Mp, int nrhs) {
  extern __shared__ unsigned char smem[];
  int Pm = pc > pp ? pc : pp;
  cplx<T> *buf = (cplx<T> *)smem;
  cplx<T> *ph = buf + Pm * Pm;
  int pb = blockIdx.x;
  int c0 = cstart[pb], c1 = cstart[pb + 1];
  for (int r = 0; r < nrhs; r++) {
    cplx<T> acc[R];
#pragma unroll
    for (int k = 0; k < R; k++) acc[k] = cmk<T>(0, 0);
    for (int c = c0; c < c1; c++) {
      int oct = ckeys[c] & 7;
      __syncthreads();
      fill_phase<T>(ph, Pm, ophi[oct]);
      __syncthreads();
      cplx<T> out[R];
      rcr_job<T, GS, R>(Hall + hstride * obeta[oct], C, P, pc, pp,
                        Mc + ((size_t)c * nrhs + r) * pc * pc, mtab, buf, ph,
                        out);
#pragma unroll
      for (int k = 0; k < R; k++) acc[k] = cadd(acc[k], out[k]);
    }
    cplx<T> *dst = Mp + ((size_t)pb * nrhs + r) * pp * pp;
#pragma unroll
    for (int k = 0; k < R; k++) {
      int f = threadIdx.x + GS * k;
      if (f < pp * pp) dst[f] = acc[k];
    }
  }
}

// L2L: one block per child, parent at level l-1 -> child at level l (adds)
template <typename T, int GS, int R>
__global__ void __launch_bounds__(GS)
    k_l2l(const int *__restrict__ parent, const int *__restrict__ ckeys,
          const int *__restrict__ obeta, const double *__restrict__ ophi,
          const T *__restrict__ Hall, size_t hstride,
          const cplx<T> *__restrict__ C, int P, int pp, int pc,
          const int *__restrict__ mtab, const cplx<T> *__restrict__ Lp,
          cplx<T> *__restrict__ Lc, int nrhs) {
  extern __shared__ unsigned char smem[];
  int Pm = pc > pp ? pc : pp;
  cplx<T> *buf = (cplx<T> *)smem;
  cplx<T> *ph = buf + Pm * Pm;
  int cb = blockIdx.x;
  int oct = ckeys[cb] & 7, pb = parent[cb];
  fill_phase<T>(ph, Pm, ophi[oct]);
  __syncthreads();
  for (int r = 0; r < nrhs; r++) {
    cplx<T> out[R];
    rcr_job<T, GS, R>(Hall + hstride * obeta[oct], C, P, pp, pc,
                      Lp + ((size_t)pb * nrhs + r) * pp * pp, mtab, buf, ph,
                      out);
    cplx<T> *dst = Lc + ((size_t)cb * nrhs + r) * pc * pc;
#pragma unroll
    for (int k = 0; k < R; k++) {
      int f = threadIdx.x + GS * k;
      if (f < pc * pc) dst[f] = cadd(dst[f], out[k]);
    }
  }
}

// Start of a pass, one launch: a block per leaf box moves the box's elements
// from the caller's order to xs and sums M[b][r][f] = sum_{e in b} B[e][f]
// xs[r][e] (B NULL: only moves them); the blocks after those clear the
// coefficient arrays that the translations add into.  FLIP multiplies
// coefficient f = (n, m) by (-1)^n: with B = the L2P basis it is the
// transposed L2P of the transposed pass.  As a gather, a P2M and up to eight
// fills the start took 24 of the 123 us of a 1,280-triangle product, now 5.
struct Clear {
  int n;
  size_t end[2 * FMB_MAXLEV];  // running 8-byte words
  double *p[2 * FMB_MAXLEV];
};
constexpr int kBegin = 256, kBeginE = 32;

template <typename T, bool FLIP, int RC>
__global__ void __launch_bounds__(kBegin)
    k_begin(const int *__restrict__ bstart, const int *__restrict__ perm,
            const cplx<T> *__restrict__ B, const double2 *__restrict__ x, int N, int ps,
            cplx<T> *__restrict__ xs, cplx<T> *__restrict__ M, int nrhs, int nbox, Clear cl) {
  __shared__ cplx<T> xl[RC][kBeginE];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= nbox) {
    const size_t step = (size_t)(gridDim.x - nbox) * kBegin;
    size_t i = (size_t)(blockIdx.x - nbox) * kBegin + tid, base = 0;
    for (int s = 0; s < cl.n; s++) {
      for (; i < cl.end[s]; i += step) cl.p[s][i - base] = 0.0;
      base = cl.end[s];
    }
    return;
  }
  const int b = xcd_block(blockIdx.x, nbox);
  const int e0 = bstart[b], e1 = bstart[b + 1];
  for (int r0 = 0; r0 < nrhs; r0 += RC) {
    const int nr = min(RC, nrhs - r0);
    for (int f0 = 0; f0 < ps; f0 += kBegin) {
      const int f = f0 + tid;
      cplx<T> s[RC];
#pragma unroll
      for (int r = 0; r < RC; r++) s[r] = cmk<T>(0, 0);
      for (int c0 = e0; c0 < e1; c0 += kBeginE) {
        const int ne = min(kBeginE, e1 - c0);
        __syncthreads();
        if (tid < RC * kBeginE) {
          const int r = tid / kBeginE, e = tid % kBeginE;
          if (r < nr && e < ne) {
            const double2 v = x[(size_t)(r0 + r) * N + perm[c0 + e]];
            const cplx<T> z = cmk<T>((T)v.x, (T)v.y);
            xl[r][e] = z;
            if (f0 == 0) xs[(size_t)(r0 + r) * N + c0 + e] = z;
          }
        }
        __syncthreads();
        if (!B || f >= ps) continue;
#pragma unroll 4
        for (int e = 0; e < ne; e++) {
          const cplx<T> be = B[(size_t)(c0 + e) * ps + f];
#pragma unroll
          for (int r = 0; r < RC; r++) cfma(s[r], be, xl[r][e]);
        }
      }
      if (!B) break;
      if (f >= ps) continue;
      const bool neg = FLIP && (isqrt_fix(f) & 1);
#pragma unroll
      for (int r = 0; r < RC; r++)
        if (r < nr)
          M[((size_t)b * nrhs + r0 + r) * ps + f] = neg ? cmk<T>(-s[r].re, -s[r].im) : s[r];
    }
  }
}

inline int nblk(size_t n, int b = 256) { return (int)((n + b - 1) / b); }

struct Shape {
  int gs, r;
};
inline Shape shape_for(int pm) {
  int q = pm * pm;
  if (q > 512 * 32) return {0, 0};
  if (q <= 256) return {64, 4};
  if (q <= 512) return {64, 8};
  if (q <= 1024) return {256, 4};
  if (q <= 2048) return {256, 8};
  if (q <= 4096) return {256, 16};
  if (q <= 8192) return {512, 16};
  return {512, 32};
}

template <typename K>
int set_lds(K kern, size_t bytes) {
  if (bytes > 160 * 1024)
    return fmb_set_error(FMB_ERR_RANGE, "translation needs %zu B of LDS", bytes);
  if (bytes > 64 * 1024) /* the CU's 160 KB: valid for every captured launch */
    FMB_HIP_CHECK(hipFuncSetAttribute((const void *)kern,
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      160 * 1024));
  return FMB_OK;
}

}  // namespace

// ---------------------------------------------------------------- launchers

struct fmbh_m2l_plan;  // opaque per-plan launch tables are kept on fmb_plan

extern "C" int fmbh_mmajor_table(int p, int **d_tab, void *stream) {
  int *h = (int *)malloc(sizeof(int) * p * p);
  int g = 0;
  for (int m = -(p - 1); m <= p - 1; m++) {
    int am = m < 0 ? -m : m;
    for (int np = am; np < p; np++) h[g++] = np * np + np + m;
  }
  int rc = fmbh_malloc((void **)d_tab, sizeof(int) * p * p);
  if (!rc) rc = fmbh_h2d(*d_tab, h, sizeof(int) * p * p, stream);
  free(h);
  return rc;
}

template <typename T, bool FLIP>
static int launch_begin(const fmb_plan *pl, const fmb_opset *o, const fmb_c64 *x, int nrhs,
                        const void *B, void *M, const Clear &cl, hipStream_t st) {
  const fmb_tree *t = pl->tree;
  const int nb = t->nbox[t->lmax], ps = pl->p[t->lmax] * pl->p[t->lmax];
  const size_t w = cl.n ? cl.end[cl.n - 1] : 0;
  size_t zb = (w + 4 * kBegin - 1) / (4 * kBegin);
  if (zb > 2048) zb = 2048;
  // the basis is read once for up to eight right-hand sides
  auto kern = nrhs == 1   ? k_begin<T, FLIP, 1>
              : nrhs == 2 ? k_begin<T, FLIP, 2>
              : nrhs <= 4 ? k_begin<T, FLIP, 4>
                          : k_begin<T, FLIP, 8>;
  hipLaunchKernelGGL(kern, dim3(nb + (unsigned)zb), dim3(kBegin), 0, st, t->d_box_start, t->d_perm,
                     (const cplx<T> *)B, (const double2 *)x, t->nelem, ps, (cplx<T> *)o->d_xs,
                     (cplx<T> *)M, nrhs, nb, cl);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_begin(const fmb_plan *pl, int op, int what, const fmb_c64 *x, int nrhs,
                          void *stream) {
  const fmb_tree *t = pl->tree;
  const fmb_opset *o = &pl->ops[op];
  const int L = t->lmax, trans = what == FMBH_BEGIN_T;
  hipStream_t st = (hipStream_t)stream;
  // parents receive the translations of their children as sums, and every
  // level those of the interaction lists
  Clear cl;
  cl.n = 0;
  size_t end = 0;
  for (int l = 2; l <= L && what != FMBH_BEGIN_NEAR; l++) {
    const size_t words = (size_t)t->nbox[l] * nrhs * pl->p[l] * pl->p[l] * o->csz / 8;
    for (int out = 0; out < 2; out++) {
      if (out ? what == FMBH_BEGIN_UP : l == L) continue;
      cl.p[cl.n] = (double *)(out != trans ? o->d_L[l] : o->d_M[l]);
      cl.end[cl.n++] = end += words;
    }
  }
  void *M = trans ? o->d_L[L] : o->d_M[L];
  const void *B = what == FMBH_BEGIN_NEAR ? NULL : trans ? o->d_L2P : o->d_P2M;
  if (o->prec == FMB_FP64)
    return trans ? launch_begin<double, true>(pl, o, x, nrhs, B, M, cl, st)
                 : launch_begin<double, false>(pl, o, x, nrhs, B, M, cl, st);
  return trans ? launch_begin<float, true>(pl, o, x, nrhs, B, M, cl, st)
               : launch_begin<float, false>(pl, o, x, nrhs, B, M, cl, st);
}

template <typename T, int GS, int R>
static int launch_m2l(const fmb_plan *pl, const fmb_opset *o, int l, int nrhs,
                      hipStream_t st) {
  const fmb_tree *t = pl->tree;
  int p = pl->p[l];
  size_t lds = sizeof(cplx<T>) * (size_t)(p * p + p);
  auto kern = k_m2l<T, GS, R>;
  int rc = set_lds(kern, lds);
  if (rc) return rc;
  const int4 *chunks = (const int4 *)pl->d_m2l_chunks[l];
  hipLaunchKernelGGL(kern, dim3(pl->n_m2l_chunks[l]), dim3(GS), lds, st, chunks,
                     (const OffInfo *)pl->d_off_info, t->d_pair_tgt[l],
                     t->d_pair_src[l], (const T *)o->d_H,
                     (size_t)rot_off(pl->Pmax), (const cplx<T> *)o->d_Csr[l],
                     (size_t)coax_size(p), p, pl->d_tab_mmajor[l],
                     (const cplx<T> *)o->d_M[l], (cplx<T> *)o->d_L[l], nrhs);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

template <typename T>
static int dispatch_m2l(const fmb_plan *pl, const fmb_opset *o, int l,
                        int nrhs, hipStream_t st) {
  Shape s = shape_for(pl->p[l]);
#define CASE(G, RR)                                                            \
  if (s.gs == G && s.r == RR) return launch_m2l<T, G, RR>(pl, o, l, nrhs, st);
  CASE(64, 4) CASE(64, 8) CASE(256, 4) CASE(256, 8) CASE(256, 16) CASE(512, 16)
  CASE(512, 32)
#undef CASE
  return fmb_set_error(FMB_ERR_RANGE, "no M2L shape for p=%d", pl->p[l]);
}

extern "C" int fmbh_m2l(const fmb_plan *pl, int op, int l, int nrhs,
                        void *stream) {
  if (pl->n_m2l_chunks[l] == 0) return FMB_OK;
  const fmb_opset *o = &pl->ops[op];
  if (o->prec == FMB_FP64)
    return dispatch_m2l<double>(pl, o, l, nrhs, (hipStream_t)stream);
  return dispatch_m2l<float>(pl, o, l, nrhs, (hipStream_t)stream);
}

template <typename T, int GS, int R>
static int launch_m2m(const fmb_plan *pl, const fmb_opset *o, int l, int nrhs,
                      hipStream_t st) {
  const fmb_tree *t = pl->tree;
  int pc = pl->p[l], pp = pl->p[l - 1], Pm = pc > pp ? pc : pp;
  size_t lds = sizeof(cplx<T>) * (size_t)(Pm * Pm + Pm);
  auto kern = k_m2m<T, GS, R>;
  int rc = set_lds(kern, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(t->nbox[l - 1]), dim3(GS), lds, st,
                     t->d_cstart[l - 1], t->d_keys[l], pl->d_m2m_beta,
                     pl->d_m2m_phi, (const T *)o->d_H,
                     (size_t)rot_off(pl->Pmax), (const cplx<T> *)o->d_Cm2m[l],
                     Pm, pc, pp, pl->d_tab_mmajor[l - 1],
                     (const cplx<T> *)o->d_M[l], (cplx<T> *)o->d_M[l - 1], nrhs);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

template <typename T>
static int dispatch_m2m(const fmb_plan *pl, const fmb_opset *o, int l,
                        int nrhs, hipStream_t st) {
  int pm = pl->p[l] > pl->p[l - 1] ? pl->p[l] : pl->p[l - 1];
  Shape s = shape_for(pm);
#define CASE(G, RR)                                                            \
  if (s.gs == G && s.r == RR) return launch_m2m<T, G, RR>(pl, o, l, nrhs, st);
  CASE(64, 4) CASE(64, 8) CASE(256, 4) CASE(256, 8) CASE(256, 16) CASE(512, 16)
  CASE(512, 32)
#undef CASE
  return fmb_set_error(FMB_ERR_RANGE, "no M2M shape for p=%d", pm);
}

extern "C" int fmbh_m2m(const fmb_plan *pl, int op, int l, int nrhs,
                        void *stream) {
  const fmb_opset *o = &pl->ops[op];
  if (o->prec == FMB_FP64)
    return dispatch_m2m<double>(pl, o, l, nrhs, (hipStream_t)stream);
  return dispatch_m2m<float>(pl, o, l, nrhs, (hipStream_t)stream);
}

template <typename T, int GS, int R>
static int launch_l2l(const fmb_plan *pl, const fmb_opset *o, int l, int nrhs,
                      hipStream_t st) {
  const fmb_tree *t = pl->tree;
  int pc = pl->p[l], pp = pl->p[l - 1], Pm = pc > pp ? pc : pp;
  size_t lds = sizeof(cplx<T>) * (size_t)(Pm * Pm + Pm);
  auto kern = k_l2l<T, GS, R>;
  int rc = set_lds(kern, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(t->nbox[l]), dim3(GS), lds, st, t->d_parent[l],
                     t->d_keys[l], pl->d_l2l_beta, pl->d_l2l_phi,
                     (const T *)o->d_H, (size_t)rot_off(pl->Pmax),
                     (const cplx<T> *)o->d_Cl2l[l], Pm, pp, pc,
                     pl->d_tab_mmajor[l], (const cplx<T> *)o->d_L[l - 1],
                     (cplx<T> *)o->d_L[l], nrhs);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

template <typename T>
static int dispatch_l2l(const fmb_plan *pl, const fmb_opset *o, int l,
                        int nrhs, hipStream_t st) {
  int pm = pl->p[l] > pl->p[l - 1] ? pl->p[l] : pl->p[l - 1];
  Shape s = shape_for(pm);
#define CASE(G, RR)                                                            \
  if (s.gs == G && s.r == RR) return launch_l2l<T, G, RR>(pl, o, l, nrhs, st);
  CASE(64, 4) CASE(64, 8) CASE(256, 4) CASE(256, 8) CASE(256, 16) CASE(512, 16)
  CASE(512, 32)
#undef CASE
  return fmb_set_error(FMB_ERR_RANGE, "no L2L shape for p=%d", pm);
}

extern "C" int fmbh_l2l(const fmb_plan *pl, int op, int l, int nrhs,
                        void *stream) {
  const fmb_opset *o = &pl->ops[op];
  if (o->prec == FMB_FP64)
    return dispatch_l2l<double>(pl, o, l, nrhs, (hipStream_t)stream);
  return dispatch_l2l<float>(pl, o, l, nrhs, (hipStream_t)stream);
}
