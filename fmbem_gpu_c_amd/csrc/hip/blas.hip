// blas.hip -- FP64 complex vector kernels for GMRES (batched over right-hand
// sides) and the plane-wave right-hand side.  Reductions sum the partial sums
// of a number of blocks fixed by N, in block order, so results do not depend
// on scheduling.
#include "fmb_device.h"

namespace {

constexpr int BS = 256;
// blocks per inner product and per vector update at most: an inner product has nv nrhs rows of
// blocks beside each other, an update only nrhs
constexpr int DOT_CHUNKS = 128, UPD_CHUNKS = 2048;
// Blocks up to which a reduction completes in its own launch.  Each block of such a launch releases
// its partial sum, which writes its XCD's L2 back: 16 ns a block, one after the other, against 3 us
// for a launch.  A step over 30 vectors, two right-hand sides of 10,580 elements (2,520 blocks an
// inner product): 36 us with a launch of its own for the sums, 187 without (with an acquire in
// every block too); over 29, nine of 327,680 (33,408): 1.31 ms, its bytes at the rate of a copy,
// against 8.4.
constexpr size_t kOneLaunch = 64;

// sum of v over the block in a fixed order, in every thread
__device__ __forceinline__ double block_sum(double v, double *sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0.0;
  for (int i = 0; i < BS / 64; i++) r += sh[i];
  return r;
}

// Whether this block is the last of the n of reduction q to arrive: it then reads the others'
// partial sums and completes the reduction, so a reduction takes one launch and its order does
// not depend on which block is last.  Leaves the counter at 0.  A release writes the XCD's L2
// back, so this is for launches of few blocks (kOneLaunch).
__device__ __forceinline__ bool last_block(unsigned *cnt, int q, unsigned n) {
  __shared__ unsigned seen;
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    seen = __hip_atomic_fetch_add(cnt + q, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (seen == n - 1) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      cnt[q] = 0u;
    }
  }
  __syncthreads();
  return seen == n - 1;
}

// elements [i0, i1) of chunk c of C
__device__ __forceinline__ void chunk_range(int N, int c, int C, int &i0, int &i1) {
  const int per = (N + C - 1) / C;
  i0 = min(per * c, N);
  i1 = min(i0 + per, N);
}

// partial sums of row q -> its inner product, in every thread
__device__ __forceinline__ double2 sum_dots(const double2 *part, int q, int C, double *sh) {
  double2 t = make_double2(0.0, 0.0);
  if (threadIdx.x < C) t = part[(size_t)q * C + threadIdx.x];
  t.x = block_sum(t.x, sh);
  t.y = block_sum(t.y, sh);
  return t;
}
static_assert(DOT_CHUNKS <= BS, "a thread per partial sum");
// the same of a sum of squares -> its root
__device__ __forceinline__ double sum_norm(const double *part, int r, int C, double *sh) {
  double s = 0.0;
  for (int i = threadIdx.x; i < C; i += BS) s += part[(size_t)r * C + i];
  return sqrt(block_sum(s, sh));
}

// h[j nrhs + r] = <V_j^r, w^r>, also to hp (host memory): grid (chunks, vectors x right-hand
// sides).  cnt NULL: only the partial sums, which k_sum_dots completes.
__global__ void __launch_bounds__(BS)
    k_dots(const double2 *__restrict__ V, int nrhs, int N, const double2 *__restrict__ w,
           double2 *__restrict__ part, unsigned *__restrict__ cnt, double2 *__restrict__ h,
           double2 *__restrict__ hp) {
  __shared__ double sh[BS / 64];
  const int C = gridDim.x, c = blockIdx.x, jr = blockIdx.y, r = jr % nrhs;
  const double2 *v = V + (size_t)jr * N, *x = w + (size_t)r * N;
  int i0, i1;
  chunk_range(N, c, C, i0, i1);
  double sr = 0, si = 0;
  for (int i = i0 + threadIdx.x; i < i1; i += BS) {
    const double2 a = v[i], b = x[i];
    sr += a.x * b.x + a.y * b.y;
    si += a.x * b.y - a.y * b.x;
  }
  sr = block_sum(sr, sh);
  si = block_sum(si, sh);
  if (C > 1) {
    if (threadIdx.x == 0) part[(size_t)jr * C + c] = make_double2(sr, si);
    if (!cnt || !last_block(cnt, jr, C)) return;
    const double2 t = sum_dots(part, jr, C, sh);
    sr = t.x;
    si = t.y;
  }
  if (threadIdx.x == 0) h[jr] = hp[jr] = make_double2(sr, si);
}

// a block a row
__global__ void __launch_bounds__(BS)
    k_sum_dots(const double2 *__restrict__ part, int C, double2 *__restrict__ h,
               double2 *__restrict__ hp) {
  __shared__ double sh[BS / 64];
  const int q = blockIdx.x;
  const double2 t = sum_dots(part, q, C, sh);
  if (threadIdx.x == 0) h[q] = hp[q] = t;
}
__global__ void __launch_bounds__(BS)
    k_sum_norms(const double *__restrict__ part, int C, double *__restrict__ nrm,
                double *__restrict__ hp) {
  __shared__ double sh[BS / 64];
  const int r = blockIdx.x;
  const double n = sum_norm(part, r, C, sh);
  if (threadIdx.x == 0) nrm[r] = hp[r] = n;
}

// |w|^2 of the block's chunk -> norm of right-hand side r (cnt NULL: k_sum_norms completes it)
__device__ __forceinline__ void norm_end(double s, double *sh, double *part, unsigned *cnt, int r,
                                         double *nrm, double *hp) {
  const int C = gridDim.x, c = blockIdx.x;
  s = block_sum(s, sh);
  if (C > 1) {
    if (threadIdx.x == 0) part[(size_t)r * C + c] = s;
    if (!cnt || !last_block(cnt, r, C)) return;
    s = sum_norm(part, r, C, sh);
  } else {
    s = sqrt(s);
  }
  if (threadIdx.x == 0) nrm[r] = hp[r] = s;
}

// w^r += sign sum_j h[j nrhs + r] V_j^r, and with NORM |w^r|: grid (chunks, right-hand sides)
template <bool NORM>
__global__ void __launch_bounds__(BS)
    k_gemv(const double2 *__restrict__ V, int nv, const double2 *__restrict__ h,
           double2 *__restrict__ w, int nrhs, int N, double sign, double *__restrict__ part,
           unsigned *__restrict__ cnt, double *__restrict__ nrm, double *__restrict__ hp) {
  __shared__ double sh[BS / 64];
  const int r = blockIdx.y;
  int i0, i1;
  chunk_range(N, blockIdx.x, gridDim.x, i0, i1);
  double s = 0.0;
  for (int i = i0 + threadIdx.x; i < i1; i += BS) {
    double sr = 0, si = 0;
#pragma unroll 8
    for (int j = 0; j < nv; j++) {
      const double2 a = h[(size_t)j * nrhs + r], v = V[((size_t)j * nrhs + r) * N + i];
      sr += a.x * v.x - a.y * v.y;
      si += a.x * v.y + a.y * v.x;
    }
    double2 y = w[(size_t)r * N + i];
    y.x += sign * sr;
    y.y += sign * si;
    w[(size_t)r * N + i] = y;
    s += y.x * y.x + y.y * y.y;
  }
  if constexpr (NORM) norm_end(s, sh, part, cnt, r, nrm, hp);
}

// r = b - w (w NULL: r = b; r NULL: only the norm) and |r|
__global__ void __launch_bounds__(BS)
    k_resid(const double2 *__restrict__ b, const double2 *__restrict__ w, double2 *__restrict__ res,
            int N, double *__restrict__ part, unsigned *__restrict__ cnt,
            double *__restrict__ nrm, double *__restrict__ hp) {
  __shared__ double sh[BS / 64];
  const size_t o = (size_t)blockIdx.y * N;
  int i0, i1;
  chunk_range(N, blockIdx.x, gridDim.x, i0, i1);
  double s = 0.0;
  for (int i = i0 + threadIdx.x; i < i1; i += BS) {
    double2 y = b[o + i];
    if (w) {
      const double2 v = w[o + i];
      y.x -= v.x;
      y.y -= v.y;
    }
    if (res) res[o + i] = y;
    s += y.x * y.x + y.y * y.y;
  }
  norm_end(s, sh, part, cnt, blockIdx.y, nrm, hp);
}

// y^r = x^r / nrm[r] (0 for a zero norm)
__global__ void __launch_bounds__(BS)
    k_unit(const double2 *__restrict__ x, const double *__restrict__ nrm, double2 *__restrict__ y,
           int nrhs, int N) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)N * nrhs) return;
  const double n = nrm[t / N], f = n > 0 ? 1.0 / n : 0.0;
  y[t] = make_double2(f * x[t].x, f * x[t].y);
}

// y += x
__global__ void __launch_bounds__(BS)
    k_add(const double2 *__restrict__ x, double2 *__restrict__ y, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = make_double2(y[t].x + x[t].x, y[t].y + x[t].y);
}

__global__ void k_rhs_plane(const double *__restrict__ geo,
                            const int *__restrict__ iperm, const double *__restrict__ dirs,
                            int nrhs, int N, double k, double alre, double alim,
                            double2 *__restrict__ b) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)N * nrhs) return;
  int r = (int)(t / N), e = (int)(t % N);
  const double *g = geo + 8 * (size_t)iperm[e];
  const double *d = dirs + 3 * r;
  double dx = d[0] * g[0] + d[1] * g[1] + d[2] * g[2];
  double dn = d[0] * g[3] + d[1] * g[4] + d[2] * g[5];
  double s, c;
  sincos(k * dx, &s, &c);
  // e^{ik d.x} (1 + alpha i k d.n)
  double fr = 1.0 - alim * k * dn, fi = alre * k * dn;
  b[t] = make_double2(c * fr - s * fi, c * fi + s * fr);
}

// x0 = x e^{i dk d_r . c_e}, caller order; in place when x0 == x
__global__ void k_sweep_guess(const double *__restrict__ geo,
                              const int *__restrict__ iperm,
                              const double *__restrict__ dirs, int nrhs, int N,
                              double dk, const double2 *x, double2 *x0) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)N * nrhs) return;
  int r = (int)(t / N), e = (int)(t % N);
  double2 v = x[t];
  if (dirs) {
    const double *g = geo + 8 * (size_t)iperm[e];
    const double *d = dirs + 3 * r;
    double s, c;
    sincos(dk * (d[0] * g[0] + d[1] * g[1] + d[2] * g[2]), &s, &c);
    v = make_double2(v.x * c - v.y * s, v.x * s + v.y * c);
  }
  x0[t] = v;
}

// dJ/dsigma_j = sum_r 2 conj(w_rj), w_rj = -x_rj (c_rj + s_rj)
__global__ void k_adj_combine(const double2 *__restrict__ x, const double2 *__restrict__ c,
                              const double2 *__restrict__ s, int nrhs, int N,
                              double2 *__restrict__ g) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= N) return;
  double gr = 0.0, gi = 0.0;
  for (int r = 0; r < nrhs; r++) {
    size_t i = (size_t)r * N + j;
    double2 xv = x[i], a = make_double2(c[i].x + s[i].x, c[i].y + s[i].y);
    double wr = -(xv.x * a.x - xv.y * a.y), wi = -(xv.x * a.y + xv.y * a.x);
    gr += 2.0 * wr;
    gi -= 2.0 * wi;
  }
  g[j] = make_double2(gr, gi);
}

inline int nblk(size_t n, int b = 256) { return (int)((n + b - 1) / b); }

}  // namespace

// blocks over N elements: one element a thread up to the limit
static int chunks_for(int N, int limit) {
  const int c = (N + BS - 1) / BS;
  return c < 1 ? 1 : (c > limit ? limit : c);
}

// counters of a reduction of grid g, NULL where a launch of its own completes it
static unsigned *counters(const fmbh_vecws *ws, dim3 g) {
  return (size_t)g.x * g.y <= kOneLaunch ? ws->cnt : NULL;
}
static int sum_norms(dim3 g, const fmbh_vecws *ws, hipStream_t st) {
  if (g.x == 1 || counters(ws, g)) return FMB_OK;
  hipLaunchKernelGGL(k_sum_norms, dim3(g.y), dim3(BS), 0, st, (const double *)ws->part, (int)g.x,
                     ws->nrm, ws->hpn);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}
static int dots(const double2 *V, int nv, const double2 *w, int nrhs, int N, const fmbh_vecws *ws,
                fmb_c64 *h, fmb_c64 *hp, hipStream_t st) {
  const dim3 g(chunks_for(N, DOT_CHUNKS), nv * nrhs);
  double2 *part = (double2 *)ws->part;
  unsigned *cnt = counters(ws, g);
  hipLaunchKernelGGL(k_dots, g, dim3(BS), 0, st, V, nrhs, N, w, part, cnt, (double2 *)h,
                     (double2 *)hp);
  FMB_LAUNCH_CHECK();
  if (g.x == 1 || cnt) return FMB_OK;
  hipLaunchKernelGGL(k_sum_dots, dim3(g.y), dim3(BS), 0, st, (const double2 *)part, (int)g.x,
                     (double2 *)h, (double2 *)hp);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

// Layout of the vector workspace: partial sums, counters, h1, h2, norms; the host mirror holds
// h1, h2, norms
static size_t ws_part(int nv, int nrhs, int N) {
  const size_t d = sizeof(double2) * chunks_for(N, DOT_CHUNKS) * (size_t)nv * nrhs;
  const size_t u = (sizeof(double) * chunks_for(N, UPD_CHUNKS) * (size_t)nrhs + 15) & ~(size_t)15;
  return d > u ? d : u;
}
static size_t ws_cnt(int nv, int nrhs) {
  return (sizeof(unsigned) * (size_t)nv * nrhs + 15) & ~(size_t)15;
}

extern "C" size_t fmbh_vecws_host_bytes(int nv, int nrhs) {
  return sizeof(double2) * 2 * (size_t)nv * nrhs + sizeof(double) * (size_t)nrhs;
}
extern "C" size_t fmbh_vecws_bytes(int nv, int nrhs, int N) {
  return ws_part(nv, nrhs, N) + ws_cnt(nv, nrhs) + fmbh_vecws_host_bytes(nv, nrhs);
}

extern "C" int fmbh_vecws_init(fmbh_vecws *ws, void *dev, void *host, int nv, int nrhs, int N,
                               void *stream) {
  char *d = (char *)dev + ws_part(nv, nrhs, N);
  ws->part = dev;
  ws->cnt = (unsigned *)d;
  ws->h1 = (fmb_c64 *)(d + ws_cnt(nv, nrhs));
  ws->h2 = ws->h1 + (size_t)nv * nrhs;
  ws->nrm = (double *)(ws->h2 + (size_t)nv * nrhs);
  ws->hp1 = (fmb_c64 *)host;
  ws->hp2 = ws->hp1 + (size_t)nv * nrhs;
  ws->hpn = (double *)(ws->hp2 + (size_t)nv * nrhs);
  return fmbh_memset(ws->cnt, 0, ws_cnt(nv, nrhs), stream);
}

// One Arnoldi step: w -= V (V^H w) twice (classical Gram-Schmidt with one reorthogonalisation),
// |w|, V_nv = w / |w|.  The inner products of both passes and the norms reach the host mirror; the
// caller waits for the stream once.  A small solve is bound by launches and waits: five to eight
// launches and no transfers, 21 us over ten vectors of 1,280 elements, where ten launches, six
// transfers, three allocations and eleven waits took 0.19 ms.
extern "C" int fmbh_arnoldi(fmb_c64 *d_V, int nv, fmb_c64 *d_w, int nrhs, int N,
                            const fmbh_vecws *ws, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  double2 *V = (double2 *)d_V, *w = (double2 *)d_w;
  const dim3 gv(chunks_for(N, UPD_CHUNKS), nrhs), blk(BS);
  int rc;
  if ((rc = dots(V, nv, w, nrhs, N, ws, ws->h1, ws->hp1, st))) return rc;
  hipLaunchKernelGGL(k_gemv<false>, gv, blk, 0, st, V, nv, (const double2 *)ws->h1, w, nrhs, N,
                     -1.0, nullptr, nullptr, nullptr, nullptr);
  FMB_LAUNCH_CHECK();
  if ((rc = dots(V, nv, w, nrhs, N, ws, ws->h2, ws->hp2, st))) return rc;
  hipLaunchKernelGGL(k_gemv<true>, gv, blk, 0, st, V, nv, (const double2 *)ws->h2, w, nrhs, N,
                     -1.0, (double *)ws->part, counters(ws, gv), ws->nrm, ws->hpn);
  FMB_LAUNCH_CHECK();
  if ((rc = sum_norms(gv, ws, st))) return rc;
  return fmbh_unit(d_w, ws->nrm, d_V + (size_t)nv * nrhs * N, nrhs, N, stream);
}

extern "C" int fmbh_resid(const fmb_c64 *d_b, const fmb_c64 *d_w, fmb_c64 *d_r, int nrhs, int N,
                          const fmbh_vecws *ws, void *stream) {
  const dim3 g(chunks_for(N, UPD_CHUNKS), nrhs);
  hipLaunchKernelGGL(k_resid, g, dim3(BS), 0, (hipStream_t)stream, (const double2 *)d_b,
                     (const double2 *)d_w, (double2 *)d_r, N, (double *)ws->part, counters(ws, g),
                     ws->nrm, ws->hpn);
  FMB_LAUNCH_CHECK();
  return sum_norms(g, ws, (hipStream_t)stream);
}

extern "C" int fmbh_unit(const fmb_c64 *d_x, const double *d_nrm, fmb_c64 *d_y, int nrhs, int N,
                         void *stream) {
  hipLaunchKernelGGL(k_unit, dim3(nblk((size_t)N * nrhs)), dim3(BS), 0, (hipStream_t)stream,
                     (const double2 *)d_x, d_nrm, (double2 *)d_y, nrhs, N);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_zgemv_add(const fmb_c64 *d_V, int nv, const fmb_c64 *d_y, fmb_c64 *d_x,
                              int nrhs, int N, void *stream) {
  hipLaunchKernelGGL(k_gemv<false>, dim3(chunks_for(N, UPD_CHUNKS), nrhs), dim3(BS), 0,
                     (hipStream_t)stream, (const double2 *)d_V, nv, (const double2 *)d_y,
                     (double2 *)d_x, nrhs, N, 1.0, nullptr, nullptr, nullptr, nullptr);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_zadd(const fmb_c64 *d_x, fmb_c64 *d_y, size_t n, void *stream) {
  hipLaunchKernelGGL(k_add, dim3(nblk(n)), dim3(BS), 0, (hipStream_t)stream,
                     (const double2 *)d_x, (double2 *)d_y, n);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_rhs_plane(const fmb_plan *pl, const double *h_dirs,
                              int nrhs, fmb_c64 *d_b, void *stream) {
  const fmb_tree *t = pl->tree;
  double *d_dirs;
  int rc = fmbh_malloc((void **)&d_dirs, sizeof(double) * 3 * nrhs);
  if (rc) return rc;
  if ((rc = fmbh_h2d(d_dirs, h_dirs, sizeof(double) * 3 * nrhs, stream))) return rc;
  size_t n = (size_t)t->nelem * nrhs;
  hipLaunchKernelGGL(k_rhs_plane, dim3(nblk(n)), dim3(256), 0,
                     (hipStream_t)stream, t->d_geo, t->d_iperm, d_dirs, nrhs,
                     t->nelem, pl->k, pl->alpha_re, pl->alpha_im,
                     (double2 *)d_b);
  FMB_LAUNCH_CHECK();
  FMB_HIP_CHECK(hipStreamSynchronize((hipStream_t)stream));
  fmbh_free(d_dirs);
  return FMB_OK;
}

extern "C" int fmbh_sweep_guess(const fmb_plan *pl, double dk, const fmb_c64 *d_x,
                                const double *h_dirs, int nrhs, fmb_c64 *d_x0,
                                void *stream) {
  const fmb_tree *t = pl->tree;
  double *d_dirs = NULL;
  int rc;
  if (h_dirs) {
    if ((rc = fmbh_malloc((void **)&d_dirs, sizeof(double) * 3 * nrhs))) return rc;
    if ((rc = fmbh_h2d(d_dirs, h_dirs, sizeof(double) * 3 * nrhs, stream))) return rc;
  }
  size_t n = (size_t)t->nelem * nrhs;
  hipLaunchKernelGGL(k_sweep_guess, dim3(nblk(n)), dim3(256), 0,
                     (hipStream_t)stream, t->d_geo, t->d_iperm, d_dirs, nrhs,
                     t->nelem, dk, (const double2 *)d_x, (double2 *)d_x0);
  FMB_LAUNCH_CHECK();
  FMB_HIP_CHECK(hipStreamSynchronize((hipStream_t)stream));
  return fmbh_free(d_dirs);
}

extern "C" int fmbh_adjoint_combine(const fmb_c64 *x, const fmb_c64 *c, const fmb_c64 *s,
                                    int nrhs, int N, fmb_c64 *g, void *stream) {
  hipLaunchKernelGGL(k_adj_combine, dim3(nblk((size_t)N)), dim3(256), 0,
                     (hipStream_t)stream, (const double2 *)x, (const double2 *)c,
                     (const double2 *)s, nrhs, N, (double2 *)g);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}
