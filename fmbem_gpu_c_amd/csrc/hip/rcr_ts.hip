// rcr_ts.hip -- target-stationary M2L for the fine levels (orders up to 16).
//
// The same rotate-coaxial-rotate translation as rcr_kernels.h (translation.cu:1711-1808,
// 3580-3686).  There a workgroup takes 16 vectors (pair x right-hand side) of one offset and adds
// each result into its target with device-wide float atomics: 2 p^2 adds per vector, which the
// memory side performs at 1.0-1.3 TB/s whatever the kernel does.  At low orders that is most of
// the launch: the level-6 M2L of a 60,500-triangle ellipsoid with 64 right-hand sides (order 14,
// FP32) adds 47 GB in 55.6 ms.  Here a workgroup owns a group of targets, keeps their sums in LDS
// over all their sources and adds them into the level's coefficients once: 30.1 ms.  (Level 6 of
// the 20,480-triangle sphere, one right-hand side, order 14: FP64 1.17 -> 0.85 ms, FP32 0.75 ->
// 0.64 ms.)
//
//  * Classes.  The vectors of a batch must share the rotation blocks H(theta) and the coaxial
//    matrix C(|t|).  The 316 offsets fall into 34 classes of equal |dz| and dx^2 + dy^2: offsets
//    of a class differ by a rotation about z, which is a phase e^{i m phi}, and by the reflection
//    z -> -z, which multiplies coefficient (n, m) by (-1)^(n+m) on both sides.  Both go into a
//    table of phases per offset.  A group of 32 targets fills 0.84 of its 16-vector batches (one
//    right-hand side, 81,920-triangle sphere; by single offsets: 0.33).
//  * Layout.  A batch row is (n, m >= 0) with 64 lanes: {e re, e im, o re, o im} x 16 vectors,
//    e = z_m + z_-m and o = z_m - z_-m.  In these coordinates a rotation is an even and an odd
//    block of n + 1 rows, and the coaxial block |m| acts on e and o alike.  A row is one
//    conflict-free LDS access, and its address is uniform.
//  * Products.  One instruction multiplies a row by operator elements that all its lanes share:
//    FP32: v_mfma_f32_4x4x1 with the operator block broadcast (cbsz), four output rows at once
//    and no padding beyond 4 rows; the even and odd blocks ride in the two halves of one operand.
//    FP64: v_fmac_f64 with the operator element broadcast within rows of 16 lanes (DPP
//    row_newbcast), at the full vector rate, which equals the FP64 matrix rate; a 16x16x4 tile
//    would spend half its work on padding at these orders.
//  * Order of work.  A wave owns the rows of its degrees in both rotations, so a batch needs two
//    barriers: first rotation | coaxial | back rotation and, at once, the next batch's first.
//    Sources, phases and operators of the first unit are loaded before the barrier.
//  * Sums.  FP64: LDS double atomics (6 cycles a wave).  LDS float atomics take 177 cycles a wave
//    here, so FP32 adds by plain read and write, one vector of a target after the other; no two
//    waves share a row.  (Rows and sums: rcr_ts_rows.h.)
//
// What bounds it: instruction latency and the stages' serial chain at 16 waves per CU (FP32: two
// workgroups of 8; FP64: one of 16); the vector and matrix pipes are busy about half the time.
#include <hipcub/hipcub.hpp>
#include <type_traits>

#include "fmb_device.h"
#include "rcr_ts_rows.h"

namespace {

using namespace fmb_ts;
constexpr int kNC = FMB_NCLASS;

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, -1, 0x00020000);
}
__device__ __forceinline__ void ldz(cplx<float> &z, __amdgpu_buffer_rsrc_t r, int vo, int so) {
  z = __builtin_bit_cast(cplx<float>, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
}
__device__ __forceinline__ void ldz(cplx<double> &z, __amdgpu_buffer_rsrc_t r, int vo, int so) {
  z = __builtin_bit_cast(cplx<double>, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0));
}

// c[r] += a0[r] b0 + a1[r] b1 for 4 RG rows r, where lane r of every 16 lanes holds a[r].  (A
// vector instruction that writes a register read by DPP must lie two wait states back.)
#define FMB_FM(C, A, B, I) \
  "v_fmac_f64_dpp " C ", " A ", " B " row_newbcast:" I " row_mask:0xf bank_mask:0xf\n"
template <int RG>
__device__ __forceinline__ void fma_rows(double *c, double a0, double b0, double a1, double b1);
template <>
__device__ __forceinline__ void fma_rows<1>(double *c, double a0, double b0, double a1, double b1) {
  asm("s_nop 1\n"
      FMB_FM("%0", "%4", "%5", "0")
      FMB_FM("%1", "%4", "%5", "1")
      FMB_FM("%2", "%4", "%5", "2")
      FMB_FM("%3", "%4", "%5", "3")
      FMB_FM("%0", "%6", "%7", "0")
      FMB_FM("%1", "%6", "%7", "1")
      FMB_FM("%2", "%6", "%7", "2")
      FMB_FM("%3", "%6", "%7", "3")
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3])
      : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
}
template <>
__device__ __forceinline__ void fma_rows<2>(double *c, double a0, double b0, double a1, double b1) {
  asm("s_nop 1\n"
      FMB_FM("%0", "%8", "%9", "0")
      FMB_FM("%1", "%8", "%9", "1")
      FMB_FM("%2", "%8", "%9", "2")
      FMB_FM("%3", "%8", "%9", "3")
      FMB_FM("%4", "%8", "%9", "4")
      FMB_FM("%5", "%8", "%9", "5")
      FMB_FM("%6", "%8", "%9", "6")
      FMB_FM("%7", "%8", "%9", "7")
      FMB_FM("%0", "%10", "%11", "0")
      FMB_FM("%1", "%10", "%11", "1")
      FMB_FM("%2", "%10", "%11", "2")
      FMB_FM("%3", "%10", "%11", "3")
      FMB_FM("%4", "%10", "%11", "4")
      FMB_FM("%5", "%10", "%11", "5")
      FMB_FM("%6", "%10", "%11", "6")
      FMB_FM("%7", "%10", "%11", "7")
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]),
        "+&v"(c[5]), "+&v"(c[6]), "+&v"(c[7])
      : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
}
template <>
__device__ __forceinline__ void fma_rows<3>(double *c, double a0, double b0, double a1, double b1) {
  asm("s_nop 1\n"
      FMB_FM("%0", "%12", "%13", "0")
      FMB_FM("%1", "%12", "%13", "1")
      FMB_FM("%2", "%12", "%13", "2")
      FMB_FM("%3", "%12", "%13", "3")
      FMB_FM("%4", "%12", "%13", "4")
      FMB_FM("%5", "%12", "%13", "5")
      FMB_FM("%6", "%12", "%13", "6")
      FMB_FM("%7", "%12", "%13", "7")
      FMB_FM("%8", "%12", "%13", "8")
      FMB_FM("%9", "%12", "%13", "9")
      FMB_FM("%10", "%12", "%13", "10")
      FMB_FM("%11", "%12", "%13", "11")
      FMB_FM("%0", "%14", "%15", "0")
      FMB_FM("%1", "%14", "%15", "1")
      FMB_FM("%2", "%14", "%15", "2")
      FMB_FM("%3", "%14", "%15", "3")
      FMB_FM("%4", "%14", "%15", "4")
      FMB_FM("%5", "%14", "%15", "5")
      FMB_FM("%6", "%14", "%15", "6")
      FMB_FM("%7", "%14", "%15", "7")
      FMB_FM("%8", "%14", "%15", "8")
      FMB_FM("%9", "%14", "%15", "9")
      FMB_FM("%10", "%14", "%15", "10")
      FMB_FM("%11", "%14", "%15", "11")
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]),
        "+&v"(c[5]), "+&v"(c[6]), "+&v"(c[7]), "+&v"(c[8]), "+&v"(c[9]),
        "+&v"(c[10]), "+&v"(c[11])
      : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
}
template <>
__device__ __forceinline__ void fma_rows<4>(double *c, double a0, double b0, double a1, double b1) {
  asm("s_nop 1\n"
      FMB_FM("%0", "%16", "%17", "0")
      FMB_FM("%1", "%16", "%17", "1")
      FMB_FM("%2", "%16", "%17", "2")
      FMB_FM("%3", "%16", "%17", "3")
      FMB_FM("%4", "%16", "%17", "4")
      FMB_FM("%5", "%16", "%17", "5")
      FMB_FM("%6", "%16", "%17", "6")
      FMB_FM("%7", "%16", "%17", "7")
      FMB_FM("%8", "%16", "%17", "8")
      FMB_FM("%9", "%16", "%17", "9")
      FMB_FM("%10", "%16", "%17", "10")
      FMB_FM("%11", "%16", "%17", "11")
      FMB_FM("%12", "%16", "%17", "12")
      FMB_FM("%13", "%16", "%17", "13")
      FMB_FM("%14", "%16", "%17", "14")
      FMB_FM("%15", "%16", "%17", "15")
      FMB_FM("%0", "%18", "%19", "0")
      FMB_FM("%1", "%18", "%19", "1")
      FMB_FM("%2", "%18", "%19", "2")
      FMB_FM("%3", "%18", "%19", "3")
      FMB_FM("%4", "%18", "%19", "4")
      FMB_FM("%5", "%18", "%19", "5")
      FMB_FM("%6", "%18", "%19", "6")
      FMB_FM("%7", "%18", "%19", "7")
      FMB_FM("%8", "%18", "%19", "8")
      FMB_FM("%9", "%18", "%19", "9")
      FMB_FM("%10", "%18", "%19", "10")
      FMB_FM("%11", "%18", "%19", "11")
      FMB_FM("%12", "%18", "%19", "12")
      FMB_FM("%13", "%18", "%19", "13")
      FMB_FM("%14", "%18", "%19", "14")
      FMB_FM("%15", "%18", "%19", "15")
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]),
        "+&v"(c[5]), "+&v"(c[6]), "+&v"(c[7]), "+&v"(c[8]), "+&v"(c[9]),
        "+&v"(c[10]), "+&v"(c[11]), "+&v"(c[12]), "+&v"(c[13]), "+&v"(c[14]),
        "+&v"(c[15])
      : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
}
#undef FMB_FM

typedef float f4 __attribute__((ext_vector_type(4)));
struct V4 {
  float v[4];
};
struct V2 {
  double v[2];
};

// A block's operator, loaded by chunks of columns (load), and its products with the batch rows
// (run): 4 RG output rows of 64 lanes in registers.  Columns past the block are zero and meet
// rows clamped into the block, so they stay finite where the rows are.
template <typename T, int RG> struct Rot;
template <typename T, int RG> struct Coax;

template <int RG> struct Rot<float, RG> {
  static constexpr int NC = (RG + 1) / 2;  // chunks of 8 columns
  f4 c[RG];
  V4 A[NC];
  __device__ __forceinline__ float row(int i) const { return c[i >> 2][i & 3]; }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int aoff, int lane) {
#pragma unroll
    for (int h = 0; h < NC; h++)
      A[h] = __builtin_bit_cast(
          V4, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (aoff + 256 * h) * 4, 0));
  }
  __device__ __forceinline__ void run(const float *xb, int n) {
#pragma unroll
    for (int g = 0; g < RG; g++) c[g] = f4{0, 0, 0, 0};
#pragma unroll
    for (int h = 0; h < NC; h++) {
      float b[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int k = 8 * h + u;
        if (k < 4 * RG) b[u] = xb[(k <= 4 * RG - 4 ? k : min(k, n)) * kL];
      }
#define FMB_ROT(U)                                                        \
  if (8 * h + U < 4 * RG)                                                 \
    _Pragma("unroll") for (int g = 0; g < RG; g++) c[g] =                 \
        __builtin_amdgcn_mfma_f32_4x4x1f32(A[h].v[g], b[U], c[g], 3, U, 0);
      FMB_ROT(0) FMB_ROT(1) FMB_ROT(2) FMB_ROT(3) FMB_ROT(4) FMB_ROT(5) FMB_ROT(6) FMB_ROT(7)
#undef FMB_ROT
    }
  }
};

template <int RG> struct Coax<float, RG> {
  f4 c[RG];
  V4 R, I;  // 16 columns of the real and the imaginary parts
  __device__ __forceinline__ float row(int i) const { return c[i >> 2][i & 3]; }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int aoff, int lane) {
    R = __builtin_bit_cast(V4,
                           __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, aoff * 4, 0));
    I = __builtin_bit_cast(
        V4, __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (aoff + 256) * 4, 0));
  }
  __device__ __forceinline__ void run(const float *X, __amdgpu_buffer_rsrc_t, int, int m, int p,
                                      int lane) {
    const unsigned flip = (lane & 16) ? 0u : 0x80000000u;  // i z = (-im, re)
#pragma unroll
    for (int g = 0; g < RG; g++) c[g] = f4{0, 0, 0, 0};
    auto four = [&](auto kk) {
      constexpr int K = decltype(kk)::value;
      float b[4], o[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int r = min(m + K + u, p - 1), ro = (((r * (r + 1)) >> 1) + m) * kL;
        b[u] = X[ro + lane];
        o[u] = __builtin_bit_cast(float,
                                  __builtin_bit_cast(unsigned, X[ro + (lane ^ 16)]) ^ flip);
      }
#define FMB_COAX(U)                                                                            \
  _Pragma("unroll") for (int g = 0; g < RG; g++) c[g] =                                        \
      __builtin_amdgcn_mfma_f32_4x4x1f32(R.v[g], b[U], c[g], 4, K + U, 0);                     \
  _Pragma("unroll") for (int g = 0; g < RG; g++) c[g] =                                        \
      __builtin_amdgcn_mfma_f32_4x4x1f32(I.v[g], o[U], c[g], 4, K + U, 0);
      FMB_COAX(0) FMB_COAX(1) FMB_COAX(2) FMB_COAX(3)
#undef FMB_COAX
    };
    four(std::integral_constant<int, 0>{});
    if constexpr (RG > 1) four(std::integral_constant<int, 4>{});
    if constexpr (RG > 2) four(std::integral_constant<int, 8>{});
    if constexpr (RG > 3) four(std::integral_constant<int, 12>{});
  }
};

template <int RG> struct Rot<double, RG> {
  double c[4 * RG];
  V2 A[2 * RG];  // pairs of columns
  __device__ __forceinline__ double row(int i) const { return c[i]; }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int aoff, int lane) {
    const int vo = (((lane >> 5) << 4) | (lane & 15)) * 16;
#pragma unroll
    for (int u = 0; u < 2 * RG; u++)
      A[u] = __builtin_bit_cast(
          V2, __builtin_amdgcn_raw_buffer_load_b128(r, vo, (aoff + 64 * u) * 8, 0));
  }
  __device__ __forceinline__ void run(const double *xb, int n) {
#pragma unroll
    for (int i = 0; i < 4 * RG; i++) c[i] = 0.0;
#pragma unroll
    for (int u = 0; u < 2 * RG; u++) {
      const int k = 2 * u;
      if (k == 4 * RG - 2 && k > n) break;
      const double b0 = xb[k * kL], b1 = xb[(k + 1 <= 4 * RG - 4 ? k + 1 : min(k + 1, n)) * kL];
      fma_rows<RG>(c, A[u].v[0], b0, A[u].v[1], b1);
    }
  }
};

template <int RG> struct Coax<double, RG> {
  static constexpr int NC = (RG + 1) / 2;  // chunks of 8 columns
  double c[4 * RG];
  V2 A[NC][8];
  __device__ __forceinline__ double row(int i) const { return c[i]; }
  __device__ __forceinline__ void chunk(int h, __amdgpu_buffer_rsrc_t r, int aoff, int lane) {
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (8 * h + u < 4 * RG)
        A[h][u] = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b128(
                                             r, (lane & 31) * 16, (aoff + 64 * (8 * h + u)) * 8, 0));
  }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int aoff, int lane) {
    chunk(0, r, aoff, lane);
  }
  __device__ __forceinline__ void run(const double *X, __amdgpu_buffer_rsrc_t rc, int aoff, int m,
                                      int p, int lane) {
#pragma unroll
    for (int i = 0; i < 4 * RG; i++) c[i] = 0.0;
#pragma unroll
    for (int h = 0; h < NC; h++) {
      if (h + 1 < NC) chunk(h + 1, rc, aoff, lane);
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int k = 8 * h + u, r = m + k;
        if (k >= 4 * RG || (k > 4 * RG - 4 && r >= p)) break;
        const int ro = (((r * (r + 1)) >> 1) + m) * kL;
        // lanes of im add Ci re, lanes of re add -Ci im: the table holds both signs
        fma_rows<RG>(c, A[h][u].v[0], X[ro + lane], A[h][u].v[1], X[ro + (lane ^ 16)]);
      }
    }
  }
};

template <typename T> struct Ctx {
  typedef T real;
  __amdgpu_buffer_rsrc_t rin, rph;
  T *X, *accr, *acci;
  int p, SA, par, lane;  // par: bytes of a phase row
};

// rows row_of of degree n: coefficients +-m of the sources, phases
template <typename T, int RG> struct Src {
  cplx<T> zp[RG], zm[RG];
  __device__ __forceinline__ void load(const Ctx<T> &x, const Vec &v, int n) {
    constexpr int CS = 2 * (int)sizeof(T);
#pragma unroll
    for (int j = 0; j < RG; j++) {
      const int mo = row_of<RG>(j, x.lane >> 4, n) * CS;
      ldz(zp[j], x.rin, v.soff + mo, (n * n + n) * CS);
      ldz(zm[j], x.rin, v.soff + n * CS - mo, n * n * CS);
    }
  }
};
template <typename T, int RG> struct Pha {
  cplx<T> w[RG];
  __device__ __forceinline__ void load(const Ctx<T> &x, const Vec &v, int n) {
#pragma unroll
    for (int j = 0; j < RG; j++)
      ldz(w[j], x.rph, v.phr + row_of<RG>(j, x.lane >> 4, n) * 2 * (int)sizeof(T),
          (n & 1) * x.par);
  }
};

// One unit of the phase between two batches: the back rotation of the current batch (vc) and the
// first rotation of the next one (vn), both of degree n.  FIRST: the wave's first unit, with the
// barrier that ends the coaxial stage behind its loads.  FP32 also loads the next batch's sources
// and operators there (order 14, one right-hand side: 0.66 -> 0.64 ms); in FP64 their registers
// would spill at 16 waves, and 16 waves with exposed loads beat 8 with prefetched ones (0.88 against
// 1.17 ms).
template <typename T, int RG, bool FIRST>
__device__ __forceinline__ void rot_unit(const Ctx<T> &x, bool cur, bool nxt, const Vec &vc,
                                         const Vec &vn, int most, __amdgpu_buffer_rsrc_t rhc,
                                         __amdgpu_buffer_rsrc_t rhn, int aoff, int n) {
  if constexpr (sizeof(T) == 4) {
    Src<T, RG> z;
    Rot<T, RG> B, N;
    Pha<T, RG> f, g;
    if (cur) {
      B.load(rhc, aoff, x.lane);
      f.load(x, vc, n);
    }
    if (nxt) {
      z.load(x, vn, n);
      N.load(rhn, aoff, x.lane);
      g.load(x, vn, n);
    }
    if constexpr (FIRST) __syncthreads();
    if (cur) back_rot<RG>(x, vc, most, f, B, n);
    if (nxt) first_rot<RG>(x, z, g, N, n);
  } else {
    if (cur) {
      Rot<T, RG> B;
      Pha<T, RG> f;
      B.load(rhc, aoff, x.lane);
      f.load(x, vc, n);
      if constexpr (FIRST) __syncthreads();
      back_rot<RG>(x, vc, most, f, B, n);
    }
    if (nxt) {
      Src<T, RG> z;
      Rot<T, RG> B;
      Pha<T, RG> f;
      z.load(x, vn, n);
      f.load(x, vn, n);
      B.load(rhn, aoff, x.lane);
      first_rot<RG>(x, z, f, B, n);
    }
  }
}

// coaxial block |m| in place: its rows belong to one wave
template <typename T, int RG, bool FIRST>
__device__ __forceinline__ void coax_unit(const Ctx<T> &x, __amdgpu_buffer_rsrc_t rc, int aoff,
                                          int m) {
  Coax<T, RG> B;
  B.load(rc, aoff, x.lane);
  if constexpr (FIRST) __syncthreads();
  B.run(x.X, rc, aoff, m, x.p, x.lane);
  coax_put<RG>(x, B, m);
}

// unit<RG> for a wave-uniform rg in [1, 4]
template <typename T, bool FIRST, typename... Args>
__device__ __forceinline__ void rot_any(int rg, const Args &...args) {
  if (rg == 4)
    rot_unit<T, 4, FIRST>(args...);
  else if (rg == 3)
    rot_unit<T, 3, FIRST>(args...);
  else if (rg == 2)
    rot_unit<T, 2, FIRST>(args...);
  else
    rot_unit<T, 1, FIRST>(args...);
}
template <typename T, bool FIRST, typename... Args>
__device__ __forceinline__ void coax_any(int rg, const Args &...args) {
  if (rg == 4)
    coax_unit<T, 4, FIRST>(args...);
  else if (rg == 3)
    coax_unit<T, 3, FIRST>(args...);
  else if (rg == 2)
    coax_unit<T, 2, FIRST>(args...);
  else
    coax_unit<T, 1, FIRST>(args...);
}

struct TsArgs {
  const int2 *pairs;    // by (group, class): {source box, target's place in the group | offset << 8}
  const int *seg;       // [group][class] first pair, and the end
  int ngroups, J, nrb;  // target groups, workgroups of a group, right-hand-side blocks
  int tgrp, nbox;       // boxes of a group, of the level
  int R, SA;            // right-hand sides of a block; row stride of the sums
  int p, nrhs;
  const void *phase;    // [offset][parity of n][pstride]
  int pstride;
  const void *H;        // per class
  int hstride;          // values
  const void *C;        // per distance
  int cstride;          // values
  int cdist[kNC];       // distance of a class
  const int *sched;
  const void *in;
  void *out;
};

// Levels of one launch: level i takes workgroups end[i - 1] .. end[i] - 1.
struct TsLevels {
  int n;
  unsigned end[FMBH_TS_LEVELS];
  TsArgs a[FMBH_TS_LEVELS];
};

// The arguments of a workgroup's level and its place among the level's workgroups.  (One level has
// its arguments to itself: choosing among levels costs the kernel 1%.)
__device__ __forceinline__ const TsArgs &level_of(const TsArgs &a, unsigned &) { return a; }
__device__ __forceinline__ const TsArgs &level_of(const TsLevels &lv, unsigned &block) {
  int i = 0;
  while (i + 1 < lv.n && block >= lv.end[i]) i++;
  if (i) block -= lv.end[i - 1];
  return lv.a[i];
}

// LDS: the batch rows, then the sums' real and imaginary planes [coefficient][slot].  Slot: place
// of the target in the group x R + right-hand side.
template <typename T, int W, typename A>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4)))
    k_m2l_ts(A args) {
  unsigned block = blockIdx.x;
  const TsArgs &a = level_of(args, block);
  constexpr int TS = (int)sizeof(T), CS = 2 * TS;
  extern __shared__ __align__(16) unsigned char smem[];
  const int p = a.p, p2 = p * p, SA = a.SA;
  T *X = (T *)smem;
  T *accr = X + (size_t)((p * (p + 1)) >> 1) * kL, *acci = accr + (size_t)p2 * SA;
  const int tid = threadIdx.x, wave = uni(tid >> 6), lane = tid & 63, li = lane & 15;
  // workgroups are dealt to the 8 XCDs in turn; XCD x takes a contiguous range of the groups, so
  // that those whose sources overlap share its L2.  The blocks of right-hand sides of a group lie
  // beside each other (FP64, 64 right-hand sides: 2% faster than one after the other) unless the
  // last is short: an XCD deals its workgroups to four shader engines in turn, and the short ones
  // would meet the same engines every time (33 right-hand sides took as long as 64).
  int g, jj, rb;
  {
    const unsigned items = (unsigned)a.ngroups * a.J, per = (items + 7) / 8;
    const unsigned i = block >> 3;
    if (i >= per * a.nrb) return;
    const bool even = a.nrhs % a.R == 0;
    rb = even ? i % a.nrb : i / per;
    const unsigned q = (block & 7) * per + (even ? i / a.nrb : i % per);
    if (q >= items) return;
    jj = q % a.J;
    g = q / a.J;
  }
  const int r0 = rb * a.R, R = min(a.R, a.nrhs - r0);
  // lane c: batches before class c, first pair of class c
  int preV, sqV;
  {
    const int q0 = a.seg[g * kNC + min(lane, kNC)], q1 = a.seg[g * kNC + min(lane + 1, kNC)];
    const int n = lane < kNC ? ((q1 - q0) * R + kV - 1) / kV : 0;
    int s = n;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(s, o, 64);
      if (lane >= o) s += v;
    }
    preV = s - n;
    sqV = q0;
  }
  const int NB = __builtin_amdgcn_readlane(preV, kNC);
  const int b0 = (int)((long long)NB * jj / a.J), b1 = (int)((long long)NB * (jj + 1) / a.J);
  if (b0 >= b1) return;
  for (int i = tid; i < 2 * p2 * SA; i += 64 * W) accr[i] = T(0);
  // lane i: the wave's i-th rotation and coaxial unit {degree or |m|, table offset}
  const int e1 = uni(a.sched[2 * wave]), n1 = uni(a.sched[2 * wave + 1]) - e1;
  const int e2 = uni(a.sched[2 * (W + wave)]), n2 = uni(a.sched[2 * (W + wave) + 1]) - e2;
  const int2 none{0, 0};
  const int2 un1 = lane < n1 ? ((const int2 *)a.sched)[e1 + lane] : none;
  const int2 un2 = lane < n2 ? ((const int2 *)a.sched)[e2 + lane] : none;
  __syncthreads();
  Ctx<T> x;
  x.rin = rsrc(a.in);
  x.rph = rsrc(a.phase);
  x.X = X;
  x.accr = accr;
  x.acci = acci;
  x.p = p;
  x.SA = SA;
  x.par = a.pstride * CS;
  x.lane = lane;
  int c = 0, most = 0, mostn = 0;
  int2 pr{0, 0};
  int fr = 0, fl = 0;
  // batch b: its class, and lane li's pair (loaded ahead of its use; absent vectors repeat the
  // batch's first) ...
  auto fetch = [&](int b) {
    while (__builtin_amdgcn_readlane(preV, c + 1) <= b) c++;
    const int q0 = __builtin_amdgcn_readlane(sqV, c);
    const int u0 = (b - __builtin_amdgcn_readlane(preV, c)) * kV;
    const int nv = min(kV, (__builtin_amdgcn_readlane(sqV, c + 1) - q0) * R - u0);
    fl = li < nv;
    const int u = u0 + (fl ? li : 0), qq = R == 1 ? u : u / R;
    fr = u - qq * R;
    pr = a.pairs[q0 + qq];
  };
  // ... and its vector
  auto vec = [&]() {
    Vec v;
    v.soff = (int)((unsigned)(pr.x * a.nrhs + r0 + fr) * (unsigned)(p2 * CS));
    v.phr = (pr.y >> 8) * 2 * x.par;
    v.slot = fl ? (pr.y & 255) * a.R + fr : -1;
    v.rank = 0;
    mostn = 0;
    if constexpr (TS == 4) {
      if (R < kV) {  // else the batch holds one pair, whose slots differ
#define FMB_ROR(S)                                                                    \
  {                                                                                   \
    const int o = __builtin_amdgcn_update_dpp(0, v.slot, 0x120 + S, 0xf, 0xf, false); \
    v.rank += (li >= S && o == v.slot) ? 1 : 0;                                       \
  }
        FMB_ROR(1) FMB_ROR(2) FMB_ROR(3) FMB_ROR(4) FMB_ROR(5) FMB_ROR(6) FMB_ROR(7) FMB_ROR(8)
        FMB_ROR(9) FMB_ROR(10) FMB_ROR(11) FMB_ROR(12) FMB_ROR(13) FMB_ROR(14) FMB_ROR(15)
#undef FMB_ROR
        while (__ballot(v.slot >= 0 && v.rank > mostn)) mostn++;
      }
      if (v.slot < 0) v.rank = -1;
    }
    return v;
  };
  auto hrsrc = [&](int cl) { return rsrc((const T *)a.H + (size_t)a.hstride * cl); };
  auto unit = [](int2 u, int i) {
    return int2{__builtin_amdgcn_readlane(u.x, i), __builtin_amdgcn_readlane(u.y, i)};
  };
  fetch(b0);
  Vec vn = vec(), vc = vn;
  __amdgpu_buffer_rsrc_t rhn = hrsrc(c), rhc = rhn;
  for (int i = 0; i < n1; i++) {
    const int2 u = unit(un1, i);
    rot_any<T, false>((u.x + 4) >> 2, x, false, true, vc, vn, 0, rhc, rhn, u.y, u.x);
  }
  for (int b = b0; b < b1; b++) {
    const __amdgpu_buffer_rsrc_t rc = rsrc((const T *)a.C + (size_t)a.cstride * a.cdist[c]);
    vc = vn;
    rhc = rhn;
    most = mostn;
    const bool nxt = b + 1 < b1;
    if (nxt) fetch(b + 1);
    if (n2) {
      int2 u = unit(un2, 0);
      coax_any<T, true>((p - u.x + 3) >> 2, x, rc, u.y, u.x);
      for (int i = 1; i < n2; i++) {
        u = unit(un2, i);
        coax_any<T, false>((p - u.x + 3) >> 2, x, rc, u.y, u.x);
      }
    } else {
      __syncthreads();
    }
    if (nxt) {
      vn = vec();
      rhn = hrsrc(c);
    }
    if (n1) {
      int2 u = unit(un1, 0);
      rot_any<T, true>((u.x + 4) >> 2, x, true, nxt, vc, vn, most, rhc, rhn, u.y, u.x);
      for (int i = 1; i < n1; i++) {
        u = unit(un1, i);
        rot_any<T, false>((u.x + 4) >> 2, x, true, nxt, vc, vn, most, rhc, rhn, u.y, u.x);
      }
    } else {
      __syncthreads();
    }
  }
  __syncthreads();
  // the group's sums into the level's coefficients (L2L and the group's other workgroups add there
  // too)
  const int t0 = g * a.tgrp, ns = min(a.tgrp, a.nbox - t0);
  for (int s = wave; s < ns * R; s += W) {
    const int tb = s / R, r = s - tb * R, sl = tb * a.R + r;
    T *dst = (T *)a.out + ((size_t)(t0 + tb) * a.nrhs + r0 + r) * 2 * p2;
    for (int e = lane; e < 2 * p2; e += 64)
      unsafeAtomicAdd(dst + e, (e & 1 ? acci : accr)[(e >> 1) * SA + sl]);
  }
}

// the offset bucket of pair q of the tree's offset-major list
__device__ __forceinline__ int offset_of(const int *__restrict__ start, int q) {
  int lo = 0, hi = FMB_NOFF;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= q)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// (group, class) of each pair, and its index
__global__ void k_ts_keys(const int *__restrict__ tgt, int np, int tgrp,
                          const int *__restrict__ start, const int *__restrict__ cls,
                          unsigned *__restrict__ key, int *__restrict__ idx) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  key[q] = (unsigned)(tgt[q] / tgrp) * kNC + cls[offset_of(start, q)];
  idx[q] = q;
}

// the sorted pairs and the first pair of every (group, class)
__global__ void k_ts_pairs(const unsigned *__restrict__ key, const int *__restrict__ idx, int np,
                           const int *__restrict__ tgt, const int *__restrict__ src,
                           const int *__restrict__ start, int tgrp, int nseg,
                           int2 *__restrict__ pairs, int *__restrict__ seg) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const int q = idx[i];
  pairs[i] = make_int2(src[q], (tgt[q] % tgrp) | offset_of(start, q) << 8);
  const int k = (int)key[i], k0 = i ? (int)key[i - 1] + 1 : 0;
  for (int s = k0; s <= k; s++) seg[s] = i;
  if (i == np - 1)
    for (int s = k + 1; s <= nseg; s++) seg[s] = np;
}

// Rotation tables of the classes, halved.  Even element (m', m) of degree n: H^{m'm} + H^{m',-m}
// (H^{m'0} for m = 0); odd: their difference, with a zero row and column 0.  With rg = the row
// groups (4 rows) of the block:
//   FP32: [n][8 columns][lane][4 row groups]: lane 4 k + i holds row i of the groups and column k
//         of the even block, lane 32 + 4 k + i of the odd block;
//   FP64: [n][2 columns][lane][column], 4 rg columns: lanes 0..15 the rows of the even block,
//         16..31 of the odd block.
template <typename T>
__global__ void k_ts_rot(const double *__restrict__ H, size_t hs, const int *__restrict__ cbeta,
                         const int *__restrict__ hoff, int hstride, T *__restrict__ out) {
  const int n = blockIdx.x, c = blockIdx.y, s = 2 * n + 1, rg = (n + 4) >> 2;
  const double *src = H + hs * cbeta[c] + rot_off(n);
  auto h = [&](int mp, int m) { return src[(size_t)(m + n) * s + (mp + n)]; };
  T *dst = out + (size_t)hstride * c + hoff[n];
  const int tot = sizeof(T) == 4 ? ((rg + 1) >> 1) * 256 : 2 * rg * 64;
  for (int x = threadIdx.x; x < tot; x += blockDim.x) {
    int mp, m, odd;
    if (sizeof(T) == 4) {
      const int lane = (x >> 2) & 63;
      mp = 4 * (x & 3) + (lane & 3);
      m = 8 * (x >> 8) + ((lane >> 2) & 7);
      odd = lane >> 5;
    } else {
      const int lane = (x >> 1) & 31;
      mp = lane & 15;
      m = 2 * (x >> 6) + (x & 1);
      odd = lane >> 4;
    }
    double v = 0.0;
    if (mp <= n && m <= n) {
      if (!odd)
        v = m ? h(mp, m) + h(mp, -m) : h(mp, 0);
      else if (mp && m)
        v = h(mp, m) - h(mp, -m);
    }
    dst[x] = (T)(0.5 * v);
  }
}

// Coaxial tables of the distances, doubled (which undoes the halves of the two rotations).
//   FP32: [m][re, im][lane][4 row groups]: lane 4 k + i holds row i of the groups, column k < 16;
//   FP64: [m][column][lane][2], 4 rg columns: lanes 0..15 the rows' {re, -im}, 16..31 {re, im}.
template <typename T>
__global__ void k_ts_coax(const cplx<T> *__restrict__ C, size_t cs, int p,
                          const int *__restrict__ coff, int cstride, T *__restrict__ out) {
  const int am = blockIdx.x, d = blockIdx.y, s = p - am;
  const cplx<T> *src = C + cs * d + coax_blk(p, am);
  T *dst = out + (size_t)cstride * d + coff[am];
  const int tot = sizeof(T) == 4 ? 512 : ((s + 3) & ~3) * 64;
  for (int x = threadIdx.x; x < tot; x += blockDim.x) {
    int i, k;
    bool im, neg = false;
    if (sizeof(T) == 4) {
      const int lane = (x >> 2) & 63;
      im = x >> 8;
      i = 4 * (x & 3) + (lane & 3);
      k = lane >> 2;
    } else {
      const int lane = (x >> 1) & 31;
      im = x & 1;
      neg = im && lane < 16;
      i = lane & 15;
      k = x >> 6;
    }
    T v = T(0);
    if (i < s && k < s) {
      const cplx<T> z = src[k * s + i];
      v = 2 * (im ? (neg ? -z.im : z.im) : z.re);
    }
    dst[x] = v;
  }
}

template <typename T, int W> int launch_ts(const fmbh_ts_job *jobs, int n, int nrhs, hipStream_t st) {
  TsLevels lv;
  lv.n = n;
  double per[FMBH_TS_LEVELS];
  long long wg[FMBH_TS_LEVELS], most[FMBH_TS_LEVELS], total = 0;
  size_t lds = 0;
  for (int i = 0; i < n; i++) {
    const fmbh_ts_job *j = jobs + i;
    TsArgs &a = lv.a[i];
    a.pairs = (const int2 *)j->pairs;
    a.seg = j->seg;
    a.ngroups = j->ngroups;
    a.tgrp = j->tgrp;
    a.nbox = j->nbox;
    a.SA = j->slots | 1;  // odd: neighbouring coefficients fall into different LDS banks
    // right-hand sides of a block: what the slots hold, in even blocks, which from 16 on are
    // multiples of a batch
    a.R = j->slots / j->tgrp;
    a.nrb = (nrhs + a.R - 1) / a.R;
    int even = (nrhs + a.nrb - 1) / a.nrb;
    if (even >= kV) even = (even + kV - 1) / kV * kV;
    if (even < a.R) a.R = even;
    a.nrb = (nrhs + a.R - 1) / a.R;
    a.p = j->p;
    a.nrhs = nrhs;
    a.phase = j->phase;
    a.pstride = j->pstride;
    a.H = j->H;
    a.hstride = j->hstride;
    a.C = j->C;
    a.cstride = j->cstride;
    for (int c = 0; c < kNC; c++) a.cdist[c] = j->cdist[c];
    a.sched = j->sched;
    a.in = j->in;
    a.out = j->out;
    wg[i] = (long long)a.ngroups * a.nrb;
    // batches of a group: its classes leave half a batch each
    per[i] = (double)j->npairs * nrhs / kV / wg[i] + (a.R < kV ? 0.5 * kNC : 0.0);
    most[i] = (long long)j->npairs * nrhs / kV / wg[i];
    if (most[i] > 8192 / wg[i] + 1) most[i] = 8192 / wg[i] + 1;
    if (most[i] < 1) most[i] = 1;
    const size_t b = fmbh_ts_lds_bytes(j->p, sizeof(T) == 8 ? FMB_FP64 : FMB_MIXED, j->slots);
    lds = b > lds ? b : lds;
  }
  if (lds > 160 * 1024)
    return fmb_set_error(FMB_ERR_RANGE, "M2L sums need %zu B of LDS", lds);
  // Workgroups of a group (J): setting up and flushing costs one about two batches, and the last
  // round of workgroups may be nearly empty, so the batches of a workgroup, the same at each level,
  // have the least (rounds) x (2 + batches), and the most workgroups within 2% of it (an even
  // finish).  The search takes two passes over J, at most the finest level's batches of a group:
  // 32 vectors of 189 sources, 378.  Against about 2,048 workgroups for every launch (FP64): level 4
  // of the 5,120-triangle sphere 131 -> 90 us (560 -> 248 workgroups), levels 6 and 5 of 20,480 with
  // the levels beside them 1.85 -> 1.73 ms a product.
  const int cu = 160 * 1024 / (int)lds, fit = cu < 1 ? 1 : (cu < 16 / W ? cu : 16 / W);
  auto split = [&](int i, double b) {
    const long long J = (long long)(per[i] / b + 0.999);
    return J < 1 ? 1 : (J > most[i] ? most[i] : J);
  };
  auto cost = [&](double b) {
    long long x = 0;
    double longest = 0.0;
    for (int i = 0; i < n; i++) {
      const long long J = split(i, b);
      x += (lv.a[i].ngroups * J + 7) / 8 * lv.a[i].nrb;
      longest = per[i] / J > longest ? per[i] / J : longest;
    }
    return ((x + 32 * fit - 1) / (32 * fit)) * (2.0 + longest);
  };
  double least = 1e300, batches = per[0];
  for (long long J = 1; J <= most[0]; J++) {
    const double c = cost(per[0] / J);
    least = c < least ? c : least;
  }
  for (long long J = most[0]; J >= 1; J--)
    if (cost(per[0] / J) <= 1.02 * least) {
      batches = per[0] / J;
      break;
    }
  for (int i = 0; i < n; i++) {
    lv.a[i].J = (int)split(i, batches);
    total += 8 * (((long long)lv.a[i].ngroups * lv.a[i].J + 7) / 8) * lv.a[i].nrb;
    if (total > 0x7fffffffLL) return fmb_set_error(FMB_ERR_RANGE, "M2L grid too large");
    lv.end[i] = (unsigned)total;
  }
  auto one = k_m2l_ts<T, W, TsArgs>;
  auto more = k_m2l_ts<T, W, TsLevels>;
  FMB_HIP_CHECK(hipFuncSetAttribute(n == 1 ? (const void *)one : (const void *)more,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  if (n == 1)
    hipLaunchKernelGGL(one, dim3((unsigned)total), dim3(64 * W), lds, st, lv.a[0]);
  else
    hipLaunchKernelGGL(more, dim3((unsigned)total), dim3(64 * W), lds, st, lv);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

}  // namespace

extern "C" size_t fmbh_ts_lds_bytes(int p, int prec, int slots) {
  const size_t tsz = prec == FMB_FP64 ? 8 : 4, p2 = (size_t)p * p;
  return (p2 + p) / 2 * kL * tsz + 2 * p2 * (slots | 1) * tsz;
}

extern "C" int fmbh_ts_run(const fmbh_ts_job *jobs, int n, int prec, int nrhs, void *stream) {
  fmbh_ts_job j[FMBH_TS_LEVELS];
  int m = 0;
  if (n < 0 || n > FMBH_TS_LEVELS)
    return fmb_set_error(FMB_ERR_RANGE, "target-stationary M2L of %d levels", n);
  for (int i = 0; i < n; i++) {
    if (!jobs[i].npairs) continue;
    if (jobs[i].p > FMBH_TS_PMAX || jobs[i].tgrp < 1 || jobs[i].tgrp > jobs[i].slots ||
        jobs[i].slots > 255)
      return fmb_set_error(FMB_ERR_RANGE, "no target-stationary M2L for order %d", jobs[i].p);
    j[m++] = jobs[i];
  }
  if (!m) return FMB_OK;
  if (prec == FMB_FP64) return launch_ts<double, FMBH_TS_WAVES64>(j, m, nrhs, (hipStream_t)stream);
  return launch_ts<float, FMBH_TS_WAVES32>(j, m, nrhs, (hipStream_t)stream);
}

extern "C" int fmbh_ts_lists(const fmb_tree *t, int l, int tgrp, const int *h_cls, void **d_pairs,
                             int **d_seg, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  const int np = t->npairs[l], ng = (t->nbox[l] + tgrp - 1) / tgrp, nseg = ng * kNC;
  int rc, *d_start = nullptr, *d_cls = nullptr, *idx = nullptr, *idx2 = nullptr;
  unsigned *key = nullptr, *key2 = nullptr;
  void *tmp = nullptr;
  size_t tb = 0;
  *d_pairs = nullptr;
  *d_seg = nullptr;
  if ((rc = fmbh_malloc(d_pairs, sizeof(int2) * (size_t)np))) return rc;
  if ((rc = fmbh_malloc((void **)d_seg, sizeof(int) * (size_t)(nseg + 1)))) return rc;
  if (!np) return fmbh_memset(*d_seg, 0, sizeof(int) * (size_t)(nseg + 1), stream);
  rc = fmbh_malloc((void **)&d_start, sizeof(int) * (FMB_NOFF + 1));
  if (!rc) rc = fmbh_malloc((void **)&d_cls, sizeof(int) * FMB_NOFF);
  if (!rc) rc = fmbh_malloc((void **)&key, sizeof(unsigned) * (size_t)np);
  if (!rc) rc = fmbh_malloc((void **)&key2, sizeof(unsigned) * (size_t)np);
  if (!rc) rc = fmbh_malloc((void **)&idx, sizeof(int) * (size_t)np);
  if (!rc) rc = fmbh_malloc((void **)&idx2, sizeof(int) * (size_t)np);
  if (!rc) rc = fmbh_h2d(d_start, t->h_off_start[l], sizeof(int) * (FMB_NOFF + 1), stream);
  if (!rc) rc = fmbh_h2d(d_cls, h_cls, sizeof(int) * FMB_NOFF, stream);
  if (!rc) {
    int bits = 1;
    while (bits < 32 && ((unsigned)nseg >> bits)) bits++;
    auto ok = [&](hipError_t e) {
      if (e != hipSuccess && !rc)
        rc = fmb_set_error(FMB_ERR_HIP, "M2L lists: %s", hipGetErrorString(e));
      return e == hipSuccess;
    };
    const dim3 gr((np + 255) / 256);
    hipLaunchKernelGGL(k_ts_keys, gr, dim3(256), 0, st, t->d_pair_tgt[l], np, tgrp, d_start, d_cls,
                       key, idx);
    ok(hipGetLastError());
    ok(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, key, key2, idx, idx2, np, 0, bits, st));
    if (!rc) rc = fmbh_malloc(&tmp, tb);
    if (!rc)
      ok(hipcub::DeviceRadixSort::SortPairs(tmp, tb, key, key2, idx, idx2, np, 0, bits, st));
    if (!rc) {
      hipLaunchKernelGGL(k_ts_pairs, gr, dim3(256), 0, st, key2, idx2, np, t->d_pair_tgt[l],
                         t->d_pair_src[l], d_start, tgrp, nseg, (int2 *)*d_pairs, *d_seg);
      ok(hipGetLastError());
    }
    const int rs = fmbh_sync(stream);
    if (!rc) rc = rs;
  }
  fmbh_free(tmp);
  fmbh_free(d_start);
  fmbh_free(d_cls);
  fmbh_free(key);
  fmbh_free(key2);
  fmbh_free(idx);
  fmbh_free(idx2);
  return rc;
}

extern "C" int fmbh_ts_rot(int prec, const double *d_H64, int Pmax, int P, const int *d_cbeta,
                           const int *d_hoff, int hstride, void *out, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  const dim3 gr(P, kNC);
  if (prec == FMB_FP64)
    hipLaunchKernelGGL(k_ts_rot<double>, gr, dim3(256), 0, st, d_H64, (size_t)rot_off(Pmax),
                       d_cbeta, d_hoff, hstride, (double *)out);
  else
    hipLaunchKernelGGL(k_ts_rot<float>, gr, dim3(256), 0, st, d_H64, (size_t)rot_off(Pmax),
                       d_cbeta, d_hoff, hstride, (float *)out);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}

extern "C" int fmbh_ts_coax(int prec, const void *d_C, int p, const int *d_coff, int cstride,
                            void *out, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  const dim3 gr(p, FMB_NDIST);
  if (prec == FMB_FP64)
    hipLaunchKernelGGL(k_ts_coax<double>, gr, dim3(256), 0, st, (const cplx<double> *)d_C,
                       (size_t)coax_size(p), p, d_coff, cstride, (double *)out);
  else
    hipLaunchKernelGGL(k_ts_coax<float>, gr, dim3(256), 0, st, (const cplx<float> *)d_C,
                       (size_t)coax_size(p), p, d_coff, cstride, (float *)out);
  FMB_LAUNCH_CHECK();
  return FMB_OK;
}
