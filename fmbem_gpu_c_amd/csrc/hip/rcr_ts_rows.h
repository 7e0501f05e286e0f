// rcr_ts_rows.h -- the batch rows of the target-stationary M2L (rcr_ts.hip) and the targets' sums
// in LDS: what the lanes of a wavefront write there for each other.  The accesses are written over
// a context with the arrays X (rows), accr and acci (sums), so that tests/ts_rows_check.cpp can run
// them on the CPU lane by lane, with every access checked.
#ifndef FMB_TS_ROWS_H
#define FMB_TS_ROWS_H

#ifdef __HIPCC__
#define FMB_TS_FN __device__ __forceinline__
#else
#define FMB_TS_FN inline
#endif

namespace fmb_ts {

constexpr int kV = 16;  // vectors of a batch
constexpr int kL = 64;  // reals of a batch row

// what a wave needs of the batch: lanes li, li + 16, .. stand for vector li
struct Vec {
  int soff, phr, slot;  // byte offsets of its source and phase row; its target's slot, or -1
  int rank;             // FP32: its place among the batch's vectors of that slot, or -1
};

#ifdef __HIPCC__
// What the lanes of this wave wrote to LDS before is seen by all of them after, and nothing that
// they read before changes: the hardware keeps a wave's LDS accesses in order, so this is for the
// compiler, which may reorder or fold what it sees as the accesses of one lane.  No instruction.
FMB_TS_FN void order_lanes() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
FMB_TS_FN void add_sum(double *p, double v) { unsafeAtomicAdd(p, v); }
#else
void order_lanes();
#endif

// row m = 4 j + lane / 16 of degree n, clamped to n
template <int RG> FMB_TS_FN int row_of(int j, int lk, int n) {
  return j < RG - 1 ? 4 * j + lk : (4 * j + lk < n ? 4 * j + lk : n);
}

// sources to e and o with their phases, then the first rotation: rows of degree n
template <int RG, typename C, typename Z, typename F, typename B>
FMB_TS_FN void first_rot(const C &x, const Z &z, const F &f, B &rot, int n) {
  typedef typename C::real T;
  auto xn = x.X + ((n * (n + 1)) >> 1) * kL;
  const int li = x.lane & 15, lk = x.lane >> 4;
#pragma unroll
  for (int j = 0; j < RG; j++) {
    const T sr = z.zp[j].re + z.zm[j].re, dr = z.zp[j].re - z.zm[j].re;
    const T si = z.zp[j].im + z.zm[j].im, di = z.zp[j].im - z.zm[j].im;
    const auto w = f.w[j];
    auto y = xn + (row_of<RG>(j, lk, n) * kL + li);
    y[0] = sr * w.re - di * w.im;
    y[16] = si * w.re + dr * w.im;
    y[32] = dr * w.re - si * w.im;
    y[48] = di * w.re + sr * w.im;
  }
  order_lanes();
  rot.run(xn + x.lane, n);
#pragma unroll
  for (int i = 0; i < 4 * RG; i++)
    if (i <= 4 * RG - 4 || i <= n) xn[i * kL + x.lane] = rot.row(i);
}

// rows of coaxial block |m|, which a lane's product has read for itself and for the lane of the
// other part (re, im)
template <int RG, typename C, typename B> FMB_TS_FN void coax_put(const C &x, const B &cx, int m) {
  order_lanes();
#pragma unroll
  for (int i = 0; i < 4 * RG; i++)
    if (i <= 4 * RG - 4 || m + i < x.p) {
      const int r = m + i;
      x.X[(((r * (r + 1)) >> 1) + m) * kL + x.lane] = cx.row(i);
    }
}

// back rotation of degree n, output phases, sums into the targets' slots; most: the largest rank
// of the batch (FP32)
template <int RG, typename C, typename F, typename B>
FMB_TS_FN void back_rot(const C &x, const Vec &v, int most, const F &f, B &rot, int n) {
  typedef typename C::real T;
  auto xn = x.X + ((n * (n + 1)) >> 1) * kL;
  const int li = x.lane & 15, lk = x.lane >> 4;
  rot.run(xn + x.lane, n);
#pragma unroll
  for (int i = 0; i < 4 * RG; i++)
    if (i <= 4 * RG - 4 || i <= n) xn[i * kL + x.lane] = rot.row(i);
  order_lanes();
  T y0[RG], y1[RG], y2[RG], y3[RG];
#pragma unroll
  for (int j = 0; j < RG; j++) {
    const auto y = xn + (row_of<RG>(j, lk, n) * kL + li);
    const T er = y[0], ei = y[16], orr = y[32], oi = y[48];
    const T pr = er + orr, pi = ei + oi, qr = er - orr, qi = ei - oi;
    const auto w = f.w[j];
    y0[j] = pr * w.re + pi * w.im;
    y1[j] = pi * w.re - pr * w.im;
    y2[j] = qr * w.re - qi * w.im;
    y3[j] = qi * w.re + qr * w.im;
  }
  const int c0 = n * n + n;
  const int fp0 = (c0 + lk) * x.SA + v.slot, fm0 = (c0 - lk) * x.SA + v.slot;
  const bool tail = 4 * RG - 4 + lk <= n;  // the last rows may lie past the block
  if constexpr (sizeof(T) == 8) {
    if (v.slot >= 0) {
#pragma unroll
      for (int j = 0; j < RG; j++) {
        if (j == RG - 1 && !tail) break;
        add_sum(x.accr + (fp0 + 4 * j * x.SA), y0[j]);
        add_sum(x.acci + (fp0 + 4 * j * x.SA), y1[j]);
        if (j > 0 || lk) {
          add_sum(x.accr + (fm0 - 4 * j * x.SA), y2[j]);
          add_sum(x.acci + (fm0 - 4 * j * x.SA), y3[j]);
        }
      }
    }
    order_lanes();  // (the next batch writes these rows)
  } else {
    for (int q = 0; q <= most; q++) {
      if (v.rank == q) {
        T s0[RG], s1[RG], s2[RG], s3[RG];
#pragma unroll
        for (int j = 0; j < RG; j++) {
          if (j == RG - 1 && !tail) break;  // (rows past the block lie outside the sums)
          const int d = 4 * j * x.SA;
          s0[j] = x.accr[fp0 + d];
          s1[j] = x.acci[fp0 + d];
          s2[j] = x.accr[fm0 - d];
          s3[j] = x.acci[fm0 - d];
        }
#pragma unroll
        for (int j = 0; j < RG; j++) {
          if (j == RG - 1 && !tail) break;
          const int d = 4 * j * x.SA;
          x.accr[fm0 - d] = s2[j] + y2[j];
          x.acci[fm0 - d] = s3[j] + y3[j];
          x.accr[fp0 + d] = s0[j] + y0[j];  // (m = 0: the same element, written last)
          x.acci[fp0 + d] = s1[j] + y1[j];
        }
      }
      order_lanes();  // (the next rank adds to the same sums, the next batch writes these rows)
    }
  }
}

}  // namespace fmb_ts

#endif
