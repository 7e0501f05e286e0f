// Runs the batch rows and target sums of the target-stationary M2L (csrc/hip/rcr_ts_rows.h) on the
// CPU: the 64 lanes of one wavefront as fibres that run one after another up to the next point that
// orders them, two batches of every order, with each access checked:
//   range  inside its array (rows, real sums, imaginary sums);
//   order  no element that one lane writes is touched by another lane before such a point (but
//          for the same value written again).
// The sums are compared with the same translation by plain loops.  Argument "range": only the
// ranges; "order": everything.
#include <ucontext.h>

#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "rcr_ts_rows.h"

namespace fmb_ts {

int g_lane, g_faults;
long g_epoch;
bool g_order;
char g_case[128];

void fault(const char *what, const char *array, long i) {
  if (g_faults++ < 8) printf("%s: %s, %s[%ld], lane %d\n", g_case, what, array, i, g_lane);
}

template <typename T> struct Mem {
  struct Use {
    long epoch = -1;
    int lane = 0;  // -1: several
    void add() {
      lane = epoch == g_epoch && lane != g_lane ? -1 : g_lane;
      epoch = g_epoch;
    }
    bool other() const { return epoch == g_epoch && lane != g_lane; }
  };
  const char *name;
  std::vector<T> v;
  std::vector<Use> rd, wr, at;
  Mem(const char *n, size_t size) : name(n), v(size), rd(size), wr(size), at(size) {}
  bool ok(long i) const {
    if (i >= 0 && i < (long)v.size()) return true;
    fault("out of range", name, i);
    return false;
  }
  void conflict(bool c, long i) const {
    if (c && g_order) fault("unordered lanes", name, i);
  }
  T get(long i) {
    if (!ok(i)) return T(0);
    conflict(wr[i].other() || at[i].other(), i);
    rd[i].add();
    return v[i];
  }
  void put(long i, T x) {
    if (!ok(i)) return;
    // (lanes past a block's last row repeat it: the same value)
    conflict((wr[i].other() && memcmp(&v[i], &x, sizeof(T))) || at[i].other() || rd[i].other(), i);
    wr[i].add();
    v[i] = x;
  }
  void atomic(long i, T x) {
    if (!ok(i)) return;
    conflict(wr[i].other() || rd[i].other(), i);
    at[i].add();
    v[i] += x;
  }
};

template <typename T> struct Ref {
  Mem<T> *m;
  long i;
  operator T() const { return m->get(i); }
  void operator=(T x) const { m->put(i, x); }
};
template <typename T> struct Ptr {
  Mem<T> *m;
  long i;
  Ptr operator+(long d) const { return Ptr{m, i + d}; }
  Ref<T> operator[](long d) const { return Ref<T>{m, i + d}; }
};
template <typename T> void add_sum(Ptr<T> p, T x) { p.m->atomic(p.i, x); }

// lanes as fibres
ucontext_t g_main, g_fibre[64];
bool g_done[64];
void (*g_body)();
void fibre() {
  g_body();
  g_done[g_lane] = true;
}
void run_wave(void (*body)()) {
  static std::vector<char> stacks(64 * 65536);
  g_body = body;
  for (int l = 0; l < 64; l++) {
    getcontext(&g_fibre[l]);
    g_fibre[l].uc_stack.ss_sp = &stacks[l * 65536];
    g_fibre[l].uc_stack.ss_size = 65536;
    g_fibre[l].uc_link = &g_main;
    makecontext(&g_fibre[l], fibre, 0);
    g_done[l] = false;
  }
  for (int left = 64; left;) {
    int ended = 0;
    for (g_lane = 0; g_lane < 64; g_lane++) {
      swapcontext(&g_main, &g_fibre[g_lane]);
      ended += g_done[g_lane];
    }
    if (ended && ended != 64) {
      printf("%s: lanes pass different numbers of points\n", g_case);
      exit(1);
    }
    left -= ended;
    g_epoch++;
  }
}
void order_lanes() { swapcontext(&g_fibre[g_lane], &g_main); }

template <typename T> struct Ctx {
  typedef T real;
  Ptr<T> X, accr, acci;
  int p, SA, lane;
  void sync() const { order_lanes(); }
};

// operators: rotations by degree (even, odd: row and column 0 of odd are zero), coaxial by |m|
template <typename T> struct Ops {
  int p;
  std::vector<T> H[16][2][2];  // [degree][rotation][even, odd], (n + 1)^2
  std::vector<std::complex<T>> C[16];
};
template <typename T> struct Batch {
  std::complex<T> src[16][256];
  std::complex<T> w[16][2][16];  // [vector][in, out][m]
  int slot[16], rank[16], most;
};
struct C2f {
  float re, im;
};
struct C2d {
  double re, im;
};
template <typename T> struct C2;
template <> struct C2<float> : C2f {};
template <> struct C2<double> : C2d {};

template <typename T, int RG> struct ZS {
  C2<T> zp[RG], zm[RG];
};
template <typename T, int RG> struct FS {
  C2<T> w[RG];
};
template <typename T, int RG> struct RotS {
  T c[4 * RG];
  const std::vector<T> *A;
  T row(int i) const { return c[i]; }
  void run(Ptr<T> xb, int n) {
    for (int i = 0; i < 4 * RG; i++) c[i] = 0;
    for (int k = 0; k < 4 * RG; k++) {
      const T b = xb[(k < n ? k : n) * kL];
      for (int i = 0; i <= n && k <= n; i++) c[i] += (*A)[i * (n + 1) + k] * b;
    }
  }
};
template <typename T, int RG> struct CoaxS {
  T c[4 * RG];
  T row(int i) const { return c[i]; }
  void run(const Ctx<T> &x, const std::vector<std::complex<T>> &C, int m) {
    const int s = x.p - m;
    for (int i = 0; i < 4 * RG; i++) c[i] = 0;
    for (int k = 0; k < s; k++) {
      const int r = m + k, ro = (((r * (r + 1)) >> 1) + m) * kL;
      const T b = x.X[ro + x.lane], o = x.X[ro + (x.lane ^ 16)];
      for (int i = 0; i < s; i++)
        c[i] += C[k * s + i].real() * b + (x.lane & 16 ? o : -o) * C[k * s + i].imag();
    }
  }
};

template <typename T> struct Case {
  Mem<T> X, accr, acci;
  int p, SA;
  const Ops<T> *op;
  const Batch<T> *b;
  int nb;
};
template <typename T> Case<T> *g_now;

template <typename T, int RG> void back(const Ctx<T> &x, const Batch<T> &b, const Ops<T> &op, int n) {
  const int li = x.lane & 15, lk = x.lane >> 4;
  Vec v{0, 0, b.slot[li], b.rank[li]};
  FS<T, RG> f;
  for (int j = 0; j < RG; j++) {
    const auto w = b.w[li][1][row_of<RG>(j, lk, n)];
    f.w[j].re = w.real();
    f.w[j].im = w.imag();
  }
  RotS<T, RG> R;
  R.A = &op.H[n][1][x.lane >> 5];
  back_rot<RG>(x, v, b.most, f, R, n);
}
template <typename T, int RG> void first(const Ctx<T> &x, const Batch<T> &b, const Ops<T> &op, int n) {
  const int li = x.lane & 15, lk = x.lane >> 4;
  ZS<T, RG> z;
  FS<T, RG> f;
  for (int j = 0; j < RG; j++) {
    const int m = row_of<RG>(j, lk, n);
    const auto zp = b.src[li][n * n + n + m], zm = b.src[li][n * n + n - m], w = b.w[li][0][m];
    z.zp[j].re = zp.real(), z.zp[j].im = zp.imag();
    z.zm[j].re = zm.real(), z.zm[j].im = zm.imag();
    f.w[j].re = w.real(), f.w[j].im = w.imag();
  }
  RotS<T, RG> R;
  R.A = &op.H[n][0][x.lane >> 5];
  first_rot<RG>(x, z, f, R, n);
}
template <typename T, int RG> void coax(const Ctx<T> &x, const Ops<T> &op, int m) {
  CoaxS<T, RG> B;
  B.run(x, op.C[m], m);
  coax_put<RG>(x, B, m);
}
template <typename F> void by_rows(int rg, F f) {
  if (rg == 1) f(std::integral_constant<int, 1>{});
  if (rg == 2) f(std::integral_constant<int, 2>{});
  if (rg == 3) f(std::integral_constant<int, 3>{});
  if (rg == 4) f(std::integral_constant<int, 4>{});
}

// the order of k_m2l_ts, one wave with all units
template <typename T> void lane_body() {
  Case<T> &c = *g_now<T>;
  Ctx<T> x{{&c.X, 0}, {&c.accr, 0}, {&c.acci, 0}, c.p, c.SA, g_lane};
  auto firsts = [&](int q, int n) {
    by_rows((n + 4) >> 2, [&](auto r) { first<T, decltype(r)::value>(x, c.b[q], *c.op, n); });
  };
  for (int n = 0; n < c.p; n++) firsts(0, n);
  for (int q = 0; q < c.nb; q++) {
    order_lanes();
    for (int m = 0; m < c.p; m++)
      by_rows((c.p - m + 3) >> 2, [&](auto r) { coax<T, decltype(r)::value>(x, *c.op, m); });
    order_lanes();
    for (int n = 0; n < c.p; n++) {
      by_rows((n + 4) >> 2, [&](auto r) { back<T, decltype(r)::value>(x, c.b[q], *c.op, n); });
      if (q + 1 < c.nb) firsts(q + 1, n);
    }
  }
}

// the same translation of one vector by plain loops
template <typename T>
std::vector<std::complex<T>> plain(const Ops<T> &op, const Batch<T> &b, int li) {
  typedef std::complex<T> Z;
  const int p = op.p;
  std::vector<Z> e(p * (p + 1) / 2), o(e), out(p * p);
  auto at = [](int n, int m) { return n * (n + 1) / 2 + m; };
  auto rot = [&](int which) {
    for (int n = 0; n < p; n++) {
      std::vector<Z> re(n + 1), ro(n + 1);
      for (int i = 0; i <= n; i++)
        for (int k = 0; k <= n; k++) {
          re[i] += op.H[n][which][0][i * (n + 1) + k] * e[at(n, k)];
          ro[i] += op.H[n][which][1][i * (n + 1) + k] * o[at(n, k)];
        }
      for (int i = 0; i <= n; i++) e[at(n, i)] = re[i], o[at(n, i)] = ro[i];
    }
  };
  for (int n = 0; n < p; n++)
    for (int m = 0; m <= n; m++) {
      const Z w = b.w[li][0][m], u = b.src[li][n * n + n + m] * w,
              d = b.src[li][n * n + n - m] * std::conj(w);
      e[at(n, m)] = u + d;
      o[at(n, m)] = u - d;
    }
  rot(0);
  for (int m = 0; m < p; m++) {
    const int s = p - m;
    std::vector<Z> ce(s), co(s);
    for (int i = 0; i < s; i++)
      for (int k = 0; k < s; k++) {
        ce[i] += op.C[m][k * s + i] * e[at(m + k, m)];
        co[i] += op.C[m][k * s + i] * o[at(m + k, m)];
      }
    for (int i = 0; i < s; i++) e[at(m + i, m)] = ce[i], o[at(m + i, m)] = co[i];
  }
  rot(1);
  for (int n = 0; n < p; n++)
    for (int m = 0; m <= n; m++) {
      const Z w = b.w[li][1][m], E = e[at(n, m)], O = o[at(n, m)];
      if (m) out[n * n + n - m] = (E - O) * w;
      out[n * n + n + m] = (E + O) * std::conj(w);
    }
  return out;
}

template <typename T> void check(int p, int pattern, std::mt19937 &rng) {
  std::normal_distribution<double> g;
  auto rnd = [&] { return (T)g(rng); };
  Ops<T> op;
  op.p = p;
  for (int n = 0; n < p; n++) {
    for (int r = 0; r < 2; r++)
      for (int odd = 0; odd < 2; odd++) {
        auto &H = op.H[n][r][odd];
        H.resize((n + 1) * (n + 1));
        for (auto &h : H) h = rnd() / std::sqrt((T)(n + 1));
        for (int i = 0; i <= n && odd; i++) H[i] = H[i * (n + 1)] = 0;
      }
    op.C[n].resize((p - n) * (p - n));
    for (auto &z : op.C[n]) z = std::complex<T>(rnd(), rnd()) / std::sqrt((T)(p - n));
  }
  const int S = 7, NB = 2;
  auto b = std::make_unique<Batch<T>[]>(NB);
  for (int q = 0; q < NB; q++) {
    b[q].most = 0;
    for (int li = 0; li < 16; li++) {
      for (int f = 0; f < p * p; f++) b[q].src[li][f] = {rnd(), rnd()};
      for (int i = 0; i < 2; i++)
        for (int m = 0; m < 16; m++)
          b[q].w[li][i][m] = m ? std::polar((T)1, rnd()) : std::complex<T>(1);
      // one target; targets in turn; two targets; runs, and a batch that is not full
      b[q].slot[li] = pattern == 0 ? 3 : pattern == 1 ? (li + q) % S : pattern == 2 ? li & 1 : li / 3;
      if (pattern == 3 && li >= 11 - q) b[q].slot[li] = -1;
      b[q].rank[li] = 0;
      for (int k = 0; k < li; k++) b[q].rank[li] += b[q].slot[k] == b[q].slot[li];
      if (b[q].slot[li] < 0) b[q].rank[li] = -1;
      b[q].most = std::max(b[q].most, b[q].rank[li]);
    }
  }
  snprintf(g_case, sizeof(g_case), "%s order %d pattern %d", sizeof(T) == 8 ? "fp64" : "fp32", p,
           pattern);
  Case<T> c{{"rows", (size_t)(p * (p + 1) / 2) * kL},
            {"real sums", (size_t)p * p * S},
            {"imaginary sums", (size_t)p * p * S},
            p,
            S,
            &op,
            b.get(),
            NB};
  g_now<T> = &c;
  run_wave(lane_body<T>);
  if (!g_order) return;
  std::vector<std::complex<T>> want(p * p * S);
  for (int q = 0; q < NB; q++)
    for (int li = 0; li < 16; li++)
      if (b[q].slot[li] >= 0) {
        const auto y = plain(op, b[q], li);
        for (int f = 0; f < p * p; f++) want[f * S + b[q].slot[li]] += y[f];
      }
  double err = 0, ref = 0;
  for (size_t i = 0; i < want.size(); i++) {
    err += std::norm(std::complex<T>(c.accr.v[i], c.acci.v[i]) - want[i]);
    ref += std::norm(want[i]);
  }
  // three stages of at most 32 products and 32 sums a target, random signs
  const double tol = sizeof(T) == 8 ? 1e-13 : 1e-5;
  if (!(std::sqrt(err) <= tol * std::sqrt(ref))) {
    if (g_faults++ < 8) printf("%s: sums differ by %.1e\n", g_case, std::sqrt(err / ref));
  }
}

}  // namespace fmb_ts

int main(int argc, char **argv) {
  using namespace fmb_ts;
  g_order = argc > 1 && !strcmp(argv[1], "order");
  std::mt19937 rng(1);
  for (int p = 1; p <= 16; p++)
    for (int pattern = 0; pattern < 4; pattern++) {
      check<float>(p, pattern, rng);
      check<double>(p, pattern, rng);
    }
  printf("%d faults\n", g_faults);
  return g_faults ? 1 : 0;
}
