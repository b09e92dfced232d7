// Floating-point operations of the crystal-frame point form, counted by running it on a number type that counts: an
// addition, a multiplication, a division or a square root is one, an fma two, and signs, absolute values and
// comparisons none; a rate's power counts what its series take.  Test infrastructure only.
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

struct Num {
  double v;
  static long n;
  constexpr Num() : v(0.0) {}
  constexpr Num(double x) : v(x) {}
  constexpr Num(int x) : v(x) {}
  explicit operator int() const { return (int)v; }
};
long Num::n = 0;
#define OP(o)                                                             \
  static inline Num operator o(Num a, Num b) { return ++Num::n, Num(a.v o b.v); }  \
  static inline Num operator o(Num a, double b) { return ++Num::n, Num(a.v o b); } \
  static inline Num operator o(double a, Num b) { return ++Num::n, Num(a o b.v); }
OP(+)
OP(-)
OP(*)
OP(/)
#define AS(o) \
  static inline Num& operator o##=(Num& a, Num b) { return a = a o b; }
AS(+)
AS(-)
AS(*)
AS(/)
#define CMP(o)                                                    \
  static inline bool operator o(Num a, Num b) { return a.v o b.v; }  \
  static inline bool operator o(Num a, double b) { return a.v o b; }
CMP(<)
CMP(>)
CMP(<=)
CMP(>=)
CMP(==)
CMP(!=)
static inline Num operator-(Num a) { return Num(-a.v); }
static inline Num fabs(Num a) { return Num(fabs(a.v)); }
static inline Num sqrt(Num a) { return ++Num::n, Num(sqrt(a.v)); }
static inline Num fmax(Num a, Num b) { return Num(fmax(a.v, b.v)); }
static inline Num rint(Num a) { return Num(rint(a.v)); }
static inline Num frexp(Num a, int* e) { return Num(frexp(a.v, e)); }
static inline Num ldexp(Num a, int e) { return Num(ldexp(a.v, e)); }
static inline Num fma(Num a, Num b, Num c) { return Num::n += 2, Num(fma(a.v, b.v, c.v)); }

#define double Num
#include "../../jax-cpfem_amd/csrc/cp_crystal.hpp"
using namespace cpfem;

// Operations of one residual, of the elastic one, of a Jacobian with its factorisation and solution, of the
// set-up, of the outputs (P, stress), and of the tangent kernel's work behind its set-up (pull-back,
// residual, tangent).
template <int N>
static void count(long* out) {
  SlipTable<N> tab;
  for (int a = 0; a < N; ++a)
    for (int d = 0; d < 3; ++d) {
      const int i = a % 3, j = (a + 1) % 3;
      tab.d[a][d] = d == i ? 1.0 : 0.0;
      tab.n[a][d] = d == j ? 1.0 : 0.0;
    }
  SlipSys<N> sys;
  make_slip_sys(tab, &sys);
  const Num R[9] = {1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0};
  Num F[9], g[N], gp[N], gi[N], x[6], d[6], P[9], s[6];
  for (int i = 0; i < 9; ++i) F[i] = i % 4 == 0 ? 1.001 : 0.0005;
  for (int a = 0; a < N; ++a) g[a] = 90.0;
  for (int q = 0; q < 6; ++q) x[q] = 50.0 + q;
  const PointMat m{20.0, 1e-3, 2.0, 500.0, 300.0, 1.4, 2.0e5, 1.3e5, 1.2e5};
  const auto lap = [&](int k) {
    out[k] = Num::n;
    Num::n = 0;
  };
  Crystal<N> pt;
  Num::n = 0;
  pt.setup(F, R, R, g, 1, m, gp, gi, 1, 1, 0, gi + Crystal<N>::K);
  lap(3);
  pt.eval_zero();
  lap(1);
  pt.eval(sys, x);
  lap(0);
  pt.step(sys, d);
  lap(2);
  crystal_pk1(pt, F, R, R, x, P);
  pt.stress(x, R, s);
  lap(4);
  Crystal<N>::pull_back(s, R, x);
  pt.eval(sys, x);
  crystal_tangent(pt, sys, F, R, R, x, [](int, const Num*) {});
  lap(5);
}

#undef double
int main() {
  long a[6], b[6];
  count<12>(a);
  count<24>(b);
  for (int k = 0; k < 6; ++k) printf("%ld %ld\n", a[k], b[k]);
  return 0;
}
