// Local Newton of one quadrature point in its crystal's frame: the form of cp_point.hpp's
// Point<N> that the kernels use where R is a rotation times a scalar (any quaternion gives one)
// and the Schmid dyads are traceless (slip directions lie in their planes).  Same unknown, same
// residual, same decisions; other orders of the sums.
//
// With R^T R = B and S' = R^T S R the equations of cp_point.hpp become, exactly for any R,
//   tau_a = P0_a : S',  Fh = Fe R = A R (I - Lpc B),  E' = 1/2 (Fh^T Fh - B),
//   r' = S' - B (C_cubic : E') B,
// and with B = bb I the rotated stiffness (21 values, 36 products per use) becomes three
// constants, a resolved shear stress 5 products with constants shared by all lanes instead of 12,
// the Jacobian's sum over slip systems 40 instead of 87.  What else is cheaper than in Point:
//  * S' = 0 has no slip, so the first residual is the elastic one and the first step is -r': no
//    slip loop, no Jacobian, no factorisation.
//  * The step solves (C^-1 + G) ds' = -C^-1 r', G = sum_a g'_a sym(K z_a) b_a^T with K near
//    the identity: nearly symmetric positive definite, so it is factorised without row
//    exchanges (which are most of a 6x6 factorisation's instructions); a point whose
//    multipliers exceed GROWTH is handed to the general form, from the start.
//  * dgamma and its derivative come from one power |tau/g|^(1/m - 1), without branches.
//  * The tangent reuses G's sums sum_a g'_a z_a b_a^T as the derivative of the plastic velocity
//    gradient, instead of six more loops over the slip systems.
// dgamma/dtau and 1/g_old live outside the register file, in LDS (whose 20 KB a wave at two waves
// per SIMD hold 1/g_old of 14 of 24 systems) and, for the others, in the lane's private memory, and
// the slip loops are rolled:
// unrolled, with dgamma/dtau in registers, the kernels spilled 160 to 240 registers and took
// twice the time.
//
// L lanes (adjacent, a power of two up to 8) may share one point: each takes N / L slip systems in
// a row, the sums are exchanged by DPP in an order that gives every lane the same bits, and
// everything else is computed by all of them alike.
#pragma once
#include "cp_point.hpp"

namespace cpfem {

// Schmid dyads z = d (x) n and db = d tau / d s' (shear components count twice) of the slip systems.
template <int N>
struct SlipSys {
  double z[N][8];  // without the last diagonal component, -(z0 + z4)
  double b[N][5];  // components 0, 1, 3, 4, 5; component 2 is -(b0 + b1)
};

// False if a dyad is not traceless (to rounding).
template <int N>
inline bool make_slip_sys(const SlipTable<N>& t, SlipSys<N>* o) {
  bool ok = true;
  for (int a = 0; a < N; ++a) {
    const double* d = t.d[a];
    const double* n = t.n[a];
    for (int k = 0; k < 8; ++k) o->z[a][k] = d[k / 3] * n[k % 3];
    o->b[a][0] = d[0] * n[0];
    o->b[a][1] = d[1] * n[1];
    o->b[a][2] = d[1] * n[2] + d[2] * n[1];
    o->b[a][3] = d[0] * n[2] + d[2] * n[0];
    o->b[a][4] = d[0] * n[1] + d[1] * n[0];
    ok = ok && fabs(d[0] * n[0] + d[1] * n[1] + d[2] * n[2]) <= 1e-15;
  }
  return ok;
}

// a b + c for a constant c.  On the device the instruction is written out: the compiler otherwise
// copies c into the accumulator first, a second instruction for each term of a polynomial.
CPFEM_HD double fma_c(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
#else
  return fma(a, b, c);
#endif
}

// 1 / x for x away from the ends of the exponent range, and n / d likewise (about 1 ulp; without the
// scaling and special cases of the division).
CPFEM_HD double fast_rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
#else
  return 1.0 / x;
#endif
}
CPFEM_HD double fast_div(double n, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = fast_rcp(d), q = n * r;
  return fma(fma(-d, q, n), r, q);
#else
  return n / d;
#endif
}

// x^p for x >= 0 and finite p ln x, without branches: ln_pos and exp_arg (cp_point.hpp: their
// reductions, series and constants) without the special cases that ldexp's overflow and
// underflow already give.  x = 0 gives 0, NaN gives NaN.
CPFEM_HD double rate_power(double x, double p) {
  int e;
#if defined(__HIP_DEVICE_COMPILE__)
  double m = __builtin_amdgcn_frexp_mant(x);
  e = __builtin_amdgcn_frexp_exp(x);
#else
  double m = frexp(x, &e);
#endif
  const bool low = m < 0.70710678118654752440;
  m = low ? m + m : m;
  e -= low ? 1 : 0;
  const double s = fast_div(m - 1.0, m + 1.0), z = s * s;
  double t = fma_c(1.0 / 23.0, z, 1.0 / 21.0);
  t = fma_c(t, z, 1.0 / 19.0);
  t = fma_c(t, z, 1.0 / 17.0);
  t = fma_c(t, z, 1.0 / 15.0);
  t = fma_c(t, z, 1.0 / 13.0);
  t = fma_c(t, z, 1.0 / 11.0);
  t = fma_c(t, z, 1.0 / 9.0);
  t = fma_c(t, z, 1.0 / 7.0);
  t = fma_c(t, z, 1.0 / 5.0);
  t = fma_c(t, z, 1.0 / 3.0);
  const double lm = 2.0 * fma(s * z, t, s);
  const double y = p * fma((double)e, LN2_D, lm);
  const double k = rint(y * (1.0 / LN2_D));
  const double r = fma(-k, LN2_TAIL, fma(-k, LN2_HEAD, y));
  double q = fma_c(1.0 / 6227020800.0, r, 1.0 / 479001600.0);
  q = fma_c(q, r, 1.0 / 39916800.0);
  q = fma_c(q, r, 1.0 / 3628800.0);
  q = fma_c(q, r, 1.0 / 362880.0);
  q = fma_c(q, r, 1.0 / 40320.0);
  q = fma_c(q, r, 1.0 / 5040.0);
  q = fma_c(q, r, 1.0 / 720.0);
  q = fma_c(q, r, 1.0 / 120.0);
  q = fma_c(q, r, 1.0 / 24.0);
  q = fma_c(q, r, 1.0 / 6.0);
  q = fma_c(q, r, 0.5);
  q = fma_c(q, r, 1.0);
  q = fma_c(q, r, 1.0);
#if defined(__HIP_DEVICE_COMPILE__)
  const double w = __builtin_amdgcn_ldexp(q, (int)k);
#else
  const double w = k > 4000.0 ? INFINITY : k < -4000.0 ? 0.0 : ldexp(q, (int)k);
#endif
  return x > 0.0 ? w : x;
}

template <int N, int L = 1, int KS = (N / L > 12 ? 14 : N / L)>
struct Crystal {
  static constexpr int M = N / L;  // slip systems of this lane
  static_assert(N % L == 0 && M % 3 == 0, "a lane takes whole blocks of three slip systems");
  static constexpr int K = KS;  // how many of them have |1/g_old| in the gi store, the others in gr
  double Ah[9];          // A R
  double B[6];           // R^T R (Voigt)
  double bb, ibb;        // its mean diagonal, and the reciprocal
  double k1, k2, k3;     // bb^2 (C11 - C12), bb^2 C12, bb^2 C44
  double i1, i2, i3;     // inverse: (C^-1 t)_ii = i1 t_ii - i2 tr t, shear i3 t
  double p, p1, c;       // 1/m, 1/m - 1, gamma0 dt
  double* gpv;           // d dgamma / d tau of this lane's systems, stride st
  const double* gi;      // |1 / g_old| of the first K, stride sti
  const double* gr;      // of the others
  int st;
  int64_t sti;
  int a0;                // first slip system of this lane
  double zero;           // 0 times the sum of 1 / g_old: carries a NaN, or a zero resistance, to S' = 0
  // last evaluated point
  double Lpc[9];
  double Fh[9];
  double r[6];
  double nr;
  int nev;

  CPFEM_HD double& gp(int j) const { return gpv[j * st]; }

  // Whether a point may run in this form: R a scaled rotation, C positive definite, m not 1 (where
  // the rate has a slope at zero stress).
  CPFEM_HD static bool applies(const double* R, const PointMat& m) {
    double G[9];
    mtm3(R, R, G);
    const double q = (G[0] + G[4] + G[8]) * (1.0 / 3.0), e = 1e-14 * q;
    return q > 0.0 && q < 1e100 && fabs(G[0] - q) <= e && fabs(G[4] - q) <= e && fabs(G[8] - q) <= e && fabs(G[1]) <= e &&
           fabs(G[2]) <= e && fabs(G[5]) <= e && m.C11 - m.C12 > 0.0 && m.C11 + 2.0 * m.C12 > 0.0 && m.C44 > 0.0 && m.p != 1.0;
  }

  // Set-up from F, Fp_inv_old, R and the constants; stores |1/g_old| of the lane's systems at gi_store.
  CPFEM_HD void setup(const double* F, const double* Fpi_old, const double* R, const double* g_old, int64_t gstride,
                      const PointMat& m, double* gp_store, double* gi_store, int stride, int64_t stride_gi, int sub = 0,
                      double* gr_store = nullptr) {
    {
      double A[9];
      mm3(F, Fpi_old, A);
      mm3(A, R, Ah);
    }
    B[0] = R[0] * R[0] + R[3] * R[3] + R[6] * R[6];
    B[1] = R[1] * R[1] + R[4] * R[4] + R[7] * R[7];
    B[2] = R[2] * R[2] + R[5] * R[5] + R[8] * R[8];
    B[3] = R[1] * R[2] + R[4] * R[5] + R[7] * R[8];
    B[4] = R[0] * R[2] + R[3] * R[5] + R[6] * R[8];
    B[5] = R[0] * R[1] + R[3] * R[4] + R[6] * R[7];
    bb = (B[0] + B[1] + B[2]) * (1.0 / 3.0);
    ibb = 1.0 / bb;
    const double b2 = bb * bb;
    k1 = b2 * (m.C11 - m.C12);
    k2 = b2 * m.C12;
    k3 = b2 * m.C44;
    i1 = 1.0 / k1;
    i2 = k2 * i1 / (k1 + 3.0 * k2);
    i3 = 1.0 / k3;
    p = m.p;
    p1 = m.p - 1.0;
    c = m.c;
    gpv = gp_store;
    gi = gi_store;
    st = stride;
    sti = stride_gi;
    a0 = sub * M;
    gr = gr_store;
    nev = 0;
    double z = 0.0;
#pragma unroll 3
    for (int j = 0; j < M; ++j) {
      const double v = fabs(1.0 / g_old[(a0 + j) * gstride]);
      if (j < K)
        gi_store[j * stride_gi] = v;
      else
        gr_store[j - K] = v;
      z += 0.0 * v;
    }
    zero = lane_sum<L>(z);
  }

  CPFEM_HD void cubic(const double* e, double* t) const {  // t = C : e (e engineering)
    const double tr = k2 * (e[0] + e[1] + e[2]);
    t[0] = k1 * e[0] + tr;
    t[1] = k1 * e[1] + tr;
    t[2] = k1 * e[2] + tr;
    t[3] = k3 * e[3];
    t[4] = k3 * e[4];
    t[5] = k3 * e[5];
  }

  // Residual from Fh.
  CPFEM_HD void residual(const double* x) {
    double e[6], t[6];
    e[0] = 0.5 * (Fh[0] * Fh[0] + Fh[3] * Fh[3] + Fh[6] * Fh[6] - B[0]);
    e[1] = 0.5 * (Fh[1] * Fh[1] + Fh[4] * Fh[4] + Fh[7] * Fh[7] - B[1]);
    e[2] = 0.5 * (Fh[2] * Fh[2] + Fh[5] * Fh[5] + Fh[8] * Fh[8] - B[2]);
    e[3] = Fh[1] * Fh[2] + Fh[4] * Fh[5] + Fh[7] * Fh[8] - B[3];
    e[4] = Fh[0] * Fh[2] + Fh[3] * Fh[5] + Fh[6] * Fh[8] - B[4];
    e[5] = Fh[0] * Fh[1] + Fh[3] * Fh[4] + Fh[6] * Fh[7] - B[5];
    cubic(e, t);
#pragma unroll
    for (int q = 0; q < 6; ++q) r[q] = x[q] - t[q];
    // |r| of the unrotated residual: r = R r' R^T / bb^2
    nr = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + 2.0 * (r[3] * r[3] + r[4] * r[4] + r[5] * r[5])) * ibb;
  }

  // At S' = 0: no slip.
  CPFEM_HD void eval_zero() {
    ++nev;
    const double x[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      Lpc[i] = zero;
      Fh[i] = Ah[i] + zero;
    }
#pragma unroll 3
    for (int j = 0; j < M; ++j) gp(j) = zero;
    residual(x);
  }

  // Slip increment over tau and its derivative over p, of |tau| / g = ax.
  CPFEM_HD double rate(double ax, double gia) const {
    return c * gia * rate_power(ax, p1);
  }

  template <class Tab>
  CPFEM_HD double tau(const Tab& tab, int a, const double* x) const {
    return tab.b[a][0] * (x[0] - x[2]) + tab.b[a][1] * (x[1] - x[2]) + tab.b[a][2] * x[3] + tab.b[a][3] * x[4] + tab.b[a][4] * x[5];
  }
  // Slip increment of this lane's system j at the last evaluated point x.
  template <class Tab>
  CPFEM_HD double increment(const Tab& tab, int j, const double* x) const {
    return gp(j) / p * tau(tab, a0 + j, x);
  }

  // Residual at x = S'; fills gp, Lpc, Fh, r, nr.
  template <class Tab>
  CPFEM_HD void eval(const Tab& tab, const double* x) {
    ++nev;
    double l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) l[i] = 0.0;
    const double u0 = x[0] - x[2], u1 = x[1] - x[2];
    const auto system = [&](int j, double gia) {
      const int a = L == 1 ? j : a0 + j;
      const double t = tab.b[a][0] * u0 + tab.b[a][1] * u1 + tab.b[a][2] * x[3] + tab.b[a][3] * x[4] + tab.b[a][4] * x[5];
      const double y = rate(fabs(t) * gia, gia), dg = y * t;
      gp(j) = p * y;
#pragma unroll
      for (int i = 0; i < 8; ++i) l[i] += dg * tab.z[a][i];
    };
    double rest = K < M ? gr[0] : 0.0;
    double next = gi[0];
    // (a lane of three systems evaluates them together: their chains fill each other's latency)
#pragma unroll(M == 3 ? 3 : 2)
    for (int j = 0; j < K; ++j) {
      const double gia = next;
      next = gi[(j + 1 < K ? j + 1 : j) * sti];  // in flight during this system
      system(j, gia);
    }
#pragma unroll 2
    for (int j = K; j < M; ++j) {
      const double gia = rest;
      rest = gr[(j + 1 < M ? j + 1 : j) - K];
      system(j, gia);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) Lpc[i] = lane_sum<L>(l[i]);
    Lpc[8] = -(Lpc[0] + Lpc[4]);
    double W[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) W[i] = ((i % 4) == 0 ? 1.0 : 0.0) - bb * Lpc[i];
    mm3(Ah, W, Fh);
    residual(x);
  }

  // Z[8 j + i] = sum_a g'_a z_a,i b_a,j: the stored components of dLpc / ds'_q for q = 0, 1, 3, 4, 5
  // (column 2 is minus the sum of the first two).
  template <class Tab>
  CPFEM_HD void dyads(const Tab& tab, double* Z) const {
#pragma unroll
    for (int i = 0; i < 40; ++i) Z[i] = 0.0;
#pragma unroll(M == 3 ? 3 : 1)
    for (int m = 0; m < M; ++m) {
      const int a = L == 1 ? m : a0 + m;
      const double g = gp(m);
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const double w = g * tab.b[a][j];
#pragma unroll
        for (int i = 0; i < 8; ++i) Z[8 * j + i] += w * tab.z[a][i];
      }
    }
    if (L > 1) {
#pragma unroll
      for (int i = 0; i < 40; ++i) Z[i] = lane_sum<L>(Z[i]);
    }
  }
  CPFEM_HD static void column(const double* Z, int j, double* D) {
#pragma unroll
    for (int i = 0; i < 8; ++i) D[i] = Z[8 * j + i];
    D[8] = -(D[0] + D[4]);
  }
  CPFEM_HD void coupling(double* K) const {  // bb Fh^T A R
    mtm3(Fh, Ah, K);
#pragma unroll
    for (int i = 0; i < 9; ++i) K[i] *= bb;
  }
  // Column q of G: sym(K D), engineering.
  CPFEM_HD static void strain(const double* K, const double* D, int q, double* J) {
    double X[9];
    mm3(K, D, X);
    J[q] = X[0];
    J[6 + q] = X[4];
    J[12 + q] = X[8];
    J[18 + q] = X[5] + X[7];
    J[24 + q] = X[2] + X[6];
    J[30 + q] = X[1] + X[3];
  }
  // Completes column 2 of G and adds C^-1.
  CPFEM_HD void compliance(double* J) const {
#pragma unroll
    for (int i = 0; i < 6; ++i) J[6 * i + 2] = -(J[6 * i] + J[6 * i + 1]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int j = 0; j < 3; ++j) J[6 * i + j] += i == j ? i1 - i2 : -i2;
      J[7 * (i + 3)] += i3;
    }
  }
  // C^-1 + G (6x6, row-major).
  template <class Tab>
  CPFEM_HD void matrix(const Tab& tab, double* J) const {
    double K[9], Z[40];
    dyads(tab, Z);
    coupling(K);
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      double D[9];
      column(Z, j, D);
      strain(K, D, j < 2 ? j : j + 1, J);
    }
    compliance(J);
  }

  // Factorisation without row exchanges, the reciprocal pivots on the diagonal; false if a
  // multiplier exceeds GROWTH (or is not finite).
  static constexpr double GROWTH = 1e3;
  CPFEM_HD static bool lu(double* J) {
    double big = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double inv = fast_rcp(J[7 * k]);
      J[7 * k] = inv;
#pragma unroll
      for (int i = k + 1; i < 6; ++i) {
        const double f = J[6 * i + k] * inv;
        J[6 * i + k] = f;
        big = fmax(big, fabs(f));
#pragma unroll
        for (int j = k + 1; j < 6; ++j) J[6 * i + j] -= f * J[6 * k + j];
      }
    }
    return big <= GROWTH && fabs(J[35]) <= 1.7976931348623157e308;
  }
  CPFEM_HD static void lu_solve(const double* J, double* b) {
#pragma unroll
    for (int i = 1; i < 6; ++i)
#pragma unroll
      for (int j = 0; j < i; ++j) b[i] -= J[6 * i + j] * b[j];
#pragma unroll
    for (int i = 5; i >= 0; --i) {
#pragma unroll
      for (int j = i + 1; j < 6; ++j) b[i] -= J[6 * i + j] * b[j];
      b[i] *= J[7 * i];
    }
  }

  CPFEM_HD void rhs(double* d) const {  // -C^-1 r'
    const double tr = i2 * (r[0] + r[1] + r[2]);
    d[0] = tr - i1 * r[0];
    d[1] = tr - i1 * r[1];
    d[2] = tr - i1 * r[2];
    d[3] = -i3 * r[3];
    d[4] = -i3 * r[4];
    d[5] = -i3 * r[5];
  }
  // Newton step ds' at the last evaluated point; false if the factorisation needs row exchanges.
  template <class Tab>
  CPFEM_HD bool step(const Tab& tab, double* d) const {
    double J[36];
    matrix(tab, J);
    const bool ok = lu(J);
    rhs(d);
    lu_solve(J, d);
    return ok;
  }

  // Stress S = R S' R^T / bb^2 (Voigt) of x = S'.
  CPFEM_HD void stress(const double* x, const double* R, double* s) const {
    double S[9], T[9], U[9];
    sym_full(x, S);
    mm3(R, S, T);
    mm3t(T, R, U);
    const double f = ibb * ibb;
#pragma unroll
    for (int q = 0; q < 6; ++q) s[q] = f * U[3 * vi(q) + vj(q)];
  }
  // x = S' = R^T S R of the stress s.
  CPFEM_HD static void pull_back(const double* s, const double* R, double* x) {
    double S[9], T[9], U[9];
    sym_full(s, S);
    mm3(S, R, T);
    mtm3(R, T, U);
#pragma unroll
    for (int q = 0; q < 6; ++q) x[q] = U[3 * vi(q) + vj(q)];
  }
};

// One point's Newton iteration (models_copper.py:204-249), a residual per pass: the wave's lanes that
// search a step length and those that form a step share the passes.
template <int N, int L>
struct CrystalNewton {
  double s[6], d[6];  // accepted S', step
  double nr0, lam;
  int it, k;          // Newton iterations; residuals of the current step (0: the step is to be formed)
  bool lost;          // the factorisation needs row exchanges: the point belongs to the general form

  CPFEM_HD bool start(Crystal<N, L>& pt, double tol) {
#pragma unroll
    for (int q = 0; q < 6; ++q) s[q] = 0.0;
    it = 0;
    k = 0;
    lost = false;
    pt.eval_zero();
    return pt.nr > tol;
  }
  // Resumes from s with `it` iterations done.
  template <class Tab>
  CPFEM_HD bool resume(Crystal<N, L>& pt, const Tab& tab, double tol) {
    k = 0;
    lost = false;
    if (it == 0)
      pt.eval_zero();
    else
      pt.eval(tab, s);
    return pt.nr > tol;
  }
  // The next residual; true while the point goes on.  Sets PT_CAPPED at max_iter.
  template <class Tab>
  CPFEM_HD bool advance(Crystal<N, L>& pt, const Tab& tab, double tol, int max_sub_step, int max_iter, int32_t* stat) {
    if (k == 0) {
      if (it >= max_iter) {
        *stat |= PT_CAPPED;
        return false;
      }
      if (it == 0) {  // no slip at S' = 0: J = I
#pragma unroll
        for (int q = 0; q < 6; ++q) d[q] = -pt.r[q];
      } else if (!pt.step(tab, d)) {
        lost = true;
        return false;
      }
      nr0 = pt.nr;
      lam = 1.0;
      ++it;
    }
    double x[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) x[q] = s[q] + lam * d[q];
    pt.eval(tab, x);
    lam *= 0.5;
    ++k;
    if (pt.nr >= nr0 && k < max_sub_step) return true;
#pragma unroll
    for (int q = 0; q < 6; ++q) s[q] = x[q];
    k = 0;
    return pt.nr > tol;
  }
  template <class Tab>
  // Converged, or false if the point is to be solved in the general form.
  CPFEM_HD bool solve(Crystal<N, L>& pt, const Tab& tab, double tol, int max_sub_step, int max_iter, int32_t* stat) {
    bool act = start(pt, tol);
    while (act) act = advance(pt, tab, tol, max_sub_step, max_iter, stat);
    finite(pt, stat);
    return !lost;
  }
  CPFEM_HD static void finite(const Crystal<N, L>& pt, int32_t* stat) {
    if (!(fabs(pt.nr) <= 1.7976931348623157e308)) *stat |= PT_NONFINITE;
  }
};

// First Piola-Kirchhoff stress P = F Y, Y = Ph S' Ph^T / (bb^2 det Fp_inv_new), Ph = Fp_inv_new R, and
// the consistent tangent's ingredients.  Q = Fp_inv_old R, W = I - bb Lpc: Ph = Q W and
// det Fp_inv_new = det Fp_inv_old det W.
template <int N, int L, int KS>
CPFEM_HD void crystal_pk1(const Crystal<N, L, KS>& pt, const double* F, const double* Fpi_old, const double* R, const double* x,
                          double* P) {
  double W[9], Q[9], Ph[9], S[9], U[9], Y[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) W[i] = ((i % 4) == 0 ? 1.0 : 0.0) - pt.bb * pt.Lpc[i];
  mm3(Fpi_old, R, Q);
  mm3(Q, W, Ph);
  sym_full(x, S);
  mm3t(S, Ph, U);
  mm3(Ph, U, Y);
  const double f = 1.0 / (pt.bb * pt.bb * det3(Fpi_old) * det3(W));
#pragma unroll
  for (int i = 0; i < 9; ++i) Y[i] *= f;
  mm3(F, Y, P);
}

// Consistent tangent dP/dH at the converged point x = S' (IFT of f_jvp, models_copper.py:251-259):
//   (C^-1 + G) ds' = sym(Fh^T dH Ph) (engineering),  dLpc = sum_q D_q ds'_q,
//   dP = dH Y + F dY,  dY = Ycal ds'.
// Column m = 3 k + l (dH = e_k e_l^T) goes to sink(m, dP[9]).  False, and nothing to the sink, if the
// factorisation needs row exchanges.
template <int N, int L, int KS, class Tab, class Sink>
CPFEM_HD bool crystal_tangent(const Crystal<N, L, KS>& pt, const Tab& tab, const double* F, const double* Fpi_old, const double* R,
                              const double* x, Sink sink) {
  double Ph[9], Yv[9], Yc[36], J[36];
  double f;  // 1 / (bb^2 det Fp_inv_new)
  {
    double K[9], W[9], Wi[9], Q[9], S[9], U[9], Z[40];
    pt.dyads(tab, Z);
    pt.coupling(K);
#pragma unroll
    for (int i = 0; i < 9; ++i) W[i] = ((i % 4) == 0 ? 1.0 : 0.0) - pt.bb * pt.Lpc[i];
    mm3(Fpi_old, R, Q);
    mm3(Q, W, Ph);
    const double dW = det3(W);
    inv3(W, dW, Wi);
    f = 1.0 / (pt.bb * pt.bb * det3(Fpi_old) * dW);
    sym_full(x, S);
    mm3t(S, Ph, U);
    mm3(Ph, U, Yv);
    // Yc first holds the part through Fp_inv_new, -bb (V + V^T - Yv tr)
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      const int q = j < 2 ? j : j + 1;
      double D[9], T[9], V[9];
      Crystal<N, L>::column(Z, j, D);
      Crystal<N, L>::strain(K, D, q, J);
      mm3(Q, D, T);
      mm3(T, U, V);  // -dPh S' Ph^T / bb
      double tr = 0.0;  // -tr(W^-1 dW) / bb
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) tr += Wi[3 * a + b] * D[3 * b + a];
#pragma unroll
      for (int m = 0; m < 6; ++m) {
        const int a = vi(m), b = vj(m);
        Yc[6 * m + q] = -pt.bb * (V[3 * a + b] + V[3 * b + a] - Yv[3 * a + b] * tr);
      }
    }
#pragma unroll
    for (int m = 0; m < 6; ++m) Yc[6 * m + 2] = -(Yc[6 * m] + Yc[6 * m + 1]);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const int i = vi(q), j = vj(q);
#pragma unroll
      for (int m = 0; m < 6; ++m) {
        const int a = vi(m), b = vj(m);
        const double mid = (i == j) ? Ph[3 * a + i] * Ph[3 * b + i] : Ph[3 * a + i] * Ph[3 * b + j] + Ph[3 * a + j] * Ph[3 * b + i];
        Yc[6 * m + q] = (Yc[6 * m + q] + mid) * f;
      }
    }
    pt.compliance(J);
  }
  if (!Crystal<N, L>::lu(J)) return false;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const double f0 = pt.Fh[3 * k], f1 = pt.Fh[3 * k + 1], f2 = pt.Fh[3 * k + 2];
      const double q0 = Ph[3 * l], q1 = Ph[3 * l + 1], q2 = Ph[3 * l + 2];
      double ds[6];
      ds[0] = f0 * q0; ds[1] = f1 * q1; ds[2] = f2 * q2;
      ds[3] = f1 * q2 + f2 * q1; ds[4] = f0 * q2 + f2 * q0; ds[5] = f0 * q1 + f1 * q0;
      Crystal<N, L>::lu_solve(J, ds);
      double dy[6], dY[9], dP[9];
#pragma unroll
      for (int m = 0; m < 6; ++m) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q) acc += Yc[6 * m + q] * ds[q];
        dy[m] = acc;
      }
      sym_full(dy, dY);
      mm3(F, dY, dP);
#pragma unroll
      for (int jj = 0; jj < 3; ++jj) dP[3 * k + jj] += Yv[3 * l + jj] * f;
      sink(3 * k + l, dP);
    }
  }
  return true;
}

}  // namespace cpfem
