// Reverse-mode product of one material point through its converged local solve, written out by
// hand (cp_dual.hpp holds the same map in forward mode, one input direction at a time).
//
// With the point's outputs o (P, sigma, Fp_inv_new, g_new, slip increments), inputs x (u_grad,
// Fp_inv_old, g_old, the eight constants, R) and r(s, x) = 0 at the converged stress s, the
// implicit-function theorem gives
//   xbar = (do/dx)^T obar - (dr/dx)^T mu,   (dr/ds)^T mu = (do/ds)^T obar.
// Both products are one reverse sweep over the point's map: the first without residual cotangent
// for its s component, the second with obar and -mu for all inputs together, where forward mode
// needs an evaluation of the map for each of the 6 stress and 35 + N input directions.  The
// powers and logarithms of the N slip systems are evaluated twice instead of 41 + N times.
//
// Conventions at the kinks are those of the forward-mode form: |x| has slope 0 at 0, and x^y has
// slope 0 in both arguments at x = 0.
// R need not be a rotation: the stiffness is that of the closed form in R and G = R R^T.
#pragma once
#include "cp_dual.hpp"

namespace cpfem {

// c += a b, c += a b^T, c += a^T b
CPFEM_HD void acc_mm(const double* a, const double* b, double* c) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) c[3 * i + j] += a[3 * i] * b[j] + a[3 * i + 1] * b[3 + j] + a[3 * i + 2] * b[6 + j];
}
CPFEM_HD void acc_mmt(const double* a, const double* b, double* c) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) c[3 * i + j] += a[3 * i] * b[3 * j] + a[3 * i + 1] * b[3 * j + 1] + a[3 * i + 2] * b[3 * j + 2];
}
CPFEM_HD void acc_mtm(const double* a, const double* b, double* c) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) c[3 * i + j] += a[i] * b[j] + a[3 + i] * b[3 + j] + a[6 + i] * b[6 + j];
}
// c += k cof(a), the derivative of det a
CPFEM_HD void acc_cof(double k, const double* a, double* c) {
  c[0] += k * (a[4] * a[8] - a[5] * a[7]);
  c[1] += k * (a[5] * a[6] - a[3] * a[8]);
  c[2] += k * (a[3] * a[7] - a[4] * a[6]);
  c[3] += k * (a[2] * a[7] - a[1] * a[8]);
  c[4] += k * (a[0] * a[8] - a[2] * a[6]);
  c[5] += k * (a[1] * a[6] - a[0] * a[7]);
  c[6] += k * (a[1] * a[5] - a[2] * a[4]);
  c[7] += k * (a[2] * a[3] - a[0] * a[5]);
  c[8] += k * (a[0] * a[4] - a[1] * a[3]);
}
CPFEM_HD double dot9(const double* a, const double* b) {
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < 9; ++i) s += a[i] * b[i];
  return s;
}

// Inputs of a point from plain arrays.  load() may be called more than once: on the device it reads
// memory again, so that the inputs need no registers in between.
struct ReverseIn {
  const double* H;
  const double* Fpi;
  const double* g_;  // g_old of this point, stride gs
  int64_t gs;
  const double* mp_;  // xm, gss_a, h, t_sat, r, C11, C12, C44
  const double* R_;
  CPFEM_HD void load(double* F, double* Fo, double* R) const {
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      F[i] = H[i] + ((i % 4) == 0 ? 1.0 : 0.0);
      Fo[i] = Fpi[i];
      R[i] = R_[i];
    }
  }
  CPFEM_HD double g(int a) const { return g_[a * gs]; }
  CPFEM_HD double mp(int m) const { return mp_[m]; }
};

// x^y of x = 0 (or NaN), as pow gives it
CPFEM_HD double pow_at_zero(double x, double y) { return y > 0.0 ? x : y == 0.0 ? 1.0 : y < 0.0 ? 1.0 / x : y; }

// One slip system: increment, its slopes, and the hardening term t = h |dgamma| |1 - g/t_sat|^a sgn.
struct SlipRate {
  double dg, kt, kg, kp;  // dgamma and its derivatives over tau, g, 1/m
};
CPFEM_HD SlipRate slip_rate(double tau, double g, double p, double c) {
  const double x = tau / g, ax = fabs(x), st = sgn(tau), sx = sgn(x);
  SlipRate o;
  if (ax > 0.0) {
    const double lx = ln_pos(ax), pw = c * st * exp_arg(p * lx), k = pw * p / ax * sx / g;
    o.dg = pw;
    o.kt = k;
    o.kg = -k * x;
    o.kp = pw * lx;
  } else {
    o.dg = c * pow_at_zero(ax, p) * st;
    o.kt = o.kg = o.kp = 0.0;
  }
  return o;
}
struct HardRate {
  double f, fa, fx;  // |xh|^a sgn(xh), its derivatives over a and xh
};
CPFEM_HD HardRate hard_rate(double g, double tsat, double ga) {
  const double xh = 1.0 - g / tsat, ax = fabs(xh), sx = sgn(xh);
  HardRate o;
  if (ax > 0.0) {
    const double lx = ln_pos(ax), pw = exp_arg(ga * lx);
    o.f = pw * sx;
    o.fa = pw * lx * sx;
    o.fx = pw * ga / ax;  // sgn^2 = 1
  } else {
    o.f = pow_at_zero(ax, ga) * sx;
    o.fa = o.fx = 0.0;
  }
  return o;
}

// store: 2 N doubles with stride js (the lane's LDS column on the device); park: 27 doubles that
// are written before and read after the loop over the Jacobian's terms, which needs the registers.
// Pb, sb, Fb: accessors of the cotangents of P, sigma and Fp_inv_new (component -> value).
// The rest as point_vjp.
template <int N, class In, class CP, class CS, class CF, class Emit>
CPFEM_HD void point_vjp_reverse(const In& in, const double* s, const SlipTable<N>& tab, double ao, double dt, int self_block,
                                CP Pb, CS sb, CF Fb, const double* gbq, const double* slq, int64_t gs, double* store, int js,
                                double* park, int mask, Emit emit) {
  double* kap = store;           // d dgamma / d tau
  double* har = store + N * js;  // d t / d dgamma
  const double p = 1.0 / in.mp(0), c = ao * dt, rr = in.mp(4);
  double Sc[9], blk[N / 3], gblk[N / 3], tot = 0.0, gsum = 0.0;
  const auto crystal_stress = [&](const double* R) {
    double S[9], U[9];
    sym_full(s, S);
    mm3(S, R, U);
    mtm3(R, U, Sc);
  };
  const auto tau_of = [&](int a) {
    const double* d = tab.d[a];
    const double* n = tab.n[a];
    return d[0] * (Sc[0] * n[0] + Sc[1] * n[1] + Sc[2] * n[2]) + d[1] * (Sc[3] * n[0] + Sc[4] * n[1] + Sc[5] * n[2]) +
           d[2] * (Sc[6] * n[0] + Sc[7] * n[1] + Sc[8] * n[2]);
  };
#pragma unroll
  for (int b = 0; b < N / 3; ++b) blk[b] = gblk[b] = 0.0;
  // value pass: plastic velocity gradient, hardening sums
  {
    double Lpc[9];
    {
      double F[9], Fo[9], R[9];
      in.load(F, Fo, R);
      crystal_stress(R);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) Lpc[i] = 0.0;
    const double ga = in.mp(1), hh = in.mp(2), tsat = in.mp(3);
#pragma unroll 1
    for (int a = 0; a < N; ++a) {
      const double g = in.g(a);
      const SlipRate sr = slip_rate(tau_of(a), g, p, c);
      const HardRate hr = hard_rate(g, tsat, ga);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Lpc[3 * i + j] += sr.dg * (tab.d[a][i] * tab.n[a][j]);
      const double t = hh * fabs(sr.dg) * hr.f, gb = gbq ? gbq[a * gs] : 0.0;
      tot += t;
      gsum += gb;
#pragma unroll
      for (int b = 0; b < N / 3; ++b)
        if (b == a / 3) {
          blk[b] += t;
          gblk[b] += gb;
        }
      kap[a * js] = sr.kt;
      har[a * js] = hh * hr.f * sgn(sr.dg);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) park[i] = Lpc[i];
  }
  // cotangent of t: q^T gbar with the latent matrix q
  const double own = self_block ? 1.0 - rr : 0.0;
  const auto tbar_of = [&](int a) {
    double gl = 0.0;
#pragma unroll
    for (int b = 0; b < N / 3; ++b)
      if (b == a / 3) gl = gblk[b];
    return rr * gsum + own * gl;
  };
  // Lp = R Lpc R^T and Fp_inv_new = Fo (I - Lp)
  const auto plastic = [&](const double* Fo, const double* R, const double* Lpc, double* Lp, double* Fpn) {
    double X[9], Z[9];
    mm3(R, Lpc, X);
    mm3t(X, R, Lp);
    mm3(Fo, Lp, Z);
#pragma unroll
    for (int i = 0; i < 9; ++i) Fpn[i] = Fo[i] - Z[i];
  };
  // cotangent of Lpc = sum dgamma_a d_a n_a^T from that of Fp_inv_new
  const auto lpc_bar = [&](const double* Fo, const double* R, const double* Fn, double* Lb) {
    double U[9], V[9];
    mtm3(Fo, Fn, U);
    mm3(U, R, V);
    mtm3(R, V, Lb);
#pragma unroll
    for (int i = 0; i < 9; ++i) Lb[i] = -Lb[i];
  };

  double J[36], mu[6], R[9], Lb[9], Scbar[9];
  {
    // cotangents of the outputs on F, Fp_inv_new and S
    double F[9], Fo[9], Lp[9], Fpn[9], S[9], Fbar[9], Fnbar[9], Bm[9];
    in.load(F, Fo, R);
    sym_full(s, S);
    plastic(Fo, R, park, Lp, Fpn);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      Fbar[i] = 0.0;
      Fnbar[i] = Fb(i);
    }
    const double idFp = 1.0 / det3(Fpn), idF = 1.0 / det3(F);
    double Q[9], FS[9], Y[9], P[9], Pt[9], T[9];
    mm3(Fpn, S, FS);
    mm3t(FS, Fpn, Q);
#pragma unroll
    for (int i = 0; i < 9; ++i) Y[i] = Q[i] * idFp;
    mm3(F, Y, P);
    // sigma = P F^T / det F
    {
      double PFt[9], sdot = 0.0;
      mm3t(P, F, PFt);
#pragma unroll
      for (int i = 0; i < 9; ++i) {
        const double v = sb(i);
        sdot += v * PFt[i];
        T[i] = v * idF;
        Pt[i] = Pb(i);
      }
      acc_cof(-sdot * idF * idF, F, Fbar);
    }
    acc_mm(T, F, Pt);
    acc_mtm(T, P, Fbar);
    // P = F Y, Y = Fp_inv_new S Fp_inv_new^T / det Fp_inv_new
    acc_mmt(Pt, Y, Fbar);
    mtm3(F, Pt, T);
    acc_cof(-dot9(T, Q) * idFp * idFp, Fpn, Fnbar);
    {
      double Tt[9];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Tt[3 * i + j] = idFp * (T[3 * i + j] + T[3 * j + i]);
      acc_mm(Tt, FS, Fnbar);
    }
    {
      double U[9], V[9];
      mm3(T, Fpn, U);
      mtm3(Fpn, U, V);
#pragma unroll
      for (int q = 0; q < 6; ++q) mu[q] = idFp * (q < 3 ? V[4 * q] : V[3 * vi(q) + vj(q)] + V[3 * vj(q) + vi(q)]);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      park[9 + i] = Fbar[i];
      park[18 + i] = Fnbar[i];
    }
    lpc_bar(Fo, R, Fnbar, Lb);
    double A[9], Fe[9];
    mm3(F, Fo, A);
    mm3(F, Fpn, Fe);
    mtm3(Fe, A, Bm);

    // Jacobian dr/ds = I + C sum_a kappa_a e_a w_a^T (e the strain of -dFe, w = d tau / d s), and the
    // stress cotangent of the outputs through the slip systems
#pragma unroll
    for (int i = 0; i < 36; ++i) J[i] = 0.0;
#pragma unroll
    for (int i = 0; i < 9; ++i) Scbar[i] = 0.0;
#pragma unroll 1
    for (int a = 0; a < N; ++a) {
      const double* d = tab.d[a];
      const double* n = tab.n[a];
      double dl[3], nl[3], x[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        dl[i] = R[3 * i] * d[0] + R[3 * i + 1] * d[1] + R[3 * i + 2] * d[2];
        nl[i] = R[3 * i] * n[0] + R[3 * i + 1] * n[1] + R[3 * i + 2] * n[2];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) x[i] = Bm[3 * i] * dl[0] + Bm[3 * i + 1] * dl[1] + Bm[3 * i + 2] * dl[2];
      const double e[6] = {x[0] * nl[0], x[1] * nl[1], x[2] * nl[2], x[1] * nl[2] + x[2] * nl[1], x[0] * nl[2] + x[2] * nl[0],
                           x[0] * nl[1] + x[1] * nl[0]};
      const double k = kap[a * js];
      const double w[6] = {k * dl[0] * nl[0], k * dl[1] * nl[1], k * dl[2] * nl[2], k * (dl[1] * nl[2] + dl[2] * nl[1]),
                           k * (dl[0] * nl[2] + dl[2] * nl[0]), k * (dl[0] * nl[1] + dl[1] * nl[0])};
#pragma unroll
      for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int q = 0; q < 6; ++q) J[6 * i + q] += e[i] * w[q];
      double db = (slq ? slq[a * gs] : 0.0) + tbar_of(a) * har[a * js];
#pragma unroll
      for (int i = 0; i < 3; ++i) db += d[i] * (Lb[3 * i] * n[0] + Lb[3 * i + 1] * n[1] + Lb[3 * i + 2] * n[2]);
      db *= k;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Scbar[3 * i + j] += db * (d[i] * n[j]);
    }
  }
  const double C11 = in.mp(5), C12 = in.mp(6), C44 = in.mp(7), Ac = C11 - C12 - 2.0 * C44;
  {
    double C6[21];
    rotated_stiffness(R, C11, C12, C44, C6);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      double e[6], t[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) e[i] = J[6 * i + q];
      c6mul(C6, e, t);
#pragma unroll
      for (int i = 0; i < 6; ++i) J[6 * i + q] = t[i] + (i == q ? 1.0 : 0.0);
    }
    double U[9], T[9];
    mm3(R, Scbar, U);
    mm3t(U, R, T);
#pragma unroll
    for (int q = 0; q < 6; ++q) mu[q] += q < 3 ? T[4 * q] : T[3 * vi(q) + vj(q)] + T[3 * vj(q) + vi(q)];
    int piv[6];
    lu6(J, piv);
    lu6_solve_T(J, piv, mu);
  }

  // residual cotangent -mu: r = s - C E, E = (Fe^T Fe - I) / 2.  M is the tensor of mu (mu : C : E),
  // Y = C : M.
  double Rbar[9], mbar[NPAR];
  {
    double F[9], Fo[9], Lpc[9], Lp[9], Fpn[9], Fe[9], Fbar[9], Fnbar[9], G[9];
    in.load(F, Fo, R);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      Rbar[i] = 0.0;
      Lpc[i] = park[i];
      Fbar[i] = park[9 + i];
      Fnbar[i] = park[18 + i];
    }
    plastic(Fo, R, Lpc, Lp, Fpn);
    mm3(F, Fpn, Fe);
    mm3t(R, R, G);
    {
      const double M[9] = {mu[0], 0.5 * mu[5], 0.5 * mu[4], 0.5 * mu[5], mu[1], 0.5 * mu[3], 0.5 * mu[4], 0.5 * mu[3], mu[2]};
      double E[9], MG[9], EG[9], GMG[9], T[9];
      mtm3(Fe, Fe, E);
#pragma unroll
      for (int i = 0; i < 9; ++i) E[i] = 0.5 * (E[i] - ((i % 4) == 0 ? 1.0 : 0.0));
      mm3(M, G, MG);
      mm3(E, G, EG);
      mm3(G, EG, T);
      const double bm = dot9(M, G), be = dot9(E, G), mg = dot9(M, T);
      mm3(G, MG, GMG);
      double cub = 0.0, Y[9], Mr[9], Er[9];
      mm3(M, R, Mr);
      mm3(E, R, Er);
#pragma unroll
      for (int i = 0; i < 9; ++i) Y[i] = C12 * bm * G[i] + 2.0 * C44 * GMG[i];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const double ba = R[a] * Mr[a] + R[3 + a] * Mr[3 + a] + R[6 + a] * Mr[6 + a];
        const double ea = R[a] * Er[a] + R[3 + a] * Er[3 + a] + R[6 + a] * Er[6 + a];
        cub += ba * ea;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          Rbar[3 * i + a] += 2.0 * Ac * (ea * Mr[3 * i + a] + ba * Er[3 * i + a]);
#pragma unroll
          for (int j = 0; j < 3; ++j) Y[3 * i + j] += Ac * ba * R[3 * i + a] * R[3 * j + a];
        }
      }
      mbar[5] = cub;
      mbar[6] = bm * be - cub;
      mbar[7] = 2.0 * mg - 2.0 * cub;
      // G: C12 (M:G)(G:E) + 2 C44 M:(G E G), symmetric in the sum of both orders
      mm3(MG, E, T);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int ij = 3 * i + j;
          GMG[ij] = 2.0 * (C12 * (be * M[ij] + bm * E[ij]) + 2.0 * C44 * (T[ij] + T[3 * j + i]));
        }
      acc_mm(GMG, R, Rbar);
      // E: dFe = Fe Y
      mm3(Fe, Y, T);
      acc_mmt(T, Fpn, Fbar);
      acc_mtm(F, T, Fnbar);
    }
    if (mask & 1) {
#pragma unroll
      for (int i = 0; i < 9; ++i) emit(1, i, Fbar[i]);
    }
    if (mask & 2) {  // Fp_inv_new = Fo (I - Lp)
      double T[9];
      mm3t(Fnbar, Lp, T);
#pragma unroll
      for (int i = 0; i < 9; ++i) emit(2, i, Fnbar[i] - T[i]);
    }
    {  // Lp = R Lpc R^T
      double Lpb[9], U[9];
      mtm3(Fo, Fnbar, Lpb);
#pragma unroll
      for (int i = 0; i < 9; ++i) Lpb[i] = -Lpb[i];
      mm3t(R, Lpc, U);
      acc_mm(Lpb, U, Rbar);
      mm3(R, Lpc, U);
      acc_mtm(Lpb, U, Rbar);
    }
    lpc_bar(Fo, R, Fnbar, Lb);
    crystal_stress(R);
  }
  // the slip systems again, with the total cotangents
#pragma unroll
  for (int i = 0; i < 9; ++i) Scbar[i] = 0.0;
  double pb = 0.0, ab = 0.0, hb = 0.0, tb = 0.0, rb = 0.0;
  {
    const double ga = in.mp(1), hh = in.mp(2), tsat = in.mp(3), it = 1.0 / tsat;
#pragma unroll 1
    for (int a = 0; a < N; ++a) {
      const double* d = tab.d[a];
      const double* n = tab.n[a];
      const double g = in.g(a);
      const SlipRate sr = slip_rate(tau_of(a), g, p, c);
      const HardRate hr = hard_rate(g, tsat, ga);
      const double tbar = tbar_of(a), ad = fabs(sr.dg), gb = gbq ? gbq[a * gs] : 0.0;
      double bl = 0.0;
#pragma unroll
      for (int b = 0; b < N / 3; ++b)
        if (b == a / 3) bl = blk[b];
      rb += gb * (self_block ? tot - bl : tot);
      double db = (slq ? slq[a * gs] : 0.0) + tbar * har[a * js];
#pragma unroll
      for (int i = 0; i < 3; ++i) db += d[i] * (Lb[3 * i] * n[0] + Lb[3 * i + 1] * n[1] + Lb[3 * i + 2] * n[2]);
      const double xhb = tbar * hh * ad * hr.fx;
      hb += tbar * ad * hr.f;
      ab += tbar * hh * ad * hr.fa;
      tb += xhb * g * it * it;
      pb += db * sr.kp;
      if (mask & 4) emit(4, a, gb + db * sr.kg - xhb * it);
      const double tt = db * sr.kt;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Scbar[3 * i + j] += tt * (d[i] * n[j]);
    }
  }
  if (mask & 8) {
    mbar[0] = -pb * p * p;
    mbar[1] = ab;
    mbar[2] = hb;
    mbar[3] = tb;
    mbar[4] = rb;
#pragma unroll
    for (int i = 0; i < NPAR; ++i) emit(8, i, mbar[i]);
  }
  if (mask & 16) {  // Sc = R^T S R
    double S[9], U[9], V[9];
    sym_full(s, S);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) V[3 * i + j] = Scbar[3 * i + j] + Scbar[3 * j + i];
    mm3(S, R, U);
    acc_mm(U, V, Rbar);
#pragma unroll
    for (int i = 0; i < 9; ++i) emit(16, i, Rbar[i]);
  }
}

}  // namespace cpfem
