// Reverse-mode (adjoint) kernels: the per-point vector-Jacobian product through the converged
// local Newton (implicit-function theorem), the residual cotangent field, and the transpose of
// the block-ELL Jacobian.
//
// Reference: the backward pass of the custom_jvp local solver (models_copper.py:251-259, as
// transposed by JAX when differentiating update_int_vars_gp / compute_avg_stress) and
// implicit_vjp (crystal_plasticity_OR_design/solver.py:801-853): A^T lambda = v, then
// -(dc/dp)^T lambda.
#include <type_traits>

#include "cp_internal.hpp"
#include "cp_points.hpp"
#include "cp_reverse.hpp"

namespace cpfem {

constexpr int VBS = 64;  // threads per block of the point VJP kernel: one wave

// Converged stress of a point that the crystal-frame form does not cover.
template <int N, int L>
__device__ __attribute__((noinline)) void general_stress(const Geom& G, const double* __restrict__ u, const StateView& sv,
                                                         const MatView& mv, const SlipTable<N>* table, const SolveCfg& cfg, int64_t q,
                                                         int sub, LdsDouble* sh, double* s) {
  PointIn in;
  in.load(G, u, sv, mv, q);
  int32_t st = 0;
  Point<N, L, Crystal<N, L>::K> pt;
  CrystalRest<N, L> rest;
  setup_general<VBS>(pt, in, sv, q, sub, sh, rest);
  pt.solve(uniform_table(table), cfg.tol, cfg.max_sub_step, cfg.max_iter, s, &st);
}

// A point's inputs, read from memory again at each load().
struct PointRead {
  const Geom& G;
  const double* __restrict__ u;
  const StateView& sv;
  const MatView& mv;
  int64_t q;
  __device__ __forceinline__ void load(double* F, double* Fo, double* R) const {
    const int64_t k = reread(q);
    ugrad_from_dofs(G, u, k, F);
    load_point(sv, k, Fo, R);
    F[0] += 1.0;
    F[4] += 1.0;
    F[8] += 1.0;
  }
  __device__ __forceinline__ double g(int a) const { return sv.g[a * sv.ld + q]; }
  __device__ __forceinline__ double mp(int m) const { return mv.ptr[m][q * mv.stride[m]]; }
};

// Per-point VJP.  Output cotangents: Pbar [9][Q] (may be null), sigma cotangent given per
// cell (sbar_cell [9][n_cells], spread to points with the JxW cell-average weights; may be
// null), Fbar [9][Q], gbar [N][Q] (may be null).  Input cotangents written (or added when
// accumulate) for the direction groups in `mask`: 1 u_grad -> Hbar [9][Q], 2 Fp_inv_old ->
// Fpibar [9][Q], 4 g_old -> gbar_old [N][Q], 8 material -> pbar [8][Q], 16 R -> Rbar [9][Q].
//
// The local Newton is solved again (by L lanes a point, as in the other point kernels); the first
// lane of a point then runs the reverse sweep, with 269 to 318 registers spilled outside its loops
// (two waves per SIMD are worth more to the re-solve).  16^3, FCC: 174 us, half of it the re-solve;
// 1938 us with one forward evaluation of the map per input direction.
template <int N, int L>
__global__ void __launch_bounds__(VBS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_local_vjp(Geom G, const double* __restrict__ u, StateView sv, MatView mv, SlipSys<N> arg, const SlipTable<N>* __restrict__ gen,
            int crystal, SolveCfg cfg, int self_block, VjpArgs va) {
  constexpr int solve = lds_columns<N, L> * VBS, sweep = 2 * N * (VBS / L);
  __shared__ double sh[solve > sweep ? solve : sweep];
  __shared__ SlipSys<L == 1 ? 3 : N> tabs;
  const SlipSys<N>& tab = slip_constants<N, L, VBS>(arg, reinterpret_cast<SlipSys<N>*>(&tabs));
  const int sub = L == 1 ? 0 : (int)(threadIdx.x % L);
  const int64_t q = (int64_t)blockIdx.x * (VBS / L) + threadIdx.x / L;
  const bool valid = q < G.n_qp;
  double s[6];
  if (valid) {
    PointIn in;
    in.load(G, u, sv, mv, q);
    Crystal<N, L> pt;
    CrystalRest<N, L> rest;
    CrystalNewton<N, L> nw;
    int32_t st = 0;
    bool fits = crystal && Crystal<N, L>::applies(in.R, in.m);
    if (fits) {
      setup_crystal<VBS>(pt, in, sv, q, sub, sh, rest);
      fits = nw.solve(pt, tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, &st);
    }
    if (fits) {
      double R[9], Fpi[9];
      load_point(sv, reread(q), Fpi, R);
      pt.stress(nw.s, R, s);
    } else {
      const OutOfLine f{G, sv, mv, cfg};
      double sg[6];
      general_stress<N, L>(f.G, u, f.sv, f.mv, gen, f.cfg, q, sub, (LdsDouble*)sh, sg);
#pragma unroll
      for (int i = 0; i < 6; ++i) s[i] = sg[i];
    }
  }
  __syncthreads();  // the sweep's columns are shared out by point, not by lane
  if (!valid || sub != 0) return;
  const int64_t Q = G.n_qp;
  double wsum = 0.0;
#pragma unroll
  for (int j = 0; j < 8; ++j) wsum += jxw_at(G, (q & ~(int64_t)7) + j);
  const double w = jxw_at(G, q) / wsum;
  int mask = va.mask;
  if (!va.Hbar) mask &= ~1;
  if (!va.Fpibar) mask &= ~2;
  if (!va.gbar_old) mask &= ~4;
  if (!va.pbar) mask &= ~8;
  if (!va.Rbar) mask &= ~16;
  double park[27];
  asm volatile("" ::"v"(park) : "memory");  // in private memory: its address escapes
  const PointRead in{G, u, sv, mv, q};
  point_vjp_reverse<N>(
      in, s, *gen, mv.ao, mv.dt, self_block, [&](int i) { return va.Pbar ? va.Pbar[i * Q + q] : 0.0; },
      [&](int i) { return va.sbar_cell ? va.sbar_cell[i * G.n_cells + (q >> 3)] * w : 0.0; },
      [&](int i) { return va.Fbar ? va.Fbar[i * Q + q] : 0.0; }, va.gbar ? va.gbar + q : nullptr,
      va.slipbar ? va.slipbar + q : nullptr, Q, sh + threadIdx.x / L, VBS / L, park, mask, [&](int grp, int off, double xb) {
        double* out = grp == 1 ? va.Hbar : grp == 2 ? va.Fpibar : grp == 4 ? va.gbar_old : grp == 8 ? va.pbar : va.Rbar;
        double* dst = out + (int64_t)off * Q + q;
        *dst = va.accumulate ? *dst + xb : xb;
      });
}

// Residual cotangent of implicit_vjp: Pbar_q = -JxW_q * grad(lambda)_q with lambda zero on
// Dirichlet dofs (those rows of the constraint do not depend on the parameters).
__global__ void __launch_bounds__(256) k_grad_field(Geom G, const double* __restrict__ lam, const uint8_t* __restrict__ is_bc,
                                                   double scale_by_w, double* __restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= G.n_qp) return;
  const int64_t cell = q >> 3;
  double Gq[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) Gq[i] = 0.0;
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const int64_t nd = G.cells[cell * 8 + a];
    const double g0 = sg_at(G, 3 * a, q), g1 = sg_at(G, 3 * a + 1, q), g2 = sg_at(G, 3 * a + 2, q);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double li = is_bc[3 * nd + i] ? 0.0 : lam[3 * nd + i];
      Gq[3 * i] += li * g0;
      Gq[3 * i + 1] += li * g1;
      Gq[3 * i + 2] += li * g2;
    }
  }
  const double sc = scale_by_w != 0.0 ? scale_by_w * jxw_at(G, q) : 1.0;
#pragma unroll
  for (int i = 0; i < 9; ++i) out[i * G.n_qp + q] = sc * Gq[i];
}

// A^T in the same block-ELL layout: block (j, s') of A^T is the transpose of block
// (i = col[s'][j], tslot[s'][j]) of A; padding slots stay zero.
__global__ void __launch_bounds__(256) k_transpose(BellView M, const int32_t* __restrict__ tslot, const double* __restrict__ A,
                                                  double* __restrict__ At) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t nrow = 3 * M.n_nodes;
  if (t >= nrow * M.n_slots) return;
  const int sp = (int)(t / nrow);
  const int64_t r = t - (int64_t)sp * nrow;
  const int64_t j = r / 3;
  const int c = (int)(r - 3 * j);
  double v0 = 0.0, v1 = 0.0, v2 = 0.0;
  if (sp < M.nslot[j]) {
    const int64_t i = M.col[(int64_t)sp * M.n_nodes + j];
    const int s = tslot[(int64_t)sp * M.n_nodes + j];
    const double* src = A + (3 * (int64_t)s + c) * nrow + 3 * i;
    v0 = src[0];
    v1 = src[1];
    v2 = src[2];
  }
  At[(3 * (int64_t)sp + 0) * nrow + r] = v0;
  At[(3 * (int64_t)sp + 1) * nrow + r] = v1;
  At[(3 * (int64_t)sp + 2) * nrow + r] = v2;
}

template <int N>
void launch_local_vjp(const Geom& G, const double* u, const StateView& sv, const MatView& mv, const PointTables<N>& tb,
                      const SolveCfg& cfg, int self_block, const VjpArgs& va, hipStream_t st) {
  const int L = point_lanes(N, G.n_qp);
  const dim3 grid((unsigned)((G.n_qp * L + VBS - 1) / VBS)), block(VBS);
  const auto go = [&](auto lanes) {
    hipLaunchKernelGGL((k_local_vjp<N, decltype(lanes)::value>), grid, block, 0, st, G, u, sv, mv, tb.sys, tb.gen, tb.crystal, cfg,
                       self_block, va);
  };
  if (L == 1) go(std::integral_constant<int, 1>{});
  if (L == 2) go(std::integral_constant<int, 2>{});
  if (L == 4) go(std::integral_constant<int, 4>{});
  if constexpr (N == 24) {
    if (L == 8) go(std::integral_constant<int, 8>{});
  }
}

void launch_grad_field(const Geom& G, const double* lam, const uint8_t* is_bc, double scale_by_w, double* out,
                       hipStream_t st) {
  hipLaunchKernelGGL(k_grad_field, dim3((unsigned)((G.n_qp + 255) / 256)), dim3(256), 0, st, G, lam, is_bc, scale_by_w, out);
}

void launch_transpose(const BellView& M, const int32_t* tslot, const double* A, double* At, hipStream_t st) {
  const int64_t n = 3 * M.n_nodes * M.n_slots;
  hipLaunchKernelGGL(k_transpose, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, M, tslot, A, At);
}

template void launch_local_vjp<12>(const Geom&, const double*, const StateView&, const MatView&, const PointTables<12>&,
                                   const SolveCfg&, int, const VjpArgs&, hipStream_t);
template void launch_local_vjp<24>(const Geom&, const double*, const StateView&, const MatView&, const PointTables<24>&,
                                   const SolveCfg&, int, const VjpArgs&, hipStream_t);

}  // namespace cpfem
