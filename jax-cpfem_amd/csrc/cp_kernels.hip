// Element-level kernels of the CP hot path: quadrature-point constitutive update,
// element residual / stiffness, scatter-free gathers into the block-ELL matrix and the
// residual vector, cell-averaged Cauchy stress and the history update.
//
// Upstream element semantics (jax-fem, used through solver.py:392 and restated by
// models_copper.py:277-278,315): u_grad_q = sum_a u_a (x) dN_a(q);
// r_e[a,i] = sum_q P_q,ij dN_a,j JxW_q; K_e[a i, b k] = sum_q dN_a,j A_q[ij,kl] dN_b,l JxW_q.
#include <algorithm>
#include <type_traits>

#include "cp_internal.hpp"
#include "cp_points.hpp"

namespace cpfem {

// Sum of a 32-bit count over the 64 lanes of a wave (every lane takes part).
__device__ __forceinline__ uint32_t wave_count(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ void add_counts(unsigned long long* counts, uint32_t n_it, uint32_t n_ev) {
  if (!counts) return;
  n_it = wave_count(n_it);
  n_ev = wave_count(n_ev);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&counts[0], (unsigned long long)n_it);
    atomicAdd(&counts[1], (unsigned long long)n_ev);
  }
}

// ---------------------------------------------------------------------------------
// Quadrature-point kernels of the assembly.  k_element_res: H from dofs, local Newton,
// JxW-weighted P (SoA [9][Q]) and, for Jacobian assemblies, the converged stress (sout, [6][Q]);
// k_point_tangent then forms the JxW-weighted consistent tangent ([81][Q]: each of the 81
// stores of a wave writes 512 contiguous bytes) from it, re-evaluating the residual there.  Bound by FP64 VALU issue where the points fill the
// device, by the serial chain of one point's iterations where they do not: then L lanes share a
// point (point_lanes).
// The lanes of a wave run their Newton iterations in lockstep; a wave whose points need very
// different iteration counts would otherwise run until its slowest lane converges.  With
// parking (pk.lanes > 0), once at most pk.lanes lanes of the wave are still iterating, those
// store their point's iterate in the park queue and the wave finishes the others;
// k_element_qp_park completes the parked points.  The iterates, and so every output, are the
// same either way: a parked point resumes from its stored S' with the residual re-evaluated
// there.  counts (optional): [0] += local Newton iterations, [1] += residual evaluations (one
// atomic per wave), the measured inputs of the algorithmic flop count.
//
// Points that the crystal-frame form does not cover (Crystal::applies) take the general one, by the same lanes
// in a function of its own (cp_points.hpp).
template <int N, int L>
__device__ __attribute__((noinline)) void general_res(const Geom& G, const double* __restrict__ u, const StateView& sv,
                                                      const MatView& mv, const SlipTable<N>* table, const SolveCfg& cfg, int64_t q,
                                                      int sub, LdsDouble* sh, double* __restrict__ wP,
                                                      double* __restrict__ sout, int32_t* __restrict__ iters,
                                                      int32_t* __restrict__ status, uint32_t* n_it, uint32_t* n_ev) {
  PointIn in;
  in.load(G, u, sv, mv, q);
  double s[6], P[9];
  int32_t st = 0;
  ConstTable<N>& tab = uniform_table(table);
  Point<N, L, Crystal<N, L>::K> pt;
  CrystalRest<N, L> rest;
  setup_general<QBS>(pt, in, sv, q, sub, sh, rest);
  const int it = pt.solve(tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, s, &st);
  in.load(G, u, sv, mv, reread(q));
  pk1(pt, in.F, in.Fpi, s, P);
  const double w = jxw_at(G, q);
#pragma unroll
  for (int i = 0; i < 9; ++i)
    if (L == 1 || i % L == sub) wP[i * G.n_qp + q] = w * P[i];
  if (sout) {
#pragma unroll
    for (int j = 0; j < 6; ++j)
      if (L == 1 || j % L == sub) sout[j * G.n_qp + q] = s[j];
  }
  if (sub != 0) return;
  if (iters) iters[q] = it;
  if (st) atomicOr(status, st);
  *n_it = (uint32_t)it;
  *n_ev = (uint32_t)pt.nev;
}

// Outputs of a converged point: JxW P, the stress, iterations, status bits; each lane writes its
// share.
template <int N, int L>
__device__ __forceinline__ void finish_point(const Geom& G, int64_t q, int sub, const Crystal<N, L>& pt, const PointIn& in,
                                             const CrystalNewton<N, L>& nw, int32_t st, double* __restrict__ wP,
                                             double* __restrict__ sout, int32_t* __restrict__ iters,
                                             int32_t* __restrict__ status) {
  const double w = jxw_at(G, q);
  double P[9];
  crystal_pk1(pt, in.F, in.Fpi, in.R, nw.s, P);
#pragma unroll
  for (int i = 0; i < 9; ++i)
    if (L == 1 || i % L == sub) wP[i * G.n_qp + q] = w * P[i];
  if (sout) {
    double s[6];
    pt.stress(nw.s, in.R, s);
#pragma unroll
    for (int j = 0; j < 6; ++j)
      if (L == 1 || j % L == sub) sout[j * G.n_qp + q] = s[j];
  }
  if (sub == 0) {
    if (iters) iters[q] = nw.it;
    if (st) atomicOr(status, st);
  }
}

template <int N, int L>
__global__ void __launch_bounds__(QBS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_element_res(Geom G, const double* __restrict__ u, StateView sv, MatView mv, SlipSys<N> arg, const SlipTable<N>* __restrict__ gen,
              int crystal, SolveCfg cfg, double* __restrict__ wP, double* __restrict__ sout, int32_t* __restrict__ iters,
              int32_t* __restrict__ status, unsigned long long* __restrict__ counts, PointPark pk) {
  __shared__ double sh[lds_columns<N, L> * QBS];
  __shared__ SlipSys<L == 1 ? 3 : N> tabs;
  const SlipSys<N>& tab = slip_constants<N, L>(arg, reinterpret_cast<SlipSys<N>*>(&tabs));
  const int sub = L == 1 ? 0 : (int)(threadIdx.x % L);
  const int64_t q = (int64_t)blockIdx.x * (QBS / L) + threadIdx.x / L;
  const bool valid = q < G.n_qp;
  Crystal<N, L> pt;
  CrystalRest<N, L> rest;
  CrystalNewton<N, L> nw;
  int32_t st = 0;
  bool fits = false, act = false;
  pt.nev = 0;
  pt.nr = 0.0;
  nw.it = 0;
  nw.k = 0;
  nw.lost = false;
  if (valid) {
    PointIn in;
    in.load(G, u, sv, mv, q);
    fits = crystal && Crystal<N, L>::applies(in.R, in.m);
    if (fits) {
      setup_crystal(pt, in, sv, q, sub, sh, rest);
      act = nw.start(pt, cfg.tol);
    }
  }
  for (;;) {  // wave-uniform exits: every lane sees the same ballot
    const int nact = __popcll(__ballot(act));
    if (nact == 0 || nact <= pk.lanes) break;
    if (act) act = nw.advance(pt, tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, &st);
  }
  const unsigned long long park = __ballot(act && sub == 0);
  if (park) {  // park the points still iterating (one queue reservation per wave)
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll(park) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(&pk.ctr[0], (uint32_t)__popcll(park));
    base = __shfl(base, leader, 64);
    if (act && sub == 0) {
      const int64_t k = (int64_t)base + __popcll(park & ((1ull << lane) - 1ull));
      pk.idx[k] = (int32_t)q;
      pk.it[k] = nw.k ? nw.it - 1 : nw.it;  // a step whose length is still searched is formed again
#pragma unroll
      for (int j = 0; j < 6; ++j) pk.s[j * pk.cap + k] = nw.s[j];
    }
  }
  uint32_t n_it = 0, n_ev = fits && sub == 0 ? (uint32_t)pt.nev : 0u;
  if (fits) fits = !nw.lost;
  if (fits && !act) {
    PointIn in;
    in.load(G, u, sv, mv, reread(q));
    CrystalNewton<N, L>::finite(pt, &st);
    finish_point<N, L>(G, q, sub, pt, in, nw, st, wP, sout, iters, status);
    n_it = sub == 0 ? (uint32_t)nw.it : 0u;
  } else if (valid && !fits) {
    // (its residuals here are not counted twice)
    OutOfLine f{G, sv, mv, cfg};
    general_res<N, L>(f.G, u, f.sv, f.mv, gen, f.cfg, q, sub, (LdsDouble*)sh, wP, sout, iters, status, &f.n_it, &f.n_ev);
    n_it = f.n_it;
    n_ev = f.n_ev;
  }
  add_counts(counts, n_it, n_ev);
}

template <int N>
__device__ __attribute__((noinline)) void general_tangent(const Geom& G, const double* __restrict__ u, const StateView& sv,
                                                          const MatView& mv, const SlipTable<N>* table, int64_t q, LdsDouble* sh,
                                                          const double* __restrict__ sin, double* __restrict__ wA) {
  PointIn in;
  in.load(G, u, sv, mv, q);
  double s[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) s[j] = sin[j * G.n_qp + q];
  ConstTable<N>& tab = uniform_table(table);
  Point<N> pt;
  CrystalRest<N, 1, N> rest;
  setup_general<QBS>(pt, in, sv, q, 0, sh, rest);
  pt.eval(tab, s);
  const double w = jxw_at(G, q);
  tangent<N>(pt, tab, in.F, in.Fpi, s, [&](int m9, const double* dP) {
#pragma unroll
    for (int i = 0; i < 9; ++i) wA[(int64_t)(9 * i + m9) * G.n_qp + q] = w * dP[i];
  });
}

// Consistent tangent of every point from its converged stress (sin, [6][Q]).
template <int N>
__global__ void __launch_bounds__(QBS) k_point_tangent(Geom G, const double* __restrict__ u, StateView sv, MatView mv,
                                                      SlipSys<N> tab, const SlipTable<N>* __restrict__ gen, int crystal,
                                                      const double* __restrict__ sin, double* __restrict__ wA) {
  __shared__ double sh[2 * N * QBS];  // one wave per SIMD anyway
  const int64_t q = (int64_t)blockIdx.x * QBS + threadIdx.x;
  if (q >= G.n_qp) return;
  PointIn in;
  in.load(G, u, sv, mv, q);
  bool done = false;
  if (crystal && Crystal<N>::applies(in.R, in.m)) {
    double s[6], x[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) s[j] = sin[j * G.n_qp + q];
    Crystal<N>::pull_back(s, in.R, x);
    Crystal<N, 1, N> pt;
    CrystalRest<N, 1, N> rest;
    setup_crystal(pt, in, sv, q, 0, sh, rest);
    pt.eval(tab, x);
    const double w = jxw_at(G, q);
    done = crystal_tangent(pt, tab, in.F, in.Fpi, in.R, x, [&](int m9, const double* dP) {
#pragma unroll
      for (int i = 0; i < 9; ++i) wA[(int64_t)(9 * i + m9) * G.n_qp + q] = w * dP[i];
    });
  }
  if (!done) {
    const OutOfLine f{G, sv, mv, {}};
    general_tangent<N>(f.G, u, f.sv, f.mv, gen, q, (LdsDouble*)sh, sin, wA);
  }
}

// The parked points of k_element_res, one queue entry per point: each point's iterate is
// restored, its residual re-evaluated there and its Newton iterations continued to
// convergence.  The grid covers the longest possible queue; blocks past the queue's length
// (final when this kernel starts: k_element_res ran before it on the same stream) exit at once,
// so only as many blocks as parked points run, dispatched as earlier blocks retire.
template <int N, int L>
__global__ void __launch_bounds__(QBS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_element_qp_park(Geom G, const double* __restrict__ u, StateView sv, MatView mv, SlipSys<N> arg,
                  const SlipTable<N>* __restrict__ gen, SolveCfg cfg,
                  double* __restrict__ wP, double* __restrict__ sout, int32_t* __restrict__ iters, int32_t* __restrict__ status,
                  unsigned long long* __restrict__ counts, PointPark pk) {
  __shared__ double sh[lds_columns<N, L> * QBS];
  __shared__ SlipSys<L == 1 ? 3 : N> tabs;
  const uint32_t total = __hip_atomic_load(&pk.ctr[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((int64_t)blockIdx.x * (QBS / L) >= (int64_t)total) return;  // uniform over the block
  const SlipSys<N>& tab = slip_constants<N, L>(arg, reinterpret_cast<SlipSys<N>*>(&tabs));
  if (counts && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&counts[2], (unsigned long long)total);
  const int sub = L == 1 ? 0 : (int)(threadIdx.x % L);
  const int64_t k = (int64_t)blockIdx.x * (QBS / L) + threadIdx.x / L;
  uint32_t n_it = 0, n_ev = 0;
  if (k < (int64_t)total) {
    const int64_t q = pk.idx[k];
    PointIn in;
    Crystal<N, L> pt;
    CrystalRest<N, L> rest;
    CrystalNewton<N, L> nw;
    int32_t st = 0;
    in.load(G, u, sv, mv, q);
    setup_crystal(pt, in, sv, q, sub, sh, rest);
#pragma unroll
    for (int j = 0; j < 6; ++j) nw.s[j] = pk.s[j * pk.cap + k];
    nw.it = pk.it[k];
    bool act = nw.resume(pt, tab, cfg.tol);
    while (act) act = nw.advance(pt, tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, &st);
    if (nw.lost) {
      OutOfLine f{G, sv, mv, cfg};
      general_res<N, L>(f.G, u, f.sv, f.mv, gen, f.cfg, q, sub, (LdsDouble*)sh, wP, sout, iters, status, &f.n_it, &f.n_ev);
      n_it = f.n_it;
      n_ev = f.n_ev;
    } else {
      CrystalNewton<N, L>::finite(pt, &st);
      in.load(G, u, sv, mv, reread(q));
      finish_point<N, L>(G, q, sub, pt, in, nw, st, wP, sout, iters, status);
      if (sub == 0) {
        n_it = (uint32_t)nw.it;
        n_ev = (uint32_t)pt.nev;
      }
    }
  }
  add_counts(counts, n_it, n_ev);
}

// ---------------------------------------------------------------------------------
// Element stiffness / residual: one thread per (cell, local node a) and row index i; writes the 24
// values (b, k) of its row (KE[cell][a][i][b][k]) and r_e[cell][a][i].  A block takes 16 cells (128
// points, contiguous in the [component][Q] layouts) and one i, and stages their JxW P_ij and
// the 27 tangent components dP_(ij)/dH_(kl) in LDS with coalesced loads: each value is read
// once.  The rows leave through the same LDS, 192 contiguous bytes each.  The three i of a cell are
// blocks of the same XCD, which then finds the cells' gradients in its L2.
// Bound by memory (2.6 GB at 64^3).  64^3: 950 us; with the three i in one thread's 72 accumulators
// and 16-byte stores 576 bytes apart, 1550.  19x14x11 (183 blocks of that kind): 24 us, 52.
constexpr int EK_CELLS = 16;
constexpr int EK_BS = 8 * EK_CELLS;  // threads = points per block
constexpr int EK_PITCH = 25;         // doubles between the rows in LDS
constexpr int XCDS = 8;

template <bool UNIFORM>
__global__ void __launch_bounds__(EK_BS) k_element_K(Geom G, const double* __restrict__ wP, const double* __restrict__ wA,
                                                    double* __restrict__ KE, double* __restrict__ RE) {
  static_assert(EK_PITCH * EK_BS <= 27 * EK_BS, "the rows use the tangents' LDS");
  __shared__ double sP[3][EK_BS];
  __shared__ double sA[27 * EK_BS];
  __shared__ double sG[UNIFORM ? 192 : 1];
  const int i = (int)(blockIdx.x / XCDS) % 3;
  const int64_t q0 = ((int64_t)(blockIdx.x / (3 * XCDS)) * XCDS + blockIdx.x % XCDS) * EK_BS;  // first point of the block
  const int tid = threadIdx.x;
  const int64_t t = q0 + tid;  // (cell, a) of this thread
  const bool valid = t < G.n_qp;
  const int64_t cell = t >> 3;
  const int a = tid & 7;
  const int cl = tid >> 3;  // cell within the block
#pragma unroll
  for (int j = 0; j < 3; ++j) sP[j][tid] = valid ? wP[(3 * i + j) * G.n_qp + t] : 0.0;
#pragma unroll
  for (int c = 0; c < 27; ++c) sA[c * EK_BS + tid] = valid ? wA[(int64_t)(27 * i + c) * G.n_qp + t] : 0.0;
  if (UNIFORM)
    for (int e = tid; e < 192; e += EK_BS) sG[e] = G.sg[e];
  __syncthreads();
  double K[24], re = 0.0;
#pragma unroll
  for (int k = 0; k < 24; ++k) K[k] = 0.0;
  if (valid) {
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
      const int p = 8 * cl + q;
      const int64_t qp = cell * 8 + q;
      double ga[3], gb[24];
#pragma unroll
      for (int c = 0; c < 24; ++c) gb[c] = UNIFORM ? G.sg[c * 8 + q] : G.sg[c * G.n_qp + qp];
#pragma unroll
      for (int j = 0; j < 3; ++j) ga[j] = UNIFORM ? sG[(3 * a + j) * 8 + q] : G.sg[(3 * a + j) * G.n_qp + qp];
      double sr = 0.0;
#pragma unroll
      for (int j = 0; j < 3; ++j) sr += sP[j][p] * ga[j];
      re += sr;
      double Z[9];  // Z[k][l] = sum_j ga_j A[(i j),(k l)]
#pragma unroll
      for (int kl = 0; kl < 9; ++kl) {
        double z = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) z += ga[j] * sA[(9 * j + kl) * EK_BS + p];
        Z[kl] = z;
      }
#pragma unroll
      for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int k = 0; k < 3; ++k) K[b * 3 + k] += Z[3 * k] * gb[3 * b] + Z[3 * k + 1] * gb[3 * b + 1] + Z[3 * k + 2] * gb[3 * b + 2];
    }
    RE[t * 3 + i] = re;
  }
  __syncthreads();  // the tangents have been read
#pragma unroll
  for (int k = 0; k < 24; ++k) sA[tid * EK_PITCH + k] = K[k];
  __syncthreads();
  const int n = (int)std::max<int64_t>(0, std::min<int64_t>(EK_BS, G.n_qp - q0)) * 12;
#pragma unroll
  for (int m = 0; m < 12; ++m) {
    const int e = tid + m * EK_BS, r = e / 12, c = 2 * (e % 12);
    if (e < n)
      *reinterpret_cast<double2*>(KE + ((q0 + r) * 3 + i) * 24 + c) = make_double2(sA[r * EK_PITCH + c], sA[r * EK_PITCH + c + 1]);
  }
}

// ---------------------------------------------------------------------------------
// Block-ELL gather.  A block takes 16 nodes and sums, in ascending cell order (the order in which
// scipy's COO->CSR sum_duplicates adds them, solver.py:281-282), the rows of the element matrices
// at each node into an LDS tile of 27 slots (in turns where a pattern has more); a node's rows in one
// cell are 576 contiguous bytes.  24 lanes (b, c) take a node, two nodes a wave; slots: the slot of
// node b in the row of node a, per (cell, a, b), and above it (GATHER_RANK) the number of earlier b
// of the same cell with the same node (degenerate cells only, ranks > 1), which take turns.
// The tile leaves with the row elimination of get_A (solver.py:290-293): a Dirichlet row becomes zero
// with a unit diagonal.
// Bound by memory (1.2 GB of element matrices read, 0.53 GB written at 64^3): 565 us; with a thread per
// (slot, row), whose reads of 72 bytes use their lines about half, 620.
constexpr int GN = 16, GBS = 32 * GN, GPITCH = 3 * GN + 1;
__global__ void __launch_bounds__(GBS) k_gather_matrix(BellView M, const double* __restrict__ KE, const int32_t* __restrict__ nptr,
                                                      const int32_t* __restrict__ nlist, const uint32_t* __restrict__ slots, int ranks,
                                                      const int32_t* __restrict__ dslot, const uint8_t* __restrict__ is_bc,
                                                      double* __restrict__ vals) {
  __shared__ double T[81 * GPITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t node0 = (int64_t)blockIdx.x * GN, nrow = 3 * M.n_nodes;
  const int half = lane / 24, j = lane - 24 * half, b = j / 3, c = j - 3 * b;
  for (int s0 = 0; s0 < M.n_slots; s0 += 27) {
    for (int e = tid; e < 81 * GPITCH; e += GBS) T[e] = 0.0;
    __syncthreads();
    const int nl = 2 * wave + half;
    const int64_t i = node0 + nl;
    if (half < 2 && i < M.n_nodes) {
      const int e1 = nptr[i + 1];
      for (int e0 = nptr[i]; e0 < e1; e0 += 8) {
        double v[8][3];
        int sl[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          sl[m] = -1;
          if (e0 + m < e1) {
            const int64_t ca = nlist[e0 + m];
            const double* src = KE + (ca * 3 + c) * 24 + 3 * b;
            sl[m] = (int)slots[ca * 8 + b];
            v[m][0] = src[0];
            v[m][1] = src[1];
            v[m][2] = src[2];
          }
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const int s = (sl[m] & (GATHER_RANK - 1)) - s0;
          for (int r = 0; r < ranks; ++r) {
            if (sl[m] >= 0 && sl[m] / GATHER_RANK == r && s >= 0 && s < 27) {
              double* d = T + 3 * s * GPITCH + 3 * nl + c;
              d[0] += v[m][0];
              d[GPITCH] += v[m][1];
              d[2 * GPITCH] += v[m][2];
            }
            asm volatile("" ::: "memory");  // another lane may add to the same entry next: LDS keeps a wave's order
          }
        }
      }
    }
    __syncthreads();
    const int rows = 3 * min(27, M.n_slots - s0);
    for (int e = tid; e < rows * 3 * GN; e += GBS) {
      const int row = e / (3 * GN), col = e - row * (3 * GN);
      const int64_t r = 3 * node0 + col;
      if (r >= nrow) continue;
      double v = T[row * GPITCH + col];
      if (is_bc[r]) v = s0 + row / 3 == dslot[node0 + col / 3] && row % 3 == col % 3 ? 1.0 : 0.0;
      vals[(3 * (int64_t)s0 + row) * nrow + r] = v;
    }
    __syncthreads();  // before the tile is cleared for the next slots
  }
}

// Residual gather + apply_bc_vec (solver.py:119-133): res[bc] = u[bc] - ubar.
// Also writes per-block partial sums of res^2 (deterministic reduction finished on device).
__global__ void __launch_bounds__(256) k_gather_residual(int64_t n_nodes, const double* __restrict__ RE,
                                                        const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist,
                                                        const uint8_t* __restrict__ is_bc, const double* __restrict__ ubar,
                                                        const double* __restrict__ u, double* __restrict__ res) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= 3 * n_nodes) return;
  const int64_t i = r / 3;
  const int c = (int)(r - 3 * i);
  double v = 0.0;
  if (is_bc[r]) {
    v = u[r] - ubar[r];
  } else {
    for (int64_t e = nptr[i]; e < nptr[i + 1]; ++e) v += RE[(int64_t)nlist[e] * 3 + c];
  }
  res[r] = v;
}

// Element residual only: thread per (cell, a)
// A block stages the JxW P of its 128 points in LDS with coalesced loads (read from memory by each
// of a cell's eight threads, eight lines per load: 33 us at 40^3, now 14).
template <bool UNIFORM>
__global__ void __launch_bounds__(EK_BS) k_element_R(Geom G, const double* __restrict__ wP, double* __restrict__ RE) {
  __shared__ double sP[9][EK_BS];
  __shared__ double sG[UNIFORM ? 192 : 1];
  const int tid = threadIdx.x, a = tid & 7, cl = tid >> 3;
  const int64_t t = (int64_t)blockIdx.x * EK_BS + tid, cell = t >> 3;
  const bool valid = t < G.n_qp;
#pragma unroll
  for (int c = 0; c < 9; ++c) sP[c][tid] = valid ? wP[c * G.n_qp + t] : 0.0;
  if (UNIFORM)
    for (int e = tid; e < 192; e += EK_BS) sG[e] = G.sg[e];
  __syncthreads();
  if (!valid) return;
  double re[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
  for (int q = 0; q < 8; ++q) {
    const int p = 8 * cl + q;
    double ga[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) ga[j] = UNIFORM ? sG[(3 * a + j) * 8 + q] : G.sg[(3 * a + j) * G.n_qp + cell * 8 + q];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double sr = 0.0;  // the sum of k_element_K, to the bit
#pragma unroll
      for (int j = 0; j < 3; ++j) sr += sP[3 * i + j][p] * ga[j];
      re[i] += sr;
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) RE[t * 3 + i] = re[i];
}

// ---------------------------------------------------------------------------------
// Point-level update (tensor_map / update_int_vars_map, models_copper.py:263-269) on explicit
// u_grad arrays [9][Q] (or from dofs when Hd == nullptr).  Any output pointer may be null.
struct LocalOut {
  double *P, *A, *sig;
  StateOut so;
  int32_t *iters, *status;
};

__device__ __forceinline__ void load_local(PointIn& in, const double* __restrict__ Hd, int64_t n_qp, const Geom& G,
                                           const double* __restrict__ u, const StateView& sv, const MatView& mv, int64_t q) {
  if (Hd) {
    double H[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) H[i] = Hd[i * n_qp + q];
    in.load(H, sv, mv, q);
  } else {
    in.load(G, u, sv, mv, q);
  }
}

template <int N, bool TANGENT, int L>
__device__ __attribute__((noinline)) void general_local(int64_t n_qp, const double* __restrict__ Hd, const Geom& G,
                                                        const double* __restrict__ u, const StateView& sv, const MatView& mv,
                                                        const SlipTable<N>* table, const SolveCfg& cfg, int self_block, int64_t q,
                                                        int sub, LdsDouble* sh, const LocalOut& o) {
  PointIn in;
  load_local(in, Hd, n_qp, G, u, sv, mv, q);
  double s[6], P[9];
  int32_t st = 0;
  ConstTable<N>& tab = uniform_table(table);
  Point<N, L, Crystal<N, L>::K> pt;
  CrystalRest<N, L> rest;
  setup_general<QBS>(pt, in, sv, q, sub, sh, rest);
  const int it = pt.solve(tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, s, &st);
  load_local(in, Hd, n_qp, G, u, sv, mv, reread(q));
  pk1(pt, in.F, in.Fpi, s, P);
  if constexpr (TANGENT) {
    if (o.A) {
      tangent<N>(pt, tab, in.F, in.Fpi, s, [&](int m9, const double* dP) {
#pragma unroll
        for (int i = 0; i < 9; ++i) o.A[(9 * i + m9) * n_qp + q] = dP[i];
      });
    }
  }
  if (o.P) {
#pragma unroll
    for (int i = 0; i < 9; ++i)
      if (L == 1 || i % L == sub) o.P[i * n_qp + q] = P[i];
  }
  if (o.sig) {
    double sg[9];
    mm3t(P, in.F, sg);
    const double idF = 1.0 / det3(in.F);
#pragma unroll
    for (int i = 0; i < 9; ++i)
      if (L == 1 || i % L == sub) o.sig[i * n_qp + q] = sg[i] * idF;
  }
  if (o.so.Fpi) {
    double Fn[9], Sc[9];
    fp_inv_new(in.Fpi, in.R, pt.Lpc, Fn);
#pragma unroll
    for (int i = 0; i < 9; ++i)
      if (L == 1 || i % L == sub) o.so.Fpi[i * sv.ld + q] = Fn[i];
    pt.crystal_stress(s, Sc);
    point_history<N, L>(pt, tab, Sc, in.m, self_block, sv.g + q, sv.slip + q, sv.ld, o.so.g + q, o.so.slip + q);
  }
  if (sub != 0) return;
  if (o.iters) o.iters[q] = it;
  if (st) atomicOr(o.status, st);
}

template <int N, bool TANGENT, int L>
__global__ void __launch_bounds__(QBS) __attribute__((amdgpu_waves_per_eu(TANGENT ? 1 : 2, TANGENT ? 1 : 2)))
k_local(int64_t n_qp, const double* __restrict__ Hd, Geom G, const double* __restrict__ u, StateView sv, MatView mv, SlipSys<N> arg,
        const SlipTable<N>* __restrict__ gen, int crystal, SolveCfg cfg, int self_block, LocalOut o) {
  __shared__ double sh[lds_columns<N, L> * QBS];
  __shared__ SlipSys<L == 1 ? 3 : N> tabs;
  const SlipSys<N>& tab = slip_constants<N, L>(arg, reinterpret_cast<SlipSys<N>*>(&tabs));
  const int sub = L == 1 ? 0 : (int)(threadIdx.x % L);
  const int64_t q = (int64_t)blockIdx.x * (QBS / L) + threadIdx.x / L;
  if (q >= n_qp) return;
  PointIn in;
  load_local(in, Hd, n_qp, G, u, sv, mv, q);
  Crystal<N, L> pt;
  CrystalRest<N, L> rest;
  CrystalNewton<N, L> nw;
  int32_t st = 0;
  bool fits = crystal && Crystal<N, L>::applies(in.R, in.m);
  if (fits) {
    setup_crystal(pt, in, sv, q, sub, sh, rest);
    fits = nw.solve(pt, tab, cfg.tol, cfg.max_sub_step, cfg.max_iter, &st);
  }
  if (fits) load_local(in, Hd, n_qp, G, u, sv, mv, reread(q));
  if (TANGENT && fits && o.A) {  // a separate instantiation: the tangent's registers cost the others occupancy
    // The point is set up again at its S' and read again behind the tangent: with the Newton's state and the
    // inputs kept through it, 420 registers spilled.  Us a call, 262,144 points, elastic / plastic (8.6 and
    // 4.5 iterations): FCC 242 / 648, now 140 / 493; BCC24 301 / 588, now 217 / 487.
    setup_crystal(pt, in, sv, reread(q), sub, sh, rest);
    pt.eval(tab, nw.s);
    fits = crystal_tangent(pt, tab, in.F, in.Fpi, in.R, nw.s, [&](int m9, const double* dP) {
#pragma unroll
      for (int i = 0; i < 9; ++i) o.A[(9 * i + m9) * n_qp + q] = dP[i];
    });
    load_local(in, Hd, n_qp, G, u, sv, mv, reread(q));
  }
  if (!fits) {
    const OutOfLine f{G, sv, mv, cfg};
    const LocalOut out = o;
    general_local<N, TANGENT, L>(n_qp, Hd, f.G, u, f.sv, f.mv, gen, f.cfg, self_block, q, sub, (LdsDouble*)sh, out);
    return;
  }
  // every lane of a point writes its share of the components
  if (o.P || o.sig) {
    double P[9];
    crystal_pk1(pt, in.F, in.Fpi, in.R, nw.s, P);
    if (o.P) {
#pragma unroll
      for (int i = 0; i < 9; ++i)
        if (L == 1 || i % L == sub) o.P[i * n_qp + q] = P[i];
    }
    if (o.sig) {  // sigma = P F^T / det F (compute_avg_stress, models_copper.py:308-313)
      double sg[9];
      mm3t(P, in.F, sg);
      const double idF = 1.0 / det3(in.F);
#pragma unroll
      for (int i = 0; i < 9; ++i)
        if (L == 1 || i % L == sub) o.sig[i * n_qp + q] = sg[i] * idF;
    }
  }
  if (o.so.Fpi) {  // update_int_vars (models_copper.py:164-169,186-187)
    double Fn[9];
    fp_inv_new(in.Fpi, in.R, pt.Lpc, Fn);
#pragma unroll
    for (int i = 0; i < 9; ++i)
      if (L == 1 || i % L == sub) o.so.Fpi[i * sv.ld + q] = Fn[i];
    point_history<N, L>(pt, tab, nw.s, in.m, self_block, sv.g + q, sv.slip + q, sv.ld, o.so.g + q, o.so.slip + q);
  }
  if (sub == 0) {
    if (o.iters) o.iters[q] = nw.it;
    if (st) atomicOr(o.status, st);
  }
}

// Cell average of sigma with JxW weights (models_copper.py:315)
__global__ void k_cell_average(Geom G, const double* __restrict__ sig, double* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= G.n_cells * 9) return;
  const int64_t cell = t / 9;
  const int comp = (int)(t - cell * 9);
  double num = 0.0, den = 0.0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const double w = jxw_at(G, cell * 8 + q);
    num += sig[comp * G.n_qp + cell * 8 + q] * w;
    den += w;
  }
  out[cell * 9 + comp] = num / den;
}

// x0 of linear_incremental_solver (solver.py:221-227): ubar - u on Dirichlet dofs, 0 elsewhere
__global__ void k_bc_x0(int64_t n, const uint8_t* __restrict__ is_bc, const double* __restrict__ ubar,
                        const double* __restrict__ u, double* __restrict__ x0) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x0[i] = is_bc[i] ? ubar[i] - u[i] : 0.0;
}

// ---------------------------------------------------------------------------------
// Launch helpers (host)

// Lanes per point: one where the points fill the device (two waves per SIMD hold 131,072 lanes),
// more where a launch would otherwise be one point's serial chain of iterations in a few waves.
// Residual calls, us (FCC / BCC24), with 1, 2, 4 and 8 lanes: 4,096 points 119, 95, 67, - / 200, 150,
// 108, 81; 13,824 points 109, 95, 92, - / 186, 157, 143, 123; 32,768 points 112, 119, 102, - / 190,
// 201, 158, 180; 64,000 points 153, 133, 174, - / 260, 214, 249, 280; 110,592 points 161, 208, 241, -
// / 270, 340, 374, 451.
int point_lanes(int n_slip, int64_t n_qp) {
  if (n_qp > SHARED_POINTS) return 1;
  if (n_qp > 48000) return 2;
  return n_slip == 24 && n_qp <= 20000 ? 8 : 4;
}

template <int N>
void launch_element_qp(const Geom& G, const double* u, const StateView& sv, const MatView& mv, const PointTables<N>& tb,
                       const SolveCfg& cfg, double* wP, double* sout, int32_t* iters, int32_t* status,
                       unsigned long long* counts, const PointPark& park, hipStream_t st) {
  const int L = point_lanes(N, G.n_qp);
  const dim3 grid((unsigned)((G.n_qp * L + QBS - 1) / QBS)), block(QBS);
  const auto go = [&](auto lanes) {
    hipLaunchKernelGGL((k_element_res<N, decltype(lanes)::value>), grid, block, 0, st, G, u, sv, mv, tb.sys, tb.gen, tb.crystal, cfg,
                       wP, sout, iters, status, counts, park);
  };
  if (L == 1) go(std::integral_constant<int, 1>{});
  if (L == 2) go(std::integral_constant<int, 2>{});
  if (L == 4) go(std::integral_constant<int, 4>{});
  if constexpr (N == 24) {
    if (L == 8) go(std::integral_constant<int, 8>{});
  }
}

template <int N>
void launch_element_qp_park(const Geom& G, const double* u, const StateView& sv, const MatView& mv, const PointTables<N>& tb,
                            const SolveCfg& cfg, double* wP, double* sout, int32_t* iters, int32_t* status,
                            unsigned long long* counts, const PointPark& park, hipStream_t st) {
  const int L = point_lanes(N, G.n_qp);
  const dim3 grid((unsigned)((park.cap * L + QBS - 1) / QBS)), block(QBS);
  const auto go = [&](auto lanes) {
    hipLaunchKernelGGL((k_element_qp_park<N, decltype(lanes)::value>), grid, block, 0, st, G, u, sv, mv, tb.sys, tb.gen, cfg, wP, sout,
                       iters, status, counts, park);
  };
  if (L == 1) go(std::integral_constant<int, 1>{});
  if (L == 2) go(std::integral_constant<int, 2>{});
  if (L == 4) go(std::integral_constant<int, 4>{});
  if constexpr (N == 24) {
    if (L == 8) go(std::integral_constant<int, 8>{});
  }
}

template <int N>
void launch_point_tangent(const Geom& G, const double* u, const StateView& sv, const MatView& mv, const PointTables<N>& tb,
                          const double* sin, double* wA, hipStream_t st) {
  const int64_t nb = (G.n_qp + QBS - 1) / QBS;
  hipLaunchKernelGGL(k_point_tangent<N>, dim3((unsigned)nb), dim3(QBS), 0, st, G, u, sv, mv, tb.sys, tb.gen, tb.crystal, sin, wA);
}

template <int N>
void launch_local(int64_t n_qp, const double* Hd, const Geom& G, const double* u, const StateView& sv, const MatView& mv,
                  const PointTables<N>& tb, const SolveCfg& cfg, int self_block, double* P, double* A, double* sig,
                  const StateOut& so, int32_t* iters, int32_t* status, hipStream_t st) {
  const int L = A ? 1 : point_lanes(N, n_qp);
  const dim3 grid((unsigned)((n_qp * L + QBS - 1) / QBS)), block(QBS);
  const auto go = [&](auto tangent, auto lanes) {
    hipLaunchKernelGGL((k_local<N, decltype(tangent)::value, decltype(lanes)::value>), grid, block, 0, st, n_qp, Hd, G, u, sv, mv,
                       tb.sys, tb.gen, tb.crystal, cfg, self_block, LocalOut{P, A, sig, so, iters, status});
  };
  if (A) {
    go(std::true_type{}, std::integral_constant<int, 1>{});
    return;
  }
  if (L == 1) go(std::false_type{}, std::integral_constant<int, 1>{});
  if (L == 2) go(std::false_type{}, std::integral_constant<int, 2>{});
  if (L == 4) go(std::false_type{}, std::integral_constant<int, 4>{});
  if constexpr (N == 24) {
    if (L == 8) go(std::false_type{}, std::integral_constant<int, 8>{});
  }
}

void launch_element_K(const Geom& G, const double* wP, const double* wA, double* KE, double* RE, hipStream_t st) {
  if (wA)
    hipLaunchKernelGGL(G.uniform ? k_element_K<true> : k_element_K<false>,
                       dim3((unsigned)((G.n_qp + XCDS * EK_BS - 1) / (XCDS * EK_BS) * 3 * XCDS)), dim3(EK_BS), 0, st, G, wP, wA, KE, RE);
  else
    hipLaunchKernelGGL(G.uniform ? k_element_R<true> : k_element_R<false>, dim3((unsigned)((G.n_qp + EK_BS - 1) / EK_BS)), dim3(EK_BS),
                       0, st, G, wP, RE);
}

void launch_gather_matrix(const BellView& M, const double* KE, const int32_t* nptr, const int32_t* nlist, const uint32_t* slots,
                          int ranks, const int32_t* dslot, const uint8_t* is_bc, double* vals, hipStream_t st) {
  hipLaunchKernelGGL(k_gather_matrix, dim3((unsigned)((M.n_nodes + GN - 1) / GN)), dim3(GBS), 0, st, M, KE, nptr, nlist, slots, ranks,
                     dslot, is_bc, vals);
}

void launch_gather_residual(int64_t n_nodes, const double* RE, const int32_t* nptr, const int32_t* nlist, const uint8_t* is_bc,
                            const double* ubar, const double* u, double* res, hipStream_t st) {
  const int bs = 256;
  const int64_t n = 3 * n_nodes;
  hipLaunchKernelGGL(k_gather_residual, dim3((unsigned)((n + bs - 1) / bs)), dim3(bs), 0, st, n_nodes, RE, nptr, nlist, is_bc,
                     ubar, u, res);
}

void launch_bc_x0(int64_t n, const uint8_t* is_bc, const double* ubar, const double* u, double* x0, hipStream_t st) {
  hipLaunchKernelGGL(k_bc_x0, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, is_bc, ubar, u, x0);
}

__global__ void k_zero_words(uint32_t* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

void launch_zero_words(uint32_t* p, int64_t n, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
}

void launch_cell_average(const Geom& G, const double* sig, double* out, hipStream_t st) {
  const int bs = 256;
  const int64_t n = G.n_cells * 9;
  hipLaunchKernelGGL(k_cell_average, dim3((unsigned)((n + bs - 1) / bs)), dim3(bs), 0, st, G, sig, out);
}

#define CPFEM_INST(N)                                                                                                      \
  template void launch_element_qp<N>(const Geom&, const double*, const StateView&, const MatView&, const PointTables<N>&,  \
                                     const SolveCfg&, double*, double*, int32_t*, int32_t*, unsigned long long*,           \
                                     const PointPark&, hipStream_t);                                              \
  template void launch_element_qp_park<N>(const Geom&, const double*, const StateView&, const MatView&,                    \
                                          const PointTables<N>&, const SolveCfg&, double*, double*, int32_t*, int32_t*,    \
                                          unsigned long long*, const PointPark&, hipStream_t);                    \
  template void launch_point_tangent<N>(const Geom&, const double*, const StateView&, const MatView&,                      \
                                        const PointTables<N>&, const double*, double*, hipStream_t);              \
  template void launch_local<N>(int64_t, const double*, const Geom&, const double*, const StateView&, const MatView&,      \
                                const PointTables<N>&, const SolveCfg&, int, double*, double*, double*, const StateOut&,   \
                                int32_t*, int32_t*, hipStream_t);
CPFEM_INST(12)
CPFEM_INST(24)

}  // namespace cpfem
