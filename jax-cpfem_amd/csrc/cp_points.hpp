// What the kernels over quadrature points share: a point's inputs, the slip-system constants and
// the set-up of its local Newton.
#pragma once
#include "cp_internal.hpp"

namespace cpfem {

__device__ __forceinline__ PointMat load_mat(const MatView& mv, int64_t q) {
  PointMat m;
  m.p = 1.0 / mv.ptr[MP_XM][q * mv.stride[MP_XM]];
  m.c = mv.ao * mv.dt;
  m.gss_a = mv.ptr[MP_GSS_A][q * mv.stride[MP_GSS_A]];
  m.h = mv.ptr[MP_H][q * mv.stride[MP_H]];
  m.tsat = mv.ptr[MP_TSAT][q * mv.stride[MP_TSAT]];
  m.r = mv.ptr[MP_R][q * mv.stride[MP_R]];
  m.C11 = mv.ptr[MP_C11][q * mv.stride[MP_C11]];
  m.C12 = mv.ptr[MP_C12][q * mv.stride[MP_C12]];
  m.C44 = mv.ptr[MP_C44][q * mv.stride[MP_C44]];
  return m;
}

__device__ __forceinline__ double sg_at(const Geom& G, int comp, int64_t qp) {
  return G.uniform ? G.sg[comp * 8 + (qp & 7)] : G.sg[comp * G.n_qp + qp];
}
__device__ __forceinline__ double jxw_at(const Geom& G, int64_t qp) { return G.uniform ? G.jxw[qp & 7] : G.jxw[qp]; }

// u_grad at quadrature point qp from the nodal solution (AoS dofs, 3 per node)
__device__ __forceinline__ void ugrad_from_dofs(const Geom& G, const double* __restrict__ u, int64_t qp, double* H) {
  const int64_t cell = qp >> 3;
#pragma unroll
  for (int i = 0; i < 9; ++i) H[i] = 0.0;
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const int64_t nd = G.cells[cell * 8 + a];
    const double g0 = sg_at(G, 3 * a, qp), g1 = sg_at(G, 3 * a + 1, qp), g2 = sg_at(G, 3 * a + 2, qp);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double ui = u[3 * nd + i];
      H[3 * i] += ui * g0;
      H[3 * i + 1] += ui * g1;
      H[3 * i + 2] += ui * g2;
    }
  }
}

__device__ __forceinline__ void load_point(const StateView& sv, int64_t q, double* Fpi, double* R) {
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    Fpi[i] = sv.Fpi[i * sv.ld + q];
    R[i] = sv.rot[i * sv.ld + q];
  }
}

constexpr int QBS = 128;  // threads per block of the point kernels

// Point q's inputs: F = I + u_grad, Fp_inv_old, R and the constants.
struct PointIn {
  double F[9], Fpi[9], R[9];
  PointMat m;
  __device__ __forceinline__ void load(const double* H, const StateView& sv, const MatView& mv, int64_t q) {
#pragma unroll
    for (int i = 0; i < 9; ++i) F[i] = H[i] + ((i % 4) == 0 ? 1.0 : 0.0);
    load_point(sv, q, Fpi, R);
    m = load_mat(mv, q);
  }
  __device__ __forceinline__ void load(const Geom& G, const double* __restrict__ u, const StateView& sv, const MatView& mv,
                                       int64_t q) {
    double H[9];
    ugrad_from_dofs(G, u, q, H);
    load(H, sv, mv, q);
  }
};

// The same index, opaque to the compiler: inputs read again behind it are not kept in registers
// across the Newton iterations.
__device__ __forceinline__ int64_t reread(int64_t q) {
  int lo = (int)q, hi = (int)(q >> 32);
  asm volatile("" : "+v"(lo), "+v"(hi));
  return ((int64_t)hi << 32) | (uint32_t)lo;
}

// The slip-system constants of a point kernel: its argument where a lane does a whole point (the
// same system in every lane: scalar loads), a copy in LDS where the lanes of a point take
// different systems.
template <int N, int L, int BS = QBS>
__device__ __forceinline__ const SlipSys<N>& slip_constants(const SlipSys<N>& arg, SlipSys<N>* lds) {
  if constexpr (L == 1) {
    return arg;
  } else {
    const double* src = reinterpret_cast<const double*>(&arg);
    double* dst = reinterpret_cast<double*>(lds);
    for (int i = threadIdx.x; i < (int)(sizeof(SlipSys<N>) / sizeof(double)); i += BS) dst[i] = src[i];
    __syncthreads();
    return *lds;
  }
}

// LDS doubles per lane of a point kernel, and the set-up of point q's crystal-frame form in the
// lane's column: d dgamma / d tau and |1/g_old| behind it, what LDS does not hold in private memory
// (whose address escapes, or the compiler would index it in registers).
template <int N, int L>
constexpr int lds_columns = Crystal<N, L>::M + Crystal<N, L>::K;
template <int N, int L, int KS = Crystal<N, L>::K>
struct CrystalRest {
  static constexpr int n = N / L - KS;
  double gi[n > 0 ? n : 1];
};
template <int BS = QBS, int N, int L, int KS>
__device__ __forceinline__ void setup_crystal(Crystal<N, L, KS>& pt, const PointIn& in, const StateView& sv, int64_t q, int sub,
                                              double* sh, CrystalRest<N, L, KS>& rest) {
  if (rest.n > 0) asm volatile("" ::"v"(rest.gi) : "memory");
  pt.setup(in.F, in.Fpi, in.R, sv.g + q, sv.ld, in.m, sh + threadIdx.x, sh + Crystal<N, L>::M * BS + threadIdx.x, BS, BS, sub,
           rest.gi);
}

// Kernel arguments that go to a function out of line by reference, copied in the branch that calls it:
// the arguments themselves would be stored to every lane's private memory at the kernel's start
// (0.5 GB a launch at 64^3).
struct OutOfLine {
  Geom G;
  StateView sv;
  MatView mv;
  SolveCfg cfg;
  uint32_t n_it = 0, n_ev = 0;
};

// The general form (cp_point.hpp) runs in functions out of line, so that its registers do not weigh on the
// points of the crystal-frame form; the lanes of a point and their LDS columns are the same.  What crosses
// the call keeps its address space, or every access would be a flat one: the columns are an LDS pointer, the
// slip table one to constant memory, the same in every lane (scalar loads where a lane does a whole point).
// Batches whose every R is a rotation to 32 bits only, and so of this form, us per call (the crystal-frame
// form's call; one lane of each point at work, gp and 1/g_old in private memory, flat accesses): stress map of 4,096
// FCC points 101 (82; 251), residual 8^3 98 (61; 249), 16^3 BCC24 135 (86; 292), 40^3 BCC24 748 (378; 1076),
// assembly 64^3 BCC24 8,680 (5,510; 11,990), stress and history 32^3 842 (510; 1143).
typedef __attribute__((address_space(3))) double LdsDouble;
template <int N>
using ConstTable = const __attribute__((address_space(4))) SlipTable<N>;

template <int N>
__device__ __forceinline__ ConstTable<N>& uniform_table(const SlipTable<N>* table) {
  const uint64_t t = (uint64_t)table;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)t), hi = __builtin_amdgcn_readfirstlane((uint32_t)(t >> 32));
  return *(ConstTable<N>*)((uint64_t)hi << 32 | lo);
}
// (rest: no member of the point, whose registers it would drag into memory)
template <int BS, int N, int L, int KS>
__device__ __forceinline__ void setup_general(Point<N, L, KS>& pt, const PointIn& in, const StateView& sv, int64_t q, int sub,
                                              LdsDouble* sh, CrystalRest<N, L, KS>& rest) {
  if (rest.n > 0) asm volatile("" ::"v"(rest.gi) : "memory");
  pt.setup(in.F, in.Fpi, in.R, sv.g + q, sv.ld, in.m, (double*)sh + threadIdx.x, (double*)sh + Point<N, L, KS>::M * BS + threadIdx.x,
           BS, BS, sub, rest.n > 0 ? rest.gi : nullptr);
}

}  // namespace cpfem
