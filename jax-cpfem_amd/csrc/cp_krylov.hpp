// Device helpers shared by the Krylov kernels and the multigrid preconditioner: wave and block
// sums in a fixed order, partial sums of a grid, XCD-local block order, and the one-row-per-thread
// product with the block-ELL matrix.
#pragma once
#include "cp_internal.hpp"

namespace cpfem {

constexpr int KBS = 256;
constexpr int KMAXB = 512;  // blocks of the BiCGSTAB kernels (grid-stride beyond)

// PS_RS and PS_RT (<rhat,s>, <rhat,t>: the one-operand recurrence) share PS_BB's slot
// (<b,b>, read once by k_kinit2) and the last one.
enum { PS_RR = 0, PS_RHR, PS_RQ, PS_SS, PS_TS, PS_TT, PS_BB, PS_RT, PS_COUNT };
constexpr int PS_RS = PS_BB;

// One DPP step on a double: the value of the lane selected by CTRL (0 where the source is
// out of range or the row is masked off).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_from(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROW_MASK, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over the 64 lanes of a wave, returned in every lane.  DPP row shifts 1, 2, 4, 8 leave
// each 16-lane row's sum in its lane 15, row broadcasts 15 and 31 carry those into lane 63;
// the order of the additions is fixed, so every wave that sums the same values gets the
// bitwise-same result.
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_from<0x111, 0xf>(v);  // row_shr:1
  v += dpp_from<0x112, 0xf>(v);  // row_shr:2
  v += dpp_from<0x114, 0xf>(v);  // row_shr:4
  v += dpp_from<0x118, 0xf>(v);  // row_shr:8
  v += dpp_from<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_from<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Writes this block's NSL sums into entry `own` (a permutation of the block index over the
// grid; the block index by default) of their slots; a grid smaller than the stride ps also
// clears the entries no block of it owns, so every consumer sums exactly ps values.  sh: NSL
// doubles per wave of the block.
template <int BS, int NSL>
__device__ __forceinline__ void put_partials(const double (&v)[NSL], const int (&slot)[NSL], double* partial, int ps, double* sh,
                                             int own = -1) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NSL; ++j) {
    const double t = wave_sum(v[j]);
    if (lane == 0) sh[j * (BS / 64) + wid] = t;
  }
  __syncthreads();
  if (threadIdx.x < NSL) {
    const int j = threadIdx.x;
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < BS / 64; ++i) t += sh[j * (BS / 64) + i];
    partial[slot[j] * ps + (own < 0 ? (int)blockIdx.x : own)] = t;
  }
  for (int i = blockIdx.x + (threadIdx.x + 1) * gridDim.x; i < ps; i += BS * gridDim.x) {
#pragma unroll
    for (int j = 0; j < NSL; ++j) partial[slot[j] * ps + i] = 0.0;
  }
}

// Sums of the first `count` entries of NSL partial slots (stride ps), computed by the whole block (all
// slots' loads in one pass); returned in every thread, identical in every block.
template <int BS, int NSL>
__device__ __forceinline__ void get_sums(const double* __restrict__ partial, const int (&slot)[NSL], int count, int ps, double* sh,
                                         double (&out)[NSL]) {
  double s[NSL];
#pragma unroll
  for (int j = 0; j < NSL; ++j) s[j] = 0.0;
  // unrolled so that several iterations' loads are in flight together (the flat SpMV form
  // leaves thousands of partials per sum); the additions keep their order
#pragma unroll 4
  for (int i = threadIdx.x; i < count; i += BS) {
#pragma unroll
    for (int j = 0; j < NSL; ++j) s[j] += partial[slot[j] * ps + i];
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NSL; ++j) {
    const double t = wave_sum(s[j]);
    if (lane == 0) sh[j * (BS / 64) + wid] = t;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NSL; ++j) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < BS / 64; ++i) t += sh[j * (BS / 64) + i];
    out[j] = t;
  }
  __syncthreads();
}

constexpr int N_XCD = 8;
__device__ __forceinline__ int xcd_rank(int b, int nb) {
  const int x = b % N_XCD, per = nb / N_XCD, rem = nb % N_XCD;
  return x * per + min(x, rem) + b / N_XCD;
}
// Node columns of row r.  With a box numbering (M.box_b > 0) a node off the box's faces
// computes them (i + dz A + dy B + dx, the ascending order its stored slots have), so only
// face nodes load theirs: 27 x 4 bytes per node and the loads' round trip before the operand
// gathers saved.  The node's (ix, iy, iz) come from two floor divisions in FP64: (i + 0.5) / A
// lies at least 0.5 / A from an integer, far beyond the product's rounding for i < 2^30.
__device__ __forceinline__ void flat_cols(const BellView& M, int64_t r, int32_t (&j)[27]) {
  const int64_t i = r / 3;
  if (M.box_b > 0) {  // uniform over the grid
    const int32_t ii = (int32_t)i;
    const int32_t iz = (int32_t)(((double)ii + 0.5) * M.box_inv_a);
    const int32_t rz = ii - iz * M.box_a;
    const int32_t iy = (int32_t)(((double)rz + 0.5) * M.box_inv_b);
    const int32_t ix = rz - iy * M.box_b;
    if ((uint32_t)(ix - 1) < (uint32_t)(M.box_b - 2) && (uint32_t)(iy - 1) < (uint32_t)(M.box_ny - 2) &&
        (uint32_t)(iz - 1) < (uint32_t)(M.box_nz - 2)) {
#pragma unroll
      for (int s = 0; s < 27; ++s) j[s] = ii + (s / 9 - 1) * M.box_a + (s / 3 % 3 - 1) * M.box_b + (s % 3 - 1);
      return;
    }
  }
#pragma unroll
  for (int s = 0; s < 27; ++s) j[s] = M.col[(int64_t)s * M.n_nodes + i];
}

// A u of row r for one stored operand u, slots in order.
template <typename TM>
__device__ __forceinline__ double spmv1_flat(const BellView& M, const TM* __restrict__ vals, const double* __restrict__ u,
                                             int64_t r, const int32_t (&j)[27]) {
  const int64_t nrow = 3 * M.n_nodes;
  double a = 0.0;
#pragma unroll
  for (int s = 0; s < 27; ++s) {
    const TM* m = vals + (3 * (int64_t)s) * nrow + r;
    const int64_t jj = 3 * (int64_t)j[s];
#pragma unroll
    for (int c = 0; c < 3; ++c) a += (double)m[c * nrow] * u[jj + c];
  }
  return a;
}

}  // namespace cpfem
