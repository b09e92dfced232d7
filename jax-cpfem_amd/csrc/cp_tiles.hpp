// Dense 64 x 64 tiles in FP64: products on the matrix cores, inverses, row products.  Used by the
// direct solver's band and by the last level of the multigrid preconditioner.
#pragma once
#include "cp_internal.hpp"

namespace cpfem {

constexpr int NB = BAND_NB;
constexpr int TILE = NB * NB;
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

// Products of 64 x 64 tiles on the matrix cores (v_mfma_f64_16x16x4: a lane holds A[l % 16][l / 16],
// B[l / 16][l % 16] and D[4 v + l / 16][l % 16]).  A wave owns 16 rows of the left operand, kept
// in "operand layout": x[t] = X[l % 16][4 t + l / 16].  That is both the A operand of X M and the
// B operand of (X M)^T = M^T X^T, and the D of the latter comes out in operand layout again
// (t = 4 c + v), so chains of right multiplications need no exchange between lanes.  M is read
// from LDS, where a row-major tile (P = NB) has its columns exchanged in groups of 16 by row, so
// that the four rows that one read takes lie in different banks.
__device__ __forceinline__ int lds_swizzle(int r, int c) { return r * NB + (c ^ ((r & 3) << 4)); }
template <int P, bool CHAIN>
__device__ __forceinline__ void mul_tile(v4d (&acc)[4], const double (&x)[16], const double* S, int l) {
  const double* m[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) m[c] = S + (P == NB ? lds_swizzle(l / 16, 16 * c + l % 16) : (l / 16) * P + 16 * c + l % 16);
  double e[2][4];
#pragma unroll
  for (int c = 0; c < 4; ++c) e[0][c] = m[c][0];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    if (t < 15) {
#pragma unroll
      for (int c = 0; c < 4; ++c) e[(t + 1) & 1][c] = m[c][4 * (t + 1) * P];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
      acc[c] = CHAIN ? __builtin_amdgcn_mfma_f64_16x16x4f64(e[t & 1][c], x[t], acc[c], 0, 0, 0)
                     : __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], e[t & 1][c], acc[c], 0, 0, 0);
    // one step of LDS reads ahead is enough; the scheduler would hoist them all, and spill
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int P>
__device__ __forceinline__ void mul_chain(v4d (&acc)[4], const double (&x)[16], const double* S, int l) {
  mul_tile<P, true>(acc, x, S, l);
}
template <int P>
__device__ __forceinline__ void mul_last(v4d (&acc)[4], const double (&x)[16], const double* S, int l) {
  mul_tile<P, false>(acc, x, S, l);
}

// A tile on its way to LDS: 256 threads, 8 x 16 bytes each.
struct Stage {
  v2d v[8];
  __device__ __forceinline__ void load(const double* g) {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = reinterpret_cast<const v2d*>(g)[threadIdx.x + 256 * k];
  }
  __device__ __forceinline__ void store(double* S) const {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int e = 2 * (threadIdx.x + 256 * k);
      *reinterpret_cast<v2d*>(S + lds_swizzle(e / NB, e % NB)) = v[k];
    }
  }
  template <int P>
  __device__ __forceinline__ void store_transposed(double* S) const {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int e = 2 * (threadIdx.x + 256 * k), r = e / NB, c = e % NB;
      S[c * P + r] = v[k].x;
      S[(c + 1) * P + r] = v[k].y;
    }
  }
};

// Inverse of a tile held by 256 threads in D layout (wave w: a[c][v] is row 16 w + 4 v + l / 16,
// column 16 c + l % 16), in place, by Gauss-Jordan steps of four pivots: the four pivot rows and
// columns go through LDS, every lane forms its column of the 4 x 4 pivot block's inverse, and the
// rank-4 update is one matrix instruction per 16 columns, the tile column of the next pivots
// first, the others under the next pivot block's elimination.  What bounds it is the chain LDS -
// four reciprocals - two matrix instructions, 16 times.  Returns whether an entry that the lane
// holds is not finite, as after a zero or non-finite pivot.
struct InvLds {
  double row[2][4][NB];
  double col[2][NB][4];
};
__device__ __forceinline__ bool tile_inverse(v4d (&a)[4], InvLds& s) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lk = l >> 4;
  const auto put_col = [&](int q) {
    if (lr / 4 == q % 4) {
#pragma unroll
      for (int v = 0; v < 4; ++v) s.col[q & 1][16 * w + 4 * v + lk][lr % 4] = a[q / 4][v];
    }
  };
  double nw = 0.0, rk[4] = {};
  put_col(0);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int pc = q / 4, pv = q % 4, buf = q & 1;  // rows 4q.. are a[.][pv] of wave pc
    __syncthreads();
    double p[4][4], u[4], x[4], inv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) p[i][j] = s.col[buf][4 * q + i][j];
    const double ci = s.col[buf][16 * w + lr][lk];
    // x = P^-1 e_{lr % 4} by elimination without exchanges
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = lr % 4 == i ? 1.0 : 0.0;
    const auto pivot = [&](int k) {
      inv[k] = fast_rcp(p[k][k]);
#pragma unroll
      for (int i = k + 1; i < 4; ++i) {
        const double f = p[i][k] * inv[k];
#pragma unroll
        for (int j = k + 1; j < 4; ++j) p[i][j] -= f * p[k][j];
        u[i] -= f * u[k];
      }
    };
    // the previous step's update of the tile columns that its successor's pivots did not need
    if (q > 0) {
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        const int c = (pc + k) % 4;
        a[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(nw, rk[c], a[c], 0, 0, 0);
      }
    }
    pivot(0);
    pivot(1);
    if (w == pc) {
#pragma unroll
      for (int c = 0; c < 4; ++c) s.row[buf][lk][16 * c + lr] = a[c][pv];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) rk[c] = s.row[buf][lk][16 * c + lr];
    pivot(2);
    pivot(3);
#pragma unroll
    for (int i = 3; i >= 0; --i) {
      double v = u[i];
#pragma unroll
      for (int j = i + 1; j < 4; ++j) v -= p[i][j] * x[j];
      x[i] = v * inv[i];
    }
    // -W^T = P^-T (-A_iP)^T, with rows of the unit matrix in place of -A_iP for the pivot rows
    // (whose old values go), as a product whose D is in operand layout
    const bool prow = w == pc && lr / 4 == pv;
    const double pt = lr >= 4 ? 0.0 : lk == 0 ? x[0] : lk == 1 ? x[1] : lk == 2 ? x[2] : x[3];
    const v4d zero = {};
    const v4d wt = __builtin_amdgcn_mfma_f64_16x16x4f64(pt, prow ? (lr % 4 == lk ? 1.0 : 0.0) : -ci, zero, 0, 0, 0);
    nw = wt[0];
    if (w == pc) {
#pragma unroll
      for (int c = 0; c < 4; ++c) a[c][pv] = 0.0;
    }
    if (lr / 4 == pv) {
#pragma unroll
      for (int v = 0; v < 4; ++v) a[pc][v] = 0.0;
      rk[pc] = lr % 4 == lk ? 1.0 : 0.0;
    }
    const int pn = (q + 1) / 4 % 4;
    a[pn] = __builtin_amdgcn_mfma_f64_16x16x4f64(nw, rk[pn], a[pn], 0, 0, 0);
    if (q < 15) {
      put_col(q + 1);
    } else {
#pragma unroll
      for (int c = 1; c < 4; ++c) a[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(nw, rk[c], a[c], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // a zero or non-finite pivot has a NaN reciprocal (fast_rcp), which reaches every entry
  double sum = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int v = 0; v < 4; ++v) sum += 0.0 * a[c][v];
  return sum != 0.0;
}

__device__ __forceinline__ void load_d(v4d (&a)[4], const double* g, int w, int l) {
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int c = 0; c < 4; ++c) a[c][v] = g[(16 * w + 4 * v + l / 16) * NB + 16 * c + l % 16];
}
__device__ __forceinline__ void store_d(const v4d (&a)[4], double* g, int w, int l) {
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int c = 0; c < 4; ++c) g[(16 * w + 4 * v + l / 16) * NB + 16 * c + l % 16] = a[c][v];
}

// A row of a tile times 64 values, by 16 threads (sub: 0..15), two 16-byte pieces each.
__device__ __forceinline__ double row_dot(const double* row, const double* y, int sub) {
  double acc = 0.0;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const v2d a = reinterpret_cast<const v2d*>(row)[sub + 16 * m];
    const v2d b = reinterpret_cast<const v2d*>(y)[sub + 16 * m];
    acc = fma(a.x, b.x, fma(a.y, b.y, acc));
  }
  return acc;
}
__device__ __forceinline__ double sum16(double v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 16);
  return v;
}

}  // namespace cpfem
