// Geometric multigrid preconditioner for the Newton matrices of box-numbered meshes, and the
// BiCGSTAB that uses it.
//
// The reference solves every Newton system by Jacobi-preconditioned BiCGSTAB
// (crystal_plasticity_OR_design/solver.py:19-48), whose iteration count grows with the number of
// elements per side (about 200 at 16^3, 370 at 32^3, 900 at 64^3 to 1e-12), each iteration two
// passes over the whole matrix.  Here the same recurrence runs to the same stopping rule with
// one multigrid V-cycle in the place of the diagonal scaling: about 10 iterations at every
// size, in the elastic and in the plastic state.
//
// Cycle: levels coarsen every direction by two (node 2I; an odd last element stays as one),
// trilinear interpolation P, coarse operators P^T A P, Dirichlet dofs masked out on every level
// (on the finest they are scaled by the diagonal alone, on the others they stay zero); before the coarse correction a Chebyshev polynomial
// of the diagonally scaled operator over [0.1, 1.1] lambda_max (coarser levels: [0.07, 1.1]), none
// after it.  With scalar-diagonal smoothing before the correction only, degree 4 needs the fewest
// matrix passes (per iteration 2 + 2 x 4 on the finest level; degree 2 takes 16 iterations, 3 takes
// 12, 4 takes 10; smoothing after the correction as well, 3x3 block diagonals and W-cycles gain
// nothing).  Degree 4 over the wider range on the coarser levels takes 664 iterations for 72
// systems of 24 shapes, where degree 3 over [0.1, 1.1] takes 731, and 16.3 ms at 64^3 (17.5), 3.0 at
// 40^3 (3.2).  The last level is the first of at most DENSE_ROWS rows; its inverse is formed by
// tiles (k_dense_step) and applied as one dense product.
// lambda_max comes from a power iteration on the second level: on boxes of eight and more elements a
// side the levels' values differ by a few percent, the polynomial's range by ten.  On thinner ones the
// second level has one to three elements across, between faces that may both be held, and its value
// can lie far below the finest level's (a polynomial over too short a range amplifies instead of
// smoothing): there (mg_fine_range) the finest level's own value is found too, and the larger one taken.
//
// The polynomial is run as the three-term recurrence on the iterate,
//   x' = x + c1 (x - x_prev) + c2 D^-1 (b - A x),
// which reads and writes two vectors fewer per pass than the form that carries the residual.
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "cp_krylov.hpp"
#include "cp_tiles.hpp"

namespace cpfem {

constexpr int DEG_FINE = 4, DEG_COARSE = 4;
constexpr double LOW_FINE = 0.1, LOW_COARSE = 0.07;  // the polynomials' ranges start at this times lambda_max
constexpr int DENSE_ROWS = 768;    // the first level of at most this many rows is the last, and is inverted
// Steps of the power iteration: BiCGSTAB iterations over 24 shapes at 6, 8, 10, 12, 14, 16, 20 steps:
// 4991 (some solves run to the limit), 737, 670, 664, 667, 669, 669.
constexpr int POWER_STEPS = 12;
// When the iteration gives up.  mg_pays keeps most systems that are not for this preconditioner from it;
// for those that it lets through (48^3 of 1:1:0.1 elements, 3x20x20 of 1:1:4 held on two faces) this bounds
// what the attempt costs: 24^3 of 1:1:10, tried all the same, 27.0 ms with all MG_MAXITER iterations, 18.0
// with this, Jacobi alone 15.3.  What converges is left alone: 24 shapes of 1:1:1 elements, and 1:1:3
// (32 iterations), 1:1:0.1 (37) take the iterations they took.
constexpr int STALL_FROM = 7;
constexpr float STALL_SLACK = 6.65f;  // log2(100)
constexpr int FLAT_ROWS = 60000;   // one thread per row from here on; below, three waves per 64 rows
constexpr int PLAIN_ROWS = 700000; // row blocks in launch order from here on; below, XCD-local ranges

// Chebyshev recurrence over [lo, 1.1] lambda_max in units of 1 / lambda_max (the kernels multiply
// by the device-resident 1 / lambda_max): x1 = ith D^-1 b, then step k uses c1[k], c2[k].
struct Cheb {
  double ith;
  double c1[4], c2[4];
};

static Cheb cheb(int deg, double lo) {
  Cheb c{};
  const double hi = 1.1, th = 0.5 * (hi + lo), de = 0.5 * (hi - lo), sg = th / de;
  double rho = 1.0 / sg;
  c.ith = 1.0 / th;
  for (int k = 0; k + 1 < deg; ++k) {
    const double rn = 1.0 / (2.0 * sg - rho);
    c.c1[k] = rn * rho;
    c.c2[k] = 2.0 * rn / de;
    rho = rn;
  }
  return c;
}

// ---------------------------------------------------------------------------------
// Grids (host)
static MgGrid make_grid(int64_t nx, int64_t ny, int64_t nz) {
  MgGrid g;
  g.nx = (int32_t)nx;
  g.ny = (int32_t)ny;
  g.nz = (int32_t)nz;
  g.n = (int32_t)(3 * nx * ny * nz);
  g.inv_a = 1.0 / (double)(nx * ny);
  g.inv_b = 1.0 / (double)nx;
  return g;
}
static int64_t coarse_nodes(int64_t m) { return (m - 1 + 1) / 2 + 1; }  // m nodes, ceil((m - 1) / 2) + 1

bool mg_plan(const int64_t box[3], Multigrid* mg) {
  if (box[0] < 3 || box[1] < 3 || box[2] < 3 || 3 * box[0] * box[1] * box[2] >= (1LL << 28)) return false;
  mg->nl = 0;
  int64_t m[3] = {box[0], box[1], box[2]};
  for (;;) {
    mg->lv[mg->nl] = MgLevel{};
    mg->lv[mg->nl].g = make_grid(m[0], m[1], m[2]);
    ++mg->nl;
    const int64_t c[3] = {coarse_nodes(m[0]), coarse_nodes(m[1]), coarse_nodes(m[2])};
    if (3 * m[0] * m[1] * m[2] <= DENSE_ROWS || (c[0] == m[0] && c[1] == m[1] && c[2] == m[2])) break;
    if (mg->nl == MG_MAXL) break;
    for (int d = 0; d < 3; ++d) m[d] = c[d];
  }
  return mg->nl >= 2 && mg->lv[mg->nl - 1].g.n <= DENSE_ROWS;
}

void mg_scratch(const Multigrid& mg, int64_t* n1, int64_t* n2) {
  const MgGrid &f = mg.lv[0].g, &c = mg.lv[1].g;
  *n1 = 81LL * 3 * c.nx * f.ny * f.nz;
  *n2 = 81LL * 3 * c.nx * c.ny * f.nz;
}

// ---------------------------------------------------------------------------------
// Which preconditioner (host).  Multigrid wants elements that are not too stretched (point smoothing,
// coarsening in all directions), and a system that is hard for the Jacobi iteration: held on close
// faces, that one needs a few dozen iterations, each a fraction of a multigrid one.  Both counts are
// estimated from the mesh and its Dirichlet dofs.
//
// Multigrid, from elements of proportions a <= b <= c: 2.5 + 4.6 c/a + 1.2 (c/b - 1), measured 6..8 for
// cubes, 12 for 1:1:2, 18 for 1:1:3, 25 for 1:1:4, 31 for 1:1:5, 53 for 1:1:10, 24 for 1:5:5 and 49 for
// 1:10:10.  Above 40 some run into MG_MAXITER; they are let through to 50 only where the longest way to a
// held node (below) runs in the direction of the displacement itself.
//
// Jacobi, from the longest way to a node where a displacement component is held, over components and
// directions, in elements: 38 + 6 w along the component, w weighted by the square root of
// the element's length over the shortest one; 35 + 9 w across it (a bar held at its ends), w weighted by
// that length.  These are low estimates: 24^3 under symmetry planes 182 (measured 233..239), 16^3 134
// (156..192), 24x24x6 182 (165..177), 24^3 held on two faces 143 (182..199), 24x24x6 62 (64), 32x32x4 53
// (45), 24^3 of 1:1:10 266 (385..410), of 1:10:10 493 (815).
//
// A multigrid iteration takes the time of 4.5 Jacobi ones with two levels (10^3), 6.8 with three (16^3),
// 8 with four (24^3; 5.5 to 7 where the finest level's passes outweigh the launches), its set-up that of about
// fifteen.
// Without this, against the Jacobi solve: 24x24x6 held on two faces 1.29 -> 2.70 ms, 16^3 so held of
// 1:1:0.2 1.77 -> 3.10, 24^3 of 1:1:10 9.4 -> 10.3, 16^3 of it 4.5 -> 5.8, each now the Jacobi solve.  Of
// 1:1:4 elements 24^3 would gain 1.5, and takes the Jacobi solve too.
static double mg_iterations(double x, double y, double z) {
  const double a = std::min({x, y, z}), c = std::max({x, y, z}), b = std::max(std::min(x, y), std::min(std::max(x, y), z));
  return a > 0.0 ? 2.5 + 4.6 * c / a + 1.2 * (c / b - 1.0) : 1e30;
}

MgMesh mg_mesh(const int64_t box[3], const double* points) {
  MgMesh m;
  const int64_t step[3] = {1, box[0], box[0] * box[1]};
  double run[3][3] = {}, count[3] = {};
  for (int64_t z = 0, i = 0; z < box[2]; ++z)
    for (int64_t y = 0; y < box[1]; ++y)
      for (int64_t x = 0; x < box[0]; ++x, ++i) {
        const bool in[3] = {x + 1 < box[0], y + 1 < box[1], z + 1 < box[2]};
        double len[3];
        for (int d = 0; d < 3; ++d) {
          if (!in[d]) continue;
          double s = 0.0;
          for (int c = 0; c < 3; ++c) {
            const double v = points[3 * (i + step[d]) + c] - points[3 * i + c];
            s += v * v;
            run[d][c] += std::fabs(v);
          }
          len[d] = std::sqrt(s);
          m.h[d] += len[d];
          count[d] += 1.0;
        }
        if (in[0] && in[1] && in[2]) {
          m.its = std::max(m.its, mg_iterations(len[0], len[1], len[2]));
          m.stretch = std::max(m.stretch, std::max({len[0], len[1], len[2]}) / std::min({len[0], len[1], len[2]}));
        }
      }
  for (int d = 0; d < 3; ++d) {
    m.h[d] /= std::max(count[d], 1.0);
    m.axis[d] = (int)(std::max_element(run[d], run[d] + 3) - run[d]);
  }
  return m;
}

// Boxes of fewer than eight elements in a direction, if the elements are not nearly cubes, and of fewer than
// four: there the second level's lambda_max was up to 1.8 times below the finest one's; cubes, four to
// seven across between held faces, 1.01 to 1.04.
bool mg_fine_range(const int64_t box[3], const MgMesh& mesh) {
  const int64_t across = std::min({box[0], box[1], box[2]}) - 1;
  return across < 4 || (across < 8 && mesh.stretch > 1.25);
}

bool mg_pays(const int64_t box[3], const MgMesh& mesh, int64_t n, const int64_t* dofs) {
  const double h0 = std::min({mesh.h[0], mesh.h[1], mesh.h[2]});
  Multigrid plan;
  if (!(h0 > 0.0) || !mg_plan(box, &plan)) return false;
  std::vector<uint8_t> held[3][3];  // coordinates of the nodes where a component is held
  for (int c = 0; c < 3; ++c)
    for (int d = 0; d < 3; ++d) held[c][d].assign((size_t)box[d], 0);
  for (int64_t k = 0; k < n; ++k) {
    const int64_t i = dofs[k] / 3, z = i / (box[0] * box[1]), y = i / box[0] % box[1], x = i % box[0];
    std::vector<uint8_t>* h = held[dofs[k] % 3];
    h[0][x] = h[1][y] = h[2][z] = 1;
  }
  double jacobi = 0.0;
  bool along = true;
  for (int c = 0; c < 3; ++c) {
    for (int d = 0; d < 3; ++d) {
      int64_t far = 0, last = -1;  // last: the held coordinate before
      for (int64_t k = 0; k <= box[d]; ++k) {
        if (k < box[d] && !held[c][d][k]) continue;
        const bool open = last < 0 || k == box[d];  // an end of the box, not held
        far = std::max(far, last < 0 && k == box[d] ? box[d] - 1 : open ? (last < 0 ? k : k - 1 - last) : (k - last) / 2);
        last = k;
      }
      const double l = mesh.h[d] / h0;
      const double it = mesh.axis[d] == c ? 38.0 + 6.0 * (double)far * std::sqrt(l) : 35.0 + 9.0 * (double)far * l;
      if (it > jacobi) {
        jacobi = it;
        along = mesh.axis[d] == c;
      }
    }
  }
  return mesh.its <= (along ? 50.0 : 40.0) && jacobi >= 15.0 + std::min(8.0, 0.4 + 2.2 * plan.nl) * mesh.its;
}

// ---------------------------------------------------------------------------------
// Interpolation in one direction with n elements: fine node of coarse node X, and the weight of
// coarse node X at fine node i.
__device__ __forceinline__ int mg_fine(int X, int n) { return min(2 * X, n); }
__device__ __forceinline__ double mg_weight(int i, int f, int n) {
  if (i == f) return 1.0;
  return (i & 1) && i != n && (i == f + 1 || i == f - 1) ? 0.5 : 0.0;
}

struct NodeXYZ {
  int x, y, z;
};
// Node coordinates of node i: (i + 0.5) / A lies at least 0.5 / A from an integer, far beyond the
// product's rounding.
__device__ __forceinline__ NodeXYZ mg_node(const MgGrid& g, int i) {
  NodeXYZ p;
  p.z = (int)(((double)i + 0.5) * g.inv_a);
  const int rz = i - p.z * g.nx * g.ny;
  p.y = (int)(((double)rz + 0.5) * g.inv_b);
  p.x = rz - p.y * g.nx;
  return p;
}

// A x of row r over the slots of one part (27 / P of them): FINE: the caller's block-ELL matrix
// (columns of face nodes loaded, the others computed), else a coarse operator in offset order.
template <typename TM, bool FINE, int P>
__device__ __forceinline__ double mg_dot(const BellView& M, const MgGrid& g, const TM* __restrict__ A,
                                         const double* __restrict__ x, int r, int part) {
  constexpr int NSL = 27 / P;
  const int i = (int)((uint32_t)r / 3u);
  const NodeXYZ p = mg_node(g, i);
  const int a = g.nx * g.ny, b = g.nx;
  const int s0 = P == 1 ? 0 : NSL * part;
  const bool inner = (uint32_t)(p.x - 1) < (uint32_t)(g.nx - 2) && (uint32_t)(p.y - 1) < (uint32_t)(g.ny - 2) &&
                     (uint32_t)(p.z - 1) < (uint32_t)(g.nz - 2);
  int32_t j[NSL];
  if (inner) {
    const int base = P == 1 ? i - a : i + (part - 1) * a;
#pragma unroll
    for (int k = 0; k < NSL; ++k) j[k] = base + (k / 9) * a + (k / 3 % 3 - 1) * b + (k % 3 - 1);
  } else if (FINE) {
#pragma unroll
    for (int k = 0; k < NSL; ++k) j[k] = M.col[(int64_t)(s0 + k) * M.n_nodes + i];
  } else {  // an offset out of the box holds zeros: any node of the box will do
    const int xm = p.x > 0 ? 1 : 0, xp = p.x < g.nx - 1 ? 1 : 0, ym = p.y > 0 ? b : 0, yp = p.y < g.ny - 1 ? b : 0;
    const int zm = p.z > 0 ? a : 0, zp = p.z < g.nz - 1 ? a : 0;
#pragma unroll
    for (int k = 0; k < NSL; ++k) {
      const int dz = P == 1 ? k / 9 - 1 : part - 1, dy = k / 3 % 3 - 1, dx = k % 3 - 1;
      j[k] = i + (dz < 0 ? -zm : dz > 0 ? zp : 0) + (dy < 0 ? -ym : dy > 0 ? yp : 0) + (dx < 0 ? -xm : dx > 0 ? xp : 0);
    }
  }
  const int64_t n = g.n;
  const TM* __restrict__ v = A + 3 * (int64_t)s0 * n + r;
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < NSL; ++k) {
#pragma unroll
    for (int c = 0; c < 3; ++c) acc += (double)v[(3 * k + c) * n] * x[3 * j[k] + c];
  }
  return acc;
}

// Rows of a block: P = 1: 256 rows, one per thread; P = 3: 64 rows, the slots of each split over
// the block's three waves (planes of the stencil), so that small levels fill more of the device.
template <int P>
struct MgShape {
  static constexpr int BS = P == 1 ? 256 : 64 * P;
  static constexpr int ROWS = P == 1 ? 256 : 64;
};

// order: bit 0: row blocks in reverse, bit 1: XCD-local ranges.  Consecutive passes over the same
// matrix alternate their direction, so that each starts on the rows the last one read last (the
// matrix outgrows the 256 MB Infinity Cache at 56^3).
template <int P>
__device__ __forceinline__ int mg_row0(int order) {
  int b = (order & 2) ? xcd_rank((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
  if (order & 1) b = (int)gridDim.x - 1 - b;
  return b * MgShape<P>::ROWS;
}

// A x of this thread's row; true in the thread that owns the row (whose acc is complete).
template <typename TM, bool FINE, int P>
__device__ __forceinline__ bool mg_row(const BellView& M, const MgGrid& g, const TM* __restrict__ A,
                                       const double* __restrict__ x, int order, int& r, double& acc, double* red) {
  if constexpr (P == 1) {
    r = mg_row0<1>(order) + (int)threadIdx.x;
    acc = 0.0;
    if (r < g.n) acc = mg_dot<TM, FINE, 1>(M, g, A, x, r, 0);
    return r < g.n;
  } else {
    const int lane = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    r = mg_row0<P>(order) + lane;
    acc = 0.0;
    if (r < g.n) acc = mg_dot<TM, FINE, P>(M, g, A, x, r, part);
    if (part) red[(part - 1) * 64 + lane] = acc;
    __syncthreads();
    if (part) return false;
#pragma unroll
    for (int k = 0; k < P - 1; ++k) acc += red[k * 64 + lane];
    return r < g.n;
  }
}

// The finest level is smoothed once more while the host waits for the convergence test (see
// mg_krylov_begin): a pass over its matrix (14 us at 32^3, 108 at 64^3) is not made when that has ended
// the solve.  Smaller levels make theirs: it is shorter than the test's round trip to memory.  No kernel
// in flight writes `done`, so it is the same in every wave of the grid.
template <bool FINE, int P>
__device__ __forceinline__ bool mg_idle(const int32_t* __restrict__ done) {
  return FINE && P == 1 && *done;
}

// One Chebyshev step: xo <- x + c1 (x - xo) + c2 D^-1 (b - A x) (first: xo counts as zero).
template <typename TM, bool FINE, int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mg_smooth(BellView M, const TM* __restrict__ A, MgGrid g,
                                                             const double* __restrict__ minv, const double* __restrict__ b,
                                                             const double* __restrict__ x, double* __restrict__ xo, int first,
                                                             double c1, double c2, const double* __restrict__ lam,
                                                             const int32_t* __restrict__ done, int order) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  if (mg_idle<FINE, P>(done)) return;
  const double c2l = c2 * lam[0];
  int r;
  double acc;
  if (!mg_row<TM, FINE, P>(M, g, A, x, order, r, acc, red)) return;
  const double xv = x[r], xp = first ? 0.0 : xo[r];
  xo[r] = xv + (c1 * (xv - xp) + c2l * minv[r] * (b[r] - acc));
}

// r = b - A x on the free dofs, 0 on Dirichlet dofs.
template <typename TM, bool FINE, int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mg_resid(BellView M, const TM* __restrict__ A, MgGrid g,
                                                            const double* __restrict__ minv, const double* __restrict__ b,
                                                            const double* __restrict__ x, double* __restrict__ out,
                                                            const int32_t* __restrict__ done, int order) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  if (mg_idle<FINE, P>(done)) return;
  int r;
  double acc;
  if (!mg_row<TM, FINE, P>(M, g, A, x, order, r, acc, red)) return;
  out[r] = minv[r] != 0.0 ? b[r] - acc : 0.0;
}

// Power iteration: xo = D^-1 A x, and the partial sums of <xo, xo> and <x, x>.
template <typename TM, bool FINE, int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mg_power(BellView M, const TM* __restrict__ A, MgGrid g,
                                                            const double* __restrict__ minv, const double* __restrict__ x,
                                                            double* __restrict__ xo, double* __restrict__ partial, int ps) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  __shared__ double sh[2 * (MgShape<P>::BS / 64)];
  int r;
  double acc, v[2] = {0.0, 0.0};
  if (mg_row<TM, FINE, P>(M, g, A, x, 0, r, acc, red)) {
    const double y = minv[r] * acc;
    xo[r] = y;
    v[0] = y * y;
    v[1] = x[r] * x[r];
  }
  put_partials<MgShape<P>::BS, 2>(v, {0, 1}, partial, ps, sh);
}
// Start vector: an alternating sign per node with a hashed amplitude (the largest eigenvectors
// oscillate from node to node).
__global__ void __launch_bounds__(256) k_mg_power_start(MgGrid g, const double* __restrict__ minv, double* __restrict__ x) {
  const int r = (int)(blockIdx.x * 256 + threadIdx.x);
  if (r >= g.n) return;
  const NodeXYZ p = mg_node(g, (int)((uint32_t)r / 3u));
  uint32_t h = (uint32_t)r * 2654435761u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  const double s = ((p.x + p.y + p.z) & 1) ? -1.0 : 1.0;
  x[r] = minv[r] != 0.0 ? s * (0.5 + (double)(h >> 8) * (1.0 / 16777216.0)) : 0.0;
}
// lam[1 + which] = 1 / lambda_max; lam[0] the least of those found.
__global__ void __launch_bounds__(256) k_mg_power_finish(const double* __restrict__ partial, int count, int ps, int which,
                                                        double* __restrict__ lam) {
  __shared__ double sh[2 * 4];
  double v[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < count; i += 256) {
    v[0] += partial[i];
    v[1] += partial[ps + i];
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const double s = wave_sum(v[j]);
    if (lane == 0) sh[j * 4 + wid] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const double il = sqrt((sh[4] + sh[5] + sh[6] + sh[7]) / (sh[0] + sh[1] + sh[2] + sh[3]));
    lam[1 + which] = il;
    lam[0] = which ? fmin(lam[0], il) : il;
  }
}

// P^T r at coarse row t (res: the residual of grid f).
__device__ __forceinline__ double mg_restrict_row(const MgGrid& f, const MgGrid& g, int t, const double* __restrict__ res) {
  const int I = (int)((uint32_t)t / 3u), c = t - 3 * I;
  const NodeXYZ p = mg_node(g, I);
  const int ex = f.nx - 1, ey = f.ny - 1, ez = f.nz - 1;
  const int fx = mg_fine(p.x, ex), fy = mg_fine(p.y, ey), fz = mg_fine(p.z, ez);
  double acc = 0.0;
#pragma unroll
  for (int dz = -1; dz <= 1; ++dz) {
    const int z = fz + dz;
    const bool okz = z >= 0 && z <= ez;
    const double wz = okz ? mg_weight(z, fz, ez) : 0.0;
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy) {
      const int y = fy + dy;
      const bool oky = okz && y >= 0 && y <= ey;
      const double wy = oky ? wz * mg_weight(y, fy, ey) : 0.0;
#pragma unroll
      for (int dx = -1; dx <= 1; ++dx) {
        const int xx = fx + dx;
        const bool ok = oky && xx >= 0 && xx <= ex;
        const double w = ok ? wy * mg_weight(xx, fx, ex) : 0.0;
        const int node = ok ? xx + f.nx * (y + f.ny * z) : fx + f.nx * (fy + f.ny * fz);
        acc += w * res[3 * node + c];
      }
    }
  }
  return acc;
}

// Restriction b_c = P^T r and the first coarse iterate x_c = ith D^-1 b_c.
__global__ void __launch_bounds__(256) k_mg_restrict(MgGrid f, MgGrid g, const double* __restrict__ rf,
                                                    const double* __restrict__ minv, double* __restrict__ b,
                                                    double* __restrict__ x, double ith, const double* __restrict__ lam) {
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t >= g.n) return;
  const double il = ith * lam[0], mi = minv[t];
  double acc = mg_restrict_row(f, g, t, rf);
  acc = mi != 0.0 ? acc : 0.0;
  b[t] = acc;
  x[t] = il * mi * acc;
}

// P e at fine node (x, y, z), component c.
__device__ __forceinline__ double mg_interp(const MgGrid& f, const MgGrid& g, const NodeXYZ& p, int c,
                                            const double* __restrict__ e) {
  // the one or two parents of a direction: first, step to the second (0: none), weight
  const auto par = [](int i, int n, int& X, int& d) {
    if (!(i & 1)) {
      X = i >> 1;
      d = 0;
    } else if (i == n) {
      X = (i + 1) >> 1;
      d = 0;
    } else {
      X = i >> 1;
      d = 1;
    }
  };
  int X, Y, Z, dx, dy, dz;
  par(p.x, f.nx - 1, X, dx);
  par(p.y, f.ny - 1, Y, dy);
  par(p.z, f.nz - 1, Z, dz);
  const int b = 3 * (X + g.nx * (Y + g.ny * Z)) + c;
  const int sx = 3 * dx, sy = 3 * dy * g.nx, sz = 3 * dz * g.nx * g.ny;
  // a direction without a second parent reads the first one twice: the mean is its value
  const double v0 = 0.5 * (e[b] + e[b + sx]), v1 = 0.5 * (e[b + sy] + e[b + sy + sx]);
  const double v2 = 0.5 * (e[b + sz] + e[b + sz + sx]), v3 = 0.5 * (e[b + sz + sy] + e[b + sz + sy + sx]);
  return 0.5 * (0.5 * (v0 + v1) + 0.5 * (v2 + v3));
}

// out = x + P e on the free dofs; on Dirichlet dofs b / diagonal (finest level) or 0.
__global__ void __launch_bounds__(256) k_mg_prolong(MgGrid f, MgGrid g, const double* __restrict__ e, const double* __restrict__ x,
                                                   const double* __restrict__ minv, const double* __restrict__ b,
                                                   const double* __restrict__ invd, double* __restrict__ out) {
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t >= f.n) return;
  const int i = (int)((uint32_t)t / 3u);
  const NodeXYZ p = mg_node(f, i);
  const double v = x[t] + mg_interp(f, g, p, t - 3 * i, e);
  out[t] = minv[t] != 0.0 ? v : (invd ? b[t] * invd[t] : 0.0);
}

// ---------------------------------------------------------------------------------
// Coarse operators.  P is a product of one-dimensional interpolations, so P^T A P is formed one
// direction at a time: each pass halves the rows and reads and writes each value once (1.2 GB in
// all at 64^3), where the direct triple product reads every fine row 27 times.  A thread
// makes the three values of one coarse row, transverse offset pair and component from nine fine
// values.  DIR: direction coarsened; FINE: reads the block-ELL matrix with the masks of Dirichlet
// rows and columns; LAST: applies the coarse masks, writes the inverse diagonal and rounds to the level's
// value type.  Masked rows and columns are zero, their diagonals too: a number put there would be carried into
// the free dofs of the levels below, in units that are not the matrix's (k_dense_fill puts 1 there).
// Slot of offset (dx, dy, dz) in node p's row (existing neighbours in ascending order).
__device__ __forceinline__ int mg_slot(const MgGrid& f, const NodeXYZ& p, int dx, int dy, int dz) {
  const int xl = p.x > 0 ? -1 : 0, yl = p.y > 0 ? -1 : 0, zl = p.z > 0 ? -1 : 0;
  const int cx = (p.x < f.nx - 1 ? 2 : 1) - xl, cy = (p.y < f.ny - 1 ? 2 : 1) - yl;
  return ((dz - zl) * cy + (dy - yl)) * cx + (dx - xl);
}

template <int DIR, bool FINE, bool LAST, typename TI, typename TO>
__global__ void __launch_bounds__(256) k_mg_coarsen(MgGrid f, MgGrid g, const TI* __restrict__ A, const uint8_t* __restrict__ fixed,
                                                   const uint8_t* __restrict__ cfixed, TO* __restrict__ out,
                                                   double* __restrict__ minv) {
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t >= g.n) return;
  const int q = (int)blockIdx.y;  // (transverse offsets, component)
  const int k = q % 3, t1 = q / 3 % 3 - 1, t2 = q / 9 - 1;
  const int I = (int)((uint32_t)t / 3u), c = t - 3 * I;
  const NodeXYZ pc = mg_node(g, I);
  const int fn[3] = {f.nx, f.ny, f.nz};
  const int e = fn[DIR] - 1, X = DIR == 0 ? pc.x : DIR == 1 ? pc.y : pc.z;
  const int gX = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
  const int fX = mg_fine(X, e);
  // transverse directions in ascending order carry the offsets (t1, t2)
  NodeXYZ d{DIR == 0 ? 0 : t1, DIR == 1 ? 0 : (DIR == 0 ? t1 : t2), DIR == 2 ? 0 : t2};
  const bool inside = (uint32_t)(pc.x + d.x) < (uint32_t)(DIR == 0 ? g.nx : f.nx) &&
                      (uint32_t)(pc.y + d.y) < (uint32_t)(DIR == 1 ? g.ny : f.ny) &&
                      (uint32_t)(pc.z + d.z) < (uint32_t)(DIR == 2 ? g.nz : f.nz);
  double acc[3] = {0.0, 0.0, 0.0};
  if (inside) {
#pragma unroll
    for (int a = -1; a <= 1; ++a) {
      const int i = fX + a;
      if (i < 0 || i > e) continue;
      const double wi = mg_weight(i, fX, e);
      if (wi == 0.0) continue;
      const NodeXYZ pf{DIR == 0 ? i : pc.x, DIR == 1 ? i : pc.y, DIR == 2 ? i : pc.z};
      const int node = pf.x + f.nx * (pf.y + f.ny * pf.z);
      const int64_t row = 3 * (int64_t)node + c;
      if (FINE && fixed[row]) continue;
#pragma unroll
      for (int m = -1; m <= 1; ++m) {
        const int j = i + m;
        if (j < 0 || j > e) continue;
        const int dx = DIR == 0 ? m : d.x, dy = DIR == 1 ? m : d.y, dz = DIR == 2 ? m : d.z;
        int64_t s;
        if (FINE) {
          const int col = node + dx + f.nx * (dy + f.ny * dz);
          if (fixed[3 * (int64_t)col + k]) continue;
          s = mg_slot(f, pf, dx, dy, dz);
        } else {
          s = (dz + 1) * 9 + (dy + 1) * 3 + dx + 1;
        }
        const double v = wi * (double)A[(3 * s + k) * (int64_t)f.n + row];
#pragma unroll
        for (int o = -1; o <= 1; ++o) {
          const int Xo = X + o;
          if (Xo < 0 || Xo >= gX) continue;
          acc[o + 1] += mg_weight(j, mg_fine(Xo, e), e) * v;
        }
      }
    }
  }
  const int64_t gn = g.n;
#pragma unroll
  for (int o = -1; o <= 1; ++o) {
    const int dx = DIR == 0 ? o : d.x, dy = DIR == 1 ? o : d.y, dz = DIR == 2 ? o : d.z;
    const int64_t s = (dz + 1) * 9 + (dy + 1) * 3 + dx + 1;
    double v = acc[o + 1];
    if (LAST) {
      const bool in = inside && (uint32_t)(X + o) < (uint32_t)gX;
      const bool diag = dx == 0 && dy == 0 && dz == 0 && k == c;
      const bool fr = cfixed[t] != 0;
      const bool fc = in && cfixed[3 * (int64_t)(I + dx + g.nx * (dy + g.ny * dz)) + k] != 0;
      if (diag) minv[t] = fr ? 0.0 : 1.0 / v;
      if (fr || fc) v = 0.0;
    }
    out[(3 * s + k) * gn + t] = (TO)v;
  }
}

// ---------------------------------------------------------------------------------
// The last level: n rows in nt x nt dense tiles (unit rows beyond n), inverted by Gauss-Jordan
// steps over the tiles, one launch each, between two buffers:
//   A_kk' = D, A_kj' = D A_kj, A_ik' = -A_ik D, A_ij' = A_ij - (A_ik D) A_kj,  D = A_kk^-1,
// where the workgroup that finishes the next diagonal tile inverts it too.  The diagonal is raised
// by 1e-6, so that a floating box (a singular operator, as where only corners are held) keeps a
// bounded inverse.  Bound by the chain through the diagonal tiles, 17 us a step.
// Applying the inverse is one launch (375 rows 7 us, 648 rows 10), and takes the place of smoothing
// this level and the ones below it, 375 rows in one block of one CU 21 us, 648 rows in launches 45;
// forming it takes 6 x 17 or 11 x 18 us, where the inverse of 81 rows took 67.
template <typename TM>
__global__ void __launch_bounds__(256) k_dense_fill(MgGrid g, int nt, const TM* __restrict__ A, const double* __restrict__ minv,
                                                    double* __restrict__ out) {
  const int c = (int)(blockIdx.x * 256 + threadIdx.x), r = (int)blockIdx.y, ld = nt * NB;
  if (c >= ld) return;
  double v = r == c ? 1.0 : 0.0;
  if (r < g.n && c < g.n && (r != c || minv[r] != 0.0)) {
    const NodeXYZ p = mg_node(g, (int)((uint32_t)r / 3u)), q = mg_node(g, (int)((uint32_t)c / 3u));
    const int dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
    v = 0.0;
    if (abs(dx) <= 1 && abs(dy) <= 1 && abs(dz) <= 1)
      v = (double)A[(3 * ((dz + 1) * 9 + (dy + 1) * 3 + dx + 1) + c % 3) * (int64_t)g.n + r] * (r == c ? 1.0 + 1e-6 : 1.0);
  }
  out[((int64_t)(r / NB) * nt + c / NB) * TILE + (r % NB) * NB + c % NB] = v;
}

__global__ void __launch_bounds__(256) k_dense_first(const double* __restrict__ A, double* __restrict__ D) {
  __shared__ InvLds s;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  v4d a[4];
  load_d(a, A, w, l);
  (void)tile_inverse(a, s);
  store_d(a, D, w, l);
}

// Step k: `in` to `out`; D holds the inverse of tile (k, k), the next one goes to Dn.
__global__ void __launch_bounds__(256, 2) k_dense_step(int nt, int k, const double* __restrict__ in, double* __restrict__ out,
                                                       const double* __restrict__ D, double* __restrict__ Dn) {
  __shared__ double S[2][TILE];
  const int i = (int)blockIdx.y, j = (int)blockIdx.x, w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const auto tile = [&](const double* m, int r, int c) { return m + ((int64_t)r * nt + c) * TILE; };
  double* o = out + ((int64_t)i * nt + j) * TILE;
  v4d c[4] = {};
  if (i == k && j == k) {  // uniform over the block, as the other cases
    load_d(c, D, w, l);
    store_d(c, o, w, l);
    return;
  }
  Stage st;
  double x[16];
  // left operand: rows of D (row k), else of A_ik
  const double* g = (i == k ? D : tile(in, i, k)) + (16 * w + l % 16) * NB + l / 16;
#pragma unroll
  for (int t = 0; t < 16; ++t) x[t] = g[4 * t];
  if (i == k || j == k) {
    st.load(i == k ? tile(in, k, j) : D);
    st.store(S[0]);
    __syncthreads();
    mul_last<NB>(c, x, S[0], l);
    if (j == k) {
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = -c[q];
    }
  } else {
    st.load(D);
    st.store(S[0]);
    st.load(tile(in, k, j));
    load_d(c, tile(in, i, j), w, l);
    __syncthreads();
    {
      v4d acc[4] = {};
      mul_chain<NB>(acc, x, S[0], l);
#pragma unroll
      for (int t = 0; t < 16; ++t) x[t] = -acc[t / 4][t % 4];
    }
    st.store(S[1]);
    __syncthreads();
    mul_last<NB>(c, x, S[1], l);
  }
  store_d(c, o, w, l);
  if (i == k + 1 && j == k + 1) {
    static_assert(sizeof(InvLds) <= sizeof(S[0]), "");  // S[0] is free since the second barrier
    (void)tile_inverse(c, *reinterpret_cast<InvLds*>(S[0]));
    store_d(c, Dn, w, l);
  }
}

// x = inverse (P^T rf) of the last level, P^T rf formed by every workgroup for itself (its right-hand
// side in LDS), 16 rows a workgroup, 16 threads a row.
__global__ void __launch_bounds__(256) k_mg_dense(MgGrid f, MgGrid g, int nt, const double* __restrict__ rf,
                                                  const double* __restrict__ minv, const double* __restrict__ inv,
                                                  double* __restrict__ x) {
  __shared__ __align__(16) double b[DENSE_ROWS];
  for (int t = threadIdx.x; t < nt * NB; t += 256) b[t] = t < g.n && minv[t] != 0.0 ? mg_restrict_row(f, g, t, rf) : 0.0;
  __syncthreads();
  const int r = (int)blockIdx.x * 16 + threadIdx.x / 16, sub = threadIdx.x % 16;
  const double* row = inv + (int64_t)(r / NB) * nt * TILE + (r % NB) * NB;
  double acc = 0.0;
  for (int j = 0; j < nt; ++j) acc += row_dot(row + (int64_t)j * TILE, b + j * NB, sub);
  acc = sum16(acc);
  if (sub == 0 && r < g.n) x[r] = acc;
}

// Inverse diagonal of the finest level with Dirichlet dofs masked, and the Dirichlet flags of the
// next level (those of the fine node it stands on).
__global__ void __launch_bounds__(256) k_mg_mask(int n, const double* __restrict__ invd, const uint8_t* __restrict__ fixed,
                                                double* __restrict__ minv) {
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t < n) minv[t] = fixed[t] ? 0.0 : invd[t];
}
__global__ void __launch_bounds__(256) k_mg_inject(MgGrid f, MgGrid g, const uint8_t* __restrict__ fixed, uint8_t* __restrict__ out) {
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t >= g.n) return;
  const int I = (int)((uint32_t)t / 3u), c = t - 3 * I;
  const NodeXYZ p = mg_node(g, I);
  const int node = mg_fine(p.x, f.nx - 1) + f.nx * (mg_fine(p.y, f.ny - 1) + f.ny * mg_fine(p.z, f.nz - 1));
  out[t] = fixed[3 * (int64_t)node + c];
}

static inline unsigned blocks256(int64_t n) { return (unsigned)((n + 255) / 256); }
static inline int level_parts(int64_t n) { return n >= FLAT_ROWS ? 1 : 3; }
static inline unsigned level_blocks(int64_t n) { return (unsigned)(level_parts(n) == 1 ? (n + 255) / 256 : (n + 63) / 64); }
static inline int level_order(int64_t n, int rev) { return (rev & 1) | (n < PLAIN_ROWS ? 2 : 0); }
int mg_spmv_blocks(int64_t n) { return (int)level_blocks(n); }
// Dirichlet flags of a coarse level, in its residual until the first cycle.
static inline uint8_t* level_flags(const Multigrid& mg, int l) { return reinterpret_cast<uint8_t*>(mg.lv[l].r); }
int mg_dense_tiles(int64_t n) { return (int)((n + NB - 1) / NB); }

// Coarse operators of levels first + 1 to last; fixed: Dirichlet flags of level `first`.
template <typename TM>
static void coarsen(const Multigrid& mg, int first, int last, const double* vals, const uint8_t* fixed, hipStream_t st) {
  double *w1 = static_cast<double*>(mg.rap1), *w2 = static_cast<double*>(mg.rap2);
  for (int l = first; l < last; ++l) {
    const MgGrid f = mg.lv[l].g, g = mg.lv[l + 1].g;
    const MgGrid gx = make_grid(g.nx, f.ny, f.nz), gy = make_grid(g.nx, g.ny, f.nz);
    uint8_t* cfixed = level_flags(mg, l + 1);
    hipLaunchKernelGGL(k_mg_inject, dim3(blocks256(g.n)), dim3(256), 0, st, f, g, fixed, cfixed);
    if (l == 0)
      hipLaunchKernelGGL((k_mg_coarsen<0, true, false, double, double>), dim3(blocks256(gx.n), 27), dim3(256), 0, st, f, gx, vals,
                         fixed, cfixed, w1, (double*)nullptr);
    else
      hipLaunchKernelGGL((k_mg_coarsen<0, false, false, TM, double>), dim3(blocks256(gx.n), 27), dim3(256), 0, st, f, gx,
                         static_cast<const TM*>(mg.lv[l].A), fixed, cfixed, w1, (double*)nullptr);
    hipLaunchKernelGGL((k_mg_coarsen<1, false, false, double, double>), dim3(blocks256(gy.n), 27), dim3(256), 0, st, gx, gy, w1,
                       fixed, cfixed, w2, (double*)nullptr);
    hipLaunchKernelGGL((k_mg_coarsen<2, false, true, double, TM>), dim3(blocks256(g.n), 27), dim3(256), 0, st, gy, g, w2, fixed,
                       cfixed, static_cast<TM*>(mg.lv[l + 1].A), mg.lv[l + 1].minv);
    fixed = cfixed;
  }
}

// Power iteration on one level; which: 0 the second level's, 1 the finest one's, after it.
template <typename TM, bool FINE>
static void power(const Multigrid& mg, int l, const BellView& M, const TM* A, int which, double* partial, hipStream_t st) {
  const MgLevel& L = mg.lv[l];
  const unsigned nb = level_blocks(L.g.n);
  double *a = L.x0, *b = L.x1;
  hipLaunchKernelGGL(k_mg_power_start, dim3(blocks256(L.g.n)), dim3(256), 0, st, L.g, L.minv, a);
  for (int k = 0; k < POWER_STEPS; ++k) {
    if (level_parts(L.g.n) == 1)
      hipLaunchKernelGGL((k_mg_power<TM, FINE, 1>), dim3(nb), dim3(MgShape<1>::BS), 0, st, M, A, L.g, L.minv, a, b, partial, (int)nb);
    else
      hipLaunchKernelGGL((k_mg_power<TM, FINE, 3>), dim3(nb), dim3(MgShape<3>::BS), 0, st, M, A, L.g, L.minv, a, b, partial, (int)nb);
    std::swap(a, b);
  }
  hipLaunchKernelGGL(k_mg_power_finish, dim3(1), dim3(256), 0, st, partial, (int)nb, (int)nb, which, mg.lam);
}

template <typename TM>
void mg_setup_range(const Multigrid& mg, const BellView& M, const double* vals, const double* invd, const uint8_t* is_bc,
                    double* partial, hipStream_t st) {
  hipLaunchKernelGGL(k_mg_mask, dim3(blocks256(mg.lv[0].g.n)), dim3(256), 0, st, mg.lv[0].g.n, invd, is_bc, mg.lv[0].minv);
  coarsen<TM>(mg, 0, 1, vals, is_bc, st);
  power<TM, false>(mg, 1, BellView{}, static_cast<const TM*>(mg.lv[1].A), 0, partial, st);
  if (mg.fine_range) power<double, true>(mg, 0, M, vals, 1, partial, st);
}

template <typename TM>
void mg_setup_rest(const Multigrid& mg, hipStream_t st) {
  coarsen<TM>(mg, 1, mg.nl - 1, nullptr, level_flags(mg, 1), st);
  const MgLevel& E = mg.lv[mg.nl - 1];
  const int nt = mg_dense_tiles(E.g.n);
  hipLaunchKernelGGL(k_dense_fill<TM>, dim3((unsigned)((nt * NB + 255) / 256), (unsigned)(nt * NB)), dim3(256), 0, st, E.g, nt,
                     static_cast<const TM*>(E.A), (const double*)E.minv, mg.dense[0]);
  hipLaunchKernelGGL(k_dense_first, dim3(1), dim3(256), 0, st, mg.dense[0], mg.dpiv);
  for (int k = 0; k < nt; ++k)
    hipLaunchKernelGGL(k_dense_step, dim3((unsigned)nt, (unsigned)nt), dim3(256), 0, st, nt, k, mg.dense[k & 1],
                       mg.dense[(k & 1) ^ 1], mg.dpiv + (k & 1) * TILE, mg.dpiv + ((k & 1) ^ 1) * TILE);
}

template <typename F, typename... Args>
static inline void timed(Prof* prof, int cls, F kernel, dim3 grid, dim3 block, hipStream_t st, Args... args) {
  hipEvent_t a, b;
  if (prof_sample(prof, cls, &a, &b))
    hipExtLaunchKernelGGL(kernel, grid, block, 0, st, a, b, 0, args...);
  else
    hipLaunchKernelGGL(kernel, grid, block, 0, st, args...);
}

// Smoothing of level l from its first iterate (in x0) and the residual in r; returns the buffer of
// the last iterate.  pass: counts the passes over the finest matrix, for their direction.
template <typename TM, bool FINE, int P>
static double* smooth_level(const Multigrid& mg, int l, const BellView& M, const TM* A, const double* b, const Cheb& c, int deg,
                            const int32_t* done, int* pass, hipStream_t st, Prof* prof) {
  const MgLevel& L = mg.lv[l];
  const dim3 grid(level_blocks(L.g.n)), block(MgShape<P>::BS);
  const int cls = FINE ? PC_MG_FINE : PC_MG_COARSE;
  double *cur = L.x0, *oth = L.x1;
  for (int k = 0; k + 1 < deg; ++k) {
    timed(prof, cls, k_mg_smooth<TM, FINE, P>, grid, block, st, M, A, L.g, (const double*)L.minv, b, (const double*)cur, oth,
          k == 0 ? 1 : 0, c.c1[k], c.c2[k], (const double*)mg.lam, done, level_order(L.g.n, (*pass)++));
    std::swap(cur, oth);
  }
  timed(prof, cls, k_mg_resid<TM, FINE, P>, grid, block, st, M, A, L.g, (const double*)L.minv, b, (const double*)cur, L.r, done,
        level_order(L.g.n, (*pass)++));
  return cur;
}

// Smoothing of the finest level from its first iterate in x0, the first part of a V-cycle.
template <typename TM>
static double* smooth_fine(const Multigrid& mg, const BellView& M, const TM* vals, const double* b, const int32_t* done, int* pass,
                           hipStream_t st, Prof* prof) {
  static const Cheb cf = cheb(DEG_FINE, LOW_FINE);
  return level_parts(mg.lv[0].g.n) == 1 ? smooth_level<TM, true, 1>(mg, 0, M, vals, b, cf, DEG_FINE, done, pass, st, prof)
                                        : smooth_level<TM, true, 3>(mg, 0, M, vals, b, cf, DEG_FINE, done, pass, st, prof);
}

// The rest of the V-cycle: out = M b, from the finest level's iterate and its residual.
template <typename TM>
static void vcycle(const Multigrid& mg, const BellView& M, double* iterate, const double* invd, const double* b, double* out,
                   hipStream_t st, Prof* prof) {
  static const Cheb cc = cheb(DEG_COARSE, LOW_COARSE);
  double* cur[MG_MAXL];
  const int last = mg.nl - 1;
  cur[0] = iterate;
  for (int l = 0; l < last; ++l) {
    const MgLevel& L = mg.lv[l];
    int p = 0;
    if (l > 0) {
      const TM* A = static_cast<const TM*>(L.A);
      cur[l] = level_parts(L.g.n) == 1 ? smooth_level<TM, false, 1>(mg, l, M, A, L.b, cc, DEG_COARSE, nullptr, &p, st, prof)
                                       : smooth_level<TM, false, 3>(mg, l, M, A, L.b, cc, DEG_COARSE, nullptr, &p, st, prof);
    }
    if (l + 1 == last) break;  // the last level's kernel restricts for itself
    const MgLevel& C = mg.lv[l + 1];
    timed(prof, PC_MG_COARSE, k_mg_restrict, dim3(blocks256(C.g.n)), dim3(256), st, L.g, C.g, (const double*)L.r,
          (const double*)C.minv, C.b, C.x0, cc.ith, (const double*)mg.lam);
  }
  const MgLevel &A = mg.lv[last - 1], &E = mg.lv[last];
  const int nt = mg_dense_tiles(E.g.n);
  timed(prof, PC_MG_COARSE, k_mg_dense, dim3((unsigned)((E.g.n + 15) / 16)), dim3(256), st, A.g, E.g, nt, (const double*)A.r,
        (const double*)E.minv, (const double*)mg.dense[nt & 1], E.x0);
  const double* e = E.x0;
  for (int l = last - 1; l >= 0; --l) {
    const MgLevel& L = mg.lv[l];
    double* o = l == 0 ? out : cur[l];
    timed(prof, PC_MG_COARSE, k_mg_prolong, dim3(blocks256(L.g.n)), dim3(256), st, L.g, mg.lv[l + 1].g, e, (const double*)cur[l],
          (const double*)L.minv, b, l == 0 ? invd : (const double*)nullptr, o);
    e = o;
  }
}

// ---------------------------------------------------------------------------------
// BiCGSTAB with the V-cycle in the place of the diagonal scaling (recurrence and stopping rule of
// cp_krylov.hip's header).  Three vector kernels and two products per iteration beside the two
// cycles; sums as there: one partial per block, added by every block of the consuming kernel in
// index order.

// r0 = b - A x0 = rhat = p = q, and the partials of <r,r> (= <rhat,r>) and <b,b>.
template <int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mgb_init(BellView M, MgGrid g, const double* __restrict__ A,
                                                            const double* __restrict__ b, MgVec v, KrylovWork w, int order) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  __shared__ double sh[3 * (MgShape<P>::BS / 64)];
  int r;
  double acc, d[3] = {0.0, 0.0, 0.0};
  if (mg_row<double, true, P>(M, g, A, v.x, order, r, acc, red)) {
    const double bv = b[r], rv = bv - acc;
    v.r[r] = rv;
    v.rhat[r] = rv;
    v.p[r] = rv;
    v.q[r] = rv;
    d[0] = d[1] = rv * rv;
    d[2] = bv * bv;
  }
  put_partials<MgShape<P>::BS, 3>(d, {PS_RR, PS_RHR, PS_BB}, w.partial, w.ps, sh);
}
__global__ void __launch_bounds__(KBS) k_mgb_init2(KrylovWork w, double tol, double atol, int maxiter) {
  __shared__ double sh[KBS / 64];
  double s[1];
  get_sums<KBS, 1>(w.partial, {PS_BB}, w.ps, w.ps, sh, s);
  if (threadIdx.x == 0) {
    KrylovScalars* sc = w.sc;
    sc->bs = s[0];
    sc->atol2 = fmax(tol * tol * s[0], atol * atol);
    sc->maxiter = maxiter;
    sc->rho2[1] = sc->alpha2[1] = sc->omega2[1] = 1.0;
    sc->k2[1] = -1;
    sc->done = 0;
    sc->k = 0;
  }
}

// Convergence test of the last iteration, beta, p and the cycle's first iterate for M p.
__global__ void __launch_bounds__(KBS) k_mgb_p(MgVec v, KrylovWork w, int par, int iter, const double* __restrict__ minv,
                                              double* __restrict__ y, double ith, const double* __restrict__ lam,
                                              uint64_t* __restrict__ flag) {
  __shared__ double sh[2 * (KBS / 64)];
  // (`done` is written here and so not read: blocks of this launch would see either value)
  KrylovScalars* sc = w.sc;
  const int pv = par ^ 1;
  const double rho = sc->rho2[pv], alpha = sc->alpha2[pv], omega = sc->omega2[pv], atol2 = sc->atol2;
  const int kprev = sc->k2[pv], maxiter = sc->maxiter;
  const int64_t i0 = (int64_t)blockIdx.x * KBS + threadIdx.x;
  double sums[2];
  get_sums<KBS, 2>(w.partial, {PS_RR, PS_RHR}, iter == 0 ? w.ps : w.nb, w.ps, sh, sums);
  const double rs = sums[0], rho_ = sums[1];
  int k = (omega == 0.0 || alpha == 0.0) ? -11 : kprev + 1;
  if (rho == 0.0) k = -10;
  // A solve that is not on its way to the threshold within MG_MAXITER iterations (not the caller's own
  // limit, which may be lower) is left to the Jacobi solve: from STALL_FROM on, the squared residual has to
  // be under a straight line (in its logarithm) from a hundredfold of the first one.  See STALL_FROM for
  // what it costs without this.
  if (k >= STALL_FROM && rs > atol2) {
    const float line = log2f(fmaxf((float)(atol2 / sc->rs0), 1e-30f)) * ((float)k / (float)MG_MAXITER);
    if (log2f((float)(rs / sc->rs0)) > STALL_SLACK + line) k = -12;
  }
  const bool go = (rs > atol2) && (k < maxiter) && (k >= 0);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->k2[par] = k;
    sc->rho2[par] = rho_;
    sc->rs = rs;
    if (iter == 0) sc->rs0 = rs;
    sc->k = k;
    if (!go) sc->done = 1;
    __hip_atomic_store(flag, ((uint64_t)(iter + 1) << 33) | ((uint64_t)(go ? 0 : 1) << 32) | (uint32_t)k, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (!go) return;
  const double beta = rho_ / rho * alpha / omega, il = ith * lam[0];
  for (int64_t i = i0; i < w.n; i += (int64_t)w.nb * KBS) {
    const double p = __fma_rn(beta, __fma_rn(-omega, v.q[i], v.p[i]), v.r[i]);
    v.p[i] = p;
    y[i] = il * minv[i] * p;
  }
}

// q = A phat and the partials of <rhat,q>.
template <int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mgb_q(BellView M, MgGrid g, const double* __restrict__ A, MgVec v, KrylovWork w,
                                                         int order) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  __shared__ double sh[MgShape<P>::BS / 64];
  int r;
  double acc, d[1] = {0.0};
  if (mg_row<double, true, P>(M, g, A, v.phat, order, r, acc, red)) {
    v.q[r] = acc;
    d[0] = v.rhat[r] * acc;
  }
  put_partials<MgShape<P>::BS, 1>(d, {PS_RQ}, w.partial, w.ps, sh);
}

// alpha, s = r - alpha q and the cycle's first iterate for M s.
__global__ void __launch_bounds__(KBS) k_mgb_s(MgVec v, KrylovWork w, int par, int nbs, const double* __restrict__ minv,
                                              double* __restrict__ y, double ith, const double* __restrict__ lam) {
  __shared__ double sh[KBS / 64];
  KrylovScalars* sc = w.sc;
  double sums[1];
  get_sums<KBS, 1>(w.partial, {PS_RQ}, nbs, w.ps, sh, sums);
  const double alpha = sc->rho2[par] / sums[0], il = ith * lam[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->alpha2[par] = alpha;
  for (int64_t i = (int64_t)blockIdx.x * KBS + threadIdx.x; i < w.n; i += (int64_t)w.nb * KBS) {
    const double s = __fma_rn(-alpha, v.q[i], v.r[i]);
    v.s[i] = s;
    y[i] = il * minv[i] * s;
  }
}

// t = A shat and the partials of <s,s>, <t,s>, <t,t>.
template <int P>
__global__ void __launch_bounds__(MgShape<P>::BS) k_mgb_t(BellView M, MgGrid g, const double* __restrict__ A, MgVec v, KrylovWork w,
                                                         int order) {
  __shared__ double red[P > 1 ? (P - 1) * 64 : 1];
  __shared__ double sh[3 * (MgShape<P>::BS / 64)];
  int r;
  double acc, d[3] = {0.0, 0.0, 0.0};
  if (mg_row<double, true, P>(M, g, A, v.shat, order, r, acc, red)) {
    const double s = v.s[r];
    v.t[r] = acc;
    d[0] = s * s;
    d[1] = acc * s;
    d[2] = acc * acc;
  }
  put_partials<MgShape<P>::BS, 3>(d, {PS_SS, PS_TS, PS_TT}, w.partial, w.ps, sh);
}

// omega, x and r, and the partials of <r,r> and <rhat,r>.
__global__ void __launch_bounds__(KBS) k_mgb_xr(MgVec v, KrylovWork w, int par, int nbs) {
  __shared__ double sh[3 * (KBS / 64)];
  KrylovScalars* sc = w.sc;
  const double alpha = sc->alpha2[par], atol2 = sc->atol2;
  double sums[3];
  get_sums<KBS, 3>(w.partial, {PS_SS, PS_TS, PS_TT}, nbs, w.ps, sh, sums);
  const double omega = sums[1] / sums[2];
  const bool early = sums[0] < atol2;
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->omega2[par] = omega;
  double rr = 0.0, rhr = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * KBS + threadIdx.x; i < w.n; i += (int64_t)w.nb * KBS) {
    const double s = v.s[i];
    double r;
    if (early) {
      v.x[i] += alpha * v.phat[i];
      r = s;
    } else {
      v.x[i] += alpha * v.phat[i] + omega * v.shat[i];
      r = s - omega * v.t[i];
    }
    v.r[i] = r;
    rr += r * r;
    rhr += v.rhat[i] * r;
  }
  // (k_mgb_p adds the first w.nb partials only: nothing to clear)
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const double t0 = wave_sum(rr), t1 = wave_sum(rhr);
  if (lane == 0) {
    sh[wid] = t0;
    sh[KBS / 64 + wid] = t1;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < KBS / 64; ++i) t += sh[threadIdx.x * (KBS / 64) + i];
    w.partial[(threadIdx.x ? PS_RHR : PS_RR) * w.ps + blockIdx.x] = t;
  }
}

void mg_krylov_init(const Multigrid& mg, const BellView& M, const double* vals, const double* b, MgVec v, KrylovWork w,
                    double tol, double atol, int maxiter, hipStream_t st) {
  const MgGrid g = mg.lv[0].g;
  if (level_parts(g.n) == 1)
    hipLaunchKernelGGL(k_mgb_init<1>, dim3((unsigned)w.nbs), dim3(MgShape<1>::BS), 0, st, M, g, vals, b, v, w, level_order(g.n, 0));
  else
    hipLaunchKernelGGL(k_mgb_init<3>, dim3((unsigned)w.nbs), dim3(MgShape<3>::BS), 0, st, M, g, vals, b, v, w, level_order(g.n, 0));
  hipLaunchKernelGGL(k_mgb_init2, dim3(1), dim3(KBS), 0, st, w, tol, atol, maxiter);
}

// An iteration in two parts, so that the host can read the first one's convergence test before it
// queues the second: what a converged solve has queued in vain is then the smoothing of one level
// and not an iteration (16^3: 18 of 115 us).
template <typename TM>
void mg_krylov_begin(const Multigrid& mg, const BellView& M, const TM* valsp, MgVec v, KrylovWork w, int iter, uint64_t* flag,
                     hipStream_t st, Prof* prof) {
  const MgLevel& L = mg.lv[0];
  const double ith = cheb(DEG_FINE, LOW_FINE).ith;
  int pass = 1;  // the product that comes before walked forwards
  timed(prof, PC_KVEC, k_mgb_p, dim3((unsigned)w.nb), dim3(KBS), st, v, w, iter & 1, iter, (const double*)L.minv, L.x0, ith,
        (const double*)mg.lam, flag);
  smooth_fine<TM>(mg, M, valsp, v.p, &w.sc->done, &pass, st, prof);
}
template <typename TM>
void mg_krylov_finish(const Multigrid& mg, const BellView& M, const double* vals, const TM* valsp, MgVec v, KrylovWork w, int iter,
                      hipStream_t st, Prof* prof) {
  const MgLevel& L = mg.lv[0];
  const MgGrid g = L.g;
  const double ith = cheb(DEG_FINE, LOW_FINE).ith;
  const bool one = level_parts(g.n) == 1;
  const dim3 vb((unsigned)w.nb), vt(KBS), sb((unsigned)w.nbs), s1(MgShape<1>::BS), s3(MgShape<3>::BS);
  const int par = iter & 1;
  int pass = 1 + DEG_FINE;  // those of mg_krylov_begin
  vcycle<TM>(mg, M, (DEG_FINE - 1) & 1 ? L.x1 : L.x0, v.invd, v.p, v.phat, st, prof);
  if (one)
    timed(prof, PC_SPMV, k_mgb_q<1>, sb, s1, st, M, g, vals, v, w, level_order(g.n, pass++));
  else
    timed(prof, PC_SPMV, k_mgb_q<3>, sb, s3, st, M, g, vals, v, w, level_order(g.n, pass++));
  timed(prof, PC_KVEC, k_mgb_s, vb, vt, st, v, w, par, w.nbs, (const double*)L.minv, L.x0, ith, (const double*)mg.lam);
  double* it = smooth_fine<TM>(mg, M, valsp, v.s, &w.sc->done, &pass, st, prof);
  vcycle<TM>(mg, M, it, v.invd, v.s, v.shat, st, prof);
  if (one)
    timed(prof, PC_SPMV, k_mgb_t<1>, sb, s1, st, M, g, vals, v, w, level_order(g.n, pass++));
  else
    timed(prof, PC_SPMV, k_mgb_t<3>, sb, s3, st, M, g, vals, v, w, level_order(g.n, pass++));
  timed(prof, PC_KVEC, k_mgb_xr, vb, vt, st, v, w, par, w.nbs);
}

#define CPFEM_MG_INST(TM)                                                                                                   \
  template void mg_setup_range<TM>(const Multigrid&, const BellView&, const double*, const double*, const uint8_t*,         \
                                   double*, hipStream_t);                                                                  \
  template void mg_setup_rest<TM>(const Multigrid&, hipStream_t);                                                          \
  template void mg_krylov_begin<TM>(const Multigrid&, const BellView&, const TM*, MgVec, KrylovWork, int, uint64_t*,          \
                                    hipStream_t, Prof*);                                                                    \
  template void mg_krylov_finish<TM>(const Multigrid&, const BellView&, const double*, const TM*, MgVec, KrylovWork, int,   \
                                     hipStream_t, Prof*);
CPFEM_MG_INST(double)
CPFEM_MG_INST(float)

}  // namespace cpfem
