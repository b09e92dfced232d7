// Banded direct solve of the Newton system for the drivers that ask for a direct solver
// ('umfpack_solver' in crystal_plasticity_OR_design/solver.py:100-101, used by
// calibration_case4_UQ_polyCrystalSteel_1D_GB.py:77,90 on a 20^3 mesh).
//
// The block-ELL matrix (Dirichlet rows already replaced by unit rows) is copied, under a node
// ordering that keeps the bandwidth small (the mesh's own order or reverse Cuthill-McKee,
// whichever is narrower), into a band of dense NB x NB tiles, factored without pivoting, and
// solved with matrix-vector sweeps.  FP64 iterative refinement against the block-ELL matrix
// follows in the caller.  Without pivoting the factorisation exists when the leading principal
// minors (in the order of elimination) are non-zero, which holds for these stiffness matrices
// (elastic-plastic tangents close to SPD, unit Dirichlet rows).  A zero or non-finite pivot is
// reported instead of being worked round: the caller factors once more with one front (nt = 0), as it
// does where the solution's backward error is large, and turns a second one into an error.
//
// A band of 1400 half bandwidth gives each pivot block only about a thousand tiles of work, so
// the solve is bound by the length of the chain of dependent launches, not by operations
// (20^3: 27783 rows, 107 GFLOP, 1.5 ms at the FP64 rate).  The chain is kept short by
//  - elimination from both ends of the band at once (two independent fronts, which meet in a
//    middle part of at least two half bandwidths that the first front then finishes): 239
//    steps at 20^3 where one front has 435;
//  - one launch per pivot block: tiles keep A_IK and A_KJ as they are and the inverse of the
//    pivot block, A_IJ -= (A_IK A_KK^-1) A_KJ, so no launch has to solve the panel first, and
//    the workgroup that finishes the next diagonal tile inverts it in the same launch;
//  - sweeps over superblocks of SUP tiles: V_I = A_IS L_S^-1 and Q_J = U_S^-1 A_SJ are formed
//    once in the factor's place (k_band_super), after which a forward sweep is
//    y_I -= V_I y_S, one product with each superblock's own inverse, and y_S -= Q_SJ y_J, one
//    matrix-vector launch per superblock.
// 20^3 on an MI355X, factor and three solves: 128.6 ms with 32-wide panels from one end (four
// launches a panel, two per panel in each sweep), 8.2 ms like this (steps 5.7, sweeps 1.8, superblocks 0.55).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <deque>
#include <vector>

#include "cp_tiles.hpp"

namespace cpfem {

constexpr int SUP = BAND_SUP;

// Tile (I, J), row-major, |J - I| <= hw.
__device__ __forceinline__ double* band_tile(const BandLU& B, int I, int J) {
  return B.band + ((int64_t)I * (2 * B.hw + 1) + (J - I + B.hw)) * TILE;
}

// Copy of the block-ELL matrix into the tiles under the node map ip (old -> new); unit rows
// fill the last tile.
__global__ void k_band_scatter(BellView M, const double* __restrict__ vals, BandLU B) {
  const int64_t n = 3 * M.n_nodes;
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= (int64_t)NB * B.nbk) return;
  if (r >= n) {
    band_tile(B, B.nbk - 1, B.nbk - 1)[(r % NB) * (NB + 1)] = 1.0;
    return;
  }
  const int64_t i = r / 3;
  const int c = (int)(r - 3 * i);
  const int64_t R = 3 * (int64_t)B.ip[i] + c;
  const int I = (int)(R / NB);
  const int ns = M.nslot[i];
  for (int s = 0; s < ns; ++s) {
    const int64_t j = M.col[(int64_t)s * M.n_nodes + i];
    const int64_t C0 = 3 * (int64_t)B.ip[j];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      band_tile(B, I, (int)((C0 + k) / NB))[(R % NB) * NB + (C0 + k) % NB] = vals[(3 * (int64_t)s + k) * n + r];
  }
}

// The first pivot block of each front.
__global__ void __launch_bounds__(256) k_band_first(BandLU B) {
  __shared__ InvLds s;
  const int K = blockIdx.x ? B.nbk - 1 : 0, w = threadIdx.x >> 6, l = threadIdx.x & 63;
  double* g = band_tile(B, K, K);
  v4d a[4];
  load_d(a, g, w, l);
  if (tile_inverse(a, s)) B.flag[0] = 1;
  store_d(a, g, w, l);
}

// Elimination step t of both fronts (blockIdx.y; front 1 runs from the last tile upwards): for
// the pivot block K, whose tile (K, K) already holds its inverse, A_IJ -= (A_IK A_KK^-1) A_KJ over
// the cnt x cnt tiles ahead.  Workgroup 0 takes the tile of the next pivot and inverts it; the
// others take `group` tiles of one row I, so that A_IK A_KK^-1 is formed once for them.
// The tiles after the current one are loaded under its product.  At cnt = 22 a step of one front
// takes 19 us, of which the chain through workgroup 0 is 17 (launch 2, loads 1.4, two products 4,
// inverse 9); two fronts take 25 us, with 62 MB of tiles read and written.  (Visiting a tile in every
// second step only, for two pivots, halves that traffic and takes 32 us: the second inverse's
// product comes before the first tile's.)
__global__ void __launch_bounds__(256, 2) k_band_step(BandLU B, int t, int cnt, int group) {
  __shared__ double S[2][TILE];
  const int f = blockIdx.y, dir = f ? -1 : 1, K = f ? B.nbk - 1 - t : t;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  int i = 0, j0 = 0, j1 = 1;
  if (blockIdx.x > 0) {
    const int ng = (cnt + group - 1) / group, b = blockIdx.x - 1;
    i = b / ng;
    j0 = (b - i * ng) * group;
    j1 = min(j0 + group, cnt);
    if (i == 0 && j0 == 0) j0 = 1;
    if (j0 >= j1) return;
  }
  const int I = K + dir * (1 + i);
  Stage st;
  st.load(band_tile(B, K, K));
  double x[16];
  {
    const double* g = band_tile(B, I, K) + (16 * w + l % 16) * NB + l / 16;
#pragma unroll
    for (int k = 0; k < 16; ++k) x[k] = g[4 * k];
  }
  st.store(S[0]);
  st.load(band_tile(B, K, K + dir * (1 + j0)));
  v4d c[4];
  load_d(c, band_tile(B, I, K + dir * (1 + j0)), w, l);
  __syncthreads();
  {
    v4d acc[4] = {};
    mul_chain<NB>(acc, x, S[0], l);
#pragma unroll
    for (int k = 0; k < 16; ++k) x[k] = -acc[k / 4][k % 4];
  }
  st.store(S[1]);
  __syncthreads();
  if (blockIdx.x > 0) {
    for (int j = j0, b = 1; j < j1; ++j, b ^= 1) {
      const int J = K + dir * (1 + j);
      const bool more = j + 1 < j1;
      v4d next[4];
      if (more) {
        st.load(band_tile(B, K, J + dir));
        load_d(next, band_tile(B, I, J + dir), w, l);
      }
      mul_last<NB>(c, x, S[b], l);
      store_d(c, band_tile(B, I, J), w, l);
      if (more) {
        st.store(S[b ^ 1]);  // last read before the previous barrier
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = next[k];
      }
    }
    return;
  }
  mul_last<NB>(c, x, S[1], l);
  // the second front's last tile belongs to the middle part, which is eliminated later
  if (!(f == 1 && t == B.nt - 1)) {
    static_assert(sizeof(InvLds) <= sizeof(S[0]), "");  // S[0] is free since the second barrier
    if (tile_inverse(c, *reinterpret_cast<InvLds*>(S[0]))) B.flag[0] = 1;
  }
  store_d(c, band_tile(B, I, I), w, l);
}

// Superblock u: its pivot blocks p0 + dir a, a < s, and the number of later blocks it reaches.
// The first front's come first, then the middle part's, then the second front's.
struct Super {
  int p0, dir, s, cnt;
  __device__ __forceinline__ int block(int a) const { return p0 + dir * a; }
};
__device__ __forceinline__ Super band_super(const BandLU& B, int u) {
  const int na = (B.nt + B.sup - 1) / B.sup, mid = B.nbk - 2 * B.nt, nm = (mid + B.sup - 1) / B.sup;
  Super S;
  int off, len;
  if (u < na || u >= na + nm) {
    off = (u < na ? u : u - na - nm) * B.sup;
    len = B.nt;
    S.p0 = u < na ? off : B.nbk - 1 - off;
    S.dir = u < na ? 1 : -1;
  } else {
    off = (u - na) * B.sup;
    len = mid;
    S.p0 = B.nt + off;
    S.dir = 1;
  }
  S.s = min(B.sup, len - off);
  const int last = S.block(S.s - 1);
  S.cnt = min(B.wb, S.dir > 0 ? B.nbk - B.nt - 1 - last : last - B.nt);
  return S;
}

// V_I = A_IS L_S^-1 (blockIdx.z = 0) and Q_J = U_S^-1 A_SJ (1) for one tile row or column beyond
// superblock blockIdx.y, in place of A_IS and A_SJ, where L_S has the pivot blocks on its diagonal
// and U_S units: block back substitution, last pivot first,
//   V_a = (A_Ia - sum_{m > a} V_m A_ma) D_a^-1,   Q_a = D_a^-1 (A_aJ - sum_{m > a} A_am Q_m).
// Q is formed transposed, with the tiles of S transposed on their way to LDS.  Bound by the matrix
// cores: 0.55 ms at 20^3, ten products for each of 4800 strips, 0.32 ms at their FP64 rate.
template <bool Q>
__device__ __forceinline__ void super_strip(const BandLU& B, const Super& S, int I, double* sh) {
  constexpr int P = Q ? NB + 1 : NB;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const auto tile = [&](int r, int c) { return Q ? band_tile(B, c, r) : band_tile(B, r, c); };
  // operand layout: element (16 w + l % 16, 4 k + l / 16) of the (transposed) strip tile
  const int o = Q ? (l / 16) * NB + 16 * w + l % 16 : (16 * w + l % 16) * NB + l / 16, os = Q ? 4 * NB : 4;
  const auto stage = [&](const double* g) {
    Stage st;
    st.load(g);
    __syncthreads();  // the tile before has been read
    if (Q)
      st.store_transposed<P>(sh);
    else
      st.store(sh);
    __syncthreads();
  };
  double x[SUP][16];
#pragma unroll
  for (int a = SUP - 1; a >= 0; --a) {
    if (a >= S.s) continue;
    double* g = tile(I, S.block(a));
    v4d acc[4];
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[k / 4][k % 4] = g[o + os * k];
#pragma unroll
    for (int m = SUP - 1; m > a; --m) {
      if (m >= S.s) continue;
      stage(tile(S.block(m), S.block(a)));
      mul_chain<P>(acc, x[m], sh, l);
    }
    double y[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) y[k] = acc[k / 4][k % 4];
    stage(band_tile(B, S.block(a), S.block(a)));
    v4d v[4] = {};
    mul_chain<P>(v, y, sh, l);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      g[o + os * k] = v[k / 4][k % 4];
      x[a][k] = -v[k / 4][k % 4];
    }
  }
}

__global__ void __launch_bounds__(256, 2) k_band_super(BandLU B) {
  __shared__ double sh[NB * (NB + 1)];
  const Super S = band_super(B, blockIdx.y);
  if ((int)blockIdx.x >= S.cnt) return;
  const int I = S.block(S.s + blockIdx.x);
  if (blockIdx.z)
    super_strip<true>(B, S, I, sh);
  else
    super_strip<false>(B, S, I, sh);
}

// ---- sweeps: one launch per superblock, 4.9 us each, nearly all of it the launch and one trip to
// memory (2.9 MB of tiles a front); tile by tile they were four times as many.  16 threads a row, 16 rows a workgroup (4 workgroups a tile row); a thread reads
// two 16-byte pieces of each tile's row, and all of a launch's reads are in flight together.
// y_I -= V_I y_S for the tile rows that superblock u0 (and, blockIdx.y = 1, u1) reaches.
__global__ void __launch_bounds__(256) k_band_fwd(BandLU B, int u0, int u1) {
  const Super S = band_super(B, blockIdx.y ? u1 : u0);
  const int x = blockIdx.x / 4;
  if (x >= S.cnt) return;
  const int I = S.block(S.s + x), r = (blockIdx.x % 4) * 16 + threadIdx.x / 16, sub = threadIdx.x % 16;
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < SUP; ++a)
    if (a < S.s) acc += row_dot(band_tile(B, I, S.block(a)) + r * NB, B.y + (int64_t)NB * S.block(a), sub);
  acc = sum16(acc);
  if (sub == 0) B.y[(int64_t)NB * I + r] -= acc;
}

// y_S = A_SS^-1 y_S (of the partly eliminated matrix) for every superblock: forward and backward
// substitution over its tiles.
__global__ void __launch_bounds__(256) k_band_mid(BandLU B) {
  __shared__ double y[SUP][NB];
  __shared__ double z[NB];
  const Super S = band_super(B, blockIdx.x);
  const int tid = threadIdx.x, sub = tid % 16;
  for (int e = tid; e < NB * S.s; e += 256) y[e / NB][e % NB] = B.y[(int64_t)NB * S.block(e / NB) + e % NB];
  __syncthreads();
  // z = (accumulated rows of tile row a), then y_a from D_a^-1 z
  const auto times = [&](const double* g, const double* v, int k) { return row_dot(g + (16 * k + tid / 16) * NB, v, sub); };
  for (int a = 0; a < S.s; ++a) {
    for (int k = 0; k < 4; ++k) {
      double acc = 0.0;
      for (int j = 0; j < a; ++j) acc += times(band_tile(B, S.block(a), S.block(j)), y[j], k);
      acc = sum16(acc);
      if (sub == 0) z[16 * k + tid / 16] = y[a][16 * k + tid / 16] - acc;
    }
    __syncthreads();
    for (int k = 0; k < 4; ++k) {
      const double v = sum16(times(band_tile(B, S.block(a), S.block(a)), z, k));
      if (sub == 0) y[a][16 * k + tid / 16] = v;
    }
    __syncthreads();
  }
  for (int a = S.s - 2; a >= 0; --a) {
    for (int k = 0; k < 4; ++k) {
      double acc = 0.0;
      for (int j = a + 1; j < S.s; ++j) acc += times(band_tile(B, S.block(a), S.block(j)), y[j], k);
      acc = sum16(acc);
      if (sub == 0) z[16 * k + tid / 16] = acc;
    }
    __syncthreads();
    for (int k = 0; k < 4; ++k) {
      const double v = sum16(times(band_tile(B, S.block(a), S.block(a)), z, k));
      if (sub == 0) y[a][16 * k + tid / 16] -= v;
    }
    __syncthreads();
  }
  for (int e = tid; e < NB * S.s; e += 256) B.y[(int64_t)NB * S.block(e / NB) + e % NB] = y[e / NB][e % NB];
}

// y_K -= Q_KJ y_J for the tile rows K that reach superblock u0 (blockIdx.y = 1: u1) and were
// eliminated before it: those behind it within hw, and, for a superblock of the middle part, those
// of the second front too.  Tiles between a superblock's reach and hw are zero.
__global__ void __launch_bounds__(256) k_band_bwd(BandLU B, int u0, int u1) {
  const Super S = band_super(B, blockIdx.y ? u1 : u0);
  const int x = blockIdx.x / 4;
  const bool mid = S.p0 >= B.nt && S.p0 < B.nbk - B.nt;
  int K;
  if (x < B.hw)
    K = S.p0 - S.dir * (1 + x);
  else {
    K = B.nbk - B.nt + x - B.hw;
    if (!mid || K - S.block(S.s - 1) > B.hw) return;
  }
  if (K < 0 || K >= B.nbk) return;
  const int r = (blockIdx.x % 4) * 16 + threadIdx.x / 16, sub = threadIdx.x % 16;
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < SUP; ++a) {
    const int J = S.block(a);
    if (a < S.s && abs(K - J) <= B.hw) acc += row_dot(band_tile(B, K, J) + r * NB, B.y + (int64_t)NB * J, sub);
  }
  acc = sum16(acc);
  if (sub == 0) B.y[(int64_t)NB * K + r] -= acc;
}

// y[new order] = in[old order], zeros beyond the matrix (dir = 0) or out[old] = y[new] (dir = 1),
// dof-wise.
__global__ void k_band_perm(BandLU B, const double* __restrict__ in, double* __restrict__ out, int dir) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= B.n) {
    if (dir == 0 && r < (int64_t)NB * B.nbk) B.y[r] = 0.0;
    return;
  }
  const int64_t i = r / 3;
  const int64_t R = 3 * (int64_t)B.ip[i] + (r - 3 * i);
  if (dir == 0)
    B.y[R] = in[r];
  else
    out[r] = B.y[R];
}

// ---------------------------------------------------------------------------------- host

// Largest |ip[i] - ip[j]| over the node graph.
static int node_bandwidth(int64_t nn, const int32_t* col, const int32_t* nslot, const std::vector<int32_t>& ip) {
  int64_t bw = 0;
  for (int64_t i = 0; i < nn; ++i)
    for (int s = 0; s < nslot[i]; ++s) {
      const int64_t j = col[(size_t)s * nn + i];
      bw = std::max<int64_t>(bw, std::llabs((int64_t)ip[i] - ip[j]));
    }
  return (int)bw;
}

// Breadth-first level structure from `start` over unvisited nodes; returns the last level.
static std::vector<int32_t> bfs_last_level(int64_t nn, const int32_t* col, const int32_t* nslot, int32_t start,
                                           const std::vector<char>& taken, int* depth) {
  std::vector<int32_t> lev(nn, -1);
  std::vector<int32_t> cur{start}, last{start};
  lev[start] = 0;
  int d = 0;
  while (!cur.empty()) {
    last = cur;
    std::vector<int32_t> nxt;
    for (int32_t u : cur)
      for (int s = 0; s < nslot[u]; ++s) {
        const int32_t v = col[(size_t)s * nn + u];
        if (lev[v] < 0 && !taken[v]) {
          lev[v] = d + 1;
          nxt.push_back(v);
        }
      }
    cur.swap(nxt);
    if (!cur.empty()) ++d;
  }
  *depth = d;
  return last;
}

int band_ordering(int64_t nn, const int32_t* col, const int32_t* nslot, int32_t* ip_out, int32_t* bw_out) {
  // candidate 1: the mesh's own order
  std::vector<int32_t> ident(nn);
  for (int64_t i = 0; i < nn; ++i) ident[i] = (int32_t)i;
  const int bw0 = node_bandwidth(nn, col, nslot, ident);
  // candidate 2: reverse Cuthill-McKee from a pseudo-peripheral node of each component
  std::vector<int32_t> deg(nn);
  for (int64_t i = 0; i < nn; ++i) deg[i] = nslot[i];
  std::vector<char> taken(nn, 0);
  std::vector<int32_t> order;
  order.reserve(nn);
  while ((int64_t)order.size() < nn) {
    int32_t start = -1;
    for (int64_t i = 0; i < nn; ++i)
      if (!taken[i] && (start < 0 || deg[i] < deg[start])) start = (int32_t)i;
    int depth = 0, prev = -1;
    for (int it = 0; it < 4 && depth > prev; ++it) {  // pseudo-peripheral node (George-Liu)
      prev = depth;
      std::vector<int32_t> last = bfs_last_level(nn, col, nslot, start, taken, &depth);
      if (depth <= prev) break;
      int32_t best = last[0];
      for (int32_t v : last)
        if (deg[v] < deg[best]) best = v;
      start = best;
    }
    std::deque<int32_t> q{start};
    taken[start] = 1;
    while (!q.empty()) {
      const int32_t u = q.front();
      q.pop_front();
      order.push_back(u);
      std::vector<int32_t> nb;
      for (int s = 0; s < nslot[u]; ++s) {
        const int32_t v = col[(size_t)s * nn + u];
        if (!taken[v]) {
          taken[v] = 1;
          nb.push_back(v);
        }
      }
      std::sort(nb.begin(), nb.end(), [&](int32_t a, int32_t b) { return deg[a] < deg[b] || (deg[a] == deg[b] && a < b); });
      for (int32_t v : nb) q.push_back(v);
    }
  }
  std::vector<int32_t> ip(nn);
  for (int64_t k = 0; k < nn; ++k) ip[order[nn - 1 - k]] = (int32_t)k;
  const int bw1 = node_bandwidth(nn, col, nslot, ip);
  const std::vector<int32_t>& best = bw1 < bw0 ? ip : ident;
  std::copy(best.begin(), best.end(), ip_out);
  *bw_out = std::min(bw0, bw1);
  return 0;
}

void band_shape(BandLU& B, int64_t n, int bw, double cap) {
  B.n = n;
  const int kl = 3 * bw + 2;
  B.nbk = (int)((n + NB - 1) / NB);
  B.wb = std::min((kl + NB - 1) / NB, B.nbk - 1);
  // a superblock's last tile reaches wb tiles on, and its first tile's row and column then store
  // that far too; where that room is above the cap, sweeps go tile by tile
  for (int sup : {SUP, 1}) {
    B.sup = sup;
    B.hw = B.wb + sup - 1;
    B.room = (int64_t)B.nbk * (2 * B.hw + 1) * TILE;
    if ((double)B.room * sizeof(double) <= cap) break;
  }
  B.nt = std::max(0, (B.nbk - 2 * B.wb) / 2);
}

void band_assemble(const BandLU& B, const BellView& M, const double* vals, hipStream_t st) {
  (void)hipMemsetAsync(B.band, 0, (size_t)B.room * sizeof(double), st);
  hipLaunchKernelGGL(k_band_scatter, dim3((unsigned)((NB * (int64_t)B.nbk + 255) / 256)), dim3(256), 0, st, M, vals, B);
}

void band_factor(const BandLU& B, hipStream_t st) {
  (void)hipMemsetAsync(B.flag, 0, sizeof(int32_t), st);
  hipLaunchKernelGGL(k_band_first, dim3(B.nt > 0 ? 2 : 1), dim3(256), 0, st, B);
  for (int t = 0; t + 1 < B.nbk - B.nt; ++t) {
    const int fronts = t < B.nt ? 2 : 1, cnt = std::min(B.wb, B.nbk - B.nt - 1 - t);
    // tiles of a row per workgroup: the fewest that leave each CU one workgroup, at most 8 (cnt =
    // 22, two fronts: 5; with 4, 266 workgroups share CUs and a step takes 35 us instead of 29)
    int group = 1;
    while (group < 8 && fronts * (1 + cnt * ((cnt + group - 1) / group)) > 256) ++group;
    hipLaunchKernelGGL(k_band_step, dim3(1 + cnt * ((cnt + group - 1) / group), fronts), dim3(256), 0, st, B, t, cnt, group);
  }
  const int na = (B.nt + B.sup - 1) / B.sup, nm = (B.nbk - 2 * B.nt + B.sup - 1) / B.sup;
  if (B.wb > 0) hipLaunchKernelGGL(k_band_super, dim3(B.wb, 2 * na + nm, 2), dim3(256), 0, st, B);
}

void band_solve(const BandLU& B, const double* b, double* x, hipStream_t st) {
  const unsigned g = (unsigned)((NB * (int64_t)B.nbk + 255) / 256);
  const int na = (B.nt + B.sup - 1) / B.sup, nm = (B.nbk - 2 * B.nt + B.sup - 1) / B.sup;
  hipLaunchKernelGGL(k_band_perm, dim3(g), dim3(256), 0, st, B, b, x, 0);
  // superblocks na + nm + u of the second front go with u of the first
  for (int u = 0; u + 1 < na + nm; ++u)
    hipLaunchKernelGGL(k_band_fwd, dim3(4 * B.wb, u < na ? 2 : 1), dim3(256), 0, st, B, u, na + nm + u);
  hipLaunchKernelGGL(k_band_mid, dim3(2 * na + nm), dim3(256), 0, st, B);
  for (int u = na + nm - 1; u > 0; --u)
    hipLaunchKernelGGL(k_band_bwd, dim3(4 * (u < na ? B.hw : B.hw + std::min(B.hw, B.nt)), u < na ? 2 : 1), dim3(256), 0, st, B,
                       u, na + nm + u);
  hipLaunchKernelGGL(k_band_perm, dim3(g), dim3(256), 0, st, B, b, x, 1);
}

}  // namespace cpfem
