// Coarsest-level direct solver: sparse Cholesky L L' = P K P' in 64x64 dense
// tiles, replacing cholesky_factorization.m:26-36 (AMD ordering + CHOLMOD
// lchol) and cholesky_solve.m:27-43 (x(perm) = L'\(L\b(perm))).
//
// Ordering: geometric nested dissection of the coarse nodes (recursive
// coordinate bisection; separator = nodes of one half adjacent to the other),
// all free dofs of a node kept together.  Every leaf and separator is a block
// whose positions are padded to a multiple of 64, so tiles never straddle two
// blocks and the tile elimination structure is the dissection tree.
//
// Numeric factorisation: level-scheduled batches of tile tasks
//   update  C_IJ = A_IJ - sum_K L_IK L_JK'   (one workgroup per target tile)
//   potrf   L_JJ = chol(C_JJ) and inv(L_JJ)  (one workgroup per column)
//   trsm    L_IJ = C_IJ inv(L_JJ)'           (one workgroup per tile)
// followed by the explicit inverse X_S = inv(L_SS) of each block's diagonal
// part (recursive doubling over the block's tiles) and the products
// Z_AS = L_AS X_S with the rows A below the block.  The
// triangular solves then take one launch per tree height and direction:
//   forward:  y_S = X_S w_S  and  w_A -= Z_AS w_S     (ancestors A)
//   backward: x_S = X_S' y_S - Z_AS' x_A
// (Z_AS w_S = L_AS y_S and X_S'(y_S - L_AS' x_A) = X_S' y_S - Z_AS' x_A), each
// a batch of independent 64-row gathers.
#include "m3_internal.h"

#include <algorithm>
#include <array>
#include <functional>
#include <unordered_map>
#include <map>
#include <numeric>
#include <type_traits>

namespace {

constexpr int TS = 64;
constexpr int TT = TS * TS;
// The solves take the blocks of the first dissection levels as one, as many
// whole levels as fit into this many tiles: fewer dependent launches against a
// longer inversion, once per factorisation.  us per factorisation, and per FP64 /
// mixed iteration of the whole solver, with 0, 36, 48, 64 and 96 tiles (medians of
// two runs, which differ by 1 % and in mixed iterations by up to 4 %):
//   34 tiles in all    522   115.5/94.0    628  100/79      one block from 36 on
//   73                 898  2282/1063      978  2268/1053  1038 2267/1050  1038 2267/1051  1118 2264/1044
//   130                999   178/143      1078   170/128   1132  165/120   1177  162/118   1178  163/118
//   275               2210  1241/594      2305  1240/592   2299 1239/589   2410 1236/586   2654 1239/584
//   1,844            15,077 1641/857    15,088 1640/860  15,082 1635/854  15,076 1638/856 15,520 1635/855
// A factorisation serves 70 iterations (a step of the time loop) to a few hundred.
// 48 is a twentieth off them at 130 columns and free or nearly so elsewhere; 64
// would take another hundredth off at 130 and a third of that at 275, for a
// factorisation a twentieth longer at both.
constexpr int ROOT_TILES = 48;
constexpr int LEAF = 80;  // nodes per leaf block (40 / 80 / 160: 309 / 306 / 305 ms per c1 solve)

// ---- host: nested dissection into tile-aligned blocks ----------------------------------
struct NDState {
  const std::vector<int64_t> *ptr;
  const std::vector<int32_t> *adj;
  const std::vector<double> *xyz;
  std::vector<int32_t> stamp;
  int cur = 0;
  std::vector<std::vector<int32_t>> blocks;  // node lists in elimination order
  std::vector<int> depth;                    // dissection depth of each block (0: the first separator)
};

// Order the nodes of a block along a 3-D Morton (Z-order) curve of their
// coordinates: the nodes of a separator that border one subtree then sit in
// few 64-row tiles, which keeps the tile-level fill of the factor small.
void spatial_order(const NDState &st, std::vector<int32_t> &nodes) {
  if (nodes.size() < 2) return;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int n : nodes)
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], (*st.xyz)[3 * n + k]);
      hi[k] = std::max(hi[k], (*st.xyz)[3 * n + k]);
    }
  auto spread = [](uint64_t v) {  // 21 bits -> every third bit of 63
    v &= 0x1fffffull;
    v = (v | v << 32) & 0x1f00000000ffffull;
    v = (v | v << 16) & 0x1f0000ff0000ffull;
    v = (v | v << 8) & 0x100f00f00f00f00full;
    v = (v | v << 4) & 0x10c30c30c30c30c3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
  };
  std::vector<std::pair<uint64_t, int32_t>> key(nodes.size());
  for (size_t i = 0; i < nodes.size(); ++i) {
    uint64_t code = 0;
    for (int k = 0; k < 3; ++k) {
      const double w = hi[k] - lo[k];
      const double t = w > 0 ? ((*st.xyz)[3 * nodes[i] + k] - lo[k]) / w : 0.0;
      code |= spread((uint64_t)(t * 2097151.0)) << k;
    }
    key[i] = {code, nodes[i]};
  }
  std::sort(key.begin(), key.end());
  for (size_t i = 0; i < nodes.size(); ++i) nodes[i] = key[i].second;
}

// Minimum vertex cover of the bipartite graph between bA and bB (edges of
// the adjacency between the two sides; bB nodes carry stamp sB): Hopcroft-
// Karp maximum matching, then (bA \ Z) + (bB & Z) with Z the nodes reachable
// from unmatched bA nodes by alternating paths.  Every A-B edge has an end in
// the cover, so it separates A and B.
std::vector<int32_t> min_cover(NDState &st, const std::vector<int32_t> &bA, const std::vector<int32_t> &bB, int sB) {
  const int na = (int)bA.size(), nb = (int)bB.size();
  if (na == 0 || nb == 0) return {};
  std::unordered_map<int32_t, int> idB;
  idB.reserve(2 * nb);
  for (int j = 0; j < nb; ++j) idB[bB[j]] = j;
  std::vector<int64_t> gp(na + 1, 0);
  std::vector<int> gadj;
  for (int i = 0; i < na; ++i) {
    const int n = bA[i];
    for (int64_t k = (*st.ptr)[n]; k < (*st.ptr)[n + 1]; ++k) {
      const int m = (*st.adj)[k];
      if (st.stamp[m] != sB) continue;
      auto it = idB.find(m);
      if (it != idB.end()) gadj.push_back(it->second);
    }
    gp[i + 1] = (int64_t)gadj.size();
  }
  // Hopcroft-Karp
  std::vector<int> mA(na, -1), mB(nb, -1), dist(na);
  const int INF = 1 << 30;
  auto bfs = [&]() {
    std::vector<int> q;
    q.reserve(na);
    bool found = false;
    for (int i = 0; i < na; ++i) {
      if (mA[i] < 0) {
        dist[i] = 0;
        q.push_back(i);
      } else {
        dist[i] = INF;
      }
    }
    for (size_t h = 0; h < q.size(); ++h) {
      const int i = q[h];
      for (int64_t k = gp[i]; k < gp[i + 1]; ++k) {
        const int j = gadj[k], i2 = mB[j];
        if (i2 < 0) found = true;
        else if (dist[i2] == INF) {
          dist[i2] = dist[i] + 1;
          q.push_back(i2);
        }
      }
    }
    return found;
  };
  std::vector<int64_t> itk(na);
  std::function<bool(int)> dfs = [&](int i) -> bool {
    for (int64_t &k = itk[i]; k < gp[i + 1]; ++k) {
      const int j = gadj[k], i2 = mB[j];
      if (i2 < 0 || (dist[i2] == dist[i] + 1 && dfs(i2))) {
        mA[i] = j;
        mB[j] = i;
        ++k;
        return true;
      }
    }
    dist[i] = INF;
    return false;
  };
  while (bfs()) {
    for (int i = 0; i < na; ++i) itk[i] = gp[i];
    for (int i = 0; i < na; ++i)
      if (mA[i] < 0) dfs(i);
  }
  // Koenig: alternating reachability from unmatched bA nodes
  std::vector<char> zA(na, 0), zB(nb, 0);
  std::vector<int> q;
  for (int i = 0; i < na; ++i)
    if (mA[i] < 0) {
      zA[i] = 1;
      q.push_back(i);
    }
  for (size_t h = 0; h < q.size(); ++h) {
    const int i = q[h];
    for (int64_t k = gp[i]; k < gp[i + 1]; ++k) {
      const int j = gadj[k];
      if (zB[j] || mA[i] == j) continue;  // non-matching edges A -> B
      zB[j] = 1;
      const int i2 = mB[j];
      if (i2 >= 0 && !zA[i2]) {
        zA[i2] = 1;
        q.push_back(i2);
      }
    }
  }
  std::vector<int32_t> cover;
  for (int i = 0; i < na; ++i)
    if (!zA[i]) cover.push_back(bA[i]);
  for (int j = 0; j < nb; ++j)
    if (zB[j]) cover.push_back(bB[j]);
  return cover;
}

// Median split of `nodes` across coordinate axis `ax` into A | B and the
// minimum vertex separator S between them (S is taken out of A and B).
void split(NDState &st, std::vector<int32_t> nodes, int ax, std::vector<int32_t> &A2, std::vector<int32_t> &B2,
           std::vector<int32_t> &S) {
  const size_t mid = nodes.size() / 2;
  std::nth_element(nodes.begin(), nodes.begin() + mid, nodes.end(), [&](int a, int b) {
    const double xa = (*st.xyz)[3 * a + ax], xb = (*st.xyz)[3 * b + ax];
    return xa < xb || (xa == xb && a < b);
  });
  std::vector<int32_t> A(nodes.begin(), nodes.begin() + mid), B(nodes.begin() + mid, nodes.end());
  const int sA = ++st.cur;
  for (int n : A) st.stamp[n] = sA;
  const int sB = ++st.cur;
  for (int n : B) st.stamp[n] = sB;
  std::vector<int32_t> bA, bB;  // boundary layers
  for (int n : A) {
    for (int64_t k = (*st.ptr)[n]; k < (*st.ptr)[n + 1]; ++k)
      if (st.stamp[(*st.adj)[k]] == sB) { bA.push_back(n); break; }
  }
  for (int n : B) {
    for (int64_t k = (*st.ptr)[n]; k < (*st.ptr)[n + 1]; ++k)
      if (st.stamp[(*st.adj)[k]] == sA) { bB.push_back(n); break; }
  }
  // smallest vertex separator between the two boundary layers: a minimum
  // vertex cover of the bipartite graph of the A-B edges (Koenig: maximum
  // matching, then the alternating-path closure of the unmatched bA nodes)
  S = min_cover(st, bA, bB, sB);
  const int sS = ++st.cur;
  for (int n : S) st.stamp[n] = sS;
  A2.clear();
  B2.clear();
  for (int n : A)
    if (st.stamp[n] != sS) A2.push_back(n);
  for (int n : B)
    if (st.stamp[n] != sS) B2.push_back(n);
}

// Nested dissection: the split across the axis with the smallest separator
// (ties: the longer extent), both halves recursively, then the separator.
void nd_rec(NDState &st, std::vector<int32_t> nodes, int depth = 0) {
  if (nodes.empty()) return;
  if (nodes.size() <= (size_t)LEAF) {
    spatial_order(st, nodes);
    st.blocks.push_back(nodes);
    st.depth.push_back(depth);
    return;
  }
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int n : nodes)
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], (*st.xyz)[3 * n + k]);
      hi[k] = std::max(hi[k], (*st.xyz)[3 * n + k]);
    }
  int order[3] = {0, 1, 2};
  std::sort(order, order + 3, [&](int a, int b) { return hi[a] - lo[a] > hi[b] - lo[b]; });
  std::vector<int32_t> A2, B2, S, bestA, bestB, bestS;
  bool have = false;
  for (int ax : order) {
    if (!(hi[ax] > lo[ax])) continue;
    split(st, nodes, ax, A2, B2, S);
    if (!have || S.size() < bestS.size()) {
      bestA.swap(A2);
      bestB.swap(B2);
      bestS.swap(S);
      have = true;
    }
  }
  if (!have) {  // all nodes at one point: one block
    st.blocks.push_back(nodes);
    st.depth.push_back(depth);
    return;
  }
  spatial_order(st, bestS);
  nd_rec(st, bestA, depth + 1);
  nd_rec(st, bestB, depth + 1);
  if (!bestS.empty()) {
    st.blocks.push_back(bestS);
    st.depth.push_back(depth);
  }
}

// ---- device kernels --------------------------------------------------------------------
__global__ void k_gather(int64_t n, const int64_t *src, const int64_t *dst, const double *val,
                         double *tiles) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) tiles[dst[i]] = val[src[i]];
}

// acc(64x64) += A * B' (transB) or A * B over a list of tile pairs, A and B
// 64x64 column-major tiles staged in LDS as sA[r][c] = A(r,c) and
// sB[j][k] = B'(j,k), so that out(i,j) = sum_k sA[i][k] sB[j][k].
// On the FP64 matrix cores: 4 waves, each a 32x32 quarter
// of the 64x64 tile as 2x2 blocks of v_mfma_f64_16x16x4 (A operand: lane l
// holds A[l%16][l/16]; B operand: lane l holds B[l/16][l%16]; accumulator:
// lane l, element r holds D[l/16 + 4r][l%16], as measured on gfx950 with a
// one-wave probe).  Operands come from the
// LDS-staged tiles, 4 doubles per lane per k-step of 4 instead of 8 LDS
// reads per k for the 4x4 register tiling.
typedef double dbl4 __attribute__((ext_vector_type(4)));
struct MfAcc {
  dbl4 d[2][2];
};
__device__ inline void mf_zero(MfAcc &m) {
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) m.d[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
}
// wave w's 32x32 quarter of sA * sB' (sA[r][k], sB[c][k] in LDS) added to m
__device__ inline void mf_lds(double (*sA)[TS + 1], double (*sB)[TS + 1], MfAcc &m, int w) {
  const int lane = threadIdx.x & 63;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1), li = lane & 15, lk = lane >> 4;
#pragma unroll 4
  for (int k0 = 0; k0 < TS; k0 += 4) {
    const double a0 = sA[r0 + li][k0 + lk], a1 = sA[r0 + 16 + li][k0 + lk];
    const double b0 = sB[c0 + li][k0 + lk], b1 = sB[c0 + 16 + li][k0 + lk];
    m.d[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, m.d[0][0], 0, 0, 0);
    m.d[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, m.d[0][1], 0, 0, 0);
    m.d[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, m.d[1][0], 0, 0, 0);
    m.d[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, m.d[1][1], 0, 0, 0);
  }
}
__device__ inline void tile_mm_mf(const double *A, const double *B, bool transB, double (*sA)[TS + 1],
                                  double (*sB)[TS + 1], MfAcc &m) {
  __syncthreads();
  double va[TT / 256], vb[TT / 256];  // all 32 loads in flight before the LDS stores
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    va[q] = A[threadIdx.x + 256 * q];
    vb[q] = B[threadIdx.x + 256 * q];
  }
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q, r = t & 63, c = t >> 6;
    sA[r][c] = va[q];
    if (transB) sB[r][c] = vb[q];
    else sB[c][r] = vb[q];
  }
  __syncthreads();
  mf_lds(sA, sB, m, threadIdx.x >> 6);
}
// sum_p A_p op(B_p) over the tile pairs p0 <= p < p1 (op(B) = B' when transB);
// the loads of a pair are in flight during the products of the one before it
// (64 v_mfma_f64_16x16x4 per wave, 1.7 us).  66 KB of LDS, so that two
// workgroups share a CU and one's first loads and last stores overlap the
// other's products: one workgroup of two groups of four waves that took turns
// (133 KB) left the matrix cores idle half of a chunk of four pairs.  1,844 tile
// columns: updates 13.2 -> 11.2 ms, Z 2.42 -> 1.96 ms, the factorisation 18.16 ->
// 15.7 ms (two groups with the loads a pair further ahead: 20.1 ms; chunks that
// share a tile dealt to one XCD: 19.2 ms).
// On return sA[r][c] holds the sum, with every thread past the final barrier.
struct PairLds {
  double A[TS][TS + 1], B[TS][TS + 1];
};
__device__ inline void pair_sum(const double *Abase, const double *Bbase, const int32_t *pairs, int64_t p0,
                                int64_t p1, bool transB, PairLds &lds) {
  auto &sA = lds.A;
  auto &sB = lds.B;
  MfAcc m;
  mf_zero(m);
  double va[TT / 256], vb[TT / 256];
  auto fetch = [&](int64_t p) {
    const double *A = Abase + (int64_t)pairs[2 * p] * TT;
    const double *B = Bbase + (int64_t)pairs[2 * p + 1] * TT;
#pragma unroll
    for (int q = 0; q < TT / 256; ++q) {
      va[q] = A[threadIdx.x + 256 * q];
      vb[q] = B[threadIdx.x + 256 * q];
    }
  };
  if (p0 < p1) fetch(p0);
  for (int64_t p = p0; p < p1; ++p) {
    if (p > p0) __syncthreads();
#pragma unroll
    for (int q = 0; q < TT / 256; ++q) {
      const int t = threadIdx.x + 256 * q, r = t & 63, c = t >> 6;
      sA[r][c] = va[q];
      if (transB) sB[r][c] = vb[q];
      else sB[c][r] = vb[q];
    }
    if (p + 1 < p1) fetch(p + 1);
    __syncthreads();
    mf_lds(sA, sB, m, threadIdx.x >> 6);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1), li = lane & 15, lq = lane >> 4;
  __syncthreads();
  for (int bi = 0; bi < 2; ++bi)
    for (int bj = 0; bj < 2; ++bj)
      for (int r = 0; r < 4; ++r) sA[r0 + 16 * bi + lq + 4 * r][c0 + 16 * bj + li] = m.d[bi][bj][r];
  __syncthreads();
}

// C_IJ -= sum_pairs L_IK L_JK'  (one workgroup per chunk of at most UCH pairs
// of a target tile; chunks of one tile subtract atomically).  Factorisation of
// 34 / 275 / 1,844 tile columns with 3, 4, 6 and 8 pairs per chunk: 628 / 2,307 /
// 15,297, 621 / 2,282 / 15,363, 628 / 2,302 / 15,045 and 670 / 2,503 / 15,510 us.
constexpr int UCH = 6;
struct UpdArgs {
  const int32_t *tile;         // per chunk: target tile
  const int64_t *pbeg, *pend;  // per chunk: range of its pairs
  const int32_t *pairs;
  double *tiles;
};
__device__ inline void update_chunk(const UpdArgs &u, int ck, PairLds &lds) {
  double *C = u.tiles + (int64_t)u.tile[ck] * TT;
  pair_sum(u.tiles, u.tiles, u.pairs, u.pbeg[ck], u.pend[ck], true, lds);
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q;
    atomicAdd(C + t, -lds.A[t & 63][t >> 6]);
  }
}
__global__ __launch_bounds__(256) void k_update(UpdArgs u, int chunk0) {
  __shared__ PairLds lds;
  update_chunk(u, chunk0 + blockIdx.x, lds);
}

// 64-bit value of lane `lane` (a compile-time constant in the unrolled loops)
__device__ inline double bcast_lane(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// Cholesky of the diagonal tile and inverse of the factor, four wavefronts
// per tile, in column blocks (panels) of PB.  Wave w keeps the tile's columns
// w, w + 4, ... of row t (lane t) in registers for the whole factorisation
// (two of each panel's eight columns).  For panel kb the waves publish the
// panel columns they own through LDS; every wave
// then factors the whole panel (step j broadcasts L[kb+j][kb+j] and the
// entries L[c][kb+j] from their owning lanes with v_readlane: the four waves
// do the same arithmetic on the same values, so the panel is computed
// redundantly rather than exchanged), keeps the two panel columns it owns,
// writes its copy of the panel to its own LDS slot and updates its columns
// right of the panel with the panel rows read back as broadcasts.  Every
// entry receives its updates in ascending column order, the order of the
// unblocked right-looking elimination, with fused multiply-adds; the pivot
// is scaled by 1/sqrt(d) (one reciprocal square root per step instead of a
// square root and a division per entry).  The inverse is formed by
// recursive doubling in LDS (3.2 us instead of 8.2 us for blocked forward
// substitution, which is a chain of 64 dependent column steps): the 8x8
// diagonal blocks by substitution, then the lower-left part of each pair of
// 8-, 16- and 32-blocks as -X_CC (B X_AA).  The error flag (16: a pivot <= 0) is
// kept per lane and written once, so the elimination has no branches: with
// branches the compiler sinks the updates past later barriers and keeps the
// panel values live (512 registers and spills); an empty asm statement after
// each column's update pins it to its panel for the same reason.
constexpr int PB = 8, PW = 4;  // panel width, waves per tile

struct PotrfLds {
  double S[TS][TS + 2];   // L, row-major, rows 16-byte aligned
  union {                 // P is done with before X is begun
    double P[PW][TS][PB];   // each wave's copy of the factored panel, row c = L[c][kb..kb+7]
    double X[TS][TS + 1];   // inv(L), row-major
  };
  double RD[PW][TS];      // each wave's copy of 1 / L[c][c]
  double Tf[1024];        // B X_AA of the doubling steps
};
__device__ inline void potrf_tile(int J, double *A, const int32_t *pos2dof, double *dinv, int *err, PotrfLds &lds) {
  auto &S = lds.S;
  auto &P = lds.P;
  auto &RD = lds.RD;
  auto &X = lds.X;
  auto &Tf = lds.Tf;
  const int t = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool pr = pos2dof[J * TS + t] < 0;
  const unsigned long long padded = __ballot(pr);  // bit c: row and column c are padding
  bool bad = false;
  double v[TS / PW];  // v[q] = A[t][w + 4q]
#pragma unroll
  for (int q = 0; q < TS / PW; ++q) v[q] = A[t + TS * (w + PW * q)];
#pragma unroll
  for (int q = 0; q < TS / PW; ++q) {
    const int c = w + PW * q;
    if (pr || ((padded >> c) & 1ull)) v[q] = (t == c) ? 1.0 : 0.0;
  }
#pragma unroll
  for (int kb = 0; kb < TS; kb += PB) {
    S[t][kb + w] = v[kb / PW];
    S[t][kb + PW + w] = v[kb / PW + 1];
    __syncthreads();
    double p[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) p[j] = S[t][kb + j];
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const double d = bcast_lane(p[j], kb + j);
      bad |= !(d > 0);
      const double dd = d > 0 ? d : 1.0;
      const double r = rsqrt(dd);
      p[j] = (t == kb + j) ? dd * r : p[j] * r;
#pragma unroll
      for (int jj = j + 1; jj < PB; ++jj) p[jj] -= p[j] * bcast_lane(p[j], kb + jj);
    }
    v[kb / PW] = p[w];
    v[kb / PW + 1] = p[PW + w];
#pragma unroll
    for (int j = 0; j < PB; ++j) P[w][t][j] = p[j];
    __syncthreads();
#pragma unroll
    for (int q = (kb + PB) / PW; q < TS / PW; ++q) {
      const int c = w + PW * q;
      double l[PB];
#pragma unroll
      for (int j = 0; j < PB; ++j) l[j] = P[w][c][j];
#pragma unroll
      for (int j = 0; j < PB; ++j) v[q] -= p[j] * l[j];
      asm volatile("" : "+v"(v[q]));
    }
  }
  // L into LDS (the inverse reads rows of it) and out; the upper part of the
  // registers is never meaningful
#pragma unroll
  for (int q = 0; q < TS / PW; ++q) {
    const int c = w + PW * q;
    S[t][c] = v[q];
    A[t + TS * c] = (t >= c) ? v[q] : 0.0;
  }
  __syncthreads();
  RD[w][t] = 1.0 / S[t][t];
#pragma unroll
  for (int q = 0; q < TS / PW; ++q) X[w + PW * q][t] = 0.0;
  __syncthreads();
  // inv(L) by recursive doubling: the 8x8 diagonal blocks by substitution
  // (lane t of wave 0 forms column t of its block's inverse), then for
  // h = 8, 16, 32 every pair of h-blocks [A 0; B C] gets its lower-left part
  // -X_CC (B X_AA), through Tf; the 16- and 32-wide products on the FP64
  // matrix cores
  if (w == 0) {
    const int b0 = t & ~7;
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = b0 + i;
      double sum = 0;
#pragma unroll
      for (int k = 0; k < i; ++k) sum += S[r][b0 + k] * x[k];
      const double v = (r < t) ? 0.0 : ((r == t) ? RD[0][t] : -sum * RD[0][r]);
      x[i] = v;
      X[r][t] = v;
    }
  }
  __syncthreads();
  {  // h = 8: four pairs, one entry per thread
    const int o = threadIdx.x, pr8 = o >> 6, i = (o >> 3) & 7, j = o & 7, base = 16 * pr8;
    double sum = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) sum += S[base + 8 + i][base + k] * X[base + k][base + j];
    Tf[o] = sum;  // Tf[64 pr8 + 8i + j]
    __syncthreads();
    double u = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) u += X[base + 8 + i][base + 8 + k] * Tf[64 * pr8 + 8 * k + j];
    X[base + 8 + i][base + j] = -u;
    __syncthreads();
  }
  const int li = t & 15, lq = t >> 4;  // v_mfma_f64_16x16x4: A[li][k0 + lq], B[k0 + lq][li] -> out[lq + 4r][li]
  {  // h = 16: two pairs, one 16x16 block each (waves 0 and 1)
    const int base = 32 * w;
    dbl4 d = {0.0, 0.0, 0.0, 0.0};
    if (w < 2) {
#pragma unroll
      for (int k0 = 0; k0 < 16; k0 += 4)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(S[base + 16 + li][base + k0 + lq], X[base + k0 + lq][base + li], d,
                                                 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) Tf[256 * w + 16 * (lq + 4 * r) + li] = d[r];
    }
    __syncthreads();
    if (w < 2) {
      d = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k0 = 0; k0 < 16; k0 += 4)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(X[base + 16 + li][base + 16 + k0 + lq],
                                                 Tf[256 * w + 16 * (k0 + lq) + li], d, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) X[base + 16 + lq + 4 * r][base + li] = -d[r];
    }
    __syncthreads();
  }
  {  // h = 32: one pair, wave w takes the output block (w >> 1, w & 1)
    const int bi = w >> 1, bj = w & 1;
    dbl4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < 32; k0 += 4)
      d = __builtin_amdgcn_mfma_f64_16x16x4f64(S[32 + 16 * bi + li][k0 + lq], X[k0 + lq][16 * bj + li], d, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) Tf[32 * (16 * bi + lq + 4 * r) + 16 * bj + li] = d[r];
    __syncthreads();
    d = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < 32; k0 += 4)
      d = __builtin_amdgcn_mfma_f64_16x16x4f64(X[32 + 16 * bi + li][32 + k0 + lq], Tf[32 * (k0 + lq) + 16 * bj + li],
                                               d, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) X[32 + 16 * bi + lq + 4 * r][16 * bj + li] = -d[r];
  }
  __syncthreads();
  double *Di = dinv + (int64_t)J * TT;
#pragma unroll 4
  for (int c = w; c < TS; c += PW) Di[t + TS * c] = X[t][c];  // Di[r + 64c] = X[r][c]
  if (threadIdx.x == 0 && bad) atomicOr(err, 16);
}

// The diagonal tiles of one level of the elimination, and beside them (ncol
// workgroups, then the rest) the part of the next level's updates that does not
// wait for this level: the chunks of columns from the levels before it.  A level
// is a chain update, potrf, trsm of 25, 19 and 8 us (275 tile columns in 43
// levels) and the diagonal tiles leave nearly all CUs idle; now the chain holds
// only the update by the level just finished.  With the updates as they were then,
// factorisation of 275 tile columns 2.74 -> 2.40 ms, of 1,844 (99 levels, bound by
// the products) 18.59 -> 18.16, of 34 columns 0.64 -> 0.63.
__global__ __launch_bounds__(64 * PW) void k_potrf_update(const int32_t *cols, int ncol, const int32_t *diagtile,
                                                      const int32_t *pos2dof, double *dinv, int *err, UpdArgs u,
                                                      int chunk0) {
  __shared__ union Lds {
    PairLds upd;
    PotrfLds potrf;
    __device__ Lds() {}
  } lds;
  const int b = blockIdx.x;
  if (b < ncol) {
    const int J = cols[b];
    potrf_tile(J, u.tiles + (int64_t)diagtile[J] * TT, pos2dof, dinv, err, lds.potrf);
  } else {
    update_chunk(u, chunk0 + b - ncol, lds.upd);
  }
}

// L_IJ = C_IJ inv(L_JJ)'
__global__ __launch_bounds__(256) void k_trsm(const int32_t *tile, const int32_t *col, int task0,
                                              double *tiles, const double *dinv) {
  const int task = task0 + blockIdx.x;
  double *C = tiles + (int64_t)tile[task] * TT;
  __shared__ double sA[TS][TS + 1];
  __shared__ double sB[TS][TS + 1];
  MfAcc m;
  mf_zero(m);
  tile_mm_mf(C, dinv + (int64_t)col[task] * TT, true, sA, sB, m);
  // the product through LDS, to be written coalesced
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1), li = lane & 15, lq = lane >> 4;
  __syncthreads();
  for (int bi = 0; bi < 2; ++bi)
    for (int bj = 0; bj < 2; ++bj)
      for (int r = 0; r < 4; ++r) sA[r0 + 16 * bi + lq + 4 * r][c0 + 16 * bj + li] = m.d[bi][bj][r];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q;
    C[t] = sA[t & 63][t >> 6];  // C[r + 64c]
  }
}

// X_jj = inv(L_jj): the diagonal tiles of each block's inverse and their
// transposed copies
__global__ __launch_bounds__(256) void k_inv(const int32_t *inv_x, const int32_t *inv_row, const double *dinv,
                                             double *X, double *XT, float *X32, float *XT32) {
  const int task = blockIdx.x;
  const int64_t o = (int64_t)inv_x[task] * TT;
  const double *Di = dinv + (int64_t)inv_row[task] * TT;
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q, r = t & 63, c = t >> 6;
    const double v = Di[t];
    X[o + t] = v;
    XT[o + c + TS * r] = v;
    X32[o + t] = (float)v;
    XT32[o + c + TS * r] = (float)v;
  }
}

// One step of the recursive doubling of a block's inverse: pool tile
// out = sign * sum_p A_p P_p, A_p from Abase (the L tiles for T = B X_AA, the
// pool for X_CA = -X_CC T), P_p from the pool.  neg: the X step, which also
// writes the transposed copy and the FP32 copies.  No pairs: the tile is zero.
__global__ __launch_bounds__(256) void k_invp(const int32_t *out, const int64_t *pair_ptr, const int32_t *pairs,
                                              int task0, const double *Abase, double *X, double *XT, float *X32,
                                              float *XT32, int neg) {
  const int task = task0 + blockIdx.x;
  __shared__ PairLds lds;
  auto &sA = lds.A;
  pair_sum(Abase, X, pairs, pair_ptr[task], pair_ptr[task + 1], false, lds);
  double *O = X + (int64_t)out[task] * TT;
  double *OT = XT + (int64_t)out[task] * TT;
  const double sg = neg ? -1.0 : 1.0;
  const int64_t o = (int64_t)out[task] * TT;
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q, r = t & 63, c = t >> 6;
    const double v = sg * sA[r][c];
    O[t] = v;
    if (neg) {
      const double vt = sg * sA[c][r];  // OT[r + 64c] = O[c + 64r]
      OT[t] = vt;
      X32[o + t] = (float)v;
      XT32[o + t] = (float)vt;
    }
  }
}

// Z_Ij = sum_k L_Ik X_kj over the block's columns k >= j, and its transposed copy
__global__ __launch_bounds__(256) void k_zprod(const int32_t *z_tile, const int64_t *pair_ptr,
                                               const int32_t *pairs, const double *tiles, double *X,
                                               double *XT, float *X32, float *XT32) {
  const int task = blockIdx.x;
  __shared__ PairLds lds;
  auto &sA = lds.A;
  pair_sum(tiles, X, pairs, pair_ptr[task], pair_ptr[task + 1], false, lds);
  double *Zo = X + (int64_t)z_tile[task] * TT;
  double *ZTo = XT + (int64_t)z_tile[task] * TT;
  const int64_t o = (int64_t)z_tile[task] * TT;
#pragma unroll
  for (int q = 0; q < TT / 256; ++q) {
    const int t = threadIdx.x + 256 * q, r = t & 63, c = t >> 6;
    const double v = sA[r][c], vt = sA[c][r];
    Zo[t] = v;
    ZTo[t] = vt;
    X32[o + t] = (float)v;
    XT32[o + t] = (float)vt;
  }
}

// One 64x64 tile times a 64-vector per workgroup: item (row, mat, vcol, sel)
// adds M[mat] in0[vcol] to out0[row] (sel 0) or subtracts M[mat] in1[vcol]
// from out1[row] (sel 1); items of one row are summed atomically.
// MT: the tiles' type (the FP32 copies for the FP32 V-cycle; the products
// and the vectors stay FP64)
template <class MT>
__global__ __launch_bounds__(256) void k_gtask(const CholTiles::Item *items, int item0, const MT *mats,
                                               const double *in0, const double *in1, double *out0,
                                               double *out1) {
  const CholTiles::Item it = items[item0 + blockIdx.x];
  const int i = threadIdx.x & 63, part = threadIdx.x >> 6;  // 4 waves split the columns
  __shared__ double red[4][TS];
  const MT *M = mats + (int64_t)it.mat * TT;
  const double *vv = (it.sel ? in1 : in0) + (int64_t)it.vcol * TS;
  // all 16 loads of this thread's columns in flight before the FMAs: the
  // phases are latency-bound, not bandwidth-bound
  double mv[TS / 4], xv[TS / 4];
#pragma unroll
  for (int j = 0; j < TS / 4; ++j) {
    mv[j] = (double)M[i + TS * (part + 4 * j)];
    xv[j] = vv[part + 4 * j];
  }
  double acc = 0;
#pragma unroll
  for (int j = 0; j < TS / 4; ++j) acc += mv[j] * xv[j];
  red[part][i] = acc;
  __syncthreads();
  if (part == 0) {
    const double s = red[0][i] + red[1][i] + red[2][i] + red[3][i];
    atomicAdd((it.sel ? out1 : out0) + (int64_t)it.row * TS + i, it.sel ? -s : s);
  }
}

// right-hand side into tile order, and the forward / backward accumulators y
// and x cleared, in one pass
__global__ void k_to_tiles(int64_t npos, const int32_t *pos2dof, const double *rhs, double *w, double *y, double *x) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= npos) return;
  const int d = pos2dof[i];
  w[i] = d >= 0 ? rhs[d] : 0.0;
  y[i] = 0.0;
  x[i] = 0.0;
}

// solution back to dof order; fixed dofs (no tile position) get 0
__global__ void k_from_tiles(int64_t n, const int32_t *dof2pos, const double *x, double *out) {
  const int64_t d = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (d >= n) return;
  const int p = dof2pos[d];
  out[d] = p >= 0 ? x[p] : 0.0;
}

inline unsigned nblk(int64_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

template <class T>
void up(DBuf<T> &b, const std::vector<T> &h) {
  if (h.empty()) b.upload(std::vector<T>{T{}});
  else b.upload(h);
}

// gather items of one direction, grouped by height
struct PhaseBuilder {
  std::vector<CholTiles::Item> items;
  std::vector<int32_t> hptr{0};
  void item(int row, int mat, int vcol, int sel) { items.push_back({row, mat, vcol, sel}); }
  void end_height() { hptr.push_back((int32_t)items.size()); }
  void upload(CholTiles::Phase &p) {
    p.h_ptr = hptr;
    up(p.items, items);
  }
};

}  // namespace

namespace m3 {

// Symbolic analysis: ordering, tile structure, schedules.
void chol_analyse(m3_ctx *c) {
  LevelDev &cl = c->L[c->nmg - 1];
  CholTiles &ch = c->chol;
  const int64_t nn = cl.nnod;
  HIPCHECK(hipStreamSynchronize(c->stream));  // plain copies do not wait for the solver stream
  const std::vector<double> mask = cl.mask.to_host();
  std::vector<int64_t> ptr(nn + 1, 0);
  std::vector<int32_t> adj;
  const Sell &K = cl.K;
  for (int64_t r = 0; r < nn; ++r) {
    const int64_t base = K.base_of(r);
    for (int k = 0; k < K.h_rowlen[r]; ++k) adj.push_back(K.h_col[base + (int64_t)k * 64]);
    ptr[r + 1] = (int64_t)adj.size();
  }
  NDState st;
  st.ptr = &ptr;
  st.adj = &adj;
  st.xyz = &c->h_coord;
  st.stamp.assign(nn, 0);
  std::vector<int32_t> nodes;
  for (int64_t n = 0; n < nn; ++n)
    if (mask[3 * n] + mask[3 * n + 1] + mask[3 * n + 2] > 0) nodes.push_back((int32_t)n);
  nd_rec(st, nodes);
  // dofs of every block; the blocks of the dissection's first levels, as many
  // whole levels as fit into ROOT_TILES tiles, come last: they are factorised
  // as blocks of their own but solved as one (below)
  std::vector<std::vector<int32_t>> bdofs(st.blocks.size());
  std::vector<int> level_tiles;
  for (size_t b = 0; b < st.blocks.size(); ++b) {
    for (int n : st.blocks[b])
      for (int k = 0; k < 3; ++k)
        if (mask[3 * (int64_t)n + k] != 0.0) bdofs[b].push_back(3 * n + k);
    if ((int)level_tiles.size() <= st.depth[b]) level_tiles.resize(st.depth[b] + 1, 0);
    level_tiles[st.depth[b]] += (int)((bdofs[b].size() + TS - 1) / TS);
  }
  int root_depth = 0;
  for (int t = 0; root_depth < (int)level_tiles.size() && t + level_tiles[root_depth] <= ROOT_TILES; ++root_depth)
    t += level_tiles[root_depth];
  std::vector<int> order;
  for (int root = 0; root < 2; ++root)
    for (size_t b = 0; b < bdofs.size(); ++b)
      if ((st.depth[b] < root_depth) == (root == 1)) order.push_back((int)b);
  // positions, padded per block
  std::vector<int32_t> pos2dof, blk_t0, blk_t1;
  int64_t nfree = 0;
  int root_blk = -1;  // first block of the root
  for (int ob : order) {
    const std::vector<int32_t> &dofs = bdofs[ob];
    if (dofs.empty()) continue;
    if (root_blk < 0 && st.depth[ob] < root_depth) root_blk = (int)blk_t0.size();
    const int t0 = (int)(pos2dof.size() / TS);
    pos2dof.insert(pos2dof.end(), dofs.begin(), dofs.end());
    nfree += (int64_t)dofs.size();
    while (pos2dof.size() % TS) pos2dof.push_back(-1);
    blk_t0.push_back(t0);
    blk_t1.push_back((int)(pos2dof.size() / TS));
  }
  ch.n = nfree;
  ch.T = (int)(pos2dof.size() / TS);
  ch.nblock = (int)blk_t0.size();
  const int T = ch.T;
  std::vector<int32_t> blk_of(T);
  for (int b = 0; b < ch.nblock; ++b)
    for (int t = blk_t0[b]; t < blk_t1[b]; ++t) blk_of[t] = b;
  std::vector<int32_t> inv(3 * nn, -1);
  for (size_t i = 0; i < pos2dof.size(); ++i)
    if (pos2dof[i] >= 0) inv[pos2dof[i]] = (int32_t)i;
  // tile structure of A (lower); blocks are dense on their diagonal part
  std::vector<std::vector<int32_t>> Acol(T);
  for (int64_t n = 0; n < nn; ++n)
    for (int64_t k = ptr[n]; k < ptr[n + 1]; ++k) {
      const int m = adj[k];
      for (int a = 0; a < 3; ++a) {
        const int pa = inv[3 * n + a];
        if (pa < 0) continue;
        for (int b = 0; b < 3; ++b) {
          const int pb = inv[3 * (int64_t)m + b];
          if (pb < 0 || pa < pb) continue;
          Acol[pb / TS].push_back(pa / TS);
        }
      }
    }
  for (int J = 0; J < T; ++J) {
    for (int I = J; I < blk_t1[blk_of[J]]; ++I) Acol[J].push_back(I);
    std::sort(Acol[J].begin(), Acol[J].end());
    Acol[J].erase(std::unique(Acol[J].begin(), Acol[J].end()), Acol[J].end());
  }
  // tile-level symbolic factorisation
  std::vector<std::vector<int32_t>> S(T), children(T);
  for (int J = 0; J < T; ++J) {
    std::vector<int32_t> s = Acol[J];
    for (int Kc : children[J])
      for (int I : S[Kc])
        if (I > Kc && I >= J) s.push_back(I);
    std::sort(s.begin(), s.end());
    s.erase(std::unique(s.begin(), s.end()), s.end());
    S[J] = s;
    if (s.size() > 1) children[s[1]].push_back(J);
  }
  ch.h_colptr.assign(T + 1, 0);
  for (int J = 0; J < T; ++J) ch.h_colptr[J + 1] = ch.h_colptr[J] + (int32_t)S[J].size();
  ch.ntile = ch.h_colptr[T];
  ch.h_rowtile.clear();
  for (int J = 0; J < T; ++J) ch.h_rowtile.insert(ch.h_rowtile.end(), S[J].begin(), S[J].end());
  auto tile_of = [&](int I, int J) -> int32_t {
    const auto b = ch.h_rowtile.begin() + ch.h_colptr[J], e = ch.h_rowtile.begin() + ch.h_colptr[J + 1];
    const auto it = std::lower_bound(b, e, I);
    return (it != e && *it == I) ? (int32_t)(it - ch.h_rowtile.begin()) : -1;
  };
  std::vector<std::vector<std::pair<int32_t, int32_t>>> rows(T);  // row I: (K, t_IK), K < I
  for (int Kc = 0; Kc < T; ++Kc)
    for (int32_t t = ch.h_colptr[Kc] + 1; t < ch.h_colptr[Kc + 1]; ++t) rows[ch.h_rowtile[t]].push_back({Kc, t});
  // factorisation levels
  std::vector<int> lev(T, 0);
  int nlev = 0;
  for (int J = 0; J < T; ++J) {
    int l = 0;
    for (auto &kt : rows[J]) l = std::max(l, lev[kt.first] + 1);
    lev[J] = l;
    nlev = std::max(nlev, l + 1);
  }
  ch.nlev = nlev;
  std::vector<int32_t> lev_cols, upd_tile, trsm_tile, trsm_col, pairs;
  std::vector<int64_t> pair_beg, pair_end;
  ch.h_lev_ptr.assign(nlev + 1, 0);
  ch.h_upd_ptr.assign(2 * nlev + 1, 0);
  ch.h_trsm_ptr.assign(nlev + 1, 0);
  std::vector<std::vector<int32_t>> cols_at(nlev);
  for (int J = 0; J < T; ++J) cols_at[lev[J]].push_back(J);
  for (int l = 0; l < nlev; ++l) {
    // updates by the columns of the levels up to l - 2, then by those of l - 1
    for (int late = 0; late < 2; ++late) {
      for (int J : cols_at[l])
        for (int32_t t = ch.h_colptr[J]; t < ch.h_colptr[J + 1]; ++t) {
          const int64_t p0 = (int64_t)pairs.size() / 2;
          for (auto &kt : rows[J]) {
            if ((lev[kt.first] == l - 1) != (late == 1)) continue;
            const int32_t tIK = tile_of(ch.h_rowtile[t], kt.first);
            if (tIK >= 0) {
              pairs.push_back(tIK);
              pairs.push_back(kt.second);
            }
          }
          const int64_t p1 = (int64_t)pairs.size() / 2;
          for (int64_t b = p0; b < p1; b += UCH) {
            upd_tile.push_back(t);
            pair_beg.push_back(b);
            pair_end.push_back(std::min<int64_t>(b + UCH, p1));
          }
        }
      ch.h_upd_ptr[2 * l + late + 1] = (int32_t)upd_tile.size();
    }
    for (int J : cols_at[l]) {
      lev_cols.push_back(J);
      for (int32_t t = ch.h_colptr[J]; t < ch.h_colptr[J + 1]; ++t)
        if (ch.h_rowtile[t] != J) {
          trsm_tile.push_back(t);
          trsm_col.push_back(J);
        }
    }
    ch.h_lev_ptr[l + 1] = (int32_t)lev_cols.size();
    ch.h_trsm_ptr[l + 1] = (int32_t)trsm_tile.size();
  }
  // the solves take the root's blocks as one: its inverse factor is one set of
  // tiles, and the launches of its blocks' heights go.  The factorisation above
  // keeps them apart (independent separators run side by side).
  if (root_blk >= 0 && root_blk + 1 < ch.nblock) {
    blk_t1[root_blk] = blk_t1.back();
    blk_t0.resize(root_blk + 1);
    blk_t1.resize(root_blk + 1);
    ch.nblock = root_blk + 1;
    for (int t = blk_t0[root_blk]; t < T; ++t) blk_of[t] = root_blk;
  }
  // block heights from the structure of L: a block comes after every block
  // that has tiles in its rows
  std::vector<int> hb(ch.nblock, 0);
  for (int b = 0; b < ch.nblock; ++b) {
    int h = 0;
    for (int I = blk_t0[b]; I < blk_t1[b]; ++I)
      for (auto &kt : rows[I]) {
        const int bk = blk_of[kt.first];
        if (bk != b) h = std::max(h, hb[bk] + 1);
      }
    hb[b] = h;
  }
  int H = 0;
  for (int b = 0; b < ch.nblock; ++b) H = std::max(H, hb[b] + 1);
  ch.H = H;
  // inverse tiles of the diagonal blocks: block-local m x m, X index
  std::vector<int64_t> offX(ch.nblock + 1, 0);
  int maxm = 0;
  for (int b = 0; b < ch.nblock; ++b) {
    const int m = blk_t1[b] - blk_t0[b];
    maxm = std::max(maxm, m);
    offX[b + 1] = offX[b] + (int64_t)m * m;
  }
  ch.maxm = maxm;
  ch.nX = offX[ch.nblock];
  auto xidx = [&](int b, int i, int j) {  // global tile rows/cols i >= j in block b
    const int m = blk_t1[b] - blk_t0[b];
    return (int32_t)(offX[b] + (i - blk_t0[b]) + (int64_t)m * (j - blk_t0[b]));
  };
  std::vector<int32_t> inv_x, inv_row;
  for (int b = 0; b < ch.nblock; ++b)
    for (int i = blk_t0[b]; i < blk_t1[b]; ++i) {
      inv_x.push_back(xidx(b, i, i));
      inv_row.push_back(i);
    }
  // tiles of X that are not zero: column j of the inverse reaches the rows that
  // the columns of L reach from j (all of them in a block with a dense factor)
  std::vector<uint8_t> x_nz((size_t)ch.nX, 0);
  for (int b = 0; b < ch.nblock; ++b)
    for (int j = blk_t0[b]; j < blk_t1[b]; ++j) {
      x_nz[xidx(b, j, j)] = 1;
      for (int k = j; k < blk_t1[b]; ++k) {
        if (!x_nz[xidx(b, k, j)]) continue;
        for (int32_t t = ch.h_colptr[k]; t < ch.h_colptr[k + 1]; ++t)
          if (ch.h_rowtile[t] < blk_t1[b]) x_nz[xidx(b, ch.h_rowtile[t], j)] = 1;
      }
    }
  // Z tiles: for each block S and row tile I below it, Z_Ij = sum_k L_Ik X_kj
  // (k >= j in S); stored after the X tiles in the same pool
  std::vector<int32_t> z_tile, z_pairs;
  std::vector<int64_t> z_pair_ptr{0};
  std::vector<std::vector<std::array<int32_t, 3>>> zlist(ch.nblock);  // (I, j, pool index)
  for (int b = 0; b < ch.nblock; ++b) {
    std::vector<int32_t> below;
    for (int k = blk_t0[b]; k < blk_t1[b]; ++k)
      for (int32_t t = ch.h_colptr[k]; t < ch.h_colptr[k + 1]; ++t)
        if (ch.h_rowtile[t] >= blk_t1[b]) below.push_back(ch.h_rowtile[t]);
    std::sort(below.begin(), below.end());
    below.erase(std::unique(below.begin(), below.end()), below.end());
    for (int j = blk_t0[b]; j < blk_t1[b]; ++j)
      for (int I : below) {
        const size_t before = z_pairs.size();
        for (int k = j; k < blk_t1[b]; ++k) {
          const int32_t tl = x_nz[xidx(b, k, j)] ? tile_of(I, k) : -1;
          if (tl >= 0) {
            z_pairs.push_back(tl);
            z_pairs.push_back(xidx(b, k, j));
          }
        }
        if (z_pairs.size() == before) continue;
        const int32_t zi = (int32_t)(ch.nX + (int64_t)z_tile.size());
        z_tile.push_back(zi);
        z_pair_ptr.push_back((int64_t)z_pairs.size() / 2);
        zlist[b].push_back({I, j, zi});
      }
  }
  ch.nZ = (int64_t)z_tile.size();
  // the off-diagonal tiles of X_S = inv(L_SS) by recursive doubling over the
  // block's tile range [a, e), split at s: with A = [a, s), C = [s, e) and
  // B = L_CA,  inv([L_AA 0; B L_CC]) has lower-left part -X_CC (B X_AA).
  // Level = height of the split in the recursion (single tiles: 0); level l
  // takes two launches, T = B X_AA (products of L tiles with X tiles) and
  // X_CA = -X_CC T, so the longest chain of dependent tile products is about
  // 2 (1 + 2 + ... + m/2) ~ 2m instead of m^2/2 for row-by-row substitution.
  // T tiles that have no product are zero and left out of the second step.
  struct InvTask {
    int32_t out;
    std::vector<int32_t> pairs;
  };
  std::vector<std::vector<InvTask>> stepT, stepX;
  int64_t nT = 0;
  const int64_t t_base = ch.nX + ch.nZ;
  std::function<int(int, int, int)> double_up = [&](int b, int a, int e) -> int {
    if (e - a == 1) return 0;
    const int sp = a + (e - a) / 2;
    const int lv = 1 + std::max(double_up(b, a, sp), double_up(b, sp, e));
    if ((int)stepT.size() <= lv) {
      stepT.resize(lv + 1);
      stepX.resize(lv + 1);
    }
    const int na = sp - a;
    std::vector<int32_t> tix((size_t)(e - sp) * na, -1);  // T_ij pool index, -1: zero
    for (int i = sp; i < e; ++i)
      for (int j = a; j < sp; ++j) {
        InvTask tk;
        for (int k = j; k < sp; ++k) {
          const int32_t tl = x_nz[xidx(b, k, j)] ? tile_of(i, k) : -1;
          if (tl >= 0) {
            tk.pairs.push_back(tl);
            tk.pairs.push_back(xidx(b, k, j));
          }
        }
        if (tk.pairs.empty()) continue;
        tk.out = (int32_t)(t_base + nT++);
        tix[(size_t)(i - sp) * na + (j - a)] = tk.out;
        stepT[lv].push_back(std::move(tk));
      }
    for (int i = sp; i < e; ++i)
      for (int j = a; j < sp; ++j) {
        if (!x_nz[xidx(b, i, j)]) continue;
        InvTask tk;
        tk.out = xidx(b, i, j);
        for (int k = sp; k <= i; ++k) {
          const int32_t tt = tix[(size_t)(k - sp) * na + (j - a)];
          if (tt >= 0 && x_nz[xidx(b, i, k)]) {
            tk.pairs.push_back(xidx(b, i, k));
            tk.pairs.push_back(tt);
          }
        }
        stepX[lv].push_back(std::move(tk));
      }
    return lv;
  };
  for (int b = 0; b < ch.nblock; ++b) double_up(b, blk_t0[b], blk_t1[b]);
  ch.nT = nT;
  std::vector<int32_t> invp_out, invp_pairs;
  std::vector<int64_t> invp_pair_ptr{0};
  ch.h_invp_ptr.assign(1, 0);
  for (size_t lv = 1; lv < stepT.size(); ++lv)
    for (auto *st : {&stepT[lv], &stepX[lv]}) {
      for (auto &tk : *st) {
        invp_out.push_back(tk.out);
        invp_pairs.insert(invp_pairs.end(), tk.pairs.begin(), tk.pairs.end());
        invp_pair_ptr.push_back((int64_t)invp_pairs.size() / 2);
      }
      ch.h_invp_ptr.push_back((int32_t)invp_out.size());
    }
  // solve phases, one launch per height and direction:
  //   forward  y_S = X_S w_S  and  w_A -= Z_AS w_S   (both read the final w_S)
  //   backward x_S = X_S' y_S - Z_AS' x_A            (x_A final from the heights above)
  std::vector<std::vector<int>> blocks_at(H);
  for (int b = 0; b < ch.nblock; ++b) blocks_at[hb[b]].push_back(b);
  PhaseBuilder fw, bw;
  for (int h = 0; h < H; ++h) {
    for (int b : blocks_at[h]) {
      for (int i = blk_t0[b]; i < blk_t1[b]; ++i)
        for (int j = blk_t0[b]; j <= i; ++j)
          if (x_nz[xidx(b, i, j)]) fw.item(i, xidx(b, i, j), j, 0);
      for (auto &z : zlist[b]) fw.item(z[0], z[2], z[1], 1);
    }
    fw.end_height();
  }
  for (int h = H - 1; h >= 0; --h) {
    for (int b : blocks_at[h]) {
      for (int j = blk_t0[b]; j < blk_t1[b]; ++j)
        for (int i = j; i < blk_t1[b]; ++i)
          if (x_nz[xidx(b, i, j)]) bw.item(j, xidx(b, i, j), i, 0);
      for (auto &z : zlist[b]) bw.item(z[1], z[2], z[0], 1);
    }
    bw.end_height();
  }
  // gather map from the coarse operator values
  std::vector<int64_t> gsrc, gdst;
  for (int64_t n = 0; n < nn; ++n) {
    const int64_t base = K.base_of(n);
    for (int k = 0; k < K.h_rowlen[n]; ++k) {
      const int64_t slot = base + (int64_t)k * 64;
      const int m = K.h_col[slot];
      for (int a = 0; a < 3; ++a) {
        const int pa = inv[3 * n + a];
        if (pa < 0) continue;
        for (int b = 0; b < 3; ++b) {
          const int pb = inv[3 * (int64_t)m + b];
          if (pb < 0 || pa < pb) continue;
          const int32_t t = tile_of(pa / TS, pb / TS);
          gsrc.push_back(kval(slot, 3 * a + b));
          gdst.push_back((int64_t)t * TT + (pa % TS) + (int64_t)TS * (pb % TS));
        }
      }
    }
  }
  std::vector<int32_t> diagt(T);
  for (int J = 0; J < T; ++J) diagt[J] = ch.h_colptr[J];
  up(ch.pos2dof, pos2dof);
  up(ch.dof2pos, inv);
  up(ch.lev_cols, lev_cols);
  up(ch.upd_tile, upd_tile);
  up(ch.upd_pair_ptr, pair_beg);
  up(ch.upd_pair_end, pair_end);
  up(ch.upd_pairs, pairs);
  up(ch.trsm_tile, trsm_tile);
  up(ch.trsm_col, trsm_col);
  up(ch.inv_x, inv_x);
  up(ch.inv_row, inv_row);
  up(ch.invp_out, invp_out);
  up(ch.invp_pairs, invp_pairs);
  up(ch.invp_pair_ptr, invp_pair_ptr);
  up(ch.diagtile, diagt);
  up(ch.gsrc, gsrc);
  up(ch.gdst, gdst);
  up(ch.z_tile, z_tile);
  up(ch.z_pairs, z_pairs);
  up(ch.z_pair_ptr, z_pair_ptr);
  fw.upload(ch.fwd);
  bw.upload(ch.bwd);
  ch.tiles.alloc((size_t)ch.ntile * TT);
  ch.dinv.alloc((size_t)T * TT);
  ch.X.alloc((size_t)(ch.nX + ch.nZ + ch.nT) * TT);
  ch.XT.alloc((size_t)(ch.nX + ch.nZ) * TT);
  ch.X32.alloc((size_t)(ch.nX + ch.nZ) * TT);
  ch.XT32.alloc((size_t)(ch.nX + ch.nZ) * TT);
  for (auto *b : {&ch.w, &ch.y, &ch.x}) b->alloc((size_t)T * TS);
  c->factored = false;
}

void chol_factor(m3_ctx *c) {
  CholTiles &ch = c->chol;
  LevelDev &cl = c->L[c->nmg - 1];
  hipStream_t s = c->stream;
  ch.tiles.zero(s);
  const int64_t ng = (int64_t)ch.gsrc.n;
  hipLaunchKernelGGL(k_gather, dim3(nblk(ng)), dim3(256), 0, s, ng, ch.gsrc.p, ch.gdst.p, cl.K.val.p,
                     ch.tiles.p);
  const UpdArgs upd{ch.upd_tile.p, ch.upd_pair_ptr.p, ch.upd_pair_end.p, ch.upd_pairs.p, ch.tiles.p};
  for (int l = 0; l < ch.nlev; ++l) {
    const int u0 = ch.h_upd_ptr[2 * l + 1], u1 = ch.h_upd_ptr[2 * l + 2];
    if (u1 > u0) hipLaunchKernelGGL(k_update, dim3(u1 - u0), dim3(256), 0, s, upd, u0);
    const int c0 = ch.h_lev_ptr[l], nc = ch.h_lev_ptr[l + 1] - c0;
    const int e1 = l + 1 < ch.nlev ? ch.h_upd_ptr[2 * l + 3] : u1;
    hipLaunchKernelGGL(k_potrf_update, dim3(nc + (e1 - u1)), dim3(64 * PW), 0, s, ch.lev_cols.p + c0, nc, ch.diagtile.p,
                       ch.pos2dof.p, ch.dinv.p, c->errflag.p, upd, u1);
    const int t0 = ch.h_trsm_ptr[l], t1 = ch.h_trsm_ptr[l + 1];
    if (t1 > t0)
      hipLaunchKernelGGL(k_trsm, dim3(t1 - t0), dim3(256), 0, s, ch.trsm_tile.p, ch.trsm_col.p, t0,
                         ch.tiles.p, ch.dinv.p);
  }
  hipLaunchKernelGGL(k_inv, dim3((unsigned)ch.inv_x.n), dim3(256), 0, s, ch.inv_x.p, ch.inv_row.p, ch.dinv.p, ch.X.p,
                     ch.XT.p, ch.X32.p, ch.XT32.p);
  for (size_t st = 0; st + 1 < ch.h_invp_ptr.size(); ++st) {
    const int a = ch.h_invp_ptr[st], b = ch.h_invp_ptr[st + 1];
    const bool xstep = (st & 1) != 0;
    if (b > a)
      hipLaunchKernelGGL(k_invp, dim3(b - a), dim3(256), 0, s, ch.invp_out.p, ch.invp_pair_ptr.p, ch.invp_pairs.p, a,
                         xstep ? ch.X.p : ch.tiles.p, ch.X.p, ch.XT.p, ch.X32.p, ch.XT32.p, xstep ? 1 : 0);
  }
  if (ch.nZ > 0)
    hipLaunchKernelGGL(k_zprod, dim3((unsigned)ch.nZ), dim3(256), 0, s, ch.z_tile.p, ch.z_pair_ptr.p,
                       ch.z_pairs.p, ch.tiles.p, ch.X.p, ch.XT.p, ch.X32.p, ch.XT32.p);
  HIPCHECK(hipGetLastError());
  c->factored = true;
}

// one launch per tree height; algorithmic bytes per item: the 64x64 tile, the
// 64-vector read and the 64 accumulated outputs (read and written)
template <class MT>
static void run_phase(m3_ctx *c, hipStream_t s, CholTiles::Phase &p, int h, const MT *mats,
                      const double *in0, const double *in1, double *out0, double *out1) {
  const int a = p.h_ptr[h], b = p.h_ptr[h + 1];
  if (b > a) {
    ProfScope ps(c, 2, true, (double)(b - a) * (TT * (double)sizeof(MT) + 3.0 * TS * 8.0));
    launch_timed(k_gtask<MT>, dim3(b - a), dim3(256), s, (const CholTiles::Item *)p.items.p, a, mats, in0, in1,
                 out0, out1);
  }
}

void chol_solve_tiles(m3_ctx *c, bool tiles32) {
  CholTiles &ch = c->chol;
  hipStream_t s = c->stream;
  // the FP32 V-cycle reads the FP32 copies of the tiles (half the bytes; the
  // cycle around it carries FP32 values anyway)
  for (int h = 0; h < ch.H; ++h) {
    if (tiles32) run_phase(c, s, ch.fwd, h, (const float *)ch.X32.p, ch.w.p, ch.w.p, ch.y.p, ch.w.p);
    else run_phase(c, s, ch.fwd, h, (const double *)ch.X.p, ch.w.p, ch.w.p, ch.y.p, ch.w.p);
  }
  for (int k = 0; k < ch.H; ++k) {
    if (tiles32) run_phase(c, s, ch.bwd, k, (const float *)ch.XT32.p, ch.y.p, ch.x.p, ch.x.p, ch.x.p);
    else run_phase(c, s, ch.bwd, k, (const double *)ch.XT.p, ch.y.p, ch.x.p, ch.x.p, ch.x.p);
  }
  HIPCHECK(hipGetLastError());
}

void chol_solve_dev(m3_ctx *c, const double *rhs, double *x) {
  CholTiles &ch = c->chol;
  LevelDev &cl = c->L[c->nmg - 1];
  hipStream_t s = c->stream;
  const int64_t npos = (int64_t)ch.T * TS, n3 = 3 * cl.nnod;
  hipLaunchKernelGGL(k_to_tiles, dim3(nblk(npos)), dim3(256), 0, s, npos, ch.pos2dof.p, rhs, ch.w.p, ch.y.p, ch.x.p);
  chol_solve_tiles(c, false);
  hipLaunchKernelGGL(k_from_tiles, dim3(nblk(n3)), dim3(256), 0, s, n3, ch.dof2pos.p, ch.x.p, x);
  HIPCHECK(hipGetLastError());
}

}  // namespace m3
