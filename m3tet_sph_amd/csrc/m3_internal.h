// Internal declarations of libm3stokes: device buffers, sliced block-sparse
// storage, per-level state, kernel launchers.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/m3stokes.h"

typedef struct m3_gnn m3_gnn;

struct M3Error : std::runtime_error {
  int code;
  M3Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define HIPCHECK(x)                                                                  \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess)                                                            \
      throw M3Error(M3_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_));      \
  } while (0)

#define M3_REQUIRE(cond, code, msg)                                                  \
  do {                                                                               \
    if (!(cond)) throw M3Error((code), (msg));                                       \
  } while (0)

namespace m3 {
// message of the last failed context-free call on this thread (m3_last_error(NULL))
const char *context_free_error();
void set_context_free_error(const char *msg);
// first-appearance numbering of n bars (2 n int32 node indices, device):
// d_bar_of[i] = number of bar i's unique bar, d_first[u] = position of the
// first occurrence of unique bar u (room for n); returns the unique count
int64_t unique_bars_device(const int32_t *dbars, int64_t n, int64_t *d_first, int64_t *d_bar_of, hipStream_t s);
// d_firstpos[i] = smallest position whose key equals key i (device arrays)
void first_position_device(const unsigned long long *dkeys, int64_t n, int64_t *d_firstpos, hipStream_t s);
// exclusive prefix sum of n int64 on the device; returns the total
int64_t exclusive_scan_device(const int64_t *d_x, int64_t n, int64_t *d_out, hipStream_t s);
}  // namespace m3

template <class T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  DBuf(DBuf &&o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
  DBuf &operator=(DBuf &&o) noexcept {
    if (this != &o) { release(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; }
    return *this;
  }
  ~DBuf() { release(); }
  void alloc(size_t count) {
    release();
    n = count;
    if (count) HIPCHECK(hipMalloc(&p, count * sizeof(T)));
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void upload(const T *h, size_t count) {
    if (count != n) alloc(count);
    if (count) HIPCHECK(hipMemcpy(p, h, count * sizeof(T), hipMemcpyHostToDevice));
  }
  void upload(const std::vector<T> &h) { upload(h.data(), h.size()); }
  void download(T *h, size_t count) const {
    if (count) HIPCHECK(hipMemcpy(h, p, count * sizeof(T), hipMemcpyDeviceToHost));
  }
  std::vector<T> to_host() const {
    std::vector<T> h(n);
    download(h.data(), n);
    return h;
  }
  void zero(hipStream_t s) {
    if (n) HIPCHECK(hipMemsetAsync(p, 0, n * sizeof(T), s));
  }
};

// Sliced (SELL-64) block-sparse storage.  Rows are grouped in slices of 64 (one
// wavefront); inside a slice the k-th stored block of each row sits at slot
// slice_ptr[s] + 64*k + (position % 64), so the 64 lanes of a wave touch 64
// consecutive slots.  Matrices with fewer than nine values per block store
// them structure-of-arrays, val[v*nslot + slot]; the 3x3 operators store each
// group of 64 slots contiguously (kval).  Columns inside a row are sorted.
//
// Rows may be placed in the slices in another order than their index:
// position q of the slices holds row perm[q], row r sits at position
// ipos[r]; both are NULL for the identity placement.  rowlen is indexed by row.
template <class T>
struct SellT {
  const int64_t *slice_ptr;
  const int32_t *rowlen;
  const int32_t *col;
  T *val;
  int64_t nslot;
  const int32_t *perm;  // position -> row (NULL: identity)
  const int32_t *ipos;  // row -> position (NULL: identity)
};
using SellView = SellT<double>;

// Index of value v (row-major in the 3x3 block) of slot p in a 3x3 operator:
// the 64 slots of a group hold their 576 doubles together, values (0,1),
// (2,3), (4,5), (6,7) as one 16-byte pair per lane and value 8 behind them, so
// that a wave reads a group in four 16-byte and one 8-byte load per lane from
// one contiguous stretch
__host__ __device__ inline int64_t kval(int64_t p, int v) {
  const int64_t lane = p & 63;
  return 9 * (p - lane) + (v < 8 ? 128 * (v >> 1) + 2 * lane + (v & 1) : 512 + lane);
}
// The same for the packed BF16 copy of the mixed V-cycle, in 32-bit words: the
// group's 64 lanes hold (v0..v7) as four words of two BF16 each (v_2i in the
// low half), then v8 in FP32: 20 bytes per block
constexpr int P16 = 5;  // words per slot
__host__ __device__ inline int64_t p16_words(int64_t p) { return P16 * (p & ~(int64_t)63) + 4 * (p & 63); }
__host__ __device__ inline int64_t p16_v8(int64_t p) { return P16 * (p & ~(int64_t)63) + 256 + (p & 63); }

// BF16 bits of x rounded to nearest even (through FP32)
__device__ inline uint32_t bf16_rne(double x) {
  uint32_t u = __float_as_uint((float)x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

// slot of the first block of row `row`; block k is at + 64 k
template <class T>
__device__ inline int64_t sell_base(const SellT<T> &K, int64_t row) {
  const int64_t q = K.ipos ? (int64_t)K.ipos[row] : row;
  return K.slice_ptr[q >> 6] + (q & 63);
}

// What a sweep reads of a 3x3 operator besides its values (k_sparse.hip).
// Without windows the rows are in index order and col holds their columns.
// With windows the vectors are in a space-filling order of the nodes; window b
// is the rows at the places win[b].x .. win[b+1].x of it (from a multiple of 64
// on, at most 512 of them); they sit in the slices by decreasing length, lrow
// being a position's place in the window's stretch of the vectors; the window
// gathers the entries list[win[b].y .. win[b+1].y) of the vector and idx is a
// slot's place among them.
struct SweepPat {
  const int64_t *slice_ptr;
  const int32_t *len;   // stored blocks per position
  const int32_t *col;
  const uint16_t *idx, *lrow;
  const int2 *win;
  const int32_t *list;
  int64_t n;
  int32_t nsl;          // slices
};

namespace m3 {
// the most workgroups of a kernel that leaves its partial sums to the host
constexpr int HOST_PARTS = 512;
// Which levels are swept in windows, and when a window is split.  The LDS of all
// workgroups of a sweep is that of its largest window: up to 2,900 gathered
// entries leave room for as many workgroups per CU as the waves allow (two in
// FP64, four in FP32; the meshes here gather 1,350 to 1,450 and at most 1,837 per
// 512 rows), so a window of more is halved, down to the 64 rows of a slice.
// A slice may gather as many as fit into the LDS of a CU beside its sums; a
// level with a slice of more (a node with thousands of neighbours) is swept
// without windows, and so is one whose windows gather more than four entries per
// row in all, because they had to be split or the space-filling order is none for
// its numbering.  337,986 rows, entries per row and us per sweep in FP64 / BF16:
// windows of 512 rows 2.7, 131 / 41.6; 256 rows 3.3, 139 / 49.3; 148 on average 3.9,
// 158 / 56.4; 64 rows 5.1, 214 / 87.3; with the coordinates of two thirds of the
// nodes dealt out anew 20, 239 / 110; without windows 157 / 56.0 on both.
constexpr int SWEEP_LIMIT = 6300;
struct SweepRule {
  int64_t rows = 131072;                      // fewest rows of a level with windows (sweep_window)
  int32_t split = 2900, limit = SWEEP_LIMIT;  // most entries of a window, of a slice
  int32_t per_row = 4;                        // most entries per row of the level
  int most(int64_t nr) const { return nr > 64 ? std::min(split, limit) : limit; }
};
enum class WindowFit { ok, oversized, scattered };
}  // namespace m3

struct Sell {
  int64_t nrow = 0, ncol = 0, nslot = 0, nnz = 0;
  int bs = 9;  // values per stored block
  std::vector<int64_t> h_slice_ptr;
  std::vector<int32_t> h_rowlen, h_col;
  std::vector<int32_t> h_perm, h_ipos;  // empty: identity placement
  DBuf<int64_t> slice_ptr;
  DBuf<int32_t> rowlen, col, perm, ipos;
  DBuf<double> val;
  DBuf<uint32_t> val16;  // packed BF16 copy of the mixed V-cycle (P16 words per slot)
  // order of the level's vectors (empty: node order): node at each place,
  // place of each node
  std::vector<int32_t> h_vperm, h_vpos;
  DBuf<int32_t> vperm, vpos;
  // windowed sweeps (SweepPat): windows (0: none), the most vector entries that
  // one of them gathers
  int nwin = 0, umax = 0;
  DBuf<int2> win;
  DBuf<int32_t> plen, list;
  DBuf<uint16_t> idx, lrow;
  // build from sorted per-row column lists (CSR); uploads pattern, allocates
  // val.  place (may be NULL): the row at each position
  void build(int64_t nrow_, int64_t ncol_, const std::vector<int64_t> &ptr,
             const std::vector<int32_t> &cols, int bs_, const std::vector<int32_t> *place = nullptr);
  // window lists; first: the first row of each window in the vector order, and
  // nrow.  Nothing is kept if a window gathers more entries than rule allows one
  // of its size (oversized) or all of them more than it allows the level (scattered)
  m3::WindowFit build_windows(const std::vector<int32_t> &order, const std::vector<int32_t> &first,
                              const m3::SweepRule &rule);
  int64_t base_of(int64_t row) const {
    const int64_t q = h_ipos.empty() ? row : (int64_t)h_ipos[row];
    return h_slice_ptr[q >> 6] + (q & 63);
  }
  const int32_t *perm_p() const { return h_perm.empty() ? nullptr : perm.p; }
  const int32_t *ipos_p() const { return h_ipos.empty() ? nullptr : ipos.p; }
  const int32_t *vperm_p() const { return h_vperm.empty() ? nullptr : vperm.p; }
  const int32_t *vpos_p() const { return h_vpos.empty() ? nullptr : vpos.p; }
  SellView view() { return SellView{slice_ptr.p, rowlen.p, col.p, val.p, nslot, perm_p(), ipos_p()}; }
  SweepPat sweep() const {
    return SweepPat{slice_ptr.p, nwin ? plen.p : rowlen.p, col.p, idx.p, lrow.p, win.p, list.p, nrow,
                    (int32_t)(h_slice_ptr.size() - 1)};
  }
};

// Coarse sparse Cholesky in 64x64 dense tiles, nested-dissection blocks
// aligned to tiles (one block = one leaf or separator = one supernode).
struct CholTiles {
  int64_t n = 0;                 // free coarse dofs
  int T = 0;                     // tile rows/cols (including padding)
  int64_t ntile = 0;             // stored lower tiles of L (incl. diagonal)
  std::vector<int32_t> h_colptr, h_rowtile;   // tile CSC (row tiles sorted)
  DBuf<int32_t> pos2dof;         // T*64: coarse dof (0-based) or -1 (padding)
  DBuf<int32_t> dof2pos;         // 3*nnod: tile position or -1 (fixed dof)
  DBuf<double> tiles;            // L tiles (column-major)
  DBuf<double> dinv;             // inverses of the diagonal tiles of L
  DBuf<int64_t> gsrc, gdst;      // gather: operator value index -> tile value index
  DBuf<int32_t> diagtile;        // T: tile index of (J,J)
  // factorisation: tile tasks by dependency level
  int nlev = 0;
  std::vector<int32_t> h_lev_ptr, h_trsm_ptr;
  std::vector<int32_t> h_upd_ptr;             // per level: chunks by levels before the last, by the last one
  DBuf<int32_t> lev_cols, upd_tile, upd_pairs, trsm_tile, trsm_col;
  DBuf<int64_t> upd_pair_ptr, upd_pair_end;  // per update chunk: pair range
  // supernodes: explicit inverse of each block's diagonal part
  int nblock = 0, H = 0, maxm = 0;
  int64_t nX = 0, nZ = 0;
  // tile pool X | Z and its transposed copies: X = inverse of each block's
  // diagonal part (block-local m x m, column-major tiles); Z_Ij = L_Ij-part
  // times X for the rows I below a block (Z_Ij = sum_k L_Ik X_kj)
  DBuf<double> X, XT;
  DBuf<float> X32, XT32;                     // FP32 copies of the X | Z tiles for the FP32 V-cycle
  DBuf<int32_t> inv_x, inv_row;              // diagonal X tiles and their tile row (for dinv)
  // the rest of X by recursive doubling: per level two steps, T = B X_AA
  // (B: L tiles) then X_CA = -X_CC T; T tiles follow Z in the pool
  int64_t nT = 0;
  std::vector<int32_t> h_invp_ptr;           // per step: task range
  DBuf<int32_t> invp_out, invp_pairs;        // target pool tile; (A tile, pool tile) pairs
  DBuf<int64_t> invp_pair_ptr;
  DBuf<int32_t> z_tile, z_pairs;             // Z target (pool index); (L tile, X tile) pairs
  DBuf<int64_t> z_pair_ptr;
  // solves: one gather phase per height and direction
  struct Item {                              // out_sel[row] +-= M[mat] in_sel[vcol]
    int32_t row, mat, vcol, sel;
  };
  struct Phase {
    std::vector<int32_t> h_ptr;  // per height: item range
    DBuf<Item> items;
  } fwd, bwd;
  DBuf<double> w, y, x;          // T*64 solve vectors
};

// sparse slots of one element's blocks: K 10x10 at [10a+b], G 10x4 at
// [100+4a+v], GT 4x10 at [140+4a+v], M 4x4 at [180+4v+w]
constexpr int ASM_SLOTS = 196;

// stored element matrix: the 55 node blocks (a >= b) of the symmetric 30x30
// matrix, block a(a+1)/2 + b, each 3x3 row-major (entry [c][d] = K[3a+c][3b+d]);
// the diagonal blocks are stored whole (and symmetric), so every block is one
// contiguous 72-byte read
constexpr int KEL = 55 * 9;

struct LevelDev {
  int64_t nel = 0, nnod = 0, nV = 0;
  std::vector<int32_t> h_el2nod;   // 0-based nel*10
  DBuf<int32_t> el2nod;
  Sell K;                          // 3x3 blocks
  DBuf<double> mask;               // 3*nnod, 1 free / 0 fixed
  // What the V-cycle and the CG hold of this level is in K's vector order
  // (the node order on small levels): the vectors below, dinv, vmask (the mask,
  // a byte per dof) and the transfers
  DBuf<uint8_t> vmask;
  DBuf<double> dinv;               // 3*nnod inverse diagonal (1 at fixed dofs)
  DBuf<float> dinv32;
  DBuf<double> Kel;                // nel*KEL rotated + masked element matrices
  // coarse levels: K summed per row from Kel (row-owner gather, no atomics)
  DBuf<int32_t> kslots;            // per element: 100 K slots (block (a,b) at 10a+b)
  DBuf<int64_t> inc_ptr;           // node -> (element, local node) incidence
  DBuf<int32_t> inc;
  bool gather = false;
  // slot-owner form of the gather: for every stored block slot the sorted
  // list of element blocks that sum into it (code = 2 * (e * 55 + stored
  // block) + transposed), CSR over the slots
  DBuf<int64_t> cptr;
  DBuf<int32_t> clist;
  // transfer to this level from level+1 (fine rows) and its transpose, rows
  // and columns in the two levels' vector orders
  DBuf<int64_t> P_ptr, R_ptr;
  DBuf<int32_t> P_col, R_col;
  DBuf<double> P_val, R_val;
  DBuf<float> P_val32, R_val32;
  DBuf<int32_t> child_type;        // per element: index into Qtab of level+1 transfer
  DBuf<double> Qtab;               // ntypes*100 (10 fine local x 10 coarse local)
  int nqtypes = 0;
  int64_t nfree = 0;
  // V-cycle work vectors (FP64 and FP32 variants)
  DBuf<double> r0, r1, d, dn, dd, rr;
  DBuf<float> r0f, r1f, df, dnf, ddf;
};

namespace m3 {
// CSC patterns of the reference-shaped global matrices (KK lower, GG, MM
// lower) of the finest level, from the element connectivity
struct CscPatterns {
  int64_t nnod = 0, nV = 0;
  std::vector<int64_t> k_ptr;  // node B -> its neighbours A >= B (sorted), incl. B first
  std::vector<int32_t> k_adj;
  std::vector<int64_t> g_ptr;  // vertex p -> velocity nodes sharing an element (sorted)
  std::vector<int32_t> g_adj;
  std::vector<int64_t> m_ptr;  // vertex q -> vertices p >= q sharing an element (sorted)
  std::vector<int32_t> m_adj;
};
CscPatterns csc_patterns(const std::vector<int32_t> &el2nod, int64_t nel, int64_t nnod, int64_t nV);
void csc_sizes(const CscPatterns &pt, m3_csc *KK, m3_csc *GG, m3_csc *MM);
void csc_fill(const CscPatterns &pt, const std::vector<int32_t> &el2nod, int64_t nel, const double *KKv,
              const double *GGv, const double *MMv, const double *Fbv, m3_csc *KK, double *Fb, m3_csc *GG,
              m3_csc *MM);
}  // namespace m3

struct m3_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr;  // learned start ready on the network's stream
  std::string err;
  int nmg = 0;
  std::vector<LevelDev> L;
  // finest-level geometry and operators
  int64_t nel = 0, nnod = 0, nV = 0, n_iso = 0;
  DBuf<uint8_t> cls;
  DBuf<int32_t> iso_idx;
  DBuf<double> X, S, X20, frames;
  DBuf<double> visc, dens;
  Sell G, GT, M;                   // GG (3x1), GG' (1x3), MM (scalar)
  DBuf<double> Fb, bc_rhs, U0, LiMM;
  DBuf<int32_t> errflag;
  DBuf<int32_t> asm_slots;         // per finest element: ASM_SLOTS sparse slots (see k_assemble)
  // row-owner assembly of the finest K from the element matrices: for each
  // node the (element, local node) pairs it belongs to, as 10*element + local
  DBuf<int64_t> inc_ptr;
  DBuf<int32_t> inc;
  bool gather_K = false;
  std::vector<int64_t> h_ifix;
  std::vector<double> h_vfix;
  bool have_mesh = false, have_bc = false, assembled = false, restricted = false,
       factored = false, have_mixed = false, have_fields = false;
  bool g_valid = false;  // G and G' assembled for the current mesh (they depend on it alone)
  // the finest level's packed BF16 values (K.val16) written by the slot
  // gather and patched by the diagonal fix of the last assembly, so that the
  // mixed V-cycle needs no separate packing pass
  bool pack16_fresh = false;
  CholTiles chol;
  std::vector<double> h_coord;     // finest GCOORD row per node (for ordering)
  // reductions
  DBuf<double> partial;            // per-block partial sums
  DBuf<double> scal;               // device scalars
  double *h_scal = nullptr;        // pinned host mirror
  double *h_part = nullptr;        // pinned: partial sums that the host adds (m3::HOST_PARTS)
  m3::SweepRule sweep_rule;        // of the meshes that are set from now on
  // CG / Patera vectors (3*nnod or nV)
  DBuf<double> cg_r, cg_q, cg_Kq, cg_x, cg_b;
  DBuf<double> Uv, Zv, Yv, Rhs;
  DBuf<double> pr, prlast, pd, pq, pSq, pP;
  DBuf<double> fbbc, gU0;  // Patera: mask (Fb - bc_rhs) and GG' U0, per solve
  // solution of the last Stokes solve, kept on the device (U with the BC
  // values, rotated frame; P)
  DBuf<double> Usol, Psol;
  bool have_solution = false;
  m3_phys phys{};
  std::unique_ptr<m3::CscPatterns> csc;  // reference-shaped assembly output patterns (built on first use)
  // embedded refined region: per finest element, inside flag and Dens0_T_bary
  bool have_ref = false;
  DBuf<uint8_t> ref_in;
  DBuf<double> ref_d0;
  // kernel timing, events recorded around launches: kind 0 the fine-level
  // FP64 sweeps, 1 the fine-level mixed-precision sweeps, 2 every other
  // V-cycle kernel (middle-level sweeps, transfers, coarse solve, entry and
  // exit); each launch with its algorithmic bytes
  struct ProfEv {
    hipEvent_t a, b;
    double bytes;
  };
  bool prof = false;
  std::vector<ProfEv> prof_ev[3];
  double prof_acc[3] = {0, 0, 0}, prof_bytes[3] = {0, 0, 0};
  int64_t prof_n[3] = {0, 0, 0};
  // thermal diffusion on linear tetrahedra (a scalar field per node)
  struct {
    bool ready = false, assembled = false, have_M = false;
    int64_t nel = 0, n = 0;
    double theta_cone = 45.0;
    DBuf<int32_t> el, slots;       // 4 nodes and 16 pattern slots per element
    DBuf<uint8_t> cls;
    Sell C;                        // pattern (1 value per slot); val = CC
    DBuf<double> M, A;             // consistent mass and system values on C's slots
    DBuf<double> ML, Adi, mask, vfix, T, rhs, x, r, d, q, Aq;
  } dif;
  std::vector<double> h_sph;       // finest GCOORD_SPH row per node
  // semi-Lagrangian temperature advection on the finest P1 tetrahedra
  struct {
    bool ready = false;
    double r_in = 0, r_out = 0;
    DBuf<int64_t> star_ptr;        // vertex -> incident tetrahedra (CSR)
    DBuf<int32_t> star_tet, tet_v; // tet_v: 4 vertices per tetrahedron
    DBuf<double> tet_geo;          // 12 per tetrahedron: inverse edge matrix, 4th vertex
    DBuf<double> uc, T, Tout, U;   // Cartesian vertex velocity, temperatures, rotated U
  } adv;
  // semi-Lagrangian advection of P2 nodal fields (advect3d_slm_p_sph)
  struct {
    bool ready = false;
    double r_cmb = 0, r_surf = 0;
    DBuf<int32_t> nbr;             // 4 per element: neighbour across the face opposite each vertex, -1 on the boundary
    DBuf<int32_t> start;           // per node: an element that holds it
    DBuf<double> Sz, Sx;           // node (theta, phi, r) in the Z-rotated and the X-rotated frames
    DBuf<double> U, T, Tout;
    DBuf<unsigned long long> cnt;  // [0] points shifted onto the boundary, [1] searches that ended unresolved
  } slm;
};

namespace m3 {
// Events for the next launch (set by ProfScope): the launch records them
// itself at the kernel's start and end (hipExtLaunchKernelGGL), so the
// interval is the kernel's execution even when the host falls behind the GPU.
extern thread_local hipEvent_t prof_start, prof_stop;

// launch (with lds bytes of dynamic LDS), with the profiling events attached
// when a ProfScope set them
template <typename... Args, typename F = void (*)(Args...)>
inline void launch_timed_lds(F kernel, dim3 grid, dim3 block, unsigned lds, hipStream_t s, Args... args) {
  if (prof_start)
    hipExtLaunchKernelGGL(kernel, grid, block, lds, s, prof_start, prof_stop, 0, args...);
  else
    hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
}
template <typename... Args, typename F = void (*)(Args...)>
inline void launch_timed(F kernel, dim3 grid, dim3 block, hipStream_t s, Args... args) {
  launch_timed_lds(kernel, grid, block, 0, s, args...);
}

// time the one launch (through launch_timed) inside the scope when profiling
// is on, recording its algorithmic bytes
struct ProfScope {
  m3_ctx *c;
  int kind;
  double bytes;
  hipEvent_t a = nullptr, b = nullptr;
  ProfScope(m3_ctx *c_, int kind_, bool active, double bytes_ = 0) : c(c_), kind(kind_), bytes(bytes_) {
    if (!active || !c->prof) return;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) {
      if (a) (void)hipEventDestroy(a);
      a = b = nullptr;
      return;
    }
    prof_start = a;
    prof_stop = b;
  }
  ~ProfScope() {
    if (!a) return;
    prof_start = prof_stop = nullptr;
    c->prof_ev[kind].push_back({a, b, bytes});
  }
};
}  // namespace m3

// ---------------------------------------------------------------- launchers
namespace m3 {
constexpr int NIP = 14;
// learned start of the next solve on the network's own stream, from the
// inputs of m3_gnn_set_inputs, without waiting: `ev` is recorded there when
// the start (*U0, *P0 on the device) is complete
void gnn_start_async(m3_gnn *g, double t, int order, int device, hipEvent_t ev, const double **U0,
                     const double **P0);
void upload_sf_tables();
void launch_assemble(m3_ctx *c, double *dbgK, double *dbgG, double *dbgM, double *dbgF,
                     bool write_global);
void launch_rap(m3_ctx *c, int l);  // level l element matrices -> level l+1
void launch_fix_diag(m3_ctx *c, int l);
void launch_gather_K(m3_ctx *c, int level = 0);  // K of a level from its element matrices (no atomics)
void launch_kslots(m3_ctx *c, int level);          // K slots of a coarse level's element blocks
bool build_contrib(m3_ctx *c, int level);          // slot-owner gather lists (false: too large)
void launch_slots(m3_ctx *c);     // per-element slot map of K, G, GT, M (errflag bit 8: missing)
void launch_diag_inv(m3_ctx *c, int l);
void launch_lumped_mm(m3_ctx *c);

// sparse kernels
// rows per sweep window of a level of n nodes (0: no windows)
int sweep_window(const SweepRule &r, int64_t n);
void nan_flag(hipStream_t s, const double *x, int64_t n, int *flag);  // atomicOr(flag, 32) on a NaN
void spmv_K(hipStream_t s, LevelDev &lv, const double *x, double *y);  // node order; lv.r0 and lv.r1 are work space
// vectors of a level between the node order and K's vector order
void to_places(hipStream_t s, const LevelDev &lv, const double *x, double *y);
void to_nodes(hipStream_t s, const LevelDev &lv, const double *x, double *y);
void launch_vmask(hipStream_t s, LevelDev &lv);  // lv.vmask from lv.mask
void spmv_G(hipStream_t s, Sell &G, const double *q, double *y, const double *mask, const double *add = nullptr);
void spmv_GT(hipStream_t s, Sell &GT, const double *z, double *y);
void spmv_M(hipStream_t s, Sell &M, const double *x, double *y);
void prolong(hipStream_t s, LevelDev &fine, const double *dc, const double *dd, double *df);
void restrict_(hipStream_t s, LevelDev &fine, LevelDev &coarse, const double *rf, double *rc);

// V-cycle building blocks (templated on FP64 / FP32 vectors in k_sparse.hip)
void vcycle(m3_ctx *c, const double *r, int precision);
void chol_factor(m3_ctx *c);
void chol_solve_dev(m3_ctx *c, const double *rhs, double *x);  // device vectors, coarse level
// the triangular solves alone, from chol.w to chol.x in tile order (chol.y and
// chol.x cleared by the caller); tiles32: on the FP32 copies of the tiles
void chol_solve_tiles(m3_ctx *c, bool tiles32);

// vector helpers
double dot(m3_ctx *c, const double *a, const double *b, int64_t n);
void axpy(hipStream_t s, double a, const double *x, double *y, int64_t n);
void slm_advect(m3_ctx *c, const double *Ux, const double *Uy, const double *Uz, double *T, double dt,
                const m3_slm_opts *opts, m3_slm_info *info);
void sl_advect(m3_ctx *c, const double *T, const double *U, double dt, double T_cmb, double T_surf,
               double *T_out);
void rock_prop(m3_ctx *c, const double *T, const m3_rock_params *rp, double *Visc, double *Dens);
double calculate_dt(m3_ctx *c, const double *U, double dt_adv_limit, double dtmax);
void copy(hipStream_t s, const double *x, double *y, int64_t n);
void scale_mask(hipStream_t s, const double *x, const double *m, double *y, int64_t n);
double mean(m3_ctx *c, const double *a, int64_t n);
void patera_direction(m3_ctx *c, int64_t n, double wm, bool restart, int ip);
double patera_step(m3_ctx *c, int64_t n, int64_t n3, double *U, const double *z, int ip);
void add_scalar(hipStream_t s, double *a, double v, int64_t n);
void scal(hipStream_t s, double a, double *y, int64_t n);
void build_mixed(m3_ctx *c);
int mgpcg_run(m3_ctx *c, double *x, const double *b, double tol, bool is_abs, int itmax,
              int precision, std::vector<double> *hist, bool x_zero = false);
// Jacobi-preconditioned CG on a scalar SELL operator (1 value per slot) whose
// fixed rows/columns are identity: x and r (initial residual, zero at fixed
// rows) in place; returns iterations, final RMS residual over nfree in *norm
// (q0, q1, Aq: work space of n values)
int pcg_diag_run(m3_ctx *c, SellView A, int64_t n, const double *Adi, double *x, double *r, double *q0, double *q1,
                 double *Aq, double nfree, double tol, int itmax, double *norm);
void spmv_scalar(hipStream_t s, SellView A, int64_t n, const double *x, double *y);
// thermal diffusion on linear tetrahedra
void diffusion_mesh(m3_ctx *c, const uint32_t *EL2NOD, int64_t nel, int64_t nnodT, double theta_cone);
void diffusion3d(m3_ctx *c, double *T, double kappa, double dt, const int64_t *ifix, const double *vfix,
                 int64_t nfix, const m3_diffusion_opts *o, m3_diffusion_info *info);
void diffusion_apply(m3_ctx *c, int which, const double *x, double *y);
}  // namespace m3
