// Bandwidth-bound kernels of the MGPCG velocity solve for gfx950:
// sliced 3x3-block SpMV and the fused Jacobi smoother sweep, the nested P2
// transfer operators, the V-cycle driver and the vector kernels of the CG
// and Patera iterations.
//
// V-cycle (mgpcg_solver_p.m:388-596, 'Setup 3' weights :674-682).  On each
// level the down path is d = w1 D^-1 r0 followed by three fused sweeps
//   r1 = r0 - K d ;  d += w D^-1 r1
// and the restriction r0' = Ic2f_U' r1; the up path is d = dd + Ic2f_U d'
// followed by three fused sweeps.  Every sweep is one kernel that reads the
// matrix once.  Vectors are full length (3*nnod) with zeros at the fixed
// dofs; the operators carry an identity at those dofs, which makes every
// iterate equal to the reference's reduced vectors padded with zeros.
//
// Precision: value type MT and vector type VT are template parameters; the
// FP64 path instantiates MT=VT=double, the mixed path runs the whole V-cycle
// in FP32 on packed BF16 matrix values (MT=B16P).
//
// Vectors of a level are in K's vector order here (Sell): the node order on
// small levels, a space-filling order on the levels whose sweeps run on
// windows.  mgpcg_run takes and returns vectors in node order.
#include "m3_internal.h"

#include <hip/hip_ext.h>

#include <hip/hip_bf16.h>

#include <cstdint>
#include <cstring>

namespace {

// BF16 values in packed groups (kval's counterpart p16_words / p16_v8): eight
// BF16 (round to nearest even) in one 16-byte load and v8 in FP32, 20 bytes
// per block
struct B16P {
  uint32_t w;
};
typedef double d2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
__device__ inline float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ inline float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
// bytes of the nine values of one stored block
template <class MT>
constexpr double block_value_bytes() {
  return std::is_same<MT, B16P>::value ? 4.0 * P16 : 9.0 * sizeof(MT);
}

// streaming load
template <bool NT, class T>
__device__ inline T lds_(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// one 3x3 block of a group of 64 slots as a lane holds it
template <class MT, bool NT>
struct Blk;
template <bool NT>
struct Blk<double, NT> {
  d2v a[4];
  double e;
  __device__ inline void load(const double *val, int64_t group, int lane) {
    const double *v = val + 576 * group;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = lds_<NT>(reinterpret_cast<const d2v *>(v + 128 * j) + lane);
    e = lds_<NT>(v + 512 + lane);
  }
  __device__ inline void apply(double x0, double x1, double x2, double &y0, double &y1, double &y2) const {
    y0 += a[0].x * x0 + a[0].y * x1 + a[1].x * x2;
    y1 += a[1].y * x0 + a[2].x * x1 + a[2].y * x2;
    y2 += a[3].x * x0 + a[3].y * x1 + e * x2;
  }
};
template <bool NT>
struct Blk<B16P, NT> {
  u4v g;
  float e;
  __device__ inline void load(const B16P *val, int64_t group, int lane) {
    const B16P *v = val + 64 * P16 * group;
    g = lds_<NT>(reinterpret_cast<const u4v *>(v) + lane);
    e = lds_<NT>(reinterpret_cast<const float *>(v + 256) + lane);
  }
  __device__ inline void apply(float x0, float x1, float x2, float &y0, float &y1, float &y2) const {
    y0 += bf_lo(g.x) * x0 + bf_hi(g.x) * x1 + bf_lo(g.y) * x2;
    y1 += bf_hi(g.y) * x0 + bf_lo(g.z) * x1 + bf_hi(g.z) * x2;
    y2 += bf_lo(g.w) * x0 + bf_hi(g.w) * x1 + e * x2;
  }
};

// the vectors of a sweep: MODE bits 1: y = K x; 2: r = r0 - K x (to r_out
// unless NULL); 4: d_out = x + w Dinv r; 8: partial sums of x . K x per workgroup
template <class VT>
struct SweepVec {
  const VT *x, *r0, *dinv;
  VT w;
  VT *y, *r_out, *d_out;
  double *part;
};
template <class VT>
struct SweepIn {
  VT r0 = 0, dinv = 0, x = 0;
};
template <class VT, int MODE>
__device__ inline SweepIn<VT> sweep_in(const SweepVec<VT> &v, int64_t o) {
  SweepIn<VT> t;
  if (MODE & 2) t.r0 = v.r0[o];
  if (MODE & 4) t.dinv = v.dinv[o];
  if (MODE & 12) t.x = v.x[o];
  return t;
}
template <class VT, int MODE>
__device__ inline void sweep_out(const SweepVec<VT> &v, const SweepIn<VT> &t, int64_t o, VT kx, double &dot) {
  if (MODE & 1) v.y[o] = kx;
  if (MODE & 2) {
    const VT q = t.r0 - kx;
    if (v.r_out) v.r_out[o] = q;
    if (MODE & 4) v.d_out[o] = t.x + v.w * t.dinv * q;
  }
  if (MODE & 8) dot += (double)t.x * (double)kx;
}
// sum of s over the workgroup's NW waves, in order, to part[blockIdx.x]
template <int NW>
__device__ inline void block_part(double s, double *sh, double *part) {
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = sh[0];
    for (int j = 1; j < NW; ++j) t += sh[j];
    part[blockIdx.x] = t;
  }
}

// Sweep of a level without windows: one slice of 64 rows per workgroup, its
// stored blocks dealt to W waves (wave w takes blocks w, w + W, ...: every load
// still one contiguous stretch per wave), partial sums added in LDS.  These
// levels are latency-bound: a vertex row of 65 blocks is a chain of dependent
// column and vector loads, and one wave per slice leaves the chip empty.  So a
// lane's blocks, the last ones too, go UNR at a time with all their loads in
// flight, and the row's own vectors are read first.  One whole iteration,
// FP64 / mixed, with the remainder block by block and after it (2 16): 5,778
// rows 121 / 92 us, 23,058 rows 206 / 143; UNR and W 4 16: 107 / 92 and 176 / 127,
// 2 16: 106 / 91 and 175 / 125, 4 8: 107 / 93 and 181 / 134, 3 8: 108 / 99 and
// 182 / 136 (43,554 rows below a swept window level: alike).  One wave per
// slice took 22.7 us per FP64 sweep at 5,778 rows, this 8.8.
constexpr int SD_UNR = 2, SD_W = 16;
template <class MT, class VT, int MODE, int W, int UNR>
__global__ __launch_bounds__(64 * W) void k_sweep(SweepPat K, const MT *__restrict__ val, SweepVec<VT> v) {
  __shared__ VT sh[W][192];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t q = (int64_t)blockIdx.x * 64 + lane;
  const int64_t g0 = K.slice_ptr[blockIdx.x] >> 6;
  const int len = q < K.n ? K.len[q] : 0;
  // the row's own vectors, ahead of the long chain
  const int64_t o = 192 * (int64_t)blockIdx.x + threadIdx.x;
  SweepIn<VT> in;
  if (threadIdx.x < 192 && o < 3 * K.n) in = sweep_in<VT, MODE>(v, o);
  VT y0 = 0, y1 = 0, y2 = 0;
  for (int k = w; k < len; k += UNR * W) {
    int cc[UNR];
    VT x[UNR][3];
    Blk<MT, false> b[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (k + u * W < len) {
        cc[u] = lds_<false>(K.col + (g0 + k + u * W) * 64 + lane);
        b[u].load(val, g0 + k + u * W, lane);
      }
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (k + u * W < len)
#pragma unroll
        for (int j = 0; j < 3; ++j) x[u][j] = v.x[3 * (int64_t)cc[u] + j];
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (k + u * W < len) b[u].apply(x[u][0], x[u][1], x[u][2], y0, y1, y2);
  }
  sh[w][3 * lane] = y0;
  sh[w][3 * lane + 1] = y1;
  sh[w][3 * lane + 2] = y2;
  __syncthreads();
  double dot = 0;
  if (threadIdx.x < 192) {
    VT s = sh[0][threadIdx.x];
#pragma unroll
    for (int j = 1; j < W; ++j) s += sh[j][threadIdx.x];
    if (o < 3 * K.n) sweep_out<VT, MODE>(v, in, o, s, dot);
  }
  if (MODE & 8) {
    __shared__ double ds[W];
    block_part<W>(dot, ds, v.part);
  }
}

// Sweep on windows: one window of rows per workgroup (they lie close together
// in space, about ten stored blocks share a column).  The window's part of x is
// gathered once into LDS through the window's list, so the matrix streams with
// no dependent load behind it, with two-byte places instead of four-byte
// columns, and x leaves the caches about twice per sweep instead of filling
// them.  Rounds of SW_TEAMS slices, SW_W waves each; a window's rows are sorted
// by length, so the slices of one round are alike.  The sums go through LDS
// into vector order, so that the vectors are read and written in whole lines.
// HBM-bound: 337,986 rows, FP64 183 us with one wave per slice and gathers from
// memory -> 132 us (5.5 TB/s on the bytes each array needs once), BF16 63.5 ->
// 43.6 us; 2,662,530 rows 1,338 -> 1,024 us and 424 -> 328 us (5.8 TB/s).
// Windows of 1,024 rows, four waves per slice or 16 waves per workgroup are
// within 5 % or slower; eight waves a SIMD matter in BF16 (57.6 us with five).
// RES: the values stay in the last-level cache between sweeps: cached loads and
// a contiguous range of windows per XCD (43.2 -> 39.5 us alone for the BF16
// values of 337,986 rows, which take 210 MB); streaming loads otherwise (FP64
// there 149 us with cached loads).
constexpr int SW_WIN = 512, SW_NW = 8, SW_W = 2, SW_TEAMS = SW_NW / SW_W;
static_assert(24 * (m3::SWEEP_LIMIT + SW_WIN) + 8 * SW_NW <= 160 * 1024, "LDS of a window");
template <class MT, class VT, int MODE, int UNR, bool RES>
__global__ __launch_bounds__(64 * SW_NW, (std::is_same<MT, double>::value ? 4 : 8)) void k_sweep_win(
    SweepPat K, int nwin, int umax, const MT *__restrict__ val, SweepVec<VT> v) {
  extern __shared__ __align__(16) unsigned char sw_lds[];
  VT *xs = reinterpret_cast<VT *>(sw_lds);  // the window's gathered part of x
  VT *ys = xs + 3 * umax;                   // K x of the window's rows, in vector order
  int b = blockIdx.x;
  if (RES) {  // workgroups go to the eight XCDs in turn
    const int per = (nwin + 7) / 8;
    b = (b & 7) * per + (b >> 3);
    if (b >= nwin) b = -1;
  }
  double dot = 0;
  if (b >= 0) {
    const int2 w0 = K.win[b], w1 = K.win[b + 1];
    const int l0 = w0.y, nl = w1.y - l0, nr = w1.x - w0.x;
    for (int t = threadIdx.x; t < 3 * nl; t += 64 * SW_NW) {
      const int i = t / 3;
      xs[t] = v.x[3 * (int64_t)K.list[l0 + i] + (t - 3 * i)];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, w = wave % SW_W, team = wave / SW_W;
    __syncthreads();
#pragma unroll 1
    for (int rd = 0; 64 * SW_TEAMS * rd < nr; ++rd) {
      const int sl = (w0.x >> 6) + rd * SW_TEAMS + team;
      const int q = sl * 64 + lane;
      VT y0 = 0, y1 = 0, y2 = 0;
      VT *yr = ys;
      if (q < w1.x) {
        const int64_t g0 = K.slice_ptr[sl] >> 6;
        const int len = K.len[q];
        yr += 3 * K.lrow[q];
        auto blocks = [&](int k0, auto cnt) {
          constexpr int N = decltype(cnt)::value;
          int cc[N];
          Blk<MT, !RES> bk[N];
#pragma unroll
          for (int u = 0; u < N; ++u) {
            const int64_t g = g0 + k0 + u * SW_W;
            cc[u] = lds_<!RES>(K.idx + g * 64 + lane);
            bk[u].load(val, g, lane);
          }
#pragma unroll
          for (int u = 0; u < N; ++u) {
            const VT *xp = xs + 3 * cc[u];
            bk[u].apply(xp[0], xp[1], xp[2], y0, y1, y2);
          }
        };
        int k = w;
        for (; k + (UNR - 1) * SW_W < len; k += UNR * SW_W) blocks(k, std::integral_constant<int, UNR>{});
        for (; k < len; k += SW_W) blocks(k, std::integral_constant<int, 1>{});
      }
      // the slice's waves add their sums in turn (a row belongs to one lane of each)
#pragma unroll
      for (int j = 0; j < SW_W; ++j) {
        if (w == j && q < w1.x) {
          yr[0] = j == 0 ? y0 : yr[0] + y0;
          yr[1] = j == 0 ? y1 : yr[1] + y1;
          yr[2] = j == 0 ? y2 : yr[2] + y2;
        }
        __syncthreads();
      }
    }
    const int64_t o0 = 3 * (int64_t)w0.x;
    for (int t = threadIdx.x; t < 3 * nr; t += 64 * SW_NW)
      sweep_out<VT, MODE>(v, sweep_in<VT, MODE>(v, o0 + t), o0 + t, ys[t], dot);
  }
  if (MODE & 8) {
    __shared__ double ds[SW_NW];
    block_part<SW_NW>(dot, ds, v.part);
  }
}

// vectors between the node order and a level's vector order
__global__ void k_to_places(int64_t n3, const int32_t *perm, const double *x, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n3) return;
  const int64_t q = i / 3;
  y[i] = x[3 * (int64_t)perm[q] + (i - 3 * q)];
}
__global__ void k_to_nodes(int64_t n3, const int32_t *perm, const double *x, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n3) return;
  const int64_t q = i / 3;
  y[3 * (int64_t)perm[q] + (i - 3 * q)] = x[i];
}
// the mask as a byte per dof in vector order (perm NULL: node order)
__global__ void k_vmask(int64_t n3, const int32_t *perm, const double *mask, uint8_t *vmask) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n3) return;
  const int64_t q = i / 3;
  vmask[i] = mask[perm ? 3 * (int64_t)perm[q] + (i - 3 * q) : i] != 0.0;
}
// r = mask b: b in node order, r and the mask in vector order
__global__ void k_rhs_in(int64_t n3, const int32_t *perm, const uint8_t *vmask, const double *b, double *r) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n3) return;
  const int64_t q = i / 3;
  r[i] = (double)vmask[i] * b[perm ? 3 * (int64_t)perm[q] + (i - 3 * q) : i];
}

// generic scalar-block SELL SpMV with bs values per block, rows with 3
// (bs==3, G) or 1 output component(s)
// G:  y[3*row+c] = mask * sum_k val[c][p] * x[col]        (3x1 blocks)
// GT: y[row]     = sum_k sum_c val[c][p] * x[3*col+c]     (1x3 blocks)
// M:  y[row]     = sum_k val[p] * x[col]
// Slices of 64 rows with their blocks dealt to a workgroup's waves, SG_UNR blocks
// of a lane in flight, sums added in LDS: one thread per row is a chain of
// dependent loads (G: 5,778 rows 10.2 -> 5.3 us, 337,986 rows 30.4 -> 23.5 us).
// G: y = mask * (G x) (+ add)
constexpr int SG_W = 4, SG_UNR = 4;
__global__ __launch_bounds__(64 * SG_W) void k_spmv_G(SellView G, int64_t nrow, const double *x, double *y,
                                                      const double *mask, const double *add) {
  __shared__ double sh[SG_W][192];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t row = 64 * (int64_t)blockIdx.x + lane;
  double a0 = 0, a1 = 0, a2 = 0;
  if (row < nrow) {
    const int64_t base = sell_base(G, row);
    const int len = G.rowlen[row];
    for (int k = w; k < len; k += SG_W * SG_UNR) {
      int cc[SG_UNR];
      double g[SG_UNR][3], xv[SG_UNR];
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * SG_W < len) {
          const int64_t p = base + (int64_t)(k + u * SG_W) * 64;
          cc[u] = G.col[p];
#pragma unroll
          for (int c = 0; c < 3; ++c) g[u][c] = G.val[c * G.nslot + p];
        }
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * SG_W < len) xv[u] = x[cc[u]];
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * SG_W < len) {
          a0 += g[u][0] * xv[u];
          a1 += g[u][1] * xv[u];
          a2 += g[u][2] * xv[u];
        }
    }
  }
  sh[w][3 * lane] = a0;
  sh[w][3 * lane + 1] = a1;
  sh[w][3 * lane + 2] = a2;
  __syncthreads();
  const int64_t o = 192 * (int64_t)blockIdx.x + threadIdx.x;
  if (threadIdx.x >= 192 || o >= 3 * nrow) return;
  double s = sh[0][threadIdx.x];
#pragma unroll
  for (int j = 1; j < SG_W; ++j) s += sh[j][threadIdx.x];
  if (mask) s *= mask[o];
  y[o] = add ? s + add[o] : s;
}

// GT with the blocks of each slice split over GTW waves: wave w of a
// workgroup takes blocks k = w, w + GTW, ... of the slice's 64 rows (each load
// still one contiguous segment per wave), and the partial sums are added in
// LDS.  The pressure rows are few (nVnod) and long: one thread per row left
// the c1 product at 170 workgroups for 256 CUs.
constexpr int GTW = 8;
__device__ inline double spmv_GT_row(const SellView &G, int64_t q, int64_t nrow, const double *x,
                                     double (*sh)[64]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double a = 0;
  if (q < nrow) {
    const int64_t row = G.perm ? (int64_t)G.perm[q] : q;
    const int64_t base = G.slice_ptr[q >> 6] + (q & 63);
    const int len = G.rowlen[row];
    for (int k = w; k < len; k += GTW * SG_UNR) {
      int cc[SG_UNR];
      double g[SG_UNR][3], xv[SG_UNR][3];
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * GTW < len) {
          const int64_t p = base + (int64_t)(k + u * GTW) * 64;
          cc[u] = G.col[p];
#pragma unroll
          for (int c = 0; c < 3; ++c) g[u][c] = G.val[c * G.nslot + p];
        }
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * GTW < len)
#pragma unroll
          for (int c = 0; c < 3; ++c) xv[u][c] = x[3 * (int64_t)cc[u] + c];
#pragma unroll
      for (int u = 0; u < SG_UNR; ++u)
        if (k + u * GTW < len) a += g[u][0] * xv[u][0] + g[u][1] * xv[u][1] + g[u][2] * xv[u][2];
    }
  }
  sh[w][lane] = a;
  __syncthreads();
  double t = sh[0][lane];
#pragma unroll
  for (int j = 1; j < GTW; ++j) t += sh[j][lane];
  return t;
}
__global__ __launch_bounds__(64 * GTW) void k_spmv_GT_split(SellView G, int64_t nrow, const double *x,
                                                            double *y) {
  __shared__ double sh[GTW][64];
  const int64_t q = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);  // position in the slices
  const double t = spmv_GT_row(G, q, nrow, x, sh);
  if (threadIdx.x < 64 && q < nrow) y[G.perm ? (int64_t)G.perm[q] : q] = t;
}

constexpr int TR_UNR = 4;  // transfer weights per lane in flight

// prolongation with the add of the saved defect: df = dd + mask_f * (P dc);
// from the coarsest level (pos not NULL) dc is read where the triangular solves
// left it, pos[dof] in tile order (-1: fixed, 0).  Four lanes per node: the
// chain of row pointer, column, place and value is the time (one lane per node
// 11.0 us at 5,778 rows FP64, this 4.2; 337,986 rows FP32 18 -> 13).
template <class VT, class WT>
__global__ void k_prolong(int64_t nf, const int64_t *ptr, const int32_t *col, const WT *w,
                          const uint8_t *mask, const VT *dc, const double *xt, const int32_t *pos, const VT *dd,
                          VT *df) {
  const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 2;
  const int sub = threadIdx.x & 3;
  VT a[3] = {0, 0, 0}, old = 0, m = 0;
  const int64_t o = 3 * i + sub;
  if (i < nf) {
    const int64_t end = ptr[i + 1];
    int64_t k = ptr[i] + sub;
    if (sub < 3) {
      old = dd ? dd[o] : (VT)0;
      m = (VT)mask[o];
    }
    for (; k < end; k += 4 * TR_UNR) {
      int64_t c3[TR_UNR];
      VT wk[TR_UNR], v[TR_UNR][3];
      int q[TR_UNR][3];
#pragma unroll
      for (int u = 0; u < TR_UNR; ++u)
        if (k + 4 * u < end) {
          c3[u] = 3 * (int64_t)col[k + 4 * u];
          wk[u] = (VT)w[k + 4 * u];
        }
      if (pos) {
#pragma unroll
        for (int u = 0; u < TR_UNR; ++u)
          if (k + 4 * u < end)
#pragma unroll
            for (int c = 0; c < 3; ++c) q[u][c] = pos[c3[u] + c];
#pragma unroll
        for (int u = 0; u < TR_UNR; ++u)
          if (k + 4 * u < end)
#pragma unroll
            for (int c = 0; c < 3; ++c) v[u][c] = q[u][c] >= 0 ? (VT)xt[q[u][c]] : (VT)0;
      } else {
#pragma unroll
        for (int u = 0; u < TR_UNR; ++u)
          if (k + 4 * u < end)
#pragma unroll
            for (int c = 0; c < 3; ++c) v[u][c] = dc[c3[u] + c];
      }
#pragma unroll
      for (int u = 0; u < TR_UNR; ++u)
        if (k + 4 * u < end)
#pragma unroll
          for (int c = 0; c < 3; ++c) a[c] += wk[u] * v[u][c];
    }
  }
#pragma unroll
  for (int off = 2; off > 0; off >>= 1)
#pragma unroll
    for (int c = 0; c < 3; ++c) a[c] += __shfl_xor(a[c], off, 4);
  if (i < nf && sub < 3) df[o] = old + m * (sub == 0 ? a[0] : sub == 1 ? a[1] : a[2]);
}

// what the restriction hands to the coarsest triangular solves: the right-hand
// side at its place in tile order, and the accumulators cleared there (padding
// places are zero in all three and stay so)
struct TileVecs {
  const int32_t *pos;
  double *w, *y, *x;
};

// restriction rc = mask_c * (P' rf); also writes the first smoother iterate
// d1 = w1 Dinv rc of the coarse level when d1 != nullptr, or the coarsest
// solve's vectors instead of rc when t.pos != nullptr
// 16 lanes cooperate on one coarse row (a coarse node gathers from up to
// ~100 fine nodes), reduced with cross-lane shuffles, TR_UNR entries of a lane
// in flight (5,778 rows FP64 6.8 -> 5.2 us).
template <class VT, class WT>
__global__ __launch_bounds__(256) void k_restrict(int64_t nc, const int64_t *ptr, const int32_t *col,
                                                  const WT *w, const uint8_t *mask, const VT *rf, VT *rc,
                                                  const VT *dinv, VT w1, VT *d1, TileVecs t) {
  const int64_t j = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 4;
  const int sub = threadIdx.x & 15;
  VT a0 = 0, a1 = 0, a2 = 0;
  if (j < nc) {
    const int64_t end = ptr[j + 1];
    for (int64_t k = ptr[j] + sub; k < end; k += 16 * TR_UNR) {
      int64_t f3[TR_UNR];
      VT wk[TR_UNR], x[TR_UNR][3];
#pragma unroll
      for (int u = 0; u < TR_UNR; ++u)
        if (k + 16 * u < end) {
          f3[u] = 3 * (int64_t)col[k + 16 * u];
          wk[u] = (VT)w[k + 16 * u];
        }
#pragma unroll
      for (int u = 0; u < TR_UNR; ++u)
        if (k + 16 * u < end)
#pragma unroll
          for (int c = 0; c < 3; ++c) x[u][c] = rf[f3[u] + c];
#pragma unroll
      for (int u = 0; u < TR_UNR; ++u)
        if (k + 16 * u < end) {
          a0 += wk[u] * x[u][0];
          a1 += wk[u] * x[u][1];
          a2 += wk[u] * x[u][2];
        }
    }
  }
  for (int off = 8; off > 0; off >>= 1) {
    a0 += __shfl_xor(a0, off, 16);
    a1 += __shfl_xor(a1, off, 16);
    a2 += __shfl_xor(a2, off, 16);
  }
  if (j >= nc || sub >= 3) return;
  const int64_t o = 3 * j + sub;
  const VT a = (sub == 0 ? a0 : sub == 1 ? a1 : a2) * (VT)mask[o];
  if (t.pos) {
    const int q = t.pos[o];
    if (q >= 0) {
      t.w[q] = (double)a;
      t.y[q] = 0.0;
      t.x[q] = 0.0;
    }
    return;
  }
  rc[o] = a;
  if (d1) d1[o] = w1 * dinv[o] * a;
}

// V-cycle entry on the finest level: r0 = (VT) r and the first smoother
// iterate d = w1 Dinv r0
template <class VT>
__global__ void k_entry(int64_t n, const double *r, const VT *dinv, VT w, VT *r0, VT *d) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const VT ri = (VT)r[i];
  r0[i] = ri;
  d[i] = w * dinv[i] * ri;
}

template <class A, class B>
__global__ void k_convert(int64_t n, const A *x, B *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = (B)x[i];
}

// ---- reductions: partial sums on the device, added by the host or by the kernel that
// needs them, in a fixed order --------------------------------------------------------
constexpr int RB = 256;
__device__ inline double rb_block(double s, double *sh) {
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}
__device__ inline double rb_total(const double *part, int nb, double *sh) {
  double s = 0;
  for (int i = threadIdx.x; i < nb; i += RB) s += part[i];
  return rb_block(s, sh);
}
// a.b, or the sum of a when b is NULL
__global__ __launch_bounds__(RB) void k_dot(int64_t n, const double *a, const double *b, double *part) {
  __shared__ double sh[4];
  double s = 0;
  for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
    s += b ? a[i] * b[i] : a[i];
  s = rb_block(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ---- CG vector kernels: three per iteration besides the V-cycle and K q ---------------
// A kernel that needs a dot product adds the partial sums of the kernel before
// it itself (every workgroup in the same order, so all hold the same value); the
// residual's partial sums go to the host's memory, which adds them.  With eight
// vector kernels, two conversions and a copy per iteration the whole of it took
// 135 / 1,403 us at 5,778 / 337,986 rows (FP64) and 106 / 682 us (mixed), so
// 129 / 1,357 and 101 / 673 us.
// scal: 0 r.d of the current direction, 3 alpha, 4 + parity: r.d by iteration
constexpr int CGB = m3::HOST_PARTS;  // workgroups (and partial sums) of these kernels, at most
// partial sums of (r - rlast).d = -alpha Kq.d (0 in the first iteration) and
// r.d, with d as the V-cycle leaves it
template <class VT>
__global__ __launch_bounds__(RB) void k_cg_dots(int64_t n, const double *r, const double *Kq, const VT *d,
                                                const double *scal, double *part, int first) {
  __shared__ double sh[4];
  double s0 = 0, s1 = 0;
  for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
    const double di = (double)d[i];
    s1 += r[i] * di;
    if (!first) s0 += Kq[i] * di;
  }
  s0 = rb_block(s0, sh);
  s1 = rb_block(s1, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = first ? 0.0 : -scal[3] * s0;
    part[gridDim.x + blockIdx.x] = s1;
  }
}
// beta = ((r - rlast) . d) / rdlast (mgpcg_solver_p.m:161), rd = r.d (:166),
// q = d + beta q
template <class VT>
__global__ __launch_bounds__(RB) void k_cg_dir(int64_t n, const VT *d, double *q, const double *part, int nb,
                                               double *scal, int it) {
  __shared__ double sh[4];
  const double rdlast = scal[4 + (it & 1)];
  const double s0 = it == 1 ? 0.0 : rb_total(part, nb, sh);
  if (blockIdx.x == 0) {
    const double rd = rb_total(part + nb, nb, sh);
    if (threadIdx.x == 0) {
      scal[0] = rd;
      scal[4 + ((it + 1) & 1)] = rd;
    }
  }
  if (it == 1) {
    for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) q[i] = (double)d[i];
  } else {
    const double beta = s0 / rdlast;
    for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
      q[i] = (double)d[i] + beta * q[i];
  }
}

// alpha = rd / qKq (:173), x += alpha q, r -= alpha Kq; partial |r|^2 to the host
__global__ __launch_bounds__(RB) void k_cg_update(int64_t n, double *x, const double *q, double *r, const double *Kq,
                                                  const double *qpart, int nq, double *scal, double *part) {
  __shared__ double sh[4];
  const double alpha = scal[0] / rb_total(qpart, nq, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[3] = alpha;
  double s = 0;
  for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
    x[i] += alpha * q[i];
    const double rn = r[i] - alpha * Kq[i];
    r[i] = rn;
    s += rn * rn;
  }
  s = rb_block(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_axpy(int64_t n, double a, const double *x, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] += a * x[i];
}
__global__ void k_scal(int64_t n, double a, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] *= a;
}
__global__ void k_copy(int64_t n, const double *x, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i];
}
__global__ void k_scale_mask(int64_t n, const double *x, const double *m, double *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i] * m[i];
}
__global__ void k_add_scalar(int64_t n, double *a, double v) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] += v;
}

// y = A x of a scalar SELL matrix: the slice's entries dealt to SP_W waves (one
// thread per row leaves the 43,554 vertex rows of a million-unknown mesh at one
// wave per CU: 9.9 us, this 5.5 us), sums added in LDS
constexpr int SP_W = 4;
__device__ inline double spmv1_row(const SellView &A, int64_t nrow, int64_t q, int w, const double *x,
                                   double (*sh)[64]) {
  const int lane = threadIdx.x & 63;
  double a = 0;
  if (q < nrow) {
    const int64_t base = sell_base(A, q);
    const int len = A.rowlen[q];
#pragma unroll 4
    for (int k = w; k < len; k += SP_W) {
      const int64_t p = base + (int64_t)k * 64;
      a += A.val[p] * x[A.col[p]];
    }
  }
  sh[w][lane] = a;
  __syncthreads();
  return (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
}
__global__ __launch_bounds__(64 * SP_W) void k_spmv1(SellView A, int64_t nrow, const double *x, double *y) {
  __shared__ double sh[SP_W][64];
  const int w = threadIdx.x >> 6;
  const int64_t q = 64 * (int64_t)blockIdx.x + (threadIdx.x & 63);
  const double a = spmv1_row(A, nrow, q, w, x, sh);
  if (w == 0 && q < nrow) y[q] = a;
}

// ---- Patera pressure iteration (flow3d_patera_mg_sph_p.m:476-560) ----------------------
// Four launches besides G q and the velocity solve, and one read by the host, the
// norm at the end: a launch that needs a dot product or a mean adds the partial
// sums of the launch before it, and the mean that is taken out of a sum comes from
// the sums of its terms.  Against 17 vector launches with six blocking reads, 27
// iterations within a whole solve at 5,778 nodes: 24.0 -> 20.7 ms; at 337,986
// nodes, 18 iterations of a time step: idle time 13.0 -> 6.0 ms.
// scal: PP_RD + parity: r.d by iteration
constexpr int PP_RD = 24, PP_BLOCKS = 1024;
// d = p + w LiMM (r - M p), p = LiMM r (precondition_P); per-workgroup sums of
// (r - rlast).d, r.d, d and the last direction q (the first and last 0 in a restart)
__global__ __launch_bounds__(64 * SP_W) void k_pp_prec(SellView M, int64_t n, const double *r, const double *rl,
                                                       const double *LiMM, const double *q, double wm, double *d,
                                                       double *part, int restart) {
  __shared__ double sh[SP_W][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double s[4] = {0, 0, 0, 0};
  for (int64_t b = blockIdx.x; 64 * b < n; b += gridDim.x) {
    const int64_t i = 64 * b + lane;
    double a = 0;
    if (i < n) {
      const int64_t base = sell_base(M, i);
      const int len = M.rowlen[i];
#pragma unroll 4
      for (int k = w; k < len; k += SP_W) {
        const int64_t p = base + (int64_t)k * 64;
        const int64_t j = M.col[p];
        a += M.val[p] * (LiMM[j] * r[j]);
      }
    }
    __syncthreads();
    sh[w][lane] = a;
    __syncthreads();
    if (w == 0 && i < n) {
      const double Mp = (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
      const double ri = r[i], l = LiMM[i], di = l * ri + wm * (l * (ri - Mp));
      d[i] = di;
      if (!restart) {
        s[0] += (ri - rl[i]) * di;
        s[3] += q[i];
      }
      s[1] += ri * di;
      s[2] += di;
    }
  }
  if (w != 0) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    for (int off = 32; off > 0; off >>= 1) s[j] += __shfl_xor(s[j], off, 64);
    if (lane == 0) part[j * gridDim.x + blockIdx.x] = s[j];
  }
}
// q = d + beta q less its mean; beta = (r - rlast).d / rdlast
__global__ __launch_bounds__(RB) void k_pp_dir(int64_t n, const double *d, double *q, const double *part, int nb,
                                               double *scal, int ip, int restart) {
  __shared__ double sh[4];
  const double rdlast = scal[PP_RD + ((ip + 1) & 1)];
  double t[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) t[j] = rb_total(part + j * nb, nb, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[PP_RD + (ip & 1)] = t[1];
  const double beta = restart ? 0.0 : t[0] / rdlast;
  const double m = (t[2] + beta * t[3]) / (double)n;
  for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
    q[i] = (restart ? d[i] : d[i] + beta * q[i]) - m;
}
// Sq = G' z; per-workgroup sums of q.Sq, Sq and r
__global__ __launch_bounds__(64 * GTW) void k_pp_S(SellView G, int64_t n, const double *z, const double *q,
                                                   const double *r, double *Sq, double *part) {
  __shared__ double sh[GTW][64];
  double s[3] = {0, 0, 0};
  for (int64_t b = blockIdx.x; 64 * b < n; b += gridDim.x) {
    const int64_t k = 64 * b + (threadIdx.x & 63);
    __syncthreads();
    const double t = spmv_GT_row(G, k, n, z, sh);
    if (threadIdx.x < 64 && k < n) {
      const int64_t i = G.perm ? (int64_t)G.perm[k] : k;
      Sq[i] = t;
      s[0] += q[i] * t;
      s[1] += t;
      s[2] += r[i];
    }
  }
  if (threadIdx.x >= 64) return;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    for (int off = 32; off > 0; off >>= 1) s[j] += __shfl_xor(s[j], off, 64);
    if (threadIdx.x == 0) part[j * gridDim.x + blockIdx.x] = s[j];
  }
}
// alpha = rd / q.Sq; P += alpha q, U += alpha Z, r -= alpha Sq and r's mean;
// partial |r|^2 to the host
__global__ __launch_bounds__(RB) void k_pp_update(int64_t n, int64_t n3, double *P, const double *q, double *U,
                                                  const double *Z, double *r, double *rl, const double *Sq,
                                                  const double *part, int nb, const double *scal, int ip,
                                                  double *out) {
  __shared__ double sh[4];
  double t[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) t[j] = rb_total(part + j * nb, nb, sh);
  const double alpha = scal[PP_RD + (ip & 1)] / t[0];
  const double m = (t[2] - alpha * t[1]) / (double)n;
  double s = 0;
  for (int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x; i < n3; i += (int64_t)gridDim.x * RB) {
    U[i] += alpha * Z[i];
    if (i < n) {
      P[i] += alpha * q[i];
      const double ri = r[i], rn = ri - alpha * Sq[i] - m;
      rl[i] = ri;
      r[i] = rn;
      s += rn * rn;
    }
  }
  s = rb_block(s, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ---- Jacobi-preconditioned CG on a scalar matrix (pcg_solver_p.m:49-186) --------------
// Two launches per iteration (three for large matrices) and no host in between: the
// direction and the product, then the update.  A workgroup that needs a dot product adds the
// previous launch's partial sums itself (all in the same order, so all hold the
// same value).  All launches end at once when the residual has met the
// tolerance, so the host can queue several iterations and read the state after
// them; the iterates are those of a loop that looks every time.  Seven launches
// and a blocking read per iteration took 55 us at 43,554 rows, this 20.
// state: 0 r.d of the current direction, 1 |r|^2, 2 iterations done, 3 stopped
// (1 converged, 2 NaN) as the direction's launches read it, 4 + parity: r.d by
// iteration, 6 stopped as a direction's launch finds it.  No launch of several
// workgroups reads a value that it writes: k_pcg_dir and k_pcg_q read 3 and write
// 6, the update after them reads 6 and writes 3.
constexpr int PC_T = RB;
__device__ inline void pc_part(double s, double *part, double *sh) {
  s = rb_block(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
// what the launch of a direction leaves: s is |r|^2, (r - rlast).d, r.d
__device__ inline void pcg_state(double *state, const double *s, bool stop, double rr_stop, int it) {
  state[1] = s[0];
  if (stop) {
    state[6] = s[0] < rr_stop ? 1.0 : 2.0;
  } else {
    state[0] = s[2];
    state[4 + ((it + 1) & 1)] = s[2];
  }
}
// partial sums: |r|^2 at up, (r - rlast).d at up + nu, r.d at up + 2 nu
__global__ __launch_bounds__(PC_T) void k_pcg_start(int64_t n, const double *r, const double *Adi, double *up, int nu) {
  __shared__ double sh[4];
  double rr = 0, rd = 0;
  for (int64_t i = blockIdx.x * (int64_t)PC_T + threadIdx.x; i < n; i += (int64_t)gridDim.x * PC_T) {
    const double ri = r[i];
    rr += ri * ri;
    rd += ri * (ri * Adi[i]);
  }
  pc_part(rr, up, sh);
  pc_part(0.0, up + nu, sh);
  pc_part(rd, up + 2 * nu, sh);
}
// iteration it: stop, or q = d + beta qlast with d = r Adi, and Aq with the
// partial sums of q.Aq.  A d and A qlast are summed apart, so that the gather
// does not wait for beta.
__global__ __launch_bounds__(64 * SP_W) void k_pcg_dir(SellView A, int64_t n, const double *r, const double *Adi,
                                                       const double *qlast, double *q, double *Aq, const double *up,
                                                       int nu, double *qp, double *state, double rr_stop, int it) {
  __shared__ double sh[2][SP_W][64], tot[3][SP_W];
  if (state[3] != 0.0) return;
  const double rdlast = state[4 + (it & 1)];  // r.d of the previous iteration
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, t = threadIdx.x;
  double s[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) s[j] = t < nu ? up[j * nu + t] : 0.0;  // nu <= 256
  const int64_t i = 64 * (int64_t)blockIdx.x + lane;
  double ad = 0, aq = 0;
  if (i < n) {
    const int64_t base = sell_base(A, i);
    const int len = A.rowlen[i];
#pragma unroll 4
    for (int k = w; k < len; k += SP_W) {
      const int64_t p = base + (int64_t)k * 64;
      const int64_t j = A.col[p];
      const double a = A.val[p];
      ad += a * (r[j] * Adi[j]);
      aq += a * qlast[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
    for (int off = 32; off > 0; off >>= 1) s[j] += __shfl_xor(s[j], off, 64);
  if (lane == 0)
#pragma unroll
    for (int j = 0; j < 3; ++j) tot[j][w] = s[j];
  sh[0][w][lane] = ad;
  sh[1][w][lane] = aq;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 3; ++j) s[j] = (tot[j][0] + tot[j][1]) + (tot[j][2] + tot[j][3]);
  const bool stop = it > 1 && !(s[0] >= rr_stop);  // |r|^2 below the tolerance's, or NaN
  if (blockIdx.x == 0 && t == 0) pcg_state(state, s, stop, rr_stop, it);
  if (stop || w != 0) return;
  const double beta = it == 1 ? 0.0 : s[1] / rdlast;
  double dot = 0;
  if (i < n) {
    const double a = ((sh[0][0][lane] + sh[0][1][lane]) + (sh[0][2][lane] + sh[0][3][lane])) +
                     beta * ((sh[1][0][lane] + sh[1][1][lane]) + (sh[1][2][lane] + sh[1][3][lane]));
    const double qi = r[i] * Adi[i] + beta * qlast[i];
    q[i] = qi;
    Aq[i] = a;
    dot = qi * a;
  }
  for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
  if (lane == 0) qp[blockIdx.x] = dot;
}
// The same as two launches for a large matrix: q in place, a vector stream, then
// Aq with one gathered vector instead of three (r, Adi and qlast), PC_BLOCKS
// workgroups and so as many partial sums at most (k_pcg_dir leaves one per
// slice, and each workgroup of the update adds all of them).
constexpr int PC_BLOCKS = 2048;
__global__ __launch_bounds__(PC_T) void k_pcg_q(int64_t n, const double *r, const double *Adi, double *q,
                                                const double *up, int nu, double *state, double rr_stop, int it) {
  __shared__ double sh[4];
  if (state[3] != 0.0) return;
  const double rdlast = state[4 + (it & 1)];
  double s[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) s[j] = rb_total(up + j * nu, nu, sh);
  const bool stop = it > 1 && !(s[0] >= rr_stop);
  if (blockIdx.x == 0 && threadIdx.x == 0) pcg_state(state, s, stop, rr_stop, it);
  if (stop) return;
  const double beta = it == 1 ? 0.0 : s[1] / rdlast;
  for (int64_t i = blockIdx.x * (int64_t)PC_T + threadIdx.x; i < n; i += (int64_t)gridDim.x * PC_T)
    q[i] = r[i] * Adi[i] + beta * q[i];
}
__global__ __launch_bounds__(64 * SP_W) void k_pcg_Aq(SellView A, int64_t n, const double *q, double *Aq, double *qp,
                                                      const double *state) {
  __shared__ double sh[SP_W][64];
  if (state[3] != 0.0 || state[6] != 0.0) return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double dot = 0;
  for (int64_t b = blockIdx.x; 64 * b < n; b += gridDim.x) {
    __syncthreads();
    const int64_t i = 64 * b + lane;
    const double a = spmv1_row(A, n, i, w, q, sh);
    if (w == 0 && i < n) {
      Aq[i] = a;
      dot += q[i] * a;
    }
  }
  for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
  if (threadIdx.x == 0) qp[blockIdx.x] = dot;
}
// x += alpha q, r -= alpha Aq, and the partial sums of the next iteration
__global__ __launch_bounds__(PC_T) void k_pcg_update(int64_t n, const double *q, const double *Aq, const double *Adi,
                                                     const double *qp, int nq, double *x, double *r, double *up,
                                                     int nu, double *state, int it) {
  __shared__ double sh[4];
  if (state[6] != 0.0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) state[3] = state[6];
    return;
  }
  const double alpha = state[0] / rb_total(qp, nq, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0) state[2] = it;
  double rr = 0, s0 = 0, s1 = 0;
  for (int64_t i = blockIdx.x * (int64_t)PC_T + threadIdx.x; i < n; i += (int64_t)gridDim.x * PC_T) {
    x[i] += alpha * q[i];
    const double ro = r[i], rn = ro - alpha * Aq[i], d = rn * Adi[i];
    r[i] = rn;
    rr += rn * rn;
    s0 += (rn - ro) * d;
    s1 += rn * d;
  }
  pc_part(rr, up, sh);
  pc_part(s0, up + nu, sh);
  pc_part(s1, up + 2 * nu, sh);
}
// |r|^2 after the last queued iteration
__global__ __launch_bounds__(PC_T) void k_pcg_look(const double *up, int nu, double *state, double rr_stop) {
  __shared__ double sh[4];
  if (state[3] != 0.0) return;  // one workgroup, and it writes behind rb_total's barriers
  const double rr = rb_total(up, nu, sh);
  if (threadIdx.x == 0) {
    state[1] = rr;
    if (state[2] > 0.0 && !(rr >= rr_stop)) state[3] = rr < rr_stop ? 1.0 : 2.0;
  }
}

// FP64 values -> packed BF16 groups (the slot gather of K writes the same bits
// itself when it assembles the finest level, k_gatherK_slots)
__global__ void k_pack16(int64_t ns, const double *val, uint32_t *out) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= ns) return;
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const d2v v = *reinterpret_cast<const d2v *>(val + kval(p, 2 * j));
    w[j] = bf16_rne(v.x) | (bf16_rne(v.y) << 16);
  }
  *reinterpret_cast<u4v *>(out + p16_words(p)) = u4v{w[0], w[1], w[2], w[3]};
  out[p16_v8(p)] = __float_as_uint((float)val[kval(p, 8)]);
}

__global__ void k_zero3(int64_t n, double *a, double *b, double *c) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = b[i] = c[i] = 0.0;
}

__global__ void k_zero64(int64_t n, double *x) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

inline unsigned nblk(int64_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

namespace m3 {

thread_local hipEvent_t prof_start = nullptr, prof_stop = nullptr;

// Windows of 512 rows pay once a level fills the chip with them; below, the
// sweeps are latency-bound and the gather into LDS adds to the chain (BF16 /
// FP64, windows of 512 against none: 92,178 rows 22.5 / 36.8 against 17.6 /
// 42.9 us, 174,114 rows 27.1 / 74.5 against 30.3 / 89.7 us, 256,050 rows 33.9 /
// 93.3 against 44.8 / 130 us).  Windows of 256 rows: 25.4 / 82.3 us on 174,114
// rows, 34.1 / 102 us on 256,050.
int sweep_window(const SweepRule &r, int64_t n) { return n >= r.rows ? SW_WIN : 0; }

// do the values stay in the last-level cache (256 MB) between sweeps?  In BF16,
// up to some 370,000 rows; FP64 values of a level that has windows do not (28
// blocks a row of 74 bytes: 270 MB at 131,072 rows)
template <class MT>
static bool sweep_resident(const Sell &K) {
  return !std::is_same<MT, double>::value && (double)K.nnz * (block_value_bytes<MT>() + 2.0) < 230e6;
}
// workgroups of a sweep, each with its partial sum (MODE bit 8)
template <class MT>
static int sweep_grid(const Sell &K) {
  if (!K.nwin) return (int)((K.nrow + 63) / 64);
  return sweep_resident<MT>(K) ? (K.nwin + 7) / 8 * 8 : K.nwin;
}

// one sweep: the values val (K.val or the packed BF16 copy) on K's pattern
template <class MT, class VT, int MODE>
static void launch_sweep(hipStream_t s, const Sell &K, const MT *val, const SweepVec<VT> &v) {
  const SweepPat P = K.sweep();
  if (K.nwin) {
    constexpr int UNR = std::is_same<MT, double>::value ? 2 : 3;
    const unsigned lds = (unsigned)(3 * ((size_t)K.umax + SW_WIN) * sizeof(VT));
    auto go = [&](auto kern) {
      if (lds > 64 * 1024)
        HIPCHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds));
      launch_timed_lds(kern, dim3((unsigned)sweep_grid<MT>(K)), dim3(64 * SW_NW), lds, s, P, K.nwin, K.umax, val, v);
    };
    if constexpr (!std::is_same<MT, double>::value) {
      if (sweep_resident<MT>(K)) {
        go(k_sweep_win<MT, VT, MODE, UNR, true>);
        return;
      }
    }
    go(k_sweep_win<MT, VT, MODE, UNR, false>);
  } else {
    launch_timed(k_sweep<MT, VT, MODE, SD_W, SD_UNR>, dim3((unsigned)P.nsl), dim3(64 * SD_W), s, P, val, v);
  }
}
void to_places(hipStream_t s, const LevelDev &lv, const double *x, double *y) {
  const int64_t n3 = 3 * lv.nnod;
  if (lv.K.vperm_p())
    hipLaunchKernelGGL(k_to_places, dim3(nblk(n3)), dim3(256), 0, s, n3, lv.K.vperm_p(), x, y);
  else
    copy(s, x, y, n3);
}
void to_nodes(hipStream_t s, const LevelDev &lv, const double *x, double *y) {
  const int64_t n3 = 3 * lv.nnod;
  if (lv.K.vperm_p())
    hipLaunchKernelGGL(k_to_nodes, dim3(nblk(n3)), dim3(256), 0, s, n3, lv.K.vperm_p(), x, y);
  else
    copy(s, x, y, n3);
}

void launch_vmask(hipStream_t s, LevelDev &lv) {
  const int64_t n3 = 3 * lv.nnod;
  if (lv.vmask.n != (size_t)n3) lv.vmask.alloc(n3);
  hipLaunchKernelGGL(k_vmask, dim3(nblk(n3)), dim3(256), 0, s, n3, lv.K.vperm_p(), lv.mask.p, lv.vmask.p);
  HIPCHECK(hipGetLastError());
}

void spmv_K(hipStream_t s, LevelDev &lv, const double *x, double *y) {
  SweepVec<double> v{};
  v.x = x;
  v.y = y;
  if (!lv.K.vperm_p()) {
    launch_sweep<double, double, 1>(s, lv.K, lv.K.val.p, v);
    return;
  }
  to_places(s, lv, x, lv.r0.p);
  v.x = lv.r0.p;
  v.y = lv.r1.p;
  launch_sweep<double, double, 1>(s, lv.K, lv.K.val.p, v);
  to_nodes(s, lv, lv.r1.p, y);
}

void spmv_G(hipStream_t s, Sell &G, const double *q, double *y, const double *mask, const double *add) {
  hipLaunchKernelGGL(k_spmv_G, dim3((unsigned)((G.nrow + 63) / 64)), dim3(64 * SG_W), 0, s, G.view(), G.nrow, q, y,
                     mask, add);
}
void spmv_GT(hipStream_t s, Sell &GT, const double *z, double *y) {
  hipLaunchKernelGGL(k_spmv_GT_split, dim3((unsigned)((GT.nrow + 63) / 64)), dim3(64 * GTW), 0, s, GT.view(),
                     GT.nrow, z, y);
}
void spmv_M(hipStream_t s, Sell &M, const double *x, double *y) { spmv_scalar(s, M.view(), M.nrow, x, y); }
void prolong(hipStream_t s, LevelDev &fine, const double *dc, const double *dd, double *df) {
  hipLaunchKernelGGL((k_prolong<double, double>), dim3(nblk(4 * fine.nnod)), dim3(256), 0, s, fine.nnod,
                     fine.P_ptr.p, fine.P_col.p, fine.P_val.p, fine.vmask.p, dc, (const double *)nullptr,
                     (const int32_t *)nullptr, dd, df);
}
void restrict_(hipStream_t s, LevelDev &fine, LevelDev &coarse, const double *rf, double *rc) {
  hipLaunchKernelGGL((k_restrict<double, double>), dim3(nblk(16 * coarse.nnod)), dim3(256), 0, s,
                     coarse.nnod, fine.R_ptr.p, fine.R_col.p, fine.R_val.p, coarse.vmask.p, rf, rc,
                     (const double *)nullptr, 0.0, (double *)nullptr, TileVecs{});
}

static void add_scalar_impl(hipStream_t s, double *a, double v, int64_t n) {
  hipLaunchKernelGGL(k_add_scalar, dim3(nblk(n)), dim3(256), 0, s, n, a, v);
}

// --------------------------------------------------------------------------------
// V-cycle.  FP64: vectors and matrices double.  Mixed: the residual is
// converted to FP32, the cycle runs in FP32 on the packed BF16 values (the
// coarsest solve in FP64 on FP32 tiles), and the defect is converted back.
// --------------------------------------------------------------------------------
static const double WDOWN1[3] = {0.9, 0.4, 0.25}, WUP1[3] = {0.25, 0.4, 0.9};
static const double WDOWN[3] = {0.25, 0.4, 0.9}, WUP[3] = {0.9, 0.4, 0.25};

template <class VT>
struct VecSet {
  VT *r0, *r1, *d, *dn, *dd;
  const VT *dinv;
};

static VecSet<double> vecs64(LevelDev &l) {
  return VecSet<double>{l.r0.p, l.r1.p, l.d.p, l.dn.p, l.dd.p, l.dinv.p};
}
static VecSet<float> vecs32(LevelDev &l) {
  return VecSet<float>{l.r0f.p, l.r1f.p, l.df.p, l.dnf.p, l.ddf.p, l.dinv32.p};
}

template <class MT>
static const MT *level_values(const LevelDev &lv) {
  if constexpr (std::is_same<MT, double>::value) return lv.K.val.p;
  else return reinterpret_cast<const MT *>(lv.K.val16.p);
}

template <class MT, class VT>
static void sweep(hipStream_t s, const LevelDev &lv, const VT *x, const VT *r0, const VT *dinv, double w, VT *r_out,
                  VT *d_out) {
  SweepVec<VT> v{x, r0, dinv, (VT)w, nullptr, r_out, d_out, nullptr};
  if (d_out) launch_sweep<MT, VT, 6>(s, lv.K, level_values<MT>(lv), v);
  else launch_sweep<MT, VT, 2>(s, lv.K, level_values<MT>(lv), v);
}

// Algorithmic bytes (each stored array once, perfect reuse of the gathered
// vector) of the V-cycle kernels, for the profile:
//   sweep: every stored 3x3 block (values and int32 column, or two-byte place
//          in the window), the row lengths, and nvec vectors of 3 components;
//   restriction / prolongation: the weights and columns, the row pointers,
//          the mask, the gathered vector once and the vectors read / written.
template <class MT>
static double sweep_bytes(const LevelDev &lv, int nvec, size_t vt) {
  return (double)lv.K.nnz * (block_value_bytes<MT>() + (lv.K.nwin ? 2.0 : 4.0)) + 4.0 * lv.nnod +
         3.0 * lv.nnod * nvec * vt;
}

template <class MT, class VT>
static void vcycle_impl(m3_ctx *c, VecSet<VT> (*vs)(LevelDev &)) {
  hipStream_t s = c->stream;
  const int nm = c->nmg;
  const int pk = std::is_same<VT, double>::value ? 0 : 1;  // profile kind of the fine fused sweeps
  const size_t sv = sizeof(VT);
  // r0 of level 0 already in place
  for (int l = 0; l < nm - 1; ++l) {
    LevelDev &lv = c->L[l];
    VecSet<VT> v = vs(lv);
    const double *wd = l == 0 ? WDOWN1 : WDOWN;
    // level 0: r0 and d = w1 Dinv r0 were written by k_entry
    // d (= w1 Dinv r0) is in v.d; v.r0 is kept
    const int kind = l == 0 ? pk : 2;
    const double b6 = sweep_bytes<MT>(lv, 4, sv), b2 = sweep_bytes<MT>(lv, 3, sv);
    { ProfScope ps(c, kind, true, b6); sweep<MT, VT>(s, lv, v.d, v.r0, v.dinv, wd[1], nullptr, v.dn); }
    { ProfScope ps(c, kind, true, b6); sweep<MT, VT>(s, lv, v.dn, v.r0, v.dinv, wd[2], nullptr, v.dd); }
    { ProfScope ps(c, 2, true, b2); sweep<MT, VT>(s, lv, v.dd, v.r0, v.dinv, 0.0, v.r1, nullptr); }
    LevelDev &cl = c->L[l + 1];
    VecSet<VT> vc = vs(cl);
    const bool coarsest = (l + 1 == nm - 1);
    const TileVecs tv = coarsest ? TileVecs{c->chol.dof2pos.p, c->chol.w.p, c->chol.y.p, c->chol.x.p} : TileVecs{};
    const double rb = (double)lv.R_col.n * (sv + 4.0) + (cl.nnod + 1.0) * sizeof(*lv.R_ptr.p) +
                      3.0 * cl.nnod + 3.0 * lv.nnod * sv + 3.0 * cl.nnod * sv * (coarsest ? 1 : 3);
    ProfScope ps(c, 2, true, rb);
    if constexpr (std::is_same<VT, double>::value)
      launch_timed(k_restrict<double, double>, dim3(nblk(16 * cl.nnod)), dim3(256), s, (int64_t)cl.nnod,
                   (const int64_t *)lv.R_ptr.p, (const int32_t *)lv.R_col.p, (const double *)lv.R_val.p,
                   (const uint8_t *)cl.vmask.p, (const double *)v.r1, vc.r0,
                   coarsest ? (const double *)nullptr : vc.dinv, WDOWN[0], coarsest ? (double *)nullptr : vc.d, tv);
    else
      launch_timed(k_restrict<float, float>, dim3(nblk(16 * cl.nnod)), dim3(256), s, (int64_t)cl.nnod,
                   (const int64_t *)lv.R_ptr.p, (const int32_t *)lv.R_col.p, (const float *)lv.R_val32.p,
                   (const uint8_t *)cl.vmask.p, (const float *)v.r1, vc.r0,
                   coarsest ? (const float *)nullptr : vc.dinv, (float)WDOWN[0], coarsest ? (float *)nullptr : vc.d, tv);
  }
  // coarsest: FP64 Cholesky, from the tile-ordered right-hand side that the
  // restriction wrote to the tile-ordered x that the prolongation reads
  chol_solve_tiles(c, !std::is_same<VT, double>::value);
  for (int l = nm - 2; l >= 0; --l) {
    LevelDev &lv = c->L[l];
    LevelDev &cl = c->L[l + 1];
    VecSet<VT> v = vs(lv);
    VecSet<VT> vc = vs(cl);
    const double *wu = l == 0 ? WUP1 : WUP;
    const bool coarsest = (l + 1 == nm - 1);
    const double *xt = coarsest ? c->chol.x.p : nullptr;
    const int32_t *pos = coarsest ? c->chol.dof2pos.p : nullptr;
    // prolongated correction into dn; three sweeps dn -> d -> dn -> d leave
    // the level's result in d
    {
      const double pb = (double)lv.P_col.n * (sv + 4.0) + (lv.nnod + 1.0) * sizeof(*lv.P_ptr.p) +
                        3.0 * lv.nnod + 3.0 * cl.nnod * sv + 3.0 * lv.nnod * sv * 2;
      ProfScope ps(c, 2, true, pb);
      if constexpr (std::is_same<VT, double>::value)
        launch_timed(k_prolong<double, double>, dim3(nblk(4 * lv.nnod)), dim3(256), s, (int64_t)lv.nnod,
                     (const int64_t *)lv.P_ptr.p, (const int32_t *)lv.P_col.p, (const double *)lv.P_val.p,
                     (const uint8_t *)lv.vmask.p, (const double *)vc.d, xt, pos, (const double *)v.dd, v.dn);
      else
        launch_timed(k_prolong<float, float>, dim3(nblk(4 * lv.nnod)), dim3(256), s, (int64_t)lv.nnod,
                     (const int64_t *)lv.P_ptr.p, (const int32_t *)lv.P_col.p, (const float *)lv.P_val32.p,
                     (const uint8_t *)lv.vmask.p, (const float *)vc.d, xt, pos, (const float *)v.dd, v.dn);
    }
    const int kind = l == 0 ? pk : 2;
    const double b6 = sweep_bytes<MT>(lv, 4, sv);
    { ProfScope ps(c, kind, true, b6); sweep<MT, VT>(s, lv, v.dn, v.r0, v.dinv, wu[0], nullptr, v.d); }
    { ProfScope ps(c, kind, true, b6); sweep<MT, VT>(s, lv, v.d, v.r0, v.dinv, wu[1], nullptr, v.dn); }
    { ProfScope ps(c, kind, true, b6); sweep<MT, VT>(s, lv, v.dn, v.r0, v.dinv, wu[2], nullptr, v.d); }
  }
}

// the cycle on r; the result is left in the finest level's d (df in the mixed
// form)
void vcycle(m3_ctx *c, const double *r, int precision) {
  hipStream_t s = c->stream;
  LevelDev &f = c->L[0];
  const int64_t n3 = 3 * f.nnod;
  if (precision == M3_PREC_FP64) {
    {
      ProfScope ps(c, 2, true, n3 * (8.0 + 3 * 8.0));
      launch_timed(k_entry<double>, dim3(nblk(n3)), dim3(256), s, n3, r, (const double *)f.dinv.p, WDOWN1[0],
                   f.r0.p, f.d.p);
    }
    vcycle_impl<double, double>(c, vecs64);
  } else {
    {
      ProfScope ps(c, 2, true, n3 * (8.0 + 3 * 4.0));
      launch_timed(k_entry<float>, dim3(nblk(n3)), dim3(256), s, n3, r, (const float *)f.dinv32.p,
                   (float)WDOWN1[0], f.r0f.p, f.df.p);
    }
    vcycle_impl<B16P, float>(c, vecs32);
  }
  HIPCHECK(hipGetLastError());
}

// FP32 / BF16 copies of the operators for the mixed-precision V-cycle
void build_mixed(m3_ctx *c) {
  hipStream_t s = c->stream;
  auto fit = [&](auto &b, size_t n) {
    if (b.n != n) b.alloc(n);
  };
  for (int l = 0; l < c->nmg; ++l) {
    LevelDev &lv = c->L[l];
    const int64_t n3 = 3 * lv.nnod;
    if (l < c->nmg - 1 && !(l == 0 && c->pack16_fresh)) {  // packed BF16 groups for the sweeps
      fit(lv.K.val16, P16 * lv.K.nslot);
      hipLaunchKernelGGL(k_pack16, dim3(nblk(lv.K.nslot)), dim3(256), 0, s, lv.K.nslot, lv.K.val.p, lv.K.val16.p);
    }
    fit(lv.dinv32, n3);
    hipLaunchKernelGGL((k_convert<double, float>), dim3(nblk(n3)), dim3(256), 0, s, n3, lv.dinv.p,
                       lv.dinv32.p);
    for (auto *b : {&lv.r0f, &lv.r1f, &lv.df, &lv.dnf, &lv.ddf}) fit(*b, n3);
    if (l < c->nmg - 1) {
      const int64_t np = lv.P_val.n, nr = lv.R_val.n;
      fit(lv.P_val32, np);
      fit(lv.R_val32, nr);
      hipLaunchKernelGGL((k_convert<double, float>), dim3(nblk(np)), dim3(256), 0, s, np, lv.P_val.p, lv.P_val32.p);
      hipLaunchKernelGGL((k_convert<double, float>), dim3(nblk(nr)), dim3(256), 0, s, nr, lv.R_val.p, lv.R_val32.p);
    }
  }
  HIPCHECK(hipGetLastError());
  c->have_mixed = true;
}

// ---- dot products and vector helpers ----------------------------------------------------
static int red_blocks(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(CGB, (n + RB - 1) / RB)); }
// the sum of the nb partial sums that the stream's last kernels leave in h_part
static double host_sum(m3_ctx *c, int nb) {
  HIPCHECK(hipStreamSynchronize(c->stream));
  double t = 0;
  for (int i = 0; i < nb; ++i) t += c->h_part[i];
  return t;
}

double dot(m3_ctx *c, const double *a, const double *b, int64_t n) {
  const int nb = red_blocks(n);
  hipLaunchKernelGGL(k_dot, dim3(nb), dim3(RB), 0, c->stream, n, a, b, c->h_part);
  return host_sum(c, nb);
}

double mean(m3_ctx *c, const double *a, int64_t n) { return dot(c, a, nullptr, n) / (double)n; }

// bit 32 of flag when x holds a NaN
__global__ void k_nan_flag(int64_t n, const double *x, int *flag) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n && x[i] != x[i]) atomicOr(flag, 32);
}
void nan_flag(hipStream_t s, const double *x, int64_t n, int *flag) {
  hipLaunchKernelGGL(k_nan_flag, dim3(nblk(n)), dim3(256), 0, s, n, x, flag);
}

void axpy(hipStream_t s, double a, const double *x, double *y, int64_t n) {
  hipLaunchKernelGGL(k_axpy, dim3(nblk(n)), dim3(256), 0, s, n, a, x, y);
}
void copy(hipStream_t s, const double *x, double *y, int64_t n) {
  hipLaunchKernelGGL(k_copy, dim3(nblk(n)), dim3(256), 0, s, n, x, y);
}
void scale_mask(hipStream_t s, const double *x, const double *m, double *y, int64_t n) {
  hipLaunchKernelGGL(k_scale_mask, dim3(nblk(n)), dim3(256), 0, s, n, x, m, y);
}
void add_scalar(hipStream_t s, double *a, double v, int64_t n) { add_scalar_impl(s, a, v, n); }
void scal(hipStream_t s, double a, double *y, int64_t n) {
  hipLaunchKernelGGL(k_scal, dim3(nblk(n)), dim3(256), 0, s, n, a, y);
}

// ---- one MGPCG iteration sequence, device-resident scalars -----------------------------
// Returns the number of iterations; rrms history appended to hist.
int mgpcg_run(m3_ctx *c, double *x, const double *b, double tol, bool is_abs, int itmax,
              int precision, std::vector<double> *hist, bool x_zero) {
  hipStream_t s = c->stream;
  LevelDev &f = c->L[0];
  const int64_t n3 = 3 * f.nnod;
  const double nfree = (double)f.nfree;
  double *r = c->cg_r.p, *q = c->cg_q.p, *Kq = c->cg_Kq.p;
  const int nb = red_blocks(n3);
  auto rms = [&]() { return std::sqrt(host_sum(c, nb) / nfree); };
  // the coarsest solve's vectors, padding places included (a failed solve may
  // have left a NaN there)
  CholTiles &ch = c->chol;
  hipLaunchKernelGGL(k_zero3, dim3(nblk(ch.w.n)), dim3(256), 0, s, (int64_t)ch.w.n, ch.w.p, ch.y.p, ch.x.p);
  const int32_t *perm = f.K.vperm_p();
  double *xi = perm ? c->cg_x.p : x;  // the iterate in vector order
  // r = b - K x  (masked: fixed entries of b are zeroed); a caller that
  // passes x = 0 (x_zero) gets r = b without the product, the same values
  if (x_zero) {
    hipLaunchKernelGGL(k_rhs_in, dim3(nblk(n3)), dim3(256), 0, s, n3, perm, f.vmask.p, b, r);
    if (perm) hipLaunchKernelGGL(k_zero64, dim3(nblk(n3)), dim3(256), 0, s, n3, xi);
  } else {
    hipLaunchKernelGGL(k_rhs_in, dim3(nblk(n3)), dim3(256), 0, s, n3, perm, f.vmask.p, b, c->cg_b.p);
    if (perm) to_places(s, f, x, xi);
    SweepVec<double> v{xi, c->cg_b.p, nullptr, 0.0, nullptr, r, nullptr, nullptr};
    launch_sweep<double, double, 2>(s, f.K, f.K.val.p, v);
  }
  hipLaunchKernelGGL(k_dot, dim3(nb), dim3(RB), 0, s, n3, r, r, c->h_part);
  double rrms = rms();
  if (std::isnan(rrms)) throw M3Error(M3_E_NUMERIC, "RHS vector contains NaNs");
  if (!is_abs) tol = tol * rrms;
  if (hist) hist->push_back(rrms);
  int it = 0;
  const int gK = sweep_grid<double>(f.K);  // partial sums of the K q product, one per workgroup of its launch
  double *qpart = c->partial.p, *dpart = c->partial.p + c->partial.n / 2;
  auto iterate = [&](const auto *d) {
    using VT = std::remove_const_t<std::remove_pointer_t<decltype(d)>>;
    hipLaunchKernelGGL(k_cg_dots<VT>, dim3(nb), dim3(RB), 0, s, n3, r, Kq, d, c->scal.p, dpart, it == 1 ? 1 : 0);
    hipLaunchKernelGGL(k_cg_dir<VT>, dim3(nb), dim3(RB), 0, s, n3, d, q, dpart, nb, c->scal.p, it);
  };
  for (it = 1; it <= itmax; ++it) {
    vcycle(c, r, precision);
    if (precision == M3_PREC_FP64) iterate((const double *)f.d.p);
    else iterate((const float *)f.df.p);
    SweepVec<double> v{q, nullptr, nullptr, 0.0, Kq, nullptr, nullptr, qpart};
    launch_sweep<double, double, 9>(s, f.K, f.K.val.p, v);
    hipLaunchKernelGGL(k_cg_update, dim3(nb), dim3(RB), 0, s, n3, xi, q, r, Kq, qpart, gK, c->scal.p, c->h_part);
    rrms = rms();
    if (hist) hist->push_back(rrms);
    if (std::isnan(rrms)) throw M3Error(M3_E_NUMERIC, "NaN in CG residual");
    if (rrms < tol) break;
  }
  if (perm) to_nodes(s, f, xi, x);
  HIPCHECK(hipGetLastError());
  return it > itmax ? itmax : it;
}

void spmv_scalar(hipStream_t s, SellView A, int64_t n, const double *x, double *y) {
  hipLaunchKernelGGL(k_spmv1, dim3((unsigned)((n + 63) / 64)), dim3(64 * SP_W), 0, s, A, n, x, y);
  HIPCHECK(hipGetLastError());
}

// the next direction of the pressure iteration, of the ip-th iteration
void patera_direction(m3_ctx *c, int64_t n, double wm, bool restart, int ip) {
  hipStream_t s = c->stream;
  const int nb = (int)std::min<int64_t>(PP_BLOCKS, (n + 63) / 64);
  hipLaunchKernelGGL(k_pp_prec, dim3(nb), dim3(64 * SP_W), 0, s, c->M.view(), n, c->pr.p, c->prlast.p, c->LiMM.p,
                     c->pq.p, wm, c->pd.p, c->partial.p, restart ? 1 : 0);
  hipLaunchKernelGGL(k_pp_dir, dim3(red_blocks(n)), dim3(RB), 0, s, n, c->pd.p, c->pq.p, c->partial.p, nb, c->scal.p,
                     ip, restart ? 1 : 0);
}
// the step along it with z = K^-1 G q: P, U, the residual; returns |r|
double patera_step(m3_ctx *c, int64_t n, int64_t n3, double *U, const double *z, int ip) {
  hipStream_t s = c->stream;
  const int nb = (int)std::min<int64_t>(PP_BLOCKS, (n + 63) / 64), ng = red_blocks(n3);
  hipLaunchKernelGGL(k_pp_S, dim3(nb), dim3(64 * GTW), 0, s, c->GT.view(), n, z, c->pq.p, c->pr.p, c->pSq.p,
                     c->partial.p);
  hipLaunchKernelGGL(k_pp_update, dim3(ng), dim3(RB), 0, s, n, n3, c->pP.p, c->pq.p, U, z, c->pr.p, c->prlast.p,
                     c->pSq.p, c->partial.p, nb, c->scal.p, ip, c->h_part);
  return std::sqrt(host_sum(c, ng));
}

// The smallest rr >= 0 that does not meet sqrt(rr / nfree) < tol, so that the
// kernels' comparison rr < rr_stop is that test for every rr, also where tol^2
// underflows; 0 (never met) for a tol <= 0 or NaN.  The test is monotone in rr,
// and non-negative doubles are ordered as their bits.
static double pcg_stop(double tol, double nfree) {
  const auto met = [&](uint64_t bits) {
    double rr;
    std::memcpy(&rr, &bits, sizeof rr);
    return std::sqrt(rr / nfree) < tol;
  };
  uint64_t lo = 0, hi = 0x7ff0000000000000ull;  // +0 and +inf, which never meets it
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if (met(mid)) lo = mid + 1;
    else hi = mid;
  }
  double rr;
  std::memcpy(&rr, &lo, sizeof rr);
  return rr;
}

// Rows from which the direction and the product are launches of their own.  Small
// ones are bound by the launches, large ones by the gathers.  20 to 23 iterations,
// one launch / two, ms: 43,554 rows 0.469 / 0.479, 84,546 0.580 / 0.581, 174,114
// 0.862 / 0.795, 337,986 1.50 / 1.21, 665,730 2.49 / 1.73, 2,662,530 12.4 / 7.3
// (with seven launches and a read per iteration 1.37, 1.26, 1.41, 1.75, 2.21, 8.2).
constexpr int64_t PC_SPLIT = 131072;

// pcg_solver_p.m:49-186 with the 'diag' preconditioner (Polak-Ribiere beta,
// alpha = r.d / q.Aq), k_pcg_dir or k_pcg_q and k_pcg_Aq, k_pcg_update; the norm is |r| / sqrt(nfree)
int pcg_diag_run(m3_ctx *c, SellView A, int64_t n, const double *Adi, double *x, double *r, double *q0, double *q1,
                 double *Aq, double nfree, double tol, int itmax, double *norm) {
  hipStream_t s = c->stream;
  double *state = c->scal.p + 16;  // 7 values
  const bool split = n >= PC_SPLIT;
  const int nu = (int)std::min<int64_t>(split ? 1024 : 256, (n + PC_T - 1) / PC_T);
  const int nq = (int)std::min<int64_t>(split ? PC_BLOCKS : n, (n + 63) / 64);
  double *up = c->partial.p, *qp = c->partial.p + 3 * nu;
  M3_REQUIRE((size_t)(3 * nu + nq) <= c->partial.n, M3_E_STATE, "partial sums do not fit");
  const double rr_stop = pcg_stop(tol, nfree);
  hipLaunchKernelGGL(k_zero64, dim3(1), dim3(256), 0, s, (int64_t)7, state);
  hipLaunchKernelGGL(k_zero64, dim3(nblk(n)), dim3(256), 0, s, n, q0);
  hipLaunchKernelGGL(k_pcg_start, dim3(nu), dim3(PC_T), 0, s, n, r, Adi, up, nu);
  // iterations queued before the host looks: a few launches that end at once
  // against a blocking read each
  constexpr int BATCH = 8;
  for (int it = 1;;) {
    for (const int last = std::min(itmax, it + BATCH - 1); it <= last; ++it) {
      if (split) {
        hipLaunchKernelGGL(k_pcg_q, dim3(nu), dim3(PC_T), 0, s, n, r, Adi, q0, up, nu, state, rr_stop, it);
        hipLaunchKernelGGL(k_pcg_Aq, dim3(nq), dim3(64 * SP_W), 0, s, A, n, q0, Aq, qp, state);
      } else {
        hipLaunchKernelGGL(k_pcg_dir, dim3(nq), dim3(64 * SP_W), 0, s, A, n, r, Adi, q0, q1, Aq, up, nu, qp, state,
                           rr_stop, it);
        std::swap(q0, q1);
      }
      hipLaunchKernelGGL(k_pcg_update, dim3(nu), dim3(PC_T), 0, s, n, q0, Aq, Adi, qp, nq, x, r, up, nu, state, it);
    }
    hipLaunchKernelGGL(k_pcg_look, dim3(1), dim3(PC_T), 0, s, up, nu, state, rr_stop);
    HIPCHECK(hipMemcpyAsync(c->h_scal + 16, state, 4 * sizeof(double), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    const double *h = c->h_scal + 16;
    *norm = std::sqrt(h[1] / nfree);
    if (h[3] == 2.0) throw M3Error(M3_E_NUMERIC, "NaN in CG residual");
    if (h[3] != 0.0 || it > itmax) return (int)h[2];
  }
}

}  // namespace m3

// ---------------------------------------------------------------------------
// Plain device copy, timed: the practical HBM rate next to the 8 TB/s peak,
// and the reference kernel for scaling hardware byte counters.
namespace {
__global__ __launch_bounds__(256) void k_copy_rate(int64_t n4, const float4 *__restrict__ x,
                                                   float4 *__restrict__ y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n4) y[i] = x[i];
}
}  // namespace

extern "C" int m3_copy_rate(int32_t device, int64_t nbytes, int32_t reps, double *gbs) {
  if (!gbs || nbytes < 16 || reps < 1) return M3_E_ARG;
  try {
    HIPCHECK(hipSetDevice(device));
    const int64_t n4 = nbytes / 16;
    DBuf<float4> x, y;
    x.alloc(n4);
    y.alloc(n4);
    hipStream_t s = nullptr;
    HIPCHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    hipEvent_t a = nullptr, b = nullptr;
    HIPCHECK(hipEventCreate(&a));
    HIPCHECK(hipEventCreate(&b));
    // one 16-byte element per thread: the most loads in flight (a grid-stride
    // loop over fewer workgroups measured 4.3-5.2 TB/s against 6.2 TB/s)
    const int64_t nb = (n4 + 255) / 256;
    M3_REQUIRE(nb < (1ll << 31), M3_E_ARG, "copy size too large");
    const unsigned grid = (unsigned)nb;
    for (int r = 0; r < 3; ++r) hipLaunchKernelGGL(k_copy_rate, dim3(grid), dim3(256), 0, s, n4, x.p, y.p);
    HIPCHECK(hipEventRecord(a, s));
    for (int r = 0; r < reps; ++r) hipLaunchKernelGGL(k_copy_rate, dim3(grid), dim3(256), 0, s, n4, x.p, y.p);
    HIPCHECK(hipEventRecord(b, s));
    HIPCHECK(hipEventSynchronize(b));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    (void)hipStreamDestroy(s);
    *gbs = 2.0 * 16.0 * (double)n4 * reps / (ms * 1e-3) / 1e9;
    return M3_OK;
  } catch (const M3Error &e) {
    return e.code;
  }
}
