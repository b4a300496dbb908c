// Graph network of the learned warm start: featurisation, forward pass,
// backward pass, Adam, warm-start assembly.  The network and the parameter
// layout are described in include/m3gnn.h.
//
// Layout in HBM: vertex-major rows, h[i*64 + c] (BF16 bit patterns) for the
// activations, FP32 for features, targets, gradients and parameters.  The
// dense layers run on the FP32 matrix cores with the weights in registers;
// weight gradients are partial sums over row chunks followed by a fixed-order
// reduction, which makes the gradient deterministic.  Every product-accumulate
// of the forward pass is an FMA in a fixed order (bias first, then input index
// ascending), which the CPU restatement follows.
#include "m3_internal.h"

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/m3gnn.h"

namespace {

constexpr int NF = M3_GNN_NF, WD = M3_GNN_WIDTH, NO = M3_GNN_NOUT, NL = M3_GNN_LAYERS;
constexpr int64_t OFF_WE = 0, OFF_BE = NF * WD, OFF_L = OFF_BE + WD, LSZ = 2 * WD * WD + WD,
                  OFF_WD = OFF_L + NL * LSZ, OFF_BD = OFF_WD + WD * NO, NPARAM = OFF_BD + NO;
static_assert(NPARAM == M3_GNN_NPARAM, "parameter layout");
constexpr int NNORM = M3_GNN_NNORM;

__device__ inline uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ inline float lanebc(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

inline int nblk(int64_t n) { return (int)((n + 255) / 256); }

// ---------------------------------------------------------------- features
// s_u, s_p: RMS vertex speed and pressure of the base state; s_T: RMS of the
// temperature's departure from the base state's temperature
// (SCB workgroups of 256 threads each, then one that adds their sums in order:
// the summation order depends on n alone, so the scales do not depend on the
// launch; one workgroup for all vertices took 28 us at 43,554 vertices, this 6.5)
constexpr int SCB = 64;
__global__ __launch_bounds__(256) void k_scales(int64_t n, const double *U, const double *P, const double *T,
                                                const double *Tb, double *part) {
  double su = 0, sp = 0, st = 0;
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += 256 * SCB) {
    su += U[3 * i] * U[3 * i] + U[3 * i + 1] * U[3 * i + 1] + U[3 * i + 2] * U[3 * i + 2];
    sp += P[i] * P[i];
    st += (T[i] - Tb[i]) * (T[i] - Tb[i]);
  }
  __shared__ double a[256], b[256], c[256];
  a[threadIdx.x] = su;
  b[threadIdx.x] = sp;
  c[threadIdx.x] = st;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      a[threadIdx.x] += a[threadIdx.x + o];
      b[threadIdx.x] += b[threadIdx.x + o];
      c[threadIdx.x] += c[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x] = a[0];
    part[SCB + blockIdx.x] = b[0];
    part[2 * SCB + blockIdx.x] = c[0];
  }
}
__global__ __launch_bounds__(64) void k_scales_fin(int64_t n, const double *part, double *sc) {
  if (threadIdx.x >= 3) return;
  double s = 0;
#pragma unroll 8
  for (int j = 0; j < SCB; ++j) s += part[SCB * threadIdx.x + j];
  const double u = sqrt(s / (double)n);
  sc[threadIdx.x] = u > 0 ? u : 1.0;
}

__global__ void k_features(int64_t n, const double *T, const double *Tp, const double *visc, const double *U,
                           const double *P, const float *rn, const double *sc, float *X) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double su = sc[0], sp = sc[1], st = sc[2];
  float *x = X + NF * i;
  x[0] = (float)T[i];
  x[1] = (float)log(visc[i]);
  x[2] = (float)(U[3 * i] / su);
  x[3] = (float)(U[3 * i + 1] / su);
  x[4] = (float)(U[3 * i + 2] / su);
  x[5] = (float)(P[i] / sp);
  x[6] = rn[i];
  x[7] = (float)((T[i] - Tp[i]) / st);
}

__global__ void k_targets(int64_t n, const double *U0, const double *P0, const double *U1, const double *P1,
                          const double *sc, float *Y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double su = sc[0] * sc[2], sp = sc[1] * sc[2];
  for (int c = 0; c < 3; ++c) Y[NO * i + c] = (float)((U1[3 * i + c] - U0[3 * i + c]) / su);
  Y[NO * i + 3] = (float)((P1[i] - P0[i]) / sp);
}

// per-channel sums and sums of squares (C <= 8) over rows
__global__ void k_chan_stats(int64_t rows, const float *X, int C, double *part) {
  double s[8], q[8];
  for (int c = 0; c < 8; ++c) s[c] = q[c] = 0;
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < rows; r += (int64_t)gridDim.x * blockDim.x)
    for (int c = 0; c < C; ++c) {
      const double v = X[r * C + c];
      s[c] += v;
      q[c] += v * v;
    }
  __shared__ double sh[16][256];
  for (int c = 0; c < 8; ++c) {
    sh[c][threadIdx.x] = s[c];
    sh[8 + c][threadIdx.x] = q[c];
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    double t = 0;
    for (int k = 0; k < 256; ++k) t += sh[threadIdx.x][k];
    part[16 * blockIdx.x + threadIdx.x] = t;
  }
}

// ---------------------------------------------------------------- forward
// h0 = relu(xn We + be), xn = (x - mu) / sigma; one wave per vertex, lane =
// column; a lane normalises one feature and the wave broadcasts them
__global__ __launch_bounds__(256) void k_enc(int64_t n, const float *X, const float *norm, const float *prm,
                                             float *Xn, uint16_t *H0) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = g >> 6;
  const int c = (int)(g & 63), f = c & (NF - 1);
  if (i >= n) return;
  const float xn = (X[NF * i + f] - norm[f]) / norm[NF + f];
  float acc = prm[OFF_BE + c];
#pragma unroll
  for (int k = 0; k < NF; ++k) acc = fmaf(lanebc(xn, k), prm[OFF_WE + k * WD + c], acc);
  if (c < NF) Xn[NF * i + c] = xn;
  H0[WD * i + c] = f2bf(fmaxf(acc, 0.f));
}

// m_i = mean of h over the neighbours of i (adjacency order).  Half a wave per
// vertex, two channels a lane; the neighbour list is loaded once and the rows
// of eight neighbours are in flight at a time (one neighbour after the other,
// a chain of dependent loads: 51 us at 43,554 vertices and 14.5 neighbours;
// this 14 us).
__global__ __launch_bounds__(256) void k_agg(int64_t n, const int64_t *ptr, const int32_t *col, const uint16_t *H,
                                             uint16_t *M) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = g >> 5;
  const int c = (int)(g & 31);
  const int64_t b = i < n ? ptr[i] : 0, e = i < n ? ptr[i + 1] : 0;
  const uint32_t *H2 = reinterpret_cast<const uint32_t *>(H);
  float s0 = 0.f, s1 = 0.f;
  for (int64_t p0 = b; p0 < e; p0 += 32) {
    const int m = (int)min((int64_t)32, e - p0);
    const int my = c < m ? col[p0 + c] : 0;
    for (int q = 0; q < m; q += 8) {
      uint32_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = __shfl(my, min(q + u, m - 1), 32);
        v[u] = H2[(WD / 2) * (int64_t)j + c];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (q + u < m) {
          s0 += __uint_as_float(v[u] << 16);
          s1 += __uint_as_float(v[u] & 0xffff0000u);
        }
    }
  }
  if (i >= n) return;
  const float d = (float)(e - b);
  const uint32_t lo = f2bf(e > b ? s0 / d : 0.f), hi = f2bf(e > b ? s1 / d : 0.f);
  reinterpret_cast<uint32_t *>(M)[(WD / 2) * i + c] = lo | (hi << 16);
}

// FP32 matrix cores: v_mfma_f32_32x32x2, lane l holds A[l%32][l/32],
// B[l/32][l%32] and of the result, element r, row 8 (r/4) + 4 (l/32) + r%4,
// column l%32.  Measured on gfx950: an entry is the chain of two fused
// multiply-adds fma(a1, b1, fma(a0, b0, c)), so a sum over ascending input
// index has the bits of the scalar loop (bias first) that the CPU restatement
// follows.
typedef float f16v __attribute__((ext_vector_type(16)));
__device__ inline int mf_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// z = relu([h, m] W + b); h' = h + z   (W: 128 x 64 row-major, then b).  A
// workgroup stages 64 rows of [h, m] in LDS; a wave takes 32 of them and 32 of
// the 64 columns: its half of W in 64 registers, 64 matrix instructions.  A
// column per lane with the inputs broadcast by v_readlane took 42 us at 43,554
// rows, rows read straight into the operands 17, this 16.6 us.
constexpr int MT_LD = WD + 1;  // LDS row stride in words: rows fall into distinct banks
__global__ __launch_bounds__(256) void k_mp(int64_t n, const uint16_t *H, const uint16_t *M, const float *Wl,
                                            uint16_t *Z, uint16_t *Hn) {
  __shared__ uint32_t in[64][MT_LD];  // words 0..31: h, 32..63: m
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5, wave = threadIdx.x >> 6;
  const int c = 32 * (wave & 1) + li, rt = 32 * (wave >> 1);
  float wt[WD];  // W[2 s + lh][c]
#pragma unroll
  for (int s = 0; s < WD; ++s) wt[s] = Wl[(2 * s + lh) * WD + c];
  const float bias = Wl[2 * WD * WD + c];
  const uint32_t *H2 = reinterpret_cast<const uint32_t *>(H), *M2 = reinterpret_cast<const uint32_t *>(M);
  for (int64_t r0 = 64 * (int64_t)blockIdx.x; r0 < n; r0 += 64 * (int64_t)gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int t = threadIdx.x + 256 * q, r = t >> 5, w = t & 31;
      const int64_t row = min(r0 + r, n - 1);
      in[r][w] = H2[32 * row + w];
      in[r][32 + w] = M2[32 * row + w];
    }
    __syncthreads();
    f16v acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = bias;
#pragma unroll
    for (int s = 0; s < WD; ++s) {
      const uint32_t u = in[rt + li][s];
      const float a = __uint_as_float(lh ? u & 0xffff0000u : u << 16);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, wt[s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rr = rt + mf_row(r, lane);
      if (r0 + rr < n) {
        const uint32_t u = in[rr][c >> 1];
        const float z = fmaxf(acc[r], 0.f), h = __uint_as_float(c & 1 ? u & 0xffff0000u : u << 16);
        Z[WD * (r0 + rr) + c] = f2bf(z);
        Hn[WD * (r0 + rr) + c] = f2bf(h + z);
      }
    }
  }
}

// y = h Wd + bd, a thread per row, in input order
__global__ __launch_bounds__(64) void k_dec(int64_t n, const uint16_t *H, const float *prm, float *Y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint4 in[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) in[q] = reinterpret_cast<const uint4 *>(H + WD * i)[q];
  float y[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) y[o] = prm[OFF_BD + o];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint32_t u[4] = {in[q].x, in[q].y, in[q].z, in[q].w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float h = __uint_as_float(k & 1 ? u[k >> 1] & 0xffff0000u : u[k >> 1] << 16);
#pragma unroll
      for (int o = 0; o < NO; ++o) y[o] = fmaf(h, prm[OFF_WD + (8 * q + k) * NO + o], y[o]);
    }
  }
  reinterpret_cast<float4 *>(Y)[i] = float4{y[0], y[1], y[2], y[3]};
}

// ---------------------------------------------------------------- backward
// dY = 2 (y - t/out_sigma) / (n NO); per-block partial sums of squares
__global__ void k_loss(int64_t n, const float *Y, const float *Tg, const float *norm, float scale, float *dY,
                       double *part) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  double s = 0;
  if (e < n * NO) {
    const int o = (int)(e % NO);
    const float d = Y[e] - Tg[e] / norm[2 * NF + o];
    dY[e] = d * scale;
    s = (double)d * (double)d;
  }
  __shared__ double sh[256];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// out[k] = sum(part[0:nb]) / denom, one block
__global__ void k_loss_fin(int nbk, const double *part, double denom, float *out) {
  __shared__ double sh[256];
  double s = 0;
  for (int b = threadIdx.x; b < nbk; b += blockDim.x) s += part[b];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = (float)(sh[0] / denom);
}

// dH[i][c] = sum_o dY[i][o] Wd[c][o]
__global__ void k_dec_bwd(int64_t n, const float *dY, const float *prm, float *dH) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = g >> 6;
  const int c = (int)(g & 63);
  if (i >= n) return;
  float acc = 0.f;
  for (int o = 0; o < NO; ++o) acc = fmaf(dY[NO * i + o], prm[OFF_WD + c * NO + o], acc);
  dH[WD * i + c] = acc;
}

// per-channel sums y*t, y*y, t*t (t = target / out_sigma); block partials
__global__ void k_chan_dot(int64_t n, const float *Y, const float *Tg, const float *norm, double *part) {
  double a[3 * NO];
  for (int k = 0; k < 3 * NO; ++k) a[k] = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    for (int o = 0; o < NO; ++o) {
      const double y = Y[NO * i + o], t = (double)(Tg[NO * i + o] / norm[2 * NF + o]);
      a[3 * o] += y * t;
      a[3 * o + 1] += y * y;
      a[3 * o + 2] += t * t;
    }
  __shared__ double sh[3 * NO][256];
  for (int k = 0; k < 3 * NO; ++k) sh[k][threadIdx.x] = a[k];
  __syncthreads();
  if (threadIdx.x < 3 * NO) {
    double t = 0;
    for (int k = 0; k < 256; ++k) t += sh[threadIdx.x][k];
    part[3 * NO * blockIdx.x + threadIdx.x] = t;
  }
}

// With dP = dH where the stored activation Z is positive, 0 elsewhere:
//   dHn[i][k] = dH[i][k] + sum_c dP[i][c] W[k][c]
//   dM[i][k] = sum_c dP[i][c] W[64+k][c] / deg(i)   (ready for k_agg_bwd)
// on the FP32 matrix cores as in k_mp: a workgroup stages 32 rows of dP in LDS,
// each of its four waves takes 32 of the 128 outputs.  43,554 rows: scalar loop
// and separate masking pass 41 us, rows read straight into the operands 43,
// this 25 us.
__global__ __launch_bounds__(256) void k_mp_bwd(int64_t n, const uint16_t *Z, const float *Wl, const int64_t *ptr,
                                                const float *dH, float *dHn, float *dM) {
  __shared__ float dP[32][MT_LD], dHs[32][MT_LD], deg[32];
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5, part = threadIdx.x >> 6;
  const int k = 32 * (part & 1) + li;
  // W by rows through LDS, a row per output (a lane's own row straight from
  // memory is 32 lines per load)
  __shared__ float ws[2 * WD][MT_LD];
  for (int t = threadIdx.x; t < 2 * WD * WD; t += 256) ws[t >> 6][t & 63] = Wl[t];
  __syncthreads();
  float wt[WD / 2];  // W[output][2 s + lh]
#pragma unroll
  for (int s = 0; s < WD / 2; ++s) wt[s] = ws[32 * part + li][2 * s + lh];
  for (int64_t r0 = 32 * (int64_t)blockIdx.x; r0 < n; r0 += 32 * (int64_t)gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int t = threadIdx.x + 256 * q, r = t >> 6, c = t & 63;
      const int64_t o = WD * min(r0 + r, n - 1) + c;
      const float d = dH[o];
      dHs[r][c] = d;
      dP[r][c] = bf2f(Z[o]) > 0.f ? d : 0.f;
    }
    if (threadIdx.x < 32) {
      const int64_t i = min(r0 + (int)threadIdx.x, n - 1);
      deg[threadIdx.x] = (float)(ptr[i + 1] - ptr[i]);
    }
    __syncthreads();
    f16v acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int s = 0; s < WD / 2; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(dP[li][2 * s + lh], wt[s], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rr = mf_row(r, lane);
      if (r0 + rr >= n) continue;
      if (part < 2) dHn[WD * (r0 + rr) + k] = dHs[rr][k] + acc[r];
      else dM[WD * (r0 + rr) + k] = acc[r] / deg[rr];
    }
  }
}

// dH[j][c] += sum over neighbours i of j of dM[i][c] (dM divided by deg(i)
// already; symmetric graph).  As k_agg (62 us with one neighbour after the
// other and a division each; this 18 us).
__global__ __launch_bounds__(256) void k_agg_bwd(int64_t n, const int64_t *ptr, const int32_t *col, const float *dM,
                                                 float *dH) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t i = g >> 5;
  const int c = (int)(g & 31);
  const int64_t b = i < n ? ptr[i] : 0, e = i < n ? ptr[i + 1] : 0;
  const float2 *D2 = reinterpret_cast<const float2 *>(dM);
  float s0 = 0.f, s1 = 0.f;
  for (int64_t p0 = b; p0 < e; p0 += 32) {
    const int m = (int)min((int64_t)32, e - p0);
    const int my = c < m ? col[p0 + c] : 0;
    for (int q = 0; q < m; q += 8) {
      float2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = __shfl(my, min(q + u, m - 1), 32);
        v[u] = D2[(WD / 2) * (int64_t)j + c];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (q + u < m) {
          s0 += v[u].x;
          s1 += v[u].y;
        }
    }
  }
  if (i >= n) return;
  float2 *o = reinterpret_cast<float2 *>(dH) + (WD / 2) * i + c;
  *o = float2{o->x + s0, o->y + s1};
}

// Weight gradients: partial sums over the row chunk of each workgroup, added in
// order by k_wreduce (deterministic).
//
// A message-passing layer: part[blk][k*64 + c] = sum_r A[r][k] dP[r][c] for
// A = [H, M] (k < 128) and the bias row k = 128 (A = 1), dP as in k_mp_bwd.  A
// product of 128 x rows by rows x 64 on the FP32 matrix cores: the eight waves
// of a workgroup take the four 32-column parts of A times two halves of the
// rows, two 32x32 results each; every load is one line per row.  Registers of
// A rows in LDS and a scalar loop took 420 us at 43,554 rows; this 18 us.
constexpr int WU = 8;  // row pairs in flight
__global__ __launch_bounds__(512) void k_wgrad_mp(int64_t n, int64_t chunk, const uint16_t *H, const uint16_t *M,
                                                  const uint16_t *Z, const float *dH, float *part) {
  __shared__ float sh[2 * WD + 1][WD];
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  const int wave = threadIdx.x >> 6, kt = wave & 3, half = wave >> 2;
  const int64_t r0 = blockIdx.x * chunk, r1 = min(n, r0 + chunk);
  const uint16_t *A = (kt < 2 ? H : M) + 32 * (kt & 1) + li;
  f16v c0, c1;
#pragma unroll
  for (int r = 0; r < 16; ++r) c0[r] = c1[r] = 0.f;
  float b0 = 0.f, b1 = 0.f;
  for (int64_t rb = r0 + 2 * half + lh; rb - lh < r1; rb += 4 * WU) {
    float a[WU], d0[WU], d1[WU];
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      const int64_t r = rb + 4 * u;
      const bool in = r < r1;
      const int64_t o = WD * (in ? r : n - 1);
      const float av = bf2f(A[o]), e0 = dH[o + li], e1 = dH[o + 32 + li];
      const float z0 = bf2f(Z[o + li]), z1 = bf2f(Z[o + 32 + li]);
      a[u] = in ? av : 0.f;
      d0[u] = in && z0 > 0.f ? e0 : 0.f;
      d1[u] = in && z1 > 0.f ? e1 : 0.f;
    }
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], d0[u], c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], d1[u], c1, 0, 0, 0);
      b0 += d0[u];
      b1 += d1[u];
    }
  }
  b0 += __shfl_xor(b0, 32, 64);
  b1 += __shfl_xor(b1, 32, 64);
  if (half == 1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sh[32 * kt + mf_row(r, lane)][li] = c0[r];
      sh[32 * kt + mf_row(r, lane)][32 + li] = c1[r];
    }
    if (kt == 0 && lh == 0) {
      sh[2 * WD][li] = b0;
      sh[2 * WD][32 + li] = b1;
    }
  }
  __syncthreads();
  if (half == 0) {
    float *o = part + (int64_t)blockIdx.x * (2 * WD + 1) * WD;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int k = 32 * kt + mf_row(r, lane);
      o[k * WD + li] = c0[r] + sh[k][li];
      o[k * WD + 32 + li] = c1[r] + sh[k][32 + li];
    }
    if (kt == 0 && lh == 0) {
      o[2 * WD * WD + li] = b0 + sh[2 * WD][li];
      o[2 * WD * WD + 32 + li] = b1 + sh[2 * WD][32 + li];
    }
  }
}

// The encoder (part[blk][k*64 + c] = sum_r Xn[r][k] dP[r][c], k = 8 the bias,
// dP masked by h0) and the decoder (part[blk][k*4 + o] = sum_r h3[r][k] dY[r][o],
// k = 64 the bias): a row per wave and step, lane = column of the wide operand,
// the narrow one uniform; the four waves' sums added in LDS.  122 us -> 17 us
// and 113 us -> 6.6 us at 43,554 rows.
__global__ __launch_bounds__(256) void k_wgrad_enc(int64_t n, int64_t chunk, const float *Xn, const uint16_t *H0,
                                                   const float *dH, float *part) {
  __shared__ float sh[4][NF + 1][WD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r0 = blockIdx.x * chunk, r1 = min(n, r0 + chunk);
  float acc[NF + 1];
#pragma unroll
  for (int k = 0; k <= NF; ++k) acc[k] = 0.f;
  for (int64_t rb = r0 + wave; rb < r1; rb += 16) {
    float d[4], x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t r = min(rb + 4 * u, n - 1);
      const float e = dH[WD * r + lane];
      d[u] = rb + 4 * u < r1 && bf2f(H0[WD * r + lane]) > 0.f ? e : 0.f;
      x[u] = Xn[NF * r + (lane & (NF - 1))];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int k = 0; k < NF; ++k) acc[k] = fmaf(lanebc(x[u], k), d[u], acc[k]);
      acc[NF] += d[u];
    }
  }
#pragma unroll
  for (int k = 0; k <= NF; ++k) sh[wave][k][lane] = acc[k];
  __syncthreads();
  for (int o = threadIdx.x; o < (NF + 1) * WD; o += 256) {
    const int k = o / WD, c = o % WD;
    part[(int64_t)blockIdx.x * (NF + 1) * WD + o] = sh[0][k][c] + sh[1][k][c] + sh[2][k][c] + sh[3][k][c];
  }
}
__global__ __launch_bounds__(256) void k_wgrad_dec(int64_t n, int64_t chunk, const uint16_t *H, const float *dY,
                                                   float *part) {
  __shared__ float sh[4][WD + 1][NO];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r0 = blockIdx.x * chunk, r1 = min(n, r0 + chunk);
  float acc[NO] = {0.f, 0.f, 0.f, 0.f}, b = 0.f;
  for (int64_t rb = r0 + wave; rb < r1; rb += 16) {
    float h[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t r = min(rb + 4 * u, n - 1);
      h[u] = bf2f(H[WD * r + lane]);
      const float e = dY[NO * r + (lane & (NO - 1))];
      y[u] = rb + 4 * u < r1 ? e : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int o = 0; o < NO; ++o) acc[o] = fmaf(h[u], lanebc(y[u], o), acc[o]);
      b += y[u];
    }
  }
#pragma unroll
  for (int o = 0; o < NO; ++o) sh[wave][lane][o] = acc[o];
  if (lane < NO) sh[wave][WD][lane] = b;
  __syncthreads();
  for (int o = threadIdx.x; o < (WD + 1) * NO; o += 256) {
    const int k = o / NO, c = o % NO;
    part[(int64_t)blockIdx.x * (WD + 1) * NO + o] = sh[0][k][c] + sh[1][k][c] + sh[2][k][c] + sh[3][k][c];
  }
}

// out[o] = sum over the nbk partial results: 64 outputs a workgroup, its four
// waves take every fourth partial (one thread for all 256 of them: 62 us for
// the 8,256 values of a layer; this 4.8 us)
__global__ __launch_bounds__(256) void k_wreduce(int nbk, int nout, const float *part, float *out) {
  __shared__ float sh[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int o = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (o < nout) {
#pragma unroll 8
    for (int b = wave; b < nbk; b += 4) s += part[(int64_t)b * nout + o];
  }
  sh[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && o < nout) out[o] = sh[0][lane] + sh[1][lane] + sh[2][lane] + sh[3][lane];
}

__global__ void k_adam(int64_t np, float *p, const float *g, float *m, float *v, float lr, float c1, float c2) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---------------------------------------------------------------- warm start
__global__ void k_apply_vert(int64_t n, const float *Y, const float *norm, const double *sc, const double *Up,
                             const double *Pp, double *dU, double *U0, double *P0) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double su = sc[0] * sc[2], sp = sc[1] * sc[2];
  for (int c = 0; c < 3; ++c) {
    const double d = (double)Y[NO * i + c] * (double)norm[2 * NF + c] * su;
    dU[3 * i + c] = d;
    U0[3 * i + c] = Up[3 * i + c] + d;
  }
  P0[i] = Pp[i] + (double)Y[NO * i + 3] * (double)norm[2 * NF + 3] * sp;
}

__global__ void k_apply_edge(int64_t nv, int64_t ne, const int32_t *par, const double *dU, const double *Up,
                             double *U0) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= ne) return;
  const int64_t a = par[2 * k], b = par[2 * k + 1], node = nv + k;
  for (int c = 0; c < 3; ++c) U0[3 * node + c] = Up[3 * node + c] + 0.5 * (dU[3 * a + c] + dU[3 * b + c]);
}

// ---------------------------------------------------------------- history
// out = sum_j w_j a_j (j = 0 is the most recent state), the Lagrange
// extrapolation of the pushed states to the new time
constexpr int NH = M3_GNN_HIST;
struct LagIn {
  const double *a[NH];
  double w[NH];
  int k;
};

__global__ void k_lagrange(int64_t n, LagIn in, double *out) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = in.w[0] * in.a[0][i];
  for (int j = 1; j < in.k; ++j) s = fma(in.w[j], in.a[j][i], s);
  out[i] = s;
}

}  // namespace

// ==========================================================================
struct m3_gnn {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  int64_t n = 0, nnod = 0;
  DBuf<int64_t> ptr;
  DBuf<int32_t> col, par;
  DBuf<float> rn;
  std::vector<float> h_prm, h_norm;
  DBuf<float> prm, norm, grad, adam_m, adam_v;
  int64_t adam_t = 0;
  // activations and work arrays
  DBuf<float> X, Xn, Y, Tg, dY, dH, dHn, dM, part;
  DBuf<uint16_t> H[NL + 1], M[NL + 1], Z[NL + 1];
  DBuf<double> dpart, sc, dU;
  DBuf<float> dloss;
  // state inputs
  DBuf<double> T, Tp, visc, Up, Pp, Un, Pn, U0, P0;
  // inputs of the next step uploaded ahead (m3_gnn_set_inputs)
  DBuf<double> Tin, viscin;
  bool have_inputs = false;
  // training set
  int32_t nsample = 0;
  DBuf<float> sX, sY;
  // converged states pushed by the caller (ring; the most recent is at head - 1)
  DBuf<double> hT[NH], hU[NH], hP[NH];
  double ht[NH] = {};
  int nhist = 0, head = 0;
  bool have_start = false;  // U0, P0 hold a warm start
};

namespace {

template <class F>
int gguard(m3_gnn *g, F &&f) {
  if (!g) return M3_E_ARG;
  try {
    HIPCHECK(hipSetDevice(g->device));
    f();
    g->err.clear();
    return M3_OK;
  } catch (const M3Error &e) {
    g->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    g->err = e.what();
    return M3_E_ARG;
  }
}

int wgrid(const m3_gnn *g) { return (int)std::min<int64_t>(256, (g->n + 63) / 64); }
// workgroups of the matrix-core layers, `rows` rows each per pass
int mgrid(const m3_gnn *g, int rows) { return (int)std::min<int64_t>(768, (g->n + rows - 1) / rows); }

void forward(m3_gnn *g, const float *X) {
  hipStream_t s = g->stream;
  const int64_t n = g->n;
  hipLaunchKernelGGL(k_enc, dim3(nblk(64 * n)), dim3(256), 0, s, n, X, g->norm.p, g->prm.p, g->Xn.p, g->H[0].p);
  for (int l = 1; l <= NL; ++l) {
    hipLaunchKernelGGL(k_agg, dim3(nblk(32 * n)), dim3(256), 0, s, n, g->ptr.p, g->col.p, g->H[l - 1].p,
                       g->M[l].p);
    hipLaunchKernelGGL(k_mp, dim3(mgrid(g, 64)), dim3(256), 0, s, n, g->H[l - 1].p, g->M[l].p,
                       g->prm.p + OFF_L + (l - 1) * LSZ, g->Z[l].p, g->H[l].p);
  }
  hipLaunchKernelGGL(k_dec, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, n, g->H[NL].p, g->prm.p, g->Y.p);
}

// loss of the current prediction against Tg (raw targets); writes *dloss_slot
void loss_and_backward(m3_gnn *g, const float *Tg, float *dloss_slot) {
  hipStream_t s = g->stream;
  const int64_t n = g->n, ne = NO * n;
  const float scale = (float)(2.0 / (double)ne);
  const int nb = nblk(ne);
  hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, s, n, g->Y.p, Tg, g->norm.p, scale, g->dY.p, g->dpart.p);
  hipLaunchKernelGGL(k_loss_fin, dim3(1), dim3(256), 0, s, nb, g->dpart.p, (double)ne, dloss_slot);
  float *grad = g->grad.p;
  const int nbk = wgrid(g);
  const int64_t chunk = (n + nbk - 1) / nbk;
  auto reduce = [&](int nout, float *out) {
    hipLaunchKernelGGL(k_wreduce, dim3((unsigned)((nout + 63) / 64)), dim3(256), 0, s, nbk, nout, g->part.p, out);
  };
  hipLaunchKernelGGL(k_wgrad_dec, dim3(nbk), dim3(256), 0, s, n, chunk, g->H[NL].p, g->dY.p, g->part.p);
  reduce((WD + 1) * NO, grad + OFF_WD);
  hipLaunchKernelGGL(k_dec_bwd, dim3(nblk(64 * n)), dim3(256), 0, s, n, g->dY.p, g->prm.p, g->dH.p);
  float *dH = g->dH.p, *dHn = g->dHn.p;
  for (int l = NL; l >= 1; --l) {
    const float *Wl = g->prm.p + OFF_L + (l - 1) * LSZ;
    hipLaunchKernelGGL(k_wgrad_mp, dim3(nbk), dim3(512), 0, s, n, chunk, g->H[l - 1].p, g->M[l].p, g->Z[l].p, dH,
                       g->part.p);
    reduce((2 * WD + 1) * WD, grad + OFF_L + (l - 1) * LSZ);
    hipLaunchKernelGGL(k_mp_bwd, dim3(mgrid(g, 32)), dim3(256), 0, s, n, g->Z[l].p, Wl, g->ptr.p, dH, dHn, g->dM.p);
    hipLaunchKernelGGL(k_agg_bwd, dim3(nblk(32 * n)), dim3(256), 0, s, n, g->ptr.p, g->col.p, g->dM.p, dHn);
    std::swap(dH, dHn);
  }
  hipLaunchKernelGGL(k_wgrad_enc, dim3(nbk), dim3(256), 0, s, n, chunk, g->Xn.p, g->H[0].p, dH, g->part.p);
  reduce((NF + 1) * WD, grad + OFF_WE);
}

void adam_step(m3_gnn *g, float lr) {
  ++g->adam_t;
  const float c1 = 1.f - std::pow(0.9f, (float)g->adam_t), c2 = 1.f - std::pow(0.999f, (float)g->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(nblk(NPARAM)), dim3(256), 0, g->stream, (int64_t)NPARAM, g->prm.p, g->grad.p,
                     g->adam_m.p, g->adam_v.p, lr, c1, c2);
}

void launch_scales(m3_gnn *g) {
  hipLaunchKernelGGL(k_scales, dim3(SCB), dim3(256), 0, g->stream, g->n, g->Up.p, g->Pp.p, g->T.p, g->Tp.p, g->dpart.p);
  hipLaunchKernelGGL(k_scales_fin, dim3(1), dim3(64), 0, g->stream, g->n, g->dpart.p, g->sc.p);
}

void upload_state(m3_gnn *g, const double *T, const double *Tp, const double *Visc, const double *Up,
                  const double *Pp) {
  M3_REQUIRE(T && Tp && Visc && Up && Pp, M3_E_ARG, "null argument");
  hipStream_t s = g->stream;
  const int64_t n = g->n;
  for (int64_t i = 0; i < n; ++i)
    M3_REQUIRE(Visc[i] > 0, M3_E_NUMERIC, "Calculated a zero or negative viscosity");
  HIPCHECK(hipMemcpyAsync(g->T.p, T, sizeof(double) * n, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(g->Tp.p, Tp, sizeof(double) * n, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(g->visc.p, Visc, sizeof(double) * n, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(g->Up.p, Up, sizeof(double) * 3 * g->nnod, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(g->Pp.p, Pp, sizeof(double) * n, hipMemcpyHostToDevice, s));
  launch_scales(g);
}

void features_to(m3_gnn *g, float *X) {
  hipLaunchKernelGGL(k_features, dim3(nblk(g->n)), dim3(256), 0, g->stream, g->n, g->T.p, g->Tp.p, g->visc.p,
                     g->Up.p, g->Pp.p, g->rn.p, g->sc.p, X);
}

void require_params(const m3_gnn *g) {
  M3_REQUIRE(!g->h_prm.empty(), M3_E_STATE, "network parameters not set (m3_gnn_set_params)");
}

// new temperature and viscosity of the step being started
void check_visc(const double *Visc, int64_t n) {
  for (int64_t i = 0; i < n; ++i)
    M3_REQUIRE(Visc[i] > 0, M3_E_NUMERIC, "Calculated a zero or negative viscosity");
}

// new temperature and viscosity into T, visc: from the host, or with
// T = Visc = NULL from the inputs uploaded ahead by m3_gnn_set_inputs
void upload_new(m3_gnn *g, const double *T, const double *Visc) {
  const int64_t n = g->n;
  if (!T && !Visc) {
    M3_REQUIRE(g->have_inputs, M3_E_STATE, "T = Visc = NULL needs m3_gnn_set_inputs first");
    HIPCHECK(hipMemcpyAsync(g->T.p, g->Tin.p, sizeof(double) * n, hipMemcpyDeviceToDevice, g->stream));
    HIPCHECK(hipMemcpyAsync(g->visc.p, g->viscin.p, sizeof(double) * n, hipMemcpyDeviceToDevice, g->stream));
    return;
  }
  M3_REQUIRE(T && Visc, M3_E_ARG, "null argument");
  check_visc(Visc, n);
  HIPCHECK(hipMemcpyAsync(g->T.p, T, sizeof(double) * n, hipMemcpyHostToDevice, g->stream));
  HIPCHECK(hipMemcpyAsync(g->visc.p, Visc, sizeof(double) * n, hipMemcpyHostToDevice, g->stream));
}

// Base state at time t in (Tp, Up, Pp): the polynomial of degree
// min(order, nhist - 1) through the most recent pushed states, evaluated at
// t (Lagrange form; order 0 is the last state itself), and, with the new
// temperature already in T, the scales of the features.
void make_base(m3_gnn *g, double t, int order, bool scales = true) {
  M3_REQUIRE(order >= 0 && order < NH, M3_E_ARG, "extrapolation order must be 0..3");
  M3_REQUIRE(g->nhist > 0, M3_E_STATE, "no converged state pushed (m3_gnn_push_state)");
  M3_REQUIRE(std::isfinite(t), M3_E_ARG, "time must be finite");
  const int k = std::min(order + 1, g->nhist);
  LagIn lt{}, lu{}, lp{};
  int slot[NH];
  for (int j = 0; j < k; ++j) slot[j] = (g->head - 1 - j + 2 * NH) % NH;
  for (int j = 0; j < k; ++j) {
    double w = 1.0;
    for (int m = 0; m < k; ++m)
      if (m != j) w *= (t - g->ht[slot[m]]) / (g->ht[slot[j]] - g->ht[slot[m]]);
    lt.w[j] = lu.w[j] = lp.w[j] = w;
    lt.a[j] = g->hT[slot[j]].p;
    lu.a[j] = g->hU[slot[j]].p;
    lp.a[j] = g->hP[slot[j]].p;
  }
  lt.k = lu.k = lp.k = k;
  hipStream_t s = g->stream;
  const int64_t n = g->n, nn = g->nnod;
  hipLaunchKernelGGL(k_lagrange, dim3(nblk(n)), dim3(256), 0, s, n, lt, g->Tp.p);
  hipLaunchKernelGGL(k_lagrange, dim3(nblk(3 * nn)), dim3(256), 0, s, 3 * nn, lu, g->Up.p);
  hipLaunchKernelGGL(k_lagrange, dim3(nblk(n)), dim3(256), 0, s, n, lp, g->Pp.p);
  if (scales)  // needs the new temperature in T
    launch_scales(g);
}

// U0 = Up + network change (vertices; edge nodes take the mean of their two
// vertices' change), P0 = Pp + change, in g->U0, g->P0 (stream-ordered)
void apply_start(m3_gnn *g) {
  hipStream_t s = g->stream;
  const int64_t n = g->n, nn = g->nnod;
  hipLaunchKernelGGL(k_apply_vert, dim3(nblk(n)), dim3(256), 0, s, n, g->Y.p, g->norm.p, g->sc.p, g->Up.p,
                     g->Pp.p, g->dU.p, g->U0.p, g->P0.p);
  if (nn > n)
    hipLaunchKernelGGL(k_apply_edge, dim3(nblk(nn - n)), dim3(256), 0, s, n, nn - n, g->par.p, g->dU.p, g->Up.p,
                       g->U0.p);
  HIPCHECK(hipGetLastError());
}

// the start, downloaded to the caller unless both outputs are NULL (it then
// stays in g->U0, g->P0)
void apply_and_download(m3_gnn *g, double *U0, double *P0) {
  hipStream_t s = g->stream;
  const int64_t n = g->n, nn = g->nnod;
  apply_start(g);
  if (U0) HIPCHECK(hipMemcpyAsync(U0, g->U0.p, sizeof(double) * 3 * nn, hipMemcpyDeviceToHost, s));
  if (P0) HIPCHECK(hipMemcpyAsync(P0, g->P0.p, sizeof(double) * n, hipMemcpyDeviceToHost, s));
  HIPCHECK(hipStreamSynchronize(s));
  g->have_start = true;
}

}  // namespace

namespace m3 {
void gnn_start_async(m3_gnn *g, double t, int order, int device, hipEvent_t ev, const double **U0,
                     const double **P0) {
  M3_REQUIRE(g->device == device, M3_E_ARG, "the network and the Stokes context must use the same GPU");
  require_params(g);
  upload_new(g, nullptr, nullptr);
  make_base(g, t, order);
  features_to(g, g->X.p);
  forward(g, g->X.p);
  apply_start(g);
  HIPCHECK(hipEventRecord(ev, g->stream));
  g->have_start = true;
  *U0 = g->U0.p;
  *P0 = g->P0.p;
}
}  // namespace m3

extern "C" {

int m3_gnn_create(m3_gnn **out, int hip_device, const m3_graph_desc *d) {
  if (!out) return M3_E_ARG;
  *out = nullptr;
  m3_gnn *g = new m3_gnn();
  g->device = hip_device;
  const int rc = gguard(g, [&] {
    int ndev = 0;
    HIPCHECK(hipGetDeviceCount(&ndev));
    M3_REQUIRE(ndev > 0, M3_E_HIP, "no HIP device visible");
    M3_REQUIRE(hip_device >= 0 && hip_device < ndev, M3_E_ARG, "invalid HIP device index");
    M3_REQUIRE(d && d->adj_ptr && d->adj_col && d->radius, M3_E_ARG, "null graph descriptor field");
    const int64_t n = d->nvert, nn = d->nnod;
    M3_REQUIRE(n > 0 && nn >= n, M3_E_ARG, "need nvert > 0 and nnod >= nvert");
    M3_REQUIRE(nn == n || d->edge_parent, M3_E_ARG, "edge_parent required when nnod > nvert");
    M3_REQUIRE(d->r_out > d->r_in, M3_E_ARG, "r_out must exceed r_in");
    M3_REQUIRE(d->adj_ptr[0] == 0, M3_E_ARG, "adj_ptr[0] must be 0");
    for (int64_t i = 0; i < n; ++i) {
      M3_REQUIRE(d->adj_ptr[i + 1] > d->adj_ptr[i], M3_E_MESH, "vertex without neighbours");
      for (int64_t p = d->adj_ptr[i]; p < d->adj_ptr[i + 1]; ++p) {
        const int64_t j = d->adj_col[p];
        M3_REQUIRE(j >= 0 && j < n && j != i, M3_E_MESH, "neighbour index out of range or self loop");
        M3_REQUIRE(p == d->adj_ptr[i] || d->adj_col[p - 1] < j, M3_E_MESH, "neighbour lists must be sorted");
      }
    }
    for (int64_t i = 0; i < n; ++i)  // symmetry: i in N(j) for every j in N(i)
      for (int64_t p = d->adj_ptr[i]; p < d->adj_ptr[i + 1]; ++p) {
        const int64_t j = d->adj_col[p];
        const int32_t *b = d->adj_col + d->adj_ptr[j], *e = d->adj_col + d->adj_ptr[j + 1];
        M3_REQUIRE(std::binary_search(b, e, (int32_t)i), M3_E_MESH, "graph must be symmetric");
      }
    for (int64_t k = 0; k < 2 * (nn - n); ++k)
      M3_REQUIRE(d->edge_parent[k] >= 0 && d->edge_parent[k] < n, M3_E_MESH, "edge parent out of range");
    HIPCHECK(hipSetDevice(hip_device));
    HIPCHECK(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
    g->n = n;
    g->nnod = nn;
    g->ptr.upload(d->adj_ptr, n + 1);
    g->col.upload(d->adj_col, d->adj_ptr[n]);
    if (nn > n) g->par.upload(d->edge_parent, 2 * (nn - n));
    std::vector<float> rn(n);
    for (int64_t i = 0; i < n; ++i) rn[i] = (float)((d->radius[i] - d->r_in) / (d->r_out - d->r_in));
    g->rn.upload(rn);
    g->prm.alloc(NPARAM);
    g->norm.alloc(NNORM);
    g->grad.alloc(NPARAM);
    g->adam_m.alloc(NPARAM);
    g->adam_v.alloc(NPARAM);
    g->X.alloc(NF * n);
    g->Xn.alloc(NF * n);
    g->Y.alloc(NO * n);
    g->Tg.alloc(NO * n);
    g->dY.alloc(NO * n);
    for (auto *b : {&g->dH, &g->dHn, &g->dM}) b->alloc(WD * n);
    for (int l = 0; l <= NL; ++l) {
      g->H[l].alloc(WD * n);
      if (l) {
        g->M[l].alloc(WD * n);
        g->Z[l].alloc(WD * n);
      }
    }
    g->part.alloc((size_t)256 * (2 * WD + 1) * WD);
    g->dpart.alloc(nblk(NO * n) + 16 * 256);
    g->sc.alloc(3);
    g->dU.alloc(3 * n);
    g->dloss.alloc(1);
    for (auto *b : {&g->T, &g->Tp, &g->visc, &g->Pp, &g->Pn, &g->P0, &g->Tin, &g->viscin}) b->alloc(n);
    for (auto *b : {&g->Up, &g->Un, &g->U0}) b->alloc(3 * nn);
  });
  *out = g;
  return rc;
}

void m3_gnn_destroy(m3_gnn *g) {
  if (!g) return;
  (void)hipSetDevice(g->device);
  if (g->stream) (void)hipStreamSynchronize(g->stream);
  hipStream_t s = g->stream;
  g->stream = nullptr;
  delete g;  // buffers are freed by their destructors
  if (s) (void)hipStreamDestroy(s);
}

const char *m3_gnn_last_error(const m3_gnn *g) { return g ? g->err.c_str() : "null network"; }

int m3_gnn_set_params(m3_gnn *g, const float *params, const float *norm) {
  return gguard(g, [&] {
    M3_REQUIRE(params, M3_E_ARG, "null parameters");
    M3_REQUIRE(norm || !g->h_norm.empty(), M3_E_ARG, "null normalisation and none fitted");
    if (norm) {
      for (int k = 0; k < NF; ++k) M3_REQUIRE(norm[NF + k] > 0, M3_E_ARG, "in_sigma must be positive");
      for (int k = 0; k < NO; ++k) M3_REQUIRE(norm[2 * NF + k] > 0, M3_E_ARG, "out_sigma must be positive");
      g->h_norm.assign(norm, norm + NNORM);
      g->norm.upload(g->h_norm);
    }
    g->h_prm.assign(params, params + NPARAM);
    g->prm.upload(g->h_prm);
    g->adam_m.zero(g->stream);
    g->adam_v.zero(g->stream);
    g->adam_t = 0;
    HIPCHECK(hipStreamSynchronize(g->stream));
  });
}

int m3_gnn_get_params(m3_gnn *g, float *params, float *norm) {
  return gguard(g, [&] {
    HIPCHECK(hipStreamSynchronize(g->stream));
    if (params) {
      require_params(g);
      g->prm.download(params, NPARAM);
    }
    if (norm) {
      M3_REQUIRE(!g->h_norm.empty(), M3_E_STATE, "normalisation not set");
      g->norm.download(norm, NNORM);
    }
  });
}

int m3_gnn_features(m3_gnn *g, const double *T, const double *T_prev, const double *Visc, const double *U_prev,
                    const double *P_prev, float *X, double *scales) {
  return gguard(g, [&] {
    upload_state(g, T, T_prev, Visc, U_prev, P_prev);
    features_to(g, g->X.p);
    HIPCHECK(hipGetLastError());
    if (X) HIPCHECK(hipMemcpyAsync(X, g->X.p, sizeof(float) * NF * g->n, hipMemcpyDeviceToHost, g->stream));
    if (scales) HIPCHECK(hipMemcpyAsync(scales, g->sc.p, sizeof(double) * 3, hipMemcpyDeviceToHost, g->stream));
    HIPCHECK(hipStreamSynchronize(g->stream));
  });
}

int m3_gnn_reserve(m3_gnn *g, int32_t nmax) {
  return gguard(g, [&] {
    M3_REQUIRE(nmax > 0, M3_E_ARG, "nsample_max must be positive");
    g->sX.alloc((size_t)nmax * NF * g->n);
    g->sY.alloc((size_t)nmax * NO * g->n);
    g->nsample = nmax;
  });
}

int m3_gnn_add_sample(m3_gnn *g, int32_t idx, const double *T, const double *T_prev, const double *Visc,
                      const double *U_prev, const double *P_prev, const double *U_next, const double *P_next) {
  return gguard(g, [&] {
    M3_REQUIRE(idx >= 0 && idx < g->nsample, M3_E_ARG, "sample index out of range (m3_gnn_reserve)");
    M3_REQUIRE(U_next && P_next, M3_E_ARG, "null argument");
    upload_state(g, T, T_prev, Visc, U_prev, P_prev);
    hipStream_t s = g->stream;
    const int64_t n = g->n;
    HIPCHECK(hipMemcpyAsync(g->Un.p, U_next, sizeof(double) * 3 * n, hipMemcpyHostToDevice, s));
    HIPCHECK(hipMemcpyAsync(g->Pn.p, P_next, sizeof(double) * n, hipMemcpyHostToDevice, s));
    features_to(g, g->sX.p + (size_t)idx * NF * n);
    hipLaunchKernelGGL(k_targets, dim3(nblk(n)), dim3(256), 0, s, n, g->Up.p, g->Pp.p, g->Un.p, g->Pn.p, g->sc.p,
                       g->sY.p + (size_t)idx * NO * n);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(s));
  });
}

int m3_gnn_fit_norm(m3_gnn *g, int32_t ns) {
  return gguard(g, [&] {
    M3_REQUIRE(ns > 0 && ns <= g->nsample, M3_E_ARG, "nsample out of range");
    const int64_t rows = (int64_t)ns * g->n;
    std::vector<float> nrm(NNORM);
    for (int pass = 0; pass < 2; ++pass) {
      const int C = pass ? NO : NF;
      hipLaunchKernelGGL(k_chan_stats, dim3(256), dim3(256), 0, g->stream, rows, pass ? g->sY.p : g->sX.p, C,
                         g->dpart.p);
      HIPCHECK(hipGetLastError());
      std::vector<double> part(16 * 256);
      HIPCHECK(hipMemcpyAsync(part.data(), g->dpart.p, sizeof(double) * part.size(), hipMemcpyDeviceToHost,
                              g->stream));
      HIPCHECK(hipStreamSynchronize(g->stream));
      for (int c = 0; c < C; ++c) {
        double s = 0, q = 0;
        for (int b = 0; b < 256; ++b) {
          s += part[16 * b + c];
          q += part[16 * b + 8 + c];
        }
        const double mean = s / (double)rows, var = std::max(q / (double)rows - mean * mean, 0.0);
        if (pass == 0) {
          nrm[c] = (float)mean;
          nrm[NF + c] = var > 1e-24 ? (float)std::sqrt(var) : 1.f;
        } else {
          const double rms = std::sqrt(q / (double)rows);
          nrm[2 * NF + c] = rms > 1e-12 ? (float)rms : 1.f;
        }
      }
    }
    g->h_norm = nrm;
    g->norm.upload(nrm);
  });
}

int m3_gnn_train(m3_gnn *g, const int32_t *samples, int32_t nsteps, float lr, float *loss) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE(samples && nsteps >= 0, M3_E_ARG, "bad sample list");
    for (int32_t k = 0; k < nsteps; ++k)
      M3_REQUIRE(samples[k] >= 0 && samples[k] < g->nsample, M3_E_ARG, "sample index out of range");
    DBuf<float> dl;
    dl.alloc(std::max(nsteps, 1));
    const int64_t n = g->n;
    for (int32_t k = 0; k < nsteps; ++k) {
      const size_t sidx = (size_t)samples[k];
      forward(g, g->sX.p + sidx * NF * n);
      loss_and_backward(g, g->sY.p + sidx * NO * n, dl.p + k);
      adam_step(g, lr);
    }
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(g->stream));  // plain copies do not wait for this stream
    if (loss && nsteps) dl.download(loss, nsteps);
    g->h_prm.resize(NPARAM);
    g->prm.download(g->h_prm.data(), NPARAM);
  });
}

int m3_gnn_sample_stats(m3_gnn *g, const int32_t *samples, int32_t ns, double *out) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE(samples && ns > 0 && out, M3_E_ARG, "bad arguments");
    const int64_t n = g->n;
    constexpr int NB = 64;
    std::vector<double> acc(3 * NO, 0.0), part(3 * NO * NB);
    for (int32_t k = 0; k < ns; ++k) {
      M3_REQUIRE(samples[k] >= 0 && samples[k] < g->nsample, M3_E_ARG, "sample index out of range");
      const size_t sidx = (size_t)samples[k];
      forward(g, g->sX.p + sidx * NF * n);
      hipLaunchKernelGGL(k_chan_dot, dim3(NB), dim3(256), 0, g->stream, n, g->Y.p, g->sY.p + sidx * NO * n,
                         g->norm.p, g->dpart.p);
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipMemcpyAsync(part.data(), g->dpart.p, sizeof(double) * part.size(), hipMemcpyDeviceToHost,
                              g->stream));
      HIPCHECK(hipStreamSynchronize(g->stream));
      for (int b = 0; b < NB; ++b)
        for (int q = 0; q < 3 * NO; ++q) acc[q] += part[3 * NO * b + q];
    }
    for (int q = 0; q < 3 * NO; ++q) out[q] = acc[q];
  });
}

int m3_gnn_eval(m3_gnn *g, const int32_t *samples, int32_t ns, float *loss) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE(samples && ns > 0 && loss, M3_E_ARG, "bad arguments");
    const int64_t n = g->n, ne = NO * n;
    double tot = 0;
    for (int32_t k = 0; k < ns; ++k) {
      M3_REQUIRE(samples[k] >= 0 && samples[k] < g->nsample, M3_E_ARG, "sample index out of range");
      const size_t sidx = (size_t)samples[k];
      forward(g, g->sX.p + sidx * NF * n);
      const int nb = nblk(ne);
      hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, g->stream, n, g->Y.p, g->sY.p + sidx * NO * n, g->norm.p,
                         1.f, g->dY.p, g->dpart.p);
      hipLaunchKernelGGL(k_loss_fin, dim3(1), dim3(256), 0, g->stream, nb, g->dpart.p, (double)ne, g->dloss.p);
      float l = 0;
      HIPCHECK(hipMemcpyAsync(&l, g->dloss.p, sizeof(float), hipMemcpyDeviceToHost, g->stream));
      HIPCHECK(hipStreamSynchronize(g->stream));
      tot += l;
    }
    *loss = (float)(tot / ns);
  });
}

int m3_gnn_forward_backward(m3_gnn *g, const float *X, const float *Y, float *pred, float *loss, float *grad) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE(X && Y, M3_E_ARG, "null argument");
    const int64_t n = g->n;
    g->X.upload(X, NF * n);
    g->Tg.upload(Y, NO * n);
    forward(g, g->X.p);
    loss_and_backward(g, g->Tg.p, g->dloss.p);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(g->stream));
    if (pred) g->Y.download(pred, NO * n);
    if (loss) g->dloss.download(loss, 1);
    if (grad) g->grad.download(grad, NPARAM);
  });
}

int m3_gnn_warm_start(m3_gnn *g, const double *T, const double *T_prev, const double *Visc, const double *U_prev,
                      const double *P_prev, double *U0, double *P0) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE((U0 == nullptr) == (P0 == nullptr), M3_E_ARG, "U0 and P0 must both be given or both be NULL");
    upload_state(g, T, T_prev, Visc, U_prev, P_prev);
    features_to(g, g->X.p);
    forward(g, g->X.p);
    apply_and_download(g, U0, P0);
  });
}

int m3_gnn_clear_history(m3_gnn *g) {
  return gguard(g, [&] {
    g->nhist = 0;
    g->head = 0;
  });
}

int m3_gnn_push_state(m3_gnn *g, double t, const double *T, const double *U, const double *P) {
  return gguard(g, [&] {
    M3_REQUIRE(T && U && P, M3_E_ARG, "null argument");
    M3_REQUIRE(std::isfinite(t), M3_E_ARG, "time must be finite");
    if (g->nhist) M3_REQUIRE(t > g->ht[(g->head + NH - 1) % NH], M3_E_ARG, "times of pushed states must increase");
    const int s = g->head;
    const int64_t n = g->n, nn = g->nnod;
    if (!g->hU[s].p) {
      g->hT[s].alloc(n);
      g->hU[s].alloc(3 * nn);
      g->hP[s].alloc(n);
    }
    HIPCHECK(hipMemcpyAsync(g->hT[s].p, T, sizeof(double) * n, hipMemcpyHostToDevice, g->stream));
    HIPCHECK(hipMemcpyAsync(g->hU[s].p, U, sizeof(double) * 3 * nn, hipMemcpyHostToDevice, g->stream));
    HIPCHECK(hipMemcpyAsync(g->hP[s].p, P, sizeof(double) * n, hipMemcpyHostToDevice, g->stream));
    HIPCHECK(hipStreamSynchronize(g->stream));
    g->ht[s] = t;
    g->head = (s + 1) % NH;
    g->nhist = std::min(g->nhist + 1, NH);
  });
}

int m3_gnn_extrapolate(m3_gnn *g, double t, int32_t order, double *T_base, double *U_base, double *P_base) {
  return gguard(g, [&] {
    make_base(g, t, order, false);
    hipStream_t s = g->stream;
    const int64_t n = g->n, nn = g->nnod;
    HIPCHECK(hipGetLastError());
    if (!T_base && !U_base && !P_base) {  // the base state becomes the device start
      HIPCHECK(hipMemcpyAsync(g->U0.p, g->Up.p, sizeof(double) * 3 * nn, hipMemcpyDeviceToDevice, s));
      HIPCHECK(hipMemcpyAsync(g->P0.p, g->Pp.p, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
      HIPCHECK(hipStreamSynchronize(s));
      g->have_start = true;
      return;
    }
    if (T_base) HIPCHECK(hipMemcpyAsync(T_base, g->Tp.p, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    if (U_base) HIPCHECK(hipMemcpyAsync(U_base, g->Up.p, sizeof(double) * 3 * nn, hipMemcpyDeviceToHost, s));
    if (P_base) HIPCHECK(hipMemcpyAsync(P_base, g->Pp.p, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
  });
}

int m3_gnn_add_sample_hist(m3_gnn *g, int32_t idx, double t, int32_t order, const double *T, const double *Visc,
                           const double *U_next, const double *P_next) {
  return gguard(g, [&] {
    M3_REQUIRE(idx >= 0 && idx < g->nsample, M3_E_ARG, "sample index out of range (m3_gnn_reserve)");
    M3_REQUIRE(U_next && P_next, M3_E_ARG, "null argument");
    upload_new(g, T, Visc);
    make_base(g, t, order);
    hipStream_t s = g->stream;
    const int64_t n = g->n;
    HIPCHECK(hipMemcpyAsync(g->Un.p, U_next, sizeof(double) * 3 * n, hipMemcpyHostToDevice, s));
    HIPCHECK(hipMemcpyAsync(g->Pn.p, P_next, sizeof(double) * n, hipMemcpyHostToDevice, s));
    features_to(g, g->sX.p + (size_t)idx * NF * n);
    hipLaunchKernelGGL(k_targets, dim3(nblk(n)), dim3(256), 0, s, n, g->Up.p, g->Pp.p, g->Un.p, g->Pn.p, g->sc.p,
                       g->sY.p + (size_t)idx * NO * n);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(s));
  });
}

int m3_gnn_warm_start_hist(m3_gnn *g, double t, int32_t order, const double *T, const double *Visc, double *U0,
                           double *P0) {
  return gguard(g, [&] {
    require_params(g);
    M3_REQUIRE((U0 == nullptr) == (P0 == nullptr), M3_E_ARG, "U0 and P0 must both be given or both be NULL");
    upload_new(g, T, Visc);
    make_base(g, t, order);
    features_to(g, g->X.p);
    forward(g, g->X.p);
    apply_and_download(g, U0, P0);
  });
}

int m3_gnn_set_inputs(m3_gnn *g, const double *T, const double *Visc) {
  return gguard(g, [&] {
    M3_REQUIRE(T && Visc, M3_E_ARG, "null argument");
    check_visc(Visc, g->n);
    HIPCHECK(hipMemcpyAsync(g->Tin.p, T, sizeof(double) * g->n, hipMemcpyHostToDevice, g->stream));
    HIPCHECK(hipMemcpyAsync(g->viscin.p, Visc, sizeof(double) * g->n, hipMemcpyHostToDevice, g->stream));
    HIPCHECK(hipStreamSynchronize(g->stream));
    g->have_inputs = true;
  });
}

int m3_gnn_start_device(m3_gnn *g, const double **U0_dev, const double **P0_dev) {
  return gguard(g, [&] {
    M3_REQUIRE(U0_dev && P0_dev, M3_E_ARG, "null argument");
    M3_REQUIRE(g->have_start, M3_E_STATE, "no warm start computed yet");
    *U0_dev = g->U0.p;
    *P0_dev = g->P0.p;
  });
}

}  // extern "C"
