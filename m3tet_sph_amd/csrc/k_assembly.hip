// Element assembly of the double-Jacobian P2P1 Stokes operators and the
// element-local Galerkin coarse operators, for gfx950.
//
// One wavefront per element.  Per integration point (14, Gellert & Harbord;
// ip_tetrahedron.m:100-122) the wave builds the double Jacobian
//   dN/dx = J_SC * inv(J_SL) * dN/dxi
// (assembly_stokes_els_out_cone_no_cross_2pi_opt.m:93-164) in the frame of
// the element's class, maps the gradients back to the original Cartesian
// frame (the un-rotation of ..._cross_2pi_opt.m:385-429 and
// ..._in_cone_no_iso_opt.m:390-496 applied to the gradient vectors instead of
// to the packed matrices), and forms in LDS
//   K  = sum_ip w eta (B' D B)      (30x30, '23rd' or '221' D matrix)
//   G  = sum_ip w NP (dN/dx)        (30x4)
//   M  = sum_ip (w/eta) NP NP'      (4x4)
//   Fb = sum_ip w Fg r_hat N        (30)
// It then applies the node rotations RR' . RR of flow3d_patera_mg_sph_p.m:
// 233-243, lifts the prescribed velocities into bc_rhs (:280-283), removes
// the fixed dofs (:297-298) and scatter-adds the G, GT and M blocks into the
// sliced block-sparse operators.  The rotated, masked element matrix Kel is
// kept (node blocks a >= b, KEL layout); the finest K is summed from it row
// by row (k_gatherK, no global atomics) and the element-local Galerkin
// product of the next multigrid level reads it too.
#include "m3_internal.h"

#include <cmath>

namespace {

constexpr int NIP = 14;

__constant__ double c_ipw[NIP];
__constant__ double c_N10[NIP][10];
__constant__ double c_dN10[NIP][10][3];
__constant__ double c_N4[NIP][4];
__constant__ double c_N20[NIP][20];
__constant__ double c_dN20[NIP][20][3];
__constant__ double c_dN4[4][3];
__constant__ uint16_t c_bq[KEL];  // stored element-matrix index -> (p | q<<8), block layout (KEL)

// ---- host restatement of the shape-function tables --------------------------

void ip_rule(double ipx[3][NIP], double ipw[NIP]) {
  // ip_tetrahedron.m:105-122 (degree 5, 14 points), weights / 6 (:189-191)
  const double g = 1.0 / (46.0 * std::sqrt(46.0));
  const double h = std::acos(g) + (2.0 / 3.0) * std::asin(g);
  const double k = (104.0 + 8.0 * std::sqrt(46.0) * std::cos(h)) / 3.0;
  const double s = std::sqrt(49.0 - k);
  const double b = (7.0 + s) / k, a = 1.0 - 3.0 * b;
  const double d = (7.0 - s) / k, c = 1.0 - 3.0 * d;
  const double p = (98.0 - k - 14.0 * s) / (1680.0 * s * std::pow(b - a, 3));
  const double q = (98.0 - k + 14.0 * s) / (1680.0 * s * std::pow(c - d, 3));
  const double r = (1.0 - 4.0 * (p + q)) / 6.0;
  const double e = (1.0 + std::pow(2.0 / (105.0 * r), 0.25)) / 4.0;
  const double f = (1.0 - 2.0 * e) / 2.0;
  const double X[3][NIP] = {{a, b, b, b, c, d, d, d, e, e, e, f, f, f},
                            {b, a, b, b, d, c, d, d, e, f, f, e, e, f},
                            {b, b, a, b, d, d, c, d, f, e, f, e, f, e}};
  const double W[NIP] = {p, p, p, p, q, q, q, q, r, r, r, r, r, r};
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < NIP; ++j) ipx[i][j] = X[i][j];
  for (int j = 0; j < NIP; ++j) ipw[j] = W[j] / 6.0;
}

void sf10(double r, double s, double t, double N[10], double dN[10][3]) {
  // 10-node tetrahedron, node order of sf_dsf_tet.m:829-840
  const double u = 1.0 - r - s - t;
  const double NN[10] = {r * (2 * r - 1), s * (2 * s - 1), t * (2 * t - 1), u * (2 * u - 1),
                         4 * r * s, 4 * s * t, 4 * t * u, 4 * r * u, 4 * r * t, 4 * s * u};
  const double D[10][3] = {{4 * r - 1, 0, 0}, {0, 4 * s - 1, 0}, {0, 0, 4 * t - 1},
                           {1 - 4 * u, 1 - 4 * u, 1 - 4 * u}, {4 * s, 4 * r, 0},
                           {0, 4 * t, 4 * s}, {-4 * t, -4 * t, 4 * (u - t)},
                           {4 * (u - r), -4 * r, -4 * r}, {4 * t, 0, 4 * r},
                           {-4 * s, 4 * (u - s), -4 * s}};
  for (int i = 0; i < 10; ++i) {
    N[i] = NN[i];
    for (int j = 0; j < 3; ++j) dN[i][j] = D[i][j];
  }
}

void sf20(double r, double s, double t, double N[20], double dN[20][3]) {
  // 20-node (cubic) tetrahedron: vertices, two nodes per edge, face centres
  const double u = 1.0 - r - s - t;
  auto cv = [](double x) { return x * (3 * x - 2) * (1.5 * x - 0.5); };
  auto ce = [](double x, double y, double z) { return x * y * (13.5 * z - 4.5); };
  const double NN[20] = {cv(r), cv(s), cv(t), cv(u),
                         ce(r, s, r), ce(r, s, s), ce(s, t, s), ce(s, t, t),
                         ce(t, u, t), ce(t, u, u), ce(r, u, u), ce(r, u, r),
                         ce(r, t, r), ce(r, t, t), ce(s, u, u), ce(s, u, s),
                         27 * s * t * u, 27 * r * t * u, 27 * r * s * u, 27 * r * s * t};
  // derivatives w.r.t. (r,s,t) with u = 1-r-s-t, by the product rule
  auto dcv = [](double x) { return 13.5 * x * x - 9 * x + 1; };  // d/dx of cv
  // edge function e(x,y,z=x or y) = x*y*(13.5 z - 4.5)
  double D[20][3] = {};
  D[0][0] = dcv(r);
  D[1][1] = dcv(s);
  D[2][2] = dcv(t);
  for (int j = 0; j < 3; ++j) D[3][j] = -dcv(u);
  // helper to accumulate derivative of x*y*(13.5 z - 4.5) where x,y,z are
  // among {r,s,t,u}; grad of variable v: r->(1,0,0) ... u->(-1,-1,-1)
  auto grad = [](int v, double g[3]) {
    g[0] = g[1] = g[2] = 0;
    if (v < 3) g[v] = 1;
    else g[0] = g[1] = g[2] = -1;
  };
  const double var[4] = {r, s, t, u};
  const int E[12][3] = {{0, 1, 0}, {0, 1, 1}, {1, 2, 1}, {1, 2, 2}, {2, 3, 2}, {2, 3, 3},
                        {0, 3, 3}, {0, 3, 0}, {0, 2, 0}, {0, 2, 2}, {1, 3, 3}, {1, 3, 1}};
  for (int k = 0; k < 12; ++k) {
    const int a = E[k][0], b = E[k][1], z = E[k][2];
    double ga[3], gb[3], gz[3];
    grad(a, ga);
    grad(b, gb);
    grad(z, gz);
    const double x = var[a], y = var[b], w = 13.5 * var[z] - 4.5;
    for (int j = 0; j < 3; ++j)
      D[4 + k][j] = ga[j] * y * w + x * gb[j] * w + x * y * 13.5 * gz[j];
  }
  const int F[4][3] = {{1, 2, 3}, {0, 2, 3}, {0, 1, 3}, {0, 1, 2}};
  for (int k = 0; k < 4; ++k) {
    const int a = F[k][0], b = F[k][1], z = F[k][2];
    double ga[3], gb[3], gz[3];
    grad(a, ga);
    grad(b, gb);
    grad(z, gz);
    for (int j = 0; j < 3; ++j)
      D[16 + k][j] = 27 * (ga[j] * var[b] * var[z] + var[a] * gb[j] * var[z] +
                           var[a] * var[b] * gz[j]);
  }
  for (int i = 0; i < 20; ++i) {
    N[i] = NN[i];
    for (int j = 0; j < 3; ++j) dN[i][j] = D[i][j];
  }
}

// ---- device helpers -----------------------------------------------------------

// slot of block (row, colv), -1 when the pattern has none (columns of a row are sorted)
__device__ inline int64_t sell_find(const SellView &K, int row, int colv) {
  const int64_t base = sell_base(K, row);
  int lo = 0, hi = K.rowlen[row] - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const int c = K.col[base + (int64_t)mid * 64];
    if (c == colv) return base + (int64_t)mid * 64;
    if (c < colv) lo = mid + 1;
    else hi = mid - 1;
  }
  return -1;
}

__device__ inline void cart2sph(double x, double y, double z, double &th, double &ph,
                                double &r) {
  r = sqrt(x * x + y * y + z * z);
  th = atan2(sqrt(x * x + y * y), z);
  ph = atan2(y, x);
  if (ph < 0) ph += 2.0 * M_PI;
}

struct AsmArgs {
  int64_t nel;
  const int32_t *el2nod;
  const uint8_t *cls;
  const int32_t *iso_idx;
  const double *X, *S, *X20, *frames, *visc, *dens, *mask, *U0;
  double g, Bscale, Dens0, minV, maxV, C2;
  // embedded refined region (MESH.els_ref): NULL for none; else per element
  // 1 inside / 0 outside and the reference density NUMSCALE.Dens0_T_bary
  const uint8_t *ref_in;
  const double *ref_d0;
  int hasMin, hasMax;
  SellView K, G, GT, M;
  const int32_t *slots;  // ASM_SLOTS per element
  double *Fb, *bc_rhs, *Kel;
  double *dbgK, *dbgG, *dbgM, *dbgF;
  int write_global;
  int scatterG;            // add the element's G and G' (0: they are already assembled)
  int scatterK;          // 0: K is summed afterwards from Kel by k_gatherK
  int *err;
};

// order the LDS accesses of one wave (the waves of a workgroup hold different elements)
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One wave per element, four elements per workgroup.  The geometry (one lane
// per integration point) is done by one of the four waves for all of them, 56
// of its 64 lanes busy (alone, 14 lanes hold a wave through two sincos and three
// divisions); the spherical coordinates of the nodes are formed before, a lane
// per node.  K is formed per lane as a 3x3 node block from
//   S = sum_ip w eta g_a g_b'   ->   K = tr(S) I + S' + C2 S,
// 12 operations per point instead of 33 for the nine entries one by one, and
// stays in registers through the rotation.  The lift of prescribed velocities
// and the removal of fixed dofs run only in elements that have any, G only when
// it is asked for.  245,760 elements: 1.44 ms -> 1.05 ms (0.22 of it the atomics
// of Fb and M, 0.13 the store of Kel, 0.97 GB); Kel's bytes alone are 0.17 ms at
// the copy rate.  Bound by latency: five waves per SIMD, six would spill (slower).
constexpr int EPB = 4;
__global__ __launch_bounds__(64 * EPB, 5) void k_assemble(AsmArgs a) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t e_ = (int64_t)blockIdx.x * EPB + wv;
  const bool live = e_ < a.nel;
  const int64_t e = live ? e_ : a.nel - 1;
  __shared__ int s_nodA[EPB][10], s_cls[EPB];
  __shared__ double s_ipA[EPB][NIP][7];  // w eta, w, w / eta, w Fg, r_hat
  // gradients at the points [NIP][10][3] and the Jacobian products [NIP][9]
  // (rows original-frame x_i, columns d xi_k), then the element matrix (KEL
  // layout: block (na >= nb) at 9 (na (na+1)/2 + nb), entry 3c+d) in their
  // place; before the gradients, the spherical coordinates of the mapping's
  // nodes [20][3] and the viscosity and density of the vertices [8]
  __shared__ double s_buf[EPB][NIP * 39];
  __shared__ double s_RRA[EPB][10][9];
  int *s_nod = s_nodA[wv];
  double(*s_RR)[9] = s_RRA[wv];
  double(*s_ip)[7] = s_ipA[wv];
  double(*s_g)[10][3] = reinterpret_cast<double(*)[10][3]>(s_buf[wv]);
  double(*s_J)[9] = reinterpret_cast<double(*)[9]>(s_buf[wv] + NIP * 30);
  double *s_Kl = s_buf[wv];
  double(*s_sph)[3] = reinterpret_cast<double(*)[3]>(s_buf[wv]);
  static_assert(KEL <= NIP * 39, "element matrix in the gradients' place");

  const int cls = a.cls[e];
  if (lane < 10) s_nod[lane] = a.el2nod[e * 10 + lane];
  if (lane == 0) s_cls[wv] = cls;
  wave_sync();
  // fixed dofs of the element, and whether any of them has a value
  double msk = 1.0, u0 = 0.0;
  if (lane < 30) {
    const int64_t d = 3 * (int64_t)s_nod[lane / 3] + lane % 3;
    msk = a.mask[d];
    u0 = a.U0[d];
  }
  const unsigned fixed = (unsigned)__ballot(msk == 0.0);
  const bool lifts = __ballot(u0 != 0.0) != 0;
  for (int t = lane; t < 90; t += 64) s_RR[t / 9][t % 9] = a.frames[(int64_t)s_nod[t / 9] * 9 + t % 9];
  if (lane >= 32 && lane < 40) {
    const int n = s_nod[lane & 3];
    s_buf[wv][60 + lane - 32] = lane < 36 ? a.visc[n] : a.dens[n];
  }
  // spherical coordinates of the mapping's nodes in the frame of the class
  if (lane < (cls == 3 ? 20 : 4)) {
    double th, ph, rr;
    if (cls >= 2) {  // 90-degree rotation about X: x'=x, y'=-z, z'=y
      const double *x = cls == 3 ? a.X20 + (int64_t)a.iso_idx[e] * 60 + 3 * lane : a.X + 3 * (int64_t)s_nod[lane];
      cart2sph(x[0], -x[2], x[1], th, ph, rr);
    } else {
      const double *sv = a.S + 3 * (int64_t)s_nod[lane];
      th = sv[0];
      ph = sv[1];
      rr = sv[2];
      if (cls == 1) {  // 180-degree rotation about Z
        ph += M_PI;
        if (ph > 2.0 * M_PI) ph -= 2.0 * M_PI;
      }
    }
    s_sph[lane][0] = th;
    s_sph[lane][1] = ph;
    s_sph[lane][2] = rr;
  }
  __syncthreads();

  // ---------------- per-IP geometry: one lane per integration point of the
  // four elements, the workgroups' choice of wave spread over the SIMDs
  if (wv == (int)(blockIdx.x & (EPB - 1)) && lane < EPB * NIP) {
    const int el = lane / NIP, ip = lane - NIP * el, cl = s_cls[el];
    const int64_t ee = (int64_t)blockIdx.x * EPB + el;
    const bool lv = ee < a.nel;
    // J_SL[k][m] = sum_n dN_n/dxi_k * X_m(n) and the IP's interpolated coordinates
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    double thi = 0, phi = 0, ri = 0;
    auto add_node = [&](const double *x, const double *dn, double N) {
      for (int k = 0; k < 3; ++k) {
        J[k][0] += dn[k] * x[0];
        J[k][1] += dn[k] * x[1];
        J[k][2] += dn[k] * x[2];
      }
      thi += N * x[0];
      phi += N * x[1];
      ri += N * x[2];
    };
    if (cl == 3) {
      for (int n = 0; n < 20; ++n) add_node(s_buf[el] + 3 * n, c_dN20[ip][n], c_N20[ip][n]);
    } else {
      for (int n = 0; n < 4; ++n) add_node(s_buf[el] + 3 * n, c_dN4[n], c_N4[ip][n]);
    }
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    if (lv && det < 0) atomicOr(a.err, 1);
    if (lv && thi == 0.0) atomicOr(a.err, 2);
    const double id = 1.0 / det;
    // inv(J_SL)[m][k] = d xi_k / d sph_m
    double I[3][3];
    I[0][0] = id * (J[1][1] * J[2][2] - J[1][2] * J[2][1]);
    I[0][1] = id * (J[0][2] * J[2][1] - J[0][1] * J[2][2]);
    I[0][2] = id * (J[0][1] * J[1][2] - J[0][2] * J[1][1]);
    I[1][0] = id * (J[1][2] * J[2][0] - J[1][0] * J[2][2]);
    I[1][1] = id * (J[0][0] * J[2][2] - J[0][2] * J[2][0]);
    I[1][2] = id * (J[0][2] * J[1][0] - J[0][0] * J[1][2]);
    I[2][0] = id * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    I[2][1] = id * (J[0][1] * J[2][0] - J[0][0] * J[2][1]);
    I[2][2] = id * (J[0][0] * J[1][1] - J[0][1] * J[1][0]);
    // note: I is inv of the matrix with rows k; I[m][k] indexes (row m, col k)
    double st, ct, sp, cp;
    sincos(thi, &st, &ct);
    sincos(phi, &sp, &cp);
    const double dCS = ri * ri * st;
    const double idCS = 1.0 / dCS;
    // J_SC[i][m] = d sph_m / d x_i (class frame)
    const double SC[3][3] = {{ri * st * ct * cp * idCS, -ri * sp * idCS, ri * ri * st * st * cp * idCS},
                             {ri * st * ct * sp * idCS, ri * cp * idCS, ri * ri * st * st * sp * idCS},
                             {-ri * st * st * idCS, 0.0, ri * ri * st * ct * idCS}};
    double D[3][3];
    for (int i = 0; i < 3; ++i)
      for (int k = 0; k < 3; ++k) {
        double acc = 0;
        for (int m = 0; m < 3; ++m) acc += SC[i][m] * I[m][k];
        D[i][k] = acc;
      }
    const double rh[3] = {st * cp, st * sp, ct};
    // class frame -> original frame for gradient rows and r_hat
    double *Jo = s_buf[el] + NIP * 30 + 9 * ip, *po = s_ipA[el][ip];
    const int r1 = cl >= 2 ? 2 : 1, r2 = cl >= 2 ? 1 : 2;  // source rows of rows 1 and 2
    const double s01 = cl == 1 ? -1.0 : 1.0, s2 = cl >= 2 ? -1.0 : 1.0;
    for (int k = 0; k < 3; ++k) {
      Jo[k] = s01 * D[0][k];
      Jo[3 + k] = s01 * (r1 == 2 ? D[2][k] : D[1][k]);
      Jo[6 + k] = s2 * (r2 == 1 ? D[1][k] : D[2][k]);
    }
    const double w = dCS * det * c_ipw[ip];
    double vi = 0, di = 0;
    for (int n = 0; n < 4; ++n) {
      vi += s_buf[el][60 + n] * c_N4[ip][n];
      di += s_buf[el][64 + n] * c_N4[ip][n];
    }
    if (a.hasMin) vi = fmax(vi, a.minV);
    if (a.hasMax) vi = fmin(vi, a.maxV);
    if (lv && !(vi > 0)) atomicOr(a.err, 4);
    // buoyancy (..._out_cone_no_cross_2pi_opt.m:188-195 and the same branch of
    // the other three class kernels): with a refined region, zero outside it
    // and relative to the element's own reference density inside
    double Fg;
    if (a.ref_in)
      Fg = lv && a.ref_in[ee] ? a.g * a.Bscale * (di - a.ref_d0[ee]) : 0.0;
    else
      Fg = a.g * a.Bscale * (di - a.Dens0);
    po[0] = w * vi;
    po[1] = w;
    po[2] = w / vi;
    po[3] = w * Fg;
    po[4] = s01 * rh[0];
    po[5] = s01 * (r1 == 2 ? rh[2] : rh[1]);
    po[6] = s2 * (r2 == 1 ? rh[1] : rh[2]);
  }
  __syncthreads();
  if (!live) return;  // from here on each wave works alone
  // ---------------- gradients in the original frame
  for (int t = lane; t < NIP * 10; t += 64) {
    const int ip = t / 10, n = t % 10;
    for (int i = 0; i < 3; ++i)
      s_g[ip][n][i] = s_J[ip][3 * i] * c_dN10[ip][n][0] + s_J[ip][3 * i + 1] * c_dN10[ip][n][1] +
                      s_J[ip][3 * i + 2] * c_dN10[ip][n][2];
  }
  wave_sync();
  // ---------------- K (original frame): K[(a,c)][(b,d)] =
  //   sum_ip w eta [delta_cd g_a.g_b + g_b[c] g_a[d] + C2 g_b[d] g_a[c]]
  //   one lane per 3x3 node block (na >= nb, 55 blocks)
  int na = (int)((sqrtf(8.0f * (float)lane + 1.0f) - 1.0f) * 0.5f);  // lane = na (na+1)/2 + nb
  if ((na + 1) * (na + 2) / 2 <= lane) ++na;
  if (na * (na + 1) / 2 > lane) --na;
  const int nb = lane - na * (na + 1) / 2;
  double R[3][3];  // the block, rotated to the nodal (theta, phi, r) frames
  if (lane < 55) {
    double S[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll 2
    for (int ip = 0; ip < NIP; ++ip) {
      const double wv_ = s_ip[ip][0];
      const double ga[3] = {wv_ * s_g[ip][na][0], wv_ * s_g[ip][na][1], wv_ * s_g[ip][na][2]};
      const double gb[3] = {s_g[ip][nb][0], s_g[ip][nb][1], s_g[ip][nb][2]};
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) S[c][d] += ga[c] * gb[d];
    }
    const double tr = S[0][0] + S[1][1] + S[2][2];
    double acc[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int d = 0; d < 3; ++d) acc[c][d] = S[d][c] + a.C2 * S[c][d] + (c == d ? tr : 0.0);
    // a diagonal block keeps its lower half (the upper entries mirror it)
    if (na == nb) {
      acc[0][1] = acc[1][0];
      acc[0][2] = acc[2][0];
      acc[1][2] = acc[2][1];
    }
    if (a.dbgK)
      for (int c = 0; c < 3; ++c)
        for (int d = 0; d < 3; ++d) {
          if (na == nb && c < d) continue;
          const int p = 3 * na + c, q = 3 * nb + d;  // p >= q
          a.dbgK[e * 465 + (30 * q - q * (q - 1) / 2 + (p - q))] = acc[c][d];
        }
    double T1[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int dd = 0; dd < 3; ++dd)
        T1[i][dd] = acc[i][0] * s_RR[nb][dd] + acc[i][1] * s_RR[nb][3 + dd] + acc[i][2] * s_RR[nb][6 + dd];
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
      for (int dd = 0; dd < 3; ++dd)
        R[cc][dd] = s_RR[na][cc] * T1[0][dd] + s_RR[na][3 + cc] * T1[1][dd] + s_RR[na][6 + cc] * T1[2][dd];
    if (na == nb) {
      R[0][1] = R[1][0];
      R[0][2] = R[2][0];
      R[1][2] = R[2][1];
    }
  }
  const int32_t *slot = a.slots + e * ASM_SLOTS;  // checked at m3_set_mesh
  // ---------------- G (original frame; scattered rotated, G_rot[a,:,v] = RR_a'
  // G[a,:,v]): it depends on the geometry only, so the host asks for it once
  // per mesh
  if ((a.scatterG || a.dbgG) && lane < 40) {
    const int ga = lane / 4, v = lane % 4;
    double g[3] = {0, 0, 0};
    for (int ip = 0; ip < NIP; ++ip) {
      const double wn = s_ip[ip][1] * c_N4[ip][v];
      for (int c = 0; c < 3; ++c) g[c] += wn * s_g[ip][ga][c];
    }
    if (a.dbgG)
      for (int c = 0; c < 3; ++c) a.dbgG[e * 120 + 30 * v + 3 * ga + c] = g[c];
    if (a.scatterG && a.write_global) {
      const int64_t p1 = slot[100 + lane], p2 = slot[140 + lane];
      for (int cc = 0; cc < 3; ++cc) {
        const double gr = s_RR[ga][cc] * g[0] + s_RR[ga][3 + cc] * g[1] + s_RR[ga][6 + cc] * g[2];
        atomicAdd(a.G.val + cc * a.G.nslot + p1, gr);
        atomicAdd(a.GT.val + cc * a.GT.nslot + p2, gr);
      }
    }
  }
  // ---------------- Fb (rotated) and M
  if (lane < 10) {
    double f[3] = {0, 0, 0};
    for (int ip = 0; ip < NIP; ++ip) {
      const double wn = s_ip[ip][3] * c_N10[ip][lane];
      for (int c = 0; c < 3; ++c) f[c] += wn * s_ip[ip][4 + c];
    }
    if (a.dbgF)
      for (int c = 0; c < 3; ++c) a.dbgF[e * 30 + 3 * lane + c] = f[c];
    if (a.write_global)
      for (int cc = 0; cc < 3; ++cc)
        atomicAdd(&a.Fb[3 * (int64_t)s_nod[lane] + cc],
                  s_RR[lane][cc] * f[0] + s_RR[lane][3 + cc] * f[1] + s_RR[lane][6 + cc] * f[2]);
  } else if (lane >= 32 && lane < 48) {
    const int mv = (lane - 32) / 4, mw = (lane - 32) % 4;
    double mval = 0;
    for (int ip = 0; ip < NIP; ++ip) mval += s_ip[ip][2] * c_N4[ip][mv] * c_N4[ip][mw];
    // packed lower column-major: column mw, row mv
    if (a.dbgM && mv >= mw) a.dbgM[e * 10 + mw * 4 - mw * (mw - 1) / 2 + (mv - mw)] = mval;
    if (a.write_global) atomicAdd(a.M.val + slot[180 + (lane - 32)], mval);
  }
  if (!a.write_global) return;
  auto put = [&] {
    wave_sync();  // the gradients (or the matrix before) have been read
    if (lane < 55) {
      double *blk = s_Kl + 9 * lane;
      for (int cc = 0; cc < 3; ++cc)
        for (int dd = 0; dd < 3; ++dd) blk[3 * cc + dd] = R[cc][dd];
    }
    wave_sync();
  };
  // ---------------- BC lift (bc_rhs = K U0)
  if (lifts) {
    put();
    if (lane < 30) {
      double acc = 0;
      const int la = lane / 3, cc = lane % 3;
      for (int lb = 0; lb < 10; ++lb) {
        // row (la, cc) of block (la, lb): stored block (la, lb), or the
        // transpose of stored block (lb, la) above the diagonal
        const bool lo = la >= lb;
        const double *blk = s_Kl + 9 * (lo ? la * (la + 1) / 2 + lb : lb * (lb + 1) / 2 + la);
        for (int dd = 0; dd < 3; ++dd) acc += (lo ? blk[3 * cc + dd] : blk[3 * dd + cc]) * a.U0[3 * (int64_t)s_nod[lb] + dd];
      }
      if (acc != 0.0) atomicAdd(&a.bc_rhs[3 * (int64_t)s_nod[la] + cc], acc);
    }
  }
  // ---------------- removal of fixed dofs
  if (fixed && lane < 55)
    for (int cc = 0; cc < 3; ++cc)
      for (int dd = 0; dd < 3; ++dd)
        if ((fixed >> (3 * na + cc) | fixed >> (3 * nb + dd)) & 1u) R[cc][dd] *= 0.0;
  put();
  if (a.Kel)
    for (int t = lane; t < KEL; t += 64) a.Kel[e * KEL + t] = s_Kl[t];
  // ---------------- scatter K blocks (unless the row-owner gather k_gatherK sums them)
  for (int t = lane; t < (a.scatterK ? 100 : 0); t += 64) {
    const int ka = t / 10, kb = t % 10;
    const int64_t pos = slot[t];
    const bool lo = ka >= kb;
    const double *blk = s_Kl + 9 * (lo ? ka * (ka + 1) / 2 + kb : kb * (kb + 1) / 2 + ka);
    for (int cc = 0; cc < 3; ++cc)
      for (int dd = 0; dd < 3; ++dd)
        atomicAdd(a.K.val + kval(pos, 3 * cc + dd), lo ? blk[3 * cc + dd] : blk[3 * dd + cc]);
  }
}

// ---- element-local Galerkin product --------------------------------------------
// Coarse element c collects its 8 children e = 8c+k (tetmesh_p2_to_p1.m:112):
//   Kc = mask_c . sum_k (Q_k (x) I3)' K_e (Q_k (x) I3) . mask_c
// which equals Ic2f_U' K Ic2f_U (restrict_stiffmat.m:40-49) because every fine
// node of a child lies in the closure of its parent, where the P2
// interpolation rows of Ic2f are the parent's shape functions.
struct RapArgs {
  int64_t nel_c;
  const double *Kf;        // fine element matrices (KEL layout)
  const int32_t *ctype;    // fine element -> Q table
  const double *Qtab;      // ntypes * 100, Q[i][a] = weight of coarse local a at fine local i
  const int32_t *el2nod_c; // coarse connectivity
  const double *mask_c;
  double *Kc;              // coarse element matrices (KEL layout)
  SellView K;              // coarse operator
  int scatter;             // 1: add the blocks into K with atomics; 0: k_gatherK sums Kc
  int *err;
};

__global__ __launch_bounds__(64) void k_rap(RapArgs a) {
  const int64_t c = blockIdx.x;
  const int lane = threadIdx.x;
  // one 30x31 LDS matrix: T of each child, then the coarse matrix (7.8 KB in
  // all, so that many waves share a CU); the child matrices are read from
  // their contiguous 4 KB blocks in global memory
  __shared__ double s_T[30][31];
  __shared__ double s_Q[10][10];
  __shared__ int s_nod[10];
  __shared__ double s_m[30];
  double(*s_Kc)[31] = s_T;
  if (lane < 10) s_nod[lane] = a.el2nod_c[c * 10 + lane];
  __syncthreads();
  if (lane < 30) s_m[lane] = a.mask_c[3 * (int64_t)s_nod[lane / 3] + lane % 3];
  // Register blocking: lane task u (< 90, two per lane) owns in the first
  // product the row p = u / 3, component d = u % 3 of T (ten entries, one
  // per coarse node b) and in the second the component c = u / 30, column
  // q = u % 30 of Kc (ten entries, one per coarse node a), accumulated over
  // the eight children in registers; Q is read from LDS by broadcast.
  // Every entry sums in the same order as an entry-per-lane loop would.
  double kc[2][10];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int aa = 0; aa < 10; ++aa) kc[r][aa] = 0.0;
  for (int k = 0; k < 8; ++k) {
    const int64_t e = 8 * c + k;
    const double *Ke = a.Kf + e * KEL;
    const double *Q = a.Qtab + (int64_t)a.ctype[e] * 100;
    for (int t = lane; t < 100; t += 64) s_Q[t / 10][t % 10] = Q[t];
    // Kf[p][3j+d] with p = 3 na + cc: stored block (na, j) when na >= j,
    // else the transpose of stored block (j, na)
    double kf[2][10];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int u = lane + 64 * r;
      if (u < 90) {
        const int p = u / 3, d = u % 3, na = p / 3, cc = p % 3;
#pragma unroll
        for (int j = 0; j < 10; ++j)
          kf[r][j] = na >= j ? Ke[9 * (na * (na + 1) / 2 + j) + 3 * cc + d] : Ke[9 * (j * (j + 1) / 2 + na) + 3 * d + cc];
      }
    }
    __syncthreads();
    // T[p][(b,d)] = sum_j Kf[p][(j,d)] Q[j][b]
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int u = lane + 64 * r;
      if (u < 90) {
        const int p = u / 3, d = u % 3;
#pragma unroll
        for (int bb = 0; bb < 10; ++bb) {
          double acc = 0;
#pragma unroll
          for (int j = 0; j < 10; ++j) acc += kf[r][j] * s_Q[j][bb];
          s_T[p][3 * bb + d] = acc;
        }
      }
    }
    __syncthreads();
    // Kc[(a,c)][q] += sum_i Q[i][a] T[(i,c)][q]
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int u = lane + 64 * r;
      if (u < 90) {
        const int cc = u / 30, q = u % 30;
        double tv[10];
#pragma unroll
        for (int i = 0; i < 10; ++i) tv[i] = s_T[3 * i + cc][q];
#pragma unroll
        for (int aa = 0; aa < 10; ++aa) {
          double acc = 0;
#pragma unroll
          for (int i = 0; i < 10; ++i) acc += s_Q[i][aa] * tv[i];
          kc[r][aa] += acc;
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int u = lane + 64 * r;
    if (u < 90) {
      const int cc = u / 30, q = u % 30;
#pragma unroll
      for (int aa = 0; aa < 10; ++aa) s_Kc[3 * aa + cc][q] = kc[r][aa];
    }
  }
  __syncthreads();
  for (int t = lane; t < 900; t += 64) {
    const int p = t / 30, q = t % 30;
    s_Kc[p][q] *= s_m[p] * s_m[q];
  }
  __syncthreads();
  if (a.Kc) {
    for (int t = lane; t < KEL; t += 64) {
      const int pq = c_bq[t];
      // symmetrise the rounding of the two triangles
      a.Kc[c * KEL + t] = 0.5 * (s_Kc[pq & 255][pq >> 8] + s_Kc[pq >> 8][pq & 255]);
    }
  }
  for (int t = lane; t < (a.scatter ? 100 : 0); t += 64) {
    const int na = t / 10, nb = t % 10;
    const int64_t pos = sell_find(a.K, s_nod[na], s_nod[nb]);
    if (pos < 0) { atomicOr(a.err, 8); continue; }
    for (int cc = 0; cc < 3; ++cc)
      for (int dd = 0; dd < 3; ++dd) {
        const double v = 0.5 * (s_Kc[3 * na + cc][3 * nb + dd] + s_Kc[3 * nb + dd][3 * na + cc]);
        atomicAdd(a.K.val + kval(pos, 3 * cc + dd), v);
      }
  }
}

// Finest K summed row by row from the element matrices Kel, without global
// atomics: one wavefront per node row i accumulates its blocks in LDS.  Lane
// work item = (incident element e with i at local node a, local column node
// b); the 3x3 block (a,b) of Kel lands in stored block k of row i, where the
// slot of (a,b) comes from the per-element slot map.  Kel holds the node
// blocks a >= b of the symmetric 30x30 rotated, masked matrix (KEL layout),
// so a work item reads one contiguous 72-byte block.
// Every stored block of the row is written, so K needs no clearing first.
constexpr int GK_ROWS = 4;      // rows (wavefronts) per block
constexpr int GK_MAXLEN = 128;  // stored blocks per row (checked at m3_set_mesh)
__global__ __launch_bounds__(64 * GK_ROWS) void k_gatherK(SellView K, int64_t nrow, const int64_t *inc_ptr,
                                                         const int32_t *inc, const int32_t *slots, int slot_stride,
                                                         const double *Kel) {
  __shared__ double acc[GK_ROWS][GK_MAXLEN * 9];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * GK_ROWS + w;
  const bool live = i < nrow;
  const int len = live ? K.rowlen[i] : 0;
  const int64_t base = live ? sell_base(K, i) : 0;
  double *A = acc[w];
  for (int t = lane; t < len * 9; t += 64) A[t] = 0.0;
  __syncthreads();
  if (live) {
    const int64_t t0 = inc_ptr[i] * 10, t1 = inc_ptr[i + 1] * 10;
    for (int64_t t = t0 + lane; t < t1; t += 64) {
      const int64_t j = t / 10;
      const int b = (int)(t - 10 * j);
      const int ea = inc[j];
      const int64_t e = ea / 10;
      const int na = ea - 10 * (int)e;
      const int k = (int)((slots[e * slot_stride + 10 * na + b] - base) >> 6);
      // block (na, b) of the symmetric element matrix: stored block (hi, lo), transposed when na < b
      const bool lower = na >= b;
      const int hi = lower ? na : b, lo = lower ? b : na;
      const double *kb = Kel + e * KEL + 9 * (hi * (hi + 1) / 2 + lo);
      double v[9];
#pragma unroll
      for (int m = 0; m < 9; ++m) v[m] = kb[m];
#pragma unroll
      for (int cc = 0; cc < 3; ++cc)
#pragma unroll
        for (int dd = 0; dd < 3; ++dd) atomicAdd(&A[9 * k + 3 * cc + dd], lower ? v[3 * cc + dd] : v[3 * dd + cc]);
    }
  }
  __syncthreads();
  for (int t = lane; t < len * 9; t += 64) {
    const int k = t / 9, v = t - 9 * k;
    K.val[kval(base + 64 * (int64_t)k, v)] = A[t];
  }
}

// The same sum with one thread per stored block slot: the slot's sorted list
// of contributing element blocks (each a contiguous 72-byte block of Kel,
// transposed when the element's local row node precedes its column node) is
// added in list order and the nine values are written once, coalesced over
// the slots of a wave; padding slots have empty lists and are never read.  p16
// (finest level): the same block also in the mixed V-cycle's packed BF16
// layout (p16_words, p16_v8).
__global__ __launch_bounds__(256) void k_gatherK_slots(SellView K, const int64_t *cptr, const int32_t *clist,
                                                       const double *Kel, uint32_t *p16) {
  const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (s >= K.nslot) return;
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  const int64_t m0 = cptr[s], m1 = cptr[s + 1];
  if (m0 == m1) return;
  for (int64_t m = m0; m < m1; ++m) {
    const int32_t code = clist[m];
    const double *kb = Kel + 9 * (int64_t)(code >> 1);
    double v[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) v[t] = kb[t];
    if (code & 1) {
#pragma unroll
      for (int cc = 0; cc < 3; ++cc)
#pragma unroll
        for (int dd = 0; dd < 3; ++dd) acc[3 * cc + dd] += v[3 * dd + cc];
    } else {
#pragma unroll
      for (int t = 0; t < 9; ++t) acc[t] += v[t];
    }
  }
  typedef double d2w __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int t = 0; t < 8; t += 2) *reinterpret_cast<d2w *>(K.val + kval(s, t)) = d2w{acc[t], acc[t + 1]};
  K.val[kval(s, 8)] = acc[8];
  if (p16) {
    typedef uint32_t u4w __attribute__((ext_vector_type(4)));
    u4w g;
    g.x = bf16_rne(acc[0]) | (bf16_rne(acc[1]) << 16);
    g.y = bf16_rne(acc[2]) | (bf16_rne(acc[3]) << 16);
    g.z = bf16_rne(acc[4]) | (bf16_rne(acc[5]) << 16);
    g.w = bf16_rne(acc[6]) | (bf16_rne(acc[7]) << 16);
    *reinterpret_cast<u4w *>(p16 + p16_words(s)) = g;
    p16[p16_v8(s)] = __float_as_uint((float)acc[8]);
  }
}

// contribution lists: count, fill (any order), then sort each list so that
// the sum runs in a fixed order
__global__ void k_ccount(int64_t n, const int32_t *slots, int stride, unsigned long long *cnt) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t e = t / 100;
  const int k = (int)(t - 100 * e);
  atomicAdd(&cnt[slots[e * stride + k]], 1ull);
}

__global__ void k_cfill(int64_t n, const int32_t *slots, int stride, unsigned long long *cursor, int32_t *clist) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t e = t / 100;
  const int k = (int)(t - 100 * e), na = k / 10, nb = k % 10;
  const int hi = na >= nb ? na : nb, lo = na >= nb ? nb : na;
  const int64_t pos = (int64_t)atomicAdd(&cursor[slots[e * stride + k]], 1ull);
  clist[pos] = (int32_t)(2 * (e * 55 + hi * (hi + 1) / 2 + lo) + (na < nb ? 1 : 0));
}

__global__ void k_csort(int64_t nslot, const int64_t *cptr, int32_t *clist) {
  const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (s >= nslot) return;
  const int64_t m0 = cptr[s], m1 = cptr[s + 1];
  for (int64_t m = m0 + 1; m < m1; ++m) {
    const int32_t v = clist[m];
    int64_t j = m - 1;
    while (j >= m0 && clist[j] > v) {
      clist[j + 1] = clist[j];
      --j;
    }
    clist[j + 1] = v;
  }
}

__global__ void k_u64_to_i64(int64_t n, const unsigned long long *x, int64_t *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = (int64_t)x[i];
}

__global__ void k_i64_to_u64(int64_t n, const int64_t *x, unsigned long long *y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = (unsigned long long)x[i];
}

// slot of every element block in K (10x10 at [10a+b]), G (10x4 at
// [100+4a+v]), GT (4x10 at [140+4a+v]) and M (4x4 at [180+4v+w]); one thread
// per (element, block), a binary search in the sorted row
__global__ void k_slots(int64_t nel, const int32_t *el2nod, SellView K, SellView G, SellView GT, SellView M,
                        int32_t *slots, int *err) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nel * ASM_SLOTS) return;
  const int64_t e = t / ASM_SLOTS;
  const int k = (int)(t - e * ASM_SLOTS);
  const int32_t *n = el2nod + 10 * e;
  int64_t pos;
  if (k < 100) {
    pos = sell_find(K, n[k / 10], n[k % 10]);
  } else if (k < 140) {
    const int j = k - 100;
    pos = sell_find(G, n[j / 4], n[j % 4]);
  } else if (k < 180) {
    const int j = k - 140;
    pos = sell_find(GT, n[j % 4], n[j / 4]);
  } else {
    const int j = k - 180;
    pos = sell_find(M, n[j / 4], n[j % 4]);
  }
  if (pos < 0) atomicOr(err, 8);
  slots[t] = (int32_t)pos;
}

// K slots of the 100 element blocks of a coarse level (block (a,b) at 10a+b)
__global__ void k_kslots(int64_t nel, const int32_t *el2nod, SellView K, int32_t *slots, int *err) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nel * 100) return;
  const int64_t e = t / 100;
  const int k = (int)(t - e * 100);
  const int64_t pos = sell_find(K, el2nod[10 * e + k / 10], el2nod[10 * e + k % 10]);
  if (pos < 0) atomicOr(err, 8);
  slots[t] = (int32_t)pos;
}

// identity at fixed dofs on the diagonal blocks, inverse diagonal
// fixed dofs get a unit diagonal; p16 (finest level): the packed BF16 copy
// that the slot gather wrote gets the same unit entries (v0 and v4 are the
// low halves of words 0 and 2 of the block's group).  dinv is in
// the level's vector order (vpos: place of each node, NULL for the node order).
__global__ void k_fix_diag(SellView K, const double *mask, const int32_t *vpos, int64_t nnod, double *dinv,
                           uint32_t *p16) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nnod) return;
  const int64_t pos = sell_find(K, (int)i, (int)i);
  if (pos < 0) return;
  const int64_t o = 3 * (vpos ? (int64_t)vpos[i] : i);
  for (int c = 0; c < 3; ++c) {
    double *b = K.val + kval(pos, 4 * c);
    if (mask[3 * i + c] == 0.0) {
      *b = 1.0;
      if (p16) {
        if (c == 2) {
          p16[p16_v8(pos)] = __float_as_uint(1.0f);
        } else {
          uint32_t *wd = p16 + p16_words(pos) + 2 * c;
          *wd = (*wd & 0xffff0000u) | bf16_rne(1.0);
        }
      }
    }
    dinv[o + c] = 1.0 / *b;
  }
}

__global__ void k_lumped(SellView M, int64_t n, double *LiMM) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t base = sell_base(M, i);
  const int len = M.rowlen[i];
  double s = 0;
  for (int k = 0; k < len; ++k) s += M.val[base + (int64_t)k * 64];
  LiMM[i] = 1.0 / s;
}

}  // namespace

namespace m3 {

void upload_sf_tables() {
  double ipx[3][NIP], ipw[NIP];
  ip_rule(ipx, ipw);
  double N10[NIP][10], dN10[NIP][10][3], N4[NIP][4], N20[NIP][20], dN20[NIP][20][3];
  for (int ip = 0; ip < NIP; ++ip) {
    const double r = ipx[0][ip], s = ipx[1][ip], t = ipx[2][ip];
    sf10(r, s, t, N10[ip], dN10[ip]);
    N4[ip][0] = r;
    N4[ip][1] = s;
    N4[ip][2] = t;
    N4[ip][3] = 1.0 - r - s - t;
    sf20(r, s, t, N20[ip], dN20[ip]);
  }
  const double dN4[4][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {-1, -1, -1}};
  uint16_t bq[KEL];
  int idx = 0;
  for (int na = 0; na < 10; ++na)
    for (int nb = 0; nb <= na; ++nb)
      for (int cc = 0; cc < 3; ++cc)
        for (int dd = 0; dd < 3; ++dd) bq[idx++] = (uint16_t)((3 * na + cc) | ((3 * nb + dd) << 8));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_bq), bq, sizeof(bq)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_ipw), ipw, sizeof(ipw)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_N10), N10, sizeof(N10)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_dN10), dN10, sizeof(dN10)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_N4), N4, sizeof(N4)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_N20), N20, sizeof(N20)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_dN20), dN20, sizeof(dN20)));
  HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_dN4), dN4, sizeof(dN4)));
}

void launch_assemble(m3_ctx *c, double *dbgK, double *dbgG, double *dbgM, double *dbgF,
                     bool write_global) {
  AsmArgs a{};
  LevelDev &f = c->L[0];
  a.nel = f.nel;
  a.el2nod = f.el2nod.p;
  a.cls = c->cls.p;
  a.iso_idx = c->iso_idx.p;
  a.X = c->X.p;
  a.S = c->S.p;
  a.X20 = c->X20.p;
  a.frames = c->frames.p;
  a.visc = c->visc.p;
  a.dens = c->dens.p;
  a.mask = f.mask.p;
  a.U0 = c->U0.p;
  a.g = c->phys.g;
  a.Bscale = c->phys.Bscale;
  a.Dens0 = c->phys.Dens0;
  a.ref_in = c->have_ref ? c->ref_in.p : nullptr;
  a.ref_d0 = c->have_ref ? c->ref_d0.p : nullptr;
  a.minV = c->phys.minVisc;
  a.maxV = c->phys.maxVisc;
  a.hasMin = c->phys.has_minVisc;
  a.hasMax = c->phys.has_maxVisc;
  a.C2 = c->phys.type_Dmat == 0 ? -2.0 / 3.0 : 0.0;
  a.K = f.K.view();
  a.slots = c->asm_slots.p;
  a.G = c->G.view();
  a.GT = c->GT.view();
  a.M = c->M.view();
  a.Fb = c->Fb.p;
  a.bc_rhs = c->bc_rhs.p;
  a.Kel = write_global ? f.Kel.p : nullptr;
  a.dbgK = dbgK;
  a.dbgG = dbgG;
  a.dbgM = dbgM;
  a.dbgF = dbgF;
  a.write_global = write_global ? 1 : 0;
  a.scatterK = c->gather_K ? 0 : 1;
  a.scatterG = write_global && !c->g_valid ? 1 : 0;
  a.err = c->errflag.p;
  hipLaunchKernelGGL(k_assemble, dim3((unsigned)((f.nel + EPB - 1) / EPB)), dim3(64 * EPB), 0, c->stream, a);
  HIPCHECK(hipGetLastError());
}

void launch_rap(m3_ctx *c, int l) {
  LevelDev &f = c->L[l];
  LevelDev &cl = c->L[l + 1];
  RapArgs a{};
  a.nel_c = cl.nel;
  a.Kf = f.Kel.p;
  a.ctype = f.child_type.p;
  a.Qtab = f.Qtab.p;
  a.el2nod_c = cl.el2nod.p;
  a.mask_c = cl.mask.p;
  a.Kc = (cl.gather || l + 1 < c->nmg - 1) ? cl.Kel.p : nullptr;
  a.K = cl.K.view();
  a.scatter = cl.gather ? 0 : 1;
  a.err = c->errflag.p;
  hipLaunchKernelGGL(k_rap, dim3((unsigned)cl.nel), dim3(64), 0, c->stream, a);
  HIPCHECK(hipGetLastError());
}

void launch_gather_K(m3_ctx *c, int level) {
  LevelDev &f = c->L[level];
  if (level == 0) c->pack16_fresh = false;
  if (f.cptr.p) {
    uint32_t *p16 = nullptr;
    if (level == 0 && c->nmg > 1) {  // the finest level's packed BF16 values, written in the same pass
      if (f.K.val16.n != (size_t)(P16 * f.K.nslot)) f.K.val16.alloc(P16 * f.K.nslot);
      p16 = f.K.val16.p;
    }
    hipLaunchKernelGGL(k_gatherK_slots, dim3((unsigned)((f.K.nslot + 255) / 256)), dim3(256), 0, c->stream,
                       f.K.view(), f.cptr.p, f.clist.p, f.Kel.p, p16);
    HIPCHECK(hipGetLastError());
    if (p16) c->pack16_fresh = true;
    return;
  }
  const bool fine = level == 0;
  hipLaunchKernelGGL(k_gatherK, dim3((unsigned)((f.nnod + GK_ROWS - 1) / GK_ROWS)), dim3(64 * GK_ROWS), 0,
                     c->stream, f.K.view(), f.nnod, fine ? c->inc_ptr.p : f.inc_ptr.p, fine ? c->inc.p : f.inc.p,
                     fine ? c->asm_slots.p : f.kslots.p, fine ? ASM_SLOTS : 100, f.Kel.p);
  HIPCHECK(hipGetLastError());
}

bool build_contrib(m3_ctx *c, int level) {
  LevelDev &f = c->L[level];
  const bool fine = level == 0;
  const int32_t *slots = fine ? c->asm_slots.p : f.kslots.p;
  const int stride = fine ? ASM_SLOTS : 100;
  const int64_t n = 100 * f.nel, nslot = f.K.nslot;
  if (2 * 55 * f.nel >= (int64_t)INT32_MAX || nslot >= (int64_t)INT32_MAX) return false;
  hipStream_t s = c->stream;
  DBuf<unsigned long long> cnt;
  DBuf<int64_t> cnt64;
  cnt.alloc(nslot);
  cnt64.alloc(nslot);
  HIPCHECK(hipMemsetAsync(cnt.p, 0, nslot * sizeof(unsigned long long), s));
  const unsigned gn = (unsigned)((n + 255) / 256), gs = (unsigned)((nslot + 255) / 256);
  hipLaunchKernelGGL(k_ccount, dim3(gn), dim3(256), 0, s, n, slots, stride, cnt.p);
  hipLaunchKernelGGL(k_u64_to_i64, dim3(gs), dim3(256), 0, s, nslot, cnt.p, cnt64.p);
  f.cptr.alloc(nslot + 1);
  const int64_t total = m3::exclusive_scan_device(cnt64.p, nslot, f.cptr.p, s);
  M3_REQUIRE(total == n, M3_E_MESH, "element block without a slot");
  HIPCHECK(hipMemcpyAsync(f.cptr.p + nslot, &total, sizeof(int64_t), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_i64_to_u64, dim3(gs), dim3(256), 0, s, nslot, f.cptr.p, cnt.p);  // cursors
  f.clist.alloc(n);
  hipLaunchKernelGGL(k_cfill, dim3(gn), dim3(256), 0, s, n, slots, stride, cnt.p, f.clist.p);
  hipLaunchKernelGGL(k_csort, dim3(gs), dim3(256), 0, s, nslot, f.cptr.p, f.clist.p);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(s));
  return true;
}

void launch_kslots(m3_ctx *c, int level) {
  LevelDev &f = c->L[level];
  const int64_t nt = f.nel * 100;
  hipLaunchKernelGGL(k_kslots, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, c->stream, f.nel, f.el2nod.p,
                     f.K.view(), f.kslots.p, c->errflag.p);
  HIPCHECK(hipGetLastError());
}

void launch_slots(m3_ctx *c) {
  LevelDev &f = c->L[0];
  const int64_t nt = f.nel * ASM_SLOTS;
  hipLaunchKernelGGL(k_slots, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, c->stream, f.nel, f.el2nod.p,
                     f.K.view(), c->G.view(), c->GT.view(), c->M.view(), c->asm_slots.p, c->errflag.p);
  HIPCHECK(hipGetLastError());
}

void launch_fix_diag(m3_ctx *c, int l) {
  LevelDev &lv = c->L[l];
  const int bs = 256;
  uint32_t *p16 = (l == 0 && c->pack16_fresh) ? lv.K.val16.p : nullptr;
  hipLaunchKernelGGL(k_fix_diag, dim3((unsigned)((lv.nnod + bs - 1) / bs)), dim3(bs), 0,
                     c->stream, lv.K.view(), lv.mask.p, lv.K.vpos_p(), lv.nnod, lv.dinv.p, p16);
  HIPCHECK(hipGetLastError());
}

void launch_lumped_mm(m3_ctx *c) {
  const int bs = 256;
  hipLaunchKernelGGL(k_lumped, dim3((unsigned)((c->nV + bs - 1) / bs)), dim3(bs), 0, c->stream,
                     c->M.view(), c->nV, c->LiMM.p);
  HIPCHECK(hipGetLastError());
}

}  // namespace m3
