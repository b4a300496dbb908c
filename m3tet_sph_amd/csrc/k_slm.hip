// Semi-Lagrangian advection of a field on the P2 nodes of the finest mesh:
// the production configuration of advect3d_slm_p_sph
// (mfiles_SPH/advect3d_slm_p_sph.m:1-140; OPTS_SLM of
// default_numerics_M3TET.m:141-153: PC2 back-tracking, quadratic
// interpolation, monotonic).  One thread per node:
//
//  1. predictor (predictor_step_with_projections, :298-397): the node
//     velocity split into its part along the node's radial unit vector and
//     the rest; the point moved by the great-circle arc |U_perp| dt/2 / r
//     against U_perp (straight length r tan(arc) along the tangent, then
//     back onto the radial line) and to the radius |r - |U_par| dt/2| (the
//     reference's unsigned radial length);
//  2. radii outside [r_cmb, r_surf] (within 1e-12 of the shell thickness)
//     moved to that bound (find_pts_outside_domain_sph.m);
//  3. the point located and the velocity interpolated with the quadratic
//     shape functions (locate_points_interp_vars_3d_sph.m, interp3d_tet.m);
//  4. corrector (corrector_step_with_projections, :399-440): the
//     interpolated velocity split along the predictor point's radial unit
//     vector, moved over dt along the node's own U_perp direction;
//  5. the field interpolated at the departure point and clipped to the
//     element's nodal minimum and maximum (interp3d_tet.m:60-67).
//
// OPTS_SLM.method_BT = 'EU1' replaces steps 1-4 by backtrack_EU1
// (:145-161), a single explicit step in spherical coordinates (k_slm_eu1);
// 'RK4' stops with the reference's message (:104-105), and so do the
// interpolations other than 'quadratic' on P2 fields
// (locate_points_interp_vars_3d_sph.m:147-149).
//
// Location: local coordinates are barycentric coordinates in the spherical
// coordinates of the element's class frame (local_coords_3d_sph.m: the
// original frame with GCOORD_SPH for elements outside the cones, the
// 180-degree Z-rotated frame for those crossing phi = 2 pi, the 90-degree
// X-rotated frame inside the cones; for the isoparametric in-cone elements
// the Newton iteration of local_coords_curved_3d_sph.m on the ten nodes,
// at most six steps, to 1e-8).  The element is found by a walk over face
// neighbours from an element of the node (then from the predictor's
// element): step across the face opposite the most negative coordinate,
// stop when all four are >= -1e-12, at the shell boundary, on returning to
// the previous element or after 64 steps (then the best element seen is
// taken and the search counted as unresolved).  Coordinates are then
// clipped to [0, 1] and rescaled when they sum to more than 1
// (adjust_local_coords, locate_points_interp_vars_3d_sph.m:180-190).  A
// point tested against an element of the original frame takes the phi of
// its own side of the phi = 2 pi meridian (such elements never cross it), so
// the walk is not sent round the sphere by a phi that differs by 2 pi.
#include "m3_internal.h"

#include <algorithm>
#include <cmath>
#include <unordered_map>

namespace {

constexpr int SLM_MAXWALK = 64;

struct SlmArgs {
  int64_t nnod;
  const int32_t *el2nod;
  const uint8_t *cls;
  const double *X, *S, *Sz, *Sx;
  const int32_t *nbr, *start;
  const double *U;  // Cartesian velocity, 3 per node
  const double *T;
  double *Tout;
  double dt, r_cmb, r_surf;
  int monotonic;
  unsigned long long *cnt;
};

struct V3d {
  double x, y, z;
};

__device__ inline V3d ld(const double *a, int64_t i) { return {a[3 * i], a[3 * i + 1], a[3 * i + 2]}; }

__device__ inline V3d c2s(V3d p) {
  const double r = sqrt(p.x * p.x + p.y * p.y + p.z * p.z);
  const double th = atan2(sqrt(p.x * p.x + p.y * p.y), p.z);
  double ph = atan2(p.y, p.x);
  if (ph < 0) ph += 2.0 * M_PI;
  return {th, ph, r};
}

__device__ inline V3d s2c(V3d s) {
  return {s.z * sin(s.x) * cos(s.y), s.z * sin(s.x) * sin(s.y), s.z * cos(s.x)};
}

// the point (original-frame spherical coordinates) in frame f: 0 original,
// 1 Z-rotated (RR_Z_180), 2 X-rotated (RR_X_90_CCW)
__device__ inline V3d in_frame(V3d p, int f) {
  if (f == 0) return p;
  const V3d c = s2c(p);
  return f == 1 ? c2s(V3d{-c.x, -c.y, c.z}) : c2s(V3d{c.x, -c.z, c.y});
}

__device__ inline int frame_of(int cls) { return cls == 0 ? 0 : (cls == 1 ? 1 : 2); }

// barycentric coordinate of vertex i from vertices j, k, m (triple products
// in (theta, phi, r), local_coords_3d_sph.m:125-141)
__device__ inline double bary(const V3d *v, int i, int j, int k, int m, V3d p) {
  const V3d a = v[j], b = v[k], c = v[m], o = v[i];
  const double num = (a.x - p.x) * (b.y - p.y) * (c.z - p.z) + (b.x - p.x) * (c.y - p.y) * (a.z - p.z) +
                     (c.x - p.x) * (a.y - p.y) * (b.z - p.z) - (a.z - p.z) * (b.y - p.y) * (c.x - p.x) -
                     (b.z - p.z) * (c.y - p.y) * (a.x - p.x) - (c.z - p.z) * (a.y - p.y) * (b.x - p.x);
  const double den = (a.x - o.x) * (b.y - o.y) * (c.z - o.z) + (b.x - o.x) * (c.y - o.y) * (a.z - o.z) +
                     (c.x - o.x) * (a.y - o.y) * (b.z - o.z) - (a.z - o.z) * (b.y - o.y) * (c.x - o.x) -
                     (b.z - o.z) * (c.y - o.y) * (a.x - o.x) - (c.z - o.z) * (a.y - o.y) * (b.x - o.x);
  return num / den;
}

__device__ inline void shape10(const double l[3], double N[10]) {
  const double r = l[0], s = l[1], t = l[2], u = 1.0 - r - s - t;
  N[0] = r * (2 * r - 1);
  N[1] = s * (2 * s - 1);
  N[2] = t * (2 * t - 1);
  N[3] = u * (2 * u - 1);
  N[4] = 4 * r * s;
  N[5] = 4 * s * t;
  N[6] = 4 * t * u;
  N[7] = 4 * r * u;
  N[8] = 4 * r * t;
  N[9] = 4 * s * u;
}

// dN/d(r, s, t) of the ten shape functions (local_coords_curved_3d_sph.m)
__device__ inline void dshape10(const double l[3], double d[3][10]) {
  const double r = l[0], s = l[1], t = l[2], u = 1.0 - r - s - t;
  const double w = -3 + 4 * (1 - u);
  const double dr[10] = {4 * r - 1, 0, 0, w, 4 * s, 0, -4 * t, 4 * (u - r), 4 * t, -4 * s};
  const double ds[10] = {0, 4 * s - 1, 0, w, 4 * r, 4 * t, -4 * t, -4 * r, 0, 4 * (u - s)};
  const double dt[10] = {0, 0, 4 * t - 1, w, 0, 4 * s, 4 * (u - t), -4 * r, 4 * r, -4 * s};
  for (int k = 0; k < 10; ++k) {
    d[0][k] = dr[k];
    d[1][k] = ds[k];
    d[2][k] = dt[k];
  }
}

// local coordinates (first three) of p (original frame) in element e
__device__ void local_coords(const SlmArgs &a, int64_t e, V3d p, double l[3]) {
  const int cls = a.cls[e];
  const int f = frame_of(cls);
  const double *F = f == 0 ? a.S : (f == 1 ? a.Sz : a.Sx);
  const int32_t *n = a.el2nod + 10 * e;
  V3d v[4];
  for (int i = 0; i < 4; ++i) v[i] = ld(F, n[i]);
  V3d q = in_frame(p, f);
  // an element of the original frame does not cross phi = 2 pi; a point
  // seen from the far side of that meridian is taken there, so that its
  // coordinates point the search the right way (for a point inside the
  // element nothing changes)
  if (f == 0) {
    if (q.y - v[0].y > M_PI) q.y -= 2.0 * M_PI;
    else if (v[0].y - q.y > M_PI) q.y += 2.0 * M_PI;
  }
  l[0] = bary(v, 0, 1, 2, 3, q);
  l[1] = bary(v, 1, 0, 2, 3, q);
  l[2] = bary(v, 2, 0, 1, 3, q);
  if (cls != 3) return;
  V3d g[10];
  for (int i = 0; i < 10; ++i) g[i] = ld(F, n[i]);
  for (int it = 0; it < 6; ++it) {
    double N[10];
    shape10(l, N);
    double x0 = 0, y0 = 0, z0 = 0;
    for (int k = 0; k < 10; ++k) {
      x0 += g[k].x * N[k];
      y0 += g[k].y * N[k];
      z0 += g[k].z * N[k];
    }
    const double d0 = q.x - x0, d1 = q.y - y0, d2 = q.z - z0;
    if (sqrt(d0 * d0 + d1 * d1 + d2 * d2) < 1e-8) break;
    double dN[3][10];
    dshape10(l, dN);
    double J[3][3];  // J[a][c] = d coordinate a / d local c
    for (int c = 0; c < 3; ++c) {
      double sx = 0, sy = 0, sz = 0;
      for (int k = 0; k < 10; ++k) {
        sx += g[k].x * dN[c][k];
        sy += g[k].y * dN[c][k];
        sz += g[k].z * dN[c][k];
      }
      J[0][c] = sx;
      J[1][c] = sy;
      J[2][c] = sz;
    }
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    const double id = 1.0 / det;
    const double I00 = id * (J[1][1] * J[2][2] - J[1][2] * J[2][1]), I01 = id * (J[0][2] * J[2][1] - J[0][1] * J[2][2]),
                 I02 = id * (J[0][1] * J[1][2] - J[0][2] * J[1][1]), I10 = id * (J[1][2] * J[2][0] - J[1][0] * J[2][2]),
                 I11 = id * (J[0][0] * J[2][2] - J[0][2] * J[2][0]), I12 = id * (J[0][2] * J[1][0] - J[0][0] * J[1][2]),
                 I20 = id * (J[1][0] * J[2][1] - J[1][1] * J[2][0]), I21 = id * (J[0][1] * J[2][0] - J[0][0] * J[2][1]),
                 I22 = id * (J[0][0] * J[1][1] - J[0][1] * J[1][0]);
    l[0] += I00 * d0 + I01 * d1 + I02 * d2;
    l[1] += I10 * d0 + I11 * d1 + I12 * d2;
    l[2] += I20 * d0 + I21 * d1 + I22 * d2;
  }
}

__device__ inline double min4(const double l[3]) {
  const double u = 1.0 - l[0] - l[1] - l[2];
  return fmin(fmin(l[0], l[1]), fmin(l[2], u));
}

// walk to the element holding p; returns it and its (clipped) coordinates
__device__ int64_t locate(const SlmArgs &a, V3d p, int64_t e, double lc[3]) {
  int64_t prev = -1, best = e;
  double bl[3] = {0.25, 0.25, 0.25}, bm = -1e300;
  for (int step = 0; step < SLM_MAXWALK; ++step) {
    double l[3];
    local_coords(a, e, p, l);
    const double m = min4(l);
    if (m > bm) {
      bm = m;
      best = e;
      bl[0] = l[0];
      bl[1] = l[1];
      bl[2] = l[2];
    }
    if (m >= -1e-12) break;
    const double u = 1.0 - l[0] - l[1] - l[2];
    int f = 0;
    double mn = l[0];
    if (l[1] < mn) { mn = l[1]; f = 1; }
    if (l[2] < mn) { mn = l[2]; f = 2; }
    if (u < mn) f = 3;
    const int64_t nb = a.nbr[4 * e + f];
    if (nb < 0 || nb == prev) break;
    if (step == SLM_MAXWALK - 1) atomicAdd(&a.cnt[1], 1ull);
    prev = e;
    e = nb;
  }
  // adjust_local_coords
  double s = 0;
  for (int i = 0; i < 3; ++i) {
    lc[i] = fmin(fmax(bl[i], 0.0), 1.0);
    s += lc[i];
  }
  if (s > 1)
    for (int i = 0; i < 3; ++i) lc[i] /= s;
  return best;
}

__device__ inline V3d shift_inside(const SlmArgs &a, V3d p) {
  const double tol = 1e-12 * (a.r_surf - a.r_cmb);
  if (p.z <= a.r_cmb + tol || p.z >= a.r_surf - tol) atomicAdd(&a.cnt[0], 1ull);
  if (p.z <= a.r_cmb + tol) p.z = a.r_cmb + tol;
  if (p.z >= a.r_surf - tol) p.z = a.r_surf - tol;
  return p;
}

// move X over the arc l_perp / r against the unit direction w and to the
// radius |r - l_par| (predictor / corrector_step_with_projections)
__device__ inline V3d step_back(V3d X, double r, V3d w, double l_par, double l_perp, V3d &unit) {
  const double lp = r * tan(l_perp / r);
  const V3d q = {X.x - w.x * lp, X.y - w.y * lp, X.z - w.z * lp};
  const double nq = sqrt(q.x * q.x + q.y * q.y + q.z * q.z);
  unit = {q.x / nq, q.y / nq, q.z / nq};
  const double rr = fabs(r - l_par);
  return c2s(V3d{unit.x * rr, unit.y * rr, unit.z * rr});
}

// quadratic interpolation of the field in element e, with the optional clip
// to the element's ten nodal values (interp3d_tet.m:51-70)
__device__ inline double interp_T(const SlmArgs &a, int64_t e, const double lc[3]) {
  double N[10];
  shape10(lc, N);
  double Tv = 0, tmin = 1e300, tmax = -1e300;
  for (int k = 0; k < 10; ++k) {
    const double tk = a.T[a.el2nod[10 * e + k]];
    Tv += N[k] * tk;
    tmin = fmin(tmin, tk);
    tmax = fmax(tmax, tk);
  }
  if (a.monotonic) Tv = fmin(fmax(Tv, tmin), tmax);
  return Tv;
}

// 128 threads per workgroup (the launch below): up to 220 VGPRs, so the
// curved-element Newton step keeps its ten node coordinates in registers
// (with the default bound of 1024 threads the compiler capped the kernel at
// 128 VGPRs and spilled 308 bytes per lane to scratch)
__global__ __launch_bounds__(128) void k_slm_pc2(SlmArgs a) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.nnod) return;
  const V3d X = ld(a.X, i);
  const double r = a.S[3 * i + 2];
  const V3d ru = {X.x / r, X.y / r, X.z / r};
  const double n2 = ru.x * ru.x + ru.y * ru.y + ru.z * ru.z;
  const V3d U = ld(a.U, i);
  // predictor
  double dp = (U.x * ru.x + U.y * ru.y + U.z * ru.z) / n2;
  V3d up = {dp * ru.x, dp * ru.y, dp * ru.z};
  V3d uq = {U.x - up.x, U.y - up.y, U.z - up.z};
  const double nperp = sqrt(uq.x * uq.x + uq.y * uq.y + uq.z * uq.z);
  const V3d w = nperp > 0 ? V3d{uq.x / nperp, uq.y / nperp, uq.z / nperp} : V3d{0, 0, 0};
  V3d rbu;
  V3d P = step_back(X, r, w, sqrt(up.x * up.x + up.y * up.y + up.z * up.z) * 0.5 * a.dt, nperp * 0.5 * a.dt, rbu);
  P = shift_inside(a, P);
  double lc[3], N[10];
  int64_t e = locate(a, P, a.start[i], lc);
  shape10(lc, N);
  V3d Ub = {0, 0, 0};
  for (int k = 0; k < 10; ++k) {
    const V3d uk = ld(a.U, a.el2nod[10 * e + k]);
    Ub.x += N[k] * uk.x;
    Ub.y += N[k] * uk.y;
    Ub.z += N[k] * uk.z;
  }
  // corrector
  const double m2 = rbu.x * rbu.x + rbu.y * rbu.y + rbu.z * rbu.z;
  dp = (Ub.x * rbu.x + Ub.y * rbu.y + Ub.z * rbu.z) / m2;
  up = {dp * rbu.x, dp * rbu.y, dp * rbu.z};
  uq = {Ub.x - up.x, Ub.y - up.y, Ub.z - up.z};
  V3d unit2;
  V3d Q = step_back(X, r, w, sqrt(up.x * up.x + up.y * up.y + up.z * up.z) * a.dt,
                    sqrt(uq.x * uq.x + uq.y * uq.y + uq.z * uq.z) * a.dt, unit2);
  Q = shift_inside(a, Q);
  e = locate(a, Q, e, lc);
  a.Tout[i] = interp_T(a, e, lc);
}

// EU1 (backtrack_EU1, advect3d_slm_p_sph.m:145-161): one explicit step in
// the node's spherical coordinates, theta - dt U1 / r, phi - dt U2 / r,
// r - dt U3.  The reference hands the three velocity arrays over as
// (v_theta, v_phi, v_r) unchanged, so the caller's first, second and third
// components are taken as those; theta or phi that leave [0, pi] / [0, 2 pi]
// are kept as they are (the point is the one their Cartesian form names),
// only the radius is moved into the shell.
__global__ __launch_bounds__(128) void k_slm_eu1(SlmArgs a) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= a.nnod) return;
  const V3d S = ld(a.S, i);
  const V3d U = ld(a.U, i);
  V3d P = {S.x - a.dt * U.x / S.z, S.y - a.dt * U.y / S.z, S.z - a.dt * U.z};
  P = shift_inside(a, P);
  double lc[3];
  const int64_t e = locate(a, P, a.start[i], lc);
  a.Tout[i] = interp_T(a, e, lc);
}

void setup(m3_ctx *c) {
  auto &A = c->slm;
  const LevelDev &f = c->L[0];
  const int64_t ne = f.nel, nn = f.nnod;
  // face neighbours: the face opposite local vertex k is the other three vertices
  std::vector<int32_t> nbr(4 * ne, -1), start(nn, -1);
  std::unordered_map<unsigned long long, int64_t> open;
  open.reserve(2 * ne);
  auto key = [](int32_t a, int32_t b, int32_t d) {
    int32_t v[3] = {a, b, d};
    std::sort(v, v + 3);
    return ((unsigned long long)v[0] << 42) | ((unsigned long long)v[1] << 21) | (unsigned long long)v[2];
  };
  M3_REQUIRE(f.nV < (1 << 21), M3_E_MESH, "too many vertices for the face table (limit 2^21)");
  for (int64_t e = 0; e < ne; ++e) {
    const int32_t *n = &f.h_el2nod[10 * e];
    for (int k = 0; k < 10; ++k)
      if (start[n[k]] < 0) start[n[k]] = (int32_t)e;
    for (int k = 0; k < 4; ++k) {
      int32_t o[3], m = 0;
      for (int j = 0; j < 4; ++j)
        if (j != k) o[m++] = n[j];
      const unsigned long long kk = key(o[0], o[1], o[2]);
      auto it = open.find(kk);
      if (it == open.end()) {
        open.emplace(kk, 4 * e + k);
      } else {
        const int64_t g = it->second;
        nbr[4 * e + k] = (int32_t)(g / 4);
        nbr[g] = (int32_t)e;
        open.erase(it);
      }
    }
  }
  for (int64_t i = 0; i < nn; ++i) M3_REQUIRE(start[i] >= 0, M3_E_MESH, "node without an element");
  // node coordinates in the two rotated frames (from GCOORD, as the reference
  // recomputes them), the shell radii from GCOORD_SPH
  std::vector<double> Sz(3 * nn), Sx(3 * nn);
  double rmin = 1e300, rmax = -1e300;
  for (int64_t i = 0; i < nn; ++i) {
    const double *x = &c->h_coord[3 * i];
    auto sph = [](double px, double py, double pz, double *o) {
      o[2] = std::sqrt(px * px + py * py + pz * pz);
      o[0] = std::atan2(std::sqrt(px * px + py * py), pz);
      double ph = std::atan2(py, px);
      if (ph < 0) ph += 2 * M_PI;
      o[1] = ph;
    };
    sph(-x[0], -x[1], x[2], &Sz[3 * i]);
    sph(x[0], -x[2], x[1], &Sx[3 * i]);
    rmin = std::min(rmin, c->h_sph[3 * i + 2]);
    rmax = std::max(rmax, c->h_sph[3 * i + 2]);
  }
  A.r_cmb = rmin;
  A.r_surf = rmax;
  A.nbr.upload(nbr);
  A.start.upload(start);
  A.Sz.upload(Sz);
  A.Sx.upload(Sx);
  A.U.alloc(3 * nn);
  A.T.alloc(nn);
  A.Tout.alloc(nn);
  A.cnt.alloc(2);
  A.ready = true;
}

}  // namespace

namespace m3 {

void slm_advect(m3_ctx *c, const double *Ux, const double *Uy, const double *Uz, double *T, double dt,
                const m3_slm_opts *opts, m3_slm_info *info) {
  M3_REQUIRE(c->have_mesh, M3_E_STATE, "m3_advect3d_slm_p_sph before m3_set_mesh");
  M3_REQUIRE(Ux && Uy && Uz && T, M3_E_ARG, "null argument");
  M3_REQUIRE(std::isfinite(dt) && dt >= 0, M3_E_ARG, "dt must be finite and non-negative");
  const int method_BT = opts ? opts->method_BT : M3_SLM_PC2;
  const int interp = opts ? opts->method_interp : M3_SLM_QUADRATIC;
  M3_REQUIRE(method_BT != M3_SLM_RK4, M3_E_ARG, "RK4 is not working for spherical coordinates (need to be coded)");
  M3_REQUIRE(method_BT == M3_SLM_PC2 || method_BT == M3_SLM_EU1, M3_E_ARG, "method_BT must be 'EU1' or 'PC2'");
  M3_REQUIRE(interp == M3_SLM_QUADRATIC, M3_E_ARG,
             "fields on P2 nodes need method_interp = 'quadratic' (the reference stops on 'linear' and 'cubic' there)");
  const int64_t nn = c->L[0].nnod;
  for (int64_t i = 0; i < nn; ++i)
    M3_REQUIRE(std::isfinite(Ux[i]) && std::isfinite(Uy[i]) && std::isfinite(Uz[i]) && std::isfinite(T[i]),
               M3_E_NUMERIC, "velocity or field contains NaN or Inf");
  if (!c->slm.ready) setup(c);
  auto &A = c->slm;
  hipStream_t s = c->stream;
  std::vector<double> U(3 * nn);
  for (int64_t i = 0; i < nn; ++i) {
    U[3 * i] = Ux[i];
    U[3 * i + 1] = Uy[i];
    U[3 * i + 2] = Uz[i];
  }
  HIPCHECK(hipMemcpyAsync(A.U.p, U.data(), sizeof(double) * 3 * nn, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(A.T.p, T, sizeof(double) * nn, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemsetAsync(A.cnt.p, 0, 2 * sizeof(unsigned long long), s));
  SlmArgs a{};
  a.nnod = nn;
  a.el2nod = c->L[0].el2nod.p;
  a.cls = c->cls.p;
  a.X = c->X.p;
  a.S = c->S.p;
  a.Sz = A.Sz.p;
  a.Sx = A.Sx.p;
  a.nbr = A.nbr.p;
  a.start = A.start.p;
  a.U = A.U.p;
  a.T = A.T.p;
  a.Tout = A.Tout.p;
  a.dt = dt;
  a.r_cmb = A.r_cmb;
  a.r_surf = A.r_surf;
  a.monotonic = opts ? (opts->monotonic != 0) : 1;
  a.cnt = A.cnt.p;
  hipLaunchKernelGGL(method_BT == M3_SLM_EU1 ? k_slm_eu1 : k_slm_pc2, dim3((unsigned)((nn + 127) / 128)), dim3(128),
                     0, s, a);
  HIPCHECK(hipGetLastError());
  unsigned long long cnt[2] = {0, 0};
  HIPCHECK(hipMemcpyAsync(T, A.Tout.p, sizeof(double) * nn, hipMemcpyDeviceToHost, s));
  HIPCHECK(hipMemcpyAsync(cnt, A.cnt.p, sizeof cnt, hipMemcpyDeviceToHost, s));
  HIPCHECK(hipStreamSynchronize(s));
  if (info) {
    info->nshift = (int64_t)cnt[0];
    info->nunresolved = (int64_t)cnt[1];
  }
}

}  // namespace m3
