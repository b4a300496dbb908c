/*
 * m3stokes.h -- C ABI of the MI355X-native Stokes hot path of M3TET_SPH.
 *
 * The entry points replace, one for one, the MATLAB functions of the
 * reference's Stokes path (paths relative to the reference repository):
 *
 *   m3_set_mesh            <- MESH fields read by the path
 *                             (mfiles_SPH/init_mesh_curved_p.m:182-246)
 *   m3_set_bc              <- UBC.ifix / UBC.vfix (SETUP_TEST/bc_sph.m:526-530)
 *   m3_set_els_ref         <- MESH.els_ref / NUMSCALE.Dens0_T_bary (refined-region buoyancy)
 *   m3_assemble            <- assembly_stokes_sph_3d_double_jacobian
 *                             (mfiles_SPH/assembly_stokes_sph_3d_double_jacobian.m:1-2)
 *                             followed by the rotation / BC elimination of
 *                             mfiles_M3TET/flow3d_patera_mg_sph_p.m:225-298
 *   m3_element_matrices    <- the element-packed ASSEMBLY.KKv/GGv/MMv/Fb arrays
 *                             (assembly_stokes_sph_3d_double_jacobian.m:365-393)
 *   m3_restrict_stiffmat   <- restrict_stiffmat (mfiles_M3TET/restrict_stiffmat.m:1)
 *   m3_cholesky_factorization / m3_cholesky_solve
 *                          <- cholesky_factorization.m:1 / cholesky_solve.m:1
 *   m3_mgpcg               <- mgpcg_solver_p (mfiles_M3TET/mgpcg_solver_p.m:1-2)
 *   m3_patera              <- flow3d_patera_mg_sph_p (flow3d_patera_mg_sph_p.m:1),
 *                             pressure iteration and final velocity solve
 *   m3_flow3d_patera_sph   <- flow3d_patera_sph (mfiles_M3TET/flow3d_patera_sph.m:1-9),
 *                             the whole solve: assembly, RAP, factorisation, Patera
 *
 * Conventions: index arrays that mirror MATLAB arrays are 1-based and
 * column-major exactly as MATLAB stores them (EL2NOD{l} is 10 x nel, so in C
 * it is nel rows of 10).  Velocity dofs are node-interleaved, dof = 3*(node-1)+c
 * (nod2dof.m:11); after rotation the components are (theta, phi, r).
 * All pointers are host pointers owned by the caller and read only during the
 * call; device state lives in the context until m3_destroy.  Every call is
 * synchronous and returns 0 on success or a nonzero M3_E* code, with the
 * message available from m3_last_error (the reference's error(...) sites).
 * One host thread per context.
 */
#ifndef M3STOKES_H
#define M3STOKES_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define M3_MAX_LEVELS 8

enum {
  M3_OK = 0,
  M3_E_ARG = 1,        /* invalid argument / inconsistent sizes */
  M3_E_HIP = 2,        /* HIP runtime failure */
  M3_E_MESH = 3,       /* mesh invariant violated (nesting, classes, ...) */
  M3_E_NUMERIC = 4,    /* negative Jacobian, non-positive viscosity, NaN, ... */
  M3_E_STATE = 5,      /* call order (e.g. solve before assemble) */
  M3_E_NOTCONV = 6     /* iteration limit reached (result still returned) */
};

typedef struct m3_ctx m3_ctx;

/* MESH fields used by the hot path.  Level 0 is the finest mesh (MATLAB's
 * MESH.EL2NOD{1}); coarse-level nodes are numbered first in every finer
 * level (tetmesh_p1_to_p2_sph.m:619-629). */
typedef struct {
  int32_t nmg;                               /* MESH.nmg, 2..M3_MAX_LEVELS */
  int64_t nel[M3_MAX_LEVELS];                /* elements per level */
  int64_t nnod[M3_MAX_LEVELS];               /* P2 nodes per level */
  int64_t nVnod[M3_MAX_LEVELS];              /* vertices (pressure dofs) per level */
  const uint32_t *EL2NOD[M3_MAX_LEVELS];     /* MESH.EL2NOD{l}: 10 x nel, 1-based */
  const double *GCOORD;                      /* MESH.GCOORD: 3 x nnod (finest) */
  const double *GCOORD_SPH;                  /* MESH.GCOORD_SPH: 3 x nnod */
  const int32_t *els_class[4];               /* MESH.els_out_cone_no_cross_2pi,
                                                els_out_cone_cross_2pi,
                                                els_in_cone_no_iso,
                                                els_in_cone_iso (1-based) */
  int64_t nels_class[4];
  const uint32_t *EL2NOD_cubic;              /* MESH.EL2NOD_cubic: 20 x n_iso, 1-based
                                                into [GCOORD GCOORD_cubic] */
  const double *GCOORD_cubic;                /* MESH.GCOORD_cubic: 3 x ncubic */
  int64_t ncubic;
  /* MESH.Ic2f{l} (fine level l <- coarse level l+1) at node level: the three
   * velocity components share the weights (intermesh_transfer_matrix.m:50-55).
   * CSR over fine nodes, 0-based coarse node columns. */
  const int64_t *Ic2f_ptr[M3_MAX_LEVELS];
  const int32_t *Ic2f_col[M3_MAX_LEVELS];
  const double *Ic2f_val[M3_MAX_LEVELS];
} m3_mesh_desc;

/* PHYSICS / NUMSCALE / OPTS fields read by the assembly. */
typedef struct {
  double g;            /* PHYSICS.g */
  double Bscale;       /* NUMSCALE.Bscale */
  double Dens0;        /* NUMSCALE.Dens0 */
  double minVisc;      /* PHYSICS.minVisc (used if has_minVisc) */
  double maxVisc;      /* PHYSICS.maxVisc (used if has_maxVisc) */
  int32_t has_minVisc;
  int32_t has_maxVisc;
  int32_t nip;         /* OPTS.nip, must be 14 */
  int32_t type_Dmat;   /* 0: '23rd' (C1=4/3, C2=-2/3), 1: '221' (C1=2, C2=0) */
} m3_phys;

/* Precision of the multigrid V-cycle (the outer CG, dot products, Patera
 * update and coarse Cholesky are FP64 in every mode).  M3_PREC_MIXED: FP32
 * vectors and accumulation, BF16 matrix values on the finest and middle
 * levels (v8 of each 3x3 block in FP32), coarse triangular solves on FP32
 * copies of the factor's inverse tiles. */
enum { M3_PREC_FP64 = 0, M3_PREC_MIXED = 1 };

/* Solver parameters: flow3d_patera_mg_sph_p.m:70-98, mgpcg_solver_p.m:674-682. */
typedef struct {
  double rtol_Pat;     /* 1e-4 */
  double rtol_U;       /* 5e-3 */
  int32_t itmax_U;     /* 20 */
  int32_t itmin_Pat;   /* 3 */
  int32_t itmax_Pat;   /* 120 */
  int32_t pc_Pat;      /* 3 (only 3 is supported) */
  double wght_MM;      /* 1 (one Jacobi sweep on MM) */
  int32_t precision;   /* M3_PREC_FP64 or M3_PREC_MIXED */
  int32_t warm_U;      /* 0: U starts from the BC values as in the reference
                          (flow3d_patera_mg_sph_p.m:230); 1: use U as given */
  double rtol_U_final; /* 0: reference behaviour.  > 0: the final velocity solve
                          (flow3d_patera_mg_sph_p.m:630-632) also stops only once
                          |r_U| <= rtol_U_final |f_U| (fixed-denominator residual),
                          with up to itmax_U_final iterations; if the pressure
                          residual -GG' U of that velocity misses tol_Pat, the
                          velocity solve is tightened 10x once and, if still
                          needed, the pressure iteration continues from the
                          true residual (up to 3 times) */
  int32_t itmax_U_final;
  double tol_Pat_abs;  /* 0: reference behaviour (tol_Pat = rtol_Pat * initial
                          pressure residual, flow3d_patera_mg_sph_p.m:436-437).
                          > 0: absolute RMS pressure-residual tolerance, so that
                          runs from different starting points stop at the same
                          residual; the second velocity solve, whose tolerance
                          the reference sets to rtol_U (rtol_restart / rtol_Pat)
                          tol_Pat (:74,437-443), keeps that relation to the fixed
                          tol_Pat */
  double rtol_U_first; /* 0: reference behaviour (the initial velocity solve stops
                          at rtol_U * rtol_restart relative to its own starting
                          residual, flow3d_patera_mg_sph_p.m:413-423).  > 0: it
                          stops once |r_U| <= rtol_U_first |f_U| (RMS over the
                          free dofs), so a better starting point needs fewer
                          iterations instead of the same relative reduction */
} m3_patera_opts;

typedef struct {
  int32_t nitP, nitU, nitZ;
  double norm_rP;            /* final pressure residual (RMS) */
  double norm_rP0;           /* initial pressure residual (RMS) */
  /* s.  Host times: the solve waits for the device once per CG iteration, so
   * pressure kernels that are queued ahead of a velocity solve end in its first
   * wait and count as t_velocity; t_pressure is the host's time between the
   * velocity solves, the wait for a pressure step's norm included. */
  double t_assemble, t_restrict, t_factor, t_pressure, t_velocity, t_total;
} m3_info;

int m3_create(m3_ctx **ctx, int hip_device);
void m3_destroy(m3_ctx *ctx);
/* Message of the last failed call on ctx; with ctx = NULL, of the last failed
 * context-free call (m3_unique_bars_noalloc) on the calling thread. */
const char *m3_last_error(const m3_ctx *ctx);

int m3_set_mesh(m3_ctx *ctx, const m3_mesh_desc *mesh);
/* Which multigrid levels the m3_set_mesh calls from now on sweep in windows: the
 * fewest rows of such a level, the most vector entries that a window of more than
 * 64 rows / one of 64 rows gathers (at most 6300; larger windows are split), and
 * the most that all windows of a level gather per row; a level that meets one of
 * the last two has no windows.  0: the library's own choice.  It moves work, not
 * results.  No reference counterpart. */
int m3_sweep_windows(m3_ctx *ctx, int64_t rows, int32_t split, int32_t limit, int32_t per_row);
/* ifix: 1-based rotated-frame dofs, vfix: values (UBC.ifix / UBC.vfix). */
int m3_set_bc(m3_ctx *ctx, const int64_t *ifix, const double *vfix, int64_t nfix);

/* Embedded high-resolution region (MESH.els_ref, init_mesh_curved_p.m:172-177,
 * 302-330, and NUMSCALE.Dens0_T_bary, SETUP_TEST/init_fields_sph.m:312-319):
 * els_ref are 1-based finest-level elements, strictly increasing;
 * Dens0_T_bary[j] is the reference density of element els_ref[j].  With a
 * region set, the buoyancy of every class kernel is zero outside it and
 * g Bscale (Dens - Dens0_T_bary) inside it
 * (assembly_stokes_els_out_cone_no_cross_2pi_opt.m:188-195, ..._cross_2pi_opt.m:
 * 194-201, ..._in_cone_no_iso_opt.m:199-206, ..._iso_20_nodes_opt.m:205-212);
 * nels_ref = 0 clears it (g Bscale (Dens - Dens0) everywhere, the default). */
int m3_set_els_ref(m3_ctx *ctx, const int32_t *els_ref, int64_t nels_ref, const double *Dens0_T_bary);

/* Assembly on the device: K1 = RR' K RR with the BC dofs eliminated, GG = RR' GG,
 * Fb = RR' Fb, MM, bc_rhs.  Visc/Dens are nodal (nnod).  Visc = Dens = NULL
 * (here and in m3_flow3d_patera_sph) uses the fields that m3_rock_prop left
 * on the device. */
int m3_assemble(m3_ctx *ctx, const double *Visc, const double *Dens, const m3_phys *phys);

/* Material law on the device (mfiles_M3TET/rock_prop.m:31-118):
 *   Dens = Dens0 (1 - alpha (T - T_ref)), clipped to [minDens, maxDens];
 *   f_T  = exp(Ea/(R T0_K) (T0_K/T_K - 1)) clipped to [1e-8, 1e8] (Ea > 0),
 *          T_K = T + 273, T0_K = T_ref + 273, R = 8.314472;
 *   f_P  = f_T exp(|g Dens0 L0 depth| Va / (R T0_K)) (Va > 0),
 *          depth = max node radius - radius;
 *   f_LM = f_T a_UM2LM (a_UM2LM > 0);
 *   Visc = Visc0 min(f_P, f_LM), clipped to [minVisc, maxVisc].
 * T is nodal (nnod).  The fields stay on the device for the next assembly
 * (pass Visc = Dens = NULL there); Visc/Dens outputs here may be NULL. */
typedef struct {
  double Visc0, Dens0, T_ref, alpha, Ea, Va, g, L0, a_UM2LM;
  double minVisc, maxVisc, minDens, maxDens;
  int32_t has_minVisc, has_maxVisc, has_minDens, has_maxDens;
} m3_rock_params;
int m3_rock_prop(m3_ctx *ctx, const double *T, const m3_rock_params *rp, double *Visc, double *Dens);

/* Advective time step (mfiles_M3TET/calculate_dt.m:40-56):
 *   dt = min(dtmax, dt_adv_limit * min(Lx/max|Ux|, Ly/max|Uy|, Lz/max|Uz|))
 * with L the mesh extents (init_mesh_curved_p.m:270) and U (3*nnod, rotated
 * frame as returned by m3_flow3d_patera_sph) turned to Cartesian on the
 * device; dt = dtmax for a zero velocity. */
int m3_calculate_dt(m3_ctx *ctx, const double *U, double dt_adv_limit, double dtmax, double *dt);

/* Compressed sparse column matrix in the layout of a MATLAB sparse mxArray
 * (0-based row indices ir and column pointers jc, as mxGetIr / mxGetJc hold
 * them; the library writes int64, which a MEX gateway copies into mwIndex). */
typedef struct {
  int64_t nrow, ncol, nnz;   /* filled by the library */
  int64_t *colptr;           /* ncol + 1, caller-allocated; NULL to query the sizes */
  int64_t *rowidx;           /* nnz, ascending within each column */
  double *val;               /* nnz */
} m3_csc;

/* [KK,Fb,GG,MM,Fpdil] = assembly_stokes_sph_3d_double_jacobian(VAR,MESH,PHYSICS,
 * NUMSCALE,OPTS) (mfiles_SPH/assembly_stokes_sph_3d_double_jacobian.m:1-2,
 * global assembly :398-490) on the finest mesh, in the reference's shapes:
 * KK (3 nnod x 3 nnod) lower triangle, GG (3 nnod x nVnod), MM (nVnod x
 * nVnod) lower triangle, Fb (3 nnod), all in the Cartesian frame before the
 * rotation and BC elimination of flow3d_patera_mg_sph_p.m:225-298, and Fpdil =
 * 0 (no dilatation on this path).  The element matrices are computed on the
 * GPU, the sums per entry on the host.  Sparsity is the element pattern (no
 * entry is dropped for being zero).  Any of KK, Fb, GG, MM, Fpdil may be
 * NULL.  A call in which a given matrix has colptr = NULL only fills the
 * sizes (nrow, ncol, nnz) and computes nothing: call once to size the
 * buffers, then again to fill them. */
int m3_assembly_stokes_sph_3d_double_jacobian(m3_ctx *ctx, const double *Visc, const double *Dens,
                                              const m3_phys *phys, m3_csc *KK, double *Fb, m3_csc *GG,
                                              m3_csc *MM, double *Fpdil);

/* Element-packed matrices in the reference layout and original Cartesian
 * frame: KKv 465 x nel, GGv 120 x nel, MMv 10 x nel, Fbv 30 x nel. */
int m3_element_matrices(m3_ctx *ctx, const double *Visc, const double *Dens,
                        const m3_phys *phys, double *KKv, double *GGv, double *MMv,
                        double *Fbv);

int m3_restrict_stiffmat(m3_ctx *ctx);
int m3_cholesky_factorization(m3_ctx *ctx);
/* Coarsest-level solve; rhs/x have 3*nnod[nmg-1] entries (fixed dofs ignored / 0). */
int m3_cholesky_solve(m3_ctx *ctx, const double *rhs, double *x);

/* MGPCG on the assembled operator: b, x have 3*nnod entries (rotated frame;
 * entries at fixed dofs are ignored / returned as 0).  rrms_vec may be NULL,
 * else it receives itmax+1 values. */
int m3_mgpcg(m3_ctx *ctx, const double *b, double *x, double tol, int32_t is_abs_tol,
             int32_t itmax, int32_t precision, int32_t *it, double *rrms_vec);

/* Patera iteration on the assembled operators.  U: 3*nnod (rotated frame,
 * output includes the BC values); P: nVnod (warm start in, solution out). */
int m3_patera(m3_ctx *ctx, double *U, double *P, const m3_patera_opts *opts, m3_info *info);

/* Whole solve: assemble, restrict, factorise, Patera. */
int m3_flow3d_patera_sph(m3_ctx *ctx, const double *Visc, const double *Dens,
                         const m3_phys *phys, double *U, double *P,
                         const m3_patera_opts *opts, m3_info *info);

/* The same solve with the starting point already in device memory on the
 * context's GPU (for instance the warm start that m3_gnn_warm_start_hist left
 * there, m3_gnn_start_device): P0_dev (nVnod) and, with opts->warm_U = 1,
 * U0_dev (3*nnod, rotated frame) are copied device to device, so the start
 * makes no round trip through host memory.  U and P are outputs only;
 * U = P = NULL leaves the solution in device memory alone (m3_solution_device,
 * m3_get_solution), and with Visc = Dens = NULL (fields of m3_set_fields or
 * m3_rock_prop) the whole solve moves no data between host and device.  No
 * reference counterpart: flow3d_patera_sph.m returns VAR.U / VAR.P to MATLAB,
 * which m3_get_solution provides. */
int m3_flow3d_patera_sph_dstart(m3_ctx *ctx, const double *Visc, const double *Dens,
                                const m3_phys *phys, const double *U0_dev, const double *P0_dev,
                                double *U, double *P, const m3_patera_opts *opts, m3_info *info);

/* Solution of the last Stokes solve of this context (any of m3_patera,
 * m3_flow3d_patera_sph, m3_flow3d_patera_sph_dstart), which stays in device
 * memory until the next solve or m3_set_mesh: its device addresses (U 3*nnod
 * with the BC values, rotated frame; P nVnod), for callers that keep the
 * time loop's state on the GPU, and a host copy (either output may be NULL).
 * No reference counterpart (device residency). */
int m3_solution_device(m3_ctx *ctx, const double **U_dev, const double **P_dev);
int m3_get_solution(m3_ctx *ctx, double *U, double *P);

/* Nodal Visc and Dens (nnod) copied to the device fields that the assembly
 * reads when it is called with Visc = Dens = NULL (as m3_rock_prop leaves
 * them).  No reference counterpart (device residency). */
int m3_set_fields(m3_ctx *ctx, const double *Visc, const double *Dens);

/* Operator application for parity checks.  which: 0 = K on level `level`
 * (level 0 = K1), 1 = GG (nVnod -> 3*nnod), 2 = GG' (3*nnod -> nVnod),
 * 3 = MM (full symmetric), 4 = prolongation level+1 -> level (masked),
 * 5 = restriction level -> level+1 (masked). */
int m3_apply(m3_ctx *ctx, int32_t which, int32_t level, const double *x, double *y);

/* Device vectors for parity checks.  which: 0 = Fb (rotated), 1 = bc_rhs,
 * 2 = diag of K on `level`, 3 = free-dof mask on `level` (1/0),
 * 4 = lumped MM. */
int m3_get_vector(m3_ctx *ctx, int32_t which, int32_t level, double *out);

/* Sizes: n[0]=levels, n[1..] per-level block nonzeros of K, then coarse factor
 * statistics (free dofs, tiles, stored tiles, levels, solve levels), then per
 * level the stored block slots of K, the windows of its sweeps (0: swept
 * without) and the most vector entries that one of them gathers. */
int m3_stats(m3_ctx *ctx, int64_t *out, int32_t nout);

/* Residuals of (U, P) for the assembled problem, RMS norms (normdf.m:22):
 * out[0] = |r_U| with r_U = Fb + GG P - bc_rhs - K1 U on the free dofs,
 * out[1] = |f_U| with f_U = Fb + GG P - bc_rhs on the free dofs,
 * out[2] = |r_P| with r_P = -GG' U (mean removed).  No reference counterpart:
 * it evaluates the fixed-denominator residual used to stop and compare solves. */
int m3_residual(m3_ctx *ctx, const double *U, const double *P, double *out);

/* Kernel timing with HIP events that each timed launch records at its own
 * start and end, on the context stream.  enable=1 starts recording every
 * V-cycle kernel, enable=0 stops.  m3_profile_read (up to 9 values): for
 * the fine-level fused Jacobi sweeps in FP64, the fine-level fused sweeps of
 * the mixed-precision V-cycle, and every other V-cycle kernel (middle-level
 * sweeps, residual sweeps, transfers, coarse triangular solves, entry and
 * exit), three values each: launches, total seconds, total algorithmic bytes
 * (each stored array counted once, perfect reuse of gathered vectors).  No
 * reference counterpart (measurement only). */
int m3_profile(m3_ctx *ctx, int32_t enable);
/* Read + write bytes per second (GB/s) of a plain copy kernel over a buffer
 * of nbytes on HIP device `device`, averaged over reps launches (HIP events):
 * the practical HBM rate next to the 8 TB/s peak.  No reference counterpart
 * (measurement only; allocates its two buffers). */
int m3_copy_rate(int32_t device, int64_t nbytes, int32_t reps, double *gbs);
int m3_profile_read(m3_ctx *ctx, double *out, int32_t nout);

/* Level operator as block CSR (3x3 blocks, row-major inside a block):
 * rowptr (nnod+1), col (nnzb), val (9*nnzb).  Pass NULL pointers to query
 * nothing but sizes via m3_stats.  No reference counterpart (diagnostics). */
int m3_get_operator(m3_ctx *ctx, int32_t level, int64_t *rowptr, int32_t *col, double *val);

/* [T] = advect3d_slm_p_sph(MESH,COMM,Ux,Uy,Uz,T,dt,OPTS_SLM,WS_SLM)
 * (mfiles_SPH/advect3d_slm_p_sph.m:1-140) for a field on the P2 nodes of the
 * finest mesh: PC2 back-tracking with the reference's projections
 * (backtrack_PC2, predictor_ / corrector_step_with_projections, :165-243,
 * :298-440; the radial length is |U_par| dt as there), radii shifted into
 * the shell (find_pts_outside_domain_sph.m), local coordinates in the
 * spherical coordinates of each element's class frame
 * (local_coords_3d_sph.m, local_coords_curved_3d_sph.m for the iso
 * elements), quadratic interpolation (interp3d_tet.m) with the optional
 * monotone clip to the element's nodal range.  Ux, Uy, Uz: Cartesian
 * velocity on the nnod P2 nodes (VAR.Ux, Uy, Uz); T (nnod) is advected in
 * place.  opts NULL: the reference defaults (default_numerics_M3TET.m:
 * 141-153, PC2, quadratic, monotonic).  The point search walks over face
 * neighbours (the reference's tsearch2_sph search workspaces are not
 * needed); info (may be NULL) counts the back-tracking points shifted onto
 * the boundary and the searches that ended on their best element after 64
 * steps. */
enum { M3_SLM_EU1 = 1, M3_SLM_PC2 = 2, M3_SLM_RK4 = 3 };          /* OPTS_SLM.method_BT */
enum { M3_SLM_LINEAR = 1, M3_SLM_QUADRATIC = 2, M3_SLM_CUBIC = 3 }; /* OPTS_SLM.method_interp */
typedef struct {
  int32_t method_BT;      /* M3_SLM_PC2, or M3_SLM_EU1 (backtrack_EU1, :145-161: theta - dt Ux / r,
                             phi - dt Uy / r, r - dt Uz, the three arrays taken as (v_theta, v_phi, v_r)
                             as there); M3_SLM_RK4 is rejected as in the reference (:104-105) */
  int32_t method_interp;  /* M3_SLM_QUADRATIC (the reference stops on the others for P2 fields,
                             locate_points_interp_vars_3d_sph.m:147-149) */
  int32_t monotonic;      /* OPTS_SLM.monotonic: 1 clip to the element's nodal range */
} m3_slm_opts;
typedef struct {
  int64_t nshift;         /* predictor and corrector points moved onto r_cmb / r_surf */
  int64_t nunresolved;    /* searches that took their best element after 64 steps */
} m3_slm_info;
int m3_advect3d_slm_p_sph(m3_ctx *ctx, const double *Ux, const double *Uy, const double *Uz, double *T, double dt,
                          const m3_slm_opts *opts, m3_slm_info *info);

/* Semi-Lagrangian temperature update on the P1 vertices over one time step,
 * the step after the Stokes solve in the time loop
 * (mfiles_SPH/advect3d_slm_p_sph.m:1, backtrack_PC2 :165-243): each vertex
 * is traced back over dt with a predictor-corrector step along great circles
 * (the tangential velocity moves a point along the sphere of its radius, the
 * radial velocity changes the radius), departure points outside the shell are
 * shifted onto the nearest boundary (find_pts_outside_domain_sph), and T is
 * interpolated linearly in the straight P1 tetrahedron that holds the point.
 * T and T_out: nVnod vertex temperatures; U: 3*nnod velocity in the rotated
 * (theta, phi, r) frame as returned by m3_flow3d_patera_sph (vertex nodes are
 * read); vertices on the CMB / surface get T_cmb / T_surf. */
int m3_sl_advect(m3_ctx *ctx, const double *T, const double *U, double dt, double T_cmb, double T_surf,
                 double *T_out);

/* Options of the thermal diffusion step, SETTINGS.OPTS_D
 * (default_numerics_M3TET.m:95-134; defaults in brackets). */
typedef struct {
  double theta;        /* OPTS_D.theta: time rule, 1 backward Euler [1], 0.5 Crank-Nicolson, 0 explicit */
  int32_t lumping;     /* OPTS_D.lumping: 1 'yes' (row-sum mass matrix) [1], 0 'no' */
  int32_t nip;         /* OPTS_D.nip: 1, 4, 5, 8, 10, 11 or 14 [4] */
  double tol;          /* OPTS_D.tol [1e-8] */
  int32_t is_abs_tol;  /* OPTS_D.is_abs_tol: 0 relative to the initial residual [0] */
  int32_t itmax;       /* OPTS_D.itmax [500] */
} m3_diffusion_opts;

typedef struct {
  int32_t nit;         /* PCG iterations (profiling.nit of pcg_solver_p) */
  double norm_r0;      /* initial residual (RMS over the free nodes) */
  double norm_r;       /* final residual */
  double tol;          /* absolute tolerance used */
  double t_assemble, t_solve; /* s */
} m3_diffusion_info;

/* Linear tetrahedra of the diffusion step: EL2NOD is 4 x nel, 1-based, over
 * the first nnodT nodes of the finest mesh (the P1 vertices with the vertex
 * tetrahedra, or all P2 nodes with each 10-node element split into 8 linear
 * ones as diffusion3d_p.m:67-70 does for OPTS_D.eltype = 'linear').  Element
 * classes are computed on these tetrahedra (check_els_in_cone.m,
 * check_phi.m; assembly_diffusion_3d_double_jacobian.m:73-93) with the cone
 * half-aperture theta_cone in degrees (SETTINGS.theta_cone). */
int m3_diffusion_mesh(m3_ctx *ctx, const uint32_t *EL2NOD, int64_t nel, int64_t nnodT, double theta_cone);

/* T = diffusion3d_p(T,kappa,MESH,COMM,SETTINGS,TBC,dt) (diffusion3d_p.m:1-116):
 * conductivity and mass matrices of the double-Jacobian linear elements
 * (assembly_diffusion_3d_double_jacobian.m, class kernels
 * mfiles_SPH/assembly_diffusion_els_*_opt.m), lumping, the theta rule, the
 * fixed temperatures TBC.ifix / TBC.vfix (1-based node indices) and the
 * Jacobi-preconditioned CG of pcg_solver_p.m:49-186.  T (nnodT) is updated
 * in place.  kappa = 0 returns T unchanged, as the reference does. */
int m3_diffusion3d(m3_ctx *ctx, double *T, double kappa, double dt, const int64_t *ifix, const double *vfix,
                   int64_t nfix, const m3_diffusion_opts *opts, m3_diffusion_info *info);

/* Operators of the last m3_diffusion3d call for parity checks: y = CC x
 * (which 0), y = MM x (which 1, the consistent mass matrix, assembled only by
 * a step with lumping = 0), y = MM_lumped x (which 2).  x, y: nnodT.  No
 * reference counterpart (diagnostics). */
int m3_diffusion_apply(m3_ctx *ctx, int32_t which, const double *x, double *y);

/* Mesh set-up: unique undirected bars in the order of their first occurrence,
 * find_unique_bars (mfiles_SPH/tetmesh_p1_to_p2_sph.m:238-254), on HIP device
 * `device` (no context).  bars: n x 2 node indices (row-major, >= 0, either
 * orientation).  Out: *nu unique bars; first[u] = position of the first
 * occurrence of unique bar u (first needs room for n entries); bar_of[i] =
 * unique index of bar i.  Returns M3_E_ARG for negative node indices. */
int m3_unique_bars(int32_t device, const int32_t *bars, int64_t n, int64_t *first, int64_t *bar_of, int64_t *nu);

/* Mesh set-up: the whole multigrid hierarchy on HIP device `device` (no
 * context), replacing the set-up chain of init_mesh_curved_p.m:60-115 from the
 * coarsest vertex mesh on:
 *   tetmesh_p1_to_p2_sph.m:183-232  curved P2 promotion of every level (element
 *       classes, mid-side nodes in the original, X-rotated or Z-rotated
 *       spherical frame, bar numbering of find_unique_bars);
 *   tetmesh_refine_sph.m:56-89, tetmesh_p2_to_p1.m:27-116  8-way refinement
 *       along the shortest interior diagonal;
 *   cubic_els_in_cone_iso.m:3-346  20-node geometry of the finest in-cone iso
 *       elements;
 *   intermesh_transfer_matrix.m:8-23  node-level transfer operators.
 * Inputs: X4 (n4 x 3, row-major), EL4 (nel4 x 4, 0-based, row-major), pid4
 * (n4, PointID: 301 CMB, 306 surface), radii of the two boundaries, nmg levels,
 * the cone half-aperture in degrees.  Geometry uses fixed IEEE operation
 * sequences for sin, cos and atan2, so the result is a deterministic function
 * of the input (the same on every GPU and equal to the host restatement in
 * m3tet_sph_amd/mesh.py).  The finest level may hold at most 2^21 vertices
 * when it has iso elements.  Results stay on the device until read with the
 * getters below (host buffers; a NULL buffer is skipped); level 0 is the
 * finest.  Errors: m3_last_error(NULL). */
typedef struct m3_hier m3_hier;
int m3_hier_build(m3_hier **out, int32_t device, const double *X4, const int32_t *EL4, const int32_t *pid4,
                  int64_t n4, int64_t nel4, double r_cmb, double r_surf, int32_t nmg, double theta_cone);
/* sizes and EL2NOD (nel x 10, 0-based) of one level; isplit (nel, not for the
 * finest level): the split type 0..2 of each element of this level */
int m3_hier_level(const m3_hier *h, int32_t level, int64_t *nel, int64_t *nnod, int64_t *nVnod, int64_t *EL2NOD,
                  int8_t *isplit);
/* finest level: GCOORD (nnod x 3), GCOORD_SPH (theta, phi, r; boundary radii
 * set), PointID, element class 0..3 (out-cone, out-cone crossing 2 pi, in-cone,
 * in-cone iso) */
int m3_hier_nodes(const m3_hier *h, double *X, double *SPH, int32_t *PointID, int8_t *cls);
/* finest in-cone iso elements (increasing, 0-based) and their 20 geometry
 * nodes (n_iso x 20 x 3, node order of sf_dsf_tet20) */
int m3_hier_iso(const m3_hier *h, int64_t *n_iso, int64_t *els, double *X20);
/* transfer from level + 1 to level: CSR with one row per fine node (indptr
 * nnod + 1, coarse node indices, weights) */
int m3_hier_transfer(const m3_hier *h, int32_t level, int64_t *nnz, int64_t *indptr, int64_t *indices, double *w);
/* GPU time of the build (ms, HIP events on its stream) */
int m3_hier_time(const m3_hier *h, double *ms);
void m3_hier_destroy(m3_hier *h);
/* The set-up's reproducible primitives evaluated on the GPU, for parity
 * checks (no reference counterpart): op 0 sin(x), 1 cos(x), 2 atan2(y, x),
 * 3 sqrt(x), 4 cartesian2spherical (x and out: n x 3), 5 spherical2cartesian
 * (n x 3).  Host buffers. */
int m3_detmath_eval(int32_t device, int32_t op, int64_t n, const double *x, const double *y, double *out);

/* m3_unique_bars without any allocation.  No counterpart in the reference:
 * it is for callers that cannot allocate device memory (code under HIP graph
 * capture, serving loops, harnesses that forbid hipMalloc).  bars (2 n int32),
 * first (room for n) and bar_of (n) are DEVICE buffers of GPU `device`; nu is
 * a host pointer.  The work space (hash table, per-bar arrays, scan sums;
 * 56 MiB) is a file-scope device array of the library, held on every GPU the
 * library runs on until the process ends; n above M3_NOALLOC_MAX_BARS is
 * rejected with M3_E_ARG.  The kernels run on `stream` (a hipStream_t, NULL
 * for the null stream) and the call returns after they finish.  Calls that
 * overlap on one GPU share the work space and race: serialise them.
 * Results equal m3_unique_bars; errors as there, with the message from
 * m3_last_error(NULL). */
#define M3_NOALLOC_MAX_BARS (1 << 20)
int m3_unique_bars_noalloc(int32_t device, const int32_t *bars, int64_t n, int64_t *first, int64_t *bar_of,
                           int64_t *nu, void *stream);

#ifdef __cplusplus
}
#endif
#endif
