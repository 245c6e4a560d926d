/*
 * allium_sweep.h -- C ABI of the MI355X DG upwind transport sweep.
 *
 * Drop-in for allium's InverseAdvectionOperator (src/sweep.hpp:13-130) and the
 * operators the chive/scallion drivers wrap around it.  Plain pointers and
 * sizes only; every call returns an allium_status (never aborts) and
 * allium_last_error() describes the last failure on the calling thread.
 *
 * Vector layouts follow src/tvector.hpp:47-70 with TRANSPORT_VECTOR_LAYOUT
 * RIGHT (the reference default, CMakeLists.txt:102-119):
 *   psi / source : idx(g, a, s) = s + Ndof * (a + Nomega * g)
 *   phi (0th moment): idx(g, s) = s + Ndof * g
 * with Ndof = Ne * (p+1)^dim, elements numbered x-fastest and the dofs of an
 * element contiguous and lexicographic (Gauss-Lobatto nodes).
 */
#ifndef ALLIUM_SWEEP_H
#define ALLIUM_SWEEP_H

#ifdef __cplusplus
extern "C" {
#endif

typedef struct allium_sweep *allium_sweep_t;

typedef enum {
    ALLIUM_OK = 0,
    ALLIUM_ERR_ARG = -1,         /* bad argument / size mismatch */
    ALLIUM_ERR_NOT_DAG = -2,     /* sweep graph has a cycle (src/sweep.cpp:205-208) */
    ALLIUM_ERR_REFLECT = -3,     /* no quadrature direction matches a reflection */
    ALLIUM_ERR_DEVICE = -4,      /* HIP runtime failure */
    ALLIUM_ERR_UNSUPPORTED = -5, /* configuration the GPU path does not implement */
    ALLIUM_ERR_NUMERIC = -6,     /* non-finite input or result */
    ALLIUM_ERR_NOT_CONVERGED = -7/* iteration limit reached */
} allium_status;

typedef enum { ALLIUM_FP64 = 0, ALLIUM_FP32_REFINED = 1 } allium_precision;
typedef enum { ALLIUM_BC_INFLOW = 0, ALLIUM_BC_REFLECTIVE = 1 } allium_bc;

/* Structured quad/hex mesh with arbitrary vertex positions
 * (mfem::Mesh::MakeCartesian2D/3D, sfc_ordering=false, src/io.cpp:343-363). */
typedef struct {
    int dim;                /* 2 or 3 */
    int nel[3];             /* elements per axis */
    const double *vertices; /* prod(nel+1) x dim, x fastest; NULL => uniform box */
    double extents[3];      /* box lengths when vertices == NULL */
    int bc[6];              /* per boundary side axis*2 + {0 low, 1 high}: allium_bc */
} allium_mesh_desc;

/* Angular quadrature (LevelSymmetricQuadrature, src/angular_quadrature.cpp:98-147):
 * nomega == 0 => level-symmetric S_order generated by the library;
 * nomega > 0  => the explicit directions/weights given. */
typedef struct {
    int order;
    int nomega;
    const double *omega;    /* nomega x dim */
    const double *weights;  /* nomega */
} allium_quad_desc;

/* Info block filled by allium_sweep_info. */
typedef struct {
    long Ne, ndof_per_elem, Ndof, Nomega, G, psi_size, phi_size;
    long levels, cells, edges;
    int uniform_geometry;   /* 1 if every element is the same axis-aligned box */
    int launch_mode;        /* current launch strategy, see allium_sweep_set_launch */
} allium_sweep_info_t;

/* ---- construction (src/sweep.cpp:10-244) ------------------------------- */
/* ≙ InverseAdvectionOperator(fes, quad, total, bc_map, lump); sigma_t[G][Ne]
 * is the element-constant total cross section of each group.  lump is the
 * reference's bit set (src/sweep.cpp:940-1022): 1 the mass matrices, 2 the
 * gradient, 4 the face masses on the vertex (lumped) rule, 7 all; lumped
 * handles (fe_order 0 and 1) run the level kernels (box sweeps take lump = 0). */
int allium_sweep_create(const allium_mesh_desc *mesh, int fe_order, const allium_quad_desc *quad,
                        int G, const double *sigma_t, int lump, int precision,
                        allium_sweep_t *out);
/* ≙ ~InverseAdvectionOperator (src/sweep.cpp:246-257) */
void allium_sweep_destroy(allium_sweep_t h);
int allium_sweep_info(allium_sweep_t h, allium_sweep_info_t *info);
/* directions (Nomega x dim) and weights actually used */
int allium_sweep_quadrature(allium_sweep_t h, double *omega, double *weights);

/* ---- mutators (src/sweep.hpp:99-111) ----------------------------------- */
/* set_sigma and set_time_absorption finish the handle's own stream before they
 * replace the tables; work a caller enqueued on other streams through the
 * *_device entry points must be finished by the caller first. */
/* ≙ AssembleLocalMatrices after the total cross section changed */
int allium_sweep_set_sigma(allium_sweep_t h, const double *sigma_t);
/* ≙ SetTimeAbsorption(tau): adds tau * M to every local system */
int allium_sweep_set_time_absorption(allium_sweep_t h, double tau);
/* ≙ GetTimeAbsorption (src/sweep.hpp:105): 0 until a time absorption is set */
int allium_sweep_get_time_absorption(allium_sweep_t h, double *tau);
/* ≙ GetLumpingType (src/sweep.hpp:127): the lump bits of allium_sweep_create;
 * ≙ IsParallelBlockJacobi (src/sweep.hpp:109): always 0, one GPU sweeps the whole mesh */
int allium_sweep_get_lumping(allium_sweep_t h, int *lump, int *parallel_block_jacobi);
/* ALLIUM_FP64 or ALLIUM_FP32_REFINED local solves: the latter assembles and
 * factors each cell's system in FP32 (FP64 vectors in and out); FP64 accuracy
 * is restored by the defect correction of allium_source_iteration.  Where FP32
 * cells are not faster the request is served by the FP64 ones: 3D p = 2 on uniform
 * geometry, and 2D p = 1, 2 on uniform geometry in mode 3 (unlumped) */
int allium_sweep_set_precision(allium_sweep_t h, int precision);
/* 0 = one launch per level, 1 = hipGraph of level launches, 2 = persistent
 * kernel with device-side level counters (disabled), 3 = one workgroup per
 * (direction, group) sweeping all levels with workgroup barriers (directions
 * must not couple: no reflective side), 4 = box sweeps: a workgroup sweeps a
 * box of elements for several directions of one octant with the face traces
 * in LDS, one launch per anti-diagonal of boxes (uniform geometry, directions
 * that do not couple), 5 = the box-sweep launches in a hipGraph, -1 = pick by
 * measurement (the autotuner: launch mode x workgroup size x lanes per cell x
 * box extents x directions per workgroup) */
int allium_sweep_set_launch(allium_sweep_t h, int mode);
/* explicit tuning: launch mode, workgroup size (64..256, multiple of 64; up
 * to 512 for mode 3, 1024 for box sweeps at p = 1) and
 * lanes per cell (1, 2 or 4: each lane owns n/lanes rows of a cell's system;
 * size and lanes are without effect on level launches at 3D p = 2 and at 3D p = 1 on
 * general geometry, where 256 threads take 16 or 8 lanes per cell, and the autotuner
 * tries and reports 256 and 1 there; 0: one lane per cell in direction-uniform waves over XCD-local spatial bins,
 * uniform geometry only; modes 3..5 take 1) */
int allium_sweep_set_tuning(allium_sweep_t h, int mode, int block, int lanes);
int allium_sweep_get_tuning(allium_sweep_t h, int *mode, int *block, int *lanes);
/* box-sweep tiling (modes 4/5): box extents in elements (clamped to the
 * mesh), directions of one octant per workgroup (1..64), workgroup size
 * (multiple of 64: 64..256, or 64..1024 at p = 1, where each cell is solved
 * by 2^(dim-1) lanes) and input prefetch (0 none, 2 the next level's source
 * and cross section loaded while the current level solves, 3 (p = 1) the
 * level after next as well).
 * ALLIUM_ERR_ARG when the tiling needs more than 64 KiB of LDS per workgroup. */
int allium_sweep_set_box_tiling(allium_sweep_t h, int bx, int by, int bz, int dirs_per_group, int threads,
                                int prefetch);
int allium_sweep_get_box_tiling(allium_sweep_t h, int *bx, int *by, int *bz, int *dirs_per_group, int *threads,
                                int *prefetch);

/* ---- negative-flux fixups (src/fixup.cpp, src/sweep.hpp:75-77,116-122) - */
/* Applied after every cell solve as Mult_Upwind does (src/sweep.cpp:465-469):
 * ZERO clips psi at psi_min; ZERO_AND_SCALE clips, then scales the cell to its
 * balance sum(rhs) = (column sums of A) . psi (failed if either is negative);
 * RYOSUKE clips, then rebalances the positive unknowns with their ratios kept
 * (at most 3 of them: beyond, the sweep returns ALLIUM_ERR_NUMERIC where the
 * reference aborts).  The local-optimization fixup (mfem::SLBQPOptimizer) is
 * not provided.  With a fixup on, sweeps run the level kernel with FP64 cell
 * solves whatever the launch mode.  2D p = 0..2 and 3D p = 0..1. */
#define ALLIUM_FIXUP_NONE 0
#define ALLIUM_FIXUP_ZERO 1
#define ALLIUM_FIXUP_ZERO_AND_SCALE 2
#define ALLIUM_FIXUP_RYOSUKE 3
/* ≙ SetFixupOperator(op) (turns it on; ALLIUM_FIXUP_NONE turns it off), with
 * the deck's psi_min (default 0).  Resets the counts. */
int allium_sweep_set_fixup(allium_sweep_t h, int type, double psi_min);
/* ≙ UseFixup(bool); IsFixupOn is *on of allium_sweep_get_fixup */
int allium_sweep_use_fixup(allium_sweep_t h, int use);
int allium_sweep_get_fixup(allium_sweep_t h, int *type, double *psi_min, int *on);
/* ≙ SetFixupMonitorData(x): d_monitor (device, G x Ne doubles, element e of
 * group g at e + g Ne) gains 1 per cell solve where the fixup applied or
 * failed; NULL stops the monitoring. */
int allium_sweep_set_fixup_monitor(allium_sweep_t h, double *d_monitor);
/* EventLog "fixup applied" / "fixup failed" (src/sweep.cpp:649-650): totals
 * since allium_sweep_set_fixup */
int allium_sweep_fixup_counts(allium_sweep_t h, long long *applied, long long *failed);

/* ---- the sweep (src/sweep.cpp:259-669) --------------------------------- */
/* ≙ InverseAdvectionOperator::Mult(source, psi): psi = L^{-1} source.
 * Host pointers, psi_size doubles each; source == psi (in place) is allowed. */
int allium_sweep_mult(allium_sweep_t h, const double *source, double *psi);
/* Same on device pointers (HBM-resident), enqueued on `stream` (hipStream_t). */
int allium_sweep_mult_device(allium_sweep_t h, const double *d_source, double *d_psi, void *stream);
/* psi = L^{-1}(source + iso): the phi-sized iso (G x Ndof) is added to every
 * direction's right-hand side (an isotropic source per steradian, i.e.
 * D^T phi = phi / sum(w) applied inside the sweep, the TransportOperator
 * composition of src/transport_op.hpp:23-33); d_source may be NULL */
int allium_sweep_mult_iso_device(allium_sweep_t h, const double *d_source, const double *d_iso, double *d_psi,
                                 void *stream);
/* The same sweep followed by DiscreteToMoment::Mult (phi = sum_a w_a psi_a,
 * src/transport_op.cpp:3-89), the pair of TransportOperator::Mult
 * (src/transport_op.hpp:23-33); d_source or d_iso may be NULL.  d_phi must
 * not alias the other vectors. */
int allium_sweep_mult_moments_device(allium_sweep_t h, const double *d_source, const double *d_iso, double *d_psi,
                                     double *d_phi, void *stream);
/* Frontier index of every (element, angle): level[e * Nomega + a]
 * (the reference's Kahn frontiers, src/sweep.cpp:308-322,477-512). */
int allium_sweep_levels(allium_sweep_t h, int *level_of_node);

/* ---- streaming operator and balance (src/sweep.cpp:1246-1462) --------- */
/* ≙ AdvectionOperator::Mult: Lpsi = L psi (device pointers) */
int allium_apply_L_device(allium_sweep_t h, const double *d_psi, double *d_Lpsi, void *stream);
int allium_apply_L(allium_sweep_t h, const double *psi, double *Lpsi);
/* ≙ AdvectionOperator::ComputeBalance: absorption + leakage (FP64 reduction) */
int allium_balance(allium_sweep_t h, const double *psi, double *out);
int allium_balance_device(allium_sweep_t h, const double *d_psi, double *out, void *stream);
/* No counterpart in the reference: allium_balance_device for callers that
 * cannot allocate device memory (code under HIP graph capture, tight serving
 * loops, harnesses that forbid hipMalloc).  The block partials and the result
 * live in a file-scope device workspace of 512 KiB per GPU, held until the
 * process ends; the call allocates nothing.  Ne * G <= 8,388,608, else
 * ALLIUM_ERR_ARG.  Every call on one GPU shares that GPU's workspace: calls
 * that overlap on one GPU (other streams or threads) race.  Synchronizes
 * `stream`. */
int allium_balance_device_noalloc(allium_sweep_t h, const double *d_psi, double *out, void *stream);

/* ---- source and moments (src/sweep.cpp:1160-1185, src/transport_op.cpp) */
/* ≙ FormTransportSource: per-steradian element-constant source Q[G][Ne]
 * (NULL = 0) and isotropic inflow[G][2*dim] per boundary side (NULL = vacuum). */
int allium_form_source(allium_sweep_t h, const double *Q, const double *inflow, double *source);
/* ≙ DiscreteToMoment::Mult / MultTranspose (0th moment), device pointers */
int allium_moments_device(allium_sweep_t h, const double *d_psi, double *d_phi, void *stream);
int allium_moments_transpose_device(allium_sweep_t h, const double *d_phi, double *d_psi, void *stream);
/* ≙ DiscreteToMoment with dim + 1 moments (src/transport_op.cpp:3-89; chive's
 * Dlin_aniso, exe/chive.cpp:482): [phi, J_0 .. J_{dim-1}] laid out (m, g, s) with
 * s fastest, J_m = sum_a w_a Omega_m psi_a; the transpose is
 * psi = (phi + 3 Omega . J) / sum w.  d_mom holds (dim + 1) G Ndof doubles. */
int allium_moments_aniso_device(allium_sweep_t h, const double *d_psi, double *d_mom, void *stream);
int allium_moments_aniso_transpose_device(allium_sweep_t h, const double *d_mom, double *d_psi, void *stream);
/* block-diagonal MassIntegrator(coef[Ne]) on each group block (the
 * scattering mass Ms of exe/chive.cpp:593-599), device pointers */
int allium_mass_device(allium_sweep_t h, const double *d_coef, const double *d_x, double *d_y,
                       void *stream);

/* ---- source iteration (src/linalg.cpp:103-153, exe/chive.cpp:700-735) -- */
/* Options for allium_source_iteration. */
typedef struct {
    double abstol, reltol;  /* SLISolver tolerances on ||phi_{k+1} - phi_k||_2 */
    int maxit;
    int precision;          /* ALLIUM_FP64: plain SI with FP64 sweeps.
                               ALLIUM_FP32_REFINED: FP32 local solves inside an
                               FP64 defect correction on the transport residual */
    int accel;              /* 0 none; 1 learned correction: accel_handle is an
                               allium_cnn_t (allium_cnn.h); 3D uniform meshes, G == 1.
                               It is switched off for the rest of the solve once
                               accel_patience iterations have passed without a new
                               lowest FP64 residual; the iterate of the lowest
                               residual is then restored and accel_fallback (an
                               allium_dsa_t or NULL) takes over.
                               2 diffusion synthetic acceleration: accel_handle is an
                               allium_dsa_t (allium_dsa.h) built on this handle; the
                               residual norm is then that of the preconditioned
                               change z = r + K^{-1} Ms r (SLISolver with prec) */
    void *accel_handle;
    void *accel_fallback;
    int accel_prolong;      /* 0 element-constant correction; 1 (p = 1) continuous:
                               each node takes the mean over the elements at its vertex */
    int accel_patience;     /* iterations without a new lowest residual tolerated (>= 1) */
    double *history;        /* optional (G == 1), maxit x 2 x Ne doubles: per iteration
                               but the last, the element-average scalar flux after the
                               iteration, then the element-average change the
                               iteration made before any learned correction */
    double *raw_norms;      /* optional, maxit doubles: the unpreconditioned change
                               ||phi_{k+1} - phi_k||_2 of each iteration (before any DSA
                               or learned correction; equals norms[] without them) */
    int *inner_iterations;  /* optional, maxit ints: CG iterations of the DSA solve in
                               each iteration (0 where DSA did not run) */
} allium_si_options;

/* ≙ chive's SI path: b = D L^{-1} q; SLISolver on T = I - D L^{-1} D^T Ms;
 * final sweep for psi.  Host pointers: sigma_s[Ne] (G == 1: scattering;
 * G > 1: group-diagonal), source[psi_size], phi[phi_size] out, psi[psi_size]
 * out (may be NULL), norms[maxit] out (may be NULL). */
int allium_source_iteration(allium_sweep_t h, const double *sigma_s, const double *source,
                            const allium_si_options *opt, double *phi, double *psi,
                            double *norms, int *iterations);
/* Same with d_source, d_phi and d_psi (may be NULL) in device memory (HBM-
 * resident inputs: no PCIe copy of the psi-sized source); sigma_s, norms and
 * the optional option arrays stay on the host. */
int allium_source_iteration_device(allium_sweep_t h, const double *sigma_s, const double *d_source,
                                   const allium_si_options *opt, double *d_phi, double *d_psi,
                                   double *norms, int *iterations);

/* ---- Krylov outer solvers (src/io.cpp:179-230, exe/chive.cpp:700-735) -- */
/* chive's "gmres" (mfem::GMRESSolver, left-preconditioned) and "fgmres"
 * (mfem::FGMRESSolver, right-preconditioned, flexible) on the same
 * T = I - D L^{-1} D^T Ms and b = D L^{-1} q as the source iteration. */
#define ALLIUM_SOLVER_GMRES 1
#define ALLIUM_SOLVER_FGMRES 2
typedef struct {
    int solver;             /* ALLIUM_SOLVER_GMRES or ALLIUM_SOLVER_FGMRES */
    int kdim;               /* restart length, 1..200 (chive's default 50) */
    double abstol, reltol;  /* stop once the residual estimate <= max(reltol * beta0, abstol);
                               beta0 = ||M b|| (GMRES with M) or ||b|| */
    int maxit;              /* operator applications */
    int accel;              /* preconditioner: 0 none; 2 DSA, accel_handle an allium_dsa_t
                               built on this handle (M = I + K^{-1} Ms); 1 learned (FGMRES
                               only), accel_handle an allium_cnn_t: M v = v + net(v), the
                               correction the source iteration adds, 3D uniform, G == 1.
                               The learned preconditioner is replaced by accel_fallback (an
                               allium_dsa_t, or NULL for none) once accel_patience
                               consecutive steps each cut the residual estimate by less than
                               10 %; FGMRES allows the change within a cycle. */
    void *accel_handle;
    void *accel_fallback;
    int accel_prolong;      /* learned: 0 element-constant, 1 (p = 1) continuous */
    int accel_patience;     /* >= 1 */
    int *inner_iterations;  /* optional, maxit ints: CG iterations of the DSA solve in each
                               step (0 where DSA did not run) */
    int *accel_steps;       /* optional out: steps that used the learned preconditioner */
    int accel_max_steps;    /* learned: used in at most this many steps, then
                               accel_fallback (0: no limit) */
} allium_krylov_options;

/* Defaults: FGMRES, kdim 50, abstol 1e-8, reltol 0, maxit 100, no preconditioner,
 * continuous learned correction, patience 3. */
int allium_krylov_default_options(allium_krylov_options *opt);
/* Host pointers as allium_source_iteration; norms[maxit + 1] out (may be NULL):
 * norms[0] = beta0, norms[j] the residual estimate after step j (mfem's
 * monitor values); when a restart finds convergence, norms[*iterations] is the
 * recomputed residual.  *iterations = mfem's final iteration count.  FP64 sweeps
 * (the handle's precision setting is not used here).  Initial guess zero. */
int allium_krylov_solve(allium_sweep_t h, const double *sigma_s, const double *source,
                        const allium_krylov_options *opt, double *phi, double *psi, double *norms,
                        int *iterations);
/* Same with d_source, d_phi and d_psi (may be NULL) in device memory; sigma_s
 * and norms stay on the host.  Work is enqueued on the handle's stream and
 * finished on return. */
int allium_krylov_solve_device(allium_sweep_t h, const double *sigma_s, const double *d_source,
                               const allium_krylov_options *opt, double *d_phi, double *d_psi, double *norms,
                               int *iterations);

/* ---- batched sweeps of independent instances -------------------------- */
/* Several handles of uneven meshes swept together: each launch runs one level
 * of every instance, so a batch takes max(levels) launches instead of
 * sum(levels).  Implemented for the cooperative 3D p = 2 path; all handles
 * must share geometry kind (uniform or not) and precision.  At most 16. */
typedef struct allium_sweep_batch *allium_sweep_batch_t;
int allium_sweep_batch_create(const allium_sweep_t *handles, int count, allium_sweep_batch_t *out);
void allium_sweep_batch_destroy(allium_sweep_batch_t b);
/* psi_i = L_i^{-1}(source_i + iso_i) for every instance; device pointers,
 * d_source and d_iso may be NULL (arrays) or hold NULL entries */
int allium_sweep_batch_mult_device(allium_sweep_batch_t b, const double *const *d_source,
                                   const double *const *d_iso, double *const *d_psi, void *stream);
/* GPU seconds of the batched sweeps and the number of batched sweeps */
int allium_sweep_batch_timing(allium_sweep_batch_t b, double *seconds, long *sweeps);

/* ---- logging (src/log.hpp; keys "sweep" and "sweeps", src/sweep.cpp:665-668) */
/* Accumulated GPU time of sweeps (seconds, hipEvent-timed) and sweep count. */
int allium_sweep_timing(allium_sweep_t h, double *sweep_seconds, long *sweeps);

/* ---- host-side setup, usable without a GPU ---------------------------- */
/* level-symmetric set (Nomega x dim directions, weights); *nomega in/out:
 * capacity in, count out */
int allium_host_quadrature(int order, int dim, double *omega, double *weights, int *nomega);
/* frontier index of every (element, angle) node and the number of levels */
int allium_host_levels(const allium_mesh_desc *mesh, const allium_quad_desc *quad, int *level_of_node,
                       long *nlevels);
/* FormTransportSource on the host (RIGHT layout, G x Nomega x Ndof) */
int allium_host_form_source(const allium_mesh_desc *mesh, int fe_order, const allium_quad_desc *quad,
                            int G, const double *Q, const double *inflow, double *source);
/* element e's unit mass (MG rule), gradient blocks -int phi_j d_d phi_i and
 * MassIntegrator-rule mass, each n x n row-major (grad: dim blocks) */
int allium_host_element_matrices(const allium_mesh_desc *mesh, int fe_order, int e, double *mass,
                                 double *grad, double *tmass);

/* Description of the last error on this thread (never NULL). */
const char *allium_last_error(void);

#ifdef __cplusplus
}
#endif
#endif
