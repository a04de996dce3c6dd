/* pansfem2_amd: MI355X (gfx950) implementation of PANSFEM2's SIMP topology-
 * optimisation inner loop behind a plain C ABI.
 *
 * Conventions
 *   - Every entry point returns int: PF_OK (0), PF_NOT_CONVERGED (>0, a valid
 *     last iterate is returned, as ScalingCG does at
 *     src/LinearAlgebra/Solvers/CG.h:451-452), or a negative error code.  The
 *     message of the last error is pf_last_error(ctx).
 *   - Host pointers are owned by the caller and only read/written during the
 *     call.  *_dev entry points take device pointers (hipMalloc'd, on the
 *     context's device) and enqueue on the context's stream; they return after
 *     the work is complete unless stated otherwise.
 *   - One context per host thread.  A context owns one HIP stream (default
 *     priority) and all device buffers of its grid.
 *   - Vectors named *_free are in the reference's free-DOF numbering
 *     (SetDirichlet + Renumbering); element arrays are in element-id order.
 *
 * The reference is header-only C++ templates (no ABI of its own); each entry
 * point below names the reference routine it replaces.  The C++ drop-in
 * facade include/pansfem2/pansfem2.hpp binds these entry points under the
 * reference's own names.
 */
#ifndef PANSFEM2_AMD_H
#define PANSFEM2_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
    PF_OK = 0,
    PF_NOT_CONVERGED = 1,
    PF_ERR_ARG = -1,
    PF_ERR_HIP = -2,
    PF_ERR_STATE = -3,
    PF_ERR_NUMERIC = -4,
    PF_ERR_NOMEM = -5,
    PF_ERR_UNSUPPORTED = -6
};

/* operators for pf_apply_K / pf_pcg (PF_OP_MG, PF_OP_MG32: pf_pcg only;
 * PF_OP_MG32: multigrid PCG in FP32 inside FP64 iterative refinement) */
enum { PF_OP_CSR64 = 0, PF_OP_EBE64 = 1, PF_OP_EBE32 = 2, PF_OP_LEARNED = 3, PF_OP_MG = 4, PF_OP_MG32 = 5 };
/* filter modes for pf_filter */
enum { PF_FILTER_VARIABLES = 0, PF_FILTER_SENSITIVITIES = 1 };

typedef struct pf_ctx pf_ctx;

typedef struct pf_solve_stats {
    int iterations;        /* loop iterations run (k+1 of the converging one)  */
    int status;            /* 1 converged, 2 itrmax reached, 3 breakdown        */
    double rel_residual;   /* recursive ||r||/||b|| at exit                     */
    double true_residual;  /* FP64 ||b - K x||/||b|| recomputed on the device   */
    double seconds;        /* device wall time of the solve                     */
    int outer;             /* refinement steps (mixed precision), else 0       */
    int fallbacks;         /* flexible-CG -> Jacobi-PCG fallbacks (learned)     */
} pf_solve_stats;

typedef struct pf_oc_params {
    double iota, lambdamin, lambdamax, lambdaeps, movelimit; /* OC<T> ctor (OC.h:45-60) */
    double vf, scale1;     /* volume closure of sample_optimize_density_oc.cpp:199-206 */
    int max_steps;         /* safety cap on bisection steps (the reference has none) */
    double beta;           /* > 0: the closure filters with HeavisideFilter at this beta
                              (src/Optimize/Filter/HeavisideFilter.h:62-75) */
} pf_oc_params;

typedef struct pf_mma_params {
    int m;                                   /* constraints; 1 supported on the device */
    double a0, a, c, d;                      /* MMA<T> ctor (MMA.h:63-88), m = 1 */
    double xmin, xmax;                       /* uniform bounds */
    double raa0, albefa, move, asyinit, asydecr, asyincr, epsvalue; /* SetParameters (MMA.h:91-100) */
    int max_newton;                          /* cap of the interior-point loop (MMA.h:199 has none) */
} pf_mma_params;

typedef struct pf_simp_params {
    double E1, E0, nu, t, p;       /* SIMP: E = E1 rho^p + E0 (1 - rho^p) (sample...oc.cpp:123) */
    double vf, R, scale0, scale1;  /* volume fraction, filter radius, objective/constraint scales */
    double cg_eps; int cg_itrmax;  /* ScalingCG(K, F, itrmax, eps) (sample...oc.cpp:132) */
    int use_mma;                   /* 0: OC update, 1: MMA update, 2: CONLIN update (uses mma's a0, a, c, d,
                                      bounds, move, epsvalue) */
    int solver;                    /* PF_OP_EBE64 (plain FP64) or PF_OP_CSR64 */
    int mixed;                     /* 1: FP32 EbE inner PCG inside FP64 refinement */
    double inner_eps;              /* inner tolerance of the mixed solve */
    int learned;                   /* 1: learned-preconditioned flexible CG (after training) */
    int stop_on_convergence;       /* honour OC/MMA IsConvergence (OC.h:67-73) */
    pf_oc_params oc;
    pf_mma_params mma;
    int collect;                   /* > 0: keep a training pair every `collect` CG chunks (32 iterations)
                                      of each solve (needs pf_precond_init) */
    int collect_max;               /* cap on pairs taken from one solve */
    int heaviside;                 /* 1: HeavisideFilter (HeavisideFilter.h:15-99) instead of DensityFilter */
    double beta0, beta_factor;     /* beta continuation of the density samples: beta0 multiplied by */
    int beta_every;                /* beta_factor at every beta_every-th iteration from 0
                                      (sample_optimize_density_oc.cpp:78,89-93: 0.5, 2, 40) */
    int iter_offset;               /* index of this call's first iteration in the continuation */
    int resume_optimizer;          /* 1: keep the context's MMA/CONLIN state (an earlier pf_simp_run or
                                      pf_mma_set_state) instead of re-initialising it: a continuation */
} pf_simp_params;

typedef struct pf_simp_history {
    double* f;        /* compliance per iteration (iters)         */
    double* g;        /* volume constraint per iteration          */
    double* lambda;   /* last OC lambda per iteration (0 for MMA) */
    int* cg_iters;    /* PCG iterations per iteration             */
    int* bisect;      /* OC bisection steps / MMA Newton steps    */
    double* seconds;  /* device wall time per iteration           */
    int iterations;   /* iterations run                           */
    double* residual; /* relative residual each solve ended at: the FP64 true residual
                         ||F - K u||/||F|| (the recursive one for pair-collecting solves) */
    int* fallbacks;   /* flexible-CG -> Jacobi-PCG fallbacks per solve (learned solves) */
} pf_simp_history;

/* ---- lifecycle --------------------------------------------------------- */
int pf_create(pf_ctx** ctx, int device);
int pf_destroy(pf_ctx* ctx);
const char* pf_last_error(pf_ctx* ctx);
/* Compiled device architecture and build flags of the library. */
const char* pf_build_info(void);

/* ---- mesh and DOFs ----------------------------------------------------- */
/* SquareMesh<T>(lx, ly, nx, ny) with GenerateNodes/GenerateElements
 * (src/PrePost/Mesher/SquareMesh.h:48-70,97-106): quad4, 2 DOF per node. */
int pf_grid2d(pf_ctx* ctx, int nx, int ny, double lx, double ly);
/* Structured hex8 grid with ShapeFunction8Cubic node order
 * (src/FEM/Controller/ShapeFunction.h:299): 3 DOF per node.  The reference
 * has no 3D mesher; numbering is documented in pf_internal.h. */
int pf_grid3d(pf_ctx* ctx, int nx, int ny, int nz, double lx, double ly, double lz);
/* SetDirichlet + Renumbering (src/FEM/Controller/BoundaryCondition.h:19-25,
 * src/FEM/Controller/Assembling.h:175-186): the listed (node, dof) pairs are
 * fixed (prescribed value 0); free DOFs are numbered in (node, dof) order. */
int pf_set_dirichlet(pf_ctx* ctx, const int32_t* node, const int32_t* dof, int nfixed, int32_t* n_free);
/* Read back nodetoglobal (nn*ndpn, -1 for fixed). */
int pf_get_dofmap(pf_ctx* ctx, int32_t* n2g);
/* Assembling(F, qfixed, nodetoglobal) (Assembling.h:151-158): nodal point
 * loads accumulated into the right-hand side used by pf_simp_run. */
int pf_set_point_loads(pf_ctx* ctx, const int32_t* node, const int32_t* dof, const double* value, int n);
/* Read back the assembled load vector in free-DOF numbering (N). */
int pf_get_load(pf_ctx* ctx, double* F_free);

/* ---- element matrices and material ------------------------------------- */
/* Shared unit element matrix K0 (nd x nd, row-major) at E = 1: the result
 * of PlaneStrainStiffness (src/FEM/Equation/PlaneStrain.h:19-58) or
 * SolidLinearIsotropicElastic (src/FEM/Equation/Solid.h:19-64) on one
 * element of the grid.  Used by the matrix-free operator and compliance. */
int pf_set_element_matrix(pf_ctx* ctx, const double* K0, int nd);
/* PlaneStrainStiffness / SolidLinearIsotropicElastic evaluated on the device
 * in the reference's operation order for element `e` with modulus E (check
 * path): Ke is nd x nd. */
int pf_element_stiffness(pf_ctx* ctx, int e, double E, double nu, double t, double* Ke);
/* SIMP material: E = E1 rho^p + E0 (1 - rho^p) (sample...oc.cpp:123,142). */
int pf_set_material(pf_ctx* ctx, double E1, double E0, double p, double nu, double t);
/* Element densities (ne) -> device; element moduli computed on the device. */
int pf_set_density(pf_ctx* ctx, const double* rho);
/* Element moduli given directly (ne), as the driver passes E to
 * PlaneStrainStiffness (sample...oc.cpp:123-126). */
int pf_set_moduli(pf_ctx* ctx, const double* E);

/* ---- assembled CSR check path ------------------------------------------ */
/* Assembling(LILCSR&, ...) over all elements + CSR<T>(LILCSR&)
 * (Assembling.h:46-66, src/LinearAlgebra/Models/LILCSR.h:92-114,
 * src/LinearAlgebra/Models/CSR.h:92-105) on the device, element matrices in
 * reference arithmetic from the current moduli.  Structure and values are
 * bit-identical to the reference's.  *nnz receives the entry count. */
int pf_assemble_csr(pf_ctx* ctx, int64_t* nnz);
/* Same structure, values from caller-given element matrices instead of the
 * device's: ke_all is ne x nd x nd (row-major, element order of the grid),
 * e.g. what the C++ facade's Assembling(LILCSR&, ...) recorded.  The values
 * are the reference's sums (Assembling.h:46-66) for any element matrices. */
int pf_assemble_csr_elements(pf_ctx* ctx, const double* ke_all, int64_t* nnz);
/* Copy the assembled CSR to the host (indptr N+1, indices/data nnz). */
int pf_get_csr(pf_ctx* ctx, int32_t* indptr, int32_t* indices, double* data);

/* ---- operators and solvers --------------------------------------------- */
/* y = K x on free-DOF vectors.  PF_OP_CSR64 is CSR<T>::operator*
 * (CSR.h:108-122), bit-identical to the reference; PF_OP_EBE64/EBE32 apply
 * sum_e E_e K0 element by element without assembly. */
int pf_apply_K(pf_ctx* ctx, int op, const double* x_free, double* y_free);
/* ScalingCG(A, b, itrmax, eps) (CG.h:419-453): Jacobi-PCG from x0 = 0 that
 * stops when ||r_k|| < eps ||b|| (recursive residual).  op selects the
 * operator; PF_OP_EBE32 runs FP32 inner solves inside FP64 iterative
 * refinement to a true FP64 residual of eps. */
int pf_pcg(pf_ctx* ctx, int op, const double* b_free, double* x_free, double eps, int itrmax, pf_solve_stats* st);
/* Form of the Jacobi-PCG recurrences for the quad4 matrix-free solves of
 * this context (pf_pcg and pf_pcg_dev with PF_OP_EBE64 / PF_OP_EBE32, and
 * pf_simp_run), until changed.  PF_PCG_SCALINGCG (the default) is
 * ScalingCG's own order (CG.h:419-453), two reductions per iteration.  The
 * single-reduction forms follow Chronopoulos and Gear (p.Kp from u.Ku): one
 * reduction per iteration, the same iterates in exact arithmetic, the same
 * stopping test on the recursive residual, the Jacobi step as a product with
 * 1/D.  Grids whose vectors fit the registers and LDS of the chip (256 compute
 * units: up to 585,000 to 614,000 nodes by the grid's shape, 769 x 769 or
 * 1086 x 543 elements) are solved by one resident kernel in the first three
 * forms; larger ones, and the recomputed form, launch every iteration:
 *   PF_PCG_SINGLE_REDUCTION_CARRIED: s = K p and w = K u carried as vectors
 *     (88 bytes per free DOF and iteration);
 *   PF_PCG_SINGLE_REDUCTION_RECOMPUTED: s = K p recomputed from p on a
 *     two-node tile halo, w = K u kept only for its sum (56 bytes);
 *   PF_PCG_SINGLE_REDUCTION: the carried kernel while its working set (nine
 *     nodal vectors and the moduli) stays below 150 MB, else the recomputing
 *     one (the two meet near 125 MB; the last-level cache holds 256 MB).
 * Only FP64 quad4 solves use them: FP32 inner solves (PF_OP_EBE32), hex8,
 * CSR and learned solves keep ScalingCG's order.  Has no counterpart in the
 * reference. */
enum {
    PF_PCG_SCALINGCG = 0,
    PF_PCG_SINGLE_REDUCTION = 1,
    PF_PCG_SINGLE_REDUCTION_CARRIED = 2,
    PF_PCG_SINGLE_REDUCTION_RECOMPUTED = 3
};
int pf_set_pcg_form(pf_ctx* ctx, int form);
/* Jacobi-PCG solves with the matrix-free operators, MMA and CONLIN updates and
 * OC bisections without projection run in one resident kernel where the grid
 * fits the chip, and in kernels launched per iteration (per Newton or bisection
 * step) otherwise: on larger grids, where the resident kernel's buffers cannot
 * be had, and after
 *   - a stall (a resident kernel's workgroups have waited two seconds for one
 *     another): the call starts over launched, and so does the next one run,
 *     after a second stall in a row the next two, and so on up to 1024;
 *   - a refused cooperative launch (another process on the GPU has made one
 *     and still runs): this call and the next 1024 are launched.
 * The two sum in different orders, so that results agree to rounding and are
 * the same bits from run to run only where the same kernels ran: beside other
 * processes, with PF_RESIDENT_OFF.  Until changed:
 *   PF_RESIDENT_AUTO: as above (the default);
 *   PF_RESIDENT_OFF: always launched;
 *   PF_RESIDENT_STALL: as AUTO, but a resident solve's launches (2048
 *     iterations each; an update or bisection is one launch) after the first
 *     `after` end as stalled;
 *   PF_RESIDENT_NOMEM: as AUTO, but of the buffers that resident kernels still
 *     have to allocate, those after the first `after` are not to be had;
 *   PF_RESIDENT_REFUSED: as AUTO, but every cooperative launch is refused.
 * The last three are for tests of what follows; `after` is not used otherwise.
 * Has no counterpart in the reference. */
enum {
    PF_RESIDENT_AUTO = 0,
    PF_RESIDENT_OFF = 1,
    PF_RESIDENT_STALL = 2,
    PF_RESIDENT_NOMEM = 3,
    PF_RESIDENT_REFUSED = 4
};
int pf_set_resident(pf_ctx* ctx, int mode, int after);
/* How many solves (inner solves of a mixed one each), updates and bisections
 * of this context have run resident to their end, and how many gave way by a
 * stall or a refused launch. */
int pf_resident_runs(pf_ctx* ctx, int64_t* done, int64_t* gave_way);
/* Kernel of the hex8 matrix-free operator inside the fused PCG iteration
 * (pf_pcg, pf_pcg_dev, pf_simp_run and the multigrid PCG's outer FP64
 * operator on hex8 grids), until changed.  Both apply the same operator as
 * the element loop of Solid.h:19-64 with Assembling.h:46-66 (one K0 scaled
 * by E_e), differing in the order of the sums:
 *   PF_H8_OP_VALU: one node per thread, the node's 3 rows of its eight
 *     elements on the vector units (K0 from scalar loads in FP64, LDS in FP32);
 *   PF_H8_OP_MFMA: the element matrix as a batched product on the matrix
 *     cores (16 elements of one colour per product, K0 in registers), the
 *     rows summed per node in LDS in colour order (deterministic).
 *   PF_H8_OP_AUTO (the default): Jacobi-PCG solves of grids that fit the chip (256
 *     compute units: up to 128 x 64 x 64 elements) run in one resident kernel, with the
 *     element matrix in its parity basis where it has one (any box element of a
 *     material with the box's mirror planes), and the others use PF_H8_OP_VALU.
 * The other two are always launched.  Has no counterpart in the reference. */
enum { PF_H8_OP_AUTO = -1, PF_H8_OP_VALU = 0, PF_H8_OP_MFMA = 1 };
int pf_set_h8_operator(pf_ctx* ctx, int kind);
/* Same on device-resident free-DOF vectors. */
int pf_pcg_dev(pf_ctx* ctx, int op, const double* b_free_dev, double* x_free_dev, double eps, int itrmax,
               pf_solve_stats* st);
/* Compliance and sensitivities (sample_optimize_density_oc.cpp:136-162):
 * f = scale0 u^T K u and dfdrho_e = -scale0 p (E1 - E0) rho_e^(p-1) u_e^T K0 u_e
 * for the current densities.  u_free is a free-DOF vector (N). */
int pf_compliance_sens(pf_ctx* ctx, const double* u_free, double scale0, double* f, double* dfdrho);
/* No counterpart in the reference.  For callers that cannot allocate device
 * memory (code under HIP graph capture, serving loops or harnesses that
 * forbid hipMalloc): pf_compliance_sens on device-resident vectors -- u_free
 * (N), dfdrho (ne) and the compliance f (one double) are device pointers --
 * with the same kernel arithmetic and the same summation order, so f and
 * dfdrho are bit-identical to pf_compliance_sens's.  The call allocates
 * nothing: its only scratch, the compliance's per-workgroup partial sums, is
 * a static device array of the library (1024 doubles, 8 KiB per GPU, held
 * until the process ends; any grid fits, because the launch is capped at
 * 1024 workgroups, and a launch needing more is rejected with PF_ERR_ARG).
 * Every call on one GPU shares that array: calls that overlap on one GPU
 * (two contexts, two host threads) race and must be serialised by the
 * caller.  Returns after the work is complete. */
int pf_compliance_sens_dev_noalloc(pf_ctx* ctx, const double* u_free_dev, double scale0, double* f_dev,
                                   double* dfdrho_dev);

/* ---- filter ------------------------------------------------------------ */
/* DensityFilter<T> with the sample's neighbour rule |cg_i - cg_j| <= R,
 * w = (R - |.|)/R (src/Optimize/Filter/DensityFilter.h:34-71,
 * sample_optimize_density_oc.cpp:44-60).  Weights are recomputed on the
 * device from the element centroids in reference arithmetic. */
int pf_filter_setup(pf_ctx* ctx, double R);
/* mode 0: GetFilteredVariables (DensityFilter.h:45-56);
 * mode 1: GetFilteredSensitivitis (DensityFilter.h:60-71). ne in, ne out. */
int pf_filter(pf_ctx* ctx, int mode, const double* in, double* out);
/* HeavisideFilter<T> at `beta` over the current filter (grid rule or lists):
 * mode 0: GetFilteredVariables (HeavisideFilter.h:62-75), out = H(filter(s));
 * mode 1: GetFilteredSensitivitis (HeavisideFilter.h:78-99), out_i =
 * sum_j dfdrho_j H'(s~_j) w_ij / sum_j w_ij with s~ = filter(s). ne in, ne out. */
int pf_heaviside(pf_ctx* ctx, double beta, int mode, const double* s, const double* dfdrho, double* out);
/* SensitivityFilter<T> (scheme 1, Sigmund's) and SensitivityFilter2<T>
 * (scheme 2) (src/Optimize/Filter/SensitivityFilter.h:44-55,88-99) over the
 * current neighbour lists or the quad4 grid rule: scheme 1 gives
 * sum_j w_ij s_j dfds_j / (s_i sum_j w_ij), scheme 2 divides by
 * sum_j w_ij s_j instead.  ne in, ne out. */
int pf_sensitivity_filter(pf_ctx* ctx, int scheme, const double* s, const double* dfds, double* out);
/* DensityFilter<T>(n, neighbors, w) with caller-given lists
 * (DensityFilter.h:34-43): element e's neighbours are idx[ptr[e]..ptr[e+1])
 * with weights w (same order); pf_filter then uses the lists (sums in list
 * order, bit-identical to the reference) until pf_filter_setup is called.
 * The device OC closure (pf_oc_update, pf_simp_run) needs the grid rule. */
int pf_filter_set_lists(pf_ctx* ctx, const int32_t* ptr, const int32_t* idx, const double* w);

/* ---- optimisers -------------------------------------------------------- */
/* OC<T>::UpdateVariables (src/Optimize/Solver/OC.h:76-107) with the
 * sample's filtered-volume closure; x (ne) updated in place.  Returns
 * PF_NOT_CONVERGED (x still the reference's result) when the bisection
 * reaches max_steps, or when every tested lambda left the constraint on one
 * side, so that lambda ran to an end of [lambdamin, lambdamax]: the
 * reference returns silently in both cases (OC.h:82-106). */
int pf_oc_update(pf_ctx* ctx, double* x, const double* dfdx, const double* dgdx, const pf_oc_params* prm,
                 double* lambda_out, int* steps_out);
/* One bisection candidate of OC<T>::UpdateVariables for a given lambda
 * (OC.h:85-92): xplus = clamp(x (-dfdx/(dgdx lambda))^iota) within the move
 * limit.  For callers that evaluate their own constraint closure (the C++
 * facade's OC<T> with a host callable). ne in, ne out. */
int pf_oc_candidate(pf_ctx* ctx, const double* x, const double* dfdx, const double* dgdx, double lambda,
                    double iota, double movelimit, double* xplus);
/* MMA<T> (src/Optimize/Solver/MMA.h:15-509), m = 1, state kept in the
 * context: pf_mma_init resets it (ctor + SetParameters), pf_mma_update runs
 * UpdateVariables(x, f, dfdx, {g}, {dgdx}).  The interior-point loop, which
 * has no cap in the reference (MMA.h:199), stops at max_newton Newton steps:
 * pf_mma_update then returns PF_NOT_CONVERGED and leaves x and the state
 * unchanged. */
int pf_mma_init(pf_ctx* ctx, const pf_mma_params* prm);
int pf_mma_update(pf_ctx* ctx, double* x, double f, const double* dfdx, double g, const double* dgdx,
                  int* newton_steps);
/* The state MMA<T> carries between UpdateVariables calls (MMA.h:31-54):
 * the outer counter k, previousvalue, x_{k-1}, x_{k-2} and the asymptotes
 * L, U (ne each).  Saving it after some iterations and restoring it into a
 * context whose MMA (or CONLIN) was initialised with the same parameters
 * continues the run bit for bit (checkpoint/resume; the reference keeps it
 * only in the object).  Null output pointers are skipped by get_state. */
int pf_mma_get_state(pf_ctx* ctx, int* k, double* previousvalue, double* xkm1, double* xkm2, double* L, double* U);
int pf_mma_set_state(pf_ctx* ctx, int k, double previousvalue, const double* xkm1, const double* xkm2,
                     const double* L, const double* U);
/* CONLIN<T> (src/Optimize/Solver/CONLIN.h:18-455), m = 1, state in the
 * context: pf_conlin_init takes the ctor's a0, a, c, d, xmin, xmax and
 * SetParameters' move and epsvalue from prm (the MMA-only fields are
 * unused); pf_conlin_update runs UpdateVariables(x, f, dfdx, {g}, {dgdx}). */
int pf_conlin_init(pf_ctx* ctx, const pf_mma_params* prm);
int pf_conlin_update(pf_ctx* ctx, double* x, double f, const double* dfdx, double g, const double* dgdx,
                     int* newton_steps);

/* ---- the whole loop ---------------------------------------------------- */
/* The SIMP loop of sample_optimize_density_oc.cpp:83-208 (or the MMA
 * variant, sample_optimize_density_mma.cpp:88-204) run device-resident for
 * `iters` iterations on the current grid, Dirichlet set, loads and K0:
 * filter -> volume -> moduli -> PCG -> compliance/sensitivities -> filtered
 * sensitivities -> OC/MMA.  s (ne) holds the initial design and receives the
 * final one; rho_out (ne, may be NULL) the final filtered density.
 * PF_ERR_NUMERIC for a non-finite s.  A solve that stops at itrmax or an OC
 * update that returns PF_NOT_CONVERGED does not stop the loop (the
 * reference goes on with the last iterate): the call then returns
 * PF_NOT_CONVERGED with the first such message.  An MMA/CONLIN update that
 * reaches max_newton stops the loop at that iteration (PF_NOT_CONVERGED;
 * hist->iterations counts it). */
int pf_simp_run(pf_ctx* ctx, const pf_simp_params* prm, int iters, double* s, double* rho_out, pf_simp_history* hist);
/* Fill prm with the defaults of the SIMP workloads (E1 1, E0 1e-9, nu 0.3,
 * t 1, p 3, vf 0.5, R 1.5, scales 1, ScalingCG(100000, 1e-10), OC(0.5, 0,
 * 1e9, 1e-3, 0.2), MMA(a0 1, a 0, c 1e4, d 0, [0.01,1], 1e-5, 0.1, 0.2, 0.5,
 * 0.7, 1.2, 1e-6), density filter; Heaviside continuation 0.5, 2, 40). */
void pf_simp_default_params(pf_simp_params* prm);

/* ---- multigrid base preconditioner (quad4 and hex8) --------------------- */
/* No counterpart in the reference.  pf_mg_setup makes a geometric multigrid
 * V-cycle the base step of the flexible CG: pf_pcg with PF_OP_MG (FCG with
 * the V-cycle alone; PF_OP_MG32 the same PCG with FP32 vectors and operator
 * as the inner solve of FP64 iterative refinement to the FP64 true residual,
 * falling back to FP64 corrections when an FP32 step does not halve it) and
 * PF_OP_LEARNED (the network correction over the
 * V-cycle instead of over the Jacobi step; train after pf_mg_setup so the
 * network learns against the same base).  Coarse levels halve both element
 * counts down to at most 90 nodal DOFs (or an odd count); a coarse
 * element's matrix is the Galerkin product of its four children's
 * (bilinear prolongation, fixed DOFs removed at the finest level), built in
 * FP64 and applied in FP32; nu damped-Jacobi sweeps (weight omega) before
 * and after the coarse correction; a dense solve on the coarsest level.  The
 * hierarchy is rebuilt from the current moduli at the start of every solve.
 * nu = 0 switches the multigrid off; omega <= 0 takes the element's default
 * (0.6 quad4, 0.4 hex8: damped Jacobi smooths only below 2 / lambda_max of
 * D^-1 K, about 0.67 and 0.48). */
int pf_mg_setup(pf_ctx* ctx, int nu, double omega);
/* Prolongation of the quad4 hierarchy (hex8 hierarchies stay trilinear),
 * for this context's multigrid, now and at later pf_mg_setup calls.
 *   PF_MG_PROLONG_BILINEAR: geometric bilinear interpolation;
 *   PF_MG_PROLONG_STIFFNESS (the default): operator-dependent -- a coarse
 *     edge's midpoint follows the stiffer half of the edge, w_A = S_A /
 *     (S_A + S_B) with S the summed trace of the two fine element matrices
 *     along each half, and a coarse element's centre node is the harmonic
 *     extension -K_cc^-1 K_cb of its corner and edge values over the four
 *     children's matrices.  Each fine node's weights depend on its own edge
 *     or coarse element only, so the element-wise Galerkin coarsening stays
 *     exact.  On SIMP designs (solid/void contrast 1e9) the bilinear
 *     coarse levels misrepresent thin members; this keeps them stiff.
 * No counterpart in the reference. */
enum { PF_MG_PROLONG_BILINEAR = 0, PF_MG_PROLONG_STIFFNESS = 1 };
int pf_mg_set_prolongation(pf_ctx* ctx, int mode);
/* How the hex8 hierarchy's coarse levels form their residual r - A x, for
 * this context's multigrid, now and at later pf_mg_setup calls:
 *   PF_MG_RESIDUAL_NODE: one pass, each node gathering three rows of each of
 *     its elements' matrices;
 *   PF_MG_RESIDUAL_ELEMENT: two passes, y_e = K_e x_e per element (each
 *     matrix read once), then each node summing its elements' y_e;
 *   PF_MG_RESIDUAL_AUTO (the default): the element form on levels of at
 *     least 1024 elements, the node form below (where both are launch
 *     latency), except on the levels of at most 1024 nodes that run in one
 *     workgroup with the coarsest solve, which take the element form.
 * The forms add the same products in different orders (FP32 rounding).
 * No counterpart in the reference. */
enum { PF_MG_RESIDUAL_AUTO = 0, PF_MG_RESIDUAL_NODE = 1, PF_MG_RESIDUAL_ELEMENT = 2 };
int pf_mg_set_residual_form(pf_ctx* ctx, int form);
/* Build the hierarchy for the current moduli now (solves do it themselves). */
int pf_mg_build(pf_ctx* ctx);
/* One V-cycle z = V(r) on free-DOF host vectors, for the current moduli. */
int pf_mg_apply(pf_ctx* ctx, const double* r_free, double* z_free);
/* Level `level` of the built hierarchy: its element counts (nz = 0 for
 * quad4), and (when the pointers are not null) its FP64 element matrices
 * (level >= 1; row-major per element, element-local nodes in the shape
 * function's order, DOFs of a node together: ne x 64 for quad4, ne x 576 for
 * hex8), FP32 diagonal and nodal fixity bits (bit d: DOF d fixed).  *levels
 * receives the level count. */
int pf_mg_level(pf_ctx* ctx, int level, int* levels, int* nx, int* ny, int* nz, double* Ke, float* D,
                uint8_t* fix);

/* ---- measurement -------------------------------------------------------- */
/* Average device duration (HIP events on the context's stream, `reps`
 * back-to-back launches each) of the two PCG iteration kernels of operator
 * `op` on the current moduli: ms[0] = operator kernel (p update + K p +
 * p.q), ms[1] = vector-update kernel (x, r, z and the z.r, r.r partials),
 * ms[2] = density filter, ms[3] = one OC bisection step (one launch on quad4 grids),
 * ms[4] = the single-reduction iteration kernel, the mean of an odd and an even
 *         launch (PF_OP_EBE64 only, else 0).
 * Diagnostic only (no counterpart in the reference); it overwrites the
 * solver's work vectors. */
int pf_profile_kernels(pf_ctx* ctx, int op, int reps, double* ms);

/* ---- learned preconditioner -------------------------------------------- */
/* 4-level convolutional network on the nodal grid, 3x3 on a quad4 problem
 * and 3x3x3 on a hex8 one (BF16 weights and activations, FP32 accumulation
 * on MFMA), input (2 rho_node - 1, r/s) with s the RMS of r, output a field
 * y.  Inside flexible CG (PF_OP_LEARNED, Notay's FCG(m)) the preconditioner
 * is M(r) = a t + c y, t the Jacobi step r ./ D or, after pf_mg_setup, the
 * multigrid V-cycle, with (a, c) minimising the energy norm of the error
 * over span{t, y}; Jacobi-PCG takes over from the current iterate on
 * breakdown, divergence or stagnation.  No counterpart in the reference.
 * pf_precond_init builds the network for the current grid with seeded
 * weights. */
int pf_precond_init(pf_ctx* ctx, int channels, uint64_t seed);
/* Number of network parameters (FP32 master copy). */
int pf_precond_num_params(pf_ctx* ctx, int64_t* count);
int pf_precond_save(pf_ctx* ctx, float* params, int64_t* count);
int pf_precond_load(pf_ctx* ctx, const float* params, int64_t count);
/* Training pairs from a plain Jacobi-PCG solve of the current system
 * (current moduli and loads): every `every` chunks of 32 iterations the
 * residual r_k and the iterate x_k are kept; after convergence e_k = x* - x_k.
 * *count receives the dataset size. */
int pf_precond_collect(pf_ctx* ctx, int every, int max_pairs, int* count);
/* Synthetic pairs (K v, v) for `count` random smooth displacement fields v
 * (seeded multi-scale lattice noise) at the current moduli. */
int pf_precond_collect_random(pf_ctx* ctx, int count, uint64_t seed, int* total);
/* Adam on the collected pairs, loss min_{a,c} ||a t + c y - e||_K^2 / (e.r) for
 * each pair (K e = r), where t is the base step: r./D, or the multigrid V-cycle
 * V(r) once pf_mg_setup has been called; loss_first/loss_last are the first and
 * last steps'.  The pairs' densities are set on the device during training and
 * the caller's densities (and moduli) are restored afterwards.  Returns
 * PF_ERR_NUMERIC, the network left untrained, when no step gave a finite loss. */
int pf_precond_train(pf_ctx* ctx, int steps, double lr, uint64_t seed, double* loss_first, double* loss_last);
/* d = M(r) for a free-DOF residual with the current moduli. */
int pf_precond_apply(pf_ctx* ctx, const double* r_free, double* d_free);
/* Raw network pass on an input tensor x0 (H x W x 16, H = nx+1, W = ny+1,
 * or H x W x Dp x 16 with Dp = nz+1 on hex8; FP32 values rounded to BF16)
 * -> y (same shape, FP32), and the parameter
 * gradient of sum(y * dy) (grad in pf_precond_save order).  For checks
 * against a CPU restatement of the network. */
int pf_precond_forward_raw(pf_ctx* ctx, const float* x0, float* y);
/* The same pass with the output in the form the solver consumes: channels
 * 0 .. ndpn-1 of each node as a nodal FP64 vector y_nodal (nn x ndpn),
 * zero at fixed DOFs (the last layer writes it directly).  For checks of
 * that form against pf_precond_forward_raw. */
int pf_precond_forward_nodal(pf_ctx* ctx, const float* x0, double* y_nodal);
int pf_precond_backward_raw(pf_ctx* ctx, const float* dy, float* grad);
/* One convolution of the network, for checks against a CPU restatement (no
 * counterpart in the reference; needs no network).  Dp = 0: 3x3 taps on an
 * H x W grid; Dp > 0: 3x3x3 taps on H x W x Dp.  Tensors are channels last,
 * values rounded to BF16 on the way in.  mode 0: out (pixels x cout, FP32) =
 * conv(x (pixels x cin), w [tap][cout][cin]) with zero padding, no
 * activation; mode 1: out [tap][cout][cin] = sum_p dz[p][cout] x[p + tap][cin]
 * (the weight gradient; w_or_dz is dz, pixels x cout).  Channel counts 16,
 * 32 or 64 (the kernels the network launches). */
int pf_conv_raw(pf_ctx* ctx, int mode, int cin, int cout, int H, int W, int Dp, const float* x, const float* w_or_dz,
                float* out);

#ifdef __cplusplus
}
#endif
#endif
