/*
 * sg.h -- C ABI of the MI355X (gfx950) self-gravity multigrid library (libsg.so).
 *
 * Plain pointers, sizes and status codes only.  Every entry point returns SG_OK (0) or a
 * non-zero SG_ERR_* code; sg_last_error() gives the message of the last failure on the calling
 * thread.  The reference prints a message and stops on the same conditions
 * (e.g. mg_data.F90:187-190, interpolation.F90:75-76); its Fortran drop-in module (code_only_amd/
 * fortran/mg_gpu.F90) turns a non-zero status into that message plus `stop`.
 *
 * Uniform-grid arrays are dense n^3 FP64, C order [k][j][i] (x fastest) -- the memory order of the
 * reference's Fortran u(i,j,k) without its ghost layer.  Periodic ghosts are generated by index
 * wrap inside the kernels instead of being stored (fmg_boundary_phys_periodic.F90:71-104).
 *
 * Entry points named *_dev take device pointers; *_host take host pointers in the reference's
 * ghosted layout u(-1:n,-1:n,-1:n) and copy in and out.
 */
#ifndef SG_H
#define SG_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define SG_OK 0
#define SG_ERR_ARG 1            /* bad size / pointer / parameter                          */
#define SG_ERR_HIP 2            /* a HIP runtime call failed                               */
#define SG_ERR_NOT_CONVERGED 3  /* solve hit maxit (stats are still filled in)             */
#define SG_ERR_NONFINITE 4      /* residual became NaN/Inf                                 */

/* Convergence test of the outer defect-correction loop. */
#define SG_STOP_REFERENCE 0     /* mg.F90:91: Resmaxg / rhomax < tol (reference default 1e-2, maxit 10) */
#define SG_STOP_TRUE_RESIDUAL 1 /* post-update max|f - L phi| / max|f| < tol, computed in FP64        */

/* Arithmetic of the inner multigrid solve (outer residual and update are always FP64). */
#define SG_PREC_FP64 1          /* plain: every kernel FP64, the reference's cycle and bits          */
#define SG_PREC_MIXED 2         /* FP32 smoothing / restriction / prolongation inside FP64 refinement */

/* Coarse-grid solve of the SG_PREC_MIXED inner cycle on the uniform and batched tiers (the FP64
 * path always follows mg_lin; the AMR mixed path always solves its base grid exactly). */
#define SG_COARSE_EXACT 0       /* the cycle ends at the first level below the finest with <= 64^3 */
                                /* cells (<= 16^3 if that has <= 16^3), solved exactly by Hartley   */
                                /* transforms; grids of <= 16^3 cells keep the V-cycle              */
#define SG_COARSE_VCYCLE 1      /* mg_lin's own levels down to 1^3, as the reference (mg.F90:142-215) */

#define SG_HIST 64

typedef struct sg_params {
    double tol;       /* relative-residual target                                   */
    int maxit;        /* maximum outer iterations (mg_cycle's nmg, mg.F90:52)       */
    int stop_mode;    /* SG_STOP_*                                                  */
    int precision;    /* SG_PREC_*                                                  */
    int ncycle;       /* V-cycles per FMG level (mg.F90:123, 2)                     */
    int npre, npost;  /* smoothing sweeps (mg.F90:124-125, 2 and 2)                 */
    int use_graph;    /* replay the inner cycle as a hipGraph (AMR FP64: fmg_lin, in */
                      /* stretches between base solves, with the fused refresh on;  */
                      /* the staged refresh is always launched eagerly)             */
    int fused;        /* fused LDS-tiled kernels (same values); uniform FP64 with 0: */
                      /* one eager launch per reference loop nest                   */
    int coarse;       /* SG_PREC_MIXED only: SG_COARSE_* (default SG_COARSE_EXACT)  */
} sg_params;

typedef struct sg_stats {
    int iterations;   /* outer iterations done (calls of the inner solve)           */
    int status;       /* SG_OK or SG_ERR_NOT_CONVERGED / SG_ERR_NONFINITE           */
    double rel_linf;  /* max|f - L phi| / max|f| after the last update              */
    double rel_l2;    /* ||f - L phi||_2 / ||f||_2 after the last update            */
    double resmaxg;   /* Resmaxg of the last smoothing call (mg.F90:12)             */
    double ms;        /* device time of the solve, HIP events                       */
    double hist[SG_HIST]; /* rel_linf before each outer iteration                   */
    double rel_h2;    /* AMR: the reference's h^2-weighted L-inf residual ratio after the last
                         update, max_l(max|f - L phi| h_l^2) / max_l(max|f| h_l^2)
                         (fmg.F90:172, 1017-1039); uniform grids: equal to rel_linf           */
} sg_stats;

typedef struct sg_uniform sg_uniform; /* opaque context: one periodic n^3 grid hierarchy */

/* Library. */
const char *sg_last_error(void);
int sg_version(void);
void sg_default_params(sg_params *p);   /* reference values: tol 1e-2, maxit 10, SG_STOP_REFERENCE */

/* Uniform periodic grid.  Replaces mg_init(fmglev) + mg_data_init (mg.F90:525-528,
 * mg_data.F90:45-90): allocates every MG level n/2^l down to 1^3 once, on the device.
 * precisions: bitmask of SG_PREC_* arrays to allocate.  n must be a power of two >= 2. */
int sg_uniform_create(sg_uniform **ctx, int n, double h, int precisions);
int sg_uniform_destroy(sg_uniform *ctx);  /* replaces mg_finalize (mg.F90:532-536) */

/* Replaces mg_cycle(ju, jrho) (mg.F90:42-94): psi (in: initial guess, out: solution) and src
 * are dense n^3 FP64 device arrays.  Blocks until done. */
int sg_uniform_cycle_dev(sg_uniform *ctx, double *psi, const double *src,
                         const sg_params *p, sg_stats *st);

/* Same, host arrays in the reference's ghosted layout (n+2)^3, u(-1:n,-1:n,-1:n) with i fastest:
 * the module arrays MGdata(0)%Psi / %Src that mg_cycle works on (mg_data.F90:398-417). */
int sg_uniform_cycle_host(sg_uniform *ctx, double *psi_gh, const double *src_gh,
                          const sg_params *p, sg_stats *st);

/* g = -grad phi by centred differences (fmg_poisson.F90:29-31); g is 3 x n^3 (gx, gy, gz). */
int sg_uniform_gradient_dev(sg_uniform *ctx, const double *psi, double *g);

/* Adjoint of the periodic solve (no reference counterpart: the reference has no derivatives).
 * The forward map is src -> phi = L^+ P src (P removes the mean, as ZERO_AVERAGE_DENSITY does,
 * fmg_data_if.F90:53-78; L is the 7-point operator of mg_poisson.F90, symmetric on a periodic
 * grid), so d loss/d src = P L^+ P (d loss/d phi): sg_uniform_adjoint_dev solves that with the
 * same multigrid solver and parameters as the forward solve.  adj, grad: dense n^3 device arrays. */
int sg_uniform_adjoint_dev(sg_uniform *ctx, const double *adj, double *grad, const sg_params *p, sg_stats *st);

/* Sampled centred gradient out[3p + d] = (phi(c_p + e_d) - phi(c_p - e_d)) / (2h) at cells c_p
 * (linear index (k n + j) n + i) -- minus fmg_psi2g's g (fmg_poisson.F90:29-31) -- and its
 * transpose: out = sum_p sum_d w[3p + d] (e(c_p + e_d) - e(c_p - e_d)) / (2h), an n^3 field. */
int sg_uniform_gradient_sample_dev(sg_uniform *ctx, const double *psi, const int *cells, int npts, double *out);
int sg_uniform_gradient_sample_adjoint_dev(sg_uniform *ctx, const int *cells, const double *w, int npts, double *out);

/* Single operators on level-0-sized dense device arrays (parity tests).  prec = SG_PREC_FP64
 * operates on double*, SG_PREC_MIXED on float* (cast the pointers accordingly). */
int sg_uniform_relax_dev(sg_uniform *ctx, int prec, void *u, const void *rhs, int n, double h,
                         double *resmaxg);                                 /* mg_poisson.F90:32-79 */
int sg_uniform_resid_dev(sg_uniform *ctx, int prec, void *res, const void *u, const void *rhs,
                         int n, double h);                                 /* mg_poisson.F90:5-28  */
/* sg_uniform_relax_dev without a context and without allocating (no counterpart in the
 * reference; for callers that cannot allocate device memory: code under HIP graph capture, tight
 * serving loops).  One red-black sweep of mg_poisson_relax on the caller's dense n^3 arrays (n a
 * power of two <= 1024; double or float as prec), queued on `stream` (a hipStream_t, NULL for the
 * default stream), Resmaxg returned as sg_uniform_relax_dev returns it.  Its scratch (the Resmaxg
 * accumulator) is a fixed 64-double static device array per GPU, held until the process ends and
 * shared by every call on that GPU: calls that overlap on one GPU race.  Blocks until done. */
int sg_uniform_relax_noalloc(int prec, void *u, const void *rhs, int n, double h, double *resmaxg, void *stream);
int sg_uniform_restrict_dev(sg_uniform *ctx, int prec, void *uc, const void *uf, int nc);
                                                                           /* restriction.F90:127-151 */
int sg_uniform_interp_dev(sg_uniform *ctx, int prec, void *uf, const void *uc, int nf, int cubic);
                                                       /* interpolation.F90:40-247 via mg.F90:608-633 */

/* Measurement helper (no reference counterpart): average device time of one full smoothing sweep
 * (both colours) on the finest level's own arrays, timed with HIP events on the library's stream.  One
 * repetition is one launch of the mixed solve's sweep kernel, of as many sweeps as sg_uniform_tile_info
 * reports for level 0 (two passes of one colour each in FP64 and for grids of n <= 16). */
int sg_uniform_time_smoother(sg_uniform *ctx, int prec, int reps, double *ms_per_sweep);

/* Autotuner result (no reference counterpart): tile shape, sweeps per launch and source staging
 * chosen for MG level `level` of a context created with SG_PREC_MIXED (cfg -1 for levels solved
 * inside the single-workgroup coarse kernel) and the measured ms per fine-level visit of a V(2,2)
 * cycle (two sweeps ending with the residual restriction, two starting with the prolongated
 * correction) of every candidate (-1 where it does not fit or is not timed): 32 candidates, the LDS
 * tiles first, indexed tile * 4 + (sweeps - 1) * 2 + staged (cfg 0..4), then the twelve streaming
 * shapes at 20 + cfg - 5, timed with two sweeps per launch: column and planes, cfg 5 and 6 64x16x32, 7
 * 64x16x64, 9 32x32x64, 8, 10 and 11 32x16x16, 12 32x32x32, 13 16x16x16, 14 64x16x128, 15 32x16x64, 16
 * 16x8x8 (6, 8 and 11, second numbers of a shape, are not timed). */
int sg_uniform_tile_info(sg_uniform *ctx, int level, int *cfg, int *ns, int *fs, float *ms, int nms);
/* Override the autotuner's choice for fused-sweep level `level` (same meaning of cfg / ns / fs; values
 * do not depend on the choice).  A cfg fits the levels whose width is a multiple of its largest extent;
 * the numbers keep that meaning (a shape may be replaced by one that fits the same widths). */
int sg_uniform_set_tile(sg_uniform *ctx, int level, int cfg, int ns, int fs);

/* ---------------------------------------------------------------------------------------------
 * Block-structured AMR hierarchy (the fmg_poisson path, fmg.F90:63-233).
 *
 * Blocks hold 8^3 cells.  Block arrays passed in and out are dense [nblk][8][8][8] FP64 (i
 * fastest) -- the interior u(0:7,0:7,0:7) of the reference's per-block FMG arrays; g is
 * [nblk][3][8^3] (gx, gy, gz).  Blocks are numbered level by level, coarsest first; the tables
 * are those fmg_make_linklist builds (fmg_data_if.F90:298-413):
 *   level[b], ijk[3b..3b+2]   AMR level and position at that level in block units
 *   parent[b]                 parent block or -1 at level 0
 *   child[8b + o]             child in octant o = lri + 2 lrj + 4 lrk (Left 0, Right 1), or -1
 *   nbr[6b + 2d + lr]         neighbour across face (d = x, y, z; lr = 0 left, 1 right): the
 *                             same-level block, else the parent's same-level neighbour
 *                             (NeighborParentLevel), else -1 on the domain boundary
 * The hierarchy must be properly nested (every face has a neighbour at its own or its parent's
 * level, or lies on the domain boundary); the base level must be the full base_dims box.
 * ------------------------------------------------------------------------------------------- */
#define SG_BC_PERIODIC 0        /* fmg_boundary_phys_periodic.F90 (+ ZERO_AVERAGE_DENSITY)       */
#define SG_BC_SPHERE 1          /* fmg_boundary_phys_sphere.F90: multipole (l <= 3) boundary     */

typedef struct sg_amr sg_amr;   /* opaque context: one hierarchy with all its FMG-level arrays */

/* Replaces fmg_data_init + fmg_alloc_LoL + fmg_make_linklist (fmg_data.F90:110-154, 280-427,
 * fmg_data_if.F90:298-413): validates the tables and allocates every FMG-level array once. */
int sg_amr_create(sg_amr **ctx, int nblk, int nlev, const int *level, const int *ijk, const int *parent,
                  const int *child, const int *nbr, const int *base_dims, double h0, const double *x0, int bc);
int sg_amr_destroy(sg_amr *ctx);  /* replaces fmg_finalize / fmg_dealloc_LoL (fmg.F90:246-258) */

/* ZERO_AVERAGE_DENSITY (fmg_data_if.F90:53-78, vmg.F90:213-216): on by default for periodic
 * hierarchies, off for the sphere. */
int sg_amr_set_zero_average(sg_amr *ctx, int on);

/* Replaces fmg_poisson / fmg_cycle (fmg.F90:63-233): psi in = initial guess, out = potential on
 * every block (covered blocks: the restriction of their children); src = 4 pi G rho per block;
 * g (may be NULL) = -grad psi as fmg_psi2g forms it (fmg_poisson.F90:4-49).  SG_PREC_FP64 is the
 * reference's solve; SG_PREC_MIXED runs fmg_lin in FP32 (base grid solved exactly) inside the FP64
 * defect correction and stops on the true residual only.  SG_STOP_REFERENCE uses tol as fmg.F90's errormax (Resh2maxg / h2absmax(src), 1e-3 there) with
 * the stall test; SG_STOP_TRUE_RESIDUAL stops on max_leaf |src - L psi| / max_leaf |src| < tol. */
int sg_amr_solve_dev(sg_amr *ctx, double *psi, const double *src, double *g, const sg_params *p, sg_stats *st);
int sg_amr_solve_host(sg_amr *ctx, double *psi, const double *src, double *g, const sg_params *p, sg_stats *st);

/* Operator-level access for parity tests (no reference counterpart): whole FMG-level arrays
 * [nblk][(n+2)^3] of code U 0, RES 1, RHS 2, RHO 3, SRC 4, PSI 5 (fmg_data.F90:90), the
 * FmgLevel_fill0 state (fmg_data.F90:92), and single reference operations on that state. */
#define SG_AMR_OP_C2P 1          /* fmg_converge_c2p(L, a, cubic=flag)                        */
#define SG_AMR_OP_GHOSTFIX 2     /* fmg_ghostcell_fix(L, a, tricubic=flag&1); flag&2: one launch per level */
#define SG_AMR_OP_FILL0 3        /* fmg_boundary_fill0(L, a)                                  */
#define SG_AMR_OP_EXTRAP 4       /* fmg_boundary_extrap(L, a)                                 */
#define SG_AMR_OP_RELAX 5        /* fmg_poisson_relax(L, a, b, boundary_fill0=flag) -> Resh2maxg */
#define SG_AMR_OP_RESID 6        /* fmg_poisson_resid(L, a, b, c, boundary_fill0=flag)        */
#define SG_AMR_OP_RSTRCT 7       /* fmg_rstrct(L, a, b)                                       */
#define SG_AMR_OP_INTERP 8       /* fmg_interp(L, a, b, cubic=flag)                           */
#define SG_AMR_OP_ADDINT 9       /* fmg_addint(L, a, b, c)                                    */
#define SG_AMR_OP_VMG_FAS 10     /* vmg_fas(U, a)                                             */
#define SG_AMR_OP_FMG_LIN 11     /* fmg_lin -> Resh2maxg                                      */
#define SG_AMR_OP_SPHERE_BC 12   /* fmg_boundary_physical_grid(a, b), sphere module           */
#define SG_AMR_OP_REMOVE_MEAN 13 /* fmg_make_physvar's leaf-mean removal on code a            */
#define SG_AMR_OP_VMG_TAU 14     /* vmg_tau(AMR level flag, jtau a, ju b) incl. vmg_tau_crop, FMG level L */
int sg_amr_set_array(sg_amr *ctx, int fmglev, int code, const double *host);
int sg_amr_get_array(sg_amr *ctx, int fmglev, int code, double *host);
int sg_amr_get_fill0_level(sg_amr *ctx, int *v);
int sg_amr_set_fill0_level(sg_amr *ctx, int v);
int sg_amr_op(sg_amr *ctx, int op, int fmglev, int a, int b, int c, int flag, double *ret);
/* Context facts (no reference counterpart): info[0] bit L set when the mixed solve's refreshes at
 * FMG level L run fused (one launch evaluating the staged fill's values, instead of the staged
 * launches; the hierarchy must allow it), info[1] kernel nodes in the captured mixed outer
 * iteration (0 before the first graphed mixed solve), info[2] blocks, info[3] coarse-fine faces,
 * info[4] bit mask of the AMR levels whose vmg_ghostcell runs as one gather in the fused mode,
 * info[5] bit L set when fmg_ghostcell_fix of the base AMR level at FMG level L runs as one gather
 * in the fused mode (L = 1, 2). */
int sg_amr_info(sg_amr *ctx, int *info, int n);
/* The AMR autotuner's choice (no reference counterpart): threads per 8^3 block (64, 128 or 256) of
 * the FMG-level-0 kernel, which 0 = relaxation FP32, 1 = residual FP32, 2 = relaxation FP64,
 * 3 = residual FP64, and the timed ms per launch of the candidates 64, 128, 256 in ms[0..2] (0
 * where not yet timed: the FP32 ones are timed at the first mixed-precision solve). */
int sg_amr_tile_info(sg_amr *ctx, int which, int *choice, float *ms, int nms);
/* How the plain FP64 solve runs the base grid's mg_cycle (vmg_slvsml -> mg_cycle, vmg.F90:387-432):
 * chip = 1 (default) the fused kernels of the uniform tier (base grids of up to 16^3 cells: the whole
 * mg_cycle with its stopping test in one launch); chip = 0 the reference's steps on ghosted arrays in
 * one workgroup.  The mixed solve's exact base solve: six multi-workgroup transform passes, or one
 * workgroup.  Same values either way. */
int sg_amr_set_base_solver(sg_amr *ctx, int chip);
/* How the plain FP64 solve refreshes ghosts (no reference counterpart): fused = 1 (default) the mixed
 * solve's launch structure in FP64 -- one table-driven refresh per pass, halo-free colour passes,
 * merged VMG steps, fmg_lin replayed as graphs (use_graph); fused = 0 the reference's staged sequence
 * (c2p, fmg_ghostcell_fix level by level and direction by direction, reflux) before every colour pass,
 * launched eagerly.  Same values either way. */
int sg_amr_set_fp64_refresh(sg_amr *ctx, int fused);
/* Adjoint of the sphere-boundary AMR solve (no reference counterpart: the reference has no
 * derivatives).  The converged solve maps the source linearly to the potential: the source's
 * fmg_converge_c2p (fmg.F90:163-164), the multipole condition's mask and ghosts
 * (fmg_boundary_phys_sphere.F90:80-354), the composite operator -- same-level faces, covered
 * neighbours' restriction, the coarse-fine ghost of fmg_ghostcell.F90:443-495 and the reflux average of
 * fmg_reflux.F90:201-258 -- and the closing c2p (fmg.F90:205-216).  sg_amr_adjoint_dev applies the
 * transpose of that map: src_bar = (d psi / d src)^T psi_bar, both dense [nblk][8^3] device arrays.
 * The transposed composite operator is assembled on first use; A^T lambda = r is solved by FGMRES to
 * p->tol (relative 2-norm residual) within p->maxit iterations, preconditioned by forward solves
 * (p->precision, p->use_graph, p->fused) with zero physical ghosts.  st->iterations: FGMRES
 * iterations; st->rel_l2: its final relative residual; st->status SG_OK, or SG_ERR_NOT_CONVERGED
 * (returned as well) when p->maxit iterations end above p->tol: the preconditioner reaches tight
 * tolerances with one refinement level (two AMR levels), not yet where refined regions nest.  The
 * hierarchy must have the sphere boundary, zero averaging off, and single-pass coarse-fine ghost
 * sources (sg_amr_info's fused levels include FMG level 0); otherwise SG_ERR_ARG. */
int sg_amr_adjoint_dev(sg_amr *ctx, double *src_bar, const double *psi_bar, const sg_params *p, sg_stats *st);
/* y = A^T x for the homogeneous composite operator A at FMG level 0 that sg_amr_adjoint_dev
 * transposes (A x is minus the residual fmg_poisson_resid forms from u = x with zero source and
 * zero physical ghosts); x, y dense [nblk][8^3] device arrays, covered blocks' entries ignored / zero. */
int sg_amr_adjoint_apply(sg_amr *ctx, double *y, const double *x);
/* Benchmark hook (no reference counterpart): ms per full red-black sweep (both colour launches) of
 * the FMG-level-0 relaxation over the leaf blocks, as the solve runs it in precision prec, HIP
 * events on the library's stream, averaged over reps sweeps; the arrays' contents are not restored
 * (every solve starts from a cleared state). */
int sg_amr_time_smoother(sg_amr *ctx, int prec, int reps, double *ms_per_sweep);

/* ---------------------------------------------------------------------------------------------
 * Hydro block memory on the device.  The reference keeps each grid's hydro state in
 * BlockMem(gid)%u(i, j, k, m) (grid.F90:146-194): i, j, k in [-ng, 8 + ng), m in [0, ncomp), i
 * fastest.  Here those arrays sit in one device pool, grid slot s at pool + s * stride doubles, so
 * that the staging into the solver (fmg_make_physvar with fmg_prepare_interp's time slices,
 * fmg_data_if.F90:13-52, 169-211), the write-back (fmg_restore_u after fmg_psi2g, fmg.F90:205-215,
 * fmg_data_if.F90:275-294) and the gravity source step (source_g_all_level) run on the device
 * with no host copy.
 * ------------------------------------------------------------------------------------------- */
#define SG_AMR_MAX_LEVELS 16

typedef struct sg_blockmem {
    int ng;              /* ghost layers of the hydro arrays, 1..8 (N_GHOST_CELL = 2, config.h:135) */
    int ncomp;           /* components per cell (NM) */
    long long stride;    /* doubles from one pool slot to the next, >= ncomp (8 + 2 ng)^3 */
    int mrho, mvx, mvy, mvz, mp, mpsi, mgx, mgy, mgz;   /* component labels (config.h:63-71), distinct */
} sg_blockmem;

typedef struct sg_timeslice {
    int source;          /* time slice of rho (fmg_prepare_interp): 0 current, 1 predictor (SINGLE_STEP),
                            2 previous corrector, 3 interpolated in time */
    double step_max;     /* Step(LevelMax) */
    double step[SG_AMR_MAX_LEVELS], dstep[SG_AMR_MAX_LEVELS];   /* Step(l), Dstep(l); slice 3 only */
} sg_timeslice;

/* The pool slots of the context's blocks, host arrays of nblk entries in the context's block
 * order: slot_u[b] the grid's own arrays (GidList), slot_u1[b] its predictor-stage arrays
 * (U1list), slot_u2[b] its past arrays (U2list); slot_u1 and slot_u2 may be NULL where no time
 * slice or source step reads them.  Checked against pool_slots and kept on the device; the
 * layout is validated here too.  No reference counterpart: fmg_make_linklist's gid map
 * (fmg_data_if.F90:298-413) fixed once per hierarchy. */
int sg_amr_set_blockmem(sg_amr *ctx, const sg_blockmem *lay, long long pool_slots, const int *slot_u,
                        const int *slot_u1, const int *slot_u2);
/* Replaces fmg_poisson over BlockMem (fmg.F90:134-233 with fmg_prepare_data and fmg_restore_u):
 * psi <- u(MPSI) (time slice 0), src <- slice(u(MRHO)) * pi4g (pi4g = MP_Gconst * Pi4), the solve
 * of sg_amr_solve_dev (p, st as there), then u(MPSI) <- the solver's U over the FMG array's extent
 * (the interior and one ghost layer) and u(MGX), u(MGY), u(MGZ) <- g over the interior.  Returns
 * what the solve returns; the pool is written back for SG_OK, SG_ERR_NOT_CONVERGED and
 * SG_ERR_NONFINITE. */
int sg_amr_solve_blockmem_dev(sg_amr *ctx, double *pool, const sg_timeslice *ts, double pi4g, const sg_params *p,
                              sg_stats *st);
/* Replaces source_g_all_level (timestep.F90:528-578, SINGLE_STEP form) with the ideal-gas u2w /
 * w2u of eos_adiabatic.F90:226-266: on every grid, over all its cells u -> w; on the interior
 * momentum += g dt dv rho1 and energy += dt dv rho1 (v1 . g) (rho1, v1 from the predictor-stage
 * grid); then w -> u.  dtime[l] = Dtime(l) for the context's nlev levels, dv = the cell volume of
 * the level, gamma the ratio of specific heats (Gamma, 1.4 in eos_adiabatic.F90:9). */
int sg_amr_source_g_dev(sg_amr *ctx, double *pool, const double *dtime, double gamma);

/* The hydro steps around the solve on the same pool (ghost exchange, restriction, refluxing; the pool's
 * slot maps from sg_amr_set_blockmem, the hierarchy the context's).  Step modes as grid.F90:14-16:
 * 0 complete, 1 predictor, 2 corrector.
 * Replaces boundary_grid(level, mode) (grid_boundary.F90:65-105, SINGLE_STEP): at level >= 1 the
 * parent level's same-level exchange on the current, predictor and past arrays, then per
 * direction x, y, z the level's faces without a same-level neighbour filled from the parent
 * level (minmod-limited linear interpolation of the coarse grid's past / predictor / current
 * array for the predictor / corrector / complete step) and those with one copied from it;
 * ng ghost layers, ng even. */
int sg_amr_hydro_boundary_dev(sg_amr *ctx, double *pool, int level, int mode);
/* Replaces fg2cg_u(level) (fg2cg.F90:22-194): every grid of the level restricted into its
 * parent's octant (ideal-gas u2w with dv 1, the eight children summed, w2u with dv 8); the
 * nine-component layout only. */
int sg_amr_fg2cg_dev(sg_amr *ctx, double *pool, int level, double gamma);
/* Replaces fluxcorrection(level) (reflux.F90:114-388): at the faces where grids of level + 1 meet
 * level `level`, the coarse boundary layer corrected in conserved form by -/+ (restricted fine
 * accumulated flux - coarse boundary flux) dt ds, dt = dtime[level].  fb: device face-flux
 * buffers in the context's block order, fb[b][kind][face][m][64], kind 0 the boundary flux
 * (Fb%..._bnd), 1 the accumulated one (Fb%..._sum), faces 2 d + lr, the 8 x 8 face values in the
 * Fortran order of the reference's face arrays (x faces (j, k), y faces (i, k), z faces (i, j));
 * the nine-component layout only. */
int sg_amr_fluxcorrection_dev(sg_amr *ctx, double *pool, const double *fb, int level, const double *dtime,
                              double gamma);

/* ---------------------------------------------------------------------------------------------
 * Batched uniform tier: nprob independent periodic mg_cycle problems (mg.F90:42-94), problem q
 * an n[q]^3 grid of spacing h[q], solved together with one launch per multigrid step.  No
 * reference counterpart (the reference solves one grid per mg_cycle call); each problem follows
 * mg_cycle / mg_lin exactly.  n <= 1024: n = 2^a (a >= 1), or n = 3 * 2^a, whose levels halve to 3^3,
 * a level the reference's level count (mg_data.F90:57-62) does not describe; that coarsest level
 * is solved exactly (the zero-mean periodic solution) where mg_slvsml (mg.F90:540-546) sweeps.
 * ------------------------------------------------------------------------------------------- */
typedef struct sg_batch sg_batch;

/* precisions: SG_PREC_* bits to allocate level arrays for. */
int sg_batch_create(sg_batch **ctx, int nprob, const int *n, const double *h, int precisions);
int sg_batch_destroy(sg_batch *ctx);

/* psi[q], src[q]: device pointers to dense n[q]^3 FP64 arrays, i fastest (psi in = initial
 * guess, out = solution).  st[q]: per-problem statistics (ms is the whole batch's).  Stops each
 * problem on max|src - L psi| / max|src| < tol (SG_STOP_TRUE_RESIDUAL only); a converged problem
 * leaves the later launches.  The inner solve runs the fused kernels in either precision
 * (SG_PREC_MIXED: FP32, with tile shapes chosen on the first call); use_graph replays each outer
 * iteration as a hipGraph.  Returns SG_OK when every
 * problem converged, else the status of a problem that did not. */
int sg_batch_solve_dev(sg_batch *ctx, double *const *psi, const double *const *src, const sg_params *p,
                       sg_stats *st);

/* Chosen fused-sweep shape of fine level `level` (configuration index as sg_uniform_tile_info's,
 * sweeps per launch, source staged in LDS), tricubic tile x extent, and the timings (ms per
 * fine-level visit of a V(2,2) cycle, -1 = did not fit) of the candidates of
 * sg_uniform_tile_info. */
int sg_batch_tile_info(sg_batch *ctx, int level, int *cfg, int *ns, int *fs, int *cubic_fx, float *ms, int nms);
/* Number of levels of problem `prob` and its first level held by the coarse kernel. */
int sg_batch_levels(sg_batch *ctx, int prob, int *nlev, int *first_coarse);

#ifdef __cplusplus
}
#endif
#endif /* SG_H */
