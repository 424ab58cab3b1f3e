/*
 * cedarhip.h — C ABI of the MI355X (gfx950) Newton-transient engine.
 *
 * This library replaces, for transient and DC operating-point analysis, the
 * part of CedarSim's stack that sits below the circuit description:
 *
 *   - the DAECompiler-generated residual  f!(out, du, u, p, t)       and
 *     Jacobian jac!(J, du, u, p, gamma, t), J = dF/du + gamma*dF/d(du)
 *     (call sites: benchmarks/benchmark_common.jl:138,155; src/ac.jl:82-89),
 *   - Sundials IDA's BDF / Newton / dense LU loop behind
 *     tran!(prob) = solve(prob, IDA())            (src/sweeps.jl:450-465),
 *   - the DC operating point behind dc!(circ) and CedarDCOp
 *     (src/sweeps.jl:437-448, src/dcop.jl:24-200),
 *   - the serial sweep broadcast dc!./tran!. over a CircuitSweep
 *     (src/sweeps.jl:471-501), as one batched launch.
 *
 * Conventions (all entry points):
 *   - return int: CS_OK (0) on success, a negative CS_E_* code on failure;
 *     cs_last_error() returns a message for the last failure on that context;
 *   - host buffers are owned by the caller, device buffers by the library;
 *   - all arithmetic is IEEE FP64;
 *   - a context is bound to one GPU and one HIP stream and is not re-entrant.
 *
 * Unknown ordering ("natural order", used for u, du, residuals, CSR patterns
 * and waveforms):  node voltages 0..n_nodes-1, then one branch current per
 * voltage source, per inductor and per VCVS, in that order.  Node index -1 is
 * ground.  This is standard MNA: the reference's DAE has one current variable
 * per branch (src/simulate_ir.jl:112-140) which DAECompiler then eliminates for
 * current-defined branches; the solution in node voltages is the same DAE.
 *
 * Residual sign convention: row r of F is the sum of device currents leaving
 * node r plus d/dt of the charge stored at node r; a voltage-source row is
 * V(a) - V(b) - E(t); an inductor row is V(a) - V(b) - d/dt(L*I).
 */
#ifndef CEDARHIP_H
#define CEDARHIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define CEDARHIP_ABI_VERSION 3

/* ---- return codes ---------------------------------------------------- */
#define CS_OK            0
#define CS_E_INVALID    -1   /* bad argument / malformed netlist            */
#define CS_E_NODEVICE   -2   /* no HIP device, or HIP runtime unavailable   */
#define CS_E_HIP        -3   /* a HIP runtime call failed                   */
#define CS_E_SINGULAR   -4   /* structurally or numerically singular matrix */
#define CS_E_NOCONV     -5   /* Newton did not converge (DC op)             */
#define CS_E_DTMIN      -6   /* transient step fell below dt_min            */
#define CS_E_RANGE      -7   /* size beyond a documented limit              */
#define CS_E_OOM        -8   /* device allocation failed                    */
#define CS_E_MAXSTEPS   -9   /* transient hit max_steps before t_stop       */

/* ---- source waveforms (src/spectre_env.jl:43-69,144-176) -------------- */
#define CS_WAVE_DC     0  /* data: [v]                                        */
#define CS_WAVE_PULSE  1  /* data: [v1 v2 td tr tf pw period]  (Inf allowed)  */
#define CS_WAVE_PWL    2  /* data: [t0 y0 t1 y1 ...] (len = 2*points)         */
#define CS_WAVE_SIN    3  /* data: [vo va freq td theta phase ncycles]        */

/* ---- analysis modes (src/simulate_ir.jl:24 sim_mode) ------------------- */
#define CS_MODE_TRAN   0  /* sources follow their waveforms at time t        */
#define CS_MODE_DCOP   1  /* sources take their DC value; $time == 0         */

/* ---- transient initialisation ---------------------------------------- */
#define CS_INIT_DCOP   0  /* CedarDCOp: DC operating point at t_start        */
#define CS_INIT_UIC    1  /* u0 given; unknowns that carry charge are pinned
                             to u0 and the remaining (algebraic) unknowns are
                             solved for consistency                          */

/* ---- batched transient kernels (cs_tran_opts.batch_kernel) -------------- */
#define CS_BATCH_KERNEL_AUTO   0  /* LDS-resident kernel when every circuit fits */
#define CS_BATCH_KERNEL_LDS    1  /* LDS-resident kernel; an error if one does not fit */
#define CS_BATCH_KERNEL_GLOBAL 2  /* plan read from global memory (any size <= 512) */

/*
 * Flat netlist: the lowered form of a circuit after netlist import
 * (make_spectre_circuit, src/spectre.jl:1656-1697).  Node lists are int32
 * arrays with the per-device terminal count as stride.
 *
 *   res   2 terminals (a, b)         SimpleResistor  src/simpledevices.jl:49-77
 *   cap   2 terminals (a, b)         SimpleCapacitor src/simpledevices.jl:99-109
 *   ind   2 terminals (a, b)         SimpleInductor  src/simpledevices.jl:122-132
 *   vsrc  2 terminals (a, b) + wave  VoltageSource   src/simpledevices.jl:274-300
 *   isrc  2 terminals (a, b) + wave  CurrentSource   src/simpledevices.jl:315-339
 *   vccs  4 terminals (a, b, c, d)   vccs            src/simpledevices.jl:358-373
 *   vcvs  4 terminals (a, b, c, d)   vcvs            src/simpledevices.jl:341-356
 *   mos   4 terminals (d, g, s, b)   square-law MOSFET, a Verilog-A module
 *         (models/sqlaw.va in this package) loaded the way the reference loads
 *         any .hdl model (src/spectre.jl:1452-1469, src/ModelLoader.jl:20);
 *         type +1 = NMOS, -1 = PMOS.
 */
typedef struct cs_netlist {
    int32_t n_nodes;
    int32_t n_res;  const int32_t* res_nodes;  const double* res_r;
    int32_t n_cap;  const int32_t* cap_nodes;  const double* cap_c;
    int32_t n_ind;  const int32_t* ind_nodes;  const double* ind_l;
    int32_t n_vsrc; const int32_t* vsrc_nodes; const int32_t* vsrc_wave;
    int32_t n_isrc; const int32_t* isrc_nodes; const int32_t* isrc_wave;
    int32_t n_vccs; const int32_t* vccs_nodes; const double* vccs_gain;
    int32_t n_vcvs; const int32_t* vcvs_nodes; const double* vcvs_gain;
    int32_t n_mos;  const int32_t* mos_nodes;  const int32_t* mos_type;
    const double* mos_vth; const double* mos_kp; const double* mos_w; const double* mos_l;
    int32_t n_wave; const int32_t* wave_kind; const int32_t* wave_off; const int32_t* wave_len;
    const double* wave_dc;     /* per wave: DC-op value; NaN = value at t=0  */
    int32_t n_wave_data; const double* wave_data;
    double gmin;               /* SimSpec.gmin (src/simulate_ir.jl:16), 1e-12 */
    /* m-factor of every device (ParallelInstances, src/simulate_ir.jl:56-75):
     * the device's currents and charges enter the KCL of its terminal nets
     * multiplied by m, its own branch equation (V source, inductor, VCVS) is
     * unchanged.  One value per device in the order res, cap, ind, vsrc, isrc,
     * vccs, vcvs, mos; m >= 0 and finite.  NULL: every m is 1. */
    const double* dev_m;
    /* Verilog-A devices (make_spice_device, src/vasim.jl:663-875): the model
     * va_model[k] of the library's compiled models (cs_va_model_info), its
     * terminals va_nodes[va_node_ptr[k] .. va_node_ptr[k+1]) in the module's
     * port order, its flat parameters (card then instance parameters in
     * declaration order, NaN = not given so the model's default applies)
     * va_prm[va_prm_ptr[k] .. va_prm_ptr[k+1]).  Resistive contributions
     * only; they run on the plain path and the global-plan batched kernel. */
    int32_t n_va; const int32_t* va_model; const int32_t* va_node_ptr; const int32_t* va_nodes;
    const int32_t* va_prm_ptr; int32_t n_va_prm; const double* va_prm;
} cs_netlist;

/*
 * Parameter vector p (the DAE's "p", src/circuitodesystem.jl:66-97): every
 * numeric value of the netlist, so that sweep / Monte Carlo instances share a
 * topology and differ only in p.  Layout, in this order:
 *   res_r[n_res] cap_c[n_cap] ind_l[n_ind] vccs_gain[n_vccs] vcvs_gain[n_vcvs]
 *   mos_vth[n_mos] mos_kp[n_mos] mos_w[n_mos] mos_l[n_mos]
 *   wave_dc[n_wave] wave_data[n_wave_data] gmin va_prm[n_va_prm]
 */
typedef struct cs_param_layout {
    int32_t res_r, cap_c, ind_l, vccs_gain, vcvs_gain;
    int32_t mos_vth, mos_kp, mos_w, mos_l;
    int32_t wave_dc, wave_data, gmin, va_prm;
    int32_t n_params;
} cs_param_layout;

typedef struct cs_circuit_info {
    int32_t n;            /* unknowns                                   */
    int32_t n_nodes;
    int32_t nnz;          /* entries of the Jacobian pattern            */
    int32_t nnz_lu;       /* entries of L+U after fill                  */
    int32_t n_params;
    int32_t lu_levels;    /* levels of the entry-level LU schedule      */
    int32_t fwd_levels;   /* levels of the forward substitution         */
    int32_t bwd_levels;   /* levels of the backward substitution        */
    int64_t lu_updates;   /* multiply-subtract pairs per refactorization */
    int32_t n_singletons; /* pivots taken by singleton peeling          */
    int32_t n_probe;      /* recorded unknowns per output sample        */
} cs_circuit_info;

typedef struct cs_tran_opts {
    double  t_start, t_stop;
    double  reltol, abstol;      /* LTE weights: reltol*|u| + abstol          */
    double  dt_init;             /* first step after a (re)start; 0 = auto    */
    double  dt_min, dt_max;      /* 0 = auto                                  */
    double  newton_tol;          /* WRMS of the Newton update, tolerance units */
    double  dt_out;              /* output grid spacing                       */
    double  dc_abstol;           /* DC-op residual tolerance (CedarDCOp 1e-10)*/
    int32_t n_out;               /* output samples at t_start + k*dt_out      */
    int32_t max_order;           /* BDF order cap: 1 or 2                     */
    int32_t newton_maxit;
    int32_t init;                /* CS_INIT_DCOP or CS_INIT_UIC               */
    int64_t max_steps;
    int32_t batch_kernel;        /* batched: CS_BATCH_KERNEL_*                */
    int32_t record_steps;        /* keep the accepted-step sequence (adjoint) */
    int32_t jac_reuse;           /* 1: modified Newton, see below             */
    int32_t reserved;            /* 0                                         */
} cs_tran_opts;
/* jac_reuse = 1 factors the Jacobian once per step attempt, at the
 * predictor, and solves the later Newton iterations of the step with those
 * factors and the new residual (modified Newton, the Jacobian reuse of IDA's
 * Newton iteration, src/sweeps.jl:456).  cs_tran and cs_tran_sens run it on
 * both solvers (level-scheduled and supernodal); the batched kernels and the
 * adjoint refuse it (CS_E_INVALID).  The DC operating point and the pinned
 * initial system always refactor. */

typedef struct cs_tran_stats {
    int64_t steps;               /* accepted steps                     */
    int64_t rejected;            /* LTE or Newton rejections           */
    int64_t newton_iters;        /* Newton iterations = refactorizations */
    double  t_end;               /* time reached                       */
    int32_t retcode;             /* CS_OK or CS_E_*                    */
    int32_t pad;
    double  busy_s;              /* device time of the instance's run (LDS-
                                    resident batched kernel), else 0      */
} cs_tran_stats;

typedef struct cs_ctx cs_ctx;

/* ---- context ----------------------------------------------------------- */
int         cs_abi_version(void);
int         cs_device_count(int32_t* count);
int         cs_create(int32_t device, cs_ctx** out);
int         cs_destroy(cs_ctx* ctx);
const char* cs_last_error(const cs_ctx* ctx);

/* ---- host-only symbolic analysis (no device needed) -------------------- */
/* Runs the same analysis as cs_circuit_load and reports it: sizes in info;
 * when the arrays are non-NULL also the filled L+U pattern over permuted rows
 * (lu_rowptr[n+1], lu_col[nnz_lu], permuted column indices) and the pivot
 * order (rownat[k] / colnat[k]: natural row / unknown of pivot k).  Lets a
 * caller inspect the static pivoting and fill without a GPU. */
int cs_analyze(const cs_netlist* nl, cs_circuit_info* info, int32_t* lu_rowptr,
               int32_t* lu_col, int32_t* rownat, int32_t* colnat);
/* The packed batched launch's chunks for counts[c] instances of each of the
 * n_circ circuits (the same packing as cs_batch_create uses for a batch of
 * more than 7 instances per CU, which fills its chunks; host only; no
 * counterpart in the reference, a check of the batching): chunk k's segments
 * (circuit index, instance count) are seg_circ/seg_count[seg_ptr[k] ..
 * seg_ptr[k+1]-1], chunks in packing order (largest circuit first, before
 * the run queue's reordering); *lds_bytes the largest chunk's LDS.  A chunk
 * holds at most 8 instances in at most 4 segments within 81,664 bytes.
 * *n_chunks and *n_segs are always set; CS_E_RANGE when cap_chunks or
 * cap_segs is too small or a circuit does not fit a workgroup alone,
 * CS_E_INVALID when a circuit's plan does not fit the 16-bit LDS image. */
int cs_pack_plan(int32_t n_circ, const cs_netlist* const* nls, const int32_t* counts, int32_t cap_chunks,
                 int32_t cap_segs, int32_t* n_chunks, int32_t* n_segs, int32_t* seg_ptr, int32_t* seg_circ,
                 int32_t* seg_count, int64_t* lds_bytes);

/* ---- large circuits: supernodal multifrontal solver -------------------- */
/* Circuits from CS_SUPERNODAL_MIN_N unknowns up (power grids, meshes) are
 * factored by a supernodal multifrontal LU: nested-dissection order of the
 * matched matrix, dense fronts on the device, level by level.  They run on
 * the plain entry points (cs_tran, cs_dcop, cs_residual, cs_jacobian,
 * cs_lu_refactor, cs_lu_solve), not in batches.  No counterpart in the
 * reference, which factors densely in IDA (src/sweeps.jl:456). */
#define CS_SOLVER_AUTO       0   /* supernodal from CS_SUPERNODAL_MIN_N unknowns */
#define CS_SOLVER_LEVEL      1   /* entry-level LU schedule (batched kernels)    */
#define CS_SOLVER_SUPERNODAL 2
#define CS_SUPERNODAL_MIN_N  8192

typedef struct cs_big_info {
    int32_t n;            /* unknowns                                      */
    int32_t n_super;      /* supernodes (fronts)                           */
    int32_t n_levels;     /* levels of the assembly tree                   */
    int32_t max_front;    /* largest front order m                         */
    int32_t max_pivots;   /* most pivots in one front                      */
    int32_t n_hub;        /* high-degree unknowns ordered last             */
    int64_t pool;         /* doubles of front storage                      */
    int64_t nnz_factor;   /* entries of L+U held in the fronts             */
    double  flops;        /* flops of one factorization                    */
} cs_big_info;

/* Symbolic analysis of the supernodal solver without a GPU: sizes, and the
 * pivot order (rownat[k] / colnat[k], may be null). */
int cs_big_analyze(const cs_netlist* nl, cs_big_info* info, int32_t* rownat, int32_t* colnat);

/* cs_circuit_load with an explicit solver choice (CS_SOLVER_*). */
int cs_circuit_load_solver(cs_ctx* ctx, const cs_netlist* nl, int32_t solver, int32_t* cid);

/* Sizes of a loaded supernodal circuit (CS_E_INVALID for other circuits). */
int cs_big_info_get(cs_ctx* ctx, int32_t cid, cs_big_info* info);

/* Device time of the last cs_lu_refactor and cs_lu_solve of a supernodal
 * circuit, milliseconds. */
int cs_big_times(cs_ctx* ctx, int32_t cid, double* factor_ms, double* solve_ms);
/* Per-launch timing of one factorization of the current Jacobian values
 * and one forward/backward solve, as plain stream launches, each between
 * two HIP events on the launch stream: for launch q, kinds[q] (CS_MFK_*),
 * levels[q] (assembly-tree level) and ms[q]; *count = number of launches
 * (at most cap are stored).  A diagnostic of the supernodal path with no
 * counterpart in the reference (its KLU/UMFPACK calls are host library
 * calls); it leaves the circuit's state as a factorization would. */
#define CS_MFK_SMALL32 0   /* fronts up to 32 rows, gathered and factored in one kernel */
#define CS_MFK_SMALL64 1   /* fronts of 33..64 rows                                     */
#define CS_MFK_SMALL96 2   /* fronts of 65..96 rows                                     */
#define CS_MFK_GATHER  3   /* contribution-block gather of the large fronts            */
#define CS_MFK_ORIG    4   /* Jacobian entries into the large fronts                   */
#define CS_MFK_DIAG    5   /* LU of a panel's diagonal block                           */
#define CS_MFK_TRSM    6   /* a panel's row and column triangular solves               */
#define CS_MFK_GEMM    7   /* a panel's trailing update                                */
#define CS_MFK_FRONT   8   /* one workgroup per large front (the fused form)          */
#define CS_MFK_FWD     9   /* forward substitution of one level                        */
#define CS_MFK_BWD     10  /* backward substitution of one level                       */
#define CS_MFK_PANEL   11  /* one panel step in one launch (diagonal block, solves, update) */
#define CS_MFK_FLUSH   12  /* factored panels of a level back from the workspace          */
#define CS_MFK_HEAD    13  /* a level's small fronts, gather tiles and the last level's flush */
int cs_big_profile(cs_ctx* ctx, int32_t cid, int32_t* kinds, int32_t* levels, float* ms, int32_t cap,
                   int32_t* count);

/* ---- circuits (host symbolic analysis, done once per topology) --------- */
/* Lowers the netlist, builds the Jacobian pattern, the slot maps for
 * deterministic assembly, the static pivot order and the LU / substitution
 * level schedules, and uploads them.  Replaces DAECompiler's per-topology
 * compile (src/circuitodesystem.jl:147-164). */
int cs_circuit_load(cs_ctx* ctx, const cs_netlist* nl, int32_t* cid);
int cs_circuit_info_get(cs_ctx* ctx, int32_t cid, cs_circuit_info* info);
int cs_circuit_layout(cs_ctx* ctx, int32_t cid, cs_param_layout* layout);
int cs_circuit_default_params(cs_ctx* ctx, int32_t cid, double* p);
/* CSR pattern of J in the natural order: rowptr[n+1], colind[nnz]
 * (the reference's jac_prototype would be this sparsity). */
int cs_circuit_pattern(cs_ctx* ctx, int32_t cid, int32_t* rowptr, int32_t* colind);
/* Unknowns recorded in waveforms (default: all n). */
int cs_circuit_set_probes(cs_ctx* ctx, int32_t cid, int32_t n_probe, const int32_t* idx);

/* ---- DAE interface, mirrors f!/jac! (benchmarks/benchmark_common.jl:138,155)
 * F(du,u,p,t) = i(u,p,t) + dQ/du(u,p) * du;  J = di/du + gamma * dQ/du.
 * out[n]; vals[nnz] in the CSR order of cs_circuit_pattern.               */
int cs_residual(cs_ctx* ctx, int32_t cid, double* out, const double* du,
                const double* u, const double* p, double t, int32_t mode);
int cs_jacobian(cs_ctx* ctx, int32_t cid, double* vals, const double* du,
                const double* u, const double* p, double gamma, double t,
                int32_t mode);
/* Sparse LU on the fixed symbolic pattern (replaces IDA's dense LU). */
int cs_lu_refactor(cs_ctx* ctx, int32_t cid, const double* vals);
int cs_lu_solve(cs_ctx* ctx, int32_t cid, double* x);            /* J x = b   */
int cs_lu_solve_transpose(cs_ctx* ctx, int32_t cid, double* x);  /* J^T x = b */

/* ---- analyses ---------------------------------------------------------- */
void cs_tran_opts_default(cs_tran_opts* o);
/* dc!(circ): Newton on F(0,u,p,0)=0 in DC mode (src/dcop.jl:53-155). */
int cs_dcop(cs_ctx* ctx, int32_t cid, const double* p, const cs_tran_opts* o,
            double* u_out, cs_tran_stats* st);
/* tran!(circ, tspan).  By default a circuit that fits runs its whole transient
 * in one launch of the LDS-resident kernel, as a batch of one; circuits that
 * do not fit (more than 256 unknowns or 512 devices, Verilog-A devices, 64 KiB
 * of LDS), supernodal ones, runs with more than 64 MiB of samples or no memory
 * for them, and modified Newton (jac_reuse) on a circuit with nonlinear devices
 * take the plain path: the host runs the BDF step control
 * and every Newton iteration is one launch of a captured hipGraph (device
 * eval -> assembly -> LU refactor -> solve -> norm).  Both follow the same
 * rules; results agree to rounding.  o->batch_kernel = CS_BATCH_KERNEL_LDS
 * asks for the first (refused for supernodal circuits, circuits that do not
 * fit, and jac_reuse), CS_BATCH_KERNEL_GLOBAL for the plain path.
 * wave: n_out x n_probe samples; u_final: n.  u0 may be NULL for INIT_DCOP.
 * cs_dcop takes the same kernel code where the circuit fits, and the plain
 * path with CS_BATCH_KERNEL_GLOBAL. */
int cs_tran(cs_ctx* ctx, int32_t cid, const double* p, const double* u0,
            const cs_tran_opts* o, double* wave, double* u_final,
            cs_tran_stats* st);

/* ---- batched transient (sweep / Monte Carlo in one launch) ------------- *
 * Instances may use different circuits (uneven sizes).  params holds each
 * instance's parameter vector back to back; u0 (may be NULL) each instance's
 * initial state back to back.  cs_batch_create uploads everything; run
 * launches one persistent kernel that walks a work queue of chunks (up to
 * four runs of same-circuit instances per workgroup, each run beside its
 * circuit's plan image in LDS, one wavefront per instance), every instance
 * doing its whole transient on the device; results downloads: wave holds
 * each instance's n_out x n_probe samples back to back (instance order),
 * u_final each instance's n unknowns, st one record per instance.          */
int cs_batch_create(cs_ctx* ctx, int32_t n_inst, const int32_t* inst_cid,
                    const double* params, const double* u0,
                    const cs_tran_opts* o, int32_t* bid);
int cs_batch_run(cs_ctx* ctx, int32_t bid, double* kernel_ms);
int cs_batch_results(cs_ctx* ctx, int32_t bid, double* wave, double* u_final,
                     cs_tran_stats* st);
int cs_batch_destroy(cs_ctx* ctx, int32_t bid);
/* Roofline bookkeeping of the last run: algorithmic bytes moved by the
 * executed Newton iterations (device eval + assembly + LU + solves). */
int cs_batch_traffic(cs_ctx* ctx, int32_t bid, double* alg_bytes,
                     double* alg_flops);
/* Which kernel a batch runs (CS_BATCH_KERNEL_LDS or _GLOBAL) and how many
 * launches one run makes. */
int cs_batch_kernel(cs_ctx* ctx, int32_t bid, int32_t* kernel, int32_t* n_launches);

/* One Newton iteration of the batched kernels' instance code, recorded: the
 * circuit's plan image and one instance in LDS exactly as the batched
 * transient kernel holds them (same device code: device evaluation,
 * assembly with the wavefront-summed long rows, the level-scheduled LU with
 * the forward substitution folded in, the backward substitution).  Inputs:
 * p, the state u (natural order), the charge terms qx (natural rows, the
 * sum_j a_j Q_j of the step) and the BDF coefficient a0 at time t in mode.
 * Outputs (any may be NULL): jac[nnz] the assembled J = dI/du + a0 dQ/du on
 * the natural CSR pattern of cs_circuit_pattern; res[n] the residual
 * I + a0 Q + qx (natural rows); lu[nnz_lu] the factors in the F order of
 * cs_analyze (L below the diagonal, unit diagonal implied; U on and above);
 * dx[n] the Newton update solving J dx = -res.  nr = rows per lane (1, 2 or
 * 4; 0 = the batch kernel's own choice).  A diagnostic with no counterpart
 * in the reference (whose f!/jac! are cs_residual / cs_jacobian). */
int cs_lds_probe(cs_ctx* ctx, int32_t cid, int32_t nr, const double* p, const double* u,
                 const double* qx, double a0, double t, int32_t mode, double* jac, double* res,
                 double* lu, double* dx);

/* ---- Verilog-A device models compiled into the library ----------------- *
 * vagen translates each model's Verilog-A source at build time (the role of
 * load_VA_model / make_spice_device, src/ModelLoader.jl:20,
 * src/vasim.jl:663-875); a circuit's Verilog-A devices name a model by its
 * index.  Host-only: no device is needed.
 * cs_va_model_count: the number of models.
 * cs_va_model_info: name (NUL-terminated, at most cap bytes), terminals,
 * flat parameters, whether it contributes charges (ddt).
 * cs_va_model_param: name of flat parameter k of model id. */
int cs_va_model_count(void);
int cs_va_model_info(int32_t id, char* name, int32_t cap, int32_t* n_ports, int32_t* n_params,
                     int32_t* has_charge);
int cs_va_model_param(int32_t id, int32_t k, char* name, int32_t cap);

/* ---- compact-model device evaluation: BSIM-CMG 107 -------------------- *
 * The model code is generated from the model's Verilog-A source at build
 * time (the reference compiles the same file through make_spice_device,
 * src/vasim.jl:663-875).  One lane per instance, FP64, partial derivatives
 * by forward-mode dual numbers.  Per instance: the internal nodes di, si
 * are solved for resistive KCL, then the six-node stamps are condensed onto
 * the terminals d, g, s, e.  out[40 per instance] = I[4], Q[4], G[16],
 * C[16] (row-major, row = terminal equation, column = terminal voltage).
 * cs_bsimcmg_available: 1 when the library was built with the model.
 * cs_bsimcmg_param: set a model-card or instance-template parameter by its
 * Verilog-A name (applies to later evaluations; CS_E_INVALID if unknown).
 * cs_bsimcmg_eval: v is [n][4] terminal voltages; temp_c in Celsius;
 * iters[n] (may be NULL) the internal-node Newton iterations or -1;
 * kernel_ms the device time of the evaluation alone (inputs resident). */
int cs_bsimcmg_available(void);
int cs_bsimcmg_param(cs_ctx* ctx, const char* name, double value);
int cs_bsimcmg_eval(cs_ctx* ctx, int64_t n, const double* L, const double* nfin,
                    const double* v, double temp_c, double* out, int32_t* iters,
                    double* kernel_ms);
/* cs_bsimcmg_eval without any device allocation.  No counterpart in the
 * reference: for callers that cannot allocate device memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc).  L,
 * nfin [n], v [n][4], out [n][40] and iters [n] (may be NULL) are DEVICE
 * pointers the caller owns; the model card, the instance template and the
 * per-lane bias-independent store live in one static device buffer of the
 * library (per GPU, for the life of the process: 16,384 lanes x the model's
 * bias-independent values, about 39 MB for BSIM-CMG 107).  The kernel walks
 * the instances grid-stride, so n is bounded only by 2^31-1 (CS_E_RANGE
 * beyond).  Returns when out is written.  Calls that overlap on one GPU
 * share that buffer and race. */
int cs_bsimcmg_eval_noalloc(cs_ctx* ctx, int64_t n, const double* L, const double* nfin,
                            const double* v, double temp_c, double* out, int32_t* iters);

/* ODEForwardSensitivityProblem + extract_local_sensitivities
 * (test/sensitivity.jl:13-66): cs_tran together with the
 * forward sensitivities d(probed unknown)/d p of n_sp parameters, sp_idx[j]
 * an index into the parameter vector: res_r, cap_c, ind_l, vccs_gain,
 * vcvs_gain, mos_vth/kp/w/l, and wave_dc of a source (its DC value, which
 * is also its transient value for a DC source); any other index is refused
 * (CS_E_INVALID).  They are the sensitivities of the discrete solution on
 * its own step sequence (staggered direct method): at every accepted step
 * J(u_m) s_m = -(dI/dp + a0 dQ/dp + a1 dQ_{m-1} + a2 dQ_{m-2}), dQ the total
 * derivative of the charges and J refactored at u_m; the initial point's
 * follow its construction (charge rows fixed at u0 under UIC; with the DC
 * operating point, the DC point's sensitivity pins them).  wave as cs_tran
 * (required); sens: n_out x n_sp x n_probe, interpolated like wave.
 * Circuits of up to 64 unknowns run in one launch; larger ones, jac_reuse,
 * Verilog-A devices, more than 512 MiB of samples (or no memory for them) and
 * CS_BATCH_KERNEL_GLOBAL take the plain path.
 * Circuits on the supernodal solver are refused. */
int cs_tran_sens(cs_ctx* ctx, int32_t cid, const double* p, const double* u0, const cs_tran_opts* o,
                 int32_t n_sp, const int32_t* sp_idx, double* wave, double* sens, double* u_final,
                 cs_tran_stats* st);

/* ---- small-signal AC and noise (src/ac.jl) ------------------------------ *
 * ac!(circ) + freqresp(ac, sym, ws) (src/ac.jl:75-102,173-180,231-240): the
 * circuit linearised at the DC point u_dc (natural order, e.g. cs_dcop's
 * answer), G = dF/du in DC mode and C = dQ/du on the pattern the transient
 * factors; for each angular frequency omega[f] (rad/s) solves
 * (G + j omega C) x = b, b the sources' AC excitation: src_ac[s] is the AC
 * magnitude of source s (voltage sources, then current sources, as in
 * cs_netlist; the reference uses |ac|, phase 0, src/simpledevices.jl:291,332).
 * out[f][i] = x at natural unknown obs[i], complex (re, im) interleaved:
 * out has 2 * n_freq * n_obs doubles.  Circuits on the supernodal solver
 * are refused (CS_E_INVALID). */
int cs_ac(cs_ctx* ctx, int32_t cid, const double* p, const double* u_dc, const double* src_ac,
          int32_t n_freq, const double* omega, int32_t n_obs, const int32_t* obs, double* out);
/* noise!(circ) + PSD(noise, sym, ws) (src/ac.jl:139-165,267-284): the
 * power spectral density of natural unknown obs at each omega[f] from the
 * thermal noise of every resistor, 4kT/R (T = temp_c + 273.15 K, times its
 * m-factor; src/simpledevices.jl:71-76), a current in parallel with it:
 * psd[f] = sum_i pwr_i |H_i(j omega_f)|^2, H_i the transfer from source i to
 * obs (one transposed solve per frequency). */
int cs_noise(cs_ctx* ctx, int32_t cid, const double* p, const double* u_dc, double temp_c, int32_t n_freq,
             const double* omega, int32_t obs, double* psd);

/* ---- batched adjoint sensitivities ------------------------------------- *
 * Replaces forward sensitivity through DAECompiler's paramjac
 * (ODEForwardSensitivityProblem, test/sensitivity.jl:29-41) for the energy
 * objective: E = energy delivered by voltage source `vsrc` over the run
 * (trapezoid on the accepted points), gradient with respect to every MOSFET
 * width.  Discrete adjoint of the BDF scheme on the recorded step sequence,
 * checkpoints every ckpt_every accepted steps, recomputation in between.
 * Requires o->init == CS_INIT_UIC.  Outputs: energy[n_inst]; grad: each
 * instance's n_mos entries back to back; n_steps[n_inst]; optional step log
 * t_log / npts_log ([n_inst][max_steps], may be NULL) for frozen-step replays
 * (npts_log[m] = points of the current segment before step m).             */
typedef struct cs_adjoint_opts {
    int32_t vsrc;           /* index of the voltage source of the objective */
    int32_t ckpt_every;     /* accepted steps between checkpoints (64)      */
    int64_t max_steps;      /* step-log capacity per instance               */
} cs_adjoint_opts;

int cs_adjoint_batch(cs_ctx* ctx, int32_t n_inst, const int32_t* inst_cid,
                     const double* params, const double* u0,
                     const cs_tran_opts* o, const cs_adjoint_opts* ao,
                     double* energy, double* grad, int64_t* n_steps,
                     double* t_log, int32_t* npts_log, cs_tran_stats* st,
                     double* kernel_ms);

#ifdef __cplusplus
}
#endif
#endif /* CEDARHIP_H */
