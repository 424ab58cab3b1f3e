// kernels.h — launch interface between the C-ABI layer (api.hip) and the
// kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/cedarhip.h"
#include "dplan.h"

namespace cedar {

// Per-iteration parameters of the single-instance path, written by the host.
struct StepDev {
    double a0, t, rtol, atol, tol;
    int32_t mode;   // CS_MODE_*
    int32_t kind;   // STEP_TRAN, STEP_DC, STEP_UIC
    int32_t pad[2];
};
enum : int32_t { STEP_TRAN = 0, STEP_DC = 1, STEP_UIC = 2 };

// norm[] slots written by the single-instance kernels
enum : int32_t { NRM_WRMS = 0, NRM_MAXD = 1, NRM_RES = 2, NRM_DONE = 3, NRM_SLOTS = 4 };

// Device workspace of one circuit instance (single-instance path).
struct InstDev {
    double *p, *linbuf, *Glin, *Clin, *F, *inv, *u, *x, *qx, *st, *u0, *norm;
    StepDev* sp;
    bool has_va;             // the circuit has Verilog-A devices
};

struct BatchArgs {
    const DPlan* plans;
    const int32_t* inst_cid;
    const int64_t* p_off;
    const double* params;
    const int64_t* u_off;
    const double* u0;        // may be null (DC-op init)
    const int64_t* w_off;
    double* wave;            // may be null
    double* u_final;
    cs_tran_stats* stats;
    const int32_t* order;    // work-queue order of instances
    int32_t* queue;          // work-queue head (zeroed before launch)
    double *glin, *clin, *linbuf;   // per-workgroup workspace
    int32_t n_inst, nnz_max, n_max, stamp_max, lin_max, n_probe_max;
    cs_tran_opts o;
};

// Small-signal AC / noise (ac.hip): one workgroup per frequency.
struct AcArgs {
    const DPlan* P;
    const double* G;          // [nnz] dF/du at the DC point on the F pattern
    const double* Cl;         // [nnz] dQ/du on the F pattern
    const double* omega;      // [n_freq] angular frequencies
    double* ws;               // per workgroup: 2 nnz + 4 n doubles
    size_t ws_stride;         // doubles per workgroup slice
    int32_t n_freq;
    int32_t transposed;       // 0: AC solve, 1: transposed (noise) solve
    // AC: right-hand side by pivot row, observed unknowns by pivot column
    const double* rhs;
    int32_t n_obs;
    const int32_t* obs_piv;
    double* out;              // [n_freq][n_obs] complex, interleaved
    // noise: unit right-hand side at pivot column obs_col; per source the
    // pivot rows of its two nodes (-1: ground), power and frequency exponent
    int32_t obs_col, n_noise;
    const int32_t* nz_rows;
    const double* nz_pwr;
    const double* nz_exp;
    double* psd;              // [n_freq]
};
// LDS for one frequency's factors, reciprocals, solution and substitution
// schedules; lds = 0 keeps the first three in the workspace
size_t ac_lds(int32_t n, int32_t nnz);
hipError_t launch_ac(const AcArgs& a, int nblocks, int nt, size_t lds, hipStream_t s);

// Forward parameter sensitivities of the plain-path transient (sens.hip):
// one parameter's stamps.  Indices are natural (-1: ground).
enum : int32_t {
    SP_R = 0,      // resistor: i0, i1 nodes, val = R, m
    SP_C = 1,      // capacitor: i0, i1 nodes, m
    SP_IND = 2,    // inductor: i0 its branch row
    SP_VCCS = 3,   // VCCS: i0, i1 output nodes, i2, i3 control nodes, m
    SP_VCVS = 4,   // VCVS: i0 branch row, i2, i3 control nodes
    SP_VTH = 5, SP_KP = 6, SP_MW = 7, SP_ML = 8,   // MOSFET dev: i0 d, i1 g, i2 s, i3 type, m
    SP_VSRC = 9,   // DC value of a voltage source: i0 branch row; dev = 1 when its transient value is that DC value
    SP_ISRC = 10,  // DC value of a current source: i0, i1 nodes, m; dev as above
};
struct SensParam {
    int32_t kind, i0, i1, i2, i3, dev, pad[2];
    double m, val;
};
struct SensArgs {
    const DPlan* P;
    const double* p;          // parameters
    const double* u;          // the state (natural)
    const double* F;          // LU of the Jacobian at u (refactored by the caller)
    const double* inv;
    const double* Clin;       // dQ/du on the F pattern
    const int32_t* prow;      // natural row -> pivot row
    const SensParam* sp;
    int32_t n_sp;
    int32_t mode;             // CS_MODE_* of the source values
    int32_t pinned;           // rows that carry charge are pinned (initial point)
    int32_t pad;
    double a0, a1, a2;        // BDF coefficients (0 at the initial point)
    const double* pin_s;      // [n_sp][n] sensitivity of the pin values, or null (0)
    const double* dq1;        // [n_sp][n] charge sensitivities one and two steps back, or null
    const double* dq2;
    double* x;                // [n_sp][n] workspace
    double* s;                // [n_sp][n] sensitivities (natural)
    double* dq0;              // [n_sp][n] C s + dQ/dp (natural rows)
};
hipError_t launch_sens(const SensArgs& a, hipStream_t s);

// A whole sensitivity run in one launch (k_tran_sens): one wavefront per
// parameter.
struct SensRunArgs {
    const DPlan* P;
    const double* p;
    const double* u0;         // may be null (DC-op init)
    const int32_t* prow;      // natural row -> pivot row
    const SensParam* sp;
    double* ws;               // per parameter: ws_stride doubles (linear slots, G, C)
    size_t ws_stride;
    double* wave;             // [n_out][n_probe], or null: no output samples
    double* sens;             // [n_out][n_sp][n_probe]
    double* u_final;
    cs_tran_stats* stats;
    int32_t n_sp, n, nnz, n_lin, n_stamp, n_probe;
    cs_tran_opts o;
};
constexpr int kSensMaxN = 64;   // one unknown per lane
size_t tran_sens_lds(int32_t n, int32_t nnz, int32_t n_stamp);
hipError_t launch_tran_sens(const SensRunArgs& a, hipStream_t s);

struct CPlan;

// Arguments of the LDS-resident kernels: the packed launch of a batch, a single
// circuit's run or DC point (tran_lds.hip), an adjoint class (adj_lds.hip).
struct LdsArgs {
    const CPlan* cplans;
    const DPlan* plans;
    const int32_t* inst_cid;
    const int64_t* p_off;
    const double* params;
    const int64_t* u_off;
    const double* u0;        // may be null (DC-op init)
    const int64_t* w_off;
    double* wave;            // may be null
    double* u_final;
    cs_tran_stats* stats;
    const int32_t* order;    // the launch's instances, in its order
    int32_t* queue;          // its queue's head (zeroed before launch)
    int32_t n_inst;          // its instances
    int32_t dbl_max;         // LDS doubles before the plan image (adjoint)
    cs_tran_opts o;
    // packed launch: a chunk is up to kPackSegs segments, each a run of
    // instances of one circuit, one wavefront each.  Segment j is segs[2j] =
    // (circuit, first index into order, count, rows per lane) and segs[2j+1] =
    // (word offset of its plan image in LDS, double offset of its first
    // wavefront's region, doubles per region, its first wavefront); chunk c
    // holds segments chunk_seg[c] .. chunk_seg[c+1]-1.
    const int4* segs;
    const int32_t* chunk_seg;
    int32_t n_chunks;
    int32_t pad_;
};

// Batched discrete adjoint on the LDS-resident kernel (adj_lds.hip): one
// launch per size class for the recording forward pass, one for the reverse.
struct AdjLdsArgs {
    LdsArgs f;              // the class's transient arguments (queue: forward)
    double* t_log;          // [n_inst][cap]
    int32_t* npts_log;      // [n_inst][cap]
    int64_t cap;
    double* ckpt;           // [n_inst][ckcap][3][ck_n] pivot-order states
    int64_t ckcap;
    int32_t K;              // checkpoint interval (accepted steps)
    int32_t ck_n;           // doubles per checkpointed state (max unknowns)
    int64_t* n_steps;       // [n_inst]
    double* energy;         // [n_inst]
    double* grad;           // per instance at g_off, n_mos entries
    const int64_t* g_off;
    const int32_t* obj;     // per circuit: a, b, j as pivot columns (0xFFFF ground)
    double* seg;            // per workgroup: K * ck_n recomputed states
    int32_t* queue2;        // the class's reverse queue head
    int32_t pad;
};

// Batched BSIM-CMG evaluation (bsimcmg.hip).
struct BsimArgs {
    const void* card;       // the model card (generated Card struct), device
    const void* inst;       // instance-parameter template (generated Inst), device
    int64_t n;
    const double* L;        // [n] gate length
    const double* nfin;     // [n] fins per finger
    const double* v;        // [n][4] terminal voltages d, g, s, e
    double temp;            // kelvin
    double* out;            // [n][40]: I[4], Q[4], G[16], C[16]
    int32_t* iters;         // [n] internal-node Newton iterations (may be null)
    double* store;          // bias-independent values: [bsim_setup_size()][stride], one column per lane
    int64_t stride;         // = lanes of the launch
};

constexpr int kSingleThreads = 256;
constexpr int kBatchThreads = 64;

// single-instance kernels (one workgroup each)
void launch_lin_setup(const DPlan* dp, const InstDev& w, hipStream_t s);
// jac = false: the residual only, F untouched
void launch_eval_assemble(const DPlan* dp, const InstDev& w, hipStream_t s, bool jac = true);
void launch_lu(const DPlan* dp, const InstDev& w, hipStream_t s);
void launch_solve(const DPlan* dp, const InstDev& w, hipStream_t s);
void launch_solve_t(const DPlan* dp, const InstDev& w, hipStream_t s);
void launch_update(const DPlan* dp, const InstDev& w, hipStream_t s);
void launch_charges(const DPlan* dp, const InstDev& w, const double* v, double* q, hipStream_t s);

// batched transient: LDS bytes per workgroup and launch
size_t batch_lds_bytes(const BatchArgs& a);
int batch_max_blocks(int nr, bool va, size_t lds);   // resident workgroups per CU
hipError_t launch_tran_batch(int nr, bool va, const BatchArgs& a, int nblocks, size_t lds, hipStream_t s);

// LDS bytes of one instance beside its image
size_t lds_kernel_bytes(int32_t dbl_max, int32_t words_max);
// packed launch: workgroups of up to kPackWaves wavefronts, each workgroup
// runs one chunk at a time: up to kPackSegs runs of same-circuit instances,
// each run sharing one plan image in LDS
constexpr int kPackWaves = 8;
constexpr int kPackSegs = 4;
struct PackShape {
    int32_t nr = 1;       // rows per lane: 1, 2 or 4 (devices per lane = 2*nr)
    int32_t waves = 1;    // wavefronts per workgroup
    int32_t occ = 2;      // wavefronts per SIMD the kernel's registers allow: 2 or 4
    bool dyn = true;      // some source is not DC
};
int pack_max_blocks(const PackShape& k, size_t lds);   // resident workgroups per CU
hipError_t launch_tran_pack(const PackShape& k, const LdsArgs* d_args, int nblocks, size_t lds, hipStream_t s);
// DC operating point of one circuit (args: its plans, params, u_final, stats, o)
hipError_t launch_lds_dcop(int nr, bool dyn, const LdsArgs* d_args, size_t lds, hipStream_t s);
// one recorded Newton iteration of the LDS-resident instance code (pivot order)
hipError_t launch_lds_probe(int nr, const CPlan* cp, const DPlan* P, const double* p, const double* u_piv,
                            const double* qx_piv, double a0, double t, int mode, double* f_asm,
                            double* res_piv, double* f_lu, double* dx_piv, size_t lds, hipStream_t s);

// LDS-resident adjoint: the recording forward or the reverse kernel's resident
// workgroups per CU, and its launch
int adj_lds_max_blocks(int nr, bool dyn, bool reverse, size_t lds);
hipError_t launch_adj_lds(int nr, bool dyn, bool reverse, const AdjLdsArgs* d_args, int nblocks, size_t lds,
                          hipStream_t s);

// BSIM-CMG: sizes of the generated structs, host helpers, launch
int bsim_card_size();
int bsim_inst_size();
int bsim_out_per();
void bsim_card_defaults(void* card);
int bsim_set_param(void* card, void* inst, const char* name, double value);
int bsim_max_blocks();
int bsim_setup_size();
hipError_t launch_bsimcmg(const BsimArgs& a, int nblocks, hipStream_t s);
// the library's own device buffer for cs_bsimcmg_eval_noalloc (bsimcmg.hip)
int bsim_noalloc_lanes();
size_t bsim_scratch_card_off();
size_t bsim_scratch_inst_off();
size_t bsim_scratch_store_off();
void* bsim_scratch(int device, std::string& err);

}  // namespace cedar
