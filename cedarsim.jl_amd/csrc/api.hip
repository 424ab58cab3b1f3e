// api.hip — implementation of the C ABI declared in include/cedarhip.h.
//
// Host responsibilities: symbolic analysis (symbolic.cpp), plan upload, the
// DAE interface (residual / Jacobian / LU on the device), the plain
// per-instance transient (host step control, one captured hipGraph launch per
// Newton iteration), and the batched transient (one persistent kernel).
// There is no CPU compute fallback: without a HIP device every compute entry
// point returns CS_E_NODEVICE.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <functional>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/cedarhip.h"
#include "big.h"
#include "compact.h"
#include "dcop_rules.h"
#include "kernels.h"
#include "plan.h"
#include "rules.h"

using namespace cedar;

namespace {

struct Circuit {
    Plan plan;
    DPlan hd{};                 // device pointers, host copy
    void* dbuf = nullptr;       // plan arrays
    DPlan* d_dplan = nullptr;   // device copy of hd
    // single-instance workspace
    void* wbuf = nullptr;
    InstDev w{};
    double* scratch = nullptr;  // n doubles (charges / du)
    double* h_norm = nullptr;   // pinned, NRM_SLOTS
    double* h_stage = nullptr;  // pinned: the plain transient's per-step copies (3 n doubles + a StepDev)
    hipGraphExec_t iter_exec = nullptr;
    hipGraph_t iter_graph_nf = nullptr;      // without the LU (modified Newton)
    hipGraphExec_t iter_exec_nf = nullptr;
    hipGraph_t iter_graph = nullptr;
    // 16-bit LDS plan image (compact.h) for the LDS-resident batched kernel
    bool compact_ok = false;
    std::string compact_why;
    CPlan hcp{};                // device pointers, host copy
    void* cbuf = nullptr;
    const CPlan* d_cplan = nullptr;
    // one instance on the LDS-resident kernel (cs_tran, cs_dcop)
    int32_t lds_nr = 0;         // rows per lane, 0: does not fit
    std::string lds_why;
    bool lds_dyn = false;
    size_t lds_bytes = 0;
    // large circuits: the supernodal path (big.h) instead of all of the above
    BigCircuit* big = nullptr;
};

constexpr size_t kLdsMaxBytes = 64 * 1024;   // dynamic LDS of one workgroup
constexpr size_t kPackLds = 80 * 1024 - 256; // packed launch: two workgroups per CU
constexpr size_t kSideStreams = 4;           // hardware queues of one process

// One launch of the adjoint's forward kernel and one of its reverse kernel:
// the instances of circuits whose LDS footprints are within a factor of each
// other.
struct LdsClass {
    int32_t nr = 1, n_inst = 0;
    bool dyn = false;                          // some source is not DC
    size_t lds[2] = {0, 0};                    // forward (the image without the adjoint's part), reverse
    LdsArgs args{};
};

struct Batch {
    std::vector<int32_t> cid;
    std::vector<int64_t> p_off, u_off, w_off;
    int32_t n_inst = 0;
    int32_t nr = 1;
    bool has_va = false;                       // some circuit has Verilog-A devices
    int32_t nblocks = 0;
    size_t lds = 0;
    BatchArgs args{};
    std::vector<void*> allocs;
    size_t wave_len = 0, u_len = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0.0;
    int32_t kernel = CS_BATCH_KERNEL_GLOBAL;   // which kernel runs this batch
    std::vector<LdsClass> classes;             // adjoint: one launch each
    std::vector<hipEvent_t> class_ev;
    int32_t* d_queues = nullptr;
    // the packed launch of the transient
    PackShape pack;
    int32_t pack_blocks = 0;
    size_t pack_lds = 0;
    LdsArgs pack_args{};
    const LdsArgs* d_pack_args = nullptr;
    std::vector<int32_t> used, c_nr;           // circuits of the batch; rows per lane by circuit id
};

}  // namespace

struct cs_ctx {
    int device = 0;
    std::vector<char> bsim_card, bsim_inst;   // host copies (generated structs)
    std::vector<char> bsim_card_full;         // bsim_card with the model's defaults filled in
    bool bsim_ready = false;
    hipStream_t stream = nullptr;
    std::vector<hipStream_t> side;   // default-priority streams for concurrent class launches
    int n_cu = 0;
    double clock_hz = 1e8;      // wall_clock64() ticks per second
    std::string err;
    std::vector<std::unique_ptr<Circuit>> circuits;
    std::vector<std::unique_ptr<Batch>> batches;
    // one-launch runs of single circuits: a device buffer and a pinned image of
    // its start, kept and grown from call to call; a call holds single_mu
    std::mutex single_mu;
    char* sbuf = nullptr;
    char* h_sbuf = nullptr;
    size_t sbuf_bytes = 0, h_sbuf_bytes = 0;
};

namespace {

int fail(cs_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    return code;
}

#define HIPCHK(ctx, expr)                                                              \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess)                                                          \
            return fail(ctx, e_ == hipErrorOutOfMemory ? CS_E_OOM : CS_E_HIP,          \
                        std::string(#expr) + ": " + hipGetErrorString(e_));            \
    } while (0)

Circuit* get_circuit(cs_ctx* ctx, int32_t cid) {
    if (!ctx || cid < 0 || cid >= (int32_t)ctx->circuits.size() || !ctx->circuits[cid]) return nullptr;
    return ctx->circuits[cid].get();
}

// ---- plan upload ------------------------------------------------------------
struct Packer {
    std::vector<char> bytes;
    template <class T>
    size_t add(const std::vector<T>& v) {
        size_t off = (bytes.size() + 15) & ~size_t(15);
        bytes.resize(off + std::max<size_t>(v.size() * sizeof(T), 16));
        if (!v.empty()) std::memcpy(bytes.data() + off, v.data(), v.size() * sizeof(T));
        return off;
    }
};

// Rows per lane of the LDS-resident kernels, or why the circuit does not fit.
void lds_shape(Circuit& C) {
    C.lds_nr = 0;
    if (!C.compact_ok) { C.lds_why = C.compact_why; return; }
    const CPlan& cp = C.hcp;
    int32_t nr = cp.n <= 64 ? 1 : cp.n <= 128 ? 2 : 4;
    while (nr < 4 && cp.n_mos > 128 * nr) nr *= 2;
    if (cp.n > 64 * nr || cp.n_mos > 128 * nr || cp.n_src > 64 * 64) {
        C.lds_why = "circuit exceeds the LDS-resident kernel's per-lane limits (256 unknowns, 512 devices)";
        return;
    }
    C.lds_bytes = lds_kernel_bytes((cp.dbl + 1) & ~1, cp.words);
    if (C.lds_bytes > kLdsMaxBytes) {
        C.lds_why = "circuit needs more LDS than one workgroup may hold";
        return;
    }
    C.lds_nr = nr;
    C.lds_dyn = false;
    for (const SrcDesc& d : C.plan.src) C.lds_dyn = C.lds_dyn || d.kind != CS_WAVE_DC;
}

// The plan header, the LDS plan image and its pivot-order side arrays in one
// allocation (the image 16-byte aligned).  A circuit whose indices do not fit 16 bits
// keeps compact_ok = false and runs on the global-plan kernel.
int upload_compact(cs_ctx* ctx, Circuit& C) {
    std::vector<uint16_t> blob;
    std::vector<int32_t> lpos, colnat, diffrow, probe, dev, devrow;
    const char* why = "";
    CPlan cp{};
    if (C.cbuf) { (void)hipFree(C.cbuf); C.cbuf = nullptr; }
    C.compact_ok = build_compact(C.plan, blob, cp, lpos, colnat, diffrow, probe, dev, devrow, &why);
    C.compact_why = why;
    if (!C.compact_ok) {
        lds_shape(C);
        return CS_OK;
    }
    Packer pk;
    const size_t o_hdr = pk.add(std::vector<CPlan>(1));
    size_t o_blob = pk.add(blob), o_lp = pk.add(lpos), o_cn = pk.add(colnat), o_df = pk.add(diffrow), o_pr = pk.add(probe),
           o_dev = pk.add(dev), o_dr = pk.add(devrow);
    HIPCHK(ctx, hipMalloc(&C.cbuf, pk.bytes.size()));
    char* b = (char*)C.cbuf;
    cp.blob = (const uint16_t*)(b + o_blob);
    cp.lpos = (const int32_t*)(b + o_lp);
    cp.colnat = (const int32_t*)(b + o_cn);
    cp.diffrow = (const int32_t*)(b + o_df);
    cp.probe = (const int32_t*)(b + o_pr);
    cp.dev = (const int32_t*)(b + o_dev);
    cp.devrow = (const int32_t*)(b + o_dr);
    cp.mos_m = C.hd.mos_m;
    cp.src_m = C.hd.src_m;
    C.hcp = cp;
    std::memcpy(pk.bytes.data() + o_hdr, &cp, sizeof(CPlan));
    HIPCHK(ctx, hipMemcpy(C.cbuf, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice));
    C.d_cplan = (const CPlan*)(b + o_hdr);
    lds_shape(C);
    return CS_OK;
}

int upload_plan(cs_ctx* ctx, Circuit& C) {
    const Plan& P = C.plan;
    Packer pk;
    std::vector<int32_t> mos4 = P.mos;
    std::vector<int4> src4;
    for (auto& s : P.src) src4.push_back(make_int4(s.kind, s.off, s.len, s.dc));
    std::vector<int4> task4;
    for (auto& t : P.lu_task) task4.push_back(make_int4(t.e, t.ub, t.ue, t.piv));
    std::vector<int2> upd2;
    for (size_t q = 0; q + 1 < P.lu_upd.size(); q += 2) upd2.push_back(make_int2(P.lu_upd[q], P.lu_upd[q + 1]));
    size_t o_rowptr = pk.add(P.rowptr), o_colperm = pk.add(P.colperm), o_colnat = pk.add(P.colnat),
           o_rownat = pk.add(P.rownat), o_pcol = pk.add(P.pcol), o_diag = pk.add(P.diag),
           o_lk = pk.add(P.lin_kind), o_li = pk.add(P.lin_idx), o_gp = pk.add(P.g_ptr),
           o_gr = pk.add(P.g_ref), o_cp = pk.add(P.c_ptr), o_cr = pk.add(P.c_ref),
           o_mos = pk.add(mos4), o_jp = pk.add(P.jnl_ptr), o_jr = pk.add(P.jnl_ref),
           o_rp = pk.add(P.rnl_ptr), o_rr = pk.add(P.rnl_ref), o_src = pk.add(src4),
           o_ll = pk.add(P.lu_lptr), o_lt = pk.add(task4), o_lu = pk.add(upd2),
           o_fl = pk.add(P.f_lptr), o_fr = pk.add(P.f_rows), o_bl = pk.add(P.b_lptr),
           o_br = pk.add(P.b_rows), o_tcp = pk.add(P.tcol_ptr), o_tcq = pk.add(P.tcol_pos),
           o_tcr = pk.add(P.tcol_row), o_tfl = pk.add(P.tf_lptr), o_tfr = pk.add(P.tf_rows),
           o_tbl = pk.add(P.tb_lptr), o_tbr = pk.add(P.tb_rows), o_isd = pk.add(P.is_diff),
           o_ps = pk.add(P.probe_slot), o_ls = pk.add(P.lin_scale), o_mm = pk.add(P.mos_m),
           o_sm = pk.add(P.src_m), o_vd = pk.add(P.va_dev), o_vn = pk.add(P.va_nodes), o_vs = pk.add(P.va_st);
    if (C.dbuf) { (void)hipFree(C.dbuf); C.dbuf = nullptr; }
    HIPCHK(ctx, hipMalloc(&C.dbuf, pk.bytes.size()));
    HIPCHK(ctx, hipMemcpy(C.dbuf, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice));
    char* b = (char*)C.dbuf;
    auto I = [&](size_t o) { return (const int32_t*)(b + o); };
    DPlan& d = C.hd;
    d.n = P.n; d.n_nodes = P.n_nodes; d.nnz = P.nnz; d.n_mos = P.n_mos; d.n_src = P.n_src;
    d.n_lin = P.n_lin; d.n_stamp = P.n_stamp;
    d.lu_nlev = (int32_t)P.lu_lptr.size() - 1; d.f_nlev = (int32_t)P.f_lptr.size() - 1;
    d.b_nlev = (int32_t)P.b_lptr.size() - 1; d.tf_nlev = (int32_t)P.tf_lptr.size() - 1;
    d.tb_nlev = (int32_t)P.tb_lptr.size() - 1;
    d.n_probe = (int32_t)P.probe.size(); d.uic_ok = P.uic_ok ? 1 : 0;
    d.p_mos_vth = P.lay.mos_vth; d.p_mos_kp = P.lay.mos_kp; d.p_mos_w = P.lay.mos_w;
    d.p_mos_l = P.lay.mos_l; d.p_gmin = P.lay.gmin; d.n_params = P.lay.n_params;
    d.rowptr = I(o_rowptr); d.colperm = I(o_colperm); d.colnat = I(o_colnat); d.rownat = I(o_rownat);
    d.pcol = I(o_pcol); d.diag = I(o_diag);
    d.lin_kind = I(o_lk); d.lin_idx = I(o_li); d.g_ptr = I(o_gp); d.g_ref = I(o_gr);
    d.c_ptr = I(o_cp); d.c_ref = I(o_cr); d.mos = I(o_mos);
    d.jnl_ptr = I(o_jp); d.jnl_ref = I(o_jr); d.rnl_ptr = I(o_rp); d.rnl_ref = I(o_rr);
    d.src = (const int4*)(b + o_src);
    d.lu_lptr = I(o_ll); d.lu_task = (const int4*)(b + o_lt); d.lu_upd = (const int2*)(b + o_lu);
    d.f_lptr = I(o_fl); d.f_rows = I(o_fr); d.b_lptr = I(o_bl); d.b_rows = I(o_br);
    d.tcol_ptr = I(o_tcp); d.tcol_pos = I(o_tcq); d.tcol_row = I(o_tcr);
    d.tf_lptr = I(o_tfl); d.tf_rows = I(o_tfr); d.tb_lptr = I(o_tbl); d.tb_rows = I(o_tbr);
    d.is_diff = I(o_isd); d.probe_slot = I(o_ps);
    d.lin_scale = (const double*)(b + o_ls);
    d.mos_m = P.mos_m.empty() ? nullptr : (const double*)(b + o_mm);
    d.src_m = P.src_m.empty() ? nullptr : (const double*)(b + o_sm);
    d.n_va = P.n_va;
    d.va_dev = (const int4*)(b + o_vd);
    d.va_nodes = I(o_vn);
    d.va_st = I(o_vs);
    if (!C.d_dplan) HIPCHK(ctx, hipMalloc(&C.d_dplan, sizeof(DPlan)));
    HIPCHK(ctx, hipMemcpy(C.d_dplan, &C.hd, sizeof(DPlan), hipMemcpyHostToDevice));
    return upload_compact(ctx, C);
}

// ---- single-instance workspace ---------------------------------------------------
int ensure_workspace(cs_ctx* ctx, Circuit& C) {
    if (C.wbuf) return CS_OK;
    const Plan& P = C.plan;
    size_t nd = (size_t)P.lay.n_params + P.n_lin + 3 * (size_t)P.nnz + 6 * (size_t)P.n +
                P.n_stamp + NRM_SLOTS + 8;
    size_t bytes = nd * sizeof(double) + sizeof(StepDev) + 64;
    HIPCHK(ctx, hipMalloc(&C.wbuf, bytes));
    double* q = (double*)C.wbuf;
    auto take = [&](size_t k) { double* r = q; q += k; return r; };
    C.w.p = take(P.lay.n_params);
    C.w.linbuf = take(P.n_lin);
    C.w.Glin = take(P.nnz);
    C.w.Clin = take(P.nnz);
    C.w.F = take(P.nnz);
    C.w.inv = take(P.n);
    C.w.u = take(P.n);
    C.w.x = take(P.n);
    C.w.qx = take(P.n);
    C.w.u0 = take(P.n);
    C.scratch = take(P.n);
    C.w.st = take(std::max(P.n_stamp, 1));
    C.w.norm = take(NRM_SLOTS);
    C.w.sp = (StepDev*)take(sizeof(StepDev) / sizeof(double) + 1);
    C.w.has_va = P.n_va > 0;
    HIPCHK(ctx, hipMemset(C.wbuf, 0, bytes));
    HIPCHK(ctx, hipHostMalloc((void**)&C.h_norm, NRM_SLOTS * sizeof(double), hipHostMallocDefault));
    HIPCHK(ctx, hipHostMalloc((void**)&C.h_stage, (3 * (size_t)P.n + sizeof(StepDev) / sizeof(double) + 1) *
                                                    sizeof(double), hipHostMallocDefault));
    return CS_OK;
}

// Graphs of one Newton iteration: eval+assemble -> LU -> solves -> update ->
// copy of the norms to pinned host memory; and the same with the residual
// alone and no LU, the solves on the factors already in F (modified Newton).
int ensure_graph(cs_ctx* ctx, Circuit& C) {
    if (C.iter_exec) return CS_OK;
    for (int full = 1; full >= 0; full--) {
        HIPCHK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        launch_eval_assemble(C.d_dplan, C.w, ctx->stream, full != 0);
        if (full) launch_lu(C.d_dplan, C.w, ctx->stream);
        launch_solve(C.d_dplan, C.w, ctx->stream);
        launch_update(C.d_dplan, C.w, ctx->stream);
        (void)hipMemcpyAsync(C.h_norm, C.w.norm, NRM_SLOTS * sizeof(double), hipMemcpyDeviceToHost,
                             ctx->stream);
        hipGraph_t& g = full ? C.iter_graph : C.iter_graph_nf;
        HIPCHK(ctx, hipStreamEndCapture(ctx->stream, &g));
        HIPCHK(ctx, hipGraphInstantiate(full ? &C.iter_exec : &C.iter_exec_nf, g, nullptr, nullptr, 0));
    }
    return CS_OK;
}

int set_step(cs_ctx* ctx, Circuit& C, const StepDev& sp) {
    HIPCHK(ctx, hipMemcpyAsync(C.w.sp, &sp, sizeof(StepDev), hipMemcpyHostToDevice, ctx->stream));
    return CS_OK;
}

int run_iteration(cs_ctx* ctx, Circuit& C, bool full = true) {
    HIPCHK(ctx, hipGraphLaunch(full ? C.iter_exec : C.iter_exec_nf, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return CS_OK;
}

int check_params(cs_ctx* ctx, const Plan& P, const double* p) {
    if (!p) return fail(ctx, CS_E_INVALID, "null parameter vector");
    return CS_OK;
}

// Why a DC point can fail on the static pivot order: a pivot that only the
// charge terms fill (with a0 = 0 it is zero) and that no reordering could fill.
std::string dc_pivot_note(const Plan& P) {
    if (P.dc_zero_pivot < 0) return "";
    return " (the static pivot order has a zero pivot at step " + std::to_string(P.dc_zero_pivot) +
           " when the charge terms vanish; start the transient from initial conditions instead)";
}

// Newton iterations from the state already in C.w.u; CS_OK when max |F| <=
// tol, CS_E_NOCONV on a non-finite residual (a singular factor shows up as
// one) or after maxit iterations.
int newton_point(cs_ctx* ctx, Circuit& C, int maxit, cs_tran_stats* st) {
    for (int it = 0; it < maxit; it++) {
        int rc = run_iteration(ctx, C);
        if (rc) return rc;
        if (C.h_norm[NRM_DONE] == 1.0) return CS_OK;
        const double r = C.h_norm[NRM_RES];
        if (!(r == r) || std::isinf(r)) return CS_E_NOCONV;
        if (st) st->newton_iters++;
    }
    return CS_E_NOCONV;
}

// Initial point on the single-instance path.  UIC: the charge rows pinned to
// u0, the algebraic rows solved (50 iterations).  DC op: the trajectories
// and the gmin ladder of dcop_rules.h (CedarDCOp, src/dcop.jl:53-94).
int init_point(cs_ctx* ctx, Circuit& C, const double* u0, const cs_tran_opts& o, bool uic,
               cs_tran_stats* st) {
    const Plan& P = C.plan;
    if (uic) {
        HIPCHK(ctx, hipMemcpyAsync(C.w.u, u0, sizeof(double) * P.n, hipMemcpyHostToDevice, ctx->stream));
        HIPCHK(ctx, hipMemcpyAsync(C.w.u0, u0, sizeof(double) * P.n, hipMemcpyHostToDevice, ctx->stream));
    }
    StepDev sp{};
    sp.a0 = 0.0; sp.t = o.t_start; sp.rtol = o.reltol; sp.atol = o.abstol; sp.tol = o.dc_abstol;
    sp.mode = uic ? CS_MODE_TRAN : CS_MODE_DCOP;
    sp.kind = uic ? STEP_UIC : STEP_DC;
    int rc = set_step(ctx, C, sp);
    if (rc) return rc;
    if (uic) return newton_point(ctx, C, 50, st);
    std::vector<double> us(P.n);
    auto start = [&](int j) -> int {
        for (int32_t i = 0; i < P.n; i++) us[i] = dc_start(j, i);
        HIPCHK(ctx, hipMemcpyAsync(C.w.u, us.data(), sizeof(double) * P.n, hipMemcpyHostToDevice, ctx->stream));
        return CS_OK;
    };
    for (int j = 0; j < kDcTrajectories; j++) {
        if ((rc = start(j))) return rc;
        rc = newton_point(ctx, C, kDcMaxIt, st);
        if (rc != CS_E_NOCONV) return rc;
    }
    // the gmin ladder, on the device's copy of p; the circuit's gmin is
    // restored afterwards
    double gc = 0.0;
    HIPCHK(ctx, hipMemcpy(&gc, C.w.p + P.lay.gmin, sizeof(double), hipMemcpyDeviceToHost));
    if ((rc = start(0))) return rc;
    for (int q = 0;; q++) {
        const double g = dc_gmin_stage(q, gc);
        if (g < 0.0) break;
        HIPCHK(ctx, hipMemcpyAsync(C.w.p + P.lay.gmin, &g, sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        rc = newton_point(ctx, C, kDcMaxIt, st);
        if (rc != CS_OK) break;
    }
    HIPCHK(ctx, hipMemcpyAsync(C.w.p + P.lay.gmin, &gc, sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return rc;
}

// CedarDCOp after the DC point (its BrownFullBasicInit step, src/dcop.jl:153):
// the rows that carry charge pinned to the DC point, the algebraic rows
// solved again with the sources at their transient values at t_start.
int reinit_at_t0(cs_ctx* ctx, Circuit& C, const cs_tran_opts& o, cs_tran_stats* st) {
    const Plan& P = C.plan;
    HIPCHK(ctx, hipMemcpyAsync(C.w.u0, C.w.u, sizeof(double) * P.n, hipMemcpyDeviceToDevice, ctx->stream));
    StepDev sp{};
    sp.a0 = 0.0; sp.t = o.t_start; sp.rtol = o.reltol; sp.atol = o.abstol; sp.tol = o.dc_abstol;
    sp.mode = CS_MODE_TRAN;
    sp.kind = STEP_UIC;
    int rc = set_step(ctx, C, sp);
    if (rc) return rc;
    return newton_point(ctx, C, 50, st);
}

}  // namespace

// =====================================================================================
extern "C" {

int cs_abi_version(void) { return CEDARHIP_ABI_VERSION; }

int cs_device_count(int32_t* count) {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (count) *count = (e == hipSuccess) ? n : 0;
    return (e == hipSuccess && n > 0) ? CS_OK : CS_E_NODEVICE;
}

#ifdef CEDAR_HAVE_BSIMCMG
static void bsim_init(cs_ctx* ctx);
#endif

int cs_create(int32_t device, cs_ctx** out) {
    if (!out) return CS_E_INVALID;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return CS_E_NODEVICE;
    if (device < 0 || device >= n) return CS_E_INVALID;
    if (hipSetDevice(device) != hipSuccess) return CS_E_HIP;
    auto* c = new cs_ctx();
    c->device = device;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return CS_E_HIP;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->n_cu = prop.multiProcessorCount;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0)
        c->clock_hz = 1e3 * khz;
#ifdef CEDAR_HAVE_BSIMCMG
    {   // the device address of the no-allocation entry's buffer on this GPU
        std::string err;
        if (!bsim_scratch(device, err)) {
            (void)hipStreamDestroy(c->stream);
            delete c;
            return CS_E_HIP;
        }
        bsim_init(c);   // host copies of the card, so that the entry allocates nothing later
    }
#endif
    *out = c;
    return CS_OK;
}

int cs_destroy(cs_ctx* ctx) {
    if (!ctx) return CS_E_INVALID;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (auto& b : ctx->batches)
        if (b) {
            for (void* p : b->allocs) (void)hipFree(p);
            if (b->ev0) (void)hipEventDestroy(b->ev0);
            if (b->ev1) (void)hipEventDestroy(b->ev1);
            for (hipEvent_t e : b->class_ev) (void)hipEventDestroy(e);
        }
    for (auto& c : ctx->circuits)
        if (c) {
            if (c->iter_exec) (void)hipGraphExecDestroy(c->iter_exec);
            if (c->iter_graph) (void)hipGraphDestroy(c->iter_graph);
            if (c->iter_exec_nf) (void)hipGraphExecDestroy(c->iter_exec_nf);
            if (c->iter_graph_nf) (void)hipGraphDestroy(c->iter_graph_nf);
            if (c->dbuf) (void)hipFree(c->dbuf);
            if (c->d_dplan) (void)hipFree(c->d_dplan);
            if (c->wbuf) (void)hipFree(c->wbuf);
            if (c->h_norm) (void)hipHostFree(c->h_norm);
            if (c->h_stage) (void)hipHostFree(c->h_stage);
            if (c->cbuf) (void)hipFree(c->cbuf);
            if (c->big) big_destroy(c->big);
        }
    if (ctx->sbuf) (void)hipFree(ctx->sbuf);
    if (ctx->h_sbuf) (void)hipHostFree(ctx->h_sbuf);
    for (hipStream_t st : ctx->side) (void)hipStreamDestroy(st);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return CS_OK;
}

const char* cs_last_error(const cs_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

// ---- host-only analysis ---------------------------------------------------------------
static void fill_info(const Plan& P, cs_circuit_info* info) {
    info->n = P.n;
    info->n_nodes = P.n_nodes;
    info->nnz = P.nnz_nat;
    info->nnz_lu = P.nnz;
    info->n_params = P.lay.n_params;
    info->lu_levels = (int32_t)P.lu_lptr.size() - 1;
    info->fwd_levels = (int32_t)P.f_lptr.size() - 1;
    info->bwd_levels = (int32_t)P.b_lptr.size() - 1;
    info->lu_updates = P.lu_updates;
    info->n_singletons = P.n_singletons;
    info->n_probe = (int32_t)P.probe.size();
}

int cs_analyze(const cs_netlist* nl, cs_circuit_info* info, int32_t* lu_rowptr,
               int32_t* lu_col, int32_t* rownat, int32_t* colnat) {
    if (!nl || !info) return CS_E_INVALID;
    Plan P;
    std::string err;
    int rc = build_plan(nl, P, err);
    if (rc != CS_OK) return rc;
    fill_info(P, info);
    if (lu_rowptr) std::memcpy(lu_rowptr, P.rowptr.data(), sizeof(int32_t) * (P.n + 1));
    if (lu_col) std::memcpy(lu_col, P.colperm.data(), sizeof(int32_t) * P.nnz);
    if (rownat) std::memcpy(rownat, P.rownat.data(), sizeof(int32_t) * P.n);
    if (colnat)
        for (int32_t i = 0; i < P.n; i++) colnat[P.pcol[i]] = i;
    return CS_OK;
}

int cs_pack_plan(int32_t n_circ, const cs_netlist* const* nls, const int32_t* counts, int32_t cap_chunks,
                 int32_t cap_segs, int32_t* n_chunks, int32_t* n_segs, int32_t* seg_ptr, int32_t* seg_circ,
                 int32_t* seg_count, int64_t* lds_bytes) {
    if (n_circ <= 0 || !nls || !counts || !n_chunks || !n_segs) return CS_E_INVALID;
    *n_chunks = *n_segs = 0;
    std::vector<size_t> img(n_circ), dblb(n_circ), rem(n_circ);
    std::vector<int32_t> dbl(n_circ), nn(n_circ), order(n_circ);
    for (int32_t c = 0; c < n_circ; c++) {
        Plan P;
        std::string err;
        if (!nls[c] || counts[c] < 0 || build_plan(nls[c], P, err) != CS_OK) return CS_E_INVALID;
        std::vector<uint16_t> blob;
        std::vector<int32_t> a, b, d, e, f, g;
        CPlan cp{};
        const char* why = "";
        if (!build_compact(P, blob, cp, a, b, d, e, f, g, &why)) return CS_E_INVALID;
        img[c] = 2 * (size_t)((cp.words + 7) & ~7);
        dblb[c] = 8 * (size_t)((cp.dbl + 1) & ~1);
        dbl[c] = cp.dbl;
        nn[c] = cp.n;
        rem[c] = (size_t)counts[c];
        order[c] = c;
    }
    std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) {
        return dbl[x] != dbl[y] ? dbl[x] > dbl[y] : nn[x] > nn[y];
    });
    size_t need = 0;
    const auto chunks = pack_chunks(order, img, dblb, rem, kPackWaves, kPackSegs, kPackLds, &need);
    size_t total = 0;
    for (size_t c = 0; c < rem.size(); c++) total += rem[c];
    if (chunks.empty() && total > 0) return CS_E_RANGE;
    size_t ns = 0;
    for (const auto& ch : chunks) ns += ch.size();
    *n_chunks = (int32_t)chunks.size();
    *n_segs = (int32_t)ns;
    if (lds_bytes) *lds_bytes = (int64_t)need;
    if ((int64_t)chunks.size() > cap_chunks || (int64_t)ns > cap_segs || !seg_ptr || !seg_circ || !seg_count)
        return CS_E_RANGE;
    int32_t q = 0;
    for (size_t k = 0; k < chunks.size(); k++) {
        seg_ptr[k] = q;
        for (const PackSeg& g : chunks[k]) {
            seg_circ[q] = g.c;
            seg_count[q] = g.cnt;
            q++;
        }
    }
    seg_ptr[chunks.size()] = q;
    return CS_OK;
}

// ---- circuits -----------------------------------------------------------------------
int cs_circuit_load(cs_ctx* ctx, const cs_netlist* nl, int32_t* cid) {
    return cs_circuit_load_solver(ctx, nl, CS_SOLVER_AUTO, cid);
}

int cs_circuit_load_solver(cs_ctx* ctx, const cs_netlist* nl, int32_t solver, int32_t* cid) {
    if (!ctx || !nl || !cid) return fail(ctx, CS_E_INVALID, "null argument");
    if (solver < CS_SOLVER_AUTO || solver > CS_SOLVER_SUPERNODAL) return fail(ctx, CS_E_INVALID, "unknown solver");
    (void)hipSetDevice(ctx->device);
    auto C = std::make_unique<Circuit>();
    std::string err;
    const int64_t n = (int64_t)nl->n_nodes + nl->n_vsrc + nl->n_ind + nl->n_vcvs;
    const bool has_va = nl->n_va > 0;
    if (has_va && solver == CS_SOLVER_SUPERNODAL)
        return fail(ctx, CS_E_INVALID, "Verilog-A devices run on the level-scheduled solver");
    const bool big = solver == CS_SOLVER_SUPERNODAL ||
                     (solver == CS_SOLVER_AUTO && n >= CS_SUPERNODAL_MIN_N && !has_va);
    int rc;
    if (big) {
        rc = big_create(nl, ctx->stream, &C->big, err);
        if (rc != CS_OK) return fail(ctx, rc, err);
        C->plan = big_plan(C->big).base;
    } else {
        rc = build_plan(nl, C->plan, err);
        if (rc != CS_OK) return fail(ctx, rc, err);
        if ((rc = upload_plan(ctx, *C)) != CS_OK) return rc;
    }
    ctx->circuits.push_back(std::move(C));
    *cid = (int32_t)ctx->circuits.size() - 1;
    return CS_OK;
}

int cs_big_analyze(const cs_netlist* nl, cs_big_info* info, int32_t* rownat, int32_t* colnat) {
    if (!nl || !info) return CS_E_INVALID;
    BigPlan B;
    std::string err;
    int rc = build_bigplan(nl, B, err);
    if (rc != CS_OK) return rc;
    big_info(B, info);
    if (rownat) std::memcpy(rownat, B.rownat.data(), sizeof(int32_t) * B.n);
    if (colnat) std::memcpy(colnat, B.colnat.data(), sizeof(int32_t) * B.n);
    return CS_OK;
}

int cs_big_info_get(cs_ctx* ctx, int32_t cid, cs_big_info* info) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !info) return fail(ctx, CS_E_INVALID, "bad argument");
    if (!C->big) return fail(ctx, CS_E_INVALID, "not a supernodal circuit");
    big_info(big_plan(C->big), info);
    return CS_OK;
}

int cs_big_times(cs_ctx* ctx, int32_t cid, double* factor_ms, double* solve_ms) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C) return fail(ctx, CS_E_INVALID, "bad circuit id");
    if (!C->big) return fail(ctx, CS_E_INVALID, "not a supernodal circuit");
    big_last_times(C->big, factor_ms, solve_ms);
    return CS_OK;
}

int cs_big_profile(cs_ctx* ctx, int32_t cid, int32_t* kinds, int32_t* levels, float* ms, int32_t cap,
                   int32_t* count) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || cap < 0) return fail(ctx, CS_E_INVALID, "bad argument");
    if (!C->big) return fail(ctx, CS_E_INVALID, "not a supernodal circuit");
    std::string err;
    int rc = big_profile(C->big, ctx->stream, kinds, levels, ms, cap, count, err);
    return rc ? fail(ctx, rc, err) : CS_OK;
}

int cs_circuit_info_get(cs_ctx* ctx, int32_t cid, cs_circuit_info* info) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !info) return fail(ctx, CS_E_INVALID, "bad circuit id");
    fill_info(C->plan, info);
    return CS_OK;
}

int cs_circuit_layout(cs_ctx* ctx, int32_t cid, cs_param_layout* lay) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !lay) return fail(ctx, CS_E_INVALID, "bad circuit id");
    *lay = C->plan.lay;
    return CS_OK;
}

int cs_circuit_default_params(cs_ctx* ctx, int32_t cid, double* p) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !p) return fail(ctx, CS_E_INVALID, "bad argument");
    std::memcpy(p, C->plan.p_default.data(), sizeof(double) * C->plan.p_default.size());
    return CS_OK;
}

int cs_circuit_pattern(cs_ctx* ctx, int32_t cid, int32_t* rowptr, int32_t* colind) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !rowptr || !colind) return fail(ctx, CS_E_INVALID, "bad argument");
    std::memcpy(rowptr, C->plan.nat_rowptr.data(), sizeof(int32_t) * (C->plan.n + 1));
    std::memcpy(colind, C->plan.nat_col.data(), sizeof(int32_t) * C->plan.nnz_nat);
    return CS_OK;
}

int cs_circuit_set_probes(cs_ctx* ctx, int32_t cid, int32_t n_probe, const int32_t* idx) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || n_probe < 0 || (n_probe > 0 && !idx)) return fail(ctx, CS_E_INVALID, "bad argument");
    std::vector<int32_t> v(idx, idx + n_probe);
    std::vector<char> seen(C->plan.n, 0);
    for (int32_t i : v) {
        if (i < 0 || i >= C->plan.n) return fail(ctx, CS_E_INVALID, "probe index out of range");
        if (seen[i]) return fail(ctx, CS_E_INVALID, "duplicate probe index");
        seen[i] = 1;
    }
    set_probes(C->plan, v);
    (void)hipSetDevice(ctx->device);
    if (C->big) {
        std::string err;
        int rc = big_set_probes(C->big, v, err);
        return rc ? fail(ctx, rc, err) : CS_OK;
    }
    return upload_plan(ctx, *C);
}

// ---- DAE interface ------------------------------------------------------------------
int cs_residual(cs_ctx* ctx, int32_t cid, double* out, const double* du, const double* u,
                const double* p, double t, int32_t mode) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !out || !u || !p) return fail(ctx, CS_E_INVALID, "bad argument");
    (void)hipSetDevice(ctx->device);
    if (C->big) {
        std::string err;
        int rc = big_residual(C->big, ctx->stream, out, du, u, p, t, mode, err);
        return rc ? fail(ctx, rc, err) : CS_OK;
    }
    int rc = ensure_workspace(ctx, *C);
    if (rc) return rc;
    const Plan& P = C->plan;
    hipStream_t s = ctx->stream;
    HIPCHK(ctx, hipMemcpyAsync(C->w.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
    HIPCHK(ctx, hipMemcpyAsync(C->w.u, u, sizeof(double) * P.n, hipMemcpyHostToDevice, s));
    launch_lin_setup(C->d_dplan, C->w, s);
    StepDev sp{};
    sp.t = t;
    sp.mode = mode;
    sp.kind = mode == CS_MODE_DCOP ? STEP_DC : STEP_TRAN;
    sp.a0 = 0.0;
    if (mode != CS_MODE_DCOP) {
        std::vector<double> z(P.n, 0.0);
        HIPCHK(ctx, hipMemcpyAsync(C->scratch, du ? du : z.data(), sizeof(double) * P.n,
                                   hipMemcpyHostToDevice, s));
        launch_charges(C->d_dplan, C->w, C->scratch, C->w.qx, s);
    }
    if ((rc = set_step(ctx, *C, sp))) return rc;
    launch_eval_assemble(C->d_dplan, C->w, s);
    std::vector<double> x(P.n);
    HIPCHK(ctx, hipMemcpyAsync(x.data(), C->w.x, sizeof(double) * P.n, hipMemcpyDeviceToHost, s));
    HIPCHK(ctx, hipStreamSynchronize(s));
    for (int k = 0; k < P.n; k++) out[P.rownat[k]] = -x[k];
    return CS_OK;
}

int cs_jacobian(cs_ctx* ctx, int32_t cid, double* vals, const double* du, const double* u,
                const double* p, double gamma, double t, int32_t mode) {
    (void)du;
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !vals || !u || !p) return fail(ctx, CS_E_INVALID, "bad argument");
    (void)hipSetDevice(ctx->device);
    if (C->big) {
        std::string err;
        int rc = big_jacobian(C->big, ctx->stream, vals, du, u, p, gamma, t, mode, err);
        return rc ? fail(ctx, rc, err) : CS_OK;
    }
    int rc = ensure_workspace(ctx, *C);
    if (rc) return rc;
    const Plan& P = C->plan;
    hipStream_t s = ctx->stream;
    HIPCHK(ctx, hipMemcpyAsync(C->w.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
    HIPCHK(ctx, hipMemcpyAsync(C->w.u, u, sizeof(double) * P.n, hipMemcpyHostToDevice, s));
    launch_lin_setup(C->d_dplan, C->w, s);
    StepDev sp{};
    sp.t = t;
    sp.mode = mode;
    sp.kind = mode == CS_MODE_DCOP ? STEP_DC : STEP_TRAN;
    sp.a0 = gamma;
    HIPCHK(ctx, hipMemsetAsync(C->w.qx, 0, sizeof(double) * P.n, s));
    if ((rc = set_step(ctx, *C, sp))) return rc;
    launch_eval_assemble(C->d_dplan, C->w, s);
    std::vector<double> F(P.nnz);
    HIPCHK(ctx, hipMemcpyAsync(F.data(), C->w.F, sizeof(double) * P.nnz, hipMemcpyDeviceToHost, s));
    HIPCHK(ctx, hipStreamSynchronize(s));
    for (int q = 0; q < P.nnz_nat; q++) vals[q] = F[P.nat_fpos[q]];
    return CS_OK;
}

int cs_lu_refactor(cs_ctx* ctx, int32_t cid, const double* vals) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !vals) return fail(ctx, CS_E_INVALID, "bad argument");
    (void)hipSetDevice(ctx->device);
    if (C->big) {
        std::string err;
        int rc = big_lu_refactor(C->big, ctx->stream, vals, err);
        return rc ? fail(ctx, rc, err) : CS_OK;
    }
    int rc = ensure_workspace(ctx, *C);
    if (rc) return rc;
    const Plan& P = C->plan;
    std::vector<double> F(P.nnz, 0.0);
    for (int q = 0; q < P.nnz_nat; q++) F[P.nat_fpos[q]] = vals[q];
    HIPCHK(ctx, hipMemcpyAsync(C->w.F, F.data(), sizeof(double) * P.nnz, hipMemcpyHostToDevice, ctx->stream));
    launch_lu(C->d_dplan, C->w, ctx->stream);
    std::vector<double> inv(P.n);
    HIPCHK(ctx, hipMemcpyAsync(inv.data(), C->w.inv, sizeof(double) * P.n, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < P.n; k++)
        if (!std::isfinite(inv[k]))
            return fail(ctx, CS_E_SINGULAR, "zero pivot at step " + std::to_string(k));
    return CS_OK;
}

static int lu_solve_common(cs_ctx* ctx, int32_t cid, double* x, bool transpose) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !x) return fail(ctx, CS_E_INVALID, "bad argument");
    if (C->big) {
        if (transpose) return fail(ctx, CS_E_INVALID, "transposed solves are not available for supernodal circuits");
        (void)hipSetDevice(ctx->device);
        std::string err;
        int rc = big_lu_solve(C->big, ctx->stream, x, err);
        return rc ? fail(ctx, rc, err) : CS_OK;
    }
    if (!C->wbuf) return fail(ctx, CS_E_INVALID, "cs_lu_refactor must be called first");
    (void)hipSetDevice(ctx->device);
    const Plan& P = C->plan;
    std::vector<double> b(P.n);
    if (!transpose)
        for (int k = 0; k < P.n; k++) b[k] = x[P.rownat[k]];
    else
        for (int i = 0; i < P.n; i++) b[P.pcol[i]] = x[i];
    HIPCHK(ctx, hipMemcpyAsync(C->w.x, b.data(), sizeof(double) * P.n, hipMemcpyHostToDevice, ctx->stream));
    if (!transpose) launch_solve(C->d_dplan, C->w, ctx->stream);
    else launch_solve_t(C->d_dplan, C->w, ctx->stream);
    HIPCHK(ctx, hipMemcpyAsync(b.data(), C->w.x, sizeof(double) * P.n, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    if (!transpose)
        for (int i = 0; i < P.n; i++) x[i] = b[P.pcol[i]];
    else
        for (int k = 0; k < P.n; k++) x[P.rownat[k]] = b[k];
    return CS_OK;
}

int cs_lu_solve(cs_ctx* ctx, int32_t cid, double* x) { return lu_solve_common(ctx, cid, x, false); }
int cs_lu_solve_transpose(cs_ctx* ctx, int32_t cid, double* x) {
    return lu_solve_common(ctx, cid, x, true);
}

// ---- analyses -------------------------------------------------------------------
void cs_tran_opts_default(cs_tran_opts* o) {
    if (!o) return;
    std::memset(o, 0, sizeof(*o));
    o->t_start = 0.0;
    o->t_stop = 1e-9;
    o->reltol = 1e-6;
    o->abstol = 1e-9;
    o->newton_tol = 1e-2;
    o->dc_abstol = 1e-10;
    o->n_out = 0;
    o->dt_out = 0.0;
    o->max_order = 2;
    o->newton_maxit = 8;
    o->init = CS_INIT_DCOP;
    o->max_steps = 10000000;
    o->batch_kernel = 0;
    o->record_steps = 0;
    o->jac_reuse = 0;
    o->reserved = 0;
}

static int dcop_single(cs_ctx* ctx, Circuit& C, const double* p, const cs_tran_opts* o, double* u_out,
                       cs_tran_stats* st);

int cs_dcop(cs_ctx* ctx, int32_t cid, const double* p, const cs_tran_opts* o, double* u_out,
            cs_tran_stats* st) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !o || !u_out) return fail(ctx, CS_E_INVALID, "bad argument");
    int rc = check_params(ctx, C->plan, p);
    if (rc) return rc;
    (void)hipSetDevice(ctx->device);
    if (C->big) {
        std::string err;
        rc = big_dcop(C->big, ctx->stream, p, o, u_out, st, err);
        if (rc) ctx->err = err;
        return rc;
    }
    if (C->lds_nr && o->batch_kernel != CS_BATCH_KERNEL_GLOBAL) {
        rc = dcop_single(ctx, *C, p, o, u_out, st);
        if (rc != CS_E_OOM || o->batch_kernel == CS_BATCH_KERNEL_LDS) return rc;
    }
    if ((rc = ensure_workspace(ctx, *C)) || (rc = ensure_graph(ctx, *C))) return rc;
    const Plan& P = C->plan;
    HIPCHK(ctx, hipMemcpyAsync(C->w.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, ctx->stream));
    launch_lin_setup(C->d_dplan, C->w, ctx->stream);
    cs_tran_stats lst{};
    if (!st) st = &lst;
    std::memset(st, 0, sizeof(*st));
    rc = init_point(ctx, *C, nullptr, *o, false, st);
    HIPCHK(ctx, hipMemcpy(u_out, C->w.u, sizeof(double) * P.n, hipMemcpyDeviceToHost));
    st->retcode = rc;
    st->t_end = o->t_start;
    if (rc == CS_E_NOCONV) ctx->err = "DC operating point analysis failed" + dc_pivot_note(P);
    return rc;
}

// Plain per-instance path: host step control, one graph launch per Newton
// iteration.  Follows the same rules as the batched kernel (rules.h).
// ---- forward sensitivities of the plain path (sens.hip) ---------------------------
namespace {

// The sensitivity state of one cs_tran_sens run: the parameters' stamps, the
// device buffers (charge-sensitivity history rotates through dq[0..2]) and
// the host history of the probed sensitivities for the output interpolation.
struct SensRun {
    int32_t n_sp = 0;
    std::vector<SensParam> sp;
    double* out = nullptr;            // [n_out][n_sp][n_probe]
    char* buf = nullptr;
    SensParam* d_sp = nullptr;
    int32_t* d_prow = nullptr;
    double *d_pin = nullptr, *d_x = nullptr, *d_s = nullptr;
    double* d_dq[3] = {nullptr, nullptr, nullptr};
    int hist = 0;                     // index of dq[m-1] in d_dq
    std::vector<double> S;            // [3][n_sp][n_probe]: s at the last three accepted points
    std::vector<double> s_nat;        // [n_sp][n]
};

// A parameter index of the layout -> its stamps; false when the parameter
// has none this path differentiates.
bool sens_param(const Plan& P, int32_t pi, SensParam& o) {
    const cs_param_layout& L = P.lay;
    o = SensParam{};
    o.m = 1.0;
    const int32_t nres = (int32_t)P.res_m.size(), ncap = (int32_t)P.topo.cap_m.size(),
                  nind = (int32_t)P.topo.ind_row.size(), nvccs = (int32_t)P.topo.vccs_m.size(),
                  nvcvs = (int32_t)P.topo.vcvs.size() / 3, nmos = P.n_mos;
    auto in = [](int32_t i, int32_t b, int32_t n) { return i >= b && i < b + n; };
    if (in(pi, L.res_r, nres)) {
        const int32_t k = pi - L.res_r;
        o.kind = SP_R; o.i0 = P.res_nodes[2 * k]; o.i1 = P.res_nodes[2 * k + 1]; o.m = P.res_m[k];
        return true;
    }
    if (in(pi, L.cap_c, ncap)) {
        const int32_t k = pi - L.cap_c;
        o.kind = SP_C; o.i0 = P.topo.cap[2 * k]; o.i1 = P.topo.cap[2 * k + 1]; o.m = P.topo.cap_m[k];
        return true;
    }
    if (in(pi, L.ind_l, nind)) {
        o.kind = SP_IND; o.i0 = P.topo.ind_row[pi - L.ind_l];
        return true;
    }
    if (in(pi, L.vccs_gain, nvccs)) {
        const int32_t k = pi - L.vccs_gain;
        o.kind = SP_VCCS; o.m = P.topo.vccs_m[k];
        o.i0 = P.topo.vccs[4 * k]; o.i1 = P.topo.vccs[4 * k + 1]; o.i2 = P.topo.vccs[4 * k + 2]; o.i3 = P.topo.vccs[4 * k + 3];
        return true;
    }
    if (in(pi, L.vcvs_gain, nvcvs)) {
        const int32_t k = pi - L.vcvs_gain;
        o.kind = SP_VCVS; o.i0 = P.topo.vcvs[3 * k]; o.i2 = P.topo.vcvs[3 * k + 1]; o.i3 = P.topo.vcvs[3 * k + 2];
        return true;
    }
    const int32_t mk[4] = {L.mos_vth, L.mos_kp, L.mos_w, L.mos_l};
    const int32_t kinds[4] = {SP_VTH, SP_KP, SP_MW, SP_ML};
    for (int q = 0; q < 4; q++)
        if (in(pi, mk[q], nmos)) {
            const int32_t k = pi - mk[q];
            o.kind = kinds[q]; o.dev = k;
            o.i0 = P.mos[4 * k]; o.i1 = P.mos[4 * k + 1]; o.i2 = P.mos[4 * k + 2]; o.i3 = P.mos[4 * k + 3];
            o.m = P.mos_m.empty() ? 1.0 : P.mos_m[k];
            return true;
        }
    const int32_t nv = (int32_t)P.topo.vsrc_row.size();
    for (int32_t sidx = 0; sidx < (int32_t)P.src.size(); sidx++) {
        if (P.src[sidx].dc != pi) continue;
        o.dev = P.src[sidx].kind == CS_WAVE_DC ? 1 : 0;
        if (sidx < nv) {
            o.kind = SP_VSRC; o.i0 = P.topo.vsrc_row[sidx];
        } else {
            const int32_t k = sidx - nv;
            o.kind = SP_ISRC; o.i0 = P.topo.isrc[2 * k]; o.i1 = P.topo.isrc[2 * k + 1];
            o.m = P.src_m.empty() ? 1.0 : P.src_m[sidx];
        }
        return true;
    }
    return false;
}

// Refactors the Jacobian at the state in C.w.u for the given step (the
// assembly also rewrites x and the norms, which nothing reads after an
// accepted step), then solves every parameter's sensitivity.
int sens_solve(cs_ctx* ctx, Circuit& C, SensRun& R, const StepDev& sp, int pinned, bool with_pin,
               bool hist1, bool hist2, double a1, double a2) {
    hipStream_t s = ctx->stream;
    int rc = set_step(ctx, C, sp);
    if (rc) return rc;
    launch_eval_assemble(C.d_dplan, C.w, s);
    launch_lu(C.d_dplan, C.w, s);
    SensArgs a{};
    a.P = C.d_dplan;
    a.p = C.w.p;
    a.u = C.w.u;
    a.F = C.w.F;
    a.inv = C.w.inv;
    a.Clin = C.w.Clin;
    a.prow = R.d_prow;
    a.sp = R.d_sp;
    a.n_sp = R.n_sp;
    a.mode = sp.mode;
    a.pinned = pinned;
    a.a0 = sp.kind == STEP_TRAN ? sp.a0 : 0.0;
    a.a1 = a1;
    a.a2 = a2;
    a.pin_s = with_pin ? R.d_pin : nullptr;
    a.dq1 = hist1 ? R.d_dq[R.hist] : nullptr;
    a.dq2 = hist2 ? R.d_dq[(R.hist + 1) % 3] : nullptr;
    a.x = R.d_x;
    a.s = R.d_s;
    a.dq0 = R.d_dq[(R.hist + 2) % 3];
    HIPCHK(ctx, launch_sens(a, s));
    return CS_OK;
}

// After a solve: the new charge sensitivities become dq[m-1]; the probed
// sensitivities enter the host history.
int sens_accept(cs_ctx* ctx, Circuit& C, SensRun& R) {
    const Plan& P = C.plan;
    const int n = P.n, np = (int)P.probe.size();
    R.hist = (R.hist + 2) % 3;
    HIPCHK(ctx, hipMemcpyAsync(R.s_nat.data(), R.d_s, sizeof(double) * n * R.n_sp, hipMemcpyDeviceToHost,
                               ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    const size_t blk = (size_t)R.n_sp * np;
    std::memmove(R.S.data() + blk, R.S.data(), sizeof(double) * 2 * blk);
    for (int j = 0; j < R.n_sp; j++)
        for (int q = 0; q < np; q++) R.S[(size_t)j * np + q] = R.s_nat[(size_t)j * n + P.probe[q]];
    return CS_OK;
}

}  // namespace

static int tran_plain(cs_ctx* ctx, int32_t cid, const double* p, const double* u0, const cs_tran_opts* o,
                      double* wave, double* u_final, cs_tran_stats* st_out, SensRun* sr) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !o) return fail(ctx, CS_E_INVALID, "bad argument");
    if (o->jac_reuse != 0 && o->jac_reuse != 1) return fail(ctx, CS_E_INVALID, "jac_reuse is 0 or 1");
    int rc = check_params(ctx, C->plan, p);
    if (rc) return rc;
    if (C->big) {
        if (sr) return fail(ctx, CS_E_INVALID, "sensitivities run on the level-scheduled plan, not the supernodal solver");
        (void)hipSetDevice(ctx->device);
        std::string err;
        rc = big_tran(C->big, ctx->stream, p, u0, o, wave, u_final, st_out, err);
        if (rc) ctx->err = err;
        return rc;
    }
    const Plan& P = C->plan;
    const bool uic = o->init == CS_INIT_UIC;
    if (uic && !u0) return fail(ctx, CS_E_INVALID, "UIC initialisation needs u0");
    if (uic && !P.uic_ok)
        return fail(ctx, CS_E_INVALID, "UIC: a charge-carrying row could not be kept on its own pivot");
    if (o->n_out > 0 && !(o->dt_out > 0)) return fail(ctx, CS_E_INVALID, "dt_out must be > 0");
    (void)hipSetDevice(ctx->device);
    if ((rc = ensure_workspace(ctx, *C)) || (rc = ensure_graph(ctx, *C))) return rc;
    hipStream_t s = ctx->stream;
    const int n = P.n;
    HIPCHK(ctx, hipMemcpyAsync(C->w.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
    launch_lin_setup(C->d_dplan, C->w, s);
    cs_tran_stats st{};
    rc = init_point(ctx, *C, u0, *o, uic, &st);
    if (rc == CS_OK && !uic && sr) {
        // the DC point's sensitivity: G s = -dF_DC/dp, G refactored at it
        StepDev d{};
        d.t = o->t_start; d.mode = CS_MODE_DCOP; d.kind = STEP_DC; d.tol = o->dc_abstol;
        rc = sens_solve(ctx, *C, *sr, d, 0, false, false, false, 0.0, 0.0);
        if (rc == CS_OK)
            HIPCHK(ctx, hipMemcpyAsync(sr->d_pin, sr->d_s, sizeof(double) * P.n * sr->n_sp,
                                       hipMemcpyDeviceToDevice, ctx->stream));
    }
    if (rc == CS_OK && !uic) rc = reinit_at_t0(ctx, *C, *o, &st);
    if (rc == CS_OK && sr) {
        // the initial point: charge rows pinned (to u0, or to the DC point
        // with its sensitivity), the algebraic rows solved at t_start
        StepDev d{};
        d.t = o->t_start; d.mode = CS_MODE_TRAN; d.kind = STEP_UIC; d.tol = o->dc_abstol;
        rc = sens_solve(ctx, *C, *sr, d, 1, !uic, false, false, 0.0, 0.0);
        if (rc == CS_OK) rc = sens_accept(ctx, *C, *sr);
    }
    std::vector<double> U(3 * (size_t)n, 0.0), QH(2 * (size_t)n, 0.0);
    // the per-step copies go through pinned memory, so they are queued without
    // a staging pass; the host writes it only after the stream has synchronized
    double* const up = C->h_stage;
    double* const q = up + n;
    double* const u = q + n;
    StepDev* const sph = (StepDev*)(u + n);
    const StepDefaults sd = step_defaults(*o);
    double t = o->t_start;
    const int n_probe = (int)P.probe.size();
    if (rc == CS_OK) {
        HIPCHK(ctx, hipMemcpyAsync(U.data(), C->w.u, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        launch_charges(C->d_dplan, C->w, C->w.u, C->scratch, s);
        HIPCHK(ctx, hipMemcpyAsync(QH.data(), C->scratch, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipStreamSynchronize(s));
        double T0 = o->t_start, T1 = 0.0, T2 = 0.0;
        int npts = 1;
        double h = sd.dt_init;
        int kout = 0;
        if (wave)
            while (kout < o->n_out && out_due(out_time(o->t_start, kout, o->dt_out), o->t_start, o->dt_out)) {
                for (int s2 = 0; s2 < n_probe; s2++) wave[(size_t)kout * n_probe + s2] = U[P.probe[s2]];
                if (sr)
                    std::copy(sr->S.begin(), sr->S.begin() + (size_t)sr->n_sp * n_probe,
                              sr->out + (size_t)kout * sr->n_sp * n_probe);
                kout++;
            }
        // host copy of the parameter vector for source breakpoints
        std::vector<double> ph(p, p + P.lay.n_params);
        StepDev sp{};
        sp.rtol = o->reltol; sp.atol = o->abstol; sp.tol = o->dc_abstol;
        sp.mode = CS_MODE_TRAN; sp.kind = STEP_TRAN;
        while (t < o->t_stop) {
            if (st.steps + st.rejected >= o->max_steps) { rc = CS_E_MAXSTEPS; break; }
            double tb = INFINITY;
            for (auto& sdsc : P.src) {
                double b = wave_next_bp(sdsc.kind, ph.data() + sdsc.off, sdsc.len, t);
                if (b < tb) tb = b;
            }
            const bool srcbp = tb < o->t_stop;
            if (!srcbp) tb = o->t_stop;
            double hh = h < sd.dt_max ? h : sd.dt_max;
            int hit;
            const double tn = clip_step(t, hh, tb, hit);
            const int k = bdf_order(npts, o->max_order);
            double a0, a1, a2, w0, w1, w2;
            bdf_coeffs(k, tn, T0, T1, a0, a1, a2);
            const int np = npts < k + 1 ? npts : k + 1;
            pred_weights(np, tn, T0, T1, T2, w0, w1, w2);
            for (int i = 0; i < n; i++) {
                double v = U[i];
                if (np == 2) v = w0 * U[i] + w1 * U[n + i];
                else if (np == 3) v = w0 * U[i] + w1 * U[n + i] + w2 * U[2 * n + i];
                up[i] = v;
                q[i] = a1 * QH[i] + (k == 2 ? a2 * QH[n + i] : 0.0);
            }
            sp.a0 = a0;
            sp.t = tn;
            HIPCHK(ctx, hipMemcpyAsync(C->w.u, up, sizeof(double) * n, hipMemcpyHostToDevice, s));
            HIPCHK(ctx, hipMemcpyAsync(C->w.qx, q, sizeof(double) * n, hipMemcpyHostToDevice, s));
            *sph = sp;
            HIPCHK(ctx, hipMemcpyAsync(C->w.sp, sph, sizeof(StepDev), hipMemcpyHostToDevice, s));
            bool conv = false;
            for (int it = 0; it < o->newton_maxit; it++) {
                // modified Newton: the step's first factors for its later iterations
                if ((rc = run_iteration(ctx, *C, it == 0 || !o->jac_reuse))) break;
                st.newton_iters++;
                const double nr = C->h_norm[NRM_WRMS];
                if (!(nr == nr)) break;
                if (nr <= o->newton_tol) { conv = true; break; }
            }
            if (rc) break;
            if (!conv) {
                st.rejected++;
                h = 0.25 * hh;
                if (h < sd.dt_min) { rc = CS_E_DTMIN; break; }
                continue;
            }
            HIPCHK(ctx, hipMemcpyAsync(u, C->w.u, sizeof(double) * n, hipMemcpyDeviceToHost, s));
            launch_charges(C->d_dplan, C->w, C->w.u, C->scratch, s);
            HIPCHK(ctx, hipMemcpyAsync(q, C->scratch, sizeof(double) * n, hipMemcpyDeviceToHost, s));
            HIPCHK(ctx, hipStreamSynchronize(s));
            double fac = 2.0;
            if (npts >= 2) {
                const double c = lte_coeff(k, tn, T0, T1, T2, a0, a1, a2);
                double ss = 0.0;
                for (int i = 0; i < n; i++) {
                    const double est = c * (u[i] - up[i]);
                    const double m = std::max(std::fabs(u[i]), std::fabs(U[i]));
                    const double r = est / (o->reltol * m + o->abstol);
                    ss += r * r;
                }
                const double err = std::sqrt(ss / n);
                if (!(err <= 1.0)) {
                    st.rejected++;
                    h = hh * reject_factor(err, k);
                    if (h < sd.dt_min) { rc = CS_E_DTMIN; break; }
                    continue;
                }
                fac = accept_factor(err, k);
            }
            if (sr) {
                // the accepted point's sensitivities, on the Jacobian at u_m
                if ((rc = sens_solve(ctx, *C, *sr, sp, 0, false, true, k == 2, a1, k == 2 ? a2 : 0.0)) ||
                    (rc = sens_accept(ctx, *C, *sr)))
                    break;
            }
            std::memmove(U.data() + n, U.data(), sizeof(double) * 2 * n);
            std::memcpy(U.data(), u, sizeof(double) * n);
            std::memcpy(QH.data() + n, QH.data(), sizeof(double) * n);
            std::memcpy(QH.data(), q, sizeof(double) * n);
            T2 = T1; T1 = T0; T0 = tn;
            if (npts < 3) npts++;
            st.steps++;
            if (wave) {
                while (kout < o->n_out) {
                    const double tq = out_time(o->t_start, kout, o->dt_out);
                    if (!out_due(tq, tn, o->dt_out)) break;
                    double l0, l1, l2 = 0.0;
                    if (npts >= 3) {
                        l0 = (tq - T1) * (tq - T2) / ((T0 - T1) * (T0 - T2));
                        l1 = (tq - T0) * (tq - T2) / ((T1 - T0) * (T1 - T2));
                        l2 = (tq - T0) * (tq - T1) / ((T2 - T0) * (T2 - T1));
                    } else {
                        const double sl = (tq - T1) / (T0 - T1);
                        l0 = sl;
                        l1 = 1.0 - sl;
                    }
                    for (int s2 = 0; s2 < n_probe; s2++) {
                        const int i = P.probe[s2];
                        wave[(size_t)kout * n_probe + s2] = l0 * U[i] + l1 * U[n + i] + l2 * U[2 * n + i];
                    }
                    if (sr) {
                        const size_t blk = (size_t)sr->n_sp * n_probe;
                        double* so = sr->out + (size_t)kout * blk;
                        for (size_t q = 0; q < blk; q++)
                            so[q] = l0 * sr->S[q] + l1 * sr->S[blk + q] + l2 * sr->S[2 * blk + q];
                    }
                    kout++;
                }
            }
            t = tn;
            h = hh * fac;
            if (hit && srcbp) {
                npts = 1;
                h = 0.1 * h;
                if (h < sd.dt_min) h = sd.dt_min;
            }
        }
    }
    st.t_end = t;
    st.retcode = rc;
    if (u_final) {
        if (st.steps > 0) std::memcpy(u_final, U.data(), sizeof(double) * n);
        else (void)hipMemcpy(u_final, C->w.u, sizeof(double) * n, hipMemcpyDeviceToHost);
    }
    if (st_out) *st_out = st;
    if (rc == CS_E_DTMIN) ctx->err = "transient: step size fell below dt_min";
    else if (rc == CS_E_NOCONV)
        ctx->err = std::string("transient: initial point did not converge") + (uic ? "" : dc_pivot_note(C->plan));
    else if (rc == CS_E_MAXSTEPS) ctx->err = "transient: max_steps reached";
    return rc;
}


// ---- one instance on the LDS-resident kernel ------------------------------------------
// The whole analysis in one launch, where the plain path takes a graph launch
// and a host round trip per Newton iteration.  The context keeps a device
// buffer and a pinned image of its start: one copy up (arguments, parameters,
// initial state), the kernel, one copy down (stats, final state and samples
// of up to kSinglePin bytes).  More samples go straight to the caller's array,
// as far as the run came: an inverter's run with 100 MiB of them took 88 ms
// through a pinned image of their size, 51 so, and the context pins no more
// than the 1 MiB.
struct SingleRun {
    LdsArgs* args;          // in the pinned image
    double *p, *u0;
    cs_tran_stats* st;      // results, in the pinned image
    double *u, *wave;       // (wave null: the samples stay on the device)
    char *d_args, *d_st;
    double* d_wave;
    size_t up, down;        // bytes to copy up; bytes of results to copy down
};

// The buffers outlive the call up to kSingleKeep bytes.  A run whose samples
// need more than kSingleMax stays on the plain path, which writes them
// straight to the caller's array: 17 ns a sample of five values in one launch
// against 8 there, so that an inverter's 1 ns takes 33 against 70 ms with 60
// MiB of them and 145 against 122 with 300.
constexpr size_t kSinglePin = (size_t)1 << 20, kSingleKeep = (size_t)96 << 20, kSingleMax = (size_t)64 << 20;

static void single_free(cs_ctx* ctx) {
    if (ctx->sbuf) (void)hipFree(ctx->sbuf);
    if (ctx->h_sbuf) (void)hipHostFree(ctx->h_sbuf);
    ctx->sbuf = ctx->h_sbuf = nullptr;
    ctx->sbuf_bytes = ctx->h_sbuf_bytes = 0;
}

// The samples a run on one launch has written: those up to the time it
// reached; one that stops early leaves the others.
static int32_t samples_written(const cs_tran_opts& o, int32_t n_out, const cs_tran_stats& st) {
    if (n_out <= 0 || st.retcode == CS_E_NOCONV) return 0;
    const double est = (st.t_end - o.t_start) / o.dt_out;   // off by less than one
    int32_t rows = est > 2.0 ? (int32_t)std::min(est - 2.0, (double)n_out) : 0;
    while (rows < n_out && out_due(out_time(o.t_start, rows, o.dt_out), st.t_end, o.dt_out)) rows++;
    return rows;
}

static int single_buffers(cs_ctx* ctx, Circuit& C, const cs_tran_opts& o, bool with_u0, int32_t n_out, SingleRun& R) {
    const Plan& P = C.plan;
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t off = at; at = (at + bytes + 15) & ~size_t(15); return off; };
    const size_t n_wave = (size_t)n_out * P.probe.size();
    const size_t o_args = take(sizeof(LdsArgs)), o_z = take(64), o_segs = take(2 * sizeof(int4)),
                 o_p = take(sizeof(double) * P.lay.n_params), o_u0 = take(sizeof(double) * P.n);
    R.up = at;
    const size_t o_st = take(sizeof(cs_tran_stats)), o_u = take(sizeof(double) * P.n);
    size_t pinned = at;
    const size_t o_w = take(sizeof(double) * n_wave);
    const bool pin_wave = sizeof(double) * n_wave <= kSinglePin;
    if (pin_wave) pinned = at;
    R.down = pinned - o_st;
    if (at > ctx->sbuf_bytes || pinned > ctx->h_sbuf_bytes) {
        single_free(ctx);
        const size_t bytes = at + at / 4, h_bytes = pinned + pinned / 4;
        if (hipMalloc((void**)&ctx->sbuf, bytes) != hipSuccess ||
            hipHostMalloc((void**)&ctx->h_sbuf, h_bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();   // later launches must not report it
            single_free(ctx);
            return fail(ctx, CS_E_OOM, "no memory for the run's parameters and samples");
        }
        ctx->sbuf_bytes = bytes;
        ctx->h_sbuf_bytes = h_bytes;
    }
    char *h = ctx->h_sbuf, *d = ctx->sbuf;
    std::memset(h, 0, o_p);
    // zeros at o_z: offsets, instance and circuit numbers; then the queue, and
    // the chunk's segment range (0, 1)
    int32_t* z = (int32_t*)(h + o_z);
    z[9] = 1;
    int4* sg = (int4*)(h + o_segs);
    sg[0] = make_int4(0, 0, 1, C.lds_nr);
    sg[1] = make_int4(0, C.hcp.words / 4, (C.hcp.dbl + 1) & ~1, 0);
    R.args = (LdsArgs*)(h + o_args);
    R.p = (double*)(h + o_p);
    R.u0 = (double*)(h + o_u0);
    R.st = (cs_tran_stats*)(h + o_st);
    R.u = (double*)(h + o_u);
    R.wave = pin_wave ? (double*)(h + o_w) : nullptr;
    R.d_args = d + o_args;
    R.d_st = d + o_st;
    R.d_wave = (double*)(d + o_w);
    LdsArgs& a = *R.args;
    a.cplans = C.d_cplan;
    a.plans = C.d_dplan;
    a.inst_cid = (const int32_t*)(d + o_z);
    a.p_off = a.u_off = a.w_off = (const int64_t*)(d + o_z);
    a.params = (const double*)(d + o_p);
    a.u0 = with_u0 ? (const double*)(d + o_u0) : nullptr;
    a.wave = n_wave ? R.d_wave : nullptr;
    a.u_final = (double*)(d + o_u);
    a.stats = (cs_tran_stats*)(d + o_st);
    a.order = (const int32_t*)(d + o_z);
    a.queue = (int32_t*)(d + o_z + 16);
    a.n_inst = 1;
    a.o = o;
    a.o.n_out = n_out;
    a.segs = (const int4*)(d + o_segs);
    a.chunk_seg = (const int32_t*)(d + o_z + 32);
    a.n_chunks = 1;
    return CS_OK;
}

static int tran_single(cs_ctx* ctx, Circuit& C, const double* p, const double* u0, const cs_tran_opts* o,
                       double* wave, double* u_final, cs_tran_stats* st_out) {
    const Plan& P = C.plan;
    if (o->init == CS_INIT_UIC && !u0) return fail(ctx, CS_E_INVALID, "UIC initialisation needs u0");
    if (o->init == CS_INIT_UIC && !P.uic_ok)
        return fail(ctx, CS_E_INVALID, "UIC: a charge-carrying row could not be kept on its own pivot");
    if (o->n_out > 0 && !(o->dt_out > 0)) return fail(ctx, CS_E_INVALID, "dt_out must be > 0");
    (void)hipSetDevice(ctx->device);
    const int32_t n_out = wave ? std::max(o->n_out, 0) : 0;
    std::lock_guard<std::mutex> lock(ctx->single_mu);
    SingleRun R{};
    int rc = single_buffers(ctx, C, *o, u0 != nullptr, n_out, R);
    if (rc) return rc;
    std::memcpy(R.p, p, sizeof(double) * P.lay.n_params);
    if (u0) std::memcpy(R.u0, u0, sizeof(double) * P.n);
    hipStream_t s = ctx->stream;
    PackShape k;
    k.nr = C.lds_nr;
    k.dyn = C.lds_dyn;
    HIPCHK(ctx, hipMemcpyAsync(ctx->sbuf, ctx->h_sbuf, R.up, hipMemcpyHostToDevice, s));
    HIPCHK(ctx, launch_tran_pack(k, (const LdsArgs*)R.d_args, 1, C.lds_bytes, s));
    HIPCHK(ctx, hipMemcpyAsync(R.st, R.d_st, R.down, hipMemcpyDeviceToHost, s));
    HIPCHK(ctx, hipStreamSynchronize(s));
    const size_t got = sizeof(double) * (size_t)samples_written(*o, n_out, *R.st) * P.probe.size();
    if (got && R.wave) std::memcpy(wave, R.wave, got);
    else if (got) HIPCHK(ctx, hipMemcpy(wave, R.d_wave, got, hipMemcpyDeviceToHost));
    if (u_final) std::memcpy(u_final, R.u, sizeof(double) * P.n);
    R.st->busy_s /= ctx->clock_hz;
    if (st_out) *st_out = *R.st;
    rc = R.st->retcode;
    if (ctx->sbuf_bytes > kSingleKeep) single_free(ctx);   // R's pointers end here
    if (rc == CS_E_DTMIN) ctx->err = "transient: step size fell below dt_min";
    else if (rc == CS_E_NOCONV)
        ctx->err = std::string("transient: initial point did not converge") +
                   (o->init == CS_INIT_UIC ? "" : dc_pivot_note(P));
    else if (rc == CS_E_MAXSTEPS) ctx->err = "transient: max_steps reached";
    return rc;
}

// The DC operating point on the same kernel code (k_lds_dcop).
static int dcop_single(cs_ctx* ctx, Circuit& C, const double* p, const cs_tran_opts* o, double* u_out,
                       cs_tran_stats* st) {
    const Plan& P = C.plan;
    std::lock_guard<std::mutex> lock(ctx->single_mu);
    SingleRun R{};
    int rc = single_buffers(ctx, C, *o, false, 0, R);
    if (rc) return rc;
    std::memcpy(R.p, p, sizeof(double) * P.lay.n_params);
    hipStream_t s = ctx->stream;
    HIPCHK(ctx, hipMemcpyAsync(ctx->sbuf, ctx->h_sbuf, R.up, hipMemcpyHostToDevice, s));
    HIPCHK(ctx, launch_lds_dcop(C.lds_nr, C.lds_dyn, (const LdsArgs*)R.d_args, C.lds_bytes, s));
    HIPCHK(ctx, hipMemcpyAsync(R.st, R.d_st, R.down, hipMemcpyDeviceToHost, s));
    HIPCHK(ctx, hipStreamSynchronize(s));
    std::memcpy(u_out, R.u, sizeof(double) * P.n);
    rc = R.st->retcode;
    if (st) {
        std::memset(st, 0, sizeof(*st));
        st->newton_iters = R.st->newton_iters;
        st->retcode = rc;
        st->t_end = o->t_start;
    }
    if (rc == CS_E_NOCONV) ctx->err = "DC operating point analysis failed" + dc_pivot_note(P);
    return rc;
}

int cs_tran(cs_ctx* ctx, int32_t cid, const double* p, const double* u0, const cs_tran_opts* o,
            double* wave, double* u_final, cs_tran_stats* st_out) {
    Circuit* C = get_circuit(ctx, cid);
    if (o && o->batch_kernel == CS_BATCH_KERNEL_LDS) {
        if (!C || !p) return fail(ctx, CS_E_INVALID, "bad argument");
        if (C->big)
            return fail(ctx, CS_E_INVALID,
                        "the LDS-resident kernel runs level-scheduled circuits, not the supernodal solver");
        if (o->jac_reuse)
            return fail(ctx, CS_E_INVALID, "jac_reuse (modified Newton) runs on cs_tran, not in batches");
        if (!C->lds_nr) return fail(ctx, CS_E_RANGE, "LDS-resident batch kernel: " + C->lds_why);
        return tran_single(ctx, *C, p, u0, o, wave, u_final, st_out);
    }
    // AUTO takes the LDS-resident kernel where the circuit fits it: the same
    // rules and step sequence, 5 us per Newton iteration of a small circuit
    // against 90 (an inverter over 4 ns 165 -> 11.9 ms).  Modified Newton,
    // Verilog-A devices and larger circuits stay on the plain path, and
    // CS_BATCH_KERNEL_GLOBAL asks for it.  Without nonlinear devices the
    // factors modified Newton keeps are those full Newton recomputes, so such
    // a circuit takes the same kernel and the same bits either way.
    if (o && C && p && !C->big && C->lds_nr && o->batch_kernel == CS_BATCH_KERNEL_AUTO &&
        (!wave || sizeof(double) * std::max(o->n_out, 0) * C->plan.probe.size() <= kSingleMax) &&
        (o->jac_reuse == 0 || (o->jac_reuse == 1 && C->plan.n_mos == 0))) {
        const int rc = tran_single(ctx, *C, p, u0, o, wave, u_final, st_out);
        if (rc != CS_E_OOM) return rc;   // without memory for its samples: the plain path needs none
    }
    return tran_plain(ctx, cid, p, u0, o, wave, u_final, st_out, nullptr);
}

// A sensitivity run goes in one launch (k_tran_sens) where a wavefront holds
// one unknown per lane, the factors fit the default LDS, and every
// parameter's wavefront is resident at once (four per CU); its samples are
// held on the device up to kSensMax bytes (an inverter's 267 MiB: 63 ms
// against 106 with the host's step control, which costs half as much a sample).  Modified Newton,
// Verilog-A devices and larger circuits keep the host's step control, and
// CS_BATCH_KERNEL_GLOBAL asks for it.
constexpr size_t kSensMax = (size_t)512 << 20;
static bool sens_fits(const cs_ctx* ctx, const Circuit& C, const cs_tran_opts& o, int32_t n_sp) {
    const Plan& P = C.plan;
    return o.batch_kernel == CS_BATCH_KERNEL_AUTO && o.jac_reuse == 0 && P.n_va == 0 && P.n <= kSensMaxN &&
           tran_sens_lds(P.n, P.nnz, P.n_stamp) <= 40 * 1024 && n_sp <= 4 * std::max(ctx->n_cu, 1) &&
           sizeof(double) * std::max(o.n_out, 0) * P.probe.size() * (n_sp + 1) <= kSensMax;
}

static int sens_single(cs_ctx* ctx, Circuit& C, const double* p, const double* u0, const cs_tran_opts* o,
                       const std::vector<SensParam>& sp, double* wave, double* sens, double* u_final,
                       cs_tran_stats* st_out) {
    const Plan& P = C.plan;
    int rc = check_params(ctx, P, p);
    if (rc) return rc;
    const bool uic = o->init == CS_INIT_UIC;
    if (uic && !u0) return fail(ctx, CS_E_INVALID, "UIC initialisation needs u0");
    if (uic && !P.uic_ok)
        return fail(ctx, CS_E_INVALID, "UIC: a charge-carrying row could not be kept on its own pivot");
    if (o->n_out > 0 && !(o->dt_out > 0)) return fail(ctx, CS_E_INVALID, "dt_out must be > 0");
    (void)hipSetDevice(ctx->device);
    const int32_t n = P.n, n_sp = (int32_t)sp.size(), np = (int32_t)P.probe.size(), n_out = std::max(o->n_out, 0);
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t off = at; at = (at + bytes + 255) & ~size_t(255); return off; };
    const size_t blk = (size_t)n_sp * np;
    SensRunArgs a{};
    a.ws_stride = (size_t)P.n_lin + 2 * (size_t)P.nnz;
    const size_t o_sp = take(sizeof(SensParam) * n_sp), o_prow = take(sizeof(int32_t) * n),
                 o_p = take(sizeof(double) * P.lay.n_params), o_u0 = take(sizeof(double) * n),
                 o_ws = take(sizeof(double) * a.ws_stride * n_sp), o_st = take(sizeof(cs_tran_stats)),
                 o_u = take(sizeof(double) * n), o_w = take(sizeof(double) * (size_t)n_out * np),
                 o_s = take(sizeof(double) * (size_t)n_out * blk);
    char* d = nullptr;
    if (hipMalloc((void**)&d, at) != hipSuccess) {
        (void)hipGetLastError();   // later launches must not report it
        return fail(ctx, CS_E_OOM, "no memory for the run's samples");
    }
    a.P = C.d_dplan;
    a.p = (const double*)(d + o_p);
    a.u0 = uic ? (const double*)(d + o_u0) : nullptr;
    a.prow = (const int32_t*)(d + o_prow);
    a.sp = (const SensParam*)(d + o_sp);
    a.ws = (double*)(d + o_ws);
    a.wave = n_out && np ? (double*)(d + o_w) : nullptr;
    a.sens = (double*)(d + o_s);
    a.u_final = (double*)(d + o_u);
    a.stats = (cs_tran_stats*)(d + o_st);
    a.n_sp = n_sp; a.n = n; a.nnz = P.nnz; a.n_lin = P.n_lin; a.n_stamp = P.n_stamp; a.n_probe = np;
    a.o = *o;
    hipStream_t s = ctx->stream;
    cs_tran_stats st{};
    std::vector<double> u(n);
    auto run = [&]() -> int {
        HIPCHK(ctx, hipMemcpyAsync(d + o_sp, sp.data(), sizeof(SensParam) * n_sp, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, hipMemcpyAsync(d + o_prow, P.prow.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, hipMemcpyAsync(d + o_p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
        if (uic) HIPCHK(ctx, hipMemcpyAsync(d + o_u0, u0, sizeof(double) * n, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, launch_tran_sens(a, s));
        HIPCHK(ctx, hipMemcpyAsync(&st, d + o_st, sizeof(st), hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipMemcpyAsync(u.data(), d + o_u, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipStreamSynchronize(s));
        const size_t rows = a.wave ? samples_written(*o, n_out, st) : 0;
        if (rows) {
            HIPCHK(ctx, hipMemcpy(wave, a.wave, sizeof(double) * rows * np, hipMemcpyDeviceToHost));
            HIPCHK(ctx, hipMemcpy(sens, a.sens, sizeof(double) * rows * blk, hipMemcpyDeviceToHost));
        }
        return CS_OK;
    };
    rc = run();
    (void)hipFree(d);
    if (rc) return rc;
    if (u_final) std::memcpy(u_final, u.data(), sizeof(double) * n);
    st.busy_s = 0.0;
    if (st_out) *st_out = st;
    rc = st.retcode;
    if (rc == CS_E_DTMIN) ctx->err = "transient: step size fell below dt_min";
    else if (rc == CS_E_NOCONV)
        ctx->err = std::string("transient: initial point did not converge") + (uic ? "" : dc_pivot_note(P));
    else if (rc == CS_E_MAXSTEPS) ctx->err = "transient: max_steps reached";
    return rc;
}

int cs_tran_sens(cs_ctx* ctx, int32_t cid, const double* p, const double* u0, const cs_tran_opts* o,
                 int32_t n_sp, const int32_t* sp_idx, double* wave, double* sens, double* u_final,
                 cs_tran_stats* st_out) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !o || n_sp <= 0 || !sp_idx || !sens || !wave) return fail(ctx, CS_E_INVALID, "bad argument");
    if (C->big) return fail(ctx, CS_E_INVALID, "sensitivities run on the level-scheduled plan, not the supernodal solver");
    const Plan& P = C->plan;
    SensRun R;
    R.n_sp = n_sp;
    R.out = sens;
    R.sp.resize(n_sp);
    for (int32_t j = 0; j < n_sp; j++) {
        if (sp_idx[j] < 0 || sp_idx[j] >= P.lay.n_params || !sens_param(P, sp_idx[j], R.sp[j]))
            return fail(ctx, CS_E_INVALID, "parameter " + std::to_string(sp_idx[j]) +
                        " has no sensitivity on this path (R, C, L, VCCS/VCVS gains, MOSFET vth/kp/w/l, "
                        "source DC values)");
        R.sp[j].val = p ? p[sp_idx[j]] : 0.0;
    }
    if (!p) return fail(ctx, CS_E_INVALID, "bad argument");
    if (sens_fits(ctx, *C, *o, n_sp)) {
        const int rs = sens_single(ctx, *C, p, u0, o, R.sp, wave, sens, u_final, st_out);
        if (rs != CS_E_OOM) return rs;   // without memory for its samples: the host's step control needs none
    }
    const int n = P.n, np = (int)P.probe.size();
    R.S.assign(3 * (size_t)n_sp * np, 0.0);
    R.s_nat.assign((size_t)n_sp * n, 0.0);
    (void)hipSetDevice(ctx->device);
    const size_t vec = sizeof(double) * (size_t)n_sp * n;
    const size_t o_sp = 0, o_prow = (sizeof(SensParam) * n_sp + 255) & ~size_t(255);
    const size_t o_vec = (o_prow + sizeof(int32_t) * n + 255) & ~size_t(255);
    const size_t bytes = o_vec + 7 * vec;
    HIPCHK(ctx, hipMalloc(&R.buf, bytes));
    R.d_sp = (SensParam*)(R.buf + o_sp);
    R.d_prow = (int32_t*)(R.buf + o_prow);
    double* v = (double*)(R.buf + o_vec);
    const size_t nv = (size_t)n_sp * n;
    R.d_pin = v; R.d_x = v + nv; R.d_s = v + 2 * nv;
    R.d_dq[0] = v + 3 * nv; R.d_dq[1] = v + 4 * nv; R.d_dq[2] = v + 5 * nv;
    int rc = CS_OK;
    if (hipMemcpy(R.d_sp, R.sp.data(), sizeof(SensParam) * n_sp, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(R.d_prow, P.prow.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(v, 0, 7 * vec) != hipSuccess)
        rc = fail(ctx, CS_E_HIP, "sensitivity buffers");
    if (rc == CS_OK) rc = tran_plain(ctx, cid, p, u0, o, wave, u_final, st_out, &R);
    (void)hipFree(R.buf);
    return rc;
}

// The arguments every LDS-resident launch of a batch shares.
static int lds_base_args(cs_ctx* ctx, const Batch& B, const std::function<int(void**, size_t)>& dalloc, LdsArgs& a) {
    std::vector<CPlan> cplans(ctx->circuits.size());
    for (size_t c = 0; c < ctx->circuits.size(); c++)
        if (ctx->circuits[c] && ctx->circuits[c]->compact_ok) cplans[c] = ctx->circuits[c]->hcp;
    void* d_cp = nullptr;
    int rc;
    if ((rc = dalloc(&d_cp, sizeof(CPlan) * cplans.size()))) return rc;
    HIPCHK(ctx, hipMemcpy(d_cp, cplans.data(), sizeof(CPlan) * cplans.size(), hipMemcpyHostToDevice));
    const BatchArgs& g = B.args;
    a = LdsArgs{};
    a.cplans = (const CPlan*)d_cp;
    a.plans = g.plans;
    a.inst_cid = g.inst_cid;
    a.p_off = g.p_off;
    a.params = g.params;
    a.u_off = g.u_off;
    a.u0 = g.u0;
    a.w_off = g.w_off;
    a.wave = g.wave;
    a.u_final = g.u_final;
    a.stats = g.stats;
    a.o = g.o;
    return CS_OK;
}

// Size classes of the adjoint.  Circuits are sorted by LDS footprint; a class
// takes circuits down to 3/4 of its largest footprint, so small circuits are
// not launched with the largest circuit's LDS reservation.  Each class is one
// persistent launch with its own largest-first queue.
static int build_lds_classes(cs_ctx* ctx, Batch& B, const std::function<int(void**, size_t)>& dalloc) {
    auto need = [&](int32_t c) {
        const CPlan& cp = ctx->circuits[c]->hcp;
        return lds_kernel_bytes((cp.dbl + 1) & ~1, cp.words_adj);
    };
    std::vector<int32_t> cs = B.used;
    std::stable_sort(cs.begin(), cs.end(), [&](int32_t a, int32_t b) { return need(a) > need(b); });
    std::vector<int32_t> cls_of(ctx->circuits.size(), -1);
    std::vector<std::vector<int32_t>> members;
    for (size_t q = 0; q < cs.size();) {
        const size_t cap = need(cs[q]);
        std::vector<int32_t> m;
        while (q < cs.size() && 4 * need(cs[q]) >= 3 * cap) m.push_back(cs[q++]);
        for (int32_t c : m) cls_of[c] = (int32_t)members.size();
        members.push_back(m);
    }
    LdsArgs base{};
    void* d_q = nullptr;
    int rc;
    if ((rc = lds_base_args(ctx, B, dalloc, base)) || (rc = dalloc(&d_q, sizeof(int32_t) * members.size()))) return rc;
    B.d_queues = (int32_t*)d_q;
    for (size_t k = 0; k < members.size(); k++) {
        LdsClass L;
        int32_t dbl_max = 2, words_max[2] = {8, 8};
        for (int32_t c : members[k]) {
            const CPlan& cp = ctx->circuits[c]->hcp;
            dbl_max = std::max(dbl_max, (cp.dbl + 1) & ~1);
            words_max[0] = std::max(words_max[0], cp.words);
            words_max[1] = std::max(words_max[1], cp.words_adj);
            L.nr = std::max(L.nr, B.c_nr[c]);
            L.dyn = L.dyn || ctx->circuits[c]->lds_dyn;
        }
        std::vector<int32_t> order;
        for (int32_t i = 0; i < B.n_inst; i++)
            if (cls_of[B.cid[i]] == (int32_t)k) order.push_back(i);
        std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return need(B.cid[a]) > need(B.cid[b]); });
        void* d_order = nullptr;
        if ((rc = dalloc(&d_order, sizeof(int32_t) * order.size()))) return rc;
        HIPCHK(ctx, hipMemcpy(d_order, order.data(), sizeof(int32_t) * order.size(), hipMemcpyHostToDevice));
        L.n_inst = (int32_t)order.size();
        for (int r = 0; r < 2; r++) L.lds[r] = lds_kernel_bytes(dbl_max, words_max[r]);
        L.args = base;
        L.args.order = (const int32_t*)d_order;
        L.args.queue = B.d_queues + k;
        L.args.n_inst = L.n_inst;
        L.args.dbl_max = dbl_max;
        B.classes.push_back(L);
    }
    while (ctx->side.size() < kSideStreams) {
        hipStream_t st;
        HIPCHK(ctx, hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        ctx->side.push_back(st);
    }
    const size_t nev = std::min(B.classes.size(), kSideStreams);
    for (size_t k = 0; k < nev; k++) {
        hipEvent_t e;
        HIPCHK(ctx, hipEventCreate(&e));
        B.class_ev.push_back(e);
    }
    return CS_OK;
}

// The packed launch.  A chunk fills one workgroup: up to kPackWaves
// wavefronts in up to kPackSegs segments, each a run of one circuit's
// instances beside that circuit's plan image, within kPackLds bytes of LDS.
// Packing (greedy, largest circuit first): a chunk takes as many instances
// of the largest circuit left as fit, and fills the rest of its wavefronts
// and LDS from the smallest circuits left; of the counts of the large
// circuit that fit, it keeps the one that fills the most wavefronts.  Large
// circuits are LDS-bound (a few instances beside their image) and small ones
// slot-bound, so mixing them lets every instance of a batch like the ring
// Monte Carlo be resident at once.  A batch that does not fill the device is
// spread over its CUs instead: a chunk takes no more instances than there
// would be per CU, since wavefronts on one CU share its LDS and issue ports
// (60 rings over 500 ps: 8 CUs at 8 wavefronts each before).  A workgroup has
// the wavefronts of the fullest chunk, no more: where LDS holds only a few
// instances, idle ones would keep a second workgroup off the CU.  Returns
// CS_E_RANGE when a circuit does not fit even one wavefront beside its image.
static int build_pack(cs_ctx* ctx, Batch& B, const std::function<int(void**, size_t)>& dalloc) {
    const std::vector<int32_t>&used = B.used, &c_nr = B.c_nr;
    const size_t nc = ctx->circuits.size();
    std::vector<int32_t> cs = used;
    std::stable_sort(cs.begin(), cs.end(), [&](int32_t a, int32_t b) {
        const CPlan &x = ctx->circuits[a]->hcp, &y = ctx->circuits[b]->hcp;
        return x.dbl != y.dbl ? x.dbl > y.dbl : x.n > y.n;
    });
    std::vector<size_t> img(nc, 0), dblb(nc, 0);
    PackShape& ks = B.pack;
    ks = PackShape{};
    ks.dyn = false;
    for (int32_t c : cs) {
        const CPlan& cp = ctx->circuits[c]->hcp;
        img[c] = 2 * (size_t)((cp.words + 7) & ~7);
        dblb[c] = 8 * (size_t)((cp.dbl + 1) & ~1);
        if (img[c] + dblb[c] > kPackLds) return CS_E_RANGE;
        ks.nr = std::max(ks.nr, c_nr[c]);
        ks.dyn = ks.dyn || ctx->circuits[c]->lds_dyn;
    }
    const int64_t n_cu = std::max(ctx->n_cu, 1);
    const int32_t spread = (int32_t)std::min<int64_t>(kPackWaves, (B.n_inst + n_cu - 1) / n_cu);
    std::vector<std::vector<int32_t>> per(nc);
    for (int32_t i = 0; i < B.n_inst; i++) per[B.cid[i]].push_back(i);
    std::vector<size_t> rem(nc, 0), next(nc, 0);
    for (int32_t c : cs) rem[c] = per[c].size();
    size_t need = 0;
    const std::vector<std::vector<PackSeg>> chunks = pack_chunks(cs, img, dblb, rem, spread, kPackSegs, kPackLds, &need);
    if (chunks.empty() && B.n_inst > 0) return CS_E_RANGE;
    const size_t C = chunks.size();
    for (const auto& ch : chunks) {
        int32_t cnt = 0;
        for (const PackSeg& g : ch) cnt += g.cnt;
        ks.waves = std::max(ks.waves, cnt);
    }
    int per_cu = pack_max_blocks(ks, need);
    // the registers for four wavefronts per SIMD where the batch has more than
    // two, or where only they hold every chunk at once
    if (ks.nr <= 2) {
        PackShape k4 = ks;
        k4.occ = 4;
        const int per_cu4 = pack_max_blocks(k4, need);
        if (B.n_inst > kPackWaves * n_cu || ((int64_t)C > per_cu * n_cu && per_cu4 > per_cu)) {
            ks = k4;
            per_cu = per_cu4;
        }
    }
    if (per_cu <= 0) return fail(ctx, CS_E_RANGE, "packed LDS kernel does not fit on a CU");
    // When the chunks outnumber the resident workgroups by E, the E extra
    // chunks start when the first workgroups finish.  The chunks come largest
    // circuit first, and a larger circuit takes longer; so the queue puts the
    // E smallest chunks first (ascending), then the large ones, then the next
    // E smallest (descending): the workgroups that finish first take a second
    // small chunk, the largest of those first, instead of a large chunk being
    // followed by a small one.
    B.pack_blocks = (int32_t)std::min<int64_t>((int64_t)C, per_cu * n_cu);
    std::vector<size_t> qorder(C);
    for (size_t i = 0; i < C; i++) qorder[i] = i;
    {
        const size_t E = C - (size_t)B.pack_blocks;
        if (E > 0 && 2 * E <= C) {
            qorder.clear();
            for (size_t i = 0; i < E; i++) qorder.push_back(C - 1 - i);
            for (size_t i = 0; i < C - 2 * E; i++) qorder.push_back(i);
            for (size_t i = C - 2 * E; i < C - E; i++) qorder.push_back(i);
        }
    }
    // segments in queue order, with their LDS offsets
    std::vector<int32_t> order, chunk_seg{0};
    std::vector<int4> segs;
    for (size_t qi : qorder) {
        const std::vector<PackSeg>& ch = chunks[qi];
        size_t words = 0, regions = 0;
        for (const PackSeg& g : ch) words += img[g.c] / 2;
        int32_t w0 = 0;
        for (const PackSeg& g : ch) {
            segs.push_back(make_int4(g.c, (int32_t)order.size(), g.cnt, c_nr[g.c]));
            order.insert(order.end(), per[g.c].begin() + next[g.c], per[g.c].begin() + next[g.c] + g.cnt);
            next[g.c] += g.cnt;
            const int32_t stride = (int32_t)(dblb[g.c] / 8);
            segs.push_back(make_int4(0, (int32_t)(words / 4 + regions), stride, w0));
            regions += (size_t)g.cnt * stride;
            w0 += g.cnt;
        }
        // image word offsets
        size_t off = 0;
        for (size_t j = 0; j < ch.size(); j++) {
            segs[segs.size() - 2 * ch.size() + 2 * j + 1].x = (int32_t)off;
            off += img[ch[j].c] / 2;
        }
        chunk_seg.push_back((int32_t)(segs.size() / 2));
    }
    if ((int32_t)order.size() != B.n_inst) return fail(ctx, CS_E_INVALID, "packing lost instances");
    void *d_order, *d_segs, *d_cseg, *d_q, *d_args;
    int rc;
    if ((rc = dalloc(&d_order, sizeof(int32_t) * order.size())) ||
        (rc = dalloc(&d_segs, sizeof(int4) * segs.size())) ||
        (rc = dalloc(&d_cseg, sizeof(int32_t) * chunk_seg.size())) || (rc = dalloc(&d_q, sizeof(int32_t))) ||
        (rc = dalloc(&d_args, sizeof(LdsArgs))))
        return rc;
    B.pack_lds = need;
    HIPCHK(ctx, hipMemcpy(d_order, order.data(), sizeof(int32_t) * order.size(), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_segs, segs.data(), sizeof(int4) * segs.size(), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_cseg, chunk_seg.data(), sizeof(int32_t) * chunk_seg.size(), hipMemcpyHostToDevice));
    LdsArgs& a = B.pack_args;
    if ((rc = lds_base_args(ctx, B, dalloc, a))) return rc;
    a.order = (const int32_t*)d_order;
    a.queue = (int32_t*)d_q;
    a.n_inst = B.n_inst;
    a.dbl_max = 0;
    a.segs = (const int4*)d_segs;
    a.chunk_seg = (const int32_t*)d_cseg;
    a.n_chunks = (int32_t)C;
    HIPCHK(ctx, hipMemcpy(d_args, &a, sizeof(LdsArgs), hipMemcpyHostToDevice));
    B.d_pack_args = (const LdsArgs*)d_args;
    return CS_OK;
}

// ---- batched transient --------------------------------------------------------------
int cs_batch_create(cs_ctx* ctx, int32_t n_inst, const int32_t* inst_cid, const double* params,
                    const double* u0, const cs_tran_opts* o, int32_t* bid) {
    if (!ctx || n_inst <= 0 || !inst_cid || !params || !o || !bid)
        return fail(ctx, CS_E_INVALID, "bad argument");
    if (o->init == CS_INIT_UIC && !u0) return fail(ctx, CS_E_INVALID, "UIC initialisation needs u0");
    if (o->n_out > 0 && !(o->dt_out > 0)) return fail(ctx, CS_E_INVALID, "dt_out must be > 0");
    (void)hipSetDevice(ctx->device);
    auto B = std::make_unique<Batch>();
    B->n_inst = n_inst;
    B->cid.assign(inst_cid, inst_cid + n_inst);
    int64_t po = 0, uo = 0, wo = 0;
    int32_t nnz_max = 1, n_max = 1, st_max = 1, lin_max = 1, np_max = 0;
    std::vector<DPlan> plans(ctx->circuits.size());
    for (size_t c = 0; c < ctx->circuits.size(); c++)
        if (ctx->circuits[c]) plans[c] = ctx->circuits[c]->hd;
    for (int32_t i = 0; i < n_inst; i++) {
        Circuit* C = get_circuit(ctx, inst_cid[i]);
        if (!C) return fail(ctx, CS_E_INVALID, "bad circuit id in batch");
        if (C->big) return fail(ctx, CS_E_INVALID, "supernodal circuits run on cs_tran, not in batches");
        const Plan& P = C->plan;
        if (o->init == CS_INIT_UIC && !P.uic_ok)
            return fail(ctx, CS_E_INVALID, "UIC: a charge-carrying row could not be kept on its own pivot");
        B->p_off.push_back(po);
        B->u_off.push_back(uo);
        B->w_off.push_back(wo);
        po += P.lay.n_params;
        uo += P.n;
        wo += (int64_t)o->n_out * (int64_t)P.probe.size();
        B->has_va = B->has_va || P.n_va > 0;
        nnz_max = std::max(nnz_max, P.nnz);
        n_max = std::max(n_max, P.n);
        st_max = std::max(st_max, P.n_stamp);
        lin_max = std::max(lin_max, P.n_lin);
        np_max = std::max<int32_t>(np_max, (int32_t)P.probe.size());
    }
    // ---- kernel choice: the LDS-resident kernel when every circuit fits ----
    const int32_t want = o->batch_kernel;
    if (want < CS_BATCH_KERNEL_AUTO || want > CS_BATCH_KERNEL_GLOBAL)
        return fail(ctx, CS_E_INVALID, "unknown batch_kernel");
    if (o->jac_reuse)
        return fail(ctx, CS_E_INVALID, "jac_reuse (modified Newton) runs on cs_tran, not in batches");
    std::vector<int32_t> used;
    {
        std::vector<char> seen(ctx->circuits.size(), 0);
        for (int32_t i = 0; i < n_inst; i++)
            if (!seen[inst_cid[i]]) { seen[inst_cid[i]] = 1; used.push_back(inst_cid[i]); }
    }
    std::string lds_why;
    std::vector<int32_t> c_nr(ctx->circuits.size(), 0);
    bool lds_fits = true;
    for (int32_t c : used) {
        const Circuit& C = *ctx->circuits[c];
        if (!C.lds_nr) { lds_fits = false; lds_why = C.lds_why; break; }
        c_nr[c] = C.lds_nr;
    }
    if (want == CS_BATCH_KERNEL_LDS && !lds_fits)
        return fail(ctx, CS_E_RANGE, "LDS-resident batch kernel: " + lds_why);
    B->kernel = (want != CS_BATCH_KERNEL_GLOBAL && lds_fits) ? CS_BATCH_KERNEL_LDS : CS_BATCH_KERNEL_GLOBAL;
    if (B->kernel == CS_BATCH_KERNEL_GLOBAL && n_max > 64 * 8)
        return fail(ctx, CS_E_RANGE, "batched path supports up to 512 unknowns per instance; use cs_tran");
    B->nr = n_max <= 64 ? 1 : n_max <= 128 ? 2 : n_max <= 256 ? 4 : 8;
    B->u_len = uo;
    B->wave_len = wo;
    // largest-first queue order (longest per-iteration work first)
    std::vector<int32_t> order(n_inst);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        return ctx->circuits[inst_cid[a]]->plan.nnz > ctx->circuits[inst_cid[b]]->plan.nnz;
    });
    auto dalloc = [&](void** p, size_t bytes) -> int {
        hipError_t e = hipMalloc(p, std::max<size_t>(bytes, 16));
        if (e != hipSuccess) return fail(ctx, CS_E_OOM, "batch allocation failed");
        B->allocs.push_back(*p);
        return CS_OK;
    };
    BatchArgs& A = B->args;
    int rc;
    void *d_plans, *d_cid, *d_poff, *d_params, *d_uoff, *d_u0 = nullptr, *d_woff, *d_wave = nullptr,
                                                    *d_uf, *d_st, *d_order, *d_queue;
    if ((rc = dalloc(&d_plans, sizeof(DPlan) * plans.size())) ||
        (rc = dalloc(&d_cid, sizeof(int32_t) * n_inst)) ||
        (rc = dalloc(&d_poff, sizeof(int64_t) * n_inst)) ||
        (rc = dalloc(&d_params, sizeof(double) * po)) ||
        (rc = dalloc(&d_uoff, sizeof(int64_t) * n_inst)) ||
        (rc = dalloc(&d_woff, sizeof(int64_t) * n_inst)) ||
        (rc = dalloc(&d_uf, sizeof(double) * uo)) ||
        (rc = dalloc(&d_st, sizeof(cs_tran_stats) * n_inst)) ||
        (rc = dalloc(&d_order, sizeof(int32_t) * n_inst)) ||
        (rc = dalloc(&d_queue, sizeof(int32_t))))
        return rc;
    if (u0 && (rc = dalloc(&d_u0, sizeof(double) * uo))) return rc;
    if (wo > 0 && (rc = dalloc(&d_wave, sizeof(double) * wo))) return rc;
    HIPCHK(ctx, hipMemcpy(d_plans, plans.data(), sizeof(DPlan) * plans.size(), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_cid, inst_cid, sizeof(int32_t) * n_inst, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_poff, B->p_off.data(), sizeof(int64_t) * n_inst, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_params, params, sizeof(double) * po, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_uoff, B->u_off.data(), sizeof(int64_t) * n_inst, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_woff, B->w_off.data(), sizeof(int64_t) * n_inst, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_order, order.data(), sizeof(int32_t) * n_inst, hipMemcpyHostToDevice));
    if (u0) HIPCHK(ctx, hipMemcpy(d_u0, u0, sizeof(double) * uo, hipMemcpyHostToDevice));
    A.plans = (const DPlan*)d_plans;
    A.inst_cid = (const int32_t*)d_cid;
    A.p_off = (const int64_t*)d_poff;
    A.params = (const double*)d_params;
    A.u_off = (const int64_t*)d_uoff;
    A.u0 = (const double*)d_u0;
    A.w_off = (const int64_t*)d_woff;
    A.wave = (double*)d_wave;
    A.u_final = (double*)d_uf;
    A.stats = (cs_tran_stats*)d_st;
    A.order = (const int32_t*)d_order;
    A.queue = (int32_t*)d_queue;
    A.n_inst = n_inst;
    A.nnz_max = nnz_max;
    A.n_max = n_max;
    A.stamp_max = st_max;
    A.lin_max = lin_max;
    A.n_probe_max = np_max;
    A.o = *o;
    if (B->kernel == CS_BATCH_KERNEL_GLOBAL) {
        B->lds = batch_lds_bytes(A);
        int per_cu = batch_max_blocks(B->nr, B->has_va, B->lds);
        if (per_cu <= 0) return fail(ctx, CS_E_RANGE, "batched kernel does not fit: LDS per instance too large");
        B->nblocks = std::min<int64_t>(n_inst, (int64_t)per_cu * std::max(ctx->n_cu, 1));
        void *d_g, *d_c, *d_l;
        if ((rc = dalloc(&d_g, sizeof(double) * (size_t)B->nblocks * nnz_max)) ||
            (rc = dalloc(&d_c, sizeof(double) * (size_t)B->nblocks * nnz_max)) ||
            (rc = dalloc(&d_l, sizeof(double) * (size_t)B->nblocks * lin_max)))
            return rc;
        A.glin = (double*)d_g;
        A.clin = (double*)d_c;
        A.linbuf = (double*)d_l;
    } else {
        B->used = used;
        B->c_nr = c_nr;
        if ((rc = build_pack(ctx, *B, dalloc)) != CS_OK)
            return rc == CS_E_RANGE ? fail(ctx, rc, "a circuit does not fit the packed LDS kernel") : rc;
    }
    HIPCHK(ctx, hipEventCreate(&B->ev0));
    HIPCHK(ctx, hipEventCreate(&B->ev1));
    ctx->batches.push_back(std::move(B));
    *bid = (int32_t)ctx->batches.size() - 1;
    return CS_OK;
}

static Batch* get_batch(cs_ctx* ctx, int32_t bid) {
    if (!ctx || bid < 0 || bid >= (int32_t)ctx->batches.size() || !ctx->batches[bid]) return nullptr;
    return ctx->batches[bid].get();
}

int cs_batch_run(cs_ctx* ctx, int32_t bid, double* kernel_ms) {
    Batch* B = get_batch(ctx, bid);
    if (!B) return fail(ctx, CS_E_INVALID, "bad batch id");
    (void)hipSetDevice(ctx->device);
    hipStream_t s = ctx->stream;
    if (B->kernel == CS_BATCH_KERNEL_GLOBAL) {
        HIPCHK(ctx, hipMemsetAsync(B->args.queue, 0, sizeof(int32_t), s));
        HIPCHK(ctx, hipEventRecord(B->ev0, s));
        HIPCHK(ctx, launch_tran_batch(B->nr, B->has_va, B->args, B->nblocks, B->lds, s));
        HIPCHK(ctx, hipEventRecord(B->ev1, s));
    } else {
        HIPCHK(ctx, hipMemsetAsync(B->pack_args.queue, 0, sizeof(int32_t), s));
        HIPCHK(ctx, hipEventRecord(B->ev0, s));
        HIPCHK(ctx, launch_tran_pack(B->pack, B->d_pack_args, B->pack_blocks, B->pack_lds, s));
        HIPCHK(ctx, hipEventRecord(B->ev1, s));
    }
    HIPCHK(ctx, hipEventSynchronize(B->ev1));
    float ms = 0.f;
    HIPCHK(ctx, hipEventElapsedTime(&ms, B->ev0, B->ev1));
    B->last_ms = ms;
    if (kernel_ms) *kernel_ms = ms;
    return CS_OK;
}

int cs_batch_results(cs_ctx* ctx, int32_t bid, double* wave, double* u_final, cs_tran_stats* st) {
    Batch* B = get_batch(ctx, bid);
    if (!B) return fail(ctx, CS_E_INVALID, "bad batch id");
    (void)hipSetDevice(ctx->device);
    if (wave && B->wave_len)
        HIPCHK(ctx, hipMemcpy(wave, B->args.wave, sizeof(double) * B->wave_len, hipMemcpyDeviceToHost));
    if (u_final)
        HIPCHK(ctx, hipMemcpy(u_final, B->args.u_final, sizeof(double) * B->u_len, hipMemcpyDeviceToHost));
    if (st) {
        HIPCHK(ctx, hipMemcpy(st, B->args.stats, sizeof(cs_tran_stats) * B->n_inst, hipMemcpyDeviceToHost));
        for (int32_t i = 0; i < B->n_inst; i++)
            st[i].busy_s = B->kernel == CS_BATCH_KERNEL_LDS ? st[i].busy_s / ctx->clock_hz : 0.0;
    }
    return CS_OK;
}

int cs_batch_destroy(cs_ctx* ctx, int32_t bid) {
    Batch* B = get_batch(ctx, bid);
    if (!B) return fail(ctx, CS_E_INVALID, "bad batch id");
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (void* p : B->allocs) (void)hipFree(p);
    if (B->ev0) (void)hipEventDestroy(B->ev0);
    if (B->ev1) (void)hipEventDestroy(B->ev1);
    for (hipEvent_t e : B->class_ev) (void)hipEventDestroy(e);
    ctx->batches[bid].reset();
    return CS_OK;
}

int cs_lds_probe(cs_ctx* ctx, int32_t cid, int32_t nr, const double* p, const double* u,
                 const double* qx, double a0, double t, int32_t mode, double* jac, double* res,
                 double* lu, double* dx) {
    Circuit* C = get_circuit(ctx, cid);
    if (!C || !p || !u || !qx) return fail(ctx, CS_E_INVALID, "bad argument");
    if (C->big || !C->compact_ok)
        return fail(ctx, CS_E_INVALID, "circuit does not run on the LDS-resident kernel");
    const CPlan& cp = C->hcp;
    if (nr == 0) {
        nr = cp.n <= 64 ? 1 : cp.n <= 128 ? 2 : 4;
        while (nr < 4 && cp.n_mos > 128 * nr) nr *= 2;
    }
    if ((nr != 1 && nr != 2 && nr != 4) || cp.n > 64 * nr || cp.n_mos > 128 * nr)
        return fail(ctx, CS_E_RANGE, "rows per lane too small for this circuit");
    const size_t lds = lds_kernel_bytes((cp.dbl + 1) & ~1, cp.words);
    if (lds > kLdsMaxBytes) return fail(ctx, CS_E_RANGE, "circuit needs more LDS than one workgroup may hold");
    (void)hipSetDevice(ctx->device);
    const Plan& P = C->plan;
    const int32_t n = P.n, nnz = P.nnz;
    std::vector<double> up(n), qp(n);
    for (int32_t r = 0; r < n; r++) {
        up[P.pcol[r]] = u[r];
        qp[P.prow[r]] = qx[r];
    }
    const size_t nb = sizeof(CPlan) + sizeof(double) * ((size_t)P.lay.n_params + 4 * (size_t)n + 2 * (size_t)nnz) + 256;
    char* buf = nullptr;
    HIPCHK(ctx, hipMalloc(&buf, nb));
    CPlan* d_cp = (CPlan*)buf;
    double* d = (double*)(buf + ((sizeof(CPlan) + 15) & ~size_t(15)));
    double *d_p = d, *d_u = d_p + P.lay.n_params, *d_q = d_u + n, *d_fa = d_q + n, *d_r = d_fa + nnz,
           *d_fl = d_r + n, *d_x = d_fl + nnz;
    hipStream_t s = ctx->stream;
    int rc = CS_OK;
    std::vector<double> fa(nnz), rp(n), fl(nnz), xp(n);
    auto run = [&]() -> int {
        HIPCHK(ctx, hipMemcpyAsync(d_cp, &cp, sizeof(CPlan), hipMemcpyHostToDevice, s));
        HIPCHK(ctx, hipMemcpyAsync(d_p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, hipMemcpyAsync(d_u, up.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, hipMemcpyAsync(d_q, qp.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        HIPCHK(ctx, launch_lds_probe(nr, d_cp, C->d_dplan, d_p, d_u, d_q, a0, t, mode, d_fa, d_r, d_fl, d_x,
                                     lds, s));
        HIPCHK(ctx, hipMemcpyAsync(fa.data(), d_fa, sizeof(double) * nnz, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipMemcpyAsync(rp.data(), d_r, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipMemcpyAsync(fl.data(), d_fl, sizeof(double) * nnz, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipMemcpyAsync(xp.data(), d_x, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipStreamSynchronize(s));
        return CS_OK;
    };
    rc = run();
    (void)hipFree(buf);
    if (rc) return rc;
    if (jac)
        for (int32_t q = 0; q < P.nnz_nat; q++) jac[q] = fa[P.nat_fpos[q]];
    if (res)
        for (int32_t r = 0; r < n; r++) res[r] = rp[P.prow[r]];
    if (lu) std::copy(fl.begin(), fl.end(), lu);
    if (dx)
        for (int32_t r = 0; r < n; r++) dx[r] = xp[P.pcol[r]];
    return CS_OK;
}

// ---- small-signal AC and noise (src/ac.jl) ----------------------------------------
namespace {

// G = dF/du at the DC point (DC mode, a0 = 0: the assembled Jacobian with
// the device stamps) into C.w.F and C = dQ/du into C.w.Clin, both on the F
// pattern.  Only linear charges exist on this path (a Verilog-A model with
// charges is rejected at load), so dQ/du is the linear C.
int ac_operands(cs_ctx* ctx, Circuit& C, const double* p, const double* u_dc) {
    int rc = ensure_workspace(ctx, C);
    if (rc) return rc;
    const Plan& P = C.plan;
    hipStream_t s = ctx->stream;
    HIPCHK(ctx, hipMemcpyAsync(C.w.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
    HIPCHK(ctx, hipMemcpyAsync(C.w.u, u_dc, sizeof(double) * P.n, hipMemcpyHostToDevice, s));
    launch_lin_setup(C.d_dplan, C.w, s);
    StepDev sp{};
    sp.t = 0.0;
    sp.mode = CS_MODE_DCOP;
    sp.kind = STEP_DC;
    sp.a0 = 0.0;
    HIPCHK(ctx, hipMemsetAsync(C.w.qx, 0, sizeof(double) * P.n, s));
    if ((rc = set_step(ctx, C, sp))) return rc;
    launch_eval_assemble(C.d_dplan, C.w, s);
    return CS_OK;
}

// One sweep of k_ac over n_freq frequencies with the operands in C.w: the
// workspace (one complex F, inv and x per workgroup), the frequencies and
// the per-analysis arrays in one allocation, freed before returning.
int ac_sweep(cs_ctx* ctx, Circuit& C, AcArgs a, const double* omega, const std::vector<double>& rhs,
             const std::vector<int32_t>& obs_piv, const std::vector<int32_t>& nz_rows,
             const std::vector<double>& nz_pwr, const std::vector<double>& nz_exp, double* out, double* psd) {
    const Plan& P = C.plan;
    // a frequency in LDS where at least two fit a CU, else in the workspace.
    // Those circuits have few hundred unknowns at most: one wavefront (four
    // measured the same on a 12 x 11 mesh)
    const size_t fit = ac_lds(P.n, P.nnz);
    const size_t lds = P.n <= 512 && fit <= 76 * 1024 ? fit : 0;
    const size_t stride = lds ? 0 : 2 * (size_t)P.nnz + 4 * (size_t)P.n + 2;
    const size_t budget = (size_t)1 << 28;   // doubles of workspace: 2 GiB
    int64_t nblocks = std::min<int64_t>(a.n_freq, std::max<int64_t>(4 * std::max(ctx->n_cu, 1), 1));
    nblocks = std::max<int64_t>(1, std::min<int64_t>(nblocks, (int64_t)(budget / std::max<size_t>(stride, 1))));
    Packer pk;
    std::vector<double> om(omega, omega + a.n_freq);
    const size_t o_om = pk.add(om), o_rhs = pk.add(rhs), o_obs = pk.add(obs_piv), o_nr = pk.add(nz_rows),
                 o_np = pk.add(nz_pwr), o_ne = pk.add(nz_exp);
    const size_t n_out = a.transposed ? (size_t)a.n_freq : 2 * (size_t)a.n_freq * std::max(a.n_obs, 1);
    const size_t n_out_al = (n_out + 1) & ~size_t(1);   // the workspace after it holds double2
    const size_t head = (pk.bytes.size() + 255) & ~size_t(255);
    const size_t bytes = head + sizeof(double) * (n_out_al + stride * (size_t)nblocks);
    char* buf = nullptr;
    HIPCHK(ctx, hipMalloc(&buf, bytes));
    hipStream_t s = ctx->stream;
    int rc = CS_OK;
    auto run = [&]() -> int {
        HIPCHK(ctx, hipMemcpyAsync(buf, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice, s));
        double* d_out = (double*)(buf + head);
        a.P = C.d_dplan;
        a.G = C.w.F;
        a.Cl = C.w.Clin;
        a.omega = (const double*)(buf + o_om);
        a.rhs = (const double*)(buf + o_rhs);
        a.obs_piv = (const int32_t*)(buf + o_obs);
        a.nz_rows = (const int32_t*)(buf + o_nr);
        a.nz_pwr = (const double*)(buf + o_np);
        a.nz_exp = (const double*)(buf + o_ne);
        a.out = d_out;
        a.psd = d_out;
        a.ws = d_out + n_out_al;
        a.ws_stride = stride;
        HIPCHK(ctx, launch_ac(a, (int)nblocks, P.n <= 512 ? 64 : 256, lds, s));
        HIPCHK(ctx, hipMemcpyAsync(a.transposed ? psd : out, d_out, sizeof(double) * n_out, hipMemcpyDeviceToHost, s));
        HIPCHK(ctx, hipStreamSynchronize(s));
        return CS_OK;
    };
    rc = run();
    (void)hipFree(buf);
    return rc;
}

int ac_check(cs_ctx* ctx, Circuit* C, const double* p, const double* u_dc, int32_t n_freq, const double* omega) {
    if (!C || !p || !u_dc || n_freq <= 0 || !omega) return fail(ctx, CS_E_INVALID, "bad argument");
    if (C->big)
        return fail(ctx, CS_E_INVALID,
                    "AC and noise analysis run on the level-scheduled plan; this circuit uses the supernodal solver");
    for (int32_t f = 0; f < n_freq; f++)
        if (!std::isfinite(omega[f]) || omega[f] < 0.0) return fail(ctx, CS_E_INVALID, "frequencies must be finite and >= 0");
    return check_params(ctx, C->plan, p);
}

}  // namespace

int cs_ac(cs_ctx* ctx, int32_t cid, const double* p, const double* u_dc, const double* src_ac, int32_t n_freq,
          const double* omega, int32_t n_obs, const int32_t* obs, double* out) {
    Circuit* C = get_circuit(ctx, cid);
    int rc = ac_check(ctx, C, p, u_dc, n_freq, omega);
    if (rc) return rc;
    const Plan& P = C->plan;
    if (!src_ac || n_obs <= 0 || !obs || !out) return fail(ctx, CS_E_INVALID, "bad argument");
    std::vector<int32_t> obs_piv(n_obs);
    for (int32_t i = 0; i < n_obs; i++) {
        if (obs[i] < 0 || obs[i] >= P.n) return fail(ctx, CS_E_INVALID, "observed unknown out of range");
        obs_piv[i] = P.pcol[obs[i]];
    }
    // b = -dR/d(eps): a source's stamp enters its rows with sign +-1 and
    // its m-factor; the AC excitation moves its value by eps * |ac|
    const int32_t s0 = 4 * P.n_mos;
    std::vector<double> rhs(P.n, 0.0);
    for (int32_t k = 0; k < P.n; k++)
        for (int32_t q = P.rnl_ptr[k]; q < P.rnl_ptr[k + 1]; q++) {
            const int32_t ref = P.rnl_ref[q], slot = ref >> 1;
            if (slot < s0 || slot >= s0 + P.n_src) continue;
            const int32_t sidx = slot - s0;
            const double m = P.src_m.empty() ? 1.0 : P.src_m[sidx];
            rhs[k] += ((ref & 1) ? 1.0 : -1.0) * m * std::fabs(src_ac[sidx]);
        }
    (void)hipSetDevice(ctx->device);
    if ((rc = ac_operands(ctx, *C, p, u_dc))) return rc;
    AcArgs a{};
    a.n_freq = n_freq;
    a.transposed = 0;
    a.n_obs = n_obs;
    return ac_sweep(ctx, *C, a, omega, rhs, obs_piv, {-1, -1}, {0.0}, {0.0}, out, nullptr);
}

int cs_noise(cs_ctx* ctx, int32_t cid, const double* p, const double* u_dc, double temp_c, int32_t n_freq,
             const double* omega, int32_t obs, double* psd) {
    Circuit* C = get_circuit(ctx, cid);
    int rc = ac_check(ctx, C, p, u_dc, n_freq, omega);
    if (rc) return rc;
    const Plan& P = C->plan;
    if (!psd || obs < 0 || obs >= P.n) return fail(ctx, CS_E_INVALID, "bad argument");
    if (!std::isfinite(temp_c) || temp_c <= -273.15) return fail(ctx, CS_E_INVALID, "bad temperature");
    // thermal noise of every resistor, 4kT/R per m-factor copy
    // (src/simpledevices.jl:71-76), a current in parallel with it
    const double kB = 1.380649e-23, T = temp_c + 273.15;
    const int32_t nres = (int32_t)P.res_m.size();
    std::vector<int32_t> rows;
    std::vector<double> pwr, ex;
    for (int32_t k = 0; k < nres; k++) {
        const int32_t a = P.res_nodes[2 * k], b = P.res_nodes[2 * k + 1];
        rows.push_back(a >= 0 ? P.prow[a] : -1);
        rows.push_back(b >= 0 ? P.prow[b] : -1);
        pwr.push_back(P.res_m[k] * 4.0 * kB * T / p[P.lay.res_r + k]);
        ex.push_back(0.0);
    }
    if (rows.empty()) {
        rows = {-1, -1};
        pwr = {0.0};
        ex = {0.0};
    }
    (void)hipSetDevice(ctx->device);
    if ((rc = ac_operands(ctx, *C, p, u_dc))) return rc;
    AcArgs a{};
    a.n_freq = n_freq;
    a.transposed = 1;
    a.obs_col = P.pcol[obs];
    a.n_noise = nres;
    return ac_sweep(ctx, *C, a, omega, {0.0}, {0}, rows, pwr, ex, nullptr, psd);
}

int cs_batch_kernel(cs_ctx* ctx, int32_t bid, int32_t* kernel, int32_t* n_launches) {
    Batch* B = get_batch(ctx, bid);
    if (!B) return fail(ctx, CS_E_INVALID, "bad batch id");
    if (kernel) *kernel = B->kernel;
    if (n_launches) *n_launches = 1;
    return CS_OK;
}

// Algorithmic traffic of the executed Newton iterations (per iteration and
// instance): MOSFET eval 8*(7 in + 4 out) B per device; assembly 8*nnz
// written + 8*(nnz Glin + nnz Clin + stamp refs) read + 4*(refs + indices);
// LU 2*8*nnz(L+U); solves 8*nnz(L+U) + 8*3n.  Flops: eval 40 per device,
// assembly 3 per entry + 1 per stamp ref, LU 2 per update, solves 2*nnz(L+U).
int cs_batch_traffic(cs_ctx* ctx, int32_t bid, double* alg_bytes, double* alg_flops) {
    Batch* B = get_batch(ctx, bid);
    if (!B) return fail(ctx, CS_E_INVALID, "bad batch id");
    std::vector<cs_tran_stats> st(B->n_inst);
    int rc = cs_batch_results(ctx, bid, nullptr, nullptr, st.data());
    if (rc) return rc;
    double bytes = 0.0, flops = 0.0;
    for (int32_t i = 0; i < B->n_inst; i++) {
        const Plan& P = ctx->circuits[B->cid[i]]->plan;
        const double refs = (double)P.jnl_ref.size() + (double)P.rnl_ref.size();
        const double b_it = 8.0 * 11.0 * P.n_mos + 8.0 * P.nnz + 8.0 * (2.0 * P.nnz + refs) +
                            4.0 * (refs + 2.0 * P.nnz) + 16.0 * P.nnz + 8.0 * P.nnz + 24.0 * P.n;
        const double f_it = 40.0 * P.n_mos + 3.0 * P.nnz + refs + 2.0 * (double)P.lu_updates +
                            2.0 * P.nnz;
        bytes += b_it * (double)st[i].newton_iters;
        flops += f_it * (double)st[i].newton_iters;
    }
    if (alg_bytes) *alg_bytes = bytes;
    if (alg_flops) *alg_flops = flops;
    return CS_OK;
}

// ---- BSIM-CMG device evaluation ---------------------------------------------------------
#ifdef CEDAR_HAVE_BSIMCMG
int cs_bsimcmg_available(void) { return 1; }

static void bsim_init(cs_ctx* ctx) {
    if (ctx->bsim_ready) return;
    ctx->bsim_card.assign(bsim_card_size(), 0);
    ctx->bsim_inst.assign(bsim_inst_size(), 0);
    ctx->bsim_card_full = ctx->bsim_card;
    bsim_card_defaults(ctx->bsim_card_full.data());
    ctx->bsim_ready = true;
}

int cs_bsimcmg_param(cs_ctx* ctx, const char* name, double value) {
    if (!ctx || !name) return fail(ctx, CS_E_INVALID, "bad argument");
    bsim_init(ctx);
    if (bsim_set_param(ctx->bsim_card.data(), ctx->bsim_inst.data(), name, value) != 0)
        return fail(ctx, CS_E_INVALID, std::string("unknown BSIM-CMG parameter ") + name);
    ctx->bsim_card_full = ctx->bsim_card;
    bsim_card_defaults(ctx->bsim_card_full.data());
    return CS_OK;
}

int cs_bsimcmg_eval(cs_ctx* ctx, int64_t n, const double* L, const double* nfin, const double* v,
                    double temp_c, double* out, int32_t* iters, double* kernel_ms) {
    if (!ctx || n <= 0 || !L || !nfin || !v || !out) return fail(ctx, CS_E_INVALID, "bad argument");
    (void)hipSetDevice(ctx->device);
    bsim_init(ctx);
    std::vector<char> card = ctx->bsim_card;   // given flags as set; defaults filled here
    bsim_card_defaults(card.data());
    std::vector<void*> allocs;
    struct Guard {
        std::vector<void*>& a;
        ~Guard() { for (void* q : a) (void)hipFree(q); }
    } guard{allocs};
    auto dalloc = [&](void** q, size_t bytes) -> int {
        hipError_t e = hipMalloc(q, std::max<size_t>(bytes, 16));
        if (e != hipSuccess) return fail(ctx, CS_E_OOM, "BSIM-CMG allocation failed");
        allocs.push_back(*q);
        return CS_OK;
    };
    const int per = bsim_out_per();
    void *d_card, *d_inst, *d_L, *d_nf, *d_v, *d_out, *d_it = nullptr;
    int rc;
    if ((rc = dalloc(&d_card, card.size())) || (rc = dalloc(&d_inst, ctx->bsim_inst.size())) ||
        (rc = dalloc(&d_L, sizeof(double) * n)) || (rc = dalloc(&d_nf, sizeof(double) * n)) ||
        (rc = dalloc(&d_v, sizeof(double) * 4 * n)) || (rc = dalloc(&d_out, sizeof(double) * per * n)) ||
        (iters && (rc = dalloc(&d_it, sizeof(int32_t) * n))))
        return rc;
    HIPCHK(ctx, hipMemcpy(d_card, card.data(), card.size(), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_inst, ctx->bsim_inst.data(), ctx->bsim_inst.size(), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_L, L, sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_nf, nfin, sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_v, v, sizeof(double) * 4 * n, hipMemcpyHostToDevice));
    BsimArgs a{};
    a.card = d_card;
    a.inst = d_inst;
    a.n = n;
    a.L = (const double*)d_L;
    a.nfin = (const double*)d_nf;
    a.v = (const double*)d_v;
    a.temp = temp_c + 273.15;
    a.out = (double*)d_out;
    a.iters = (int32_t*)d_it;
    const int per_cu = bsim_max_blocks();
    if (per_cu <= 0) return fail(ctx, CS_E_RANGE, "BSIM-CMG kernel does not fit on a CU");
    // one resident wave of lanes, each walking its instances; every lane keeps
    // the bias-independent values of its current instance in one column of store
    const int64_t want = (n + 255) / 256;
    const int nblocks = (int)std::min<int64_t>(want, (int64_t)per_cu * std::max(ctx->n_cu, 1));
    void* d_store = nullptr;
    a.stride = (int64_t)nblocks * 256;
    if ((rc = dalloc(&d_store, sizeof(double) * (size_t)bsim_setup_size() * a.stride))) return rc;
    a.store = (double*)d_store;
    hipEvent_t e0, e1;
    HIPCHK(ctx, hipEventCreate(&e0));
    HIPCHK(ctx, hipEventCreate(&e1));
    HIPCHK(ctx, hipEventRecord(e0, ctx->stream));
    HIPCHK(ctx, launch_bsimcmg(a, nblocks, ctx->stream));
    HIPCHK(ctx, hipEventRecord(e1, ctx->stream));
    HIPCHK(ctx, hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(ctx, hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (kernel_ms) *kernel_ms = ms;
    HIPCHK(ctx, hipMemcpy(out, d_out, sizeof(double) * per * n, hipMemcpyDeviceToHost));
    if (iters) HIPCHK(ctx, hipMemcpy(iters, d_it, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    return CS_OK;
}
int cs_bsimcmg_eval_noalloc(cs_ctx* ctx, int64_t n, const double* L, const double* nfin, const double* v,
                            double temp_c, double* out, int32_t* iters) {
    if (!ctx || n <= 0 || !L || !nfin || !v || !out) return fail(ctx, CS_E_INVALID, "bad argument");
    if (n > INT32_MAX) return fail(ctx, CS_E_RANGE, "at most 2^31-1 instances per call");
    (void)hipSetDevice(ctx->device);
    std::string err;
    char* base = (char*)bsim_scratch(ctx->device, err);
    if (!base) return fail(ctx, CS_E_HIP, err);
    bsim_init(ctx);
    const int per_cu = bsim_max_blocks();
    if (per_cu <= 0) return fail(ctx, CS_E_RANGE, "BSIM-CMG kernel does not fit on a CU");
    // the card with its defaults is kept on the context (bsim_init and
    // cs_bsimcmg_param refresh it); both structs go to the library's buffer
    HIPCHK(ctx, hipMemcpyAsync(base + bsim_scratch_card_off(), ctx->bsim_card_full.data(),
                               ctx->bsim_card_full.size(), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(ctx, hipMemcpyAsync(base + bsim_scratch_inst_off(), ctx->bsim_inst.data(), ctx->bsim_inst.size(),
                               hipMemcpyHostToDevice, ctx->stream));
    BsimArgs a{};
    a.card = base + bsim_scratch_card_off();
    a.inst = base + bsim_scratch_inst_off();
    a.n = n;
    a.L = L;
    a.nfin = nfin;
    a.v = v;
    a.temp = temp_c + 273.15;
    a.out = out;
    a.iters = iters;
    const int64_t want = (n + 255) / 256;
    const int64_t cap = std::min<int64_t>((int64_t)per_cu * std::max(ctx->n_cu, 1), bsim_noalloc_lanes() / 256);
    const int nblocks = (int)std::min<int64_t>(want, cap);
    a.stride = (int64_t)nblocks * 256;
    a.store = (double*)(base + bsim_scratch_store_off());
    HIPCHK(ctx, launch_bsimcmg(a, nblocks, ctx->stream));
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    return CS_OK;
}
#else
int cs_bsimcmg_available(void) { return 0; }
int cs_bsimcmg_eval_noalloc(cs_ctx* ctx, int64_t, const double*, const double*, const double*, double, double*,
                            int32_t*) {
    return fail(ctx, CS_E_INVALID, "this library was built without the BSIM-CMG model");
}
int cs_bsimcmg_param(cs_ctx* ctx, const char*, double) {
    return fail(ctx, CS_E_INVALID, "this library was built without the BSIM-CMG model");
}
int cs_bsimcmg_eval(cs_ctx* ctx, int64_t, const double*, const double*, const double*, double, double*,
                    int32_t*, double*) {
    return fail(ctx, CS_E_INVALID, "this library was built without the BSIM-CMG model");
}
#endif

// ---- batched adjoint ------------------------------------------------------------------
// Runs on the LDS-resident kernels: the instances are grouped into the same
// size classes as a batched transient (cs_batch_create with the LDS kernel);
// per class the recording forward and the reverse kernel run back to back on
// one stream.
int cs_adjoint_batch(cs_ctx* ctx, int32_t n_inst, const int32_t* inst_cid, const double* params,
                     const double* u0, const cs_tran_opts* o, const cs_adjoint_opts* ao,
                     double* energy, double* grad, int64_t* n_steps, double* t_log,
                     int32_t* npts_log, cs_tran_stats* st, double* kernel_ms) {
    if (!ctx || n_inst <= 0 || !inst_cid || !params || !u0 || !o || !ao || !energy || !grad)
        return fail(ctx, CS_E_INVALID, "bad argument");
    if (o->init != CS_INIT_UIC) return fail(ctx, CS_E_INVALID, "the adjoint needs CS_INIT_UIC");
    if (o->jac_reuse) return fail(ctx, CS_E_INVALID, "the adjoint differentiates full Newton steps (jac_reuse = 0)");
    if (ao->ckpt_every <= 0 || ao->max_steps <= 0) return fail(ctx, CS_E_INVALID, "bad adjoint options");
    (void)hipSetDevice(ctx->device);
    std::vector<int64_t> g_off;
    int64_t go = 0;
    int32_t ck_n = 1;
    std::vector<int32_t> obj(3 * ctx->circuits.size(), (int32_t)CP_GROUND);
    for (int32_t i = 0; i < n_inst; i++) {
        Circuit* C = get_circuit(ctx, inst_cid[i]);
        if (!C) return fail(ctx, CS_E_INVALID, "bad circuit id");
        if (C->big) return fail(ctx, CS_E_INVALID, "supernodal circuits have no batched adjoint");
        const Plan& P = C->plan;
        if (!P.uic_ok) return fail(ctx, CS_E_INVALID, "UIC not supported by this circuit");
        if (ao->vsrc < 0 || 2 * ao->vsrc + 1 >= (int32_t)P.vsrc_nodes.size())
            return fail(ctx, CS_E_INVALID, "objective source index out of range");
        g_off.push_back(go);
        go += P.n_mos;
        ck_n = std::max(ck_n, P.n);
        const int32_t a = P.vsrc_nodes[2 * ao->vsrc], b = P.vsrc_nodes[2 * ao->vsrc + 1];
        const size_t c = (size_t)inst_cid[i];
        obj[3 * c] = a >= 0 ? P.pcol[a] : (int32_t)CP_GROUND;
        obj[3 * c + 1] = b >= 0 ? P.pcol[b] : (int32_t)CP_GROUND;
        obj[3 * c + 2] = P.pcol[P.n_nodes + ao->vsrc];
    }
    cs_tran_opts o2 = *o;
    o2.batch_kernel = CS_BATCH_KERNEL_LDS;
    o2.n_out = 0;
    int32_t bid = -1;
    int rc = cs_batch_create(ctx, n_inst, inst_cid, params, u0, &o2, &bid);
    if (rc != CS_OK) return rc;
    std::vector<void*> allocs;
    struct Guard {
        cs_ctx* ctx;
        int32_t bid;
        std::vector<void*>& a;
        ~Guard() {
            for (void* q : a) (void)hipFree(q);
            (void)cs_batch_destroy(ctx, bid);
        }
    } guard{ctx, bid, allocs};
    Batch* B = get_batch(ctx, bid);
    auto dalloc = [&](void** q, size_t bytes) -> int {
        hipError_t e = hipMalloc(q, std::max<size_t>(bytes, 16));
        if (e != hipSuccess) return fail(ctx, CS_E_OOM, "adjoint allocation failed");
        allocs.push_back(*q);
        return CS_OK;
    };
    auto balloc = [&](void** q, size_t bytes) -> int {   // lives with the batch
        hipError_t e = hipMalloc(q, std::max<size_t>(bytes, 16));
        if (e != hipSuccess) return fail(ctx, CS_E_OOM, "adjoint allocation failed");
        B->allocs.push_back(*q);
        return CS_OK;
    };
    if ((rc = build_lds_classes(ctx, *B, balloc)) != CS_OK) return rc;
    const int64_t cap = ao->max_steps;
    const int64_t K = ao->ckpt_every;
    const int64_t ckcap = cap / K + 1;
    const size_t ncls = B->classes.size();
    void *d_tl, *d_npl, *d_ck, *d_ns, *d_E, *d_g, *d_goff, *d_obj, *d_q2;
    if ((rc = dalloc(&d_tl, sizeof(double) * cap * n_inst)) ||
        (rc = dalloc(&d_npl, sizeof(int32_t) * cap * n_inst)) ||
        (rc = dalloc(&d_ck, sizeof(double) * (size_t)ckcap * 3 * ck_n * n_inst)) ||
        (rc = dalloc(&d_ns, sizeof(int64_t) * n_inst)) || (rc = dalloc(&d_E, sizeof(double) * n_inst)) ||
        (rc = dalloc(&d_g, sizeof(double) * std::max<int64_t>(go, 1))) ||
        (rc = dalloc(&d_goff, sizeof(int64_t) * n_inst)) ||
        (rc = dalloc(&d_obj, sizeof(int32_t) * obj.size())) ||
        (rc = dalloc(&d_q2, sizeof(int32_t) * ncls)))
        return rc;
    HIPCHK(ctx, hipMemcpy(d_goff, g_off.data(), sizeof(int64_t) * n_inst, hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d_obj, obj.data(), sizeof(int32_t) * obj.size(), hipMemcpyHostToDevice));
    std::vector<AdjLdsArgs> args(ncls);
    // resident workgroups of each kernel by its own LDS: the forward kernel's
    // image is a quarter smaller (768 185-stage rings over 3 ps: 14.4 ms with
    // both at the reverse's, 11.9 now)
    std::vector<std::array<int, 2>> nblk(ncls);
    for (size_t k = 0; k < ncls; k++) {
        const LdsClass& L = B->classes[k];
        for (int r = 0; r < 2; r++) {
            const int per_cu = adj_lds_max_blocks(L.nr, L.dyn, r == 1, L.lds[r]);
            if (per_cu <= 0) return fail(ctx, CS_E_RANGE, "adjoint kernels do not fit on a CU");
            nblk[k][r] = (int)std::min<int64_t>(L.n_inst, (int64_t)per_cu * std::max(ctx->n_cu, 1));
        }
        void* d_seg;
        if ((rc = dalloc(&d_seg, sizeof(double) * (size_t)nblk[k][1] * K * ck_n))) return rc;
        AdjLdsArgs& a = args[k];
        a.f = L.args;
        a.t_log = (double*)d_tl;
        a.npts_log = (int32_t*)d_npl;
        a.cap = cap;
        a.ckpt = (double*)d_ck;
        a.ckcap = ckcap;
        a.K = (int32_t)K;
        a.ck_n = ck_n;
        a.n_steps = (int64_t*)d_ns;
        a.energy = (double*)d_E;
        a.grad = (double*)d_g;
        a.g_off = (const int64_t*)d_goff;
        a.obj = (const int32_t*)d_obj;
        a.seg = (double*)d_seg;
        a.queue2 = (int32_t*)d_q2 + k;
    }
    void* d_args;
    if ((rc = dalloc(&d_args, sizeof(AdjLdsArgs) * ncls))) return rc;
    HIPCHK(ctx, hipMemcpy(d_args, args.data(), sizeof(AdjLdsArgs) * ncls, hipMemcpyHostToDevice));
    const AdjLdsArgs* da = (const AdjLdsArgs*)d_args;
    hipStream_t s = ctx->stream;
    HIPCHK(ctx, hipMemsetAsync(B->d_queues, 0, sizeof(int32_t) * ncls, s));
    HIPCHK(ctx, hipMemsetAsync(d_q2, 0, sizeof(int32_t) * ncls, s));
    HIPCHK(ctx, hipEventRecord(B->ev0, s));
    const size_t ns = B->class_ev.size();
    for (size_t k = 0; k < ns; k++) HIPCHK(ctx, hipStreamWaitEvent(ctx->side[k], B->ev0, 0));
    for (size_t k = 0; k < ncls; k++) {
        const LdsClass& L = B->classes[k];
        for (int r = 0; r < 2; r++)
            HIPCHK(ctx, launch_adj_lds(L.nr, L.dyn, r == 1, da + k, nblk[k][r], L.lds[r], ctx->side[k % ns]));
    }
    for (size_t k = 0; k < ns; k++) {
        HIPCHK(ctx, hipEventRecord(B->class_ev[k], ctx->side[k]));
        HIPCHK(ctx, hipStreamWaitEvent(s, B->class_ev[k], 0));
    }
    HIPCHK(ctx, hipEventRecord(B->ev1, s));
    HIPCHK(ctx, hipEventSynchronize(B->ev1));
    float ms = 0.f;
    HIPCHK(ctx, hipEventElapsedTime(&ms, B->ev0, B->ev1));
    if (kernel_ms) *kernel_ms = ms;
    HIPCHK(ctx, hipMemcpy(energy, d_E, sizeof(double) * n_inst, hipMemcpyDeviceToHost));
    HIPCHK(ctx, hipMemcpy(grad, d_g, sizeof(double) * go, hipMemcpyDeviceToHost));
    if (n_steps) HIPCHK(ctx, hipMemcpy(n_steps, d_ns, sizeof(int64_t) * n_inst, hipMemcpyDeviceToHost));
    if (t_log) HIPCHK(ctx, hipMemcpy(t_log, d_tl, sizeof(double) * cap * n_inst, hipMemcpyDeviceToHost));
    if (npts_log)
        HIPCHK(ctx, hipMemcpy(npts_log, d_npl, sizeof(int32_t) * cap * n_inst, hipMemcpyDeviceToHost));
    if (st) {
        HIPCHK(ctx, hipMemcpy(st, B->args.stats, sizeof(cs_tran_stats) * n_inst, hipMemcpyDeviceToHost));
        for (int32_t i = 0; i < n_inst; i++) st[i].busy_s = 0.0;
    }
    return CS_OK;
}

}  // extern "C"
