// kernels.hip — gfx950 kernels of the Newton-transient engine.
//
// Batched path (k_tran_batch): a persistent grid of one-wavefront workgroups
// walks a work queue of circuit instances (largest first).  A workgroup runs
// its instance's whole transient on the device: consistent initialisation
// (DC op or UIC), then per step predictor -> Newton (eval -> assemble ->
// LU refactor -> solves -> update/WRMS) -> local-error test -> accept/reject
// -> output interpolation, exactly the rules of rules.h.  The per-unknown
// history lives in registers of the lane that owns the unknown; F, the
// vectors and the stamp buffer live in LDS; the per-instance linear stamp
// values (Glin, Clin) in a per-workgroup global workspace.
//
// Single-instance kernels (k_*): one workgroup each, the pieces the plain
// per-instance path captures into a hipGraph per Newton iteration and the
// DAE interface (cs_residual / cs_jacobian / cs_lu_*) calls directly.
#include "device.h"
#include "kernels.h"
#include "tran_device.h"

namespace cedar {

// ---------------------------------------------------------------------------
// single-instance kernels
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kSingleThreads) void k_lin_setup(const DPlan* dp, InstDev w) {
    const DPlan* P = dp;
    dev_lin_setup<kSingleThreads>(P, w.p, w.linbuf, w.Glin, w.Clin);
}

// JAC = false: the residual only, F keeps the factors of an earlier
// iteration (modified Newton).  VA = false: no Verilog-A device, whose models
// would hold registers and scratch memory
template <bool JAC, bool VA>
__global__ __launch_bounds__(kSingleThreads) void k_eval_assemble(const DPlan* dp, InstDev w) {
    __shared__ double red[kSingleThreads];
    const DPlan* P = dp;
    const StepDev sp = *w.sp;
    dev_sources<kSingleThreads>(P, w.p, sp.t, sp.mode, w.st);
    dev_mos<kSingleThreads>(P, w.p, w.u, w.st, w.p[P->p_gmin]);
    if constexpr (VA) dev_va<kSingleThreads>(P, w.p, w.u, w.st, w.p[P->p_gmin]);
    __syncthreads();
    const double a0 = sp.kind == STEP_TRAN ? sp.a0 : 0.0;
    const double m = dev_assemble<kSingleThreads, JAC>(P, w.Glin, w.Clin, a0, w.u,
                                                  sp.kind == STEP_TRAN ? w.qx : nullptr, w.st,
                                                  w.F, w.x, sp.kind == STEP_UIC ? w.u0 : nullptr);
    const double r = block_reduce<kSingleThreads>(m, red, OpMax());
    if (threadIdx.x == 0) w.norm[NRM_RES] = r;
}

__global__ __launch_bounds__(kSingleThreads) void k_lu(const DPlan* dp, InstDev w) {
    const DPlan* P = dp;
    dev_lu<kSingleThreads>(P, w.F, w.inv);
}

__global__ __launch_bounds__(kSingleThreads) void k_solve(const DPlan* dp, InstDev w) {
    const DPlan* P = dp;
    dev_fwd<kSingleThreads>(P, w.F, w.x);
    dev_bwd<kSingleThreads>(P, w.F, w.inv, w.x);
}

__global__ __launch_bounds__(kSingleThreads) void k_solve_t(const DPlan* dp, InstDev w) {
    const DPlan* P = dp;
    dev_tfwd<kSingleThreads>(P, w.F, w.inv, w.x);
    dev_tbwd<kSingleThreads>(P, w.F, w.x);
}

// u += d (DC/UIC: skipped once the residual met the tolerance).  norm: WRMS(d), max|d|, done flag.
__global__ __launch_bounds__(kSingleThreads) void k_update(const DPlan* dp, InstDev w) {
    __shared__ double red[kSingleThreads];
    const DPlan* P = dp;
    const StepDev sp = *w.sp;
    const int tid = threadIdx.x;
    if (sp.kind != STEP_TRAN) {
        const double res = w.norm[NRM_RES];
        if (res <= sp.tol) {
            if (tid == 0) w.norm[NRM_DONE] = 1.0;
            return;
        }
    }
    double ss = 0.0, mx = 0.0;
    for (int i = tid; i < P->n; i += kSingleThreads) {
        const double d = w.x[P->pcol[i]];
        const double ui = w.u[i] + d;
        w.u[i] = ui;
        const double r = d / (sp.rtol * fabs(ui) + sp.atol);
        ss += r * r;
        const double a = fabs(d);
        if (a != a || a > mx) mx = a;
    }
    const double s = block_reduce<kSingleThreads>(ss, red, OpSum());
    const double m = block_reduce<kSingleThreads>(mx, red, OpMax());
    if (tid == 0) {
        w.norm[NRM_WRMS] = sqrt(s / P->n);
        w.norm[NRM_MAXD] = m;
        w.norm[NRM_DONE] = 0.0;
    }
}

__global__ __launch_bounds__(kSingleThreads) void k_charges(const DPlan* dp, InstDev w,
                                                            const double* v, double* q) {
    const DPlan* P = dp;
    dev_charges<kSingleThreads>(P, w.Clin, v, q);
}

void launch_lin_setup(const DPlan* dp, const InstDev& w, hipStream_t s) {
    hipLaunchKernelGGL(k_lin_setup, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_eval_assemble(const DPlan* dp, const InstDev& w, hipStream_t s, bool jac) {
    auto* f = w.has_va ? (jac ? k_eval_assemble<true, true> : k_eval_assemble<false, true>)
                       : (jac ? k_eval_assemble<true, false> : k_eval_assemble<false, false>);
    hipLaunchKernelGGL(f, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_lu(const DPlan* dp, const InstDev& w, hipStream_t s) {
    hipLaunchKernelGGL(k_lu, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_solve(const DPlan* dp, const InstDev& w, hipStream_t s) {
    hipLaunchKernelGGL(k_solve, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_solve_t(const DPlan* dp, const InstDev& w, hipStream_t s) {
    hipLaunchKernelGGL(k_solve_t, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_update(const DPlan* dp, const InstDev& w, hipStream_t s) {
    hipLaunchKernelGGL(k_update, dim3(1), dim3(kSingleThreads), 0, s, dp, w);
}
void launch_charges(const DPlan* dp, const InstDev& w, const double* v, double* q,
                    hipStream_t s) {
    hipLaunchKernelGGL(k_charges, dim3(1), dim3(kSingleThreads), 0, s, dp, w, v, q);
}

// ---------------------------------------------------------------------------
// batched persistent transient kernel
// ---------------------------------------------------------------------------
namespace {

// Bound by the latency of one wavefront's chains through the caches and LDS, so
// by how many wavefronts are resident once a batch fills the device: registers.
// With the waveforms and step factors of wave_math.h they are 123, 126, 164
// and 216 (1, 2, 4 and 8 rows per lane; four, four, three and two wavefronts
// per SIMD) and none is spilled; with the library's sin, exp, fmod and pow
// inlined 208 to 256. Those held to 128 (74 spilled, among them the ones that
// keep spilled scalar registers) gave wrong answers in a build without
// Verilog-A models, DtLessThanMin from the first steps; the source is not at
// fault as far as a CPU build shows (address and undefined-behaviour sanitizers,
// uninitialised variables filled with patterns, lanes in any order between
// barriers: the oracle's steps, one set of bits). So no limit that spills.
// 4096 rings over 2 ps: 33 stages 7.5 ms held to 128, 8.0 without a limit, 5.2
// now; 67 stages 12.8, 14.9, 10.3; 4096 12 x 12 meshes over 20 ps 44.7, 41.7,
// 41.5.  The Verilog-A models take 175 and more (two per SIMD): 2048 inverters
// of them 36.5 ms held to 128 and 30.4 now, but 4096 of them 50.4 and 60.4.
template <int NR, bool VA>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NR <= 2 && !VA ? 4 : 1)))
void k_tran_batch(BatchArgs A) {
    extern __shared__ double lds[];
    __shared__ int s_idx;
    Lds L;
    L.F = lds;
    L.inv = L.F + A.nnz_max;
    L.u = L.inv + A.n_max;
    L.x = L.u + A.n_max;
    L.qx = L.x + A.n_max;
    L.st = L.qx + A.n_max;
    double* Glin = A.glin + (size_t)blockIdx.x * A.nnz_max;
    double* Clin = A.clin + (size_t)blockIdx.x * A.nnz_max;
    double* linbuf = A.linbuf + (size_t)blockIdx.x * A.lin_max;
    for (;;) {
        if (threadIdx.x == 0) s_idx = atomicAdd(A.queue, 1);
        __syncthreads();
        // wave-uniform queue index: the plan and instance pointers then live
        // in scalar registers
        const int qi = __builtin_amdgcn_readfirstlane(s_idx);
        __syncthreads();
        if (qi >= A.n_inst) break;
        const int inst = __builtin_amdgcn_readfirstlane(A.order[qi]);
        const int cid = __builtin_amdgcn_readfirstlane(A.inst_cid[inst]);
        const DPlan* P = A.plans + cid;
        NoRec rec;
        run_instance<NR, VA>(rec, P, A.params + A.p_off[inst], A.u0 ? A.u0 + A.u_off[inst] : nullptr,
                         A.wave ? A.wave + A.w_off[inst] : nullptr, A.u_final + A.u_off[inst],
                         A.stats + inst, A.o, L, Glin, Clin, linbuf);
    }
}

}  // namespace

size_t batch_lds_bytes(const BatchArgs& a) {
    return sizeof(double) * ((size_t)a.nnz_max + 4 * (size_t)a.n_max + a.stamp_max);
}

namespace {
typedef void (*BatchKernel)(BatchArgs);
template <bool VA>
BatchKernel batch_kernel(int nr) {
    switch (nr) {
    case 1: return k_tran_batch<1, VA>;
    case 2: return k_tran_batch<2, VA>;
    case 4: return k_tran_batch<4, VA>;
    default: return k_tran_batch<8, VA>;
    }
}
BatchKernel batch_kernel(int nr, bool va) { return va ? batch_kernel<true>(nr) : batch_kernel<false>(nr); }
}  // namespace

int batch_max_blocks(int nr, bool va, size_t lds) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, batch_kernel(nr, va), NT, lds) != hipSuccess) return 0;
    return nb;
}

hipError_t launch_tran_batch(int nr, bool va, const BatchArgs& a, int nblocks, size_t lds, hipStream_t s) {
    hipLaunchKernelGGL(batch_kernel(nr, va), dim3(nblocks), dim3(NT), lds, s, a);
    return hipGetLastError();
}

}  // namespace cedar
