// sens.hip — forward parameter sensitivities of the plain-path transient
// (the role of ODEForwardSensitivityProblem in the reference,
// test/sensitivity.jl:13-66), by the staggered direct method.
//
// The discrete equations of an accepted BDF step m are
//     I(u_m, t_m; p) + a0 Q(u_m; p) + a1 Q_{m-1} + a2 Q_{m-2} = 0,
// with Q = C u the linear charges.  Differentiating them in p_j on the
// step's own sequence gives
//     J_m s_m = -(dI/dp_j + a0 dQ/dp_j + a1 dQ_{m-1} + a2 dQ_{m-2}),
// dQ_k = C s_k + dQ/dp_j(u_k) the total derivative of the charges, J_m the
// Jacobian at u_m.  The initial point's equations are the pinned system
// (rows that carry charge fixed at the pin value, the rest I = 0): there the
// pinned rows of the right-hand side carry the pin's own sensitivity.
//
// One workgroup per parameter: it forms the right-hand side from the
// parameter's stamps (a few rows, see SensParam) and the history, solves with
// the LU the host has just refactored (the circuit's F and inv), and writes
// s in natural order and the new charge sensitivity dQ = C s + dQ/dp.
// Small circuits run whole in one launch instead, step control and solves
// together (k_tran_sens, below).
#include "device.h"
#include "kernels.h"
#include "tran_device.h"

namespace cedar {

namespace {

constexpr int kSensThreads = 256;

__device__ __forceinline__ double nodev(const double* u, int32_t i) { return i >= 0 ? u[i] : 0.0; }

// dI/dp (into di) and dQ/dp (into dq) of one parameter at u, on at most two
// natural rows r[0], r[1] (-1: none)
__device__ void param_stamps(const DPlan* P, const double* p, const double* u, const SensParam& s, int mode,
                             int32_t (&r)[2], double (&di)[2], double (&dq)[2]) {
    r[0] = r[1] = -1;
    di[0] = di[1] = dq[0] = dq[1] = 0.0;
    switch (s.kind) {
        case SP_R: {   // I = m (Va - Vb) / R on a, -I on b
            const double v = nodev(u, s.i0) - nodev(u, s.i1);
            const double g = -s.m / (s.val * s.val) * v;
            r[0] = s.i0; r[1] = s.i1; di[0] = g; di[1] = -g;
            break;
        }
        case SP_C: {   // Q = m C (Va - Vb) on a, -Q on b
            const double v = s.m * (nodev(u, s.i0) - nodev(u, s.i1));
            r[0] = s.i0; r[1] = s.i1; dq[0] = v; dq[1] = -v;
            break;
        }
        case SP_IND:   // Q_j = -L I_j on the branch row
            r[0] = s.i0; dq[0] = -u[s.i0];
            break;
        case SP_VCCS: {   // I = m g (Vc - Vd) on out+, -I on out-
            const double v = s.m * (nodev(u, s.i2) - nodev(u, s.i3));
            r[0] = s.i0; r[1] = s.i1; di[0] = v; di[1] = -v;
            break;
        }
        case SP_VCVS:     // branch row: Va - Vb - g (Vc - Vd)
            r[0] = s.i0; di[0] = -(nodev(u, s.i2) - nodev(u, s.i3));
            break;
        case SP_VTH: case SP_KP: case SP_MW: case SP_ML: {
            const int k = s.dev;
            const double vd = nodev(u, s.i0), vg = nodev(u, s.i1), vs = nodev(u, s.i2);
            const double gmin = p[P->p_gmin];
            double id, dd, dg, ds;
            sqlaw_eval(s.i3, p[P->p_mos_vth + k], p[P->p_mos_kp + k], p[P->p_mos_w + k], p[P->p_mos_l + k],
                       gmin, vd, vg, vs, id, dd, dg, ds);
            const double ich = id - gmin * (vd - vs);   // the channel current, proportional to beta
            double d;
            if (s.kind == SP_VTH) d = -dg;
            else if (s.kind == SP_KP) d = ich / p[P->p_mos_kp + k];
            else if (s.kind == SP_MW) d = ich / p[P->p_mos_w + k];
            else d = -ich / p[P->p_mos_l + k];
            r[0] = s.i0; r[1] = s.i2; di[0] = s.m * d; di[1] = -s.m * d;
            break;
        }
        case SP_VSRC:     // branch row: V - Vs; Vs is the DC value in DC mode or for a DC source
            if (mode == CS_MODE_DCOP || s.dev) { r[0] = s.i0; di[0] = -1.0; }
            break;
        case SP_ISRC:     // +m val on a, -m val on b
            if (mode == CS_MODE_DCOP || s.dev) { r[0] = s.i0; r[1] = s.i1; di[0] = s.m; di[1] = -s.m; }
            break;
        default:
            break;
    }
}

__global__ __launch_bounds__(kSensThreads) void k_sens(SensArgs A) {
    constexpr int NT = kSensThreads;   // not the transient kernels' NT
    const DPlan* P = A.P;
    const int n = P->n, j = blockIdx.x, tid = threadIdx.x;
    if (j >= A.n_sp) return;
    double* x = A.x + (size_t)j * n;
    const double* dq1 = A.dq1 ? A.dq1 + (size_t)j * n : nullptr;
    const double* dq2 = A.dq2 ? A.dq2 + (size_t)j * n : nullptr;
    const double* pin = A.pin_s ? A.pin_s + (size_t)j * n : nullptr;
    // history part, by pivot row
    for (int k = tid; k < n; k += NT) {
        const int r = P->rownat[k];
        if (A.pinned && P->is_diff[r]) {
            x[k] = pin ? pin[r] : 0.0;
        } else {
            double h = 0.0;
            if (dq1) h += A.a1 * dq1[r];
            if (dq2) h += A.a2 * dq2[r];
            x[k] = -h;
        }
    }
    __syncthreads();
    int32_t rr[2];
    double di[2], dq[2];
    param_stamps(P, A.p, A.u, A.sp[j], A.mode, rr, di, dq);
    if (tid == 0)
        for (int q = 0; q < 2; q++) {
            if (rr[q] < 0) continue;
            const int k = A.prow[rr[q]];
            if (A.pinned && P->is_diff[rr[q]]) continue;
            x[k] -= di[q] + A.a0 * dq[q];
        }
    __syncthreads();
    dev_fwd<NT>(P, A.F, x);
    dev_bwd<NT>(P, A.F, A.inv, x);
    double* s = A.s + (size_t)j * n;
    for (int i = tid; i < n; i += NT) s[i] = x[P->pcol[i]];
    __syncthreads();
    double* q0 = A.dq0 + (size_t)j * n;
    for (int k = tid; k < n; k += NT) {
        double acc = 0.0;
        for (int e = P->rowptr[k]; e < P->rowptr[k + 1]; e++) acc += A.Clin[e] * s[P->colnat[e]];
        q0[P->rownat[k]] = acc;
    }
    __syncthreads();
    if (tid == 0)
        for (int q = 0; q < 2; q++)
            if (rr[q] >= 0) q0[rr[q]] += dq[q];
}

// The sensitivity of one parameter beside a transient (run_instance's Rec):
// k_sens's solves at the DC point, at the initial point and at each accepted
// step, on the instance's own LU in LDS.  Lane i holds unknown i's
// sensitivity at the last three points.
template <bool FineGrid>
struct SensRec {
    static constexpr bool kFineGrid = FineGrid;
    const SensRunArgs& A;
    const int j;
    double *sn, *d1, *d2;          // LDS: s at the new point; charge sensitivities one and two steps back
    double pin = 0.0, s0 = 0.0, s1 = 0.0, s2 = 0.0;

    __device__ __forceinline__ bool writes() const { return j == 0; }
    // J s = -(dI/dp + a0 dQ/dp + a1 d1 + a2 d2) on the Jacobian assembled in L.F
    __device__ void solve(const DPlan* P, const double* p, const Lds& L, const double* Clin, int mode, bool pinned,
                          double a0, double a1, double a2) {
        const int n = P->n, i = threadIdx.x;
        if (i < n) sn[i] = pin;
        __syncthreads();
        dev_lu<NT>(P, L.F, L.inv);
        if (i < n) {
            const int r = P->rownat[i];
            L.x[i] = pinned && P->is_diff[r] ? sn[r] : -(a1 * d1[r] + a2 * d2[r]);
        }
        __syncthreads();
        int32_t rr[2];
        double di[2], dq[2];
        param_stamps(P, p, L.u, A.sp[j], mode, rr, di, dq);
        if (i == 0)
            for (int q = 0; q < 2; q++)
                if (rr[q] >= 0 && !(pinned && P->is_diff[rr[q]])) L.x[A.prow[rr[q]]] -= di[q] + a0 * dq[q];
        __syncthreads();
        dev_fwd<NT>(P, L.F, L.x);
        dev_bwd<NT>(P, L.F, L.inv, L.x);
        s2 = s1; s1 = s0;
        s0 = i < n ? L.x[P->pcol[i]] : 0.0;
        if (i < n) sn[i] = s0;
        __syncthreads();
        // the charge sensitivities C s + dQ/dp; the lane's own row is k's natural one
        if (i < n) {
            double acc = 0.0;
            for (int e = P->rowptr[i]; e < P->rowptr[i + 1]; e++) acc += Clin[e] * sn[P->colnat[e]];
            const int r = P->rownat[i];
            for (int q = 0; q < 2; q++)
                if (rr[q] == r) acc += dq[q];
            d2[r] = d1[r];
            d1[r] = acc;
        }
        __syncthreads();
    }
    __device__ void on_dc(const DPlan* P, const double* p, const Lds& L, const double* Clin) {
        solve(P, p, L, Clin, CS_MODE_DCOP, false, 0.0, 0.0, 0.0);
        pin = s0;
    }
    __device__ void on_initial(const DPlan* P, const double* p, const Lds& L, const double* Clin, bool uic) {
        if (uic) pin = 0.0;
        solve(P, p, L, Clin, CS_MODE_TRAN, true, 0.0, 0.0, 0.0);
    }
    __device__ void on_step(const DPlan* P, const double* p, const Lds& L, const double* Glin, const double* Clin,
                            double gmin, int k, double a0, double a1, double a2) {
        dev_mos<NT>(P, p, L.u, L.st, gmin);
        __syncthreads();
        dev_assemble<NT>(P, Glin, Clin, a0, L.u, L.qx, L.st, L.F, L.x, nullptr);
        solve(P, p, L, Clin, CS_MODE_TRAN, false, a0, a1, k == 2 ? a2 : 0.0);
    }
    __device__ void on_output(const DPlan* P, int kout, double l0, double l1, double l2) {
        const int i = threadIdx.x;
        const int sl = i < P->n ? P->probe_slot[i] : -1;
        if (sl >= 0) A.sens[((size_t)kout * A.n_sp + j) * A.n_probe + sl] = l0 * s0 + l1 * s1 + l2 * s2;
    }
    __device__ void on_outputs(const int32_t (&ps)[1], int kout, int m, double l0, double l1, double l2) {
        const double a[1] = {s0}, b[1] = {s1}, c[1] = {s2};
        put_rows<1>(A.sens + (size_t)j * A.n_probe, (size_t)A.n_sp * A.n_probe, kout, m, l0, l1, l2, ps, a, b, c);
    }
};

// One wavefront per parameter, each running the whole transient with its own
// parameter's sensitivity: they take the same steps, and the first one's
// waveform, state and statistics stand for all.  The run is a serial chain of small
// steps, and the chip is otherwise idle: repeating the transient per
// parameter costs nothing, while host step control cost a graph launch and a
// round trip per Newton iteration and another of each per accepted step.
// An inverter over 1 ns with six parameters: 82.5 -> 12.9 ms.
template <bool FineGrid>
__global__ __launch_bounds__(NT) void k_tran_sens(SensRunArgs A) {
    extern __shared__ double lds[];
    const int j = blockIdx.x;
    if (j >= A.n_sp) return;
    Lds L;
    L.F = lds;
    L.inv = L.F + A.nnz;
    L.u = L.inv + A.n;
    L.x = L.u + A.n;
    L.qx = L.x + A.n;
    L.st = L.qx + A.n;
    double* sn = L.st + A.n_stamp;
    SensRec<FineGrid> rec{A, j, sn, sn + A.n, sn + 2 * A.n};
    if ((int)threadIdx.x < A.n) rec.d1[threadIdx.x] = rec.d2[threadIdx.x] = 0.0;
    double* lin = A.ws + (size_t)j * A.ws_stride;
    run_instance<1, false>(rec, A.P, A.p, A.u0, A.wave, A.u_final, A.stats, A.o, L, lin + A.n_lin,
                    lin + A.n_lin + A.nnz, lin);
}

}  // namespace

size_t tran_sens_lds(int32_t n, int32_t nnz, int32_t n_stamp) {
    return sizeof(double) * ((size_t)nnz + 7 * (size_t)n + (size_t)n_stamp);
}

hipError_t launch_tran_sens(const SensRunArgs& a, hipStream_t s) {
    // 0.45 us a sample written one by one, 4 % of a run for the other form: an
    // inverter's 13 ms, so the line lies where they cost the same
    const size_t lds = tran_sens_lds(a.n, a.nnz, a.n_stamp);
    if (a.o.n_out > 1024) hipLaunchKernelGGL(k_tran_sens<true>, dim3(a.n_sp), dim3(NT), lds, s, a);
    else hipLaunchKernelGGL(k_tran_sens<false>, dim3(a.n_sp), dim3(NT), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_sens(const SensArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_sens, dim3(a.n_sp), dim3(kSensThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace cedar
