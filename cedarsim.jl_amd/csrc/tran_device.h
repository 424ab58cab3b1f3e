// tran_device.h — the per-instance transient loop of the global-plan batched
// kernel (k_tran_batch, kernels.hip), which reads the plan from global
// memory in natural unknown order.  One workgroup of NT = 64 threads (one
// wavefront) owns one circuit instance; lane l owns unknowns l, l+64, ...
// (NR of them) and keeps their history in registers.
//
// VA: some circuit has Verilog-A devices; without, their models' code is left
// out.  Rec is called at the points a forward sensitivity run needs (sens.hip): the
// DC point and the initial point, each with its Jacobian just assembled in
// L.F, every accepted step, and every output sample; the batch passes NoRec.
// Rec::kFineGrid writes the samples of a step together (put_samples), for
// output grids finer than the steps; it costs the run 4 %.
// Rec::writes is false for a workgroup that repeats another's run: waveform,
// state and statistics are that one's to write.
#pragma once
#include "dcop_rules.h"
#include "device.h"
#include "kernels.h"

namespace cedar {

constexpr int NT = kBatchThreads;

struct Lds {
    double *F, *inv, *u, *x, *qx, *st;
};

struct NoRec {
    static constexpr bool kFineGrid = false;
    __device__ __forceinline__ bool writes() const { return true; }
    __device__ __forceinline__ void on_dc(const DPlan*, const double*, const Lds&, const double*) {}
    __device__ __forceinline__ void on_initial(const DPlan*, const double*, const Lds&, const double*, bool) {}
    __device__ __forceinline__ void on_step(const DPlan*, const double*, const Lds&, const double*, const double*,
                                            double, int, double, double, double) {}
    __device__ __forceinline__ void on_output(const DPlan*, int, double, double, double) {}
};

template <int NR, bool VA, class Rec>
__device__ void run_instance(Rec& rec, const DPlan* __restrict__ P, const double* __restrict__ p,
                             const double* __restrict__ u0, double* __restrict__ wave,
                             double* __restrict__ ufin, cs_tran_stats* __restrict__ stp,
                             const cs_tran_opts& o, const Lds& L, double* __restrict__ Glin,
                             double* __restrict__ Clin, double* __restrict__ linbuf) {
    const int tid = threadIdx.x;
    const int n = P->n;
    const StepDefaults sd = step_defaults(o);
    dev_lin_setup<NT>(P, p, linbuf, Glin, Clin);

    double Uh0[NR], Uh1[NR], Uh2[NR], Qh0[NR], Qh1[NR], up[NR];
    long long steps = 0, rej = 0, nit = 0;
    int rc = CS_OK;
    const bool uic = (o.init == CS_INIT_UIC) && u0 != nullptr;
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int i = tid + NT * r;
        Uh0[r] = Uh1[r] = Uh2[r] = Qh0[r] = Qh1[r] = up[r] = 0.0;
        if (i < n) L.u[i] = uic ? u0[i] : 0.0;
    }
    __syncthreads();

    // ---- consistent initial point -------------------------------------
    // UIC: charge rows pinned to u0, 50 iterations.  CedarDCOp: the
    // trajectories and the gmin ladder of dcop_rules.h (src/dcop.jl:53-94),
    // then the charge rows pinned to the DC point and the algebraic rows
    // solved with the sources at t0 (its BrownFullBasicInit step, :153); one
    // Newton loop over the phases as in the LDS kernel.  The pinned values
    // of the second step are kept in L.qx, free until the charges are set.
    const double gmin = p[P->p_gmin];
    {
        dev_sources<NT, true>(P, p, o.t_start, uic ? CS_MODE_TRAN : CS_MODE_DCOP, L.st);
        int phase = uic ? -1 : 0, stage = 0, it = 0;
        const double* pin = uic ? u0 : nullptr;
        double g = gmin;
        if (!uic)
            for (int i = tid; i < n; i += NT) L.u[i] = dc_start(0, i);
        __syncthreads();
        bool ok = false;
        for (;;) {
            dev_mos<NT>(P, p, L.u, L.st, g);
            if constexpr (VA) dev_va<NT>(P, p, L.u, L.st, g);
            __syncthreads();
            const double lm = dev_assemble<NT>(P, Glin, Clin, 0.0, L.u, nullptr, L.st, L.F, L.x, pin);
            const double fn = block_reduce<NT>(lm, nullptr, OpMax());
            __syncthreads();
            if (fn <= o.dc_abstol) {
                bool dc_done = phase >= 0 && phase < kDcTrajectories;
                if (phase >= kDcTrajectories) {
                    g = dc_gmin_stage(++stage, gmin);
                    dc_done = g < 0.0;
                    if (!dc_done) {
                        it = 0;
                        continue;
                    }
                }
                if (!dc_done) { ok = true; break; }
                rec.on_dc(P, p, L, Clin);
                for (int i = tid; i < n; i += NT) L.qx[i] = L.u[i];
                dev_sources<NT, true>(P, p, o.t_start, CS_MODE_TRAN, L.st);
                pin = L.qx;
                phase = -1;
                g = gmin;
                it = 0;
                __syncthreads();
                continue;
            }
            const int maxit = phase < 0 ? 50 : kDcMaxIt;
            if (!(fn == fn) || __builtin_isinf(fn) || it >= maxit) {
                if (phase < 0 || phase >= kDcTrajectories) break;
                phase++;
                const int j = phase < kDcTrajectories ? phase : 0;
                for (int i = tid; i < n; i += NT) L.u[i] = dc_start(j, i);
                if (phase >= kDcTrajectories) {
                    stage = 0;
                    g = dc_gmin_stage(0, gmin);
                }
                it = 0;
                __syncthreads();
                continue;
            }
            dev_lu<NT>(P, L.F, L.inv);
            dev_fwd<NT>(P, L.F, L.x);
            dev_bwd<NT>(P, L.F, L.inv, L.x);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int i = tid + NT * r;
                if (i < n) L.u[i] += L.x[P->pcol[i]];
            }
            nit++;
            it++;
            __syncthreads();
        }
        if (!ok) rc = CS_E_NOCONV;
    }

    double t = o.t_start;
    if (rc == CS_OK) {
        __syncthreads();
        rec.on_initial(P, p, L, Clin, uic);
        dev_charges<NT>(P, Clin, L.u, L.qx);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int i = tid + NT * r;
            if (i < n) { Uh0[r] = L.u[i]; Qh0[r] = L.qx[i]; }
        }
        double T0 = o.t_start, T1 = 0.0, T2 = 0.0;
        int npts = 1;
        double h = sd.dt_init;
        int kout = 0;
        const int n_probe = P->n_probe;
        if (wave) {
            while (kout < o.n_out && out_due(out_time(o.t_start, kout, o.dt_out), o.t_start, o.dt_out)) {
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const int i = tid + NT * r;
                    if (i < n) {
                        const int sl = P->probe_slot[i];
                        if (sl >= 0 && rec.writes()) wave[(size_t)kout * n_probe + sl] = Uh0[r];
                    }
                }
                rec.on_output(P, kout, 1.0, 0.0, 0.0);
                kout++;
            }
        }
        __syncthreads();
        while (t < o.t_stop) {
            if (steps + rej >= o.max_steps) { rc = CS_E_MAXSTEPS; break; }
            double lb = INFINITY;
            for (int s = tid; s < P->n_src; s += NT) {
                const int4 d = P->src[s];
                const double b = next_bp(d.x, p + d.y, d.z, t);
                if (b < lb) lb = b;
            }
            double tb = block_reduce<NT>(lb, nullptr, OpMin());
            const bool srcbp = tb < o.t_stop;
            if (!srcbp) tb = o.t_stop;
            double hh = h < sd.dt_max ? h : sd.dt_max;
            int hit;
            const double tn = clip_step(t, hh, tb, hit);
            const int k = bdf_order(npts, o.max_order);
            double a0, a1, a2, w0, w1, w2;
            bdf_coeffs(k, tn, T0, T1, a0, a1, a2);
            const int np = npts < k + 1 ? npts : k + 1;
            pred_weights(np, tn, T0, T1, T2, w0, w1, w2);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int i = tid + NT * r;
                if (i < n) {
                    double v = Uh0[r];
                    if (np == 2) v = w0 * Uh0[r] + w1 * Uh1[r];
                    else if (np == 3) v = w0 * Uh0[r] + w1 * Uh1[r] + w2 * Uh2[r];
                    up[r] = v;
                    L.u[i] = v;
                    L.qx[i] = a1 * Qh0[r] + (k == 2 ? a2 * Qh1[r] : 0.0);
                }
            }
            dev_sources<NT, true>(P, p, tn, CS_MODE_TRAN, L.st);
            __syncthreads();
            bool conv = false;
            for (int it = 0; it < o.newton_maxit; it++) {
                dev_mos<NT>(P, p, L.u, L.st, gmin);
                if constexpr (VA) dev_va<NT>(P, p, L.u, L.st, gmin);
                __syncthreads();
                dev_assemble<NT>(P, Glin, Clin, a0, L.u, L.qx, L.st, L.F, L.x, nullptr);
                __syncthreads();
                dev_lu<NT>(P, L.F, L.inv);
                dev_fwd<NT>(P, L.F, L.x);
                dev_bwd<NT>(P, L.F, L.inv, L.x);
                nit++;
                double ss = 0.0;
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const int i = tid + NT * r;
                    if (i < n) {
                        const double d = L.x[P->pcol[i]];
                        const double ui = L.u[i] + d;
                        L.u[i] = ui;
                        const double q = d / (o.reltol * fabs(ui) + o.abstol);
                        ss += q * q;
                    }
                }
                const double nr = sqrt(block_reduce<NT>(ss, nullptr, OpSum()) / n);
                __syncthreads();
                if (!(nr == nr)) break;
                if (nr <= o.newton_tol) { conv = true; break; }
            }
            if (!conv) {
                rej++;
                h = 0.25 * hh;
                if (h < sd.dt_min) { rc = CS_E_DTMIN; break; }
                continue;
            }
            double fac = 2.0;
            if (npts >= 2) {
                const double c = lte_coeff(k, tn, T0, T1, T2, a0, a1, a2);
                double ss = 0.0;
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const int i = tid + NT * r;
                    if (i < n) {
                        const double ui = L.u[i];
                        const double est = c * (ui - up[r]);
                        const double m = fabs(ui) > fabs(Uh0[r]) ? fabs(ui) : fabs(Uh0[r]);
                        const double q = est / (o.reltol * m + o.abstol);
                        ss += q * q;
                    }
                }
                const double err2 = block_reduce<NT>(ss, nullptr, OpSum()) / n;
                if (!(err2 <= 1.0)) {
                    rej++;
                    h = hh * step_reject(err2, k);
                    if (h < sd.dt_min) { rc = CS_E_DTMIN; break; }
                    continue;
                }
                fac = step_accept(err2, k);
            }
            // accept
            rec.on_step(P, p, L, Glin, Clin, gmin, k, a0, a1, a2);
            dev_charges<NT>(P, Clin, L.u, L.qx);
            __syncthreads();
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int i = tid + NT * r;
                if (i < n) {
                    Uh2[r] = Uh1[r]; Uh1[r] = Uh0[r]; Uh0[r] = L.u[i];
                    Qh1[r] = Qh0[r]; Qh0[r] = L.qx[i];
                }
            }
            T2 = T1; T1 = T0; T0 = tn;
            if (npts < 3) npts++;
            steps++;
            auto weights = [&](double tq, double& l0, double& l1, double& l2) {
                l2 = 0.0;
                if (npts >= 3) {
                    l0 = (tq - T1) * (tq - T2) / ((T0 - T1) * (T0 - T2));
                    l1 = (tq - T0) * (tq - T2) / ((T1 - T0) * (T1 - T2));
                    l2 = (tq - T0) * (tq - T1) / ((T2 - T0) * (T2 - T1));
                } else {
                    const double s = (tq - T1) / (T0 - T1);
                    l0 = s;
                    l1 = 1.0 - s;
                }
            };
            if constexpr (Rec::kFineGrid) {
                if (wave)
                    put_samples(kout, o.t_start, o.dt_out, o.n_out, tn, weights,
                                [&](int k0, int m, double l0, double l1, double l2) {
                                    int32_t ps[NR];
#pragma unroll
                                    for (int r = 0; r < NR; r++)
                                        ps[r] = tid + NT * r < n ? P->probe_slot[tid + NT * r] : -1;
                                    if (rec.writes()) put_rows<NR>(wave, n_probe, k0, m, l0, l1, l2, ps, Uh0, Uh1, Uh2);
                                    rec.on_outputs(ps, k0, m, l0, l1, l2);
                                });
            } else if (wave) {
                while (kout < o.n_out) {
                    const double tq = out_time(o.t_start, kout, o.dt_out);
                    if (!out_due(tq, tn, o.dt_out)) break;
                    double l0, l1, l2;
                    weights(tq, l0, l1, l2);
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        const int i = tid + NT * r;
                        if (i < n) {
                            const int sl = P->probe_slot[i];
                            if (sl >= 0 && rec.writes())
                                wave[(size_t)kout * n_probe + sl] =
                                    l0 * Uh0[r] + l1 * Uh1[r] + l2 * Uh2[r];
                        }
                    }
                    rec.on_output(P, kout, l0, l1, l2);
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
    if (!rec.writes()) return;
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int i = tid + NT * r;
        if (i < n) ufin[i] = (rc == CS_OK || steps > 0) ? Uh0[r] : L.u[i];
    }
    if (tid == 0) {
        stp->steps = steps;
        stp->rejected = rej;
        stp->newton_iters = nit;
        stp->t_end = t;
        stp->retcode = rc;
        stp->pad = 0;
    }
    __syncthreads();
}

}  // namespace cedar
