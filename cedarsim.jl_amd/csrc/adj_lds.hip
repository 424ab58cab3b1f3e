// adj_lds.hip — batched discrete adjoint on the LDS-resident kernel.
//
// Objective per instance: energy delivered by one voltage source,
//     E = sum_m w_m P(u_m),  P(u) = -(V(a) - V(b)) * I_src,
// trapezoid weights on the accepted time points; parameters: every MOSFET
// width.  Two persistent kernels per size class, one wavefront per instance,
// the circuit's plan image in LDS (lds_core.h):
//
//   k_adj_lds_forward  the transient of run_lds with a recording policy:
//                      every accepted time and segment count goes to a step
//                      log, E is integrated, and every K accepted steps the
//                      three states the predictor needs are checkpointed;
//   k_adj_lds_reverse  walks the segments [sK, (s+1)K) from the last one
//                      back: restores checkpoint s, recomputes the segment's
//                      states from the log (same predictor and Newton, so
//                      the same bits), then for m descending solves
//                        J_m^T l_m = -( w_m dP/du(u_m) + a_{m+1,1} C^T l_{m+1}
//                                       + a_{m+2,2} C^T l_{m+2} )
//                      on J_m's LU with the transposed level schedules, and
//                      accumulates dE/dW_k += (l_m[d] - l_m[s]) * I_ch,k / W_k.
// Step 0 is the consistent-initialisation system (charge rows pinned), so
// the adjoint needs UIC.  C^T l is carried between steps in the registers of
// the lanes that own the columns and each device's gradient is accumulated
// by one lane in a fixed order, so results are bit-reproducible.
// Bound by the latency of the instance code (lds_core.h): 256 51-stage rings
// over 0.1 ns 208 ms with its earlier form, 100 ms.
#include "lds_core.h"

namespace cedar {

namespace {

using namespace lds;

// Recording policy of the forward pass; the arguments are read where a step
// is recorded, so that they hold no registers in the Newton loop.
struct AdjRec {
    ConstPtr<AdjLdsArgs> A;
    int inst, cid;
    double E, Pprev;
    long long M;

    template <int NR>
    __device__ __forceinline__ bool on_accept(Hdr c, const View& v, double tn, double tprev,
                                              int npts, long long m, const double (&Uh0)[NR],
                                              const double (&Uh1)[NR], const double (&Uh2)[NR]) {
        A = fresh(A);
        c = fresh(c);
        if (m >= A->cap) return false;
        if (lane_id() == 0) {
            A->t_log[(size_t)inst * A->cap + m] = tn;
            A->npts_log[(size_t)inst * A->cap + m] = npts;
        }
        // objective source: terminals and branch current (pivot columns)
        const uint32_t a = (uint32_t)A->obj[3 * cid], b = (uint32_t)A->obj[3 * cid + 1],
                       j = (uint32_t)A->obj[3 * cid + 2];
        const int bu = c->b_u;
        const double Pn = -((a != CP_GROUND ? v.at(bu + 8 * a) : 0.0) - (b != CP_GROUND ? v.at(bu + 8 * b) : 0.0)) *
                          v.at(bu + 8 * j);
        if (m > 0) E += 0.5 * (tn - tprev) * (Pn + Pprev);
        Pprev = Pn;
        M = m;
        const int K = A->K;
        if (m % K == 0) {
            const long long s = m / K;
            if (s >= A->ckcap) return false;
            const int ck_n = A->ck_n;
            double* cp = A->ckpt + ((size_t)inst * A->ckcap + s) * 3 * ck_n;
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = lane_id() + W * r;
                if (k < c->n) {
                    cp[k] = Uh0[r];
                    cp[ck_n + k] = Uh1[r];
                    cp[2 * ck_n + k] = Uh2[r];
                }
            }
        }
        return true;
    }
};

__device__ __forceinline__ void step_coeffs(const double* tl, const int32_t* npl, long long q,
                                            int max_order, double& a0, double& a1, double& a2) {
    const int k = bdf_order(npl[q], max_order);
    bdf_coeffs(k, tl[q], tl[q - 1], q >= 2 ? tl[q - 2] : 0.0, a0, a1, a2);
}

template <int NR, bool DYN>
__global__ __launch_bounds__(W) void k_adj_lds_forward(const AdjLdsArgs* args) {
    extern __shared__ double lds_mem[];
    ConstPtr<AdjLdsArgs> A = as_const(args);
    uint16_t* blob = reinterpret_cast<uint16_t*>(lds_mem + A->f.dbl_max);
    int cur = -1;
    for (;;) {
        A = fresh(A);
        int qi = 0;
        if (threadIdx.x == 0) qi = atomicAdd(A->f.queue, 1);
        qi = __builtin_amdgcn_readfirstlane(qi);
        if (qi >= A->f.n_inst) break;
        const int inst = __builtin_amdgcn_readfirstlane(A->f.order[qi]);
        const int cid = __builtin_amdgcn_readfirstlane(A->f.inst_cid[inst]);
        Hdr c = as_const(A->f.cplans + cid);
        if (cid != cur) {
            copy_image(c->blob, c->words, blob, lane_id(), W);
            cur = cid;
            lds_sync();
        }
        const View v{reinterpret_cast<char*>(lds_mem), blob};
        AdjRec rec{A, inst, cid, 0.0, 0.0, 0};
        run_lds<NR, DYN, (NR <= 2)>(rec, c, &A->f, A->f.plans + cid, inst, v);
        if (threadIdx.x == 0) {
            A->energy[inst] = rec.E;
            A->n_steps[inst] = rec.M;
        }
    }
}

template <int NR, bool DYN>
__device__ __forceinline__ void run_reverse(ConstPtr<AdjLdsArgs> A, Hdr c, const DPlan* __restrict__ P,
                            const double* __restrict__ p, const double* __restrict__ u0, int inst,
                            int cid, const View& v, double* __restrict__ seg) {
    constexpr int NM = 2 * NR;
    const int tid = lane_id();
    const int n = c->n, bu = c->b_u, bx = c->b_x, bst = c->b_st;
    const long long M = A->n_steps[inst];
    const int K = A->K;
    const int ck_n = A->ck_n;
    const double* tl = A->t_log + (size_t)inst * A->cap;
    const int32_t* npl = A->npts_log + (size_t)inst * A->cap;
    const double* ck = A->ckpt + (size_t)inst * A->ckcap * 3 * ck_n;
    double* grad = A->grad + A->g_off[inst];
    const uint32_t oa = (uint32_t)A->obj[3 * cid], ob = (uint32_t)A->obj[3 * cid + 1],
                   oj = (uint32_t)A->obj[3 * cid + 2];

    DevRegs<NM> dr;
    setup_instance<NM>(c, P, p, v, dr);
    const double gmin = p[P->p_gmin];
    // per device slot: width, drain / source pivot rows (and whether those
    // rows are pinned at step 0), gradient accumulator
    double wdt[NM], gacc[NM];
    uint32_t drow[NM], srow[NM], pin0[NM];
#pragma unroll
    for (int jd = 0; jd < NM; jd++) {
        const int m = tid + W * jd;
        wdt[jd] = 1.0;
        gacc[jd] = 0.0;
        drow[jd] = srow[jd] = CP_GROUND;
        pin0[jd] = 0;
        if (m < c->n_mos) {
            wdt[jd] = p[P->p_mos_w + m];
            drow[jd] = (uint32_t)c->devrow[2 * m];
            srow[jd] = (uint32_t)c->devrow[2 * m + 1];
            if (drow[jd] != CP_GROUND && c->diffrow[drow[jd]]) pin0[jd] |= 1;
            if (srow[jd] != CP_GROUND && c->diffrow[srow[jd]]) pin0[jd] |= 2;
        }
    }
    double pinv[NR], ctl1[NR], ctl2[NR];
    uint32_t flag[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = tid + W * r;
        pinv[r] = ctl1[r] = ctl2[r] = 0.0;
        flag[r] = 0;
        if (k < n) {
            pinv[r] = u0[c->colnat[k]];
            flag[r] = c->diffrow[k] ? 1u : 0u;
        }
    }
    lds_sync();
    long long nit = 0;

    for (long long s = M / K; s >= 0; s--) {
        const long long m0 = s * K;
        const long long m1 = (m0 + K < M + 1) ? m0 + K : M + 1;
        double U0[NR], U1[NR], U2[NR], Q0[NR], Q1[NR], qx[NR];
        const double* cp = ck + (size_t)s * 3 * ck_n;
        lds_sync();   // the previous segment's last step still reads u
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k = row_of(tid, r, n);   // lanes past the last row carry a copy of it
            U0[r] = cp[k];
            U1[r] = cp[ck_n + k];
            U2[r] = cp[2 * ck_n + k];
            qx[r] = 0.0;
            seg[k] = U0[r];
            v.at(bu + 8 * k) = U1[r];
        }
        lds_sync();
#pragma unroll
        for (int r = 0; r < NR; r++) {
            Q1[r] = row_charge(c, v, row_of(tid, r, n));
        }
        lds_sync();
#pragma unroll
        for (int r = 0; r < NR; r++) {
            v.at(bu + 8 * row_of(tid, r, n)) = U0[r];
        }
        lds_sync();
#pragma unroll
        for (int r = 0; r < NR; r++) {
            Q0[r] = row_charge(c, v, row_of(tid, r, n));
        }
        // ---- recompute the segment's states from the log -------------------
        for (long long m = m0 + 1; m < m1; m++) {
            const int npts = npl[m];
            const int k = bdf_order(npts, A->f.o.max_order);
            const double tn = tl[m], T0 = tl[m - 1];
            const double T1 = m >= 2 ? tl[m - 2] : 0.0, T2 = m >= 3 ? tl[m - 3] : 0.0;
            double a0, a1, a2, w0, w1, w2;
            step_bdf(k, tn, T0, T1, a0, a1, a2);
            const int np = npts < k + 1 ? npts : k + 1;
            step_pred(np, tn, T0, T1, T2, w0, w1, w2);
            lds_sync();
#pragma unroll
            for (int r = 0; r < NR; r++) {
                double val = U0[r];
                if (np == 2) val = __builtin_fma(w0, U0[r], w1 * U1[r]);
                else if (np == 3) val = __builtin_fma(w0, U0[r], __builtin_fma(w1, U1[r], w2 * U2[r]));
                v.at(bu + 8 * row_of(tid, r, n)) = val;
                qx[r] = __builtin_fma(a1, Q0[r], k == 2 ? a2 * Q1[r] : 0.0);
            }
            eval_sources<DYN>(c, v, tn, CS_MODE_TRAN);
            lds_sync();
            A = fresh(A);
            newton<NR, NM, (NR <= 2)>(c, v, dr, gmin, a0, qx, A->f.o.newton_maxit, A->f.o.newton_tol, A->f.o.reltol,
                           A->f.o.abstol, nit);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int kk = row_of(tid, r, n);
                U2[r] = U1[r]; U1[r] = U0[r]; U0[r] = v.at(bu + 8 * kk);
                Q1[r] = Q0[r]; Q0[r] = row_charge(c, v, kk);
                seg[(size_t)(m - m0) * ck_n + kk] = U0[r];
            }
        }
        // ---- backward over the segment ------------------------------------
        for (long long m = m1 - 1; m >= m0; m--) {
            lds_sync();
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = tid + W * r;
                if (k < n) v.at(bu + 8 * k) = seg[(size_t)(m - m0) * ck_n + k];
            }
            A = fresh(A);
            const int max_order = A->f.o.max_order;
            const double tm = tl[m];
            double w = 0.0;
            if (m > 0) w += 0.5 * (tm - tl[m - 1]);
            if (m < M) w += 0.5 * (tl[m + 1] - tm);
            double c1 = 0.0, c2 = 0.0, b0, b1, b2;
            if (m + 1 <= M) { step_coeffs(tl, npl, m + 1, max_order, b0, b1, b2); c1 = b1; }
            if (m + 2 <= M) { step_coeffs(tl, npl, m + 2, max_order, b0, b1, b2); c2 = b2; }
            double am0 = 0.0;
            if (m > 0) step_coeffs(tl, npl, m, max_order, am0, b1, b2);
            eval_sources<DYN>(c, v, tm, CS_MODE_TRAN);
            lds_sync();
            const Hot h = load_hot(c);
            eval_mos<NM, (NR <= 2)>(h, v, dr, gmin);
            lds_sync();
            double qz[NR];
#pragma unroll
            for (int r = 0; r < NR; r++) qz[r] = 0.0;
            assemble<NR, (NR <= 2)>(h, v, am0, qz);
            if (m == 0) apply_pins<NR>(c, v, P, pinv, flag);
            lds_sync();
            factor<(NR <= 2)>(h, v);
            const double ua = oa != CP_GROUND ? v.at(bu + 8 * oa) : 0.0;
            const double ub = ob != CP_GROUND ? v.at(bu + 8 * ob) : 0.0, uj = v.at(bu + 8 * oj);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = tid + W * r;
                if (k < n) {
                    double dP = 0.0;
                    if ((uint32_t)k == oa) dP -= uj;
                    if ((uint32_t)k == ob) dP += uj;
                    if ((uint32_t)k == oj) dP -= (ua - ub);
                    v.at(bx + 8 * k) = -w * dP - c1 * ctl1[r] - c2 * ctl2[r];
                }
            }
            lds_sync();
            solve_transposed(c, v);
            // C^T lambda for this lane's columns
            double ctl[NR];
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = tid + W * r;
                ctl[r] = k < n ? col_charge_t(c, v, k) : 0.0;
            }
            // dE/dW: lambda of the drain and source rows times I_ch / W
#pragma unroll
            for (int jd = 0; jd < NM; jd++) {
                const int md = tid + W * jd;
                if (md < c->n_mos) {
                    const uint32_t pz = m == 0 ? pin0[jd] : 0u;
                    const double ld = (drow[jd] != CP_GROUND && !(pz & 1)) ? v.at(bx + 8 * drow[jd]) : 0.0;
                    const double ls = (srow[jd] != CP_GROUND && !(pz & 2)) ? v.at(bx + 8 * srow[jd]) : 0.0;
                    const double vd = v.at(dr.dg[jd] & 0xFFFF), vs = v.at(dr.sx[jd] & 0xFFFF);
                    // channel current: the stamp minus the (m-scaled) gmin term
                    const double gm = c->mos_m ? gmin * c->mos_m[md] : gmin;
                    const double ich = v.at(bst + 8 * md) - gm * (vd - vs);
                    gacc[jd] += (ld - ls) * ich / wdt[jd];
                }
            }
#pragma unroll
            for (int r = 0; r < NR; r++) {
                ctl2[r] = ctl1[r];
                ctl1[r] = ctl[r];
            }
        }
    }
#pragma unroll
    for (int jd = 0; jd < NM; jd++) {
        const int md = tid + W * jd;
        if (md < c->n_mos) grad[md] = gacc[jd];
    }
    lds_sync();
}

template <int NR, bool DYN>
__global__ __launch_bounds__(W) void k_adj_lds_reverse(const AdjLdsArgs* args) {
    extern __shared__ double lds_mem[];
    ConstPtr<AdjLdsArgs> A = as_const(args);
    uint16_t* blob = reinterpret_cast<uint16_t*>(lds_mem + A->f.dbl_max);
    double* seg = A->seg + (size_t)blockIdx.x * A->K * A->ck_n;
    int cur = -1;
    for (;;) {
        A = fresh(A);
        int qi = 0;
        if (threadIdx.x == 0) qi = atomicAdd(A->queue2, 1);
        qi = __builtin_amdgcn_readfirstlane(qi);
        if (qi >= A->f.n_inst) break;
        const int inst = __builtin_amdgcn_readfirstlane(A->f.order[qi]);
        const int cid = __builtin_amdgcn_readfirstlane(A->f.inst_cid[inst]);
        const int rc = __builtin_amdgcn_readfirstlane(A->f.stats[inst].retcode);
        if (rc != CS_OK) continue;
        Hdr c = as_const(A->f.cplans + cid);
        if (cid != cur) {
            copy_image(c->blob, c->words_adj, blob, lane_id(), W);
            cur = cid;
            lds_sync();
        }
        const View v{reinterpret_cast<char*>(lds_mem), blob};
        run_reverse<NR, DYN>(A, c, A->f.plans + cid, A->f.params + A->f.p_off[inst], A->f.u0 + A->f.u_off[inst], inst, cid,
                        v, seg);
    }
}

}  // namespace

namespace {
typedef void (*AdjKernel)(const AdjLdsArgs*);
template <bool DYN>
AdjKernel adj_kernel(int nr, bool reverse) {
    switch (nr) {
        case 1: return reverse ? k_adj_lds_reverse<1, DYN> : k_adj_lds_forward<1, DYN>;
        case 2: return reverse ? k_adj_lds_reverse<2, DYN> : k_adj_lds_forward<2, DYN>;
        case 4: return reverse ? k_adj_lds_reverse<4, DYN> : k_adj_lds_forward<4, DYN>;
        default: return nullptr;
    }
}
AdjKernel adj_kernel(int nr, bool dyn, bool reverse) {
    return dyn ? adj_kernel<true>(nr, reverse) : adj_kernel<false>(nr, reverse);
}
}  // namespace

int adj_lds_max_blocks(int nr, bool dyn, bool reverse, size_t lds) {
    int nb = 0;
    const AdjKernel f = adj_kernel(nr, dyn, reverse);
    if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, W, lds) != hipSuccess) return 0;
    return nb;
}

hipError_t launch_adj_lds(int nr, bool dyn, bool reverse, const AdjLdsArgs* a, int nblocks, size_t lds, hipStream_t s) {
    const AdjKernel f = adj_kernel(nr, dyn, reverse);
    if (!f) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f, dim3(nblocks), dim3(W), lds, s, a);
    return hipGetLastError();
}

}  // namespace cedar
