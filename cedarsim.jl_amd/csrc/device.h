// device.h — device building blocks of one Newton iteration, written for a
// group of NT threads that owns one circuit instance (NT = 64: one wavefront,
// the batched kernel; NT = 256: the single-instance kernels).
//
//   eval       one lane per device instance: square-law MOSFET stamps
//              (id, dI/dVd, dI/dVg, dI/dVs) and source values into a stamp
//              buffer in LDS;
//   assemble   one lane per permuted row: Jacobian entries and residual are
//              gathered from fixed, ordered contributor lists into the CSR
//              slots of F (no atomics, bit-reproducible);
//   LU         entry-level level schedule, one barrier per level;
//   solves     level-scheduled forward / backward substitution (and the
//              transposed pair for adjoint solves).
#pragma once
#include "dplan.h"
#include "rules.h"
#include "va_registry.h"
#include "wave_math.h"

namespace cedar {

__device__ __forceinline__ double sref_val(const double* buf, int32_t r) {
    const double v = buf[r >> 1];
    return (r & 1) ? -v : v;
}

struct OpSum {
    __device__ double operator()(double a, double b) const { return a + b; }
};
struct OpMax {   // NaN-propagating max
    __device__ double operator()(double a, double b) const { return (a != a || a > b) ? a : b; }
};
struct OpMin {
    __device__ double operator()(double a, double b) const { return (a != a || a < b) ? a : b; }
};

// A double from another lane of the same row of 16 by a DPP move (CTRL a
// quad_perm, row_mirror or row_half_mirror pattern: every source lane is in
// the row, so no lane reads outside it).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffll), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Reduction over a full wavefront (every lane active) in a fixed order: within
// each row of 16 lanes by four DPP steps (partners xor 1 and xor 2 in the
// quad, then the other quad of the half-row, then the other half of the row),
// then the four row results, read from lanes 0, 16, 32 and 48, as
// op(op(r0, r1), op(r2, r3)).  The result is uniform.  DPP moves stay in the
// register file, where a lane shuffle would go through the LDS crossbar.
template <class Op>
__device__ __forceinline__ double wave_reduce(double v, Op op) {
    v = op(v, dpp_f64<0xB1>(v));    // quad_perm [1,0,3,2]
    v = op(v, dpp_f64<0x4E>(v));    // quad_perm [2,3,0,1]
    v = op(v, dpp_f64<0x141>(v));   // row_half_mirror
    v = op(v, dpp_f64<0x140>(v));   // row_mirror
    const double r0 = readlane_f64(v, 0), r1 = readlane_f64(v, 16);
    const double r2 = readlane_f64(v, 32), r3 = readlane_f64(v, 48);
    return op(op(r0, r1), op(r2, r3));
}

// Deterministic block reduction; every thread receives the same value.
template <int NT, class Op>
__device__ __forceinline__ double block_reduce(double v, double* red, Op op) {
    if constexpr (NT == 64) {
        return wave_reduce(v, op);
    } else {
        red[threadIdx.x] = v;
        __syncthreads();
#pragma unroll
        for (int s = NT / 2; s > 0; s >>= 1) {
            if ((int)threadIdx.x < s) red[threadIdx.x] = op(red[threadIdx.x], red[threadIdx.x + s]);
            __syncthreads();
        }
        const double r = red[0];
        __syncthreads();
        return r;
    }
}

// The output samples due at an accepted point tn, by one wavefront: up to 64
// of them at a time, their interpolation weights one sample per lane, then
// put(kout, m, l0, l1, l2) for samples kout .. kout + m - 1.
template <class Weights, class Put>
__device__ __forceinline__ void put_samples(int& kout, double t_start, double dt_out, int n_out, double tn,
                                            Weights weights, Put put) {
    while (kout < n_out && out_due(out_time(t_start, kout, dt_out), tn, dt_out)) {
        const int lane = (int)(threadIdx.x & 63);
        const double tq = out_time(t_start, kout + (lane < n_out - kout ? lane : 0), dt_out);
        const int m = __popcll(__ballot(lane < n_out - kout && out_due(tq, tn, dt_out)));
        double l0, l1, l2;
        weights(tq, l0, l1, l2);
        put(kout, m, l0, l1, l2);
        kout += m;
    }
}

// The put of rows held by the lanes: row r of a lane has the values U0, U1, U2
// at the last three points and goes to place ps[r] of a sample (-1: none).
// Few samples: one after the other, lanes over the rows.  More samples than
// rows (a fine grid): the rows one after the other, lanes over the samples.
// Written one by one a sample cost a whole pass of the wavefront, 225 ns:
// cs_tran of an inverter (five rows, 1 ns, 786,000 samples) took 169 ms, of
// which the run itself is 5; now 18.5, and six sensitivities of it at
// 1,000,001 samples 557 ms, now 63.
template <int NR>
__device__ __forceinline__ void put_rows(double* out, size_t stride, int kout, int m, double l0, double l1, double l2,
                                         const int32_t (&ps)[NR], const double (&U0)[NR], const double (&U1)[NR],
                                         const double (&U2)[NR]) {
    const int lane = (int)(threadIdx.x & 63);
    int rows = 0;
#pragma unroll
    for (int r = 0; r < NR; r++) rows += __popcll(__ballot(ps[r] >= 0));
    double* const at = out + (size_t)kout * stride;
    if (m <= rows) {
#pragma nounroll
        for (int j = 0; j < m; j++) {
            const double a = readlane_f64(l0, j), b = readlane_f64(l1, j), c = readlane_f64(l2, j);
#pragma unroll
            for (int r = 0; r < NR; r++)
                if (ps[r] >= 0)
                    at[j * stride + ps[r]] = __builtin_fma(a, U0[r], __builtin_fma(b, U1[r], c * U2[r]));
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        unsigned long long todo = __ballot(ps[r] >= 0);
#pragma nounroll
        while (todo) {
            const int j = __builtin_ctzll(todo);
            todo &= todo - 1;
            const int p = __builtin_amdgcn_readlane(ps[r], j);
            const double a = readlane_f64(U0[r], j), b = readlane_f64(U1[r], j), c = readlane_f64(U2[r], j);
            if (lane < m) at[lane * stride + p] = __builtin_fma(l0, a, __builtin_fma(l1, b, l2 * c));
        }
    }
}

// Per-instance linear stamp values -> Glin, Clin in F positions.
template <int NT>
__device__ void dev_lin_setup(const DPlan* __restrict__ P, const double* __restrict__ p,
                              double* __restrict__ linbuf, double* __restrict__ Glin,
                              double* __restrict__ Clin) {
    const int tid = threadIdx.x;
    for (int s = tid; s < P->n_lin; s += NT) {
        const int kd = P->lin_kind[s];
        const double pv = kd == 0 ? 1.0 : p[P->lin_idx[s]];
        linbuf[s] = (kd == 0 ? 1.0 : kd == 1 ? 1.0 / pv : kd == 2 ? pv : -pv) * P->lin_scale[s];
    }
    __syncthreads();
    for (int e = tid; e < P->nnz; e += NT) {
        double g = 0.0, c = 0.0;
        for (int q = P->g_ptr[e]; q < P->g_ptr[e + 1]; q++) g += sref_val(linbuf, P->g_ref[q]);
        for (int q = P->c_ptr[e]; q < P->c_ptr[e + 1]; q++) c += sref_val(linbuf, P->c_ref[q]);
        Glin[e] = g;
        Clin[e] = c;
    }
    __syncthreads();
}

// Inline: by wave_math.h's source_at, for kernels that run whole transients
template <int NT, bool Inline = false>
__device__ void dev_sources(const DPlan* __restrict__ P, const double* __restrict__ p,
                                            double t, int mode, double* __restrict__ st) {
    for (int s = threadIdx.x; s < P->n_src; s += NT) {
        const int4 d = P->src[s];
        double val;
        if constexpr (Inline) val = source_at(d.x, p + d.y, d.z, p[d.w], t, mode);
        else val = source_value(d.x, p + d.y, d.z, p[d.w], t, mode);
        st[4 * P->n_mos + s] = P->src_m ? val * P->src_m[s] : val;
    }
}

template <int NT>
__device__ void dev_mos(const DPlan* __restrict__ P, const double* __restrict__ p,
                                        const double* __restrict__ u, double* __restrict__ st, double gmin) {
    for (int m = threadIdx.x; m < P->n_mos; m += NT) {
        const int4 dv = reinterpret_cast<const int4*>(P->mos)[m];
        const double vd = dv.x >= 0 ? u[dv.x] : 0.0;
        const double vg = dv.y >= 0 ? u[dv.y] : 0.0;
        const double vs = dv.z >= 0 ? u[dv.z] : 0.0;
        double id, dd, dg, ds;
        sqlaw_eval(dv.w, p[P->p_mos_vth + m], p[P->p_mos_kp + m], p[P->p_mos_w + m],
                   p[P->p_mos_l + m], gmin, vd, vg, vs, id, dd, dg, ds);
        if (P->mos_m) {
            const double mm = P->mos_m[m];
            id *= mm; dd *= mm; dg *= mm; ds *= mm;
        }
        st[4 * m] = id;
        st[4 * m + 1] = dd;
        st[4 * m + 2] = dg;
        st[4 * m + 3] = ds;
    }
}

// Verilog-A devices, one lane per device: the model's currents leaving its
// terminals and their partial derivatives (forward-mode duals seeded on the
// terminal voltages) into the stamp buffer: I[nt], then dI[i]/dV[j].
// $temperature is SimSpec's 27 C (src/simulate_ir.jl:16) in kelvin.
template <int NT>
__device__ void dev_va(const DPlan* __restrict__ P, const double* __restrict__ p,
                       const double* __restrict__ u, double* __restrict__ st, double gmin) {
    using D = VaDual<cedar_va::max_nodes>;
    for (int d = threadIdx.x; d < P->n_va; d += NT) {
        const int4 dv = P->va_dev[d];
        const int nt = dv.z;
        D V[cedar_va::max_nodes], I[cedar_va::max_nodes], Q[cedar_va::max_nodes];
        for (int k = 0; k < cedar_va::max_nodes; k++) {
            const int node = k < nt ? P->va_nodes[dv.y + k] : -1;
            V[k] = k < nt ? D::var(node >= 0 ? u[node] : 0.0, k) : D(0.0);
        }
        cedar_va::eval<D>(dv.x, p + dv.w, kVaTempK, gmin, V, I, Q);
        double* s = st + P->va_st[d];
        for (int i = 0; i < nt; i++) {
            s[i] = I[i].v;
            for (int j = 0; j < nt; j++) s[nt + i * nt + j] = I[i].d[j];
        }
    }
}

// F[e] = Glin + a0*Clin + nonlinear stamps;  x[k] = -(residual of row k).
// qx (natural rows, may be null) is added to the residual.  With pin != null
// the rows that carry charge become u_r = pin_r (consistent initialisation).
// Returns this thread's max |x| over its rows.
// JAC = false writes the residual only and leaves F (factors) untouched.
template <int NT, bool JAC = true>
__device__ double dev_assemble(const DPlan* __restrict__ P, const double* __restrict__ Glin,
                               const double* __restrict__ Clin, double a0,
                               const double* __restrict__ u, const double* __restrict__ qx,
                               const double* __restrict__ st, double* __restrict__ F,
                               double* __restrict__ x, const double* __restrict__ pin) {
    double lmax = 0.0;
    for (int k = threadIdx.x; k < P->n; k += NT) {
        const int r = P->rownat[k];
        const int e0 = P->rowptr[k], e1 = P->rowptr[k + 1];
        double res;
        if (pin && P->is_diff[r]) {
            const int dg = P->diag[k];
            if (JAC)
                for (int e = e0; e < e1; e++) F[e] = (e == dg) ? 1.0 : 0.0;
            res = u[r] - pin[r];
        } else {
            double acc = 0.0;
            for (int e = e0; e < e1; e++) {
                const double jl = Glin[e] + a0 * Clin[e];
                acc += jl * u[P->colnat[e]];
                if (JAC) {
                    double v = jl;
                    for (int q = P->jnl_ptr[e]; q < P->jnl_ptr[e + 1]; q++) v += sref_val(st, P->jnl_ref[q]);
                    F[e] = v;
                }
            }
            if (qx) acc += qx[r];
            for (int q = P->rnl_ptr[k]; q < P->rnl_ptr[k + 1]; q++) acc += sref_val(st, P->rnl_ref[q]);
            res = acc;
        }
        x[k] = -res;
        const double a = fabs(res);
        if (a != a || a > lmax) lmax = a;
    }
    return lmax;
}

// Numeric LU on the fixed pattern, static pivots on the diagonal.
template <int NT>
__device__ void dev_lu(const DPlan* __restrict__ P, double* __restrict__ F, double* __restrict__ inv) {
    for (int l = 0; l < P->lu_nlev; l++) {
        const int b = P->lu_lptr[l], e = P->lu_lptr[l + 1];
        for (int q = b + (int)threadIdx.x; q < e; q += NT) {
            const int4 t = P->lu_task[q];
            double acc = F[t.x];
            for (int up = t.y; up < t.z; up++) {
                const int2 ab = P->lu_upd[up];
                acc -= F[ab.x] * F[ab.y];
            }
            if (t.w >= 0) {
                F[t.x] = acc * inv[t.w];
            } else {
                F[t.x] = acc;
                if (t.w <= -2) inv[-2 - t.w] = 1.0 / acc;
            }
        }
        __syncthreads();
    }
}

// L y = b (unit lower), in place
template <int NT>
__device__ void dev_fwd(const DPlan* __restrict__ P, const double* __restrict__ F, double* __restrict__ x) {
    for (int l = 0; l < P->f_nlev; l++) {
        for (int q = P->f_lptr[l] + (int)threadIdx.x; q < P->f_lptr[l + 1]; q += NT) {
            const int k = P->f_rows[q];
            double s = x[k];
            for (int e = P->rowptr[k]; e < P->diag[k]; e++) s -= F[e] * x[P->colperm[e]];
            x[k] = s;
        }
        __syncthreads();
    }
}

// U x = y, in place
template <int NT>
__device__ void dev_bwd(const DPlan* __restrict__ P, const double* __restrict__ F,
                        const double* __restrict__ inv, double* __restrict__ x) {
    for (int l = 0; l < P->b_nlev; l++) {
        for (int q = P->b_lptr[l] + (int)threadIdx.x; q < P->b_lptr[l + 1]; q += NT) {
            const int k = P->b_rows[q];
            double s = x[k];
            for (int e = P->diag[k] + 1; e < P->rowptr[k + 1]; e++) s -= F[e] * x[P->colperm[e]];
            x[k] = s * inv[k];
        }
        __syncthreads();
    }
}

// U^T z = b, in place (column access to U)
template <int NT>
__device__ void dev_tfwd(const DPlan* __restrict__ P, const double* __restrict__ F,
                         const double* __restrict__ inv, double* __restrict__ x) {
    for (int l = 0; l < P->tf_nlev; l++) {
        for (int q = P->tf_lptr[l] + (int)threadIdx.x; q < P->tf_lptr[l + 1]; q += NT) {
            const int k = P->tf_rows[q];
            double s = x[k];
            for (int c = P->tcol_ptr[k]; c < P->tcol_ptr[k + 1]; c++) {
                const int i = P->tcol_row[c];
                if (i < k) s -= F[P->tcol_pos[c]] * x[i];
            }
            x[k] = s * inv[k];
        }
        __syncthreads();
    }
}

// L^T w = z (unit upper), in place (column access to L)
template <int NT>
__device__ void dev_tbwd(const DPlan* __restrict__ P, const double* __restrict__ F, double* __restrict__ x) {
    for (int l = 0; l < P->tb_nlev; l++) {
        for (int q = P->tb_lptr[l] + (int)threadIdx.x; q < P->tb_lptr[l + 1]; q += NT) {
            const int k = P->tb_rows[q];
            double s = x[k];
            for (int c = P->tcol_ptr[k]; c < P->tcol_ptr[k + 1]; c++) {
                const int i = P->tcol_row[c];
                if (i > k) s -= F[P->tcol_pos[c]] * x[i];
            }
            x[k] = s;
        }
        __syncthreads();
    }
}

// q[natural row] = (Clin * v)[row]
template <int NT>
__device__ void dev_charges(const DPlan* __restrict__ P, const double* __restrict__ Clin,
                            const double* __restrict__ v, double* __restrict__ q) {
    for (int k = threadIdx.x; k < P->n; k += NT) {
        double acc = 0.0;
        for (int e = P->rowptr[k]; e < P->rowptr[k + 1]; e++) acc += Clin[e] * v[P->colnat[e]];
        q[P->rownat[k]] = acc;
    }
}

}  // namespace cedar
