// ac.hip — small-signal AC and noise on the circuit's own pattern and LU
// schedule (the analyses of src/ac.jl: ACSol/freqresp :75-102,215-240,
// NoiseSol/PSD :139-165,267-284).
//
// At the DC operating point the circuit linearises to G + jw C, with G the
// Jacobian dF/du in DC mode and C = dQ/du, both on the filled pattern F the
// transient factors.  One workgroup takes one frequency: it forms
// G + jw C in its own slice of a global workspace (complex, interleaved),
// factors it with the same entry-level LU schedule as the real transient
// (complex arithmetic, the same static pivots), and
//   AC:    solves (G + jw C) x = b, b the sources' AC excitation, and writes
//          x at the observed unknowns;
//   noise: solves (G + jw C)^T y = e_obs and sums, over the noise current
//          sources i (thermal noise of the resistors, 4kT/R each),
//          pwr_i / f^exp_i |y_a - y_b|^2: the output PSD of the reference's
//          PSD(), one transposed solve instead of one solve per source.
#include "device.h"
#include "kernels.h"

namespace cedar {

namespace {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// a - b*c
__device__ __forceinline__ double2 cfms(double2 a, double2 b, double2 c) {
    return make_double2(a.x - (b.x * c.x - b.y * c.y), a.y - (b.x * c.y + b.y * c.x));
}

// 1/d by Smith's method (no overflow of |d|^2 for large or small d)
__device__ __forceinline__ double2 cinv(double2 d) {
    if (fabs(d.x) >= fabs(d.y)) {
        const double r = d.y / d.x, den = d.x + d.y * r;
        return make_double2(1.0 / den, -r / den);
    }
    const double r = d.x / d.y, den = d.x * r + d.y;
    return make_double2(r / den, -1.0 / den);
}

// acc minus the products of entries [b, e), in order: pos(q), col(q) give
// product q's entry of F and of y (pos < 0: none).  Four at a time, so that
// the index reads of a row overlap.
template <class Ld>
__device__ __forceinline__ double2 sub_products(double2 acc, int b, int e, const double2* F, const double2* y,
                                                Ld ld) {
    constexpr int U = 4;
    for (int q = b; q < e; q += U) {
        int pos[U], col[U];
#pragma unroll
        for (int v = 0; v < U; v++) {
            ld(q + v < e ? q + v : e - 1, pos[v], col[v]);
            if (q + v >= e) pos[v] = -1;
        }
#pragma unroll
        for (int v = 0; v < U; v++)
            if (pos[v] >= 0) acc = cfms(acc, F[pos[v]], y[col[v]]);
    }
    return acc;
}

// The update pairs [b, b + U) of a task that ends at e, the last repeated
constexpr int kAcPairs = 8;
__device__ __forceinline__ void load_pairs(int2 (&ab)[kAcPairs], const int2* upd, int b, int e) {
    if (b < e) {
#pragma unroll
        for (int v = 0; v < kAcPairs; v++) ab[v] = upd[b + v < e ? b + v : e - 1];
    }
}

// In LDS (InLds) the factors, reciprocals and solution of one frequency and
// the index arrays of the substitutions stay on the CU: a level is a chain of
// dependent reads of them, 60 cycles each there against several hundred
// through the caches.  The tasks and update pairs of the factorization are too
// many for that: a thread reads its task two levels ahead and the task's first
// pairs one level ahead.  A 12 x 11 mesh's response and noise over 201
// frequencies: 1.37 -> 0.80 ms for the two calls.
template <int NT, bool InLds>
__global__ __launch_bounds__(NT) void k_ac(AcArgs A) {
    extern __shared__ double2 lds_ac[];
    __shared__ double red[NT];
    const DPlan* P = A.P;
    const int n = P->n, nnz = P->nnz, tid = threadIdx.x;
    double2* F = InLds ? lds_ac : reinterpret_cast<double2*>(A.ws + (size_t)blockIdx.x * A.ws_stride);
    double2* inv = F + nnz;
    double2* x = inv + n;
    // the substitutions' schedules: levels over the rows of two passes, each
    // row's entries [ptr, ptr + 1) with their columns (and places in F)
    const bool tr = A.transposed;
    const int nl1 = tr ? P->tf_nlev : P->f_nlev, nl2 = tr ? P->tb_nlev : P->b_nlev;
    const int32_t *lv1 = tr ? P->tf_lptr : P->f_lptr, *lv2 = tr ? P->tb_lptr : P->b_lptr;
    const int32_t *rows1 = tr ? P->tf_rows : P->f_rows, *rows2 = tr ? P->tb_rows : P->b_rows;
    const int32_t *ptr = tr ? P->tcol_ptr : P->rowptr, *col = tr ? P->tcol_row : P->colperm;
    const int32_t *pos = P->tcol_pos, *diag = P->diag;
    if constexpr (InLds) {
        int32_t* at = reinterpret_cast<int32_t*>(x + n);
        auto stage = [&](const int32_t* src, int cnt) {
            int32_t* d = at;
            for (int i = tid; i < cnt; i += NT) d[i] = src[i];
            at += cnt;
            return d;
        };
        const int c1 = lv1[nl1], c2 = lv2[nl2], ce = ptr[n];
        const int32_t* l1 = stage(lv1, nl1 + 1);
        const int32_t* l2 = stage(lv2, nl2 + 1);
        rows1 = stage(rows1, c1);
        rows2 = stage(rows2, c2);
        ptr = stage(ptr, n + 1);
        col = stage(col, ce);
        if (tr) pos = stage(pos, ce);
        else diag = stage(diag, n);
        lv1 = l1;
        lv2 = l2;
    }
    const int nlev = P->lu_nlev;
    const int32_t* lp = P->lu_lptr;
    const int4* task = P->lu_task;
    const int2* upd = P->lu_upd;
    // the thread's first task of level l, empty past the level's end
    auto first_task = [&](int l) {
        int4 t = make_int4(0, 0, 0, -1);
        if (l < nlev) {
            const int q = lp[l] + tid;
            if (q < lp[l + 1]) t = task[q];
        }
        return t;
    };
    for (int f = blockIdx.x; f < A.n_freq; f += gridDim.x) {
        const double w = A.omega[f];
        for (int e = tid; e < nnz; e += NT) F[e] = make_double2(A.G[e], w * A.Cl[e]);
        for (int k = tid; k < n; k += NT)
            x[k] = tr ? make_double2(k == A.obs_col ? 1.0 : 0.0, 0.0) : make_double2(A.rhs[k], 0.0);
        int4 t0 = first_task(0), t1 = first_task(1);
        int2 ab0[kAcPairs], ab1[kAcPairs];
        load_pairs(ab0, upd, t0.y, t0.z);
        __syncthreads();
        // LU on the fixed pattern (the schedule of dev_lu)
        for (int l = 0; l < nlev; l++) {
            load_pairs(ab1, upd, t1.y, t1.z);
            const int4 t2 = first_task(l + 2);
            const int qe = lp[l + 1];
            for (int q = lp[l] + tid; q < qe; q += NT) {
                double2 acc = F[t0.x];
                for (int up = t0.y; up < t0.z; up += kAcPairs) {
#pragma unroll
                    for (int v = 0; v < kAcPairs; v++)
                        if (up + v < t0.z) acc = cfms(acc, F[ab0[v].x], F[ab0[v].y]);
                    load_pairs(ab0, upd, up + kAcPairs, t0.z);
                }
                if (t0.w >= 0) {
                    F[t0.x] = cmul(acc, inv[t0.w]);
                } else {
                    F[t0.x] = acc;
                    if (t0.w <= -2) inv[-2 - t0.w] = cinv(acc);
                }
                if (q + NT < qe) {
                    t0 = task[q + NT];
                    load_pairs(ab0, upd, t0.y, t0.z);
                }
            }
            t0 = t1;
            t1 = t2;
#pragma unroll
            for (int v = 0; v < kAcPairs; v++) ab0[v] = ab1[v];
            __syncthreads();
        }
        if (!tr) {
            // L y = b (unit lower), then U x = y
            auto entry = [&](int e, int& ps, int& cl) {
                ps = e;
                cl = col[e];
            };
            for (int l = 0; l < nl1; l++) {
                for (int q = lv1[l] + tid; q < lv1[l + 1]; q += NT) {
                    const int k = rows1[q];
                    x[k] = sub_products(x[k], ptr[k], diag[k], F, x, entry);
                }
                __syncthreads();
            }
            for (int l = 0; l < nl2; l++) {
                for (int q = lv2[l] + tid; q < lv2[l + 1]; q += NT) {
                    const int k = rows2[q];
                    x[k] = cmul(sub_products(x[k], diag[k] + 1, ptr[k + 1], F, x, entry), inv[k]);
                }
                __syncthreads();
            }
            for (int i = tid; i < A.n_obs; i += NT) {
                const double2 v = x[A.obs_piv[i]];
                A.out[2 * ((size_t)f * A.n_obs + i)] = v.x;
                A.out[2 * ((size_t)f * A.n_obs + i) + 1] = v.y;
            }
        } else {
            // U^T z = e, then L^T y = z (column access to F)
            for (int l = 0; l < nl1; l++) {
                for (int q = lv1[l] + tid; q < lv1[l + 1]; q += NT) {
                    const int k = rows1[q];
                    const double2 s = sub_products(x[k], ptr[k], ptr[k + 1], F, x, [&](int c, int& ps, int& cl) {
                        const int p = pos[c];
                        cl = col[c];
                        ps = cl < k ? p : -1;
                    });
                    x[k] = cmul(s, inv[k]);
                }
                __syncthreads();
            }
            for (int l = 0; l < nl2; l++) {
                for (int q = lv2[l] + tid; q < lv2[l + 1]; q += NT) {
                    const int k = rows2[q];
                    x[k] = sub_products(x[k], ptr[k], ptr[k + 1], F, x, [&](int c, int& ps, int& cl) {
                        const int p = pos[c];
                        cl = col[c];
                        ps = cl > k ? p : -1;
                    });
                }
                __syncthreads();
            }
            // PSD = sum_i pwr_i / fHz^exp_i |y_a - y_b|^2, y by pivot row
            const double fhz = w / (2.0 * M_PI);
            double acc = 0.0;
            for (int i = tid; i < A.n_noise; i += NT) {
                const int a = A.nz_rows[2 * i], b = A.nz_rows[2 * i + 1];
                const double2 ya = a >= 0 ? x[a] : make_double2(0.0, 0.0);
                const double2 yb = b >= 0 ? x[b] : make_double2(0.0, 0.0);
                const double dr = ya.x - yb.x, di = ya.y - yb.y;
                const double ex = A.nz_exp[i];
                const double s = ex == 0.0 ? A.nz_pwr[i] : A.nz_pwr[i] / pow(fhz, ex);
                acc += s * (dr * dr + di * di);
            }
            const double tot = block_reduce<NT>(acc, red, OpSum());
            if (tid == 0) A.psd[f] = tot;
        }
        __syncthreads();
    }
}

}  // namespace

// levels and rows of a pass are at most n
size_t ac_lds(int32_t n, int32_t nnz) {
    return sizeof(double2) * ((size_t)nnz + 2 * (size_t)n) + sizeof(int32_t) * (2 * (size_t)nnz + 6 * (size_t)n + 4);
}

hipError_t launch_ac(const AcArgs& a, int nblocks, int nt, size_t lds, hipStream_t s) {
    if (nt == 64 && lds) hipLaunchKernelGGL((k_ac<64, true>), dim3(nblocks), dim3(64), lds, s, a);
    else if (nt == 64 && !lds) hipLaunchKernelGGL((k_ac<64, false>), dim3(nblocks), dim3(64), 0, s, a);
    else if (nt == 256 && !lds) hipLaunchKernelGGL((k_ac<256, false>), dim3(nblocks), dim3(256), 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace cedar
