// big.hip — large-circuit path: device-wide evaluation and assembly, the
// supernodal multifrontal LU of bigplan.h, and the transient / DC-op drivers
// with the step history kept on the device.
//
// One Newton iteration (captured once in a hipGraph and replayed):
//   eval      one lane per MOSFET / source (grid-stride)
//   assemble  one lane per natural row: Jacobian values on the natural
//             pattern (fixed-order contributor gathers) and -residual in
//             pivot order; per-block max |residual|
//   factor    for each assembly-tree level, leaves first:
//               gather  front entries = sum of the children's contribution
//                       blocks (inverse relative maps; every entry written
//                       once, children in a fixed order: no atomics)
//               orig    + the level's Jacobian entries (distinct positions)
//               small   fronts with m <= kSmallM: one workgroup each, the
//                       gather straight into LDS, right-looking partial LU
//               large   gather and entries, then blocked right-looking
//                       partial LU, panel width kNb: diagonal block (one
//                       workgroup), row / column triangular solves, trailing
//                       update by 64 x 64 MFMA tiles over many workgroups
//                       (or one workgroup per front, where the autotuner
//                       measured that faster for the level)
//   solve     forward by levels (children's update vectors gathered in a
//             fixed order), backward from the root
//   update    u += dx, WRMS / max norms (fixed-order block reductions)
// Everything is bit-reproducible run to run.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "big.h"
#include "dcop_rules.h"
#include "kernels.h"
#include "rules.h"

namespace cedar {

namespace {

constexpr int kBT = 256;      // threads of the device-wide kernels
constexpr int kSmallM = 96;   // fronts up to this size factor in LDS
constexpr int kNb = 32;       // panel width of the blocked front LU
constexpr int kTile = 64;     // trailing-update tile
constexpr int kGatherChunk = 8192;   // entries a gather tile can hold in LDS
// entries a gather tile should have: a tile is a chain of dependent loads
// per child and per 4 entries of a thread, so smaller tiles end earlier
constexpr int kGatherTile = 2048;
constexpr int kRowBlocks = 1024;

struct BigDev {
    int32_t n, nnz, n_mos, n_src, n_lin, n_stamp, n_params;
    int32_t p_mos_vth, p_mos_kp, p_mos_w, p_mos_l, p_gmin;
    const int32_t *rowptr, *col, *lin_kind, *lin_idx, *g_ptr, *g_ref, *c_ptr, *c_ref;
    const int32_t *jnl_ptr, *jnl_ref, *rnl_ptr, *rnl_ref, *is_diff, *prow, *pcol;
    const int4 *mos, *src;
    const double* lin_scale;               // m-factor per linear slot
    const double *mos_m, *src_m;           // m-factors, null when every m is 1
    const int32_t *sn_first, *sn_m, *sn_rptr, *sn_rows, *ch_ptr, *ch_sn, *rel_ptr, *rel, *inv, *olev_pos;
    const int32_t *osn_ptr, *osn_pos;
    // per entry of ch_sn: (rows of the child's contribution block, its leading
    // dimension, its rel_ptr, unused), and the block's offset in the pool
    const int4* ch_rec;
    const int64_t* ch_blk;
    const int32_t *row_long, *long_rows;   // rows too long for one lane (supply node, ...)
    const int32_t* long_cptr;              // [n_long+1] chunk range of each long row
    const int4* long_chunks;               // (row, kind, begin, end)
    int32_t n_long, n_chunks;
    const int64_t *sn_off, *inv_ptr, *nat_dest;
};

__device__ __forceinline__ double sref_v(const double* buf, int32_t r) {
    const double v = buf[r >> 1];
    return (r & 1) ? -v : v;
}

template <class Op>
__device__ __forceinline__ double blk_reduce(double v, double* red, Op op) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = kBT / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = op(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}
struct Sum {
    __device__ double operator()(double a, double b) const { return a + b; }
};
struct Max {   // NaN-propagating
    __device__ double operator()(double a, double b) const { return (a != a || a > b) ? a : b; }
};

// ---- evaluation and assembly ----------------------------------------------------------
__global__ __launch_bounds__(kBT) void k_lin_a(const BigDev* P, const double* p, double* linbuf) {
    for (int s = blockIdx.x * kBT + threadIdx.x; s < P->n_lin; s += gridDim.x * kBT) {
        const int kd = P->lin_kind[s];
        const double pv = kd == 0 ? 1.0 : p[P->lin_idx[s]];
        linbuf[s] = (kd == 0 ? 1.0 : kd == 1 ? 1.0 / pv : kd == 2 ? pv : -pv) * P->lin_scale[s];
    }
}

__global__ __launch_bounds__(kBT) void k_lin_b(const BigDev* P, const double* linbuf, double* Glin,
                                               double* Clin) {
    for (int e = blockIdx.x * kBT + threadIdx.x; e < P->nnz; e += gridDim.x * kBT) {
        double g = 0.0, c = 0.0;
        for (int q = P->g_ptr[e]; q < P->g_ptr[e + 1]; q++) g += sref_v(linbuf, P->g_ref[q]);
        for (int q = P->c_ptr[e]; q < P->c_ptr[e + 1]; q++) c += sref_v(linbuf, P->c_ref[q]);
        Glin[e] = g;
        Clin[e] = c;
    }
}

__global__ __launch_bounds__(kBT) void k_eval(const BigDev* P, const double* p, const double* u,
                                              const StepDev* spp, double* st) {
    const StepDev sp = *spp;
    const double gmin = p[P->p_gmin];
    const int total = P->n_mos + P->n_src;
    for (int q = blockIdx.x * kBT + threadIdx.x; q < total; q += gridDim.x * kBT) {
        if (q < P->n_mos) {
            const int4 dv = P->mos[q];
            const double vd = dv.x >= 0 ? u[dv.x] : 0.0;
            const double vg = dv.y >= 0 ? u[dv.y] : 0.0;
            const double vs = dv.z >= 0 ? u[dv.z] : 0.0;
            double id, dd, dg, ds;
            sqlaw_eval(dv.w, p[P->p_mos_vth + q], p[P->p_mos_kp + q], p[P->p_mos_w + q],
                       p[P->p_mos_l + q], gmin, vd, vg, vs, id, dd, dg, ds);
            if (P->mos_m) {
                const double mm = P->mos_m[q];
                id *= mm; dd *= mm; dg *= mm; ds *= mm;
            }
            st[4 * q] = id;
            st[4 * q + 1] = dd;
            st[4 * q + 2] = dg;
            st[4 * q + 3] = ds;
        } else {
            const int s = q - P->n_mos;
            const int4 d = P->src[s];
            const double val = source_value(d.x, p + d.y, d.z, p[d.w], sp.t, sp.mode);
            st[4 * P->n_mos + s] = P->src_m ? val * P->src_m[s] : val;
        }
    }
}

// Jacobian values on the natural pattern and x[prow[r]] = -residual(r)
// (x may be null).  a0 and the charge term qx apply in transient steps;
// pinned rows (UIC) become u_r = pin_r.
__global__ __launch_bounds__(kBT) void k_assemble(const BigDev* P, const double* Glin, const double* Clin,
                                                  const StepDev* spp, const double* u, const double* qx,
                                                  const double* st, const double* pin, double* Aval,
                                                  double* x, double* part) {
    __shared__ double red[kBT];
    const StepDev sp = *spp;
    const double a0 = sp.kind == STEP_TRAN ? sp.a0 : 0.0;
    const bool use_q = sp.kind == STEP_TRAN && qx;
    const bool use_pin = sp.kind == STEP_UIC && pin;
    double lmax = 0.0;
    for (int r = blockIdx.x * kBT + threadIdx.x; r < P->n; r += gridDim.x * kBT) {
        if (P->row_long[r]) continue;
        const int e0 = P->rowptr[r], e1 = P->rowptr[r + 1];
        double res;
        if (use_pin && P->is_diff[r]) {
            for (int e = e0; e < e1; e++) Aval[e] = P->col[e] == r ? 1.0 : 0.0;
            res = u[r] - pin[r];
        } else {
            double acc = 0.0;
            for (int e = e0; e < e1; e++) {
                const double jl = Glin[e] + a0 * Clin[e];
                acc += jl * u[P->col[e]];
                double v = jl;
                for (int q = P->jnl_ptr[e]; q < P->jnl_ptr[e + 1]; q++) v += sref_v(st, P->jnl_ref[q]);
                Aval[e] = v;
            }
            if (use_q) acc += qx[r];
            for (int q = P->rnl_ptr[r]; q < P->rnl_ptr[r + 1]; q++) acc += sref_v(st, P->rnl_ref[q]);
            res = acc;
        }
        if (x) x[P->prow[r]] = -res;
        const double a = fabs(res);
        if (a != a || a > lmax) lmax = a;
    }
    const double m = blk_reduce(lmax, red, Max());
    if (threadIdx.x == 0 && part) part[blockIdx.x] = m;
}

// A row with thousands of entries (a supply node touching every PMOS) is cut
// into chunks of up to 256 entries, 256 residual references or 256
// Jacobian references of one heavy entry (the supply node's diagonal takes
// one from every device on it), one workgroup per chunk; chunk = (row,
// kind, begin, end) with kind 0 entries, 1 residual refs, 2 + e the refs of
// heavy entry e.  k_long_finish adds the chunk partials of each row and of
// each heavy entry in a fixed order.
constexpr int kHeavyRefs = 64;   // an entry with more Jacobian refs is heavy
__global__ __launch_bounds__(kBT) void k_assemble_chunks(const BigDev* P, const double* Glin, const double* Clin,
                                                         const StepDev* spp, const double* u, const double* st,
                                                         const double* pin, double* Aval, double* lpart) {
    __shared__ double red[kBT];
    const StepDev sp = *spp;
    const double a0 = sp.kind == STEP_TRAN ? sp.a0 : 0.0;
    const bool pinned_row = sp.kind == STEP_UIC && pin;
    const int4 ch = P->long_chunks[blockIdx.x];
    const int r = ch.x;
    double acc = 0.0;
    const int q = ch.z + threadIdx.x;
    if (ch.y == 0) {
        if (q < ch.w) {
            if (pinned_row && P->is_diff[r]) {
                Aval[q] = P->col[q] == r ? 1.0 : 0.0;
            } else {
                const double jl = Glin[q] + a0 * Clin[q];
                acc = jl * u[P->col[q]];
                double v = jl;
                const int t0 = P->jnl_ptr[q], t1 = P->jnl_ptr[q + 1];
                if (t1 - t0 <= kHeavyRefs)
                    for (int t = t0; t < t1; t++) v += sref_v(st, P->jnl_ref[t]);
                Aval[q] = v;
            }
        }
    } else if (q < ch.w) {
        acc = sref_v(st, ch.y == 1 ? P->rnl_ref[q] : P->jnl_ref[q]);
    }
    const double t = blk_reduce(acc, red, Sum());
    if (threadIdx.x == 0) lpart[blockIdx.x] = t;
}

// One workgroup per long row: the chunk partials are staged in LDS and one
// thread adds them in chunk order (the row's entry sums, its residual
// references, then each heavy entry's references onto its Jacobian value).
__global__ __launch_bounds__(kBT) void k_long_finish(const BigDev* P, const StepDev* spp, const double* u,
                                                     const double* qx, const double* pin, const double* lpart,
                                                     double* Aval, double* x, double* part) {
    __shared__ double pl[kBT];
    __shared__ int kl[kBT];
    const StepDev sp = *spp;
    const bool use_q = sp.kind == STEP_TRAN && qx;
    const bool use_pin = sp.kind == STEP_UIC && pin;
    const int l = blockIdx.x;
    const int r = P->long_rows[l];
    const bool pinned = use_pin && P->is_diff[r];
    const int cb = P->long_cptr[l], ce = P->long_cptr[l + 1];
    double sa = 0.0, sn = 0.0, hv = 0.0;
    int he = -1;   // heavy entry being summed (value in hv)
    for (int c0 = cb; c0 < ce; c0 += kBT) {
        const int c = c0 + threadIdx.x;
        if (c < ce) {
            kl[threadIdx.x] = P->long_chunks[c].y;
            pl[threadIdx.x] = lpart[c];
        }
        __syncthreads();
        if (threadIdx.x == 0 && !pinned) {
            const int nc = (ce - c0) < kBT ? ce - c0 : kBT;
            for (int q = 0; q < nc; q++) {
                const int kind = kl[q];
                if (kind == 0) sa += pl[q];
                else if (kind == 1) sn += pl[q];
                else {
                    if (kind - 2 != he) {
                        if (he >= 0) Aval[he] = hv;
                        he = kind - 2;
                        hv = Aval[he];
                    }
                    hv += pl[q];
                }
            }
        }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    if (he >= 0) Aval[he] = hv;
    const double res = pinned ? u[r] - pin[r] : (use_q ? sa + qx[r] : sa) + sn;
    if (x) x[P->prow[r]] = -res;
    if (part) part[l] = fabs(res);
}

__global__ __launch_bounds__(kBT) void k_res_reduce(const double* part, int nb, double* norm) {
    __shared__ double red[kBT];
    double m = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBT) {
        const double v = part[b];
        if (v != v || v > m) m = v;
    }
    m = blk_reduce(m, red, Max());
    if (threadIdx.x == 0) norm[NRM_RES] = m;
}

// u += dx (DC / UIC: skipped once the residual met the tolerance); block
// partial sums of the WRMS terms and maxima of |dx|.
__global__ __launch_bounds__(kBT) void k_update(const BigDev* P, const StepDev* spp, const double* x,
                                                double* u, double* norm, double* part) {
    __shared__ double red[kBT];
    const StepDev sp = *spp;
    if (sp.kind != STEP_TRAN && norm[NRM_RES] <= sp.tol) return;
    double ss = 0.0, mx = 0.0;
    for (int i = blockIdx.x * kBT + threadIdx.x; i < P->n; i += gridDim.x * kBT) {
        const double d = x[P->pcol[i]];
        const double ui = u[i] + d;
        u[i] = ui;
        const double r = d / (sp.rtol * fabs(ui) + sp.atol);
        ss += r * r;
        const double a = fabs(d);
        if (a != a || a > mx) mx = a;
    }
    const double s = blk_reduce(ss, red, Sum());
    const double m = blk_reduce(mx, red, Max());
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = s;
        part[2 * blockIdx.x + 1] = m;
    }
}

__global__ __launch_bounds__(kBT) void k_upd_reduce(const BigDev* P, const StepDev* spp, const double* part,
                                                    int nb, double* norm) {
    __shared__ double red[kBT];
    const StepDev sp = *spp;
    if (sp.kind != STEP_TRAN && norm[NRM_RES] <= sp.tol) {
        if (threadIdx.x == 0) norm[NRM_DONE] = 1.0;
        return;
    }
    double s = 0.0, m = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBT) {
        s += part[2 * b];
        const double v = part[2 * b + 1];
        if (v != v || v > m) m = v;
    }
    s = blk_reduce(s, red, Sum());
    m = blk_reduce(m, red, Max());
    if (threadIdx.x == 0) {
        norm[NRM_WRMS] = sqrt(s / P->n);
        norm[NRM_MAXD] = m;
        norm[NRM_DONE] = 0.0;
    }
}

// ---- multifrontal factorization ----------------------------------------------------------
// Front s: m x m column-major at pool + sn_off[s]; k = pivots; CB = trailing r x r.
__device__ __forceinline__ int sn_k(const BigDev* P, int s) { return P->sn_first[s + 1] - P->sn_first[s]; }

// Global-memory phases of one workgroup: stores complete and the CU's L1 is
// invalidated before any wavefront reads what another one wrote.
__device__ __forceinline__ void gsync() {
    __threadfence();
    __syncthreads();
}

// Barrier of the NT threads that work on one front in LDS: the workgroup,
// or a wavefront of a workgroup whose wavefronts work on fronts of their own
// (a wavefront's LDS operations complete in order: only the compiler must
// keep them so).
template <int NT>
__device__ __forceinline__ void front_sync() {
    if (NT > 64) {
        __syncthreads();
        return;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Columns [j0, j1) of front s = the sum of its children's contribution
// blocks, children in order, into F (column j0 at F[0], leading dimension
// ld): the columns are zeroed, then each child's block is added (one
// wavefront per block column, lanes down the rows), with a barrier between
// children.  Update row a of child c sits at row rel[a] of the parent.  br,
// when given, holds per child the range of its block columns that land in
// [j0, j1) (rel is ascending); without it every column does.  Every entry
// sees its children's values in the same order as a sum over the children.
// NT threads, this one number tid; Global: F in global memory (fenced
// barriers), else in LDS.
template <int NT, bool Global>
__device__ __forceinline__ void scatter_cb(const BigDev* P, const double* pool, double* F, int ld, int s, int j0,
                                           int j1, const int2* br, int tid) {
    for (int q = tid; q < (j1 - j0) * ld; q += NT) F[q] = 0.0;
    if (Global) gsync();
    else front_sync<NT>();
    const int c0 = P->ch_ptr[s], c1 = P->ch_ptr[s + 1];
    // the next child's record is read while this one is added
    int4 next = c0 < c1 ? P->ch_rec[c0] : make_int4(0, 0, 0, 0);
    int64_t next_blk = c0 < c1 ? P->ch_blk[c0] : 0;
    for (int cq = c0; cq < c1; cq++) {
        const int rc = next.x, mc = next.y;
        const int* rl = P->rel + next.z;
        const double* blk = pool + next_blk;
        if (cq + 1 < c1) {
            next = P->ch_rec[cq + 1];
            next_blk = P->ch_blk[cq + 1];
        }
        int b0 = 0, b1 = rc;
        if (br) {
            const int2 r = br[cq - c0];
            b0 = r.x;
            b1 = r.y;
        }
        // entry (a, b) of the child's block, flattened; the loads of four
        // entries are issued before their adds.  A child's entries land on
        // distinct entries of F, so the order within a child is free.
        constexpr int U = 4;
        const int tot = (b1 - b0) * rc;
        for (int q0 = tid; q0 < tot; q0 += NT * U) {
            int dst[U];
            double sv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int q = q0 + u * NT;
                if (q < tot) {
                    const int b = b0 + q / rc, a = q % rc;
                    dst[u] = (rl[b] - j0) * ld + rl[a];
                    sv[u] = blk[(int64_t)b * mc + a];
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (q0 + u * NT < tot) F[dst[u]] += sv[u];
        }
        if (Global) gsync();
        else front_sync<NT>();
    }
}

// tile = (front, first column, end column, offset of its per-child column
// ranges in cbr): the tile (at most kGatherChunk entries) is summed in LDS
// and written once.  With op, the Jacobian entries of the tile's columns
// (positions op[0, n_op)) are added before that; they land on distinct
// entries, so their order is free.
__device__ __forceinline__ void gather_tile(const BigDev* P, double* pool, const int4 t, const int2* cbr, double* Ft,
                                            const double* Aval, const int32_t* op, int n_op) {
    const int s = t.x, m = P->sn_m[s];
    const int64_t off = P->sn_off[s] + (int64_t)t.y * m;
    double* G = pool + off;
    const bool fits = (t.z - t.y) * m <= kGatherChunk;
    if (fits) {
        scatter_cb<kBT, false>(P, pool, Ft, m, s, t.y, t.z, cbr + t.w, threadIdx.x);
        for (int q = threadIdx.x; q < n_op; q += kBT) Ft[P->nat_dest[op[q]] - off] += Aval[op[q]];
        if (n_op) __syncthreads();
        for (int q = threadIdx.x; q < (t.z - t.y) * m; q += kBT) G[q] = Ft[q];
    } else {   // a single column longer than the LDS tile
        scatter_cb<kBT, true>(P, pool, G, m, s, t.y, t.z, cbr + t.w, threadIdx.x);
        for (int q = threadIdx.x; q < n_op; q += kBT) G[P->nat_dest[op[q]] - off] += Aval[op[q]];
    }
}

__global__ __launch_bounds__(kBT) void k_mf_gather(const BigDev* P, double* pool, const int4* tiles,
                                                   const int2* cbr) {
    extern __shared__ double lds_f[];
    gather_tile(P, pool, tiles[blockIdx.x], cbr, lds_f, nullptr, nullptr, 0);
}

__global__ __launch_bounds__(kBT) void k_mf_orig(const BigDev* P, const double* Aval, double* pool,
                                                 const int32_t* pos_list, int b, int e) {
    for (int q = b + blockIdx.x * kBT + threadIdx.x; q < e; q += gridDim.x * kBT) {
        const int pos = pos_list[q];
        pool[P->nat_dest[pos]] += Aval[pos];
    }
}

// LU without pivoting of the nb x nb block D (column-major, leading
// dimension kNb, in LDS) by NT threads (NT a multiple of 32, at most
// 1024), each holding 1024 / NT entries in registers: with G = NT / 32 row
// groups, thread t owns column t / G, rows t % G + G v.  Before step p the
// owners of column p and of row p publish them in cb / rb (double-buffered,
// one barrier per pivot; with one wavefront the barrier is only a wavefront
// one).  The operations and their order are those of the column sweep:
// l(i,p) = a(i,p) * (1 / u(p,p)), then a(i,j) -= l(i,p) u(p,j) for pivots p
// ascending.  L (unit diagonal, below) and U overwrite D; ipv[p] = 1 / u(p,p).
template <int NT>
__device__ __forceinline__ void diag_lu_block(double* D, double* ipv, int nb, double (*cb)[kNb],
                                              double (*rb)[kNb]) {
    constexpr int G = NT / kNb, EP = kNb / G;
    const int t = threadIdx.x, j = t / G, i0 = t % G;
    double a[EP];
#pragma unroll
    for (int v = 0; v < EP; v++) {
        const int i = i0 + G * v;
        a[v] = (i < nb && j < nb) ? D[j * kNb + i] : 0.0;
        if (j == 0) cb[0][i] = a[v];
        if (i == 0) rb[0][j] = a[v];
    }
    __syncthreads();
    for (int p = 0; p < nb; p++) {
        const int b = p & 1;
        // every LDS read of the step is issued before the first use, and the
        // update is computed for all entries and selected, so no entry waits
        // in a branch of its own
        const double piv = rb[b][p];
        const double u = rb[b][j];
        double c[EP];
#pragma unroll
        for (int v = 0; v < EP; v++) c[v] = cb[b][i0 + G * v];
        const double ip = 1.0 / piv;
        if (t == 0) ipv[p] = ip;
#pragma unroll
        for (int v = 0; v < EP; v++) {
            const int i = i0 + G * v;
            const double l = c[v] * ip;
            const double upd = a[v] - l * u;
            a[v] = i > p ? (j == p ? l : (j > p ? upd : a[v])) : a[v];
            if (j == p + 1) cb[b ^ 1][i] = a[v];
            if (i == p + 1) rb[b ^ 1][j] = a[v];
        }
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < EP; v++) {
        const int i = i0 + G * v;
        if (i < nb && j < nb) D[j * kNb + i] = a[v];
    }
}

// item = (front, p0): LU of the diagonal block [p0, p0+nb) x [p0, p0+nb),
// four wavefronts (four entries per thread; one wavefront was 3x slower: it
// issues each step's updates serially)
constexpr int kDiagThreads = kBT;
__global__ __launch_bounds__(kDiagThreads) void k_mf_diag(const BigDev* P, double* pool, double* dinv,
                                                          const int2* items) {
    __shared__ double D[kNb * kNb];
    __shared__ double cb[2][kNb], rb[2][kNb];
    const int2 it = items[blockIdx.x];
    const int s = it.x, p0 = it.y;
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int nb = (k - p0) < kNb ? (k - p0) : kNb;
    double* G = pool + P->sn_off[s];
    for (int q = threadIdx.x; q < nb * nb; q += kDiagThreads) {
        const int j = q / nb, i = q % nb;
        D[j * kNb + i] = G[(int64_t)(p0 + j) * m + p0 + i];
    }
    __syncthreads();
    diag_lu_block<kDiagThreads>(D, dinv + f0 + p0, nb, cb, rb);
    __syncthreads();
    for (int q = threadIdx.x; q < nb * nb; q += kDiagThreads) {
        const int j = q / nb, i = q % nb;
        G[(int64_t)(p0 + j) * m + p0 + i] = D[j * kNb + i];
    }
}

// Triangular solve of one right-hand side held in registers, right-looking:
// a[i] is the pending value of column c + i while column c is eliminated,
// so every register index is fixed (a runtime-indexed array would live in
// scratch).  The coefficient coupling column c to column c + 1 + i is
// E[c * (kNb + 1) + 1 + i]; the kNb - 1 coefficients of a step are all
// requested before the first is used.  Column c + 1 + i receives its
// updates in ascending c, the order of the left-looking dot product.  Each
// result, scaled by sc[c] when Scale, goes to put(c, x).  Columns past nb
// carry values that are never stored.
template <bool Scale, class Put>
__device__ __forceinline__ void rot_solve(double (&a)[kNb], const double* E, const double* sc, int nb, Put put) {
    for (int c = 0; c < nb; c++) {
        const double* e = E + c * (kNb + 1) + 1;
        double ev[kNb - 1];
#pragma unroll
        for (int i = 0; i < kNb - 1; i++) ev[i] = e[i];
        const double s = Scale ? sc[c] : 1.0;
        __builtin_amdgcn_sched_barrier(0);
        const double xc = Scale ? a[0] * s : a[0];
        put(c, xc);
#pragma unroll
        for (int i = 0; i < kNb - 1; i++) a[i] = a[i + 1] - xc * ev[i];
        a[kNb - 1] = 0.0;
    }
}
// Coefficient block of rot_solve: E[c kNb + j] (kNb + 1 rows of kNb, zero
// outside the nb x nb block, so reads past a row stay in bounds), from the
// factored diagonal block B (column-major, leading dimension ld):
//   rows of L21 (x U11 = a):    E[c kNb + j] = U(c, j) = B[j ld + c]
//   columns of U12 (L11 y = a): E[c kNb + j] = L(j, c) = B[c ld + j]
constexpr int kCoef = kNb * (kNb + 1);
template <bool Upper>
__device__ __forceinline__ void load_coef(double* E, const double* B, int64_t ld, int nb) {
    for (int q = threadIdx.x; q < kNb * kNb; q += kBT) {
        // the index that runs fastest in B runs fastest over the threads
        const int f = q % kNb, g = q / kNb;
        const int c = Upper ? f : g, j = Upper ? g : f;
        E[c * kNb + j] = (c < nb && j < nb) ? B[(int64_t)g * ld + f] : 0.0;
    }
    if ((int)threadIdx.x < kNb) E[kNb * kNb + threadIdx.x] = 0.0;
}

// item = (front, p0, kind, first): kind 0 solves rows [first, first+256) of
// L21 (x U11 = a), kind 1 columns [first, first+128) of U12 (L11 y = a, unit
// diagonal); the columns go through LDS so both loads and stores are
// contiguous runs of a column
constexpr int kTrsmCols = 128;
__global__ __launch_bounds__(kBT) void k_mf_trsm(const BigDev* P, double* pool, const double* dinv,
                                                 const int4* items) {
    __shared__ double E[kCoef];
    __shared__ double sc[kNb];
    __shared__ double T[kNb][kTrsmCols + 1];
    const int4 it = items[blockIdx.x];
    const int s = it.x, p0 = it.y;
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int nb = (k - p0) < kNb ? (k - p0) : kNb;
    double* G = pool + P->sn_off[s];
    const double* B = G + (int64_t)p0 * m + p0;
    if (it.z == 0) {
        load_coef<true>(E, B, m, nb);
        if ((int)threadIdx.x < nb) sc[threadIdx.x] = dinv[f0 + p0 + threadIdx.x];
        __syncthreads();
        const int r = it.w + threadIdx.x;
        if (r >= m) return;
        double a[kNb];
#pragma unroll
        for (int c = 0; c < kNb; c++) a[c] = c < nb ? G[(int64_t)(p0 + c) * m + r] : 0.0;
        rot_solve<true>(a, E, sc, nb, [&](int c, double x) { G[(int64_t)(p0 + c) * m + r] = x; });
        return;
    }
    load_coef<false>(E, B, m, nb);
    const int j0 = it.w;
    const int ncol = (m - j0) < kTrsmCols ? (m - j0) : kTrsmCols;
    for (int q = threadIdx.x; q < nb * ncol; q += kBT) {
        const int jj = q / nb, c = q % nb;
        T[c][jj] = G[(int64_t)(j0 + jj) * m + p0 + c];
    }
    __syncthreads();
    if ((int)threadIdx.x < ncol) {
        const int jj = threadIdx.x;
        double a[kNb];
#pragma unroll
        for (int c = 0; c < kNb; c++) a[c] = c < nb ? T[c][jj] : 0.0;
        rot_solve<false>(a, E, nullptr, nb, [&](int c, double x) { T[c][jj] = x; });
    }
    __syncthreads();
    for (int q = threadIdx.x; q < nb * ncol; q += kBT) {
        const int jj = q / nb, c = q % nb;
        G[(int64_t)(j0 + jj) * m + p0 + c] = T[c][jj];
    }
}

// F[i0:i0+64, j0:j0+64] -= L U for the L panel rows A[c][i] (transposed) and
// the U panel columns Bt[c][j] staged in LDS, on the vector ALUs
template <int LD>
__device__ __forceinline__ void tile_update_valu(const double (*A)[LD], const double (*Bt)[LD],
                                                 double* G, int m, int i0, int j0, int nb) {
    const int ti = (threadIdx.x % 16) * 4, tj = (threadIdx.x / 16) * 4;
    double acc[4][4] = {};
    for (int c = 0; c < nb; c++) {
        double a[4], b[4];
        for (int q = 0; q < 4; q++) { a[q] = A[c][ti + q]; b[q] = Bt[c][tj + q]; }
        for (int y = 0; y < 4; y++)
            for (int x = 0; x < 4; x++) acc[y][x] += a[x] * b[y];
    }
    for (int y = 0; y < 4; y++) {
        const int j = j0 + tj + y;
        if (j >= m) continue;
        for (int x = 0; x < 4; x++) {
            const int i = i0 + ti + x;
            if (i < m) G[(int64_t)j * m + i] -= acc[y][x];
        }
    }
}

// The panel rows i0.. of L and columns j0.. of U into LDS (zero past m and
// nb).  All loads are issued before the first LDS store, so the 16 global
// round trips overlap; consecutive threads read consecutive addresses (L:
// down a column of the panel, U: along a panel row's column segment).
__device__ __forceinline__ void load_panel_tiles(double (*A)[kTile + 1], double (*Bt)[kTile + 1], const double* G,
                                                 int m, int p0, int i0, int j0, int nb) {
    constexpr int R = kNb * kTile / kBT;
    static_assert(R * kBT == kNb * kTile, "panel tiles split evenly over the threads");
    double va[R], vb[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = (int)threadIdx.x + r * kBT;
        const int c = q / kTile, i = q % kTile;       // A: column c, row i
        const int cu = q % kNb, ju = q / kNb;         // Bt: row cu, column ju
        va[r] = (c < nb && i0 + i < m) ? G[(int64_t)(p0 + c) * m + i0 + i] : 0.0;
        vb[r] = (cu < nb && j0 + ju < m) ? G[(int64_t)(j0 + ju) * m + p0 + cu] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = (int)threadIdx.x + r * kBT;
        A[q / kTile][q % kTile] = va[r];
        Bt[q % kNb][q / kNb] = vb[r];
    }
}

// tile = (front, p0, i0, j0): F[i0:i0+64, j0:j0+64] -= L[.., p0:p0+nb] U[p0:p0+nb, ..]
__global__ __launch_bounds__(kBT) void k_mf_gemm(const BigDev* P, double* pool, const int4* tiles) {
    __shared__ double A[kNb][kTile + 1];   // L panel, transposed: A[c][i]
    __shared__ double Bt[kNb][kTile + 1];  // U panel: Bt[c][j]
    const int4 t = tiles[blockIdx.x];
    const int s = t.x, p0 = t.y, i0 = t.z, j0 = t.w;
    const int m = P->sn_m[s], k = sn_k(P, s);
    const int nb = (k - p0) < kNb ? (k - p0) : kNb;
    double* G = pool + P->sn_off[s];
    load_panel_tiles(A, Bt, G, m, p0, i0, j0, nb);
    __syncthreads();
    tile_update_valu(A, Bt, G, m, i0, j0, nb);
}

// The same update on the FP64 matrix cores: four wavefronts, each a 32 x 32
// quarter of the tile as 2 x 2 blocks of v_mfma_f64_16x16x4f64 (A: lane l
// holds A[l%16][l/16], B: B[l/16][l%16], accumulator element v of lane l is
// D[l/16 + 4v][l%16], as measured on gfx950).
typedef double dbl4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void tile_update_mfma(const double (*A)[kTile + 1], const double (*Bt)[kTile + 1],
                                                 double* G, int m, int i0, int j0, int nb) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    const int r16 = lane & 15, q4 = lane >> 4;
    dbl4 acc[2][2];
    for (int bi = 0; bi < 2; bi++)
        for (int bj = 0; bj < 2; bj++) acc[bi][bj] = dbl4{0.0, 0.0, 0.0, 0.0};
    for (int kk = 0; kk < nb; kk += 4) {
        const double a0 = A[kk + q4][wi + r16], a1 = A[kk + q4][wi + 16 + r16];
        const double b0 = Bt[kk + q4][wj + r16], b1 = Bt[kk + q4][wj + 16 + r16];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
    for (int bi = 0; bi < 2; bi++)
        for (int bj = 0; bj < 2; bj++) {
            const int j = j0 + wj + bj * 16 + r16;
            if (j >= m) continue;
            for (int v = 0; v < 4; v++) {
                const int i = i0 + wi + bi * 16 + q4 + 4 * v;
                if (i < m) G[(int64_t)j * m + i] -= acc[bi][bj][v];
            }
        }
}

// The tile entries tile_update_mfma's thread subtracts from, read ahead:
// cv[(2 bi + bj) 4 + v] (zero outside the front)
__device__ __forceinline__ void tile_load_mfma(const double* G, int m, int i0, int j0, double (&cv)[16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    const int r16 = lane & 15, q4 = lane >> 4;
#pragma unroll
    for (int bi = 0; bi < 2; bi++)
#pragma unroll
        for (int bj = 0; bj < 2; bj++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int j = j0 + wj + bj * 16 + r16, i = i0 + wi + bi * 16 + q4 + 4 * v;
                cv[(2 * bi + bj) * 4 + v] = (i < m && j < m) ? G[(int64_t)j * m + i] : 0.0;
            }
}

// tile_update_mfma with the tile's entries already in cv
template <int LD>
__device__ __forceinline__ void tile_update_mfma_c(const double (*A)[LD], const double (*Bt)[LD],
                                                   double* G, int m, int i0, int j0, int nb, const double (&cv)[16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    const int r16 = lane & 15, q4 = lane >> 4;
    dbl4 acc[2][2];
    for (int bi = 0; bi < 2; bi++)
        for (int bj = 0; bj < 2; bj++) acc[bi][bj] = dbl4{0.0, 0.0, 0.0, 0.0};
    for (int kk = 0; kk < nb; kk += 4) {
        const double a0 = A[kk + q4][wi + r16], a1 = A[kk + q4][wi + 16 + r16];
        const double b0 = Bt[kk + q4][wj + r16], b1 = Bt[kk + q4][wj + 16 + r16];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
#pragma unroll
    for (int bi = 0; bi < 2; bi++)
#pragma unroll
        for (int bj = 0; bj < 2; bj++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int j = j0 + wj + bj * 16 + r16, i = i0 + wi + bi * 16 + q4 + 4 * v;
                if (i < m && j < m) G[(int64_t)j * m + i] = cv[(2 * bi + bj) * 4 + v] - acc[bi][bj][v];
            }
}

__global__ __launch_bounds__(kBT) void k_mf_gemm_mfma(const BigDev* P, double* pool, const int4* tiles) {
    __shared__ double A[kNb][kTile + 1];
    __shared__ double Bt[kNb][kTile + 1];
    const int4 t = tiles[blockIdx.x];
    const int s = t.x, p0 = t.y, i0 = t.z, j0 = t.w;
    const int m = P->sn_m[s], k = sn_k(P, s);
    const int nb = (k - p0) < kNb ? (k - p0) : kNb;
    double* G = pool + P->sn_off[s];
    load_panel_tiles(A, Bt, G, m, p0, i0, j0, nb);
    __syncthreads();
    tile_update_mfma(A, Bt, G, m, i0, j0, nb);
}

// Lane src's value (src uniform) for the whole wavefront, by readlane.
__device__ __forceinline__ double wave_bcast(double v, int src) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), src);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Pivots [p, min(p + kStage, nb)) of a panel step, one panel row (Col:
// column) per lane in registers; lanes 0..31 carry the diagonal block's, the
// pivot's own lane p supplies the step's other operand by readlane.  The
// registers rotate by one per pivot, so a[0] is always the entry of the
// pivot's column (Col: row) and every register index is fixed:
//   row i:     l = a[0] * (1 / u(p,p)) is L(i,p);    a[j] = a[j+1] - l u(p,j)
//   column j:  a[0] is U(p,j);  a[i] = a[i+1] - l(i,p) a[0], the same l
// Lanes at or before the pivot go on computing; nothing reads what
// holds.  W registers are still needed when the stage begins.  put(p, x, ip)
// takes each finished entry x (row: L(i,p); column: U(p,j)) and 1 / u(p,p).
constexpr int kStage = 8;
constexpr int kPanLd = kNb + kTile + 1;
template <bool Col, int W, class Put>
__device__ __forceinline__ void panel_stage(double (&a)[kNb], int& p, int nb, double& ip, Put put) {
#pragma unroll 1
    for (int q = 0; q < kStage && p < nb; q++, p++) {
        const double l = Col ? a[0] : a[0] * ip;
        put(p, l, ip);
        const double ipc = ip;
        auto update = [&](int i) {
            const double o = wave_bcast(a[i + 1], p);
            a[i] = Col ? a[i + 1] - (o * ipc) * l : a[i + 1] - l * o;
        };
        // the next pivot first; the dependent operations of its reciprocal
        // then alternate with the other updates.  They are the sequence the
        // CDNA instruction set documents for a 64-bit division (scale, estimate,
        // two corrections, quotient, div_fmas, div_fixup), the one the
        // compiler makes of 1.0 / x, written out so that it can be spread
        update(0);
        const double x = wave_bcast(a[0], p + 1);
        constexpr int G = (W - 2 + 8) / 9;
        int i = 1;
        auto group = [&] {
#pragma unroll
            for (int g = 0; g < G; g++)
                if (i < W - 1) update(i++);
            __builtin_amdgcn_sched_barrier(0);
        };
        bool fd, fn;
        const double d = __builtin_amdgcn_div_scale(1.0, x, false, &fd);
        double r = __builtin_amdgcn_rcp(d);
        group();
        double e = __builtin_fma(-d, r, 1.0);
        group();
        r = __builtin_fma(r, e, r);
        group();
        e = __builtin_fma(-d, r, 1.0);
        group();
        r = __builtin_fma(r, e, r);
        group();
        const double n = __builtin_amdgcn_div_scale(1.0, x, true, &fn);
        const double t = n * r;
        group();
        e = __builtin_fma(-d, t, n);
        group();
        e = __builtin_amdgcn_div_fmas(e, r, t, fn);
        group();
        ip = __builtin_amdgcn_div_fixup(e, x, 1.0);
        group();
    }
}
template <bool Col, class Put>
__device__ __forceinline__ void panel_lu(double (&a)[kNb], int nb, Put put) {
    int p = 0;
    double ip = 1.0 / wave_bcast(a[0], 0);
    if (nb > 24) panel_stage<Col, 32>(a, p, nb, ip, put);
    if (nb > 16) panel_stage<Col, 24>(a, p, nb, ip, put);
    if (nb > 8) panel_stage<Col, 16>(a, p, nb, ip, put);
    panel_stage<Col, 8>(a, p, nb, ip, put);
}
static_assert(kNb == 4 * kStage && kTile == 64 && kBT == 256, "panel_lu's stages and wavefronts");

// One step of the blocked front LU in one launch.  item = (front, p0, i0,
// j0): every workgroup factors the diagonal block [p0, p1), solves the L
// rows [i0, i0+64) and the U columns [j0, j0+64) it needs, and updates the
// trailing tile F[i0:, j0:]; (front, p0, -1, -1) is a step with no trailing
// matrix (p1 = m).  The operations and their order are those of k_mf_diag,
// k_mf_trsm and the trailing update, so the factors are the same bits.
//
// The step is one serial chain over its pivots.  The factorization of the
// diagonal block, then staged coefficients, then the triangular solves were
// three such phases, with an LDS round trip and a barrier per pivot in the
// first.  Now four wavefronts each carry the diagonal block's 32 rows (or
// columns) beside 32 rows of L (columns of U) and go through the pivots
// once, in registers, with no barrier and no LDS read: a step
// of a 450 x 450 grid's factorization took 36 us, now 24.
//
// Workgroups of the step read the unfactored panel from the front,
// so the factored panel goes to the workspace W instead (the same layout,
// at woff[front]): the diagonal block from the tile (p1, p1) or the item
// without trailing matrix, L rows from the tiles with j0 = p1, U columns
// from those with i0 = p1.  k_mf_flush copies it back once the level's
// steps are done; later steps read only the trailing matrix.
template <bool Mfma>
__global__ __launch_bounds__(kBT) void k_mf_panel(const BigDev* P, double* pool, double* dinv, double* W,
                                                  const int64_t* woff, const int4* items) {
    // A[c][i]: rows of the panel's column c, the diagonal block's 32 first,
    // then the L rows; Bt[c][j]: columns of its row c, likewise
    __shared__ double A[kNb][kPanLd];
    __shared__ double Bt[kNb][kPanLd];
    const int4 it = items[blockIdx.x];
    const int s = it.x, p0 = it.y, i0 = it.z, j0 = it.w;
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int nb = (k - p0) < kNb ? (k - p0) : kNb, p1 = p0 + nb;
    double* G = pool + P->sn_off[s];
    double* Wf = W + woff[s];
    const bool tile = i0 >= 0;
    {
        // all loads before the first LDS store, addresses running down the
        // front's columns; zero past the block, the panel and the front
        constexpr int RD = kNb * kNb / kBT, RT = kNb * kTile / kBT;
        double vd[RD], va[RT], vb[RT];
#pragma unroll
        for (int r = 0; r < RD; r++) {
            const int q = (int)threadIdx.x + r * kBT, j = q / kNb, i = q % kNb;
            vd[r] = (i < nb && j < nb) ? G[(int64_t)(p0 + j) * m + p0 + i] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const int q = (int)threadIdx.x + r * kBT;
            const int c = q / kTile, i = q % kTile;       // A: column c, row i
            const int cu = q % kNb, ju = q / kNb;         // Bt: row cu, column ju
            va[r] = (tile && c < nb && i0 + i < m) ? G[(int64_t)(p0 + c) * m + i0 + i] : 0.0;
            vb[r] = (tile && cu < nb && j0 + ju < m) ? G[(int64_t)(j0 + ju) * m + p0 + cu] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < RD; r++) {
            const int q = (int)threadIdx.x + r * kBT, j = q / kNb, i = q % kNb;
            A[j][i] = vd[r];
            Bt[i][j] = vd[r];
        }
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const int q = (int)threadIdx.x + r * kBT;
            A[q / kTile][kNb + q % kTile] = va[r];
            Bt[q % kNb][kNb + q / kNb] = vb[r];
        }
    }
    double cv[16];   // the trailing tile, read ahead of the LU (MFMA form)
    if (Mfma && tile) tile_load_mfma(G, m, i0, j0, cv);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // wavefronts 0 and 1: rows, 2 and 3: columns
    double* mine = &(wave < 2 ? A : Bt)[0][lane < kNb ? lane : lane + (wave & 1) * kNb];
    double a[kNb];
#pragma unroll
    for (int c = 0; c < kNb; c++) a[c] = mine[c * kPanLd];
    __syncthreads();   // the diagonal block is read by two wavefronts, then overwritten (same values) by both
    const int nbu = __builtin_amdgcn_readfirstlane(nb);
    auto put = [&](int p, double x, double) { mine[p * kPanLd] = x; };
    if (wave < 2) panel_lu<false>(a, nbu, put);
    else panel_lu<true>(a, nbu, put);
    __syncthreads();
    // the diagonal block: L below the diagonal in A, U in Bt
    const bool diag_owner = !tile || (i0 == p1 && j0 == p1);
    if (diag_owner) {
        for (int q = threadIdx.x; q < nb * nb; q += kBT) {
            const int j = q / nb, i = q % nb;
            Wf[(int64_t)(p0 + j) * m + p0 + i] = i > j ? A[j][i] : Bt[i][j];
        }
        if ((int)threadIdx.x < nb) dinv[f0 + p0 + threadIdx.x] = 1.0 / Bt[threadIdx.x][threadIdx.x];
    }
    if (!tile) return;
    if (j0 == p1)
        for (int q = threadIdx.x; q < nb * kTile; q += kBT) {
            const int c = q / kTile, i = q % kTile;
            if (i0 + i < m) Wf[(int64_t)(p0 + c) * m + i0 + i] = A[c][kNb + i];
        }
    if (i0 == p1)
        for (int q = threadIdx.x; q < nb * kTile; q += kBT) {
            const int jj = q / nb, c = q % nb;
            if (j0 + jj < m) Wf[(int64_t)(j0 + jj) * m + p0 + c] = Bt[c][kNb + jj];
        }
    const double (*At)[kPanLd] = (const double (*)[kPanLd])&A[0][kNb];
    const double (*Ut)[kPanLd] = (const double (*)[kPanLd])&Bt[0][kNb];
    if (Mfma) tile_update_mfma_c(At, Ut, G, m, i0, j0, nb, cv);
    else tile_update_valu(At, Ut, G, m, i0, j0, nb);
}

// item = (front, j0): copies the factored panels of columns [j0, j0+4) back
// from the workspace, i.e. the entries (i, j) with min(i, j) < k: the whole
// column for j < k, its rows [0, k) for j >= k
constexpr int kFlushCols = 4;
__device__ __forceinline__ void flush_cols(const BigDev* P, double* pool, const double* W, const int64_t* woff,
                                           const int2 it) {
    const int s = it.x, m = P->sn_m[s], k = sn_k(P, s);
    double* G = pool + P->sn_off[s];
    const double* Wf = W + woff[s];
    const int j1 = (it.y + kFlushCols) < m ? it.y + kFlushCols : m;
    for (int j = it.y; j < j1; j++) {
        const int rows = j < k ? m : k;
        const int64_t o = (int64_t)j * m;
        for (int i = threadIdx.x; i < rows; i += kBT) G[o + i] = Wf[o + i];
    }
}
__global__ __launch_bounds__(kBT) void k_mf_flush(const BigDev* P, double* pool, const double* W,
                                                  const int64_t* woff, const int2* items) {
    const int2 it = items[blockIdx.x];
    flush_cols(P, pool, W, woff, it);
}

// ---- fused per-level front kernels (one workgroup per front) ------------------------------
// Small fronts (m <= TL * R): children's contribution blocks and the
// front's Jacobian entries are gathered into LDS, then the partial LU runs
// with the front in registers: thread t of the TL x TL threads holds rows
// t % TL + TL y and columns t / TL + TL x.  Before pivot p the owners of
// column p and row p publish them in cb / rb (double-buffered, one barrier
// per pivot); the operations and their order are those of the column
// sweep (l(i,p) = a(i,p) * (1 / u(p,p)), then a(i,j) -= l(i,p) u(p,j),
// pivots ascending).  Fronts are bucketed by size so that the small ones
// run as single wavefronts with few registers.
template <int TL, int R>
constexpr int small_doubles(int m_max) { return m_max * m_max + 4 * TL * R; }
template <int TL, int R>
__device__ __forceinline__ void small_front(const BigDev* P, double* pool, double* dinv, const double* Aval,
                                            int s, double* lds, int tid) {
    constexpr int NT = TL * TL, MX = TL * R;
    double (*cb)[MX] = (double (*)[MX])lds;
    double (*rb)[MX] = cb + 2;
    double* F = lds + 4 * MX;
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int64_t off = P->sn_off[s];
    scatter_cb<NT, false>(P, pool, F, m, s, 0, m, nullptr, tid);
    // the front's Jacobian entries (distinct positions: order free), four
    // per thread with their loads ahead of the adds
    {
        constexpr int U = 4;
        const int q1 = P->osn_ptr[s + 1];
        for (int q0 = P->osn_ptr[s] + tid; q0 < q1; q0 += NT * U) {
            int e[U];
#pragma unroll
            for (int u = 0; u < U; u++) e[u] = q0 + u * NT < q1 ? P->osn_pos[q0 + u * NT] : 0;
            int64_t d[U];
            double v[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (q0 + u * NT < q1) {
                    d[u] = P->nat_dest[e[u]] - off;
                    v[u] = Aval[e[u]];
                }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (q0 + u * NT < q1) F[d[u]] += v[u];
        }
    }
    front_sync<NT>();
    const int ti = tid % TL, tj = tid / TL;
    double a[R][R];
#pragma unroll
    for (int y = 0; y < R; y++)
#pragma unroll
        for (int x = 0; x < R; x++) {
            const int i = ti + TL * y, j = tj + TL * x;
            a[y][x] = (i < m && j < m) ? F[j * m + i] : 0.0;
            if (j == 0) cb[0][i] = a[y][x];
            if (i == 0) rb[0][j] = a[y][x];
        }
    front_sync<NT>();
    for (int p = 0; p < k; p++) {
        const int b = p & 1;
        const double ip = 1.0 / rb[b][p];
        if (tid == 0) dinv[f0 + p] = ip;
        double l[R], u[R];
        // the pivot row and column are read unconditionally (in bounds: the
        // buffers hold MX entries) and the update is selected, not branched
#pragma unroll
        for (int y = 0; y < R; y++) {
            const int i = ti + TL * y;
            const double cv = cb[b][i];
            l[y] = (i > p && i < m) ? cv * ip : 0.0;
        }
#pragma unroll
        for (int x = 0; x < R; x++) {
            const int j = tj + TL * x;
            const double rv = rb[b][j];
            u[x] = (j > p && j < m) ? rv : 0.0;
        }
#pragma unroll
        for (int y = 0; y < R; y++) {
            if (TL * y >= m) break;
            const int i = ti + TL * y;
#pragma unroll
            for (int x = 0; x < R; x++) {
                if (TL * x >= m) break;
                const int j = tj + TL * x;
                const double upd = a[y][x] - l[y] * u[x];
                a[y][x] = i > p ? (j == p ? l[y] : (j > p ? upd : a[y][x])) : a[y][x];
                if (j == p + 1) cb[b ^ 1][i] = a[y][x];
                if (i == p + 1) rb[b ^ 1][j] = a[y][x];
            }
        }
        front_sync<NT>();
    }
    double* G = pool + off;
#pragma unroll
    for (int y = 0; y < R; y++)
#pragma unroll
        for (int x = 0; x < R; x++) {
            const int i = ti + TL * y, j = tj + TL * x;
            if (i < m && j < m) G[(int64_t)j * m + i] = a[y][x];
        }
}
// Fronts of 33 to kSmallM rows, one workgroup each, in LDS (odd leading
// dimension: a wavefront reads its columns without bank conflicts): blocks
// of up to 32 pivots go as in k_mf_panel (wavefronts 0 and 1 rows, 2 and 3
// columns, the block's own in lanes [0, nb) of each; 2 (64 - nb) lanes are
// left for at most kSmallM - nb further ones), then the trailing block on
// the FP64 matrix cores, the front's own value as the first addend, so an
// entry is summed as the column sweep sums it.  Before, every pivot published
// its row and column in LDS behind a barrier, with 16 or 36 entries a thread:
// the fronts of 33 to 96 rows of a 450 x 450 grid took 0.73 ms per
// factorization, now 0.45; a 150 x 150 grid's level heads 0.57 ms, now 0.37.
static_assert(2 * (64 - kNb) >= kSmallM - kNb, "a panel's rows fit two wavefronts");
__device__ __forceinline__ void mid_front(const BigDev* P, double* pool, double* dinv, const double* Aval, int s,
                                          double* F) {
    const int m = __builtin_amdgcn_readfirstlane(P->sn_m[s]), k = __builtin_amdgcn_readfirstlane(sn_k(P, s));
    const int f0 = P->sn_first[s], ld = m | 1;
    const int64_t off = P->sn_off[s];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    scatter_cb<kBT, false>(P, pool, F, ld, s, 0, m, nullptr, threadIdx.x);
    for (int q = P->osn_ptr[s] + threadIdx.x; q < P->osn_ptr[s + 1]; q += kBT) {
        const int e = P->osn_pos[q], d = (int)(P->nat_dest[e] - off), j = d / m;
        F[j * ld + d - j * m] += Aval[e];
    }
    __syncthreads();
    const int r16 = lane & 15, q4 = lane >> 4;
    for (int p0 = 0; p0 < k; p0 += kNb) {
        const int nb = (k - p0) < kNb ? (k - p0) : kNb, p1 = p0 + nb, rows = m - p1;
        const bool col = wave >= 2, work = !(wave & 1) || rows > 64 - nb;
        const int idx = lane < nb ? p0 + lane : p1 + (wave & 1) * (64 - nb) + lane - nb;
        double* mine = F + (col ? idx * ld + p0 : p0 * ld + idx);
        const int st = col ? 1 : ld;
        double a[kNb];
        if (work) {
#pragma unroll
            for (int c = 0; c < kNb; c++) a[c] = (c < nb && idx < m) ? mine[c * st] : 0.0;
        }
        __syncthreads();   // before a block row or column is overwritten
        if (work) {
            // of the diagonal block the rows keep what is below the diagonal,
            // the columns the rest; both wavefronts of a kind store the same
            const int lc = idx < m ? lane + (col ? 1 : 0) : -1;
            auto put = [&](int p, double x, double ip) {
                if (lc > p) mine[p * st] = x;
                if (threadIdx.x == 0) dinv[f0 + p0 + p] = ip;
            };
            if (col) panel_lu<true>(a, nb, put);
            else panel_lu<false>(a, nb, put);
        }
        __syncthreads();
        const int nt = (rows + 15) >> 4;
        for (int t = wave; t < nt * nt; t += kBT / 64) {
            const int i0 = p1 + (t % nt) * 16, j0 = p1 + (t / nt) * 16;
            dbl4 acc;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + q4 + 4 * v, j = j0 + r16;
                acc[v] = (i < m && j < m) ? F[j * ld + i] : 0.0;
            }
            for (int kk = 0; kk < nb; kk += 4) {
                const int c = kk + q4, i = i0 + r16, j = j0 + r16;
                const double av = (c < nb && i < m) ? F[(p0 + c) * ld + i] : 0.0;
                const double bv = (c < nb && j < m) ? F[j * ld + p0 + c] : 0.0;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-av, bv, acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + q4 + 4 * v, j = j0 + r16;
                if (i < m && j < m) F[j * ld + i] = acc[v];
            }
        }
        __syncthreads();
    }
    double* G = pool + off;
    for (int j = wave; j < m; j += kBT / 64)
        for (int i = lane; i < m; i += 64) G[j * m + i] = F[j * ld + i];
}
__global__ __launch_bounds__(kBT) void k_mf_lvl_mid(const BigDev* P, double* pool, double* dinv, const double* Aval,
                                                    const int32_t* fronts) {
    extern __shared__ double lds_f[];
    mid_front(P, pool, dinv, Aval, fronts[blockIdx.x], lds_f);
}
template <int TL, int R>
__global__ __launch_bounds__(TL * TL) void k_mf_lvl_small(const BigDev* P, double* pool, double* dinv,
                                                          const double* Aval, const int32_t* fronts) {
    extern __shared__ double lds_f[];
    small_front<TL, R>(P, pool, dinv, Aval, fronts[blockIdx.x], lds_f, threadIdx.x);
}
// size buckets: one wavefront per front, then one workgroup (by LDS size)
constexpr int kSmallBuckets = 3;
constexpr int kBucketMax[kSmallBuckets] = {32, 64, kSmallM};
static_assert(8 * 4 >= kBucketMax[0], "small fronts exceed their kernel");

// The independent work at the head of a level in one launch: its small
// fronts of every bucket, the gather tiles of its large ones (with their
// Jacobian entries), and the copies of the previous level's factored panels
// from the workspace (this level reads only that level's contribution
// blocks).  As launches of their own these ran one after the other, each
// with too few workgroups to fill the chip: a 150 x 150 grid's factorization
// went from 1.34 to 1.00 ms (98 launches to 56).
// item = (kind, a, b, c):
//   kHeadSmall32: fronts[a, a + b), one wavefront each, b <= 4
//   kHeadMid: front fronts[a]
//   kHeadGather: tile a, Jacobian positions borig[b, c)
//   kHeadFlush: flush item a
enum { kHeadSmall32, kHeadMid, kHeadGather, kHeadFlush };
__global__ __launch_bounds__(kBT) void k_mf_head(const BigDev* P, double* pool, double* dinv, const double* Aval,
                                                 const int4* items, const int32_t* fronts, const int4* tiles,
                                                 const int2* cbr, const int32_t* borig, const double* W,
                                                 const int64_t* woff, const int2* flush, int lds32) {
    extern __shared__ double lds_f[];
    const int4 it = items[blockIdx.x];
    if (it.x == kHeadSmall32) {
        const int wave = threadIdx.x >> 6;
        if (wave < it.z)
            small_front<8, 4>(P, pool, dinv, Aval, fronts[it.y + wave], lds_f + wave * lds32, threadIdx.x & 63);
    } else if (it.x == kHeadMid) {
        mid_front(P, pool, dinv, Aval, fronts[it.y], lds_f);
    } else if (it.x == kHeadGather) {
        gather_tile(P, pool, tiles[it.y], cbr, lds_f, Aval, borig + it.z, it.w - it.z);
    } else {
        flush_cols(P, pool, W, woff, flush[it.y]);
    }
}

// Large fronts, one workgroup each: gather, then blocked right-looking
// partial LU in global memory (L2-resident): diagonal block in LDS, row and
// column triangular solves, trailing update by 64 x 64 tiles on the FP64
// matrix cores.
__global__ __launch_bounds__(kBT) void k_mf_lvl_big(const BigDev* P, double* pool, double* dinv,
                                                    const double* Aval, const int32_t* fronts) {
    __shared__ double D[kNb * kNb];
    __shared__ double EU[kCoef], EL[kCoef];
    __shared__ double invd[kNb];
    __shared__ double cb[2][kNb], rb[2][kNb];
    __shared__ double A[kNb][kTile + 1];
    __shared__ double Bt[kNb][kTile + 1];
    const int s = fronts[blockIdx.x];
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int64_t off = P->sn_off[s];
    double* G = pool + off;
    scatter_cb<kBT, true>(P, pool, G, m, s, 0, m, nullptr, threadIdx.x);
    for (int q = P->osn_ptr[s] + threadIdx.x; q < P->osn_ptr[s + 1]; q += kBT) {
        const int e = P->osn_pos[q];
        G[P->nat_dest[e] - off] += Aval[e];
    }
    gsync();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    const int r16 = lane & 15, q4 = lane >> 4;
    for (int p0 = 0; p0 < k; p0 += kNb) {
        const int nb = (k - p0) < kNb ? (k - p0) : kNb;
        const int p1 = p0 + nb;
        // diagonal block
        for (int q = threadIdx.x; q < nb * nb; q += kBT) {
            const int j = q / nb, i = q % nb;
            D[j * kNb + i] = G[(int64_t)(p0 + j) * m + p0 + i];
        }
        __syncthreads();
        diag_lu_block<kBT>(D, invd, nb, cb, rb);
        __syncthreads();
        for (int q = threadIdx.x; q < nb * nb; q += kBT) {
            const int j = q / nb, i = q % nb;
            G[(int64_t)(p0 + j) * m + p0 + i] = D[j * kNb + i];
        }
        if ((int)threadIdx.x < nb) dinv[f0 + p0 + threadIdx.x] = invd[threadIdx.x];
        load_coef<true>(EU, D, kNb, nb);
        load_coef<false>(EL, D, kNb, nb);
        __syncthreads();
        // L21 rows and U12 columns
        for (int r = p1 + threadIdx.x; r < m; r += kBT) {
            double a[kNb];
#pragma unroll
            for (int c = 0; c < kNb; c++) a[c] = c < nb ? G[(int64_t)(p0 + c) * m + r] : 0.0;
            rot_solve<true>(a, EU, invd, nb, [&](int c, double x) { G[(int64_t)(p0 + c) * m + r] = x; });
        }
        for (int r = p1 + threadIdx.x; r < m; r += kBT) {
            double* col = G + (int64_t)r * m + p0;
            double a[kNb];
#pragma unroll
            for (int c = 0; c < kNb; c++) a[c] = c < nb ? col[c] : 0.0;
            rot_solve<false>(a, EL, nullptr, nb, [&](int c, double x) { col[c] = x; });
        }
        gsync();
        // trailing update
        for (int j0 = p1; j0 < m; j0 += kTile)
            for (int i0 = p1; i0 < m; i0 += kTile) {
                for (int q = threadIdx.x; q < kNb * kTile; q += kBT) {
                    const int c = q / kTile, i = q % kTile;
                    const bool ok = c < nb;
                    A[c][i] = (ok && i0 + i < m) ? G[(int64_t)(p0 + c) * m + i0 + i] : 0.0;
                    Bt[c][i] = (ok && j0 + i < m) ? G[(int64_t)(j0 + i) * m + p0 + c] : 0.0;
                }
                __syncthreads();
                dbl4 acc[2][2];
                for (int bi = 0; bi < 2; bi++)
                    for (int bj = 0; bj < 2; bj++) acc[bi][bj] = dbl4{0.0, 0.0, 0.0, 0.0};
                for (int kk = 0; kk < nb; kk += 4) {
                    const double a0 = A[kk + q4][wi + r16], a1 = A[kk + q4][wi + 16 + r16];
                    const double b0 = Bt[kk + q4][wj + r16], b1 = Bt[kk + q4][wj + 16 + r16];
                    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
                    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
                    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
                    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
                }
                for (int bi = 0; bi < 2; bi++)
                    for (int bj = 0; bj < 2; bj++) {
                        const int j = j0 + wj + bj * 16 + r16;
                        if (j >= m) continue;
                        for (int v = 0; v < 4; v++) {
                            const int i = i0 + wi + bi * 16 + q4 + 4 * v;
                            if (i < m) G[(int64_t)j * m + i] -= acc[bi][bj][v];
                        }
                    }
                __syncthreads();
            }
        gsync();
    }
}

// ---- multifrontal solves ----------------------------------------------------------------
// forward: y = L^-1 b by levels; update vectors of the fronts in uvec
// The solves' diagonal block: S[pp * 65 + ii] = G[(b0 + pp) m + b0 + ii]
// for pp < nbk (zero for ii >= nbk); a thread's loads of each group of up to
// 16 entries are issued before the group's first store, and groups whose
// columns all lie past the block are skipped
template <int BT>
__device__ __forceinline__ void stage_solve_block(double* S, const double* G, int m, int b0, int nbk) {
    constexpr int R = 64 * 64 / BT;       // entries per thread of a full block
    constexpr int GR = R < 16 ? R : 16;   // entries per thread per group
    constexpr int PP = BT / 64;           // block columns per entry step
#pragma unroll 1
    for (int g0 = 0; g0 < R; g0 += GR) {
        if (g0 * PP >= nbk) break;
        double t[GR];
#pragma unroll
        for (int r = 0; r < GR; r++) {
            const int q = (int)threadIdx.x + (g0 + r) * BT, pp = q >> 6, ii = q & 63;
            t[r] = (pp < nbk && ii < nbk) ? G[(int64_t)(b0 + pp) * m + b0 + ii] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < GR; r++) {
            const int q = (int)threadIdx.x + (g0 + r) * BT, pp = q >> 6, ii = q & 63;
            if (pp < nbk) S[pp * 65 + ii] = t[r];
        }
    }
}

// acc - sum_j G[c_j m + i] y[c_j] over the columns c_j = c0 + j dir, j < n,
// summed in order of j, as the plain loop sums them (the same roundings).  The
// loads go out 16 at a time (the last group predicated), so a row waits for
// ceil(n / 16) memory latencies, and the address advances by one column per
// load.  Sixteen measured faster than 64 (registers) and than the compiler's
// own schedule of the plain loop on the 450 x 450 power-grid solves.
__device__ __forceinline__ double sub_cols(double acc, const double* G, int m, int i, int c0, int dir, int n,
                                           const double* y) {
    constexpr int CH = 16;
    int64_t st = (int64_t)dir * m;
    asm volatile("" : "+v"(st));   // an opaque stride: no per-column offsets hoisted into registers
    const double* gp = G + ((int64_t)c0 * m + i);
    int j = 0;
#pragma unroll 1
    for (; j + CH <= n; j += CH) {
        double g[CH];
#pragma unroll
        for (int q = 0; q < CH; q++) {
            g[q] = *gp;
            if (j + q + 1 < n) gp += st;   // never past the last column
        }
#pragma unroll
        for (int q = 0; q < CH; q++) acc -= g[q] * y[c0 + (j + q) * dir];
    }
    if (j < n) {
        double g[CH];
#pragma unroll
        for (int q = 0; q < CH; q++) {
            g[q] = j + q < n ? *gp : 0.0;
            if (j + q + 1 < n) gp += st;
        }
#pragma unroll
        for (int q = 0; q < CH; q++)
            if (j + q < n) acc -= g[q] * y[c0 + (j + q) * dir];
    }
    return acc;
}

// One workgroup of BT threads per front (64, 256 or 512 by level)
template <int BT>
__global__ __launch_bounds__(BT) void k_mf_fwd(const BigDev* P, const double* pool, double* x, double* uvec,
                                               const int32_t* fronts, int ld_off) {
    extern __shared__ double v[];
    double* Ld = v + ld_off;   // the diagonal block, row stride 65
    const int s = fronts[blockIdx.x];
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const double* G = pool + P->sn_off[s];
    for (int a = threadIdx.x; a < m; a += BT) v[a] = a < k ? x[f0 + a] : 0.0;
    __syncthreads();
    const int c0 = P->ch_ptr[s], c1 = P->ch_ptr[s + 1];
    int4 next = c0 < c1 ? P->ch_rec[c0] : make_int4(0, 0, 0, 0);
    for (int cq = c0; cq < c1; cq++) {
        const int rc = next.x, rp = next.z;
        if (cq + 1 < c1) next = P->ch_rec[cq + 1];
        for (int a = threadIdx.x; a < rc; a += BT) v[P->rel[rp + a]] += uvec[rp + a];
        __syncthreads();
    }
    // blocks of 64 pivots: the diagonal block (staged in LDS) by the first
    // wavefront, one row per lane and the pivot values by shuffle; then the
    // rows below the block (one row per thread, the block's columns of L)
    const int lane = threadIdx.x & 63;
    for (int b0 = 0; b0 < k; b0 += 64) {
        const int b1 = (k - b0) < 64 ? k : b0 + 64;
        const int nbk = b1 - b0;
        stage_solve_block<BT>(Ld, G, m, b0, nbk);
        __syncthreads();
        if (threadIdx.x < 64) {
            const int i = b0 + lane;
            double vi = i < b1 ? v[i] : 0.0;
            // the lane's row of the block, 16 columns at a time, in registers
            // before the dependent steps that use it
            for (int p0 = 0; p0 < nbk; p0 += 16) {
                double l[16];
#pragma unroll
                for (int q = 0; q < 16; q++) l[q] = p0 + q < nbk ? Ld[(p0 + q) * 65 + lane] : 0.0;
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int p = p0 + q;
                    if (p < nbk) {
                        const double y = wave_bcast(vi, p);
                        if (lane > p && lane < nbk) vi -= l[q] * y;
                    }
                }
            }
            if (i < b1) v[i] = vi;
        }
        __syncthreads();
        #pragma unroll 1
        for (int i = b1 + threadIdx.x; i < m; i += BT) v[i] = sub_cols(v[i], G, m, i, b0, 1, nbk, v);
        __syncthreads();
    }
    for (int a = threadIdx.x; a < m; a += BT) {
        if (a < k) x[f0 + a] = v[a];
        else uvec[P->rel_ptr[s] + (a - k)] = v[a];
    }
}

// backward: x = U^-1 y from the root down
template <int BT>
__global__ __launch_bounds__(BT) void k_mf_bwd(const BigDev* P, const double* pool, const double* dinv,
                                               double* x, const int32_t* fronts, int ld_off) {
    extern __shared__ double w[];
    double* Ud = w + ld_off;   // the diagonal block, row stride 65
    const int s = fronts[blockIdx.x];
    const int m = P->sn_m[s], k = sn_k(P, s), f0 = P->sn_first[s];
    const int r = m - k;
    const double* G = pool + P->sn_off[s];
    const int32_t* rows = P->sn_rows + P->sn_rptr[s];
    for (int a = threadIdx.x; a < r; a += BT) w[k + a] = x[rows[a]];
    __syncthreads();
    #pragma unroll 1
    for (int p = threadIdx.x; p < k; p += BT) w[p] = sub_cols(x[f0 + p], G, m, p, k, 1, r, w);
    __syncthreads();
    // blocks of 64 pivots from the bottom: the diagonal block of U (staged in
    // LDS) by the first wavefront (row per lane, solution values by
    // shuffle), then the rows above it
    const int lane = threadIdx.x & 63;
    for (int b1 = k; b1 > 0; b1 -= 64) {
        const int b0 = b1 > 64 ? b1 - 64 : 0;
        const int nbk = b1 - b0;
        stage_solve_block<BT>(Ud, G, m, b0, nbk);
        __syncthreads();
        if (threadIdx.x < 64) {
            const int i = b0 + lane;
            double wi = i < b1 ? w[i] : 0.0;
            const double di = i < b1 ? dinv[f0 + i] : 0.0;   // the lane's own 1 / u(i, i)
            // columns from the last, 16 at a time, the lane's entries in
            // registers before the dependent steps that use them
            for (int p1 = nbk - 1; p1 >= 0; p1 -= 16) {
                double u[16];
#pragma unroll
                for (int q = 0; q < 16; q++) u[q] = p1 - q >= 0 ? Ud[(p1 - q) * 65 + lane] : 0.0;
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int p = p1 - q;
                    if (p >= 0) {
                        if (lane == p) wi *= di;
                        const double xp = wave_bcast(wi, p);
                        if (lane < p) wi -= u[q] * xp;
                    }
                }
            }
            if (i < b1) w[i] = wi;
        }
        __syncthreads();
        #pragma unroll 1
        for (int i = threadIdx.x; i < b0; i += BT) w[i] = sub_cols(w[i], G, m, i, b1 - 1, -1, nbk, w);
        __syncthreads();
    }
    for (int p = threadIdx.x; p < k; p += BT) x[f0 + p] = w[p];
}

// ---- step controller ----------------------------------------------------------------------
__global__ __launch_bounds__(kBT) void k_predict(int n, int np, int k, double w0, double w1, double w2,
                                                 double a1, double a2, const double* U0, const double* U1,
                                                 const double* U2, const double* Q0, const double* Q1,
                                                 double* up, double* u, double* qx) {
    for (int i = blockIdx.x * kBT + threadIdx.x; i < n; i += gridDim.x * kBT) {
        double v = U0[i];
        if (np == 2) v = w0 * U0[i] + w1 * U1[i];
        else if (np == 3) v = w0 * U0[i] + w1 * U1[i] + w2 * U2[i];
        up[i] = v;
        u[i] = v;
        qx[i] = a1 * Q0[i] + (k == 2 ? a2 * Q1[i] : 0.0);
    }
}

__global__ __launch_bounds__(kBT) void k_charges_chunks(const BigDev* P, const double* Clin, const double* v,
                                                        double* lpart) {
    __shared__ double red[kBT];
    const int4 ch = P->long_chunks[blockIdx.x];
    double acc = 0.0;
    const int q = ch.z + threadIdx.x;
    if (ch.y == 0 && q < ch.w) acc = Clin[q] * v[P->col[q]];
    const double t = blk_reduce(acc, red, Sum());
    if (threadIdx.x == 0) lpart[blockIdx.x] = t;
}

__global__ __launch_bounds__(kBT) void k_charges_finish(const BigDev* P, const double* lpart, double* q) {
    __shared__ double pl[kBT];
    __shared__ int kl[kBT];
    const int l = blockIdx.x;
    const int cb = P->long_cptr[l], ce = P->long_cptr[l + 1];
    double acc = 0.0;
    for (int c0 = cb; c0 < ce; c0 += kBT) {
        const int c = c0 + threadIdx.x;
        if (c < ce) {
            kl[threadIdx.x] = P->long_chunks[c].y;
            pl[threadIdx.x] = lpart[c];
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const int nc = (ce - c0) < kBT ? ce - c0 : kBT;
            for (int t = 0; t < nc; t++)
                if (kl[t] == 0) acc += pl[t];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) q[P->long_rows[l]] = acc;
}

__global__ __launch_bounds__(kBT) void k_charges(const BigDev* P, const double* Clin, const double* v,
                                                 double* q) {
    for (int r = blockIdx.x * kBT + threadIdx.x; r < P->n; r += gridDim.x * kBT) {
        if (P->row_long[r]) continue;
        double acc = 0.0;
        for (int e = P->rowptr[r]; e < P->rowptr[r + 1]; e++) acc += Clin[e] * v[P->col[e]];
        q[r] = acc;
    }
}

__global__ __launch_bounds__(kBT) void k_lte(int n, double c, double rtol, double atol, const double* u,
                                             const double* up, const double* U0, double* part) {
    __shared__ double red[kBT];
    double ss = 0.0;
    for (int i = blockIdx.x * kBT + threadIdx.x; i < n; i += gridDim.x * kBT) {
        const double est = c * (u[i] - up[i]);
        const double m = fmax(fabs(u[i]), fabs(U0[i]));
        const double r = est / (rtol * m + atol);
        ss += r * r;
    }
    const double s = blk_reduce(ss, red, Sum());
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBT) void k_sum_reduce(const double* part, int nb, double* out) {
    __shared__ double red[kBT];
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBT) s += part[b];
    s = blk_reduce(s, red, Sum());
    if (threadIdx.x == 0) *out = s;
}

// output samples: wave[(kout) * n_probe + slot] = l0 U0 + l1 U1 + l2 U2 at the probes
__global__ __launch_bounds__(kBT) void k_wave(int n_probe, const int32_t* probe, const double* U0,
                                              const double* U1, const double* U2, double l0, double l1,
                                              double l2, double* row) {
    for (int s = blockIdx.x * kBT + threadIdx.x; s < n_probe; s += gridDim.x * kBT) {
        const int i = probe[s];
        row[s] = l0 * U0[i] + l1 * U1[i] + l2 * U2[i];
    }
}

__global__ __launch_bounds__(kBT) void k_perm_in(int n, const int32_t* prow, const double* b, double* x) {
    for (int r = blockIdx.x * kBT + threadIdx.x; r < n; r += gridDim.x * kBT) x[prow[r]] = b[r];
}
__global__ __launch_bounds__(kBT) void k_perm_out(int n, const int32_t* pcol, const double* x, double* out) {
    for (int c = blockIdx.x * kBT + threadIdx.x; c < n; c += gridDim.x * kBT) out[c] = x[pcol[c]];
}

int grid_for(int64_t work) {
    const int64_t b = (work + kBT - 1) / kBT;
    return (int)std::max<int64_t>(1, std::min<int64_t>(b, kRowBlocks));
}

}  // namespace

// ============================================================================================
struct BigCircuit {
    BigPlan B;
    BigDev hd{};
    BigDev* d_dev = nullptr;
    void* dbuf = nullptr;   // plan arrays
    void* wbuf = nullptr;   // workspace
    double *p = nullptr, *linbuf = nullptr, *Glin = nullptr, *Clin = nullptr, *Aval = nullptr, *pool = nullptr;
    double *dinv = nullptr, *u = nullptr, *x = nullptr, *qx = nullptr, *u0 = nullptr, *st = nullptr;
    double *uvec = nullptr, *part = nullptr, *norm = nullptr, *up = nullptr, *qn = nullptr, *lpart = nullptr;
    double* H[3] = {nullptr, nullptr, nullptr};
    double* Q[2] = {nullptr, nullptr};
    double* scal = nullptr;
    StepDev* sp = nullptr;
    double* h_norm = nullptr;   // pinned
    int32_t* d_probe = nullptr;
    // launch tables
    struct Panel {
        int diag_b, diag_n, trsm_b, trsm_n, gemm_b, gemm_n;
        int pan_b, pan_n;   // one-launch form (k_mf_panel)
    };
    struct Level {
        int tile_b, tile_n, fr_b, fr_n, orig_b, orig_e, big_b, big_n;
        int small_b[kSmallBuckets], small_n[kSmallBuckets];   // fronts up to kBucketMax[bucket]
        size_t small_lds[kSmallBuckets], solve_lds;
        int ld_off;   // offset of the solves' diagonal block in their LDS
        int solve_bt;   // the solves' workgroup size (64, 256 or 512)
        int flush_b, flush_n;
        int tile_lds;                 // bytes of the largest gather tile in LDS
        int head_b, head_n, head_nf, head_lds;   // one-launch head (k_mf_head) without and with the
                                                 // previous level's flush; head_n 0: separate launches
        int head_lds32;               // its LDS per small32 front, in doubles
        std::vector<Panel> panels;
    };
    std::vector<Level> levels;
    int4* d_tiles = nullptr;
    int2* d_cbr = nullptr;
    int32_t* d_fronts = nullptr;
    int2* d_diag = nullptr;
    int4* d_trsm = nullptr;
    int4* d_gemm = nullptr;
    int4* d_pan = nullptr;
    int2* d_flush = nullptr;
    int4* d_head = nullptr;
    int64_t* d_woff = nullptr;   // per front: offset of its factored panels in wpan
    double* wpan = nullptr;
    int32_t* d_borig = nullptr;   // Jacobian positions of the large fronts, by level
    void* tbuf = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph_nf = nullptr;      // the iteration without the factorization (modified Newton)
    hipGraphExec_t exec_nf = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    double factor_ms = 0.0, solve_ms = 0.0;
    bool mfma = false;   // trailing updates on the matrix cores
    // panel steps as diagonal block, solves and trailing update in three
    // launches instead of k_mf_panel's one (CEDAR_MF_PANEL=split)
    bool split_panels = false;
    bool use_graph = true;
    // per level: fused (one workgroup per front) or multi-launch panels;
    // chosen by tune_levels unless CEDAR_MF_FRONT=fused|panel fixes it
    std::vector<char> lvl_fused;
    bool tuned = false;
    std::vector<float> tune_ms_panel, tune_ms_fused;
    // per-launch timing (cs_big_profile): an event pair around each launch
    struct LaunchProf {
        std::vector<hipEvent_t> ev;
        std::vector<int32_t> kind, level;
    };
    LaunchProf* prof = nullptr;
};

// Launch of a factor or solve kernel; under cs_big_profile it is bracketed
// by two events on the stream.
void prof_mark(BigCircuit& C, hipStream_t s, int kind, int level) {
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return;
    (void)hipEventRecord(e, s);
    if (kind >= 0) {
        C.prof->kind.push_back(kind);
        C.prof->level.push_back(level);
    }
    C.prof->ev.push_back(e);
}
#define MF_LAUNCH(kind, lvl, ...)                                   \
    do {                                                            \
        if (C.prof) prof_mark(C, s, kind, lvl);                     \
        hipLaunchKernelGGL(__VA_ARGS__);                            \
        if (C.prof) prof_mark(C, s, -1, lvl);                       \
    } while (0)

namespace {

// Levels of up to this many head items go as one launch.  k_mf_head holds the
// registers and LDS of its largest kind for every item, so where the small
// fronts alone fill the chip many times over the separate kernels are faster:
// the leaf levels of a 450 x 450 grid took 79 + 23, 50 + 41 and 34 + 38 us
// apart and 157, 91 and 64 us as one; of a 150 x 150 grid 34 + 13 and 36 us.
constexpr int kHeadItems = 4096;

template <class T>
size_t pack_add(std::vector<char>& bytes, const std::vector<T>& v) {
    size_t off = (bytes.size() + 15) & ~size_t(15);
    bytes.resize(off + std::max<size_t>(v.size() * sizeof(T), 16));
    if (!v.empty()) std::memcpy(bytes.data() + off, v.data(), v.size() * sizeof(T));
    return off;
}

#define BCHK(expr)                                                                  \
    do {                                                                            \
        hipError_t e_ = (expr);                                                     \
        if (e_ != hipSuccess) {                                                     \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);                \
            return e_ == hipErrorOutOfMemory ? CS_E_OOM : CS_E_HIP;                 \
        }                                                                           \
    } while (0)

int upload(BigCircuit& C, std::string& err) {
    const BigPlan& B = C.B;
    const Plan& P = B.base;
    std::vector<char> by;
    std::vector<int4> mos4, src4;
    std::vector<int32_t> row_long(B.n, 0), long_rows;
    for (int32_t r = 0; r < B.n; r++) {
        int64_t w = P.nat_rowptr[r + 1] - P.nat_rowptr[r] + (P.rnl_ptr[r + 1] - P.rnl_ptr[r]);
        for (int32_t e = P.nat_rowptr[r]; e < P.nat_rowptr[r + 1]; e++) w += P.jnl_ptr[e + 1] - P.jnl_ptr[e];
        if (w > 256) { row_long[r] = 1; long_rows.push_back(r); }
    }
    std::vector<int32_t> long_cptr(1, 0);
    std::vector<int4> long_chunks;
    for (int32_t r : long_rows) {
        for (int32_t e = P.nat_rowptr[r]; e < P.nat_rowptr[r + 1]; e += kBT)
            long_chunks.push_back(make_int4(r, 0, e, std::min(e + kBT, P.nat_rowptr[r + 1])));
        for (int32_t q = P.rnl_ptr[r]; q < P.rnl_ptr[r + 1]; q += kBT)
            long_chunks.push_back(make_int4(r, 1, q, std::min(q + kBT, P.rnl_ptr[r + 1])));
        for (int32_t e = P.nat_rowptr[r]; e < P.nat_rowptr[r + 1]; e++) {
            const int32_t t0 = P.jnl_ptr[e], t1 = P.jnl_ptr[e + 1];
            if (t1 - t0 <= kHeavyRefs) continue;
            for (int32_t t = t0; t < t1; t += kBT) long_chunks.push_back(make_int4(r, 2 + e, t, std::min(t + kBT, t1)));
        }
        long_cptr.push_back((int32_t)long_chunks.size());
    }
    for (int32_t q = 0; q < P.n_mos; q++)
        mos4.push_back(make_int4(P.mos[4 * q], P.mos[4 * q + 1], P.mos[4 * q + 2], P.mos[4 * q + 3]));
    for (auto& s : P.src) src4.push_back(make_int4(s.kind, s.off, s.len, s.dc));
    std::vector<int4> ch_rec;
    std::vector<int64_t> ch_blk;
    for (int32_t c : B.ch_sn) {
        const int kc = B.sn_first[c + 1] - B.sn_first[c], mc = B.sn_m[c];
        ch_rec.push_back(make_int4(mc - kc, mc, B.rel_ptr[c], 0));
        ch_blk.push_back(B.sn_off[c] + (int64_t)kc * mc + kc);
    }
    size_t o_rp = pack_add(by, P.nat_rowptr), o_col = pack_add(by, P.nat_col), o_lk = pack_add(by, P.lin_kind),
           o_li = pack_add(by, P.lin_idx), o_gp = pack_add(by, P.g_ptr), o_gr = pack_add(by, P.g_ref),
           o_cp = pack_add(by, P.c_ptr), o_cr = pack_add(by, P.c_ref), o_jp = pack_add(by, P.jnl_ptr),
           o_jr = pack_add(by, P.jnl_ref), o_rnp = pack_add(by, P.rnl_ptr), o_rnr = pack_add(by, P.rnl_ref),
           o_isd = pack_add(by, P.is_diff), o_prow = pack_add(by, B.prow), o_pcol = pack_add(by, B.pcol),
           o_mos = pack_add(by, mos4), o_src = pack_add(by, src4), o_sf = pack_add(by, B.sn_first),
           o_sm = pack_add(by, B.sn_m), o_srp = pack_add(by, B.sn_rptr), o_srow = pack_add(by, B.sn_rows),
           o_chp = pack_add(by, B.ch_ptr), o_chs = pack_add(by, B.ch_sn), o_relp = pack_add(by, B.rel_ptr),
           o_rel = pack_add(by, B.rel), o_inv = pack_add(by, B.inv), o_olp = pack_add(by, B.olev_pos),
           o_soff = pack_add(by, B.sn_off), o_invp = pack_add(by, B.inv_ptr), o_nd = pack_add(by, B.nat_dest),
           o_probe = pack_add(by, P.probe), o_osp = pack_add(by, B.osn_ptr), o_osq = pack_add(by, B.osn_pos),
           o_rl = pack_add(by, row_long), o_lr = pack_add(by, long_rows), o_lcp = pack_add(by, long_cptr),
           o_lch = pack_add(by, long_chunks), o_ls = pack_add(by, P.lin_scale), o_mm = pack_add(by, P.mos_m),
           o_smm = pack_add(by, P.src_m), o_crec = pack_add(by, ch_rec), o_cblk = pack_add(by, ch_blk);
    BCHK(hipMalloc(&C.dbuf, by.size()));
    BCHK(hipMemcpy(C.dbuf, by.data(), by.size(), hipMemcpyHostToDevice));
    char* b = (char*)C.dbuf;
    auto I = [&](size_t o) { return (const int32_t*)(b + o); };
    auto L = [&](size_t o) { return (const int64_t*)(b + o); };
    BigDev& d = C.hd;
    d.n = B.n; d.nnz = P.nnz_nat; d.n_mos = P.n_mos; d.n_src = P.n_src; d.n_lin = P.n_lin;
    d.n_stamp = P.n_stamp; d.n_params = P.lay.n_params;
    d.p_mos_vth = P.lay.mos_vth; d.p_mos_kp = P.lay.mos_kp; d.p_mos_w = P.lay.mos_w;
    d.p_mos_l = P.lay.mos_l; d.p_gmin = P.lay.gmin;
    d.rowptr = I(o_rp); d.col = I(o_col); d.lin_kind = I(o_lk); d.lin_idx = I(o_li);
    d.g_ptr = I(o_gp); d.g_ref = I(o_gr); d.c_ptr = I(o_cp); d.c_ref = I(o_cr);
    d.jnl_ptr = I(o_jp); d.jnl_ref = I(o_jr); d.rnl_ptr = I(o_rnp); d.rnl_ref = I(o_rnr);
    d.is_diff = I(o_isd); d.prow = I(o_prow); d.pcol = I(o_pcol);
    d.mos = (const int4*)(b + o_mos); d.src = (const int4*)(b + o_src);
    d.lin_scale = (const double*)(b + o_ls);
    d.mos_m = P.mos_m.empty() ? nullptr : (const double*)(b + o_mm);
    d.src_m = P.src_m.empty() ? nullptr : (const double*)(b + o_smm);
    d.sn_first = I(o_sf); d.sn_m = I(o_sm); d.sn_rptr = I(o_srp); d.sn_rows = I(o_srow);
    d.ch_ptr = I(o_chp); d.ch_sn = I(o_chs); d.rel_ptr = I(o_relp); d.rel = I(o_rel); d.inv = I(o_inv);
    d.olev_pos = I(o_olp); d.sn_off = L(o_soff); d.inv_ptr = L(o_invp); d.nat_dest = L(o_nd);
    d.ch_rec = (const int4*)(b + o_crec); d.ch_blk = L(o_cblk);
    d.osn_ptr = I(o_osp); d.osn_pos = I(o_osq);
    d.row_long = I(o_rl); d.long_rows = I(o_lr); d.n_long = (int32_t)long_rows.size();
    d.long_cptr = I(o_lcp); d.long_chunks = (const int4*)(b + o_lch); d.n_chunks = (int32_t)long_chunks.size();
    C.d_probe = (int32_t*)(b + o_probe);
    BCHK(hipMalloc(&C.d_dev, sizeof(BigDev)));
    BCHK(hipMemcpy(C.d_dev, &C.hd, sizeof(BigDev), hipMemcpyHostToDevice));

    // launch tables
    std::vector<int4> tiles, trsm, gemm, pan, head;
    std::vector<int32_t> fronts, borig;
    std::vector<int2> diag, cbr, flush;
    std::vector<int64_t> woff(std::max(B.ns, 1), 0);
    int64_t wpan_n = 0;   // largest sum of m^2 over one level's large fronts
    // the scatter gathers find a tile's block columns by bisection of the
    // relative maps, which the symbolic analysis builds ascending
    for (int c = 0; c < B.ns; c++)
        for (int a = B.rel_ptr[c] + 1; a < B.rel_ptr[c + 1]; a++)
            if (B.rel[a] <= B.rel[a - 1]) {
                err = "supernodal plan: relative map not ascending";
                return CS_E_INVALID;
            }
    const int nlev = (int)B.lev_ptr.size() - 1;
    C.levels.resize(nlev);
    for (int l = 0; l < nlev; l++) {
        auto& Lv = C.levels[l];
        Lv.tile_b = (int)tiles.size();
        int small_max[kSmallBuckets] = {}, m_max = 0;
        std::vector<int32_t> small[kSmallBuckets], large;
        std::vector<int4> h_gather;
        Lv.tile_lds = 0;
        Lv.orig_b = (int)borig.size();
        for (int q = B.lev_ptr[l]; q < B.lev_ptr[l + 1]; q++) {
            const int s = B.lev_sn[q], m = B.sn_m[s];
            if (m <= kSmallM) {
                int bk = 0;
                while (m > kBucketMax[bk]) bk++;
                small[bk].push_back(s);
                small_max[bk] = std::max(small_max[bk], m);
            } else {
                large.push_back(s);
                // the front's Jacobian positions by column, so that those of a
                // tile are one range
                const size_t ob = borig.size();
                borig.insert(borig.end(), B.osn_pos.begin() + B.osn_ptr[s], B.osn_pos.begin() + B.osn_ptr[s + 1]);
                auto col_of = [&](int32_t pos) { return (int)((B.nat_dest[pos] - B.sn_off[s]) / m); };
                std::stable_sort(borig.begin() + ob, borig.end(),
                                 [&](int32_t a, int32_t b) { return col_of(a) < col_of(b); });
                size_t op = ob;
                const int step = std::max(1, kGatherTile / std::max(m, 1));
                for (int j = 0; j < m; j += step) {
                    const int j1 = std::min(m, j + step);
                    const size_t o0 = op;
                    while (op < borig.size() && col_of(borig[op]) < j1) op++;
                    h_gather.push_back(make_int4(kHeadGather, (int)tiles.size(), (int)o0, (int)op));
                    Lv.tile_lds = std::max<int>(Lv.tile_lds, sizeof(double) * std::min((j1 - j) * m, kGatherChunk));
                    tiles.push_back(make_int4(s, j, j1, (int)cbr.size()));
                    for (int cq = B.ch_ptr[s]; cq < B.ch_ptr[s + 1]; cq++) {
                        const int c = B.ch_sn[cq];
                        const int32_t* rl = B.rel.data() + B.rel_ptr[c];
                        const int rc = B.rel_ptr[c + 1] - B.rel_ptr[c];
                        cbr.push_back(make_int2((int)(std::lower_bound(rl, rl + rc, j) - rl),
                                                (int)(std::lower_bound(rl, rl + rc, j1) - rl)));
                    }
                }
            }
            m_max = std::max(m_max, m);
        }
        Lv.orig_e = (int)borig.size();
        Lv.tile_n = (int)tiles.size() - Lv.tile_b;
        for (int bk = 0; bk < kSmallBuckets; bk++) {
            Lv.small_b[bk] = (int)fronts.size();
            fronts.insert(fronts.end(), small[bk].begin(), small[bk].end());
            Lv.small_n[bk] = (int)small[bk].size();
            const int sm = small_max[bk];
            Lv.small_lds[bk] = sizeof(double) * (bk == 0 ? small_doubles<8, 4>(sm) : sm * (sm | 1));
        }
        // the head's items: what takes longest first, the previous level's
        // panel copies last (left out when that level wrote no workspace)
        Lv.head_b = (int)head.size();
        Lv.head_lds32 = (int)(Lv.small_lds[0] / sizeof(double));
        Lv.head_lds = 0;
        for (int bk = 2; bk >= 1; bk--) {
            for (int q = 0; q < Lv.small_n[bk]; q++)
                head.push_back(make_int4(kHeadMid, Lv.small_b[bk] + q, 0, 0));
            if (Lv.small_n[bk]) Lv.head_lds = std::max(Lv.head_lds, (int)Lv.small_lds[bk]);
        }
        head.insert(head.end(), h_gather.begin(), h_gather.end());
        Lv.head_lds = std::max(Lv.head_lds, Lv.tile_lds);
        for (int q = 0; q < Lv.small_n[0]; q += 4)
            head.push_back(make_int4(kHeadSmall32, Lv.small_b[0] + q, std::min(4, Lv.small_n[0] - q), 0));
        if (Lv.small_n[0])
            Lv.head_lds = std::max(Lv.head_lds, std::min(4, Lv.small_n[0]) * (int)Lv.small_lds[0]);
        Lv.head_n = (int)head.size() - Lv.head_b;
        if (l > 0)
            for (int q = 0; q < C.levels[l - 1].flush_n; q++)
                head.push_back(make_int4(kHeadFlush, C.levels[l - 1].flush_b + q, 0, 0));
        Lv.head_nf = (int)head.size() - Lv.head_b;
        if (Lv.head_n > kHeadItems) Lv.head_n = 0;
        Lv.fr_b = (int)fronts.size();
        for (int q = B.lev_ptr[l]; q < B.lev_ptr[l + 1]; q++) fronts.push_back(B.lev_sn[q]);
        Lv.fr_n = (int)fronts.size() - Lv.fr_b;
        Lv.big_b = (int)fronts.size();
        fronts.insert(fronts.end(), large.begin(), large.end());
        Lv.big_n = (int)large.size();
        int k_lev = 0;
        for (int q = B.lev_ptr[l]; q < B.lev_ptr[l + 1]; q++) {
            const int sq = B.lev_sn[q];
            k_lev = std::max(k_lev, B.sn_first[sq + 1] - B.sn_first[sq]);
        }
        // solves: the front's vector, then its diagonal block (up to 64 x 65)
        Lv.ld_off = (std::max(m_max, 1) + 1) & ~1;
        Lv.solve_lds = sizeof(double) * ((size_t)Lv.ld_off + (size_t)std::min(k_lev, 64) * 65);
        // workgroup size of the solves: fronts of up to 64 rows one wavefront
        // each, so that four times as many are resident; levels of at most 64
        // wider fronts 512 threads, so that a front's rows below a pivot
        // block are updated in one pass with twice the loads in flight
        Lv.solve_bt = m_max <= 64 ? 64 : Lv.fr_n <= 64 ? 512 : kBT;
        int kmax = 0;
        int64_t wl = 0;
        Lv.flush_b = (int)flush.size();
        for (int s : large) {
            const int m = B.sn_m[s];
            kmax = std::max(kmax, B.sn_first[s + 1] - B.sn_first[s]);
            woff[s] = wl;
            wl += ((int64_t)m * m + 1) & ~int64_t(1);
            for (int j0 = 0; j0 < m; j0 += kFlushCols) flush.push_back(make_int2(s, j0));
        }
        Lv.flush_n = (int)flush.size() - Lv.flush_b;
        wpan_n = std::max(wpan_n, wl);
        for (int p0 = 0; p0 < kmax; p0 += kNb) {
            BigCircuit::Panel pn{};
            pn.diag_b = (int)diag.size();
            pn.trsm_b = (int)trsm.size();
            pn.gemm_b = (int)gemm.size();
            pn.pan_b = (int)pan.size();
            for (int s : large) {
                const int k = B.sn_first[s + 1] - B.sn_first[s], m = B.sn_m[s];
                if (p0 >= k) continue;
                const int p1 = std::min(p0 + kNb, k);
                diag.push_back(make_int2(s, p0));
                for (int r0 = p1; r0 < m; r0 += kBT) trsm.push_back(make_int4(s, p0, 0, r0));
                for (int r0 = p1; r0 < m; r0 += kTrsmCols) trsm.push_back(make_int4(s, p0, 1, r0));
                for (int j0 = p1; j0 < m; j0 += kTile)
                    for (int i0 = p1; i0 < m; i0 += kTile) {
                        gemm.push_back(make_int4(s, p0, i0, j0));
                        pan.push_back(make_int4(s, p0, i0, j0));
                    }
                if (p1 >= m) pan.push_back(make_int4(s, p0, -1, -1));
            }
            pn.pan_n = (int)pan.size() - pn.pan_b;
            pn.diag_n = (int)diag.size() - pn.diag_b;
            pn.trsm_n = (int)trsm.size() - pn.trsm_b;
            pn.gemm_n = (int)gemm.size() - pn.gemm_b;
            Lv.panels.push_back(pn);
        }
    }
    std::vector<char> tb;
    size_t o_t = pack_add(tb, tiles), o_f = pack_add(tb, fronts), o_d = pack_add(tb, diag),
           o_tr = pack_add(tb, trsm), o_g = pack_add(tb, gemm), o_bo = pack_add(tb, borig), o_cb = pack_add(tb, cbr),
           o_pa = pack_add(tb, pan), o_fl = pack_add(tb, flush), o_he = pack_add(tb, head), o_wo = pack_add(tb, woff);
    BCHK(hipMalloc(&C.tbuf, tb.size()));
    BCHK(hipMemcpy(C.tbuf, tb.data(), tb.size(), hipMemcpyHostToDevice));
    char* t = (char*)C.tbuf;
    C.d_tiles = (int4*)(t + o_t);
    C.d_fronts = (int32_t*)(t + o_f);
    C.d_diag = (int2*)(t + o_d);
    C.d_trsm = (int4*)(t + o_tr);
    C.d_gemm = (int4*)(t + o_g);
    C.d_borig = (int32_t*)(t + o_bo);
    C.d_cbr = (int2*)(t + o_cb);
    C.d_pan = (int4*)(t + o_pa);
    C.d_flush = (int2*)(t + o_fl);
    C.d_head = (int4*)(t + o_he);
    C.d_woff = (int64_t*)(t + o_wo);

    // workspace
    const size_t n = B.n, nnz = P.nnz_nat;
    const size_t nd = P.lay.n_params + P.n_lin + 3 * nnz + (size_t)B.pool + 16 * n + P.n_stamp +
                      B.rel_ptr[B.ns] + 2 * kRowBlocks + (size_t)C.hd.n_long + (size_t)C.hd.n_chunks + 32 +
                      NRM_SLOTS + 8 + (size_t)wpan_n +
                      sizeof(StepDev) / 8 + 64;
    BCHK(hipMalloc(&C.wbuf, nd * sizeof(double)));
    BCHK(hipMemset(C.wbuf, 0, nd * sizeof(double)));
    double* q = (double*)C.wbuf;
    auto take = [&](size_t k) { double* r = q; q += (k + 1) & ~size_t(1); return r; };
    C.p = take(P.lay.n_params);
    C.linbuf = take(P.n_lin);
    C.Glin = take(nnz);
    C.Clin = take(nnz);
    C.Aval = take(nnz);
    C.pool = take(B.pool);
    C.wpan = take((size_t)wpan_n);
    C.dinv = take(n);
    C.u = take(n);
    C.x = take(n);
    C.qx = take(n);
    C.u0 = take(n);
    C.up = take(n);
    C.qn = take(n);
    for (auto& h : C.H) h = take(n);
    for (auto& h : C.Q) h = take(n);
    C.st = take(std::max<int32_t>(P.n_stamp, 1));
    C.uvec = take(std::max<int32_t>(B.rel_ptr[B.ns], 1));
    C.part = take(2 * kRowBlocks + (size_t)C.hd.n_long + 16);
    C.lpart = take((size_t)C.hd.n_chunks + 16);
    C.norm = take(NRM_SLOTS);
    C.scal = take(4);
    C.sp = (StepDev*)take(sizeof(StepDev) / 8 + 1);
    BCHK(hipHostMalloc((void**)&C.h_norm, 8 * sizeof(double), hipHostMallocDefault));
    for (auto& e : C.ev) BCHK(hipEventCreate(&e));
    return CS_OK;
}

// One assembly-tree level of the factorization, in either form:
//   fused  one workgroup per front (gather, Jacobian entries, partial LU);
//   panel  gather tiles, Jacobian entries, LDS fronts, then per panel of the
//          large fronts: diagonal block, triangular solves, trailing update
//          spread over many workgroups.
// Both compute the same values in the same order (bit-identical fronts).
// pend: the level whose factored panels still wait in the workspace, or -1;
// with pend null the level's own are copied back at once.
void launch_flush(BigCircuit& C, hipStream_t s, int l) {
    auto& Lv = C.levels[l];
    MF_LAUNCH(CS_MFK_FLUSH, l, k_mf_flush, dim3(Lv.flush_n), dim3(kBT), 0, s, C.d_dev, C.pool, C.wpan, C.d_woff,
              C.d_flush + Lv.flush_b);
}
void launch_level(BigCircuit& C, hipStream_t s, int l, bool fused, int* pend = nullptr) {
    const BigDev* P = C.d_dev;
    auto& Lv = C.levels[l];
    const bool head = Lv.head_n > 0 && !fused;
    if (pend && *pend >= 0 && !(head && *pend == l - 1)) {
        launch_flush(C, s, *pend);
        *pend = -1;
    }
    if (head) {
        const int n_head = pend && *pend >= 0 ? Lv.head_nf : Lv.head_n;
        MF_LAUNCH(CS_MFK_HEAD, l, k_mf_head, dim3(n_head), dim3(kBT), Lv.head_lds, s, P, C.pool, C.dinv, C.Aval,
                  C.d_head + Lv.head_b, C.d_fronts, C.d_tiles, C.d_cbr, C.d_borig, C.wpan, C.d_woff, C.d_flush,
                  Lv.head_lds32);
        if (pend) *pend = -1;
        if (!Lv.big_n) return;
    } else {
        if (Lv.small_n[0])
            MF_LAUNCH(CS_MFK_SMALL32, l, (k_mf_lvl_small<8, 4>), dim3(Lv.small_n[0]), dim3(64), Lv.small_lds[0], s,
                      P, C.pool, C.dinv, C.Aval, C.d_fronts + Lv.small_b[0]);
        if (Lv.small_n[1])
            MF_LAUNCH(CS_MFK_SMALL64, l, k_mf_lvl_mid, dim3(Lv.small_n[1]), dim3(256), Lv.small_lds[1],
                      s, P, C.pool, C.dinv, C.Aval, C.d_fronts + Lv.small_b[1]);
        if (Lv.small_n[2])
            MF_LAUNCH(CS_MFK_SMALL96, l, k_mf_lvl_mid, dim3(Lv.small_n[2]), dim3(256), Lv.small_lds[2],
                      s, P, C.pool, C.dinv, C.Aval, C.d_fronts + Lv.small_b[2]);
        if (!Lv.big_n) return;
        if (fused) {
            MF_LAUNCH(CS_MFK_FRONT, l, k_mf_lvl_big, dim3(Lv.big_n), dim3(kBT), 0, s, P, C.pool, C.dinv, C.Aval,
                      C.d_fronts + Lv.big_b);
            return;
        }
        if (Lv.tile_n)
            MF_LAUNCH(CS_MFK_GATHER, l, k_mf_gather, dim3(Lv.tile_n), dim3(kBT), Lv.tile_lds, s, P, C.pool,
                      C.d_tiles + Lv.tile_b, C.d_cbr);
        if (Lv.orig_e > Lv.orig_b)
            MF_LAUNCH(CS_MFK_ORIG, l, k_mf_orig, dim3(grid_for(Lv.orig_e - Lv.orig_b)), dim3(kBT), 0, s, P, C.Aval,
                      C.pool, C.d_borig, Lv.orig_b, Lv.orig_e);
    }
    if (!C.split_panels) {
        for (auto& pn : Lv.panels) {
            if (C.mfma)
                MF_LAUNCH(CS_MFK_PANEL, l, k_mf_panel<true>, dim3(pn.pan_n), dim3(kBT), 0, s, P, C.pool, C.dinv,
                          C.wpan, C.d_woff, C.d_pan + pn.pan_b);
            else
                MF_LAUNCH(CS_MFK_PANEL, l, k_mf_panel<false>, dim3(pn.pan_n), dim3(kBT), 0, s, P, C.pool, C.dinv,
                          C.wpan, C.d_woff, C.d_pan + pn.pan_b);
        }
        if (pend) *pend = l;
        else launch_flush(C, s, l);
        return;
    }
    for (auto& pn : Lv.panels) {
        MF_LAUNCH(CS_MFK_DIAG, l, k_mf_diag, dim3(pn.diag_n), dim3(kDiagThreads), 0, s, P, C.pool, C.dinv,
                  C.d_diag + pn.diag_b);
        if (pn.trsm_n)
            MF_LAUNCH(CS_MFK_TRSM, l, k_mf_trsm, dim3(pn.trsm_n), dim3(kBT), 0, s, P, C.pool, C.dinv,
                      C.d_trsm + pn.trsm_b);
        if (pn.gemm_n) {
            if (C.mfma)
                MF_LAUNCH(CS_MFK_GEMM, l, k_mf_gemm_mfma, dim3(pn.gemm_n), dim3(kBT), 0, s, P, C.pool,
                          C.d_gemm + pn.gemm_b);
            else
                MF_LAUNCH(CS_MFK_GEMM, l, k_mf_gemm, dim3(pn.gemm_n), dim3(kBT), 0, s, P, C.pool,
                          C.d_gemm + pn.gemm_b);
        }
    }
}

void launch_factor(BigCircuit& C, hipStream_t s) {
    int pend = -1;
    for (int l = 0; l < (int)C.levels.size(); l++) launch_level(C, s, l, C.lvl_fused[l] != 0, &pend);
    if (pend >= 0) launch_flush(C, s, pend);
}

// The autotuner: for every level of this pattern, time both forms (the
// second of two runs each, on the current Jacobian values) and keep the
// faster.  The choice changes timing only, never the factors.
int tune_levels(BigCircuit& C, hipStream_t s, std::string& err) {
    const int nl = (int)C.levels.size();
    hipEvent_t ev[4];
    for (auto& e : ev) BCHK(hipEventCreate(&e));
    for (int l = 0; l < nl; l++) {
        if (!C.levels[l].big_n) {   // small fronts only: one form
            launch_level(C, s, l, false);
            C.tune_ms_panel.push_back(0.f);
            C.tune_ms_fused.push_back(0.f);
            continue;
        }
        // as launch_factor runs them: the factored panels go back in the next
        // level's head where it has one, and count here only where it has not
        const bool folds = l + 1 < nl && C.levels[l + 1].head_n > 0;
        for (int rep = 0; rep < 2; rep++) {   // the first one warms up
            int pend = -1;
            BCHK(hipEventRecord(ev[0], s));
            launch_level(C, s, l, false, folds ? &pend : nullptr);
            BCHK(hipEventRecord(ev[1], s));
            if (pend >= 0) launch_flush(C, s, pend);
            BCHK(hipEventRecord(ev[2], s));
            launch_level(C, s, l, true);
            BCHK(hipEventRecord(ev[3], s));
        }
        BCHK(hipEventSynchronize(ev[3]));
        float tp = 0.f, tf = 0.f;
        BCHK(hipEventElapsedTime(&tp, ev[0], ev[1]));
        BCHK(hipEventElapsedTime(&tf, ev[2], ev[3]));
        C.lvl_fused[l] = tf < tp ? 1 : 0;
        C.tune_ms_panel.push_back(tp);
        C.tune_ms_fused.push_back(tf);
    }
    for (auto& e : ev) (void)hipEventDestroy(e);
    BCHK(hipGetLastError());
    C.tuned = true;
    return CS_OK;
}

void launch_solve(BigCircuit& C, hipStream_t s) {
    const BigDev* P = C.d_dev;
    const int nl = (int)C.levels.size();
    for (int l = 0; l < nl; l++) {
        auto& Lv = C.levels[l];
        const int32_t* fr = C.d_fronts + Lv.fr_b;
        if (Lv.solve_bt == 512)
            MF_LAUNCH(CS_MFK_FWD, l, (k_mf_fwd<512>), dim3(Lv.fr_n), dim3(512), Lv.solve_lds, s, P, C.pool, C.x,
                      C.uvec, fr, Lv.ld_off);
        else if (Lv.solve_bt == 64)
            MF_LAUNCH(CS_MFK_FWD, l, (k_mf_fwd<64>), dim3(Lv.fr_n), dim3(64), Lv.solve_lds, s, P, C.pool, C.x,
                      C.uvec, fr, Lv.ld_off);
        else
            MF_LAUNCH(CS_MFK_FWD, l, (k_mf_fwd<kBT>), dim3(Lv.fr_n), dim3(kBT), Lv.solve_lds, s, P, C.pool, C.x,
                      C.uvec, fr, Lv.ld_off);
    }
    for (int l = nl - 1; l >= 0; l--) {
        auto& Lv = C.levels[l];
        const int32_t* fr = C.d_fronts + Lv.fr_b;
        if (Lv.solve_bt == 512)
            MF_LAUNCH(CS_MFK_BWD, l, (k_mf_bwd<512>), dim3(Lv.fr_n), dim3(512), Lv.solve_lds, s, P, C.pool, C.dinv,
                      C.x, fr, Lv.ld_off);
        else if (Lv.solve_bt == 64)
            MF_LAUNCH(CS_MFK_BWD, l, (k_mf_bwd<64>), dim3(Lv.fr_n), dim3(64), Lv.solve_lds, s, P, C.pool, C.dinv,
                      C.x, fr, Lv.ld_off);
        else
            MF_LAUNCH(CS_MFK_BWD, l, (k_mf_bwd<kBT>), dim3(Lv.fr_n), dim3(kBT), Lv.solve_lds, s, P, C.pool, C.dinv,
                      C.x, fr, Lv.ld_off);
    }
}

// Jacobian and residual: short rows one lane each, long rows one workgroup
// each; per-block residual maxima in part[0, gr + n_long)
int launch_assemble(BigCircuit& C, hipStream_t s, const double* qx, const double* pin, double* x, double* part) {
    const BigDev* P = C.d_dev;
    const int gr = grid_for(C.B.n);
    hipLaunchKernelGGL(k_assemble, dim3(gr), dim3(kBT), 0, s, P, C.Glin, C.Clin, C.sp, C.u, qx, C.st, pin,
                       C.Aval, x, part);
    if (C.hd.n_long) {
        hipLaunchKernelGGL(k_assemble_chunks, dim3(C.hd.n_chunks), dim3(kBT), 0, s, P, C.Glin, C.Clin, C.sp, C.u,
                           C.st, pin, C.Aval, C.lpart);
        hipLaunchKernelGGL(k_long_finish, dim3(C.hd.n_long), dim3(kBT), 0, s, P, C.sp, C.u, qx, pin, C.lpart,
                           C.Aval, x, part ? part + gr : nullptr);
    }
    return gr + C.hd.n_long;
}

void launch_charges(BigCircuit& C, hipStream_t s, const double* v, double* q) {
    hipLaunchKernelGGL(k_charges, dim3(grid_for(C.B.n)), dim3(kBT), 0, s, C.d_dev, C.Clin, v, q);
    if (C.hd.n_long) {
        hipLaunchKernelGGL(k_charges_chunks, dim3(C.hd.n_chunks), dim3(kBT), 0, s, C.d_dev, C.Clin, v, C.lpart);
        hipLaunchKernelGGL(k_charges_finish, dim3(C.hd.n_long), dim3(kBT), 0, s, C.d_dev, C.lpart, q);
    }
}

// One Newton iteration; with factor = false the solves reuse the factors in
// the pool from an earlier iteration (the assembly rewrites Aval, the
// matrix the factorization reads, but not the pool).
void launch_iteration(BigCircuit& C, hipStream_t s, bool factor = true) {
    const BigDev* P = C.d_dev;
    const int gr = grid_for(C.B.n);
    const int ge = grid_for(C.B.base.n_mos + C.B.base.n_src);
    hipLaunchKernelGGL(k_eval, dim3(ge), dim3(kBT), 0, s, P, C.p, C.u, C.sp, C.st);
    const int nb = launch_assemble(C, s, C.qx, C.u0, C.x, C.part);
    hipLaunchKernelGGL(k_res_reduce, dim3(1), dim3(kBT), 0, s, C.part, nb, C.norm);
    if (factor) launch_factor(C, s);
    launch_solve(C, s);
    hipLaunchKernelGGL(k_update, dim3(gr), dim3(kBT), 0, s, P, C.sp, C.x, C.u, C.norm, C.part);
    hipLaunchKernelGGL(k_upd_reduce, dim3(1), dim3(kBT), 0, s, P, C.sp, C.part, gr, C.norm);
    (void)hipMemcpyAsync(C.h_norm, C.norm, NRM_SLOTS * sizeof(double), hipMemcpyDeviceToHost, s);
}

int run_iter(BigCircuit& C, hipStream_t s, std::string& err, bool factor = true) {
    hipGraphExec_t g = factor ? C.exec : C.exec_nf;
    if (g) BCHK(hipGraphLaunch(g, s));
    else launch_iteration(C, s, factor);
    BCHK(hipStreamSynchronize(s));
    return CS_OK;
}

// The Newton iteration as one hipGraph (CEDAR_MF_GRAPH=0: plain stream
// launches, for A/B timing).
int ensure_graph(BigCircuit& C, hipStream_t s, std::string& err) {
    if (C.exec || !C.use_graph) return CS_OK;
    BCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    launch_iteration(C, s);
    BCHK(hipStreamEndCapture(s, &C.graph));
    BCHK(hipGraphInstantiate(&C.exec, C.graph, nullptr, nullptr, 0));
    BCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    launch_iteration(C, s, false);
    BCHK(hipStreamEndCapture(s, &C.graph_nf));
    BCHK(hipGraphInstantiate(&C.exec_nf, C.graph_nf, nullptr, nullptr, 0));
    return CS_OK;
}

int set_params(BigCircuit& C, hipStream_t s, const double* p, std::string& err) {
    const Plan& P = C.B.base;
    BCHK(hipMemcpyAsync(C.p, p, sizeof(double) * P.lay.n_params, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_lin_a, dim3(grid_for(P.n_lin)), dim3(kBT), 0, s, C.d_dev, C.p, C.linbuf);
    hipLaunchKernelGGL(k_lin_b, dim3(grid_for(P.nnz_nat)), dim3(kBT), 0, s, C.d_dev, C.linbuf, C.Glin, C.Clin);
    BCHK(hipGetLastError());
    return CS_OK;
}


int set_step(BigCircuit& C, hipStream_t s, const StepDev& sp, std::string& err) {
    BCHK(hipMemcpyAsync(C.sp, &sp, sizeof(StepDev), hipMemcpyHostToDevice, s));
    return CS_OK;
}

// Tune the factorization once per circuit, on a Jacobian assembled at the
// current state (the values only need to be finite).
int ensure_tuned(BigCircuit& C, hipStream_t s, double t, std::string& err) {
    if (C.tuned) return CS_OK;
    StepDev sp{};
    sp.t = t;
    sp.mode = CS_MODE_DCOP;
    sp.kind = STEP_DC;
    int rc = set_step(C, s, sp, err);
    if (rc) return rc;
    hipLaunchKernelGGL(k_eval, dim3(grid_for(C.B.base.n_mos + C.B.base.n_src)), dim3(kBT), 0, s, C.d_dev, C.p, C.u,
                       C.sp, C.st);
    launch_assemble(C, s, nullptr, nullptr, nullptr, nullptr);
    return tune_levels(C, s, err);
}

// Newton iterations from the state in C.u: CS_OK when max |F| <= tol,
// CS_E_NOCONV on a non-finite residual or after maxit iterations.
int newton_point(BigCircuit& C, hipStream_t s, int maxit, cs_tran_stats* st, std::string& err) {
    for (int it = 0; it < maxit; it++) {
        int rc = run_iter(C, s, err);
        if (rc) return rc;
        if (C.h_norm[NRM_DONE] == 1.0) return CS_OK;
        const double r = C.h_norm[NRM_RES];
        if (!(r == r) || std::isinf(r)) return CS_E_NOCONV;
        if (st) st->newton_iters++;
    }
    return CS_E_NOCONV;
}

// Initial point: UIC (charge rows pinned, 50 iterations) or the DC operating
// point by the trajectories and the gmin ladder of dcop_rules.h.
int init_point(BigCircuit& C, hipStream_t s, const double* u0, const cs_tran_opts& o, bool uic,
               cs_tran_stats* st, std::string& err) {
    const int32_t n = C.B.n;
    if (uic) {
        BCHK(hipMemcpyAsync(C.u, u0, sizeof(double) * n, hipMemcpyHostToDevice, s));
        BCHK(hipMemcpyAsync(C.u0, u0, sizeof(double) * n, hipMemcpyHostToDevice, s));
    }
    StepDev sp{};
    sp.a0 = 0.0; sp.t = o.t_start; sp.rtol = o.reltol; sp.atol = o.abstol; sp.tol = o.dc_abstol;
    sp.mode = uic ? CS_MODE_TRAN : CS_MODE_DCOP;
    sp.kind = uic ? STEP_UIC : STEP_DC;
    int rc = set_step(C, s, sp, err);
    if (rc) return rc;
    if (uic) return newton_point(C, s, 50, st, err);
    std::vector<double> us(n);
    auto start = [&](int j) -> int {
        for (int32_t i = 0; i < n; i++) us[i] = dc_start(j, i);
        BCHK(hipMemcpyAsync(C.u, us.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
        return CS_OK;
    };
    for (int j = 0; j < kDcTrajectories; j++) {
        if ((rc = start(j))) return rc;
        rc = newton_point(C, s, kDcMaxIt, st, err);
        if (rc != CS_E_NOCONV) return rc;
    }
    const int32_t pg = C.B.base.lay.gmin;
    double gc = 0.0;
    BCHK(hipMemcpy(&gc, C.p + pg, sizeof(double), hipMemcpyDeviceToHost));
    if ((rc = start(0))) return rc;
    for (int q = 0;; q++) {
        const double g = dc_gmin_stage(q, gc);
        if (g < 0.0) break;
        BCHK(hipMemcpyAsync(C.p + pg, &g, sizeof(double), hipMemcpyHostToDevice, s));
        rc = newton_point(C, s, kDcMaxIt, st, err);
        if (rc != CS_OK) break;
    }
    BCHK(hipMemcpyAsync(C.p + pg, &gc, sizeof(double), hipMemcpyHostToDevice, s));
    BCHK(hipStreamSynchronize(s));
    return rc;
}

// CedarDCOp after the DC point (its BrownFullBasicInit step, src/dcop.jl:153):
// the charge rows pinned to the DC point, the algebraic rows solved again
// with the sources at their transient values at t_start.
int reinit_at_t0(BigCircuit& C, hipStream_t s, const cs_tran_opts& o, cs_tran_stats* st, std::string& err) {
    BCHK(hipMemcpyAsync(C.u0, C.u, sizeof(double) * C.B.n, hipMemcpyDeviceToDevice, s));
    StepDev sp{};
    sp.a0 = 0.0; sp.t = o.t_start; sp.rtol = o.reltol; sp.atol = o.abstol; sp.tol = o.dc_abstol;
    sp.mode = CS_MODE_TRAN;
    sp.kind = STEP_UIC;
    int rc = set_step(C, s, sp, err);
    if (rc) return rc;
    return newton_point(C, s, 50, st, err);
}

}  // namespace

int big_create(const cs_netlist* nl, hipStream_t s, BigCircuit** out, std::string& err) {
    (void)s;
    auto* C = new BigCircuit();
    // trailing updates of the large fronts: FP64 matrix cores unless
    // CEDAR_MF_GEMM=valu asks for the vector-ALU kernel (A/B comparison)
    const char* g = std::getenv("CEDAR_MF_GEMM");
    C->mfma = !(g && std::strcmp(g, "valu") == 0);
    const char* sp = std::getenv("CEDAR_MF_PANEL");
    C->split_panels = sp && std::strcmp(sp, "split") == 0;
    const char* fm = std::getenv("CEDAR_MF_FRONT");
    const bool fix_fused = fm && std::strcmp(fm, "fused") == 0;
    const bool fix_panel = fm && std::strcmp(fm, "panel") == 0;
    const char* gg = std::getenv("CEDAR_MF_GRAPH");
    C->use_graph = !(gg && std::strcmp(gg, "0") == 0);
    int rc = build_bigplan(nl, C->B, err);
    if (rc == CS_OK) rc = upload(*C, err);
    if (rc == CS_OK) {
        C->lvl_fused.assign(C->levels.size(), fix_fused ? 1 : 0);
        C->tuned = fix_fused || fix_panel;
    }
    if (rc != CS_OK) {
        big_destroy(C);
        return rc;
    }
    *out = C;
    return CS_OK;
}

void big_destroy(BigCircuit* C) {
    if (!C) return;
    if (C->exec) (void)hipGraphExecDestroy(C->exec);
    if (C->graph) (void)hipGraphDestroy(C->graph);
    if (C->exec_nf) (void)hipGraphExecDestroy(C->exec_nf);
    if (C->graph_nf) (void)hipGraphDestroy(C->graph_nf);
    for (auto& e : C->ev)
        if (e) (void)hipEventDestroy(e);
    if (C->h_norm) (void)hipHostFree(C->h_norm);
    if (C->wbuf) (void)hipFree(C->wbuf);
    if (C->tbuf) (void)hipFree(C->tbuf);
    if (C->dbuf) (void)hipFree(C->dbuf);
    if (C->d_dev) (void)hipFree(C->d_dev);
    delete C;
}

const BigPlan& big_plan(const BigCircuit* C) { return C->B; }

void big_info(const BigPlan& B, cs_big_info* info) {
    info->n = B.n;
    info->n_super = B.ns;
    info->n_levels = (int32_t)B.lev_ptr.size() - 1;
    info->max_front = B.max_m;
    info->max_pivots = B.max_k;
    info->n_hub = B.n_hub;
    info->pool = B.pool;
    info->nnz_factor = B.nnz_factor;
    info->flops = B.flops;
}

int big_set_probes(BigCircuit* C, const std::vector<int32_t>& idx, std::string& err) {
    set_probes(C->B.base, idx);
    if (!idx.empty())
        BCHK(hipMemcpy(C->d_probe, idx.data(), sizeof(int32_t) * idx.size(), hipMemcpyHostToDevice));
    return CS_OK;
}

void big_last_times(const BigCircuit* C, double* f, double* s) {
    if (f) *f = C->factor_ms;
    if (s) *s = C->solve_ms;
}

int big_dcop(BigCircuit* C, hipStream_t s, const double* p, const cs_tran_opts* o, double* u_out,
             cs_tran_stats* st, std::string& err) {
    int rc;
    if ((rc = set_params(*C, s, p, err)) || (rc = ensure_tuned(*C, s, o->t_start, err)) ||
        (rc = ensure_graph(*C, s, err)))
        return rc;
    cs_tran_stats stt{};
    rc = init_point(*C, s, nullptr, *o, false, &stt, err);
    if (u_out) BCHK(hipMemcpy(u_out, C->u, sizeof(double) * C->B.n, hipMemcpyDeviceToHost));
    stt.retcode = rc;
    stt.t_end = o->t_start;
    if (st) *st = stt;
    if (rc == CS_E_NOCONV) err = "dc operating point did not converge";
    return rc;
}

// Transient with the step rules of rules.h; the history lives on the device
// and the host reads two scalars per Newton iteration and one per step.
int big_tran(BigCircuit* C, hipStream_t s, const double* p, const double* u0, const cs_tran_opts* o,
             double* wave, double* u_final, cs_tran_stats* st_out, std::string& err) {
    const BigPlan& B = C->B;
    const Plan& P = B.base;
    const int32_t n = B.n;
    const bool uic = o->init == CS_INIT_UIC;
    if (uic && !u0) { err = "UIC initialisation needs u0"; return CS_E_INVALID; }
    if (uic && !P.uic_ok) { err = "UIC: a charge-carrying row could not be kept on its own pivot"; return CS_E_INVALID; }
    if (o->n_out > 0 && !(o->dt_out > 0)) { err = "dt_out must be > 0"; return CS_E_INVALID; }
    int rc;
    if ((rc = set_params(*C, s, p, err)) || (rc = ensure_tuned(*C, s, o->t_start, err)) ||
        (rc = ensure_graph(*C, s, err)))
        return rc;
    cs_tran_stats st{};
    rc = init_point(*C, s, u0, *o, uic, &st, err);
    if (rc == CS_OK && !uic) rc = reinit_at_t0(*C, s, *o, &st, err);
    const int gr = grid_for(n);
    const int n_probe = (int)P.probe.size();
    double* d_wave = nullptr;
    if (wave && o->n_out > 0) BCHK(hipMalloc(&d_wave, sizeof(double) * (size_t)o->n_out * n_probe));
    const StepDefaults sd = step_defaults(*o);
    double t = o->t_start;
    int kout = 0;
    if (rc == CS_OK) {
        BCHK(hipMemcpyAsync(C->H[0], C->u, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        launch_charges(*C, s, C->u, C->Q[0]);
        double T0 = o->t_start, T1 = 0.0, T2 = 0.0;
        int npts = 1;
        double h = sd.dt_init;
        if (d_wave)
            while (kout < o->n_out && o->t_start + kout * o->dt_out <= o->t_start + 1e-9 * o->dt_out) {
                hipLaunchKernelGGL(k_wave, dim3(grid_for(n_probe)), dim3(kBT), 0, s, n_probe, C->d_probe, C->H[0],
                                   C->H[0], C->H[0], 1.0, 0.0, 0.0, d_wave + (size_t)kout * n_probe);
                kout++;
            }
        std::vector<double> ph(p, p + P.lay.n_params);
        StepDev sp{};
        sp.rtol = o->reltol; sp.atol = o->abstol; sp.tol = o->dc_abstol;
        sp.mode = CS_MODE_TRAN; sp.kind = STEP_TRAN;
        while (t < o->t_stop) {
            if (st.steps + st.rejected >= o->max_steps) { rc = CS_E_MAXSTEPS; break; }
            double tb = INFINITY;
            for (auto& sdsc : P.src) {
                const double bp = wave_next_bp(sdsc.kind, ph.data() + sdsc.off, sdsc.len, t);
                if (bp < tb) tb = bp;
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
            hipLaunchKernelGGL(k_predict, dim3(gr), dim3(kBT), 0, s, n, np, k, w0, w1, w2, a1, a2, C->H[0],
                               C->H[1], C->H[2], C->Q[0], C->Q[1], C->up, C->u, C->qx);
            sp.a0 = a0;
            sp.t = tn;
            if ((rc = set_step(*C, s, sp, err))) break;
            bool conv = false;
            for (int it = 0; it < o->newton_maxit; it++) {
                // modified Newton: the step's first factors for its later iterations
                if ((rc = run_iter(*C, s, err, it == 0 || !o->jac_reuse))) break;
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
            launch_charges(*C, s, C->u, C->qn);
            double fac = 2.0;
            if (npts >= 2) {
                const double c = lte_coeff(k, tn, T0, T1, T2, a0, a1, a2);
                hipLaunchKernelGGL(k_lte, dim3(gr), dim3(kBT), 0, s, n, c, o->reltol, o->abstol, C->u, C->up,
                                   C->H[0], C->part);
                hipLaunchKernelGGL(k_sum_reduce, dim3(1), dim3(kBT), 0, s, C->part, gr, C->scal);
                BCHK(hipMemcpyAsync(C->h_norm + 4, C->scal, sizeof(double), hipMemcpyDeviceToHost, s));
                BCHK(hipStreamSynchronize(s));
                const double err_ = std::sqrt(C->h_norm[4] / n);
                if (!(err_ <= 1.0)) {
                    st.rejected++;
                    h = hh * reject_factor(err_, k);
                    if (h < sd.dt_min) { rc = CS_E_DTMIN; break; }
                    continue;
                }
                fac = accept_factor(err_, k);
            }
            // accept: rotate the history buffers, u becomes the newest point
            std::swap(C->H[2], C->H[1]);
            std::swap(C->H[1], C->H[0]);
            BCHK(hipMemcpyAsync(C->H[0], C->u, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
            std::swap(C->Q[1], C->Q[0]);
            std::swap(C->Q[0], C->qn);
            T2 = T1; T1 = T0; T0 = tn;
            if (npts < 3) npts++;
            st.steps++;
            if (d_wave) {
                while (kout < o->n_out) {
                    const double tq = o->t_start + kout * o->dt_out;
                    if (tq > tn + 1e-9 * o->dt_out) break;
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
                    hipLaunchKernelGGL(k_wave, dim3(grid_for(n_probe)), dim3(kBT), 0, s, n_probe, C->d_probe,
                                       C->H[0], C->H[1], C->H[2], l0, l1, l2, d_wave + (size_t)kout * n_probe);
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
    if (d_wave) {
        (void)hipStreamSynchronize(s);
        (void)hipMemcpy(wave, d_wave, sizeof(double) * (size_t)kout * n_probe, hipMemcpyDeviceToHost);
        (void)hipFree(d_wave);
    }
    if (u_final) {
        (void)hipStreamSynchronize(s);
        (void)hipMemcpy(u_final, st.steps > 0 ? C->H[0] : C->u, sizeof(double) * n, hipMemcpyDeviceToHost);
    }
    if (st_out) *st_out = st;
    if (rc == CS_E_DTMIN) err = "transient: step size fell below dt_min";
    else if (rc == CS_E_NOCONV) err = "transient: initial point did not converge";
    else if (rc == CS_E_MAXSTEPS) err = "transient: max_steps reached";
    return rc;
}

// ---- DAE interface ------------------------------------------------------------------------------
int big_residual(BigCircuit* C, hipStream_t s, double* out, const double* du, const double* u,
                 const double* p, double t, int32_t mode, std::string& err) {
    const int32_t n = C->B.n;
    int rc;
    if ((rc = set_params(*C, s, p, err))) return rc;
    BCHK(hipMemcpyAsync(C->u, u, sizeof(double) * n, hipMemcpyHostToDevice, s));
    StepDev sp{};
    sp.a0 = 0.0; sp.t = t; sp.mode = mode;
    sp.kind = mode == CS_MODE_DCOP ? STEP_DC : STEP_TRAN;
    if (mode != CS_MODE_DCOP) {
        // the charge term d/dt q(u) = C du enters as qx with a0 = 0
        if (du) BCHK(hipMemcpyAsync(C->up, du, sizeof(double) * n, hipMemcpyHostToDevice, s));
        else BCHK(hipMemsetAsync(C->up, 0, sizeof(double) * n, s));
        launch_charges(*C, s, C->up, C->qx);
    }
    if ((rc = set_step(*C, s, sp, err))) return rc;
    hipLaunchKernelGGL(k_eval, dim3(grid_for(C->B.base.n_mos + C->B.base.n_src)), dim3(kBT), 0, s, C->d_dev, C->p,
                       C->u, C->sp, C->st);
    launch_assemble(*C, s, C->qx, nullptr, C->x, C->part);
    // x[prow[r]] = -F(r)
    hipLaunchKernelGGL(k_perm_out, dim3(grid_for(n)), dim3(kBT), 0, s, n, C->hd.prow, C->x, C->up);
    std::vector<double> h(n);
    BCHK(hipMemcpyAsync(h.data(), C->up, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    BCHK(hipStreamSynchronize(s));
    for (int32_t i = 0; i < n; i++) out[i] = -h[i];
    return CS_OK;
}

int big_jacobian(BigCircuit* C, hipStream_t s, double* vals, const double* du, const double* u,
                 const double* p, double gamma, double t, int32_t mode, std::string& err) {
    (void)du;
    const int32_t n = C->B.n;
    int rc;
    if ((rc = set_params(*C, s, p, err))) return rc;
    BCHK(hipMemcpyAsync(C->u, u, sizeof(double) * n, hipMemcpyHostToDevice, s));
    StepDev sp{};
    sp.a0 = gamma; sp.t = t; sp.mode = mode;
    sp.kind = mode == CS_MODE_DCOP ? STEP_DC : STEP_TRAN;
    if ((rc = set_step(*C, s, sp, err))) return rc;
    hipLaunchKernelGGL(k_eval, dim3(grid_for(C->B.base.n_mos + C->B.base.n_src)), dim3(kBT), 0, s, C->d_dev, C->p,
                       C->u, C->sp, C->st);
    launch_assemble(*C, s, nullptr, nullptr, nullptr, nullptr);
    BCHK(hipMemcpyAsync(vals, C->Aval, sizeof(double) * C->B.base.nnz_nat, hipMemcpyDeviceToHost, s));
    BCHK(hipStreamSynchronize(s));
    return CS_OK;
}

int big_lu_refactor(BigCircuit* C, hipStream_t s, const double* vals, std::string& err) {
    BCHK(hipMemcpyAsync(C->Aval, vals, sizeof(double) * C->B.base.nnz_nat, hipMemcpyHostToDevice, s));
    if (!C->tuned) {
        int rc = tune_levels(*C, s, err);
        if (rc) return rc;
    }
    BCHK(hipEventRecord(C->ev[0], s));
    launch_factor(*C, s);
    BCHK(hipEventRecord(C->ev[1], s));
    BCHK(hipGetLastError());
    BCHK(hipEventSynchronize(C->ev[1]));
    float ms = 0.f;
    BCHK(hipEventElapsedTime(&ms, C->ev[0], C->ev[1]));
    C->factor_ms = ms;
    std::vector<double> d(C->B.n);
    BCHK(hipMemcpy(d.data(), C->dinv, sizeof(double) * C->B.n, hipMemcpyDeviceToHost));
    for (int32_t k = 0; k < C->B.n; k++)
        if (!std::isfinite(d[k])) {
            err = "zero pivot at step " + std::to_string(k);
            return CS_E_SINGULAR;
        }
    return CS_OK;
}

int big_lu_solve(BigCircuit* C, hipStream_t s, double* x, std::string& err) {
    const int32_t n = C->B.n;
    BCHK(hipMemcpyAsync(C->up, x, sizeof(double) * n, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_perm_in, dim3(grid_for(n)), dim3(kBT), 0, s, n, C->hd.prow, C->up, C->x);
    BCHK(hipEventRecord(C->ev[2], s));
    launch_solve(*C, s);
    BCHK(hipEventRecord(C->ev[3], s));
    hipLaunchKernelGGL(k_perm_out, dim3(grid_for(n)), dim3(kBT), 0, s, n, C->hd.pcol, C->x, C->up);
    BCHK(hipMemcpyAsync(x, C->up, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    BCHK(hipStreamSynchronize(s));
    BCHK(hipGetLastError());
    float ms = 0.f;
    BCHK(hipEventElapsedTime(&ms, C->ev[2], C->ev[3]));
    C->solve_ms = ms;
    return CS_OK;
}

int big_profile(BigCircuit* C, hipStream_t s, int32_t* kinds, int32_t* levels, float* ms, int32_t cap,
                int32_t* count, std::string& err) {
    if (!C->tuned) {
        int rc = tune_levels(*C, s, err);
        if (rc) return rc;
    }
    BigCircuit::LaunchProf P;
    C->prof = &P;
    launch_factor(*C, s);
    launch_solve(*C, s);
    C->prof = nullptr;
    hipError_t e = hipStreamSynchronize(s);
    const int nlaunch = (int)P.kind.size();
    int rc = CS_OK;
    if (e != hipSuccess || (int)P.ev.size() != 2 * nlaunch) {
        err = e != hipSuccess ? std::string("hipStreamSynchronize: ") + hipGetErrorString(e)
                              : std::string("event creation failed");
        rc = CS_E_HIP;
    }
    for (int q = 0; rc == CS_OK && q < nlaunch; q++) {
        float t = 0.f;
        if (hipEventElapsedTime(&t, P.ev[2 * q], P.ev[2 * q + 1]) != hipSuccess) {
            err = "hipEventElapsedTime failed";
            rc = CS_E_HIP;
            break;
        }
        if (q < cap) {
            if (kinds) kinds[q] = P.kind[q];
            if (levels) levels[q] = P.level[q];
            if (ms) ms[q] = t;
        }
    }
    for (auto ev : P.ev) (void)hipEventDestroy(ev);
    if (count) *count = nlaunch;
    return rc;
}

}  // namespace cedar
