// lds_core.h — building blocks of the LDS-resident batched kernels
// (tran_lds.hip: transient; adj_lds.hip: adjoint).
//
// One 64-lane wavefront owns one circuit instance.  The circuit's 16-bit
// plan image (compact.h) and the instance's numbers live in LDS; a Newton
// iteration touches only LDS and registers:
//
//   eval      lane m evaluates MOSFETs m, m+64, ...: terminals (offsets of
//             u), beta = kp*W/L and type*Vth stay in registers;
//             (id, dI/dVd, dI/dVg) go to the stamp buffer;
//   assemble  one lane per matrix entry: F from fixed records (no atomics,
//             fixed summation order); one lane per pivot row: -residual -> x;
//   steps     the solve program: LU with the forward substitution folded in,
//             then the backward substitution, up to 64 records at a time;
//   update    u[k] += x[k] (pivot order: no permutation), WRMS norm by a
//             cross-lane reduction.
//
// What bounds it: one iteration is a chain of about 30 dependent LDS round
// trips of one wavefront (a read 60 cycles, a read after a write 113, a taken
// branch about 28), so it is latency-bound until 16 wavefronts share a CU;
// then the LDS pipe is (87 % busy on the 4096-ring batch).  Hence records
// whose operands are direct byte offsets (two reads deep where row
// descriptors, pointers and index pairs took five), the next step's record
// requested before the current step computes, and few register spills: with
// the plan header's 44 words in scalar registers the packed kernel spilled
// 233 scalar and 146 vector registers (now 147 and 0), and reloaded them
// inside the iteration.  Instructions per iteration, averaged over that
// batch, before and after: vector 1895 -> 1093, scalar 1087 -> 531, LDS 359 ->
// 218.
//
// Step control, predictor, local-error test and output interpolation follow
// rules.h as the global-plan kernel (tran_device.h) does; history (u and
// charges of the last three accepted points) lives in the registers of the
// lane that owns the row/column.
#pragma once
#include "compact.h"
#include "dcop_rules.h"
#include "device.h"
#include "kernels.h"
#include "wave_math.h"

// Multiplications and additions are fused only where the source says fma: the
// adjoint's reverse kernel must repeat the forward kernel's bits, and the
// compiler's own choice may differ from kernel to kernel.
#pragma clang fp contract(off)

namespace cedar {
namespace lds {

constexpr int W = 64;

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (W - 1)); }

// 1/a: the hardware estimate and two Newton corrections (error below one
// ulp), which an infinite or zero a turns into NaN; the fix-up instruction of
// the division gives 0 or an infinity there.  It lies on the chain of every
// pivot, so it is one instruction: a select on the result or on the first
// residual cost a 33-stage ring's transient 1.4 and 1.9 %, this 0.4.
__device__ __forceinline__ double recip(double a) {
    double r = __builtin_amdgcn_rcp(a);
    double e = __builtin_fma(-a, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-a, r, 1.0);
    r = __builtin_fma(r, e, r);
    return __builtin_amdgcn_div_fixup(r, a, 1.0);
}

// a / b for step control: the quotient by recip, corrected once by its
// residual (which is not defined for an infinite a or quotient).
__device__ __forceinline__ double quot(double a, double b) {
    const double r = recip(b), q = a * r;
    const double e = __builtin_fma(-q, b, a);
    return e == e ? __builtin_fma(e, r, q) : q;
}

// Value of lane src (uniform) for the whole wavefront.
__device__ __forceinline__ double bcast(double v, int src) { return readlane_f64(v, src); }

// A value that every lane holds, moved to scalar registers: the step control's
// numbers live across the Newton iterations, and as vector registers they
// would be two each in every lane.
__device__ __forceinline__ double uniform(double v) { return readlane_f64(v, 0); }

// Sum over the wavefront in a fixed order (wave_reduce): every lane ends
// with the same value, the same on every run.
__device__ __forceinline__ double wave_sum(double v) { return wave_reduce(v, OpSum()); }
// two of them, their steps interleaved
__device__ __forceinline__ void wave_sum2(double& a, double& b) {
    a += dpp_f64<0xB1>(a);   b += dpp_f64<0xB1>(b);
    a += dpp_f64<0x4E>(a);   b += dpp_f64<0x4E>(b);
    a += dpp_f64<0x141>(a);  b += dpp_f64<0x141>(b);
    a += dpp_f64<0x140>(a);  b += dpp_f64<0x140>(b);
    a = (readlane_f64(a, 0) + readlane_f64(a, 16)) + (readlane_f64(a, 32) + readlane_f64(a, 48));
    b = (readlane_f64(b, 0) + readlane_f64(b, 16)) + (readlane_f64(b, 32) + readlane_f64(b, 48));
}

// Synchronisation of the instance's own wavefront.  An instance is owned by
// one wavefront, so its phases need only wavefront-scope ordering of LDS
// accesses (other wavefronts of the workgroup own other instances): a fence
// that keeps the compiler from moving memory accesses across, and the
// wavefront barrier.  The LDS serves one wavefront's accesses in order.
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int K>
struct Count { static constexpr int value = K; };

// Row of slot r of lane tid: lanes past the last row hold a copy of it.
__device__ __forceinline__ int row_of(int tid, int r, int n) { return tid + W * r < n ? tid + W * r : n - 1; }

// Per-lane MOSFET constants of NM device slots.
template <int NM>
struct DevRegs {
    double beta[NM], tpvth[NM];
    uint32_t dg[NM], sx[NM];   // byte offsets of u: d | g << 16;  s | (type < 0) << 31
};

// The instance's region and the circuit's image.
struct View {
    char* R;
    const uint16_t* B;
    __device__ __forceinline__ double& at(uint32_t off) const { return *reinterpret_cast<double*>(R + off); }
    // stamp reference: the sign goes straight into the sign bit
    __device__ __forceinline__ double ref(uint32_t r) const {
        const double v = at(r & 0xFFF8u);
        return __longlong_as_double(__double_as_longlong(v) ^ ((long long)r << 63));
    }
    __device__ __forceinline__ double2 gc(uint32_t l16) const { return *reinterpret_cast<const double2*>(R + l16); }
};

// Uniform tables (the plan headers, the launch's arguments and options) are
// read through the scalar cache where they are used.  fresh() makes the
// compiler forget what it read through a pointer, so that a phase's fields
// occupy scalar registers only within the phase: carried across the whole
// transient they exceed the 102 there are.
template <class T>
using ConstPtr = const __attribute__((address_space(4))) T*;
template <class T>
__device__ __forceinline__ ConstPtr<T> as_const(const T* p) {
    return (ConstPtr<T>)p;
}
template <class T>
__device__ __forceinline__ ConstPtr<T> fresh(ConstPtr<T> p) {
    asm volatile("" : "+s"(p));
    return p;
}
// The same for a lane's own values: what is derived from them (addresses,
// lane masks) is recomputed where it is used instead of being kept.
__device__ __forceinline__ int fresh_lane(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
typedef ConstPtr<CPlan> Hdr;

// What one Newton iteration reads of the plan header, loaded together at the
// start of a step's iterations.
struct Hot {
    int n, nm, ns, b_x, b_u, b_st;
    int o_ea, n_ea, o_eb, n_eb, o_ec, n_ec, o_ed, n_ed, o_ez, n_ez;
    int o_rr, o_lcol, o_items, n_items, o_refs, wide, wide_ed, b_trash;
    int o_steps, n_lu, n_steps, o_rec, o_upd;
    const double* mos_m;
};
__device__ __forceinline__ Hot load_hot(Hdr c) {
    c = fresh(c);
    Hot h;
    h.n = c->n; h.nm = c->n_mos; h.ns = c->n_src; h.b_x = c->b_x; h.b_u = c->b_u; h.b_st = c->b_st;
    h.o_ea = c->o_ea; h.n_ea = c->n_ea; h.o_eb = c->o_eb; h.n_eb = c->n_eb; h.o_ec = c->o_ec; h.n_ec = c->n_ec;
    h.o_ed = c->o_ed; h.n_ed = c->n_ed; h.o_ez = c->o_ez; h.n_ez = c->n_ez;
    h.o_rr = c->o_rr; h.o_lcol = c->o_lcol; h.o_items = c->o_items; h.n_items = c->n_items; h.o_refs = c->o_refs;
    h.wide = c->wide_rows; h.wide_ed = c->wide_ed; h.b_trash = c->b_trash;
    h.o_steps = c->o_steps; h.n_lu = c->n_lu; h.n_steps = c->n_steps; h.o_rec = c->o_rec; h.o_upd = c->o_upd;
    h.mos_m = c->mos_m;
    return h;
}

// Copy the first `words` uint16 of a plan image (a multiple of 8, the image
// 16-byte aligned in both places) with threads t0, t0 + nt, ...  The caller
// synchronises.
__device__ __forceinline__ void copy_image(const uint16_t* image, int words, uint16_t* blob, int t0, int nt) {
    const uint4* src = reinterpret_cast<const uint4*>(image);
    uint4* dst = reinterpret_cast<uint4*>(blob);
#pragma nounroll
    for (int q = t0; q < words / 8; q += nt) dst[q] = src[q];
}

// Square-law MOSFET stamps (sqlaw_core of rules.h without branches: in
// saturation vx is vov, in cutoff vov is 0).
__device__ __forceinline__ void mos_eval(bool pmos, double beta, double tpvth, double gmin, double vd, double vg,
                                         double vs, double& id, double& dd, double& dg) {
    const double vdif = vd - vs;
    const double vds = pmos ? -vdif : vdif;
    const bool fwd = vds >= 0.0;
    const double vgx = vg - (fwd ? vs : vd);
    const double vo = (pmos ? -vgx : vgx) - tpvth;
    const double vov = vo > 0.0 ? vo : 0.0;
    const double va = fabs(vds);
    const double vx = va < vov ? va : vov;
    const double cur = beta * (__builtin_fma(-0.5, vx, vov) * vx);
    const double gm = beta * vx, gds = beta * (vov - vx);
    id = __builtin_fma(gmin, vdif, (pmos == fwd) ? -cur : cur);
    dd = (fwd ? gds : gm + gds) + gmin;
    dg = fwd ? gm : -gm;
}

// ILP: device slots in pairs, so that two evaluations are in flight
// together; lanes past the last device hold a copy of it and store the same
// stamps.
template <int NM, bool ILP>
__device__ __forceinline__ void eval_mos(const Hot& h, const View& v, const DevRegs<NM>& dr, double gmin) {
    const int nm = h.nm, st = h.b_st;
    if constexpr (!ILP) {
#pragma unroll
        for (int j = 0; j < NM; j++) {
            const int m = fresh_lane(lane_id()) + W * j;
            if (m < nm) {
                double id, dd, dg;
                const uint32_t t = (uint32_t)fresh_lane((int)dr.dg[j]), u = (uint32_t)fresh_lane((int)dr.sx[j]);
                mos_eval((int32_t)u < 0, dr.beta[j], dr.tpvth[j], gmin, v.at(t & 0xFFFF), v.at(t >> 16),
                         v.at(u & 0xFFFF), id, dd, dg);
                if (h.mos_m) {
                    const double mm = h.mos_m[m];
                    id *= mm; dd *= mm; dg *= mm;
                }
                v.at(st + 8 * m) = id;
                v.at(st + 8 * (nm + m)) = dd;
                v.at(st + 8 * (2 * nm + m)) = dg;
            }
        }
        return;
    }
    auto slots = [&](auto count, int j0) {
        constexpr int K = decltype(count)::value;
        double id[K], dd[K], dg[K];
#pragma unroll
        for (int i = 0; i < K; i++) {
            const uint32_t t = (uint32_t)fresh_lane((int)dr.dg[j0 + i]), u = (uint32_t)fresh_lane((int)dr.sx[j0 + i]);
            mos_eval((int32_t)u < 0, dr.beta[j0 + i], dr.tpvth[j0 + i], gmin, v.at(t & 0xFFFF), v.at(t >> 16),
                     v.at(u & 0xFFFF), id[i], dd[i], dg[i]);
        }
        const int tid = fresh_lane(lane_id());
#pragma unroll
        for (int i = 0; i < K; i++) {
            const int m = tid + W * (j0 + i) < nm ? tid + W * (j0 + i) : nm - 1;
            if (h.mos_m) {   // uniform: only circuits with m-factors read them
                const double mm = h.mos_m[m];
                id[i] *= mm; dd[i] *= mm; dg[i] *= mm;
            }
            v.at(st + 8 * m) = id[i];
            v.at(st + 8 * (nm + m)) = dd[i];
            v.at(st + 8 * (2 * nm + m)) = dg[i];
        }
    };
#pragma unroll
    for (int j0 = 0; j0 < NM; j0 += 2) {
        if (W * j0 >= nm) break;   // uniform
        if (W * (j0 + 1) < nm) slots(Count<2>(), j0);
        else slots(Count<1>(), j0);
    }
}

// DYN = false: every source of the circuit is a DC one; the waveform code is
// left out, and with it the registers it holds across the transient.
template <bool DYN>
__device__ __forceinline__ void eval_sources(Hdr c, const View& v, double t, int mode) {
    c = fresh(c);
    const int ns = c->n_src;
#pragma nounroll
    for (int s = lane_id(); s < ns; s += W) {
        const uint16_t* d = v.B + c->o_src + 4 * s;
        const double* wd = &v.at(d[1]);
        double val;
        if constexpr (DYN) {
            val = source_at(d[0], wd, d[2], wd[d[2]], t, mode);
        } else {
            const double dc = wd[d[2]];
            val = mode == CS_MODE_DCOP && dc == dc ? dc : wd[0];
        }
        v.at(d[3]) = c->src_m ? val * c->src_m[s] : val;
    }
}

// Partial sums of one wavefront item: references and linear entries by
// lane, the row's charge term by its owner lane.
template <int NR>
__device__ __forceinline__ double item_part(const Hot& h, const View& v, double a0, const double (&qx)[NR], uint4 p) {
    const int tid = fresh_lane(lane_id());
    const uint16_t* refs = v.B + h.o_refs;
    const int q1 = p.y & 0xFFFF, l1 = p.z & 0xFFFF, k = p.z >> 16;
    const bool row = (p.w & 0xFFFF) != 0;
    double s = 0.0;
#pragma nounroll
    for (int q = (int)(p.x >> 16) + tid; q < q1; q += 2 * W) {
        const int q2 = q + W;
        const double s0 = v.ref(refs[q]), s1 = v.ref(refs[q2 < q1 ? q2 : q]);
        s += q2 < q1 ? s0 + s1 : s0;
    }
#pragma nounroll
    for (int l = (int)(p.y >> 16) + tid; l < l1; l += W) {
        const double2 g = v.gc(16 * l);
        const double j = __builtin_fma(a0, g.y, g.x);
        s = row ? __builtin_fma(j, v.at((v.B + h.o_lcol)[l]), s) : s + j;
    }
    if (row) {
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (k == tid + W * r) s += qx[r];
    }
    return s;
}

// F = G + a0*C + nonlinear stamps (and the inverse of the diagonals the
// factorization does not update); x = -residual, qx added per row.
// The records of a class's first rounds and of the rows are read together,
// then their operands, then everything is stored: two LDS latencies where a
// loop per class took two each.  Lanes past a class's end read its last
// record and store the same value to the same place, which costs the LDS
// latency nothing (measured), where masking them off costs two branches a
// store.  ILP = false is the form for a CU full of wavefronts, where the LDS
// pipe bounds instead (87 % busy on the 4096-ring batch) and every lane
// masked off saves its cycles: one record at a time, lanes past the end off.  Entries with many references and the residuals of long rows (the
// supply node: one reference per device on it) are summed by the whole
// wavefront, two sums at a time, in a fixed order, so that runs are
// bit-identical.
template <int NR, bool ILP>
__device__ __forceinline__ void assemble(const Hot& h, const View& v, double a0, const double (&qx)[NR]) {
    constexpr int EA = ILP ? 2 * NR : 0, ED = ILP ? NR : 0, EB = ILP ? 1 : 0;
    const uint16_t* B = v.B;
    const int tid = fresh_lane(lane_id());
    const uint2* ra = reinterpret_cast<const uint2*>(B + h.o_ea);
    const uint2* rb = reinterpret_cast<const uint2*>(B + h.o_eb);
    const uint4* rd = reinterpret_cast<const uint4*>(B + h.o_ed);
    const uint4* rr = reinterpret_cast<const uint4*>(B + h.o_rr);
    auto last = [&](int i, int n) { return i < n ? i : n - 1; };
    // -residual of the row of record p, without the sums of a long row
    auto row = [&](const uint4& p, double q) {
        const double2 g = v.gc(16 * (p.x & 0xFFFF));
        double f = __builtin_fma(__builtin_fma(a0, g.y, g.x), v.at(p.y & 0xFFFF),
                                 q + (v.ref(p.y >> 16) + v.ref(p.z & 0xFFFF)));
        if (h.wide) {
            f += v.ref(p.z >> 16) + (v.ref(p.w & 0xFFFF) + v.ref(p.w >> 16));
            const uint32_t nl = p.x >> 16;
            if (nl != 0xFFFF) {
#pragma nounroll
                for (uint32_t l = (p.x & 0xFFFF) + 1, le = l + nl; l + 1 < le; l++) {
                    const double2 g = v.gc(16 * l);
                    f = __builtin_fma(__builtin_fma(a0, g.y, g.x), v.at((B + h.o_lcol)[l]), f);
                }
            }
        }
        return -f;
    };
    if constexpr (ILP) {
        uint2 pa[EA];
        uint4 pd[ED], pr[NR];
#pragma unroll
        for (int r = 0; r < EA; r++) pa[r] = ra[last(tid + W * r, h.n_ea)];
#pragma unroll
        for (int r = 0; r < ED; r++) pd[r] = rd[last(tid + W * r, h.n_ed)];
        const uint2 pb = rb[last(tid, h.n_eb)];
#pragma unroll
        for (int r = 0; r < NR; r++) pr[r] = rr[last(tid + W * r, h.n)];
        double fa[EA], fd[ED], id[ED], fx[NR], fb;
#pragma unroll
        for (int r = 0; r < EA; r++) fa[r] = v.ref(pa[r].x >> 16) + v.ref(pa[r].y & 0xFFFF);
#pragma unroll
        for (int r = 0; r < ED; r++) {
            const double2 g = v.gc(pd[r].x >> 16);
            fd[r] = __builtin_fma(a0, g.y, g.x) + (v.ref(pd[r].y & 0xFFFF) + v.ref(pd[r].y >> 16));
        }
        if (h.wide_ed) {
#pragma unroll
            for (int r = 0; r < ED; r++) fd[r] += v.ref(pd[r].z >> 16) + v.ref(pd[r].w & 0xFFFF);
        }
        {
            const double2 g = v.gc(pb.x >> 16);
            fb = __builtin_fma(a0, g.y, g.x) + (v.ref(pb.y & 0xFFFF) + v.ref(pb.y >> 16));
        }
#pragma unroll
        for (int r = 0; r < NR; r++) fx[r] = row(pr[r], qx[r]);
#pragma unroll
        for (int r = 0; r < ED; r++) id[r] = recip(fd[r]);
        const int lane = fresh_lane(tid);
#pragma unroll
        for (int r = 0; r < EA; r++)
            v.at(pa[r].x & 0xFFFF) = fa[r];
#pragma unroll
        for (int r = 0; r < ED; r++)
        {
            v.at(pd[r].x & 0xFFFF) = fd[r];
            v.at(pd[r].z & 0xFFFF) = id[r];
        }
        v.at(pb.x & 0xFFFF) = fb;
#pragma unroll
        for (int r = 0; r < NR; r++)
            v.at((pr[r].x >> 16) != 0xFFFF ? h.b_x + 8 * last(lane + W * r, h.n) : h.b_trash) = fx[r];
    } else {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k = tid + W * r;
            if (k < h.n) {
                const uint4 p = rr[k];
                const double f = row(p, qx[r]);
                if ((p.x >> 16) != 0xFFFF) v.at(h.b_x + 8 * k) = f;
            }
        }
    }
    // the entries left
#pragma nounroll
    for (int i = tid + W * EA; i < h.n_ea; i += 2 * W) {
        const uint2 p = ra[i], q = ra[i + W < h.n_ea ? i + W : i];
        const double p0 = v.ref(p.x >> 16) + v.ref(p.y & 0xFFFF), q0 = v.ref(q.x >> 16) + v.ref(q.y & 0xFFFF);
        v.at(p.x & 0xFFFF) = p0;
        v.at(q.x & 0xFFFF) = q0;
    }
#pragma nounroll
    for (int i = tid + W * ED; i < h.n_ed; i += W) {
        const uint4 p = rd[i];
        const double2 g = v.gc(p.x >> 16);
        double s = __builtin_fma(a0, g.y, g.x) + (v.ref(p.y & 0xFFFF) + v.ref(p.y >> 16));
        if (h.wide_ed) s += v.ref(p.z >> 16) + v.ref(p.w & 0xFFFF);
        v.at(p.x & 0xFFFF) = s;
        v.at(p.z & 0xFFFF) = recip(s);
    }
#pragma nounroll
    for (int i = tid + W * EB; i < h.n_eb; i += W) {
        const uint2 p = rb[i];
        const double2 g = v.gc(p.x >> 16);
        v.at(p.x & 0xFFFF) = __builtin_fma(a0, g.y, g.x) + (v.ref(p.y & 0xFFFF) + v.ref(p.y >> 16));
    }
#pragma nounroll
    for (int i = tid; i < h.n_ec; i += W) {
        const uint4 p = reinterpret_cast<const uint4*>(B + h.o_ec)[i];
        const double2 g = v.gc(p.x >> 16);
        const double s = (v.ref(p.y & 0xFFFF) + v.ref(p.y >> 16)) + (v.ref(p.z & 0xFFFF) + v.ref(p.z >> 16));
        v.at(p.x & 0xFFFF) = __builtin_fma(a0, g.y, g.x) + (s + (v.ref(p.w & 0xFFFF) + v.ref(p.w >> 16)));
    }
#pragma nounroll
    for (int i = tid; i < h.n_ez; i += W) v.at((B + h.o_ez)[i]) = 0.0;
    // wavefront sums
    const uint4* items = reinterpret_cast<const uint4*>(B + h.o_items);
#pragma nounroll
    for (int i = 0; i < h.n_items; i += 2) {
        const uint4 p = items[i], q = items[i + 1];
        double s = item_part<NR>(h, v, a0, qx, p), t = item_part<NR>(h, v, a0, qx, q);
        wave_sum2(s, t);
        if (tid == 0) {
            v.at(p.x & 0xFFFF) = p.w & 0xFFFF ? -s : s;
            v.at(q.x & 0xFFFF) = q.w & 0xFFFF ? -t : t;
        }
    }
}

// Rows that carry charge pinned: F's row k becomes the unit row, x[k] =
// pin - u[k] (consistent initialisation; runs after the assembly).
template <int NR>
__device__ __forceinline__ void apply_pins(Hdr c, const View& v, const DPlan* __restrict__ P,
                                           const double (&pinv)[NR], const uint32_t (&flag)[NR]) {
    c = fresh(c);
    lds_sync();
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = lane_id() + W * r;
        if (k < c->n && (flag[r] & 1)) {
            const int dg = P->diag[k];
#pragma nounroll
            for (int e = P->rowptr[k]; e < P->rowptr[k + 1]; e++) v.at(c->b_F + 8 * e) = e == dg ? 1.0 : 0.0;
            v.at(c->b_inv + 8 * k) = 1.0;
            v.at(c->b_x + 8 * k) = pinv[r] - v.at(c->b_u + 8 * k);
        }
    }
}

// Largest |residual|, NaN-propagating; x holds the negated residuals.
template <int NR>
__device__ __forceinline__ double residual_max(Hdr c, const View& v) {
    double m = 0.0;
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = lane_id() + W * r;
        if (k < c->n) {
            const double a = fabs(v.at(c->b_x + 8 * k));
            if (a != a || a > m) m = a;
        }
    }
    return wave_reduce(m, OpMax());
}

// One long record by the whole wavefront: lane l subtracts products ub + l,
// ub + l + 64, ... in order, then one wave_sum of the lanes' partial sums.
__device__ __forceinline__ void long_task(const View& v, const uint16_t* upd, uint32_t w0, uint32_t w1, bool dia) {
    const uint32_t* up = reinterpret_cast<const uint32_t*>(upd);
    const int tid = fresh_lane(lane_id());
    const int ue = w1 >> 16;
    const double x0 = v.at(w0 & 0xFFFF), sc = v.at(w0 >> 16);
    double s = 0.0;
#pragma nounroll
    for (int q = (int)(w1 & 0xFFFF) + tid; q < ue; q += 2 * W) {
        const int q2 = q + W;
        const uint32_t a = up[q], b = up[q2 < ue ? q2 : q];
        const double fa = v.at(a & 0xFFFF), xa = v.at(a >> 16), fb = v.at(b & 0xFFFF), xb = v.at(b >> 16);
        s = __builtin_fma(fa, xa, s);
        if (q2 < ue) s = __builtin_fma(fb, xb, s);
    }
    s = x0 - wave_sum(s);
    const double t = dia ? recip(s) : s * sc;
    if (tid == 0) {
        v.at(w0 & 0xFFFF) = dia ? s : t;
        if (dia) v.at(w0 >> 16) = t;
    }
}

// One record of a step of products or scalings, for the lanes that have one.
__device__ __forceinline__ void masked_step(const View& v, uint32_t kind, const uint4& w) {
    if (kind == SP_SCALE) {
        const double r0 = v.at(w.x & 0xFFFF) * v.at(w.x >> 16), r1 = v.at(w.y & 0xFFFF) * v.at(w.y >> 16);
        const double r2 = v.at(w.z & 0xFFFF) * v.at(w.z >> 16), r3 = v.at(w.w & 0xFFFF) * v.at(w.w >> 16);
        v.at(w.x & 0xFFFF) = r0;
        v.at(w.y & 0xFFFF) = r1;
        v.at(w.z & 0xFFFF) = r2;
        v.at(w.w & 0xFFFF) = r3;
        return;
    }
    double r = __builtin_fma(-v.at(w.y & 0xFFFF), v.at(w.y >> 16), v.at(w.x & 0xFFFF));
    if (kind != SP_MUL1)
        r = __builtin_fma(-v.at(w.w & 0xFFFF), v.at(w.w >> 16),
                          __builtin_fma(-v.at(w.z & 0xFFFF), v.at(w.z >> 16), r));
    if (kind == SP_DIA3) {
        v.at(w.x & 0xFFFF) = r;
        v.at(w.x >> 16) = recip(r);
    } else {
        v.at(w.x & 0xFFFF) = r * v.at(w.x >> 16);
    }
}

// Run ns steps of the solve program (descriptors at steps).  The descriptors
// come one per lane, 63 steps and the following one at a time, and each
// step's through a lane read; the next step's record is requested before this
// step's operands, so that its latency lies under this step, and all operands
// of a record before any is used.  Lanes past the count run the step's last
// record again and store the same values: with the store masked, a step of
// one product took 350 cycles for 120 (measured alone, one wavefront).  ILP =
// false masks them off, for a CU whose LDS pipe is full.
template <bool ILP>
__device__ __forceinline__ void run_steps(const View& v, const uint16_t* steps, int ns, const uint16_t* recs,
                                          const uint16_t* upd) {
    const uint32_t* sd = reinterpret_cast<const uint32_t*>(steps);
    const uint4* rec = reinterpret_cast<const uint4*>(recs);
    const int tid = fresh_lane(lane_id());
    auto fetch = [&](uint32_t d) {
        const int c1 = (int)(d >> 16) & 63;
        if constexpr (ILP) return rec[(d & 0xFFFF) + (tid < c1 ? tid : c1)];
        uint4 w = make_uint4(0, 0, 0, 0);
        if (tid <= c1) w = rec[(d & 0xFFFF) + tid];
        return w;
    };
#pragma nounroll
    for (int s0 = 0; s0 < ns; s0 += W - 1) {
        const int m = ns - s0 < W - 1 ? ns - s0 : W - 1;
        const int dv = (int)sd[s0 + (tid < m ? tid : m)];
        uint32_t dn = (uint32_t)__builtin_amdgcn_readlane(dv, 0);
        uint4 next = fetch(dn);
#pragma nounroll
        for (int q = 1; q <= m; q++) {
            const uint32_t d = dn;
            const uint4 w = next;
            dn = (uint32_t)__builtin_amdgcn_readlane(dv, q);
            next = fetch(dn);
            const uint32_t kind = d >> 22;
            if (!ILP && kind <= SP_DIA3) {
                if (tid <= ((int)(d >> 16) & 63)) masked_step(v, kind, w);
            } else if (kind == SP_MUL1) {
                const double x = v.at(w.x & 0xFFFF), a0 = v.at(w.y & 0xFFFF), b0 = v.at(w.y >> 16), k = v.at(w.x >> 16);
                const double r = __builtin_fma(-a0, b0, x) * k;
                lds_sync();
                v.at(w.x & 0xFFFF) = r;
            } else if (kind == SP_MUL3) {
                const double x = v.at(w.x & 0xFFFF), a0 = v.at(w.y & 0xFFFF), b0 = v.at(w.y >> 16);
                const double a1 = v.at(w.z & 0xFFFF), b1 = v.at(w.z >> 16), a2 = v.at(w.w & 0xFFFF), b2 = v.at(w.w >> 16);
                const double k = v.at(w.x >> 16);
                const double r = __builtin_fma(-a2, b2, __builtin_fma(-a1, b1, __builtin_fma(-a0, b0, x))) * k;
                lds_sync();
                v.at(w.x & 0xFFFF) = r;
            } else if (kind == SP_SCALE) {
                const double r0 = v.at(w.x & 0xFFFF) * v.at(w.x >> 16), r1 = v.at(w.y & 0xFFFF) * v.at(w.y >> 16);
                const double r2 = v.at(w.z & 0xFFFF) * v.at(w.z >> 16), r3 = v.at(w.w & 0xFFFF) * v.at(w.w >> 16);
                lds_sync();
                v.at(w.x & 0xFFFF) = r0;
                v.at(w.y & 0xFFFF) = r1;
                v.at(w.z & 0xFFFF) = r2;
                v.at(w.w & 0xFFFF) = r3;
            } else if (kind == SP_DIA3) {
                const double x = v.at(w.x & 0xFFFF), a0 = v.at(w.y & 0xFFFF), b0 = v.at(w.y >> 16);
                const double a1 = v.at(w.z & 0xFFFF), b1 = v.at(w.z >> 16), a2 = v.at(w.w & 0xFFFF), b2 = v.at(w.w >> 16);
                const double r = __builtin_fma(-a2, b2, __builtin_fma(-a1, b1, __builtin_fma(-a0, b0, x)));
                const double ri = recip(r);
                lds_sync();
                v.at(w.x & 0xFFFF) = r;
                v.at(w.x >> 16) = ri;
            } else {
                const int c1 = (int)(d >> 16) & 63;
#pragma nounroll
                for (int i = 0; i <= c1; i++)
                    long_task(v, upd, (uint32_t)__builtin_amdgcn_readlane((int)w.x, i),
                              (uint32_t)__builtin_amdgcn_readlane((int)w.y, i), kind == SP_LDIA);
            }
            lds_sync();
        }
    }
}

// LU with the forward substitution of x folded in.
template <bool ILP>
__device__ __forceinline__ void factor(const Hot& h, const View& v) {
    run_steps<ILP>(v, v.B + h.o_steps, h.n_lu, v.B + h.o_rec, v.B + h.o_upd);
}

// Newton step: LU + forward, then backward.
template <bool ILP>
__device__ __forceinline__ void factor_solve(const Hot& h, const View& v) {
    run_steps<ILP>(v, v.B + h.o_steps, h.n_steps, v.B + h.o_rec, v.B + h.o_upd);
}

// J^T x = b on the factors in F (U^T then L^T); b and the result in x.
__device__ __forceinline__ void solve_transposed(Hdr c, const View& v) {
    c = fresh(c);
    run_steps<true>(v, v.B + c->o_tsteps, c->n_tsteps, v.B + c->o_rec, v.B + c->o_upd);
}

// charge of pivot row k: sum over its linear entries C * u
__device__ __forceinline__ double row_charge(Hdr c, const View& v, int k) {
    const uint4 p = reinterpret_cast<const uint4*>(v.B + c->o_rr)[k];
    const uint32_t l0 = p.x & 0xFFFF;
    const uint32_t nl = (p.x >> 16) == 0xFFFF ? p.y >> 16 : p.x >> 16;   // a long row's count: its first reference
    double acc = v.gc(16 * l0).y * v.at(p.y & 0xFFFF);
#pragma nounroll
    for (uint32_t l = l0 + 1; l < l0 + nl; l++) acc = __builtin_fma(v.gc(16 * l).y, v.at((v.B + c->o_lcol)[l]), acc);
    return acc;
}

// (C^T x)[j] for column j: sum over the linear entries of column j
__device__ __forceinline__ double col_charge_t(Hdr c, const View& v, int j) {
    const uint16_t* B = v.B;
    const uint32_t cz = reinterpret_cast<const uint32_t*>(B + c->o_cdesc)[j];
    double acc = 0.0;
#pragma nounroll
    for (int q = cz & 0xFFFF; q < (int)(cz >> 16); q++)
        acc = __builtin_fma(v.gc(16 * (uint32_t)B[c->o_lcl + q]).y, v.at(c->b_x + 8 * B[c->o_lrow + q]), acc);
    return acc;
}

__device__ __forceinline__ double lin_value(const DPlan* __restrict__ P, const double* __restrict__ p,
                                            int32_t ref) {
    const int s = ref >> 1;
    const int kd = P->lin_kind[s];
    double val = 1.0;
    if (kd != 0) {
        const double pv = p[P->lin_idx[s]];
        val = kd == 1 ? 1.0 / pv : kd == 2 ? pv : -pv;
    }
    val *= P->lin_scale[s];
    return (ref & 1) ? -val : val;
}

// Instance set-up: linear stamps G, C, constants and source data into LDS,
// device constants into registers.  The caller synchronises.
template <int NM>
__device__ __forceinline__ void setup_instance(Hdr c, const DPlan* __restrict__ P, const double* __restrict__ p,
                                               const View& v, DevRegs<NM>& dr) {
    c = fresh(c);
    const int tid = lane_id(), nlin = c->nlin;
    // the F position of a linear entry, from the global plan's patterns: the
    // entries with a G or C contribution, in F order
    const int32_t* lp = c->lpos;
#pragma nounroll
    for (int l = tid; l < nlin; l += W) {
        const int e = lp[l];
        double g = 0.0, cc = 0.0;
#pragma nounroll
        for (int q = P->g_ptr[e]; q < P->g_ptr[e + 1]; q++) g += lin_value(P, p, P->g_ref[q]);
#pragma nounroll
        for (int q = P->c_ptr[e]; q < P->c_ptr[e + 1]; q++) cc += lin_value(P, p, P->c_ref[q]);
        v.at(16 * l) = g;
        v.at(16 * l + 8) = cc;
    }
    if (tid == 0) {
        v.at(16 * nlin) = v.at(16 * nlin + 8) = 0.0;
        v.at(c->b_zero) = 0.0;
        v.at(c->b_one) = 1.0;
        v.at(c->b_trash) = 0.0;
    }
#pragma nounroll
    for (int s = tid; s < c->n_src; s += W) {
        const int4 d = P->src[s];
        double* wd = &v.at(v.B[c->o_src + 4 * s + 1]);
#pragma nounroll
        for (int j = 0; j < d.z; j++) wd[j] = p[d.y + j];
        wd[d.z] = p[d.w];
    }
#pragma unroll
    for (int j = 0; j < NM; j++) {
        const int m = tid + W * j < c->n_mos ? tid + W * j : c->n_mos - 1;   // past the last: a copy of it
        dr.beta[j] = 0.0;
        dr.tpvth[j] = 0.0;
        dr.dg[j] = (uint32_t)c->b_zero * 0x10001u;
        dr.sx[j] = (uint32_t)c->b_zero;
        if (m >= 0) {
            const int4 dv = reinterpret_cast<const int4*>(c->dev)[m];
            dr.beta[j] = p[P->p_mos_kp + m] * p[P->p_mos_w + m] / p[P->p_mos_l + m];
            dr.tpvth[j] = (double)dv.w * p[P->p_mos_vth + m];
            dr.dg[j] = (uint32_t)dv.x | ((uint32_t)dv.y << 16);
            dr.sx[j] = (uint32_t)dv.z | (dv.w > 0 ? 0u : 0x80000000u);
        }
    }
}

// Newton iterations of one BDF step from the predictor already in u:
// eval -> assemble -> LU + solves -> u += x, until WRMS(x) <= tol.
template <int NR, int NM, bool ILP>
__device__ __forceinline__ bool newton(Hdr c, const View& v, const DevRegs<NM>& dr, double gmin, double a0,
                                       const double (&qx)[NR], int maxit, double tol, double reltol, double abstol,
                                       long long& nit) {
    const Hot h = load_hot(c);
    const int n = h.n, bx = h.b_x, bu = h.b_u;
    const double lim = uniform(tol * tol * n);   // WRMS <= tol
#pragma nounroll
    for (int it = 0; it < maxit; it++) {
        eval_mos<NM, ILP>(h, v, dr, gmin);
        lds_sync();
        assemble<NR, ILP>(h, v, a0, qx);
        lds_sync();
        factor_solve<ILP>(h, v);
        nit++;
        double ss = 0.0;
        const int tid = fresh_lane(lane_id());
        double un[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k8 = 8 * row_of(tid, r, n);
            const double d = v.at(bx + k8);
            un[r] = v.at(bu + k8) + d;
            const double q = d * recip(__builtin_fma(reltol, fabs(un[r]), abstol));
            ss = tid + W * r < n ? __builtin_fma(q, q, ss) : ss;
        }
        lds_sync();
#pragma unroll
        for (int r = 0; r < NR; r++) v.at(bu + 8 * row_of(tid, r, n)) = un[r];
        ss = wave_sum(ss);
        lds_sync();
        if (!(ss == ss)) return false;
        if (ss <= lim) return true;
    }
    return false;
}

// Start of DC trajectory j in u (pivot order; the draw is by natural index).
__device__ __forceinline__ void dc_set_start(Hdr c, const View& v, int j) {
#pragma nounroll
    for (int k = lane_id(); k < c->n; k += W) v.at(c->b_u + 8 * k) = dc_start(j, c->colnat[k]);
}

// Consistent initial point: (UIC) the charge rows pinned to u0 and the
// algebraic rows solved, u holding the start; or CedarDCOp: the DC operating
// point by the trajectories and the gmin ladder of dcop_rules.h
// (src/dcop.jl:53-94), then, as its BrownFullBasicInit step (:153), the
// rows that carry charge pinned to that point and the algebraic rows solved
// again with the sources at their transient values at t0.  One Newton loop
// serves every phase:
//   phase -1   pinned (UIC, or after the DC point), at most 50 iterations;
//   phase 0-9  trajectory j from its own start, at most 200 iterations;
//   phase 10   the gmin ladder from trajectory 0's start, stage by stage.
// dc_only ends with the DC point.
template <int NR, int NM, bool DYN, bool ILP>
__device__ __forceinline__ bool init_point(Hdr c, const View& v, const DPlan* __restrict__ P, const DevRegs<NM>& dr,
                                           double gmin, bool uic, double (&pinv)[NR], const uint32_t (&flag)[NR],
                                           double t0, double dc_abstol, long long& nit, bool dc_only = false) {
    const int tid = lane_id();
    double qx0[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) qx0[r] = 0.0;
    eval_sources<DYN>(c, v, t0, uic ? CS_MODE_TRAN : CS_MODE_DCOP);
    int phase = uic ? -1 : 0, stage = 0, it = 0;
    bool pin = uic;
    double g = gmin;
    if (!uic) dc_set_start(c, v, 0);
    lds_sync();
    for (;;) {
        const Hot h = load_hot(c);
        eval_mos<NM, ILP>(h, v, dr, g);
        lds_sync();
        assemble<NR, ILP>(h, v, 0.0, qx0);
        if (pin) apply_pins<NR>(c, v, P, pinv, flag);
        lds_sync();
        const double fn = residual_max<NR>(c, v);
        lds_sync();
        if (fn <= dc_abstol) {
            bool dc_done = phase >= 0 && phase < kDcTrajectories;
            if (phase >= kDcTrajectories) {                  // next ladder stage
                g = dc_gmin_stage(++stage, gmin);
                dc_done = g < 0.0;
                if (!dc_done) {
                    it = 0;
                    continue;
                }
            }
            if (!dc_done || dc_only) return true;            // the pinned phase converged, or the DC point is all
            // the DC point: pin its charge rows, sources at their t0 values
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = tid + W * r;
                pinv[r] = k < c->n ? v.at(c->b_u + 8 * k) : 0.0;
            }
            eval_sources<DYN>(c, v, t0, CS_MODE_TRAN);
            phase = -1;
            pin = true;
            g = gmin;
            it = 0;
            lds_sync();
            continue;
        }
        const int maxit = phase < 0 ? 50 : kDcMaxIt;
        if (!(fn == fn) || __builtin_isinf(fn) || it >= maxit) {
            if (phase < 0 || phase >= kDcTrajectories) return false;
            phase++;
            dc_set_start(c, v, phase < kDcTrajectories ? phase : 0);
            if (phase >= kDcTrajectories) {                  // the gmin ladder
                stage = 0;
                g = dc_gmin_stage(0, gmin);
            }
            it = 0;
            lds_sync();
            continue;
        }
        factor_solve<ILP>(h, v);
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k = tid + W * r;
            if (k < c->n) v.at(c->b_u + 8 * k) += v.at(c->b_x + 8 * k);
        }
        nit++;
        it++;
        lds_sync();
    }
}

// bdf_coeffs, pred_weights and lte_coeff of rules.h with quot() for the
// divisions
__device__ __forceinline__ void step_bdf(int k, double tn, double T0, double T1, double& a0, double& a1, double& a2) {
    const double r0 = quot(1.0, tn - T0);
    a0 = r0;
    a1 = -r0;
    a2 = 0.0;
    if (k != 1) {
        a0 = r0 + quot(1.0, tn - T1);
        a1 = quot(tn - T1, (T0 - tn) * (T0 - T1));
        a2 = quot(tn - T0, (T1 - tn) * (T1 - T0));
    }
}
__device__ __forceinline__ void step_pred(int np, double tn, double T0, double T1, double T2, double& l0, double& l1,
                                          double& l2) {
    l0 = 1.0;
    l1 = l2 = 0.0;
    if (np == 2) {
        const double s = quot(tn - T0, T0 - T1);
        l0 = 1.0 + s;
        l1 = -s;
    } else if (np == 3) {
        l0 = quot((tn - T1) * (tn - T2), (T0 - T1) * (T0 - T2));
        l1 = quot((tn - T0) * (tn - T2), (T1 - T0) * (T1 - T2));
        l2 = quot((tn - T0) * (tn - T1), (T2 - T0) * (T2 - T1));
    }
}
__device__ __forceinline__ double step_lte(int k, double tn, double T0, double T1, double T2, double a0, double a1,
                                           double a2) {
    const double d1 = T0 - tn, d2 = T1 - tn;
    if (k == 1) return quot(a1 * d1 * d1, a0 * (tn - T0) * (tn - T1));
    return quot(a1 * d1 * d1 * d1 + a2 * d2 * d2 * d2, a0 * (tn - T0) * (tn - T1) * (tn - T2));
}

// Recording policy of run_lds that records nothing.
struct NoRec {
    template <int NR>
    __device__ __forceinline__ bool on_accept(Hdr, const View&, double, double, int,
                                              long long, const double (&)[NR], const double (&)[NR],
                                              const double (&)[NR]) {
        return true;
    }
};

// One instance's whole transient (the step loop of rules.h).  Rec::on_accept
// is called for the initial point (m = 0) and after every accepted step m
// with the new state in u and the history registers; returning false stops
// the run with CS_E_RANGE.
template <int NR, bool DYN, bool ILP, class Rec>
__device__ __forceinline__ void run_lds(Rec& rec, Hdr c, ConstPtr<LdsArgs> A, const DPlan* __restrict__ P, int inst,
                                        const View& v) {
    constexpr int NM = 2 * NR;
    const int tid = lane_id();
    const int n = c->n, bu = c->b_u;
    const uint64_t clk0 = wall_clock64();
    const double* const p = A->params + A->p_off[inst];
    const double* const u0 = A->u0 ? A->u0 + A->u_off[inst] : nullptr;
    const bool uic = A->o.init == CS_INIT_UIC && u0 != nullptr;

    DevRegs<NM> dr;
    setup_instance<NM>(c, P, p, v, dr);
    const double gmin = p[P->p_gmin];
    double Uh0[NR], Uh1[NR], Uh2[NR], Qh0[NR], Qh1[NR], up[NR], qx[NR], pinv[NR];
    uint32_t flag[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = tid + W * r;
        Uh0[r] = Uh1[r] = Uh2[r] = Qh0[r] = Qh1[r] = up[r] = qx[r] = pinv[r] = 0.0;
        flag[r] = 0;
        if (k < n) {
            flag[r] = c->diffrow[k] ? 1u : 0u;
            pinv[r] = uic ? u0[c->colnat[k]] : 0.0;
            v.at(bu + 8 * k) = pinv[r];
        }
    }
    lds_sync();

    long long steps = 0, rej = 0, nit = 0;
    int rc = init_point<NR, NM, DYN, ILP>(c, v, P, dr, gmin, uic, pinv, flag, A->o.t_start, A->o.dc_abstol, nit)
                 ? CS_OK : CS_E_NOCONV;

    A = fresh(A);
    const double t_start = A->o.t_start;
    double t = t_start;
    if (rc == CS_OK) {
        lds_sync();
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int k = row_of(tid, r, n);
            Uh0[r] = v.at(bu + 8 * k);
            Qh0[r] = row_charge(c, v, k);
        }
        if (!rec.template on_accept<NR>(c, v, t_start, t_start, 0, 0, Uh0, Uh1, Uh2)) rc = CS_E_RANGE;
        double T0 = t_start, T1 = 0.0, T2 = 0.0;
        int npts = 1;
        // step_defaults of rules.h
        const double span = A->o.t_stop - t_start;
        double h = uniform(A->o.dt_init > 0 ? A->o.dt_init : span * 1e-9);
        const double dt_min = uniform(A->o.dt_min > 0 ? A->o.dt_min : span * 1e-15);
        double* const wave = A->wave ? A->wave + A->w_off[inst] : nullptr;
        int kout = 0;
        const int n_probe = P->n_probe;
        // a row's place in a sample, read where samples are written: kept, it
        // would hold registers across the transient
        auto places = [&](int32_t (&ps)[NR]) {
            c = fresh(c);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int k = lane_id() + W * r;
                ps[r] = k < c->n ? c->probe[k] : -1;
            }
        };
        if (wave) {
            int32_t ps[NR];
            places(ps);
            while (kout < A->o.n_out && out_due(out_time(t_start, kout, A->o.dt_out), t_start, A->o.dt_out)) {
#pragma unroll
                for (int r = 0; r < NR; r++)
                    if (ps[r] >= 0) wave[(size_t)kout * n_probe + ps[r]] = Uh0[r];
                kout++;
            }
        }
        // with only DC sources there is no breakpoint and, in transient mode,
        // no source value that changes with t: the per-step breakpoint
        // search is skipped and the sources are evaluated at the first step
        bool dyn_src = false;
        if constexpr (DYN) {
            int dyn = 0;
#pragma nounroll
            for (int s = tid; s < c->n_src; s += W)
                if (v.B[c->o_src + 4 * s] != CS_WAVE_DC) dyn = 1;
            dyn_src = wave_reduce((double)dyn, OpMax()) > 0.0;
        }
        bool src_set = false;
        lds_sync();
        for (;;) {
            lds_sync();
            A = fresh(A);
            const double t_stop = A->o.t_stop;
            if (!(rc == CS_OK && t < t_stop)) break;
            if (steps + rej >= A->o.max_steps) { rc = CS_E_MAXSTEPS; break; }
            double tb = t_stop;
            bool srcbp = false;
            if constexpr (DYN) {
                if (dyn_src) {
                    double lb = INFINITY;
#pragma nounroll
                    for (int s = tid; s < c->n_src; s += W) {
                        const uint16_t* d = v.B + c->o_src + 4 * s;
                        const double b = next_bp(d[0], &v.at(d[1]), d[2], t);
                        if (b < lb) lb = b;
                    }
                    tb = uniform(wave_reduce(lb, OpMin()));
                    srcbp = tb < t_stop;
                    if (!srcbp) tb = t_stop;
                }
            }
            const double dt_max = A->o.dt_max > 0 ? A->o.dt_max : quot(t_stop - t_start, 10.0);
            double hh = h < dt_max ? h : dt_max;
            int hit;
            const double tn = uniform(clip_step(t, hh, tb, hit));
            hh = uniform(hh);
            const int k = bdf_order(npts, A->o.max_order);
            double a0, a1, a2, w0, w1, w2;
            step_bdf(k, tn, T0, T1, a0, a1, a2);
            a0 = uniform(a0);
            a1 = uniform(a1);
            a2 = uniform(a2);
            const int np = npts < k + 1 ? npts : k + 1;
            step_pred(np, tn, T0, T1, T2, w0, w1, w2);
            w0 = uniform(w0);
            w1 = uniform(w1);
            w2 = uniform(w2);
            const int lane = fresh_lane(tid);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                double val = Uh0[r];
                if (np == 2) val = __builtin_fma(w0, Uh0[r], w1 * Uh1[r]);
                else if (np == 3) val = __builtin_fma(w0, Uh0[r], __builtin_fma(w1, Uh1[r], w2 * Uh2[r]));
                up[r] = val;
                v.at(bu + 8 * row_of(lane, r, n)) = val;
                qx[r] = __builtin_fma(a1, Qh0[r], k == 2 ? a2 * Qh1[r] : 0.0);
            }
            if (dyn_src || !src_set) eval_sources<DYN>(c, v, tn, CS_MODE_TRAN);
            src_set = true;
            lds_sync();
            if (!newton<NR, NM, ILP>(c, v, dr, gmin, a0, qx, A->o.newton_maxit, A->o.newton_tol, A->o.reltol,
                                A->o.abstol, nit)) {
                rej++;
                h = uniform(0.25 * hh);
                if (h < dt_min) { rc = CS_E_DTMIN; break; }
                continue;
            }
            A = fresh(A);
            double fac = 2.0;
            if (npts >= 2) {
                const double cl = uniform(step_lte(k, tn, T0, T1, T2, a0, a1, a2));
                double ss = 0.0;
                const int lane = fresh_lane(tid);
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const double ui = v.at(bu + 8 * row_of(lane, r, n));
                    const double est = cl * (ui - up[r]);
                    const double m = fabs(ui) > fabs(Uh0[r]) ? fabs(ui) : fabs(Uh0[r]);
                    const double q = est * recip(__builtin_fma(A->o.reltol, m, A->o.abstol));
                    ss = lane + W * r < n ? __builtin_fma(q, q, ss) : ss;
                }
                const double err2 = quot(wave_sum(ss), (double)n);
                if (!(err2 <= 1.0)) {
                    rej++;
                    h = uniform(hh * step_reject(err2, k));
                    if (h < dt_min) { rc = CS_E_DTMIN; break; }
                    continue;
                }
                fac = uniform(step_accept(err2, k));
            }
            // accept
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int kk = row_of(fresh_lane(tid), r, n);
                Uh2[r] = Uh1[r]; Uh1[r] = Uh0[r]; Uh0[r] = v.at(bu + 8 * kk);
                Qh1[r] = Qh0[r]; Qh0[r] = row_charge(c, v, kk);
            }
            if (!rec.template on_accept<NR>(c, v, tn, T0, npts, steps + 1, Uh0, Uh1, Uh2)) {
                rc = CS_E_RANGE;
                break;
            }
            T2 = T1; T1 = T0; T0 = tn;
            if (npts < 3) npts++;
            steps++;
            if (wave)
                put_samples(kout, A->o.t_start, A->o.dt_out, A->o.n_out, tn,
                            [&](double tq, double& l0, double& l1, double& l2) {
                                step_pred(npts, tq, T0, T1, T2, l0, l1, l2);
                            },
                            [&](int k0, int m, double l0, double l1, double l2) {
                                int32_t ps[NR];
                                places(ps);
                                put_rows<NR>(wave, n_probe, k0, m, l0, l1, l2, ps, Uh0, Uh1, Uh2);
                            });
            t = tn;
            h = hh * fac;
            if (hit && srcbp) {
                npts = 1;
                h = 0.1 * h;
                if (h < dt_min) h = dt_min;
            }
            h = uniform(h);
        }
    }
    A = fresh(A);
    c = fresh(c);
    double* const ufin = A->u_final + A->u_off[inst];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = tid + W * r;
        if (k < n) ufin[c->colnat[k]] = (rc == CS_OK || steps > 0) ? Uh0[r] : v.at(bu + 8 * k);
    }
    if (tid == 0) {
        cs_tran_stats* const stp = A->stats + inst;
        stp->steps = steps;
        stp->rejected = rej;
        stp->newton_iters = nit;
        stp->t_end = t;
        stp->retcode = rc;
        stp->pad = 0;
        stp->busy_s = (double)(wall_clock64() - clk0);   // ticks; the host scales them
    }
    lds_sync();
}

}  // namespace lds
}  // namespace cedar
