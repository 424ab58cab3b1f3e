// wave_math.h — the waveforms and step factors of rules.h for kernels that run
// whole transients: every operation inline, few registers.  The library's sin,
// exp, fmod and pow, inlined, set the register count of such a kernel (k_tran_batch
// 208 vector registers with them, 123 without).  Multiplications and additions
// are fused only where the source says fma, as lds_core.h explains.
#pragma once
#include "rules.h"

namespace cedar {

// s^(-1/(2(k+1))), k = 1 or 2, for s within [1e-6, 1e8]: the step factor's
// root of the error err = sqrt(s), by a single-precision estimate and two
// Newton steps on z^-(2(k+1)) = s.
__device__ __forceinline__ double inv_root(double s, int k) {
#pragma clang fp contract(off)
    const float p = k == 1 ? -0.25f : -1.0f / 6.0f;
    double z = (double)__builtin_amdgcn_exp2f(p * __builtin_amdgcn_logf((float)s));
    const double w = k == 1 ? 0.25 : 1.0 / 6.0;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const double z2 = z * z, zp = k == 1 ? z2 * z2 : z2 * z2 * z2;
        z = __builtin_fma(z * w, __builtin_fma(-s, zp, 1.0), z);
    }
    return z;
}

// reject_factor and accept_factor of rules.h from the mean square of the
// error: outside err in [0.09, 729] (k = 2) or [0.2, 81] (k = 1) their clamps
// decide.
__device__ __forceinline__ double step_reject(double s, int k) {
#pragma clang fp contract(off)
    if (!(s < 1e8)) return 0.1;
    const double f = 0.9 * inv_root(s, k);
    return f < 0.1 ? 0.1 : f;
}
__device__ __forceinline__ double step_accept(double s, int k) {
#pragma clang fp contract(off)
    if (!(s > 1e-6)) return 2.0;
    const double f = 0.9 * inv_root(s, k);
    return f > 2.0 ? 2.0 : f;
}

// fmod(t, per), exactly: the remainder by fma is exact and the quotient off
// by one at most while t / per is below 2^52; larger ratios are first reduced
// modulo multiples of per.
__device__ __forceinline__ double fmod_exact(double t, double per) {
#pragma clang fp contract(off)
    double a = fabs(t);
    const double p = fabs(per);
    if (!(p > 0.0) || !(a < INFINITY)) return __builtin_nan("");
    if (!(p < INFINITY)) return t;
    auto part = [](double x, double m) {
        double r = __builtin_fma(-floor(x / m), m, x);
        if (r < 0.0) r += m;
        return r >= m ? r - m : r;
    };
    while (!(a < p * 0x1p52)) {
        int ea, ep;
        (void)frexp(a, &ea);
        (void)frexp(p, &ep);
        a = part(a, ldexp(p, ea - ep - 41));
    }
    return copysign(part(a, p), t);
}

// Taylor coefficients of sine (odd, 1/17! first) and cosine (even, 1/16!
// first), in memory: as literals they would be held in registers across the
// whole transient.
static __device__ const double kSinCos[2][8] = {
    {1.0 / 355687428096000.0, -1.0 / 1307674368000.0, 1.0 / 6227020800.0, -1.0 / 39916800.0, 1.0 / 362880.0,
     -1.0 / 5040.0, 1.0 / 120.0, -1.0 / 6.0},
    {1.0 / 20922789888000.0, -1.0 / 87178291200.0, 1.0 / 479001600.0, -1.0 / 3628800.0, 1.0 / 40320.0,
     -1.0 / 720.0, 1.0 / 24.0, -0.5}};

// sin_deg of rules.h: reduced to [-45, 45] degrees without rounding, then the
// Taylor sum of sine or cosine (next terms below 1e-18).
__device__ __forceinline__ double sin_degrees(double x) {
#pragma clang fp contract(off)
    const double r = fmod_exact(x, 360.0);
    const double q = rint(r / 90.0);
    const double y = __builtin_fma(-90.0, q, r) * (3.14159265358979323846 / 180.0);
    const double z = y * y;
    const int k = (int)q & 3;
    const double* t = kSinCos[k & 1];
    double s = t[0];
#pragma nounroll
    for (int j = 1; j < 8; j++) s = __builtin_fma(s, z, t[j]);
    s = k & 1 ? __builtin_fma(s, z, 1.0) : __builtin_fma(s * z, y, y);
    return k & 2 ? -s : s;
}

// 1/13! .. 1/0! and the two parts of ln 2, in memory as above.
static __device__ const double kExp[16] = {
    1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0, 1.0 / 3628800.0, 1.0 / 362880.0, 1.0 / 40320.0,
    1.0 / 5040.0, 1.0 / 720.0, 1.0 / 120.0, 1.0 / 24.0, 1.0 / 6.0, 0.5, 1.0, 1.0,
    0x1.62e42fefa0000p-1, 0x1.cf79abc9e3b3ap-40};

// e^x: x = k ln 2 + r, the Taylor sum of e^r (next term below 1e-17), scaled.
__device__ __forceinline__ double exp_taylor(double x) {
#pragma clang fp contract(off)
    const double y = x < -1100.0 ? -1100.0 : x > 1100.0 ? 1100.0 : x;
    const double k = rint(y / kExp[14]);
    const double r = __builtin_fma(-k, kExp[15], __builtin_fma(-k, kExp[14], y));
    double s = kExp[0];
#pragma nounroll
    for (int j = 1; j < 14; j++) s = __builtin_fma(s, r, kExp[j]);
    s = ldexp(s, (int)k);
    return x == x ? s : x;
}

// source_value of rules.h without calls: every operation inline, so that the
// transient loop keeps its registers across it.
__device__ __forceinline__ double source_at(int kind, const double* d, int len, double dc, double t, int mode) {
#pragma clang fp contract(off)
    if (mode == CS_MODE_DCOP) {
        if (dc == dc) return dc;
        t = 0.0;
    }
    if (kind == CS_WAVE_DC) return d[0];
    if (kind == CS_WAVE_PULSE) {
        const double c0 = d[2], c1 = d[2] + d[3], c2 = d[2] + d[3] + d[5];
        const double c3 = d[2] + d[3] + d[5] + d[4];
        return pulse_at(d[0], d[1], c0, c1, c2, c3, fmod_exact(t, d[6]));
    }
    if (kind == CS_WAVE_PWL) return pwl_at(d, len / 2, t);
    // CS_WAVE_SIN: vo va freq td theta phase ncycles
    double ang = d[5], amp = d[1];
    if (d[3] < t && t < d[6] / d[2]) {
        ang = 360.0 * d[2] * (t - d[3]) + d[5];
        if (d[4] != 0.0) amp *= exp_taylor(-(t - d[3]) * d[4]);
    }
    return d[0] + amp * sin_degrees(ang);
}

// wave_next_bp of rules.h, the corners of a pulse one at a time
__device__ __forceinline__ double next_bp(int kind, const double* d, int len, double t) {
#pragma clang fp contract(off)
    const double thr = t + 8.0 * 2.220446049250313e-16 * fabs(t) + 1e-300;
    double best = INFINITY;
    if (kind == CS_WAVE_PULSE) {
        const double per = d[6];
        const bool once = __builtin_isinf(per);
        const double m = once ? 0.0 : floor(t / per);
#pragma nounroll
        for (int j = 0; j < 4; j++) {
            double c = d[2];
            if (j > 0) c += d[3];
            if (j > 1) c += d[5];
            if (j > 2) c += d[4];
            if (once) {
                if (c > thr && c < best) best = c;
            } else if (c < per) {
#pragma nounroll
                for (int r = -1; r <= 1; r++) {
                    const double b = (m + r) * per + c;
                    if (b > thr && b < best) best = b;
                }
            }
        }
    } else if (kind == CS_WAVE_PWL) {
#pragma nounroll
        for (int j = 0; j < len / 2; j++) {
            const double b = d[2 * j];
            if (b > thr && b < best) best = b;
        }
    } else if (kind == CS_WAVE_SIN) {
        if (d[3] > thr) best = d[3];
    }
    return best;
}

}  // namespace cedar
