// FP64 elementary functions for the delay samplers, sized for sampling:
// results within a few ulp of the correctly rounded value, in a fraction of the
// instructions of a general-purpose libm.  Each is written from the textbook
// method named on it; the test suite compares them with the host libm over
// their sampling domains.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mcdp_log_table.hpp"

namespace mcdp {

// p * z + c for a polynomial coefficient c.  The compiler's accumulate form
// (v_fmac_f64) wants c in vector registers and rebuilds each 64-bit constant
// with two v_mov_b32 per use; here c is bound to a scalar register pair, so a
// Horner step is one v_fma_f64 (the pair is set up by scalar moves, which
// issue beside the vector pipeline).
__device__ __forceinline__ double fma_k(double p, double z, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(z), "s"(c));
    return r;
#else
    return __builtin_fma(p, z, c);
#endif
}

// The table of log_tab (the lookups are per lane): kLogInv and kLogHiLo from
// mcdp_log_table.hpp, written by gen_log_table.py.  Kernels that sample many
// activities per workgroup stage it in LDS (6 KB); the others read it where it
// lies (global_log_table).
struct LogTable {
    const double *inv;    // [kLogTableSize]: 1/c_j rounded to 2^-10
    const double2 *hilo;  // [kLogTableSize]: -log(inv_j) = hi + lo, hi a multiple of 2^-32
};
__device__ __forceinline__ LogTable global_log_table() {
    return LogTable{kLogInv, reinterpret_cast<const double2 *>(kLogHiLo)};
}
struct LogTableLds {
    double inv[kLogTableSize];
    double2 hilo[kLogTableSize];
    __device__ LogTable view() const { return LogTable{inv, hilo}; }
};
// Every thread of the workgroup calls it; the caller's next barrier makes the
// table visible to all waves.
__device__ __forceinline__ void stage_log_table(LogTableLds &t) {
    for (int i = threadIdx.x; i < kLogTableSize; i += blockDim.x) {
        t.inv[i] = kLogInv[i];
        t.hilo[i] = double2{kLogHiLo[2 * i], kLogHiLo[2 * i + 1]};
    }
}

// Natural logarithms of N positive normal x, table-driven (P. T. P. Tang,
// "Table-driven implementation of the logarithm function in IEEE
// floating-point arithmetic", ACM TOMS 16(4), 1990), the scale and interval
// taken from x's high word with integer operations (half an FP64 operation's
// issue time each, against frexp, rint and conversions): z = x 2^m in (0.69,
// 1.38), c the middle of z's interval of 256, inv = 1/c rounded to 2^-10;
// log x = -m ln2 - log(inv) + log(1 + r) with r = z inv - 1, |r| <= 2^-8.7.
//   * r is one fma, and exact but for its last bits (a multiple of 2^-63);
//   * log(1 + r) = r + r^2 P(r), Taylor to r^6 (remainder < 2^-55 of r);
//   * hi - m ln2_hi is exact (both multiples of 2^-32, sum below 2^10), and
//     the small terms lo - m ln2_lo + log(1 + r) are added to it last.
// c = 1 is the middle of an interval, so near 1 the result is log(1 + r) alone
// and its relative error stays within an ulp; log 1 = 0.  Measured against
// extended precision: at most 0.78 ulp for uniforms, 0.98 ulp in (1 - 2^-8, 1).
// The N logarithms advance step by step together: a wave issues independent
// instructions back to back, and a dependent one half as often.
template <int N>
__device__ __forceinline__ void log_tab_n(const double (&x)[N], const LogTable &t, double (&out)[N]) {
    double kd[N], z[N], inv[N];
    double2 lf[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t d = kLogBase - (uint32_t)__double2hiint(x[i]);
        const int m = (int)d >> 20;
        const uint32_t j = (d >> 12) & 255u;
        inv[i] = t.inv[j];
        lf[i] = t.hilo[j];
        z[i] = __builtin_amdgcn_ldexp(x[i], m);
        kd[i] = (double)m;
    }
    constexpr double ln2_hi = 6.93147180369123816490e-01;  // 0x3fe62e42fee00000
    constexpr double ln2_lo = 1.90821492927058770002e-10;
    double r[N], p[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        r[i] = __builtin_fma(z[i], inv[i], -1.0);
        p[i] = -1.0 / 6.0;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = fma_k(p[i], r[i], 1.0 / 5.0);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = fma_k(p[i], r[i], -1.0 / 4.0);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = fma_k(p[i], r[i], 1.0 / 3.0);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(p[i], r[i], -0.5);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double log1p_r = __builtin_fma(r[i] * r[i], p[i], r[i]);
        const double hi = __builtin_fma(-kd[i], ln2_hi, lf[i].x);
        const double lo = __builtin_fma(-kd[i], ln2_lo, lf[i].y) + log1p_r;
        out[i] = hi + lo;
    }
}
__device__ __forceinline__ double log_tab(double x, const LogTable &t) {
    const double v[1] = {x};
    double out[1];
    log_tab_n<1>(v, t, out);
    return out[0];
}

// cos(2 pi u) for u in [0, 1], to within ~3e-16 absolute, N at a time.
// Reduce to w in [0, 1/4] by the symmetries of cosine (period 1, even,
// cos(pi - a) = -cos a), then the Taylor polynomial of cos in a = 2 pi w,
// |a| <= pi/2, to degree 22 (remainder (pi/2)^24 / 24! < 1e-22).  Near
// a = pi/2 the result is small and its error is absolute, which is what the
// samplers need (they use cos as a factor of a normal deviate).
template <int N>
__device__ __forceinline__ void cos2pi_n(const double (&u)[N], double (&out)[N]) {
    constexpr double two_pi = 6.28318530717958647693;
    constexpr double q[10] = {1.0 / 24.0,                        //  1/4!
                              -1.0 / 720.0,                      // -1/6!
                              1.0 / 40320.0,                     //  1/8!
                              -1.0 / 3628800.0,                  // -1/10!
                              1.0 / 479001600.0,                 //  1/12!
                              -1.0 / 87178291200.0,              // -1/14!
                              1.0 / 20922789888000.0,            //  1/16!
                              -1.0 / 6402373705728000.0,         // -1/18!
                              1.0 / 2432902008176640000.0,       //  1/20!
                              -1.0 / 1.1240007277776077e21};     // -1/22!
    double a2[N], c[N];
    bool neg[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        double w = u[i] - __builtin_rint(u[i]);  // [-1/2, 1/2]
        w = __builtin_fabs(w);                   // cos is even
        neg[i] = w > 0.25;                       // cos(2pi w) = -cos(2pi (1/2 - w))
        w = neg[i] ? 0.5 - w : w;                // [0, 1/4]
        const double a = w * two_pi;
        a2[i] = a * a;
        c[i] = q[9];
    }
#pragma unroll
    for (int k = 8; k >= 0; --k)
#pragma unroll
        for (int i = 0; i < N; ++i) c[i] = fma_k(c[i], a2[i], q[k]);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        c[i] = __builtin_fma(c[i], a2[i], -0.5);
        c[i] = __builtin_fma(c[i], a2[i], 1.0);
        out[i] = neg[i] ? -c[i] : c[i];
    }
}
__device__ __forceinline__ double cos2pi_fast(double u) {
    const double v[1] = {u};
    double out[1];
    cos2pi_n<1>(v, out);
    return out[0];
}

// e^x for x <= 0 down to about -745 (the only range the samplers use):
// x = k ln 2 + r with |r| <= ln2 / 2 (Cody-Waite split of ln 2), Taylor
// polynomial of e^r to degree 13 (remainder < 2^-56), times 2^k by ldexp.
__device__ __forceinline__ double exp_fast(double x) {
    constexpr double inv_ln2 = 1.44269504088896338700;
    constexpr double ln2_hi = 6.93147180369123816490e-01;
    constexpr double ln2_lo = 1.90821492927058770002e-10;
    const double kd = __builtin_rint(x * inv_ln2);
    const double r = __builtin_fma(-kd, ln2_lo, __builtin_fma(-kd, ln2_hi, x));
    double p = 1.0 / 6227020800.0;                 // 1/13!
    p = fma_k(p, r, 1.0 / 479001600.0);    // 1/12!
    p = fma_k(p, r, 1.0 / 39916800.0);     // 1/11!
    p = fma_k(p, r, 1.0 / 3628800.0);      // 1/10!
    p = fma_k(p, r, 1.0 / 362880.0);       // 1/9!
    p = fma_k(p, r, 1.0 / 40320.0);        // 1/8!
    p = fma_k(p, r, 1.0 / 5040.0);         // 1/7!
    p = fma_k(p, r, 1.0 / 720.0);          // 1/6!
    p = fma_k(p, r, 1.0 / 120.0);          // 1/5!
    p = fma_k(p, r, 1.0 / 24.0);           // 1/4!
    p = fma_k(p, r, 1.0 / 6.0);            // 1/3!
    p = __builtin_fma(p, r, 0.5);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    return __builtin_amdgcn_ldexp(p, (int)kd);
}

}  // namespace mcdp
