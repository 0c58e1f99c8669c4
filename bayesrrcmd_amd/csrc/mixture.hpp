// mixture.hpp -- the component draw of processColumn (BayesRBase.cpp:300-366) for one marker, and the
// FP64 exponential and reciprocal it is made of. Shared by the plain, cohort and batched sweeps.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace brr {

// exp(x): x = n ln 2 + r, |r| <= ln 2 / 2, the Taylor series of exp(r) to degree 13 (remainder below 5e-18) in
// Estrin's order, scaled by 2^n. Against long double the error is at most 1.01 ulp (24 million points in
// -745 .. 350). What bounds the decisions is the length of the dependent chain on one wave, and this has half of
// the device library's. kAny = false: |x| <= 700 (NaN stays NaN); true: any x below 700, 0 under -745.
template <bool kAny>
__device__ __forceinline__ double exp_draw(double x)
{
    double n = __builtin_rint(x * 0x1.71547652b82fep+0);        // x / ln 2
    if constexpr (kAny) n = fmax(n, -2000.0);
    double r = __builtin_fma(n, -0x1.62e42fefa39efp-1, x);      // ln 2 in two doubles
    r = __builtin_fma(n, -0x1.abc9e3b39803fp-56, r);
    const double r2 = r * r, r4 = r2 * r2;
    const double a0 = __builtin_fma(r, 1.0 / 6.0, 0.5);
    const double a1 = __builtin_fma(r, 1.0 / 120.0, 1.0 / 24.0);
    const double a2 = __builtin_fma(r, 1.0 / 5040.0, 1.0 / 720.0);
    const double a3 = __builtin_fma(r, 1.0 / 362880.0, 1.0 / 40320.0);
    const double a4 = __builtin_fma(r, 1.0 / 39916800.0, 1.0 / 3628800.0);
    const double a5 = __builtin_fma(r, 1.0 / 6227020800.0, 1.0 / 479001600.0);
    const double b0 = __builtin_fma(r2, a1, a0);
    const double b1 = __builtin_fma(r2, a3, a2);
    const double b2 = __builtin_fma(r2, a5, a4);
    const double q = __builtin_fma(r4, __builtin_fma(r4, b2, b1), b0);
    const double e = __builtin_amdgcn_ldexp(1.0 + __builtin_fma(r2, q, r), (int)n);
    return kAny && x < -745.0 ? 0.0 : e;
}

// 1 / s for a normal s: the hardware estimate and two Newton steps (within an ulp), without the scaling and
// fix-up of the IEEE division sequence. 0 and infinity give NaN.
__device__ __forceinline__ double rcp_draw(double s)
{
    double y = __builtin_amdgcn_rcp(s);
    y = __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-s, y, 1.0), y);
}

struct MixDraw {
    double e0, s;   // the zero component's probability (acum of processColumn) is e0 / s
    int sel;        // the component drawn; -1: none (u beyond the guarded sum)
    __device__ __forceinline__ double acum0() const { return prob0(e0, s); }
    // (a guarded component stays at 0 where the sum is no number: num^2 past the largest double)
    __device__ static __forceinline__ double prob0(double e0, double s) { return e0 == 0.0 ? 0.0 : e0 * rcp_draw(s); }
};

// The draw from n2 = num^2 and the uniform u. Constants per component c (any callables):
//   dg(c) = logL_c - logL_0 at num = 0, hk(c) with logL_c = lc(c) + n2 hk(c) (hk(0) = 0).
// The reference's term 1 / sum_i exp(logL_i - logL_c) is e_c / sum_i e_i with e_c = exp(logL_c - m) for any m.
// m = logL_0 while every |logL_c - logL_0| <= 350, where no 700 guard can fire; else m = max_c logL_c with the
// guards any_{i>=1} |logL_i - logL_c| > 700 evaluated (BayesRBase.cpp:335, 360). A wave without a lane of the
// second kind takes K - 1 exponentials, else K (the reference's K^2 cost about 1,000 instructions for the whole
// wave whenever one lane needed them). u <= acum is decided as u sum_i e_i <= e_0 + .. + e_c, so that no
// reciprocal stands before the choice. kExact: K == kK, so that the exponentials are straight-line code and
// overlap (with a run-time K each became a branch of its own: 900 cycles a draw on one wave instead of 300).
// kPad: straight-line code for any K <= kK. The constants of components K .. kK - 1 are kPadDg, 0 and -infinity: they add
// exp(kPadDg) to a sum of at least 1, which leaves its bits as they are, or 0, and are never drawn.
constexpr double kPadDg = -300.0;

template <int kK, bool kExact, bool kPad = false, class Dg, class Hk, class Lc>
__device__ __forceinline__ MixDraw mix_draw(int Krt, double n2, double u, Dg&& dg, Hk&& hk, Lc&& lc)
{
    const int Kg = kExact ? kK : Krt;          // components that the guards look at
    const int K = kPad ? kK : Kg;
    double x[kK];
    bool far = false;
#pragma unroll
    for (int c = 1; c < kK; ++c)
        if (c < K) {
            x[c] = __builtin_fma(n2, hk(c), dg(c));
            far = far || fabs(x[c]) > 350.0;
        }
    double e[kK];
    e[0] = 1.0;
    uint32_t guard = 0u;   // bit c: component c's guard fires
    if (!__any(far)) {
#pragma unroll
        for (int c = 1; c < kK; ++c) e[c] = c < K ? exp_draw<false>(x[c]) : 0.0;
    } else {
        x[0] = 0.0;
        if (far) {
            double m = x[0] = lc(0);
#pragma unroll
            for (int c = 1; c < kK; ++c)
                if (c < K) {
                    x[c] = __builtin_fma(n2, hk(c), lc(c));
                    m = fmax(m, x[c]);
                }
#pragma unroll
            for (int c = 0; c < kK; ++c)
#pragma unroll
                for (int i = 1; i < kK; ++i)
                    if (i != c && c < Kg && i < Kg && fabs(x[i] - x[c]) > 700.0) guard |= 1u << c;
#pragma unroll
            for (int c = 0; c < kK; ++c)
                if (c < K) x[c] = x[c] - m;
        }
#pragma unroll
        for (int c = 0; c < kK; ++c) e[c] = c < K ? exp_draw<true>(x[c]) : 0.0;
    }
    double s = e[0];
#pragma unroll
    for (int c = 1; c < kK; ++c) s += e[c];
    const double t = u * s;
    MixDraw r;
    double cum = (guard & 1u) ? 0.0 : e[0];
    r.e0 = cum;
    r.s = s;
    r.sel = t <= cum ? 0 : -1;
#pragma unroll
    for (int c = 1; c < kK; ++c) {
        cum += ((guard >> c) & 1u) ? 0.0 : e[c];
        if (c < K && r.sel < 0 && t <= cum) r.sel = c;
    }
    return r;
}

} // namespace brr
