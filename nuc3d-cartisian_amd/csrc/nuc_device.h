// nuc_device.h -- device-side numerics for the NUC3d RHS sweeps on gfx950.
//
// Point formulas restate the reference schemes (file:line cited per function);
// the arithmetic is rearranged for the GPU (x*x instead of std::pow, one
// normalising division), which changes results only at the rounding level.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nucdev {

enum { WENO5JS = 0, WENO5Z = 1, WENO7JS = 2, CRWENO5 = 3, HCCS = 4, WENO3JS = 5, UPWIND1ST = 6, HCCS78 = 7, HCCS77 = 8 };
enum { VIS_NONE = 0, VIS_CD6 = 1, VIS_CD8 = 2, VIS_CD2 = 3 };
enum { RIE_LF = 0, RIE_AUSM = 1, RIE_AUSMP = 2 };   // AUSM+ runs the AUSM kernels with its pressure splitting

template <typename T> __device__ __forceinline__ T sq(T x) { return x * x; }

// WENO7 smoothness indicators as sums of squares, for FP32 stencils (the
// mixed path).  An exact LDL^T factorisation of each of the reference's
// quadratic forms (src/weno7js.cpp:80-99) in the differences g_i = f_i - f_{i+1}
// (the forms vanish on constants):
//   is0(f0..f3) = (547 g0 - 1394 g1 + 927 g2)^2 / 547
//               + 85040 / (547 * 2126^2) * (2126 g1 - 3167 g2)^2 + 203060 / 1063 * g2^2
//   is1(f0..f3) = (267 g0 - 554 g1 + 247 g2)^2 / 267
//               + 85040 / (267 * 2126^2) * (2126 g1 - 1345 g2)^2 + 203060 / 1063 * g2^2
// and is2, is3 are is1, is0 of the mirrored stencil.  Every term is
// non-negative, so FP32 evaluates them to FP32's relative precision instead
// of cancelling terms up to 17246 f^2.  outer: the is0 form, else is1's.
template <typename T>
__device__ __forceinline__ T w7_sos(T a, T b, T c, T d, bool outer)
{
    const T g0 = a - b, g1 = b - c, g2 = c - d;
    const T e0 = outer ? T(547) * g0 - T(1394) * g1 + T(927) * g2 : T(267) * g0 - T(554) * g1 + T(247) * g2;
    const T e1 = T(2126) * g1 - (outer ? T(3167) : T(1345)) * g2;
    const T k0 = outer ? T(1.0 / 547.0) : T(1.0 / 267.0);
    const T k1 = outer ? T(85040.0 / (547.0 * 2126.0 * 2126.0)) : T(85040.0 / (267.0 * 2126.0 * 2126.0));
    return k0 * e0 * e0 + k1 * e1 * e1 + T(203060.0 / 1063.0) * g2 * g2;
}

// reciprocal: hardware estimate r (2^-25 relative) refined by one third-order
// step, r + r (e + e^2) with e = 1 - x r: e^3 is below 2^-74, and the one
// rounding left is that of the sum (|err| <= 1 ulp).  Two Newton steps reach the
// same with one instruction more; the sweeps take 15 reciprocals a variable.
__device__ __forceinline__ double frcp(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}
// Two Newton steps, for the FP64 solve behind FP32 stencils: a last bit of the
// state that differs moves an FP32 rounding somewhere, and the runs part from
// there, so these solves keep the reciprocal they have.
template <bool F32> __device__ __forceinline__ double frcp_for(double x)
{
    if constexpr (!F32) {
        return frcp(x);
    } else {
        double r = __builtin_amdgcn_rcp(x);
        double e = fma(-x, r, 1.0);
        r = fma(r, e, r);
        e = fma(-x, r, 1.0);
        return fma(r, e, r);
    }
}
// a / x from r = 1/x (two Newton steps): the product and one remainder step,
// which round as the IEEE quotient does, without its scaling (x between 1e-290
// and 1e290, and finite)
__device__ __forceinline__ double fquot(double a, double x, double r)
{
    const double q = a * r;
    return fma(fma(-x, q, a), r, q);
}
// FP32 (mixed path): the hardware reciprocal, 1 ulp
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

// 7-point WENO stencil, src/weno7js.cpp:79-118: smoothness indicators b and
// candidate values q of f[0..6].
// FP64 stencils: the smoothness indicators are the reference's expanded
// quadratic forms, whose coefficients (up to 17246) cancel to O(h^2) on smooth
// data, so any reassociation or FMA moves them by ~1e-6 relative and shifts
// the Z weights.  They are therefore evaluated without contraction and in the
// reference's operation order, which makes them bit-identical to the
// reference.  FP32 stencils (the mixed path) use the sums of squares above.
template <typename T>
__device__ __forceinline__ void weno7_stencil(const T *f, T b[4], T q[4])
{
#pragma clang fp contract(off)
    T is0, is1, is2, is3;
    if constexpr (sizeof(T) == 4) {
        is0 = w7_sos(f[0], f[1], f[2], f[3], true);
        is1 = w7_sos(f[1], f[2], f[3], f[4], false);
        is2 = w7_sos(f[5], f[4], f[3], f[2], false);
        is3 = w7_sos(f[6], f[5], f[4], f[3], true);
    } else {
        is0 = f[0] * (T(547) * f[0] - T(3882) * f[1] + T(4642) * f[2] - T(1854) * f[3])
            + f[1] * (T(7043) * f[1] - T(17246) * f[2] + T(7042) * f[3])
            + f[2] * (T(11003) * f[2] - T(9402) * f[3]) + T(2107) * f[3] * f[3];
        is1 = f[1] * (T(267) * f[1] - T(1642) * f[2] + T(1602) * f[3] - T(494) * f[4])
            + f[2] * (T(2843) * f[2] - T(5966) * f[3] + T(1922) * f[4])
            + f[3] * (T(3443) * f[3] - T(2522) * f[4]) + T(547) * f[4] * f[4];
        is2 = f[2] * (T(547) * f[2] - T(2522) * f[3] + T(1922) * f[4] - T(494) * f[5])
            + f[3] * (T(3443) * f[3] - T(5966) * f[4] + T(1602) * f[5])
            + f[4] * (T(2843) * f[4] - T(1642) * f[5]) + T(267) * f[5] * f[5];
        is3 = f[3] * (T(2107) * f[3] - T(9402) * f[4] + T(7042) * f[5] - T(1854) * f[6])
            + f[4] * (T(11003) * f[4] - T(17246) * f[5] + T(4642) * f[6])
            + f[5] * (T(7043) * f[5] - T(3882) * f[6]) + T(547) * f[6] * f[6];
    }
    q[0] = T(-3.0 / 12.0) * f[0] + T(13.0 / 12.0) * f[1] + T(-23.0 / 12.0) * f[2] + T(25.0 / 12.0) * f[3];
    q[1] = T(1.0 / 12.0) * f[1] + T(-5.0 / 12.0) * f[2] + T(13.0 / 12.0) * f[3] + T(3.0 / 12.0) * f[4];
    q[2] = T(-1.0 / 12.0) * f[2] + T(7.0 / 12.0) * f[3] + T(7.0 / 12.0) * f[4] + T(-1.0 / 12.0) * f[5];
    q[3] = T(3.0 / 12.0) * f[3] + T(13.0 / 12.0) * f[4] + T(-5.0 / 12.0) * f[5] + T(1.0 / 12.0) * f[6];
    b[0] = is0; b[1] = is1; b[2] = is2; b[3] = is3;
}

// The Z-weighted value of that stencil (eps 1e-20: src/weno7js.cpp:119-133,
// src/hccs78.cpp:246-304; 1e-40: the hccs closures, src/hccs.cpp:85-135).
// T: indicators and candidate values; TW: the nonlinear weights (they square
// tau/(eps+is) with eps 1e-20/1e-40, outside FP32's range).
// X receives the sum of the unnormalised weights less 1, sum c_k t_k^2 with
// t_k = tau/(eps+is_k), formed without the cancellation of that difference;
// the hccs family blends by theta = 1/(1 + X^2).
// Bound by FP64 issue: the eight IEEE quotients of the plain form are about
// 90 of a row's 210 instructions.  Here the four t_k share two reciprocals
// (of is_0 is_1 and is_2 is_3, whose products stay in range: eps^2 >= 1e-80)
// and the normalisation is one.  Errors over random and smooth indicators
// against 80-bit: 1.3e-16 rms in both forms.
template <typename T, typename TW>
__device__ __forceinline__ TW weno7z(const T *f, TW eps, TW &X)
{
    T is[4], q[4];
    weno7_stencil<T>(f, is, q);
    const TW s0 = eps + TW(is[0]), s1 = eps + TW(is[1]), s2 = eps + TW(is[2]), s3 = eps + TW(is[3]);
    const TW tau = fabs(TW(is[0]) - TW(is[3]));
    if constexpr (sizeof(T) == 4) {
        // FP32 stencils: the plain form, rounded as its IEEE quotients are (see
        // frcp_for), with a shared reciprocal for the four of the normalisation.
        // An indicator beyond FP32's range counts as 1e280 (weight c_k).
#pragma clang fp contract(off)
        auto t = [&](TW sk) {
            const TW x = fmin(sk, TW(1.0e280));
            return fquot(tau, x, frcp_for<true>(x));
        };
        const TW a0 = TW(1.0 / 35.0) * (TW(1) + sq(t(s0))), a1 = TW(12.0 / 35.0) * (TW(1) + sq(t(s1)));
        const TW a2 = TW(18.0 / 35.0) * (TW(1) + sq(t(s2))), a3 = TW(4.0 / 35.0) * (TW(1) + sq(t(s3)));
        const TW as = a0 + a1 + a2 + a3, ra = frcp_for<true>(as);
        X = as - TW(1);
        return fquot(a0, as, ra) * TW(q[0]) + fquot(a1, as, ra) * TW(q[1]) + fquot(a2, as, ra) * TW(q[2]) + fquot(a3, as, ra) * TW(q[3]);
    }
    const TW r01 = tau * frcp(s0 * s1), r23 = tau * frcp(s2 * s3);
    const TW x0 = TW(1.0 / 35.0) * sq(r01 * s1), x1 = TW(12.0 / 35.0) * sq(r01 * s0);
    const TW x2 = TW(18.0 / 35.0) * sq(r23 * s3), x3 = TW(4.0 / 35.0) * sq(r23 * s2);
    X = (x0 + x1) + (x2 + x3);
    const TW a0 = TW(1.0 / 35.0) + x0, a1 = TW(12.0 / 35.0) + x1;
    const TW a2 = TW(18.0 / 35.0) + x2, a3 = TW(4.0 / 35.0) + x3;
    return (a0 * TW(q[0]) + a1 * TW(q[1]) + a2 * TW(q[2]) + a3 * TW(q[3])) * frcp((a0 + a1) + (a2 + a3));
}

template <typename T, typename TW>
__device__ __forceinline__ TW weno7z(const T *f, TW eps)
{
    TW X;
    return weno7z<T, TW>(f, eps, X);
}

// hccs78, src/hccs78.cpp:66-117: on the inner interfaces the WENO7-Z value w
// (eps 1e-20) blended with the 8-point central value q8 through
// theta = 1/(1 + X^2), i.e. (X^2 w + q8)/(1 + X^2); on the edge interfaces w
// alone (:207-304).  One WENO7-Z evaluation serves both.
// f[0..7]: one downwind point more than WENO7.
template <typename T, typename TW>
__device__ __forceinline__ TW hccs78_value(const T *f, bool edge)
{
    TW X;
    const TW w = weno7z<T, TW>(f, TW(1.0e-20), X);
    const TW q8 = (TW(-3) * (TW(f[7]) + TW(f[0])) + TW(29) * (TW(f[6]) + TW(f[1])) - TW(139) * (TW(f[5]) + TW(f[2]))
                   + TW(533) * (TW(f[4]) + TW(f[3]))) * TW(1.0 / 840.0);
    const TW theta = frcp(TW(1) + sq(X));
    return edge ? w : w + theta * (q8 - w);
}

// hccs77 row, src/hccs77.cpp:86-163 (explicit rows :349-455): the 7th-order
// upwind compact row, and where theta = 1/(1 + X^2) <= 0.5 (X >= 1) its blend
// with the explicit WENO7-Z row w.  Every row is scaled by 1 + X^2 = 1/theta,
// which leaves the solution unchanged: compact row + X^2 (x = w).
// f[0..6]; TW: weights and the row.
template <typename T, typename TW>
__device__ __forceinline__ void hccs77_row(const T *f, bool expl, TW &lo, TW &di, TW &hi, TW &rhs)
{
    TW X;
    const TW w = weno7z<T, TW>(f, TW(1.0e-20), X);
    const TW q7 = (-TW(f[1]) + TW(19) * TW(f[2]) + TW(239) * TW(f[3]) + TW(159) * TW(f[4]) + TW(4) * TW(f[5])) * TW(1.0 / 420.0);
    const TW s = X < TW(1) ? TW(0) : sq(X);
    lo = expl ? TW(0) : TW(2.0 / 7.0);
    di = expl ? TW(1) : TW(4.0 / 7.0) + s;
    hi = expl ? TW(0) : TW(1.0 / 7.0);
    rhs = expl ? w : q7 + s * w;
}

// WENO3-JS, src/weno3js.cpp:80-93 (eps 1e-6): f[0..2] upwind
template <typename T, typename TW>
__device__ __forceinline__ TW weno3js(const T *f)
{
    T is0 = sq(f[0] - f[1]), is1 = sq(f[1] - f[2]);
    T q0 = T(-0.5) * f[0] + T(1.5) * f[1];
    T q1 = T(0.5) * f[1] + T(0.5) * f[2];
    TW a0 = TW(1.0 / 3.0) / sq(TW(1.0e-6) + TW(is0));
    TW a1 = TW(2.0 / 3.0) / sq(TW(1.0e-6) + TW(is1));
    return (a0 * TW(q0) + a1 * TW(q1)) / (a0 + a1);
}

// hccs interior row, src/hccs.cpp:138-183: Z-type CRWENO weights (eps 1e-40)
// blended with the 7th-order upwind compact scheme through theta.
// b0, b1, b2: four times the smoothness indicators; f0..f4 the stencil.
// T: indicators and stencil values; TW: weights and the row.
// With S_k = (is_k + eps)^2 the unnormalised weights are c_k (S_k + tau^2)/S_k.
// Their sum less 1 is X = tau^2 sum_k c_k prod_{j!=k} S_j / (S_0 S_1 S_2),
// theta = 1/(1 + X^2) and the CRWENO row's factor (1 - theta)/theta = X^2:
// two reciprocals in place of seven quotients.  X^2 holds fluxes up to about 1e17
// beside indicators of zero, the products 1e22 (LineScale keeps them below 1e14).
template <typename T, typename TW>
__device__ __forceinline__ void hccs_row(T f0, T f1, T f2, T f3, T f4, T b0, T b1, T b2, TW &lo, TW &di, TW &hi, TW &rhs)
{
    const TW eps = TW(4.0e-40);
    T q7 = T(-1.0 / 420.0) * f0 + T(19.0 / 420.0) * f1 + T(239.0 / 420.0) * f2 + T(159.0 / 420.0) * f3 + T(4.0 / 420.0) * f4;
    const TW S0 = sq(TW(b0) + eps), S1 = sq(TW(b1) + eps), S2 = sq(TW(b2) + eps);
    const TW T2 = sq(TW(b2) - TW(b0));
    const TW P12 = S1 * S2;
    const TW p0 = TW(0.2) * P12, p1 = TW(0.5) * (S0 * S2), p2 = TW(0.3) * (S0 * S1);
    const TW X = (T2 * (p0 + p1 + p2)) * frcp(S0 * P12);
    const TW n0 = (S0 + T2) * p0, n1 = (S1 + T2) * p1, n2 = (S2 + T2) * p2;
    // theta > 0.5 (X < 1): the compact row alone
    const TW s = X < TW(1) ? TW(0) : sq(X) * frcp(n0 + n1 + n2);
    const TW w0 = n0 * s, w1 = n1 * s, w2 = n2 * s;
    const TW F1 = f1, F2 = f2, F3 = f3;
    lo = (TW(2.0 / 3.0) * w0 + TW(1.0 / 3.0) * w1) + TW(2.0 / 7.0);
    di = (TW(1.0 / 3.0) * w0 + TW(2.0 / 3.0) * (w1 + w2)) + TW(4.0 / 7.0);
    hi = TW(1.0 / 3.0) * w2 + TW(1.0 / 7.0);
    rhs = (w0 * F1 + (TW(5) * (w0 + w1) + w2) * F2 + (w1 + TW(5) * w2) * F3) * TW(1.0 / 6.0) + TW(q7);
}

}  // namespace nucdev
