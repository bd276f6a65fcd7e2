// qlskum_math.h -- per-point q-LSKUM arithmetic shared by the HIP kernels.
//
// Every routine keeps the reference's expression order (Fortran a+b+c is
// (a+b)+c, a*b*c is (a*b)*c) and kernels_fp64.hip is compiled with
// -ffp-contract=off, so what it takes from here differs from the reference CPU
// build only by the device exp/log/erf (ocml vs glibc, within an ulp or two);
// its q-derivatives and time step are written apart, with fused multiply-adds.
// The sync-free sweeps take the sweep form of the split fluxes (SWEEP below:
// one refined quotient and root), the fused flux kernel its own forms
// (kernels_flux_fused.hip), and both units -ffp-contract=on (a*b + c fused
// within an expression, identically at every call site).
// Routines are templated on the arithmetic type T so the mixed-precision
// kernels reuse them with float, where division, square root and erf take
// the faster forms defined below.
#pragma once

#include <hip/hip_runtime.h>

namespace mfcfd {

// limiters.f90:26,28 compare |del_neg| with the REAL(4) literal 10e-6
constexpr double kLimiterThreshold = (double)10e-6f;

template <typename T> __device__ __forceinline__ T dexp(T x);
template <> __device__ __forceinline__ double dexp<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float dexp<float>(float x) { return __expf(x); }
template <typename T> __device__ __forceinline__ T dlog(T x);
template <> __device__ __forceinline__ double dlog<double>(double x) { return log(x); }
template <> __device__ __forceinline__ float dlog<float>(float x) { return __logf(x); }
template <typename T> __device__ __forceinline__ T dabs(T x) { return x < T(0) ? -x : x; }

// Division, square root and error function of the arithmetic type T.  FP64
// keeps IEEE division and square root and the library erf: the reference's
// arithmetic.  The mixed form's FP32 takes the hardware reciprocal and
// square root (v_rcp_f32, v_sqrt_f32: 1 ulp) and its own erf below; every
// argument here is a normal number.
template <typename T> __device__ __forceinline__ T ddiv(T a, T b);
template <> __device__ __forceinline__ double ddiv<double>(double a, double b) { return a / b; }
template <> __device__ __forceinline__ float ddiv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <typename T> __device__ __forceinline__ T dsqrt_fast(T x);
template <> __device__ __forceinline__ double dsqrt_fast<double>(double x) { return __builtin_sqrt(x); }
template <> __device__ __forceinline__ float dsqrt_fast<float>(float x) { return __builtin_amdgcn_sqrtf(x); }

// erf(x), given ex = exp(-x*x), which every flux caller forms anyway.
// FP32: for |x| < 0.5 the Maclaurin series of erf to x^13 (truncation
// < 2e-8); above it Abramowitz & Stegun 7.1.26, erf = 1 - t*(a1 + t*(a2 +
// t*(a3 + t*(a4 + t*a5))))*ex with t = 1/(1 + p|x|) (|error| <= 1.5e-7).
// In FP32 arithmetic the pair stays within 4e-7 of erf over all x; both
// branches are evaluated and one selected, so lanes do not diverge.
template <typename T> __device__ __forceinline__ T derf_e(T x, T ex);
// FP64 erf is kept out of line (list-by-list and level kernels): inlined, the
// library routine's working registers add to everything live around it
__device__ __attribute__((noinline)) inline double erf_out_of_line(double x) { return erf(x); }
template <> __device__ __forceinline__ double derf_e<double>(double x, double) { return erf_out_of_line(x); }
// a/b for normal b: the reciprocal estimate (v_rcp_f64, about 2^-23) refined by
// one Newton step, and the quotient by its residual.  Half an ulp beyond
// rounding, in 6 instructions instead of some 11.
__device__ __forceinline__ double div_refined(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = fma(r, fma(-b, r, 1.0), r);
    const double q = a * r;
    return fma(r, fma(-b, q, a), q);
}

// y ~ 1/sqrt(x) and h = x*y, with e = 1 - x*y*y to double-double accuracy, so
// that 1/sqrt(x) = y*(1 + e/2), sqrt(x) = h*(1 + e/2), 1/x = y*y*(1 + e), up
// to e*e < 2^-80: every power of x wanted is one product and one correction
// away.  The estimate (v_rsq_f64, about 2^-23) and one Newton step.
struct RootOf {
    double y, h, e;
};
__device__ __forceinline__ RootOf root_of(double x) {
    RootOf o;
    const double y0 = __builtin_amdgcn_rsq(x);
    const double h0 = x * y0;
    o.y = fma(0.5 * y0, fma(-h0, y0, 1.0), y0);
    o.h = x * o.y;
    o.e = fma(-fma(x, o.y, -o.h), o.y, fma(-o.h, o.y, 1.0));
    return o;
}
__device__ __forceinline__ double sqrt_of(const RootOf& r) { return fma(0.5 * r.h, r.e, r.h); }
// c/sqrt(x)
__device__ __forceinline__ double rsqrt_of(const RootOf& r, double c) {
    const double v = c * r.y;
    return fma(0.5 * v, r.e, v);
}

// The part of a split flux that depends on beta = 0.5*rho/p: sb = sqrt(beta),
// and what half_range takes B from.  SWEEP selects the sweep form, for
// kernels whose flux evaluations sit on a dependency chain: in FP64 one
// refined quotient and one root instead of IEEE divisions and square roots
// (1M FP64 sweep 9.0 -> 8.8 ms), and the library erf inlined: registers are
// spare there.  (erf_exp.h has fewer instructions but no shorter chain of
// them: 9.0 ms.)  FP32 is the same in both forms.
template <typename T>
struct BetaTerms {
    T beta, sb, hb;   // hb: 0.5/sqrt(pi*beta), FP64 sweep form only
};
template <typename T, bool SWEEP>
__device__ __forceinline__ BetaTerms<T> beta_terms(T rho, T pr) {
    BetaTerms<T> o;
    if constexpr (SWEEP && sizeof(T) == 8) {
        o.beta = div_refined(0.5 * rho, pr);
        const RootOf r = root_of(o.beta);
        o.sb = sqrt_of(r);
        o.hb = rsqrt_of(r, 0.28209479177387814);   // 0.5/sqrt(pi)
    } else {
        o.beta = ddiv(T(0.5) * rho, pr);
        o.sb = dsqrt_fast(o.beta);
        o.hb = T(0);
    }
    return o;
}

// erf(S) and B = 0.5*exp(-S*S)/sqrt(pi*beta) of one component, S = u*sb
template <typename T, bool SWEEP>
__device__ __forceinline__ void half_range(T u, const BetaTerms<T>& bt, T pi, T& B, T& e) {
    const T S = u * bt.sb;
    T ex;
    if constexpr (SWEEP && sizeof(T) == 8) {
        ex = exp(-S * S);
        e = erf(S);
        B = ex * bt.hb;
    } else {
        ex = dexp(-S * S);
        B = ddiv(T(0.5) * ex, dsqrt_fast(pi * bt.beta));
        e = derf_e(S, ex);
    }
}
template <> __device__ __forceinline__ float derf_e<float>(float x, float ex) {
    const float ax = x < 0.0f ? -x : x;
    const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * ax);
    const float p =
        t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
    const float far = 1.0f - p * ex;
    // 2/sqrt(pi) * sum_n (-1)^n x^(2n+1) / (n! (2n+1)), n = 0..6
    const float x2 = ax * ax;
    float s = 1.2055332981789664e-4f;
    s = s * x2 - 8.548327023450852e-4f;
    s = s * x2 + 5.223977625442188e-3f;
    s = s * x2 - 2.6866170645131252e-2f;
    s = s * x2 + 1.1283791670955126e-1f;
    s = s * x2 - 3.7612638903183754e-1f;
    s = s * x2 + 1.1283791670955126f;
    const float r = ax < 0.5f ? ax * s : far;
    return x < 0.0f ? -r : r;
}

// The six symmetric sums of a weighted least-squares stencil and the 3x3
// Cramer solve every stencil of the reference uses
// (q_derivatives.f90:85-107, interior_flux_dGxpos.f90:115-123).
template <typename T>
struct Geo6 {
    T xx, yy, zz, xy, yz, zx;
};

template <typename T>
__device__ __forceinline__ T cramer_det(const Geo6<T>& g) {
    return g.xx * (g.yy * g.zz - g.yz * g.yz)
         - g.xy * (g.xy * g.zz - g.yz * g.zx)
         + g.zx * (g.xy * g.yz - g.yy * g.zx);
}

// numerator of solution component col for the right-hand side (a, b, c)
template <typename T>
__device__ __forceinline__ T cramer_num(const Geo6<T>& g, int col, T a, T b, T c) {
    if (col == 0)
        return a * (g.yy * g.zz - g.yz * g.yz)
             - b * (g.xy * g.zz - g.zx * g.yz)
             + c * (g.xy * g.yz - g.zx * g.yy);
    if (col == 1)
        return g.xx * (b * g.zz - g.yz * c)
             - g.xy * (a * g.zz - g.zx * c)
             + g.zx * (a * g.yz - g.zx * b);
    return g.xx * (g.yy * c - b * g.yz)
         - g.xy * (g.xy * c - a * g.yz)
         + g.zx * (g.xy * b - a * g.yy);
}

template <typename T>
struct Frame {
    T t1[3], t2[3], n[3];
};

// Half-range KFVS flux of split_fluxes.f90:11-308 along axis 0/1/2
// (tan1/tan2/nor), half-space sign +1/-1.  "x - y" of the negative variants
// is written "x + (-y)", which rounds identically.
template <typename T, bool SWEEP = false>
__device__ __forceinline__ void flux_half(int axis, int sign, const Frame<T>& f, const T prim[5],
                                          T pi, T G[5]) {
    const T rho = prim[0], u1 = prim[1], u2 = prim[2], u3 = prim[3], pr = prim[4];
    const T ut1 = f.t1[0] * u1 + f.t1[1] * u2 + f.t1[2] * u3;
    const T ut2 = f.t2[0] * u1 + f.t2[1] * u2 + f.t2[2] * u3;
    const T un = f.n[0] * u1 + f.n[1] * u2 + f.n[2] * u3;
    const T ua = axis == 0 ? ut1 : (axis == 1 ? ut2 : un);
    const BetaTerms<T> bt = beta_terms<T, SWEEP>(rho, pr);
    T B, e;
    half_range<T, SWEEP>(ua, bt, pi, B, e);
    const T A = T(0.5) * (sign > 0 ? T(1) + e : T(1) - e);
    const T Bs = sign > 0 ? B : -B;
    const T u_sqr = ut1 * ut1 + ut2 * ut2 + un * un;
    T temp1 = (ua * A + Bs);
    G[0] = rho * temp1;
    G[1] = rho * ut1 * temp1;
    G[2] = rho * ut2 * temp1;
    G[3] = rho * un * temp1;
    G[1 + axis] = pr * A + rho * ua * temp1;
    temp1 = T(2.5) * pr + T(0.5) * rho * u_sqr;
    const T tail = (temp1 + T(0.5) * pr) * B;
    G[4] = (temp1 + pr) * ua * A + (sign > 0 ? tail : -tail);
}

// Quarter-range fluxes of octant_fluxes.f90:9-442: axis 0/1, sign_a along
// that axis, sign_n = -1 wall family (A3neg, -B3), +1 outer family (A3pos).
template <typename T, bool SWEEP = false>
__device__ __forceinline__ void flux_octant(int axis, int sign_a, int sign_n, const Frame<T>& f,
                                            const T prim[5], T pi, T G[5]) {
    const T rho = prim[0], u1 = prim[1], u2 = prim[2], u3 = prim[3], pr = prim[4];
    const T ut1 = f.t1[0] * u1 + f.t1[1] * u2 + f.t1[2] * u3;
    const T ut2 = f.t2[0] * u1 + f.t2[1] * u2 + f.t2[2] * u3;
    const T un = f.n[0] * u1 + f.n[1] * u2 + f.n[2] * u3;
    const T ua = axis == 0 ? ut1 : ut2;
    const BetaTerms<T> bt = beta_terms<T, SWEEP>(rho, pr);
    T Ba, ea, B3, e3;
    half_range<T, SWEEP>(ua, bt, pi, Ba, ea);
    half_range<T, SWEEP>(un, bt, pi, B3, e3);
    const T Aa = T(0.5) * (sign_a > 0 ? T(1) + ea : T(1) - ea);
    const T A3 = T(0.5) * (sign_n > 0 ? T(1) + e3 : T(1) - e3);
    const T u_sqr = ut1 * ut1 + ut2 * ut2 + un * un;
    const T temp1 = (ua * Aa + (sign_a > 0 ? Ba : -Ba));
    G[0] = rho * temp1 * A3;
    if (axis == 0) {
        G[1] = (pr * Aa + rho * ut1 * temp1) * A3;
        G[2] = rho * ut2 * temp1 * A3;
    } else {
        G[1] = rho * ut1 * temp1 * A3;
        G[2] = (pr * Aa + rho * ut2 * temp1) * A3;
    }
    G[3] = rho * temp1 * (un * A3 + (sign_n > 0 ? B3 : -B3));
    const T temp2 = T(2.5) * pr + T(0.5) * rho * u_sqr;
    const T tb = (temp2 + T(0.5) * pr) * Ba;
    const T temp3 = (temp2 + pr) * ua * Aa + (sign_a > 0 ? tb : -tb);
    const T tn = T(0.5) * rho * un * B3 * temp1;
    G[4] = temp3 * A3 + (sign_n > 0 ? tn : -tn);
}

// flux family selector: 0 half-range, 1 wall octant (Gw), 2 outer octant (Go)
template <typename T, bool SWEEP = false>
__device__ __forceinline__ void flux_eval(int family, int axis, int sign, const Frame<T>& f,
                                          const T prim[5], T pi, T G[5]) {
    if (family == 0)
        flux_half<T, SWEEP>(axis, sign, f, prim, pi, G);
    else
        flux_octant<T, SWEEP>(axis, sign, family == 2 ? 1 : -1, f, prim, pi, G);
}

// limiters.f90:18-40 for one component, from del_neg = qtilde - q
template <typename T>
__device__ __forceinline__ T venkat_phi_dn(T del_neg, T q, T qmax, T qmin, T epsi2) {
    const T thr = T(kLimiterThreshold);
    if (dabs(del_neg) <= thr) return T(1);
    if (!(dabs(del_neg) > thr)) return T(1);  // NaN: the reference leaves phi unset
    const T del_pos = del_neg > T(0) ? qmax - q : qmin - q;
    T num = (del_pos * del_pos) + epsi2;
    num = num * del_neg + T(2) * del_neg * del_neg * del_pos;
    T den = del_pos * del_pos + T(2) * del_neg * del_neg;
    den = den + del_neg * del_pos + epsi2;
    den = den * del_neg;
    const T temp = ddiv(num, den);
    return temp < T(1) ? temp : T(1);
}

template <typename T>
__device__ __forceinline__ T venkat_phi(T qt, T q, T qmax, T qmin, T epsi2) {
    return venkat_phi_dn(qt - q, q, qmax, qmin, epsi2);
}

// qvariables_to_primitive_variables.f90:16-30
template <typename T>
__device__ __forceinline__ void qtilde_to_primitive(const T q[5], T prim[5]) {
    const T beta = -q[4] * T(0.5);
    const T temp = ddiv(T(0.5), beta);
    prim[1] = q[1] * temp;
    prim[2] = q[2] * temp;
    prim[3] = q[3] * temp;
    const T temp1 = q[0] + beta * (prim[1] * prim[1] + prim[2] * prim[2] + prim[3] * prim[3]);
    const T temp2 = temp1 - (dlog(beta) * T(2.5));
    prim[0] = dexp(temp2);
    prim[4] = prim[0] * temp;
}

// get_primitive_vector.f90:10-41 / conserved_to_primitive_vector.f90:10-42:
// local-frame conserved vector of a point -> global primitive vector
// (SWEEP: 1/rho as a refined quotient)
template <typename T, bool SWEEP = false>
__device__ __forceinline__ void conserved_to_prim(const T U[5], const Frame<T>& f, T prim[5]) {
    prim[0] = U[0];
    T temp;
    if constexpr (SWEEP && sizeof(T) == 8) temp = div_refined(1.0, U[0]);
    else temp = T(1) / U[0];
    const T u2 = f.t1[0] * U[1] + f.t2[0] * U[2] + f.n[0] * U[3];
    const T u3 = f.t1[1] * U[1] + f.t2[1] * U[2] + f.n[1] * U[3];
    const T u4 = f.t1[2] * U[1] + f.t2[2] * U[2] + f.n[2] * U[3];
    prim[1] = temp * u2;
    prim[2] = temp * u3;
    prim[3] = temp * u4;
    temp = prim[1] * prim[1] + prim[2] * prim[2] + prim[3] * prim[3];
    prim[4] = T(0.4) * (U[4] - T(0.5) * prim[0] * temp);
}

}  // namespace mfcfd
