// Device arithmetic of the uniform-grid path: equation of state, HLLC / low-Mach HLLC with the shock blend,
// TVD limiters, WENO3-Z / WENO5-Z, convective and viscous ghost states.
//
// Bit-for-bit rule: every expression keeps the operation order of the reference, the file is compiled with
// -ffp-contract=off (no multiply-add is fused) and min / max are the reference's compare-and-select forms
// (std::min(a, b) = (b < a) ? b : a, std::max(a, b) = (a < b) ? b : a). Division and square root are the
// IEEE-rounded ones of the compiler's default lowering. With these, FP64 results are the reference's bits.
//
// NV is the number of conserved variables carried: 5 in 3-D, 4 in 2-D. A 2-D field has rho*w = +0
// everywhere in the reference, and with w = 0 the first four components do not depend on it (w*w adds +0 to a
// non-negative sum), so the 2-D kernels drop the fifth plane and its arithmetic.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace fvg {

constexpr double kEosEps = 1e-10;    // Core.hpp:169
constexpr double kDenomEps = 1e-14;  // Schemes.cpp:63
constexpr double kMachEps = 1e-12;   // Schemes.cpp:65
constexpr double kDtEps = 1e-10;     // TimeScheme.cpp:20

// index of the momentum component along axis a in [rho, rho u, rho v, rho E, rho w]
__host__ __device__ constexpr int mom(int a) { return a == 0 ? 1 : (a == 1 ? 2 : 4); }

template <typename T> __device__ __forceinline__ T smin(T a, T b) { return (b < a) ? b : a; }
template <typename T> __device__ __forceinline__ T smax(T a, T b) { return (a < b) ? b : a; }

// Division and square root of the flux arithmetic. FP64: the IEEE-rounded operations (the reference's bits).
// FP32 (flux_precision = fp32): the hardware reciprocal and square root (about 1 ulp), two instructions instead of
// the ten of a correctly rounded sequence; the error of the FP32 mode is measured against the FP64 path.
__device__ __forceinline__ double dv(double a, double b) { return a / b; }
__device__ __forceinline__ float dv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double sq(double a) { return sqrt(a); }
__device__ __forceinline__ float sq(float a) { return __builtin_amdgcn_sqrtf(a); }

// x / 6 correctly rounded in two operations, for x = 0 or 2^-960 <= |x| <= 2^905: with 1/6 = a + b (a = RN(1/6) =
// (1/6)(1 - 2^-54), so b = 2^-54 / 6, whose double is b to 2^-107), RN(x a + RN(x b)) rounds x/6 with an error below
// 2^-105 |x/6|. x/6 = (M/3) 2^e for an integer significand M is either representable or M/3 leaves a remainder of 1/3
// or 2/3, which puts x/6 at least 1/6 ulp from every midpoint, so the result is the IEEE quotient. Zeros keep their
// sign. Below the range the quotient may be subnormal and a midpoint (x = 9 2^-1074 gives 2^-1074, the division
// 2 2^-1074); above it, or for non-finite x, the FMA can overflow or give NaN: callers keep the IEEE division there
// (value_in_range below, whose bounds are narrower than those that quot6 needs, range_fits_quot6).
__host__ __device__ __forceinline__ double quot6(double x) {
    constexpr double a = 1.0 / 6.0, b = 0x1p-54 / 6.0;
    return __builtin_fma(x, a, x * b);
}
// v is 0 or 2^-900 <= |v| <= 2^900: the numerators of WENO5-Z's candidates (sums of 2, 7 and 11 times such values)
// are then 0 or between 2^-952 and 2^905 in magnitude, inside the range of quot6. NaN is outside.
__host__ __device__ __forceinline__ bool range_fits_quot6(double v) {
    const double m = v < 0.0 ? -v : v;
    return (v == 0.0) | ((m >= 0x1p-900) & (m <= 0x1p+900));   // no short-circuit branches
}
// ---- FP64 operations whose operands are known to be in range (IR) ----
// The IEEE division of the compiler scales its operands (two v_div_scale), ends in v_div_fmas / v_div_fixup and so
// takes about 70 cycles of a SIMD per wavefront, the IEEE square root 85; the face kernels spend a third of their time
// in them. When neither operand needs the scaling (denominator and its reciprocal normal, quotient normal or zero,
// |numerator| >= 2^-969 or zero), scaling multiplies by one and the same reciprocal, Newton steps and correction
// give the same bits without it: 57 cycles with the fixup (which keeps zeros, infinities and NaN as IEEE has them), 52
// without it, 53 for the square root. (The compiler's division, and so these, misses the IEEE quotient by one ulp for a
// few operands within 2^-53 ulp of a midpoint with a divisor just below a power of two, for instance
// 0x1.6666666666663p+52 / 0x1.ffffffffffffbp+52.)
// The kernels take these forms when every primitive that k_cells stored is zero or between 2^-400 and 2^100 in
// magnitude (value_in_range; DevState::wide) and the configuration's constants are moderate (KP::ir). Then, with
// WENO5-Z (eps at least 2^-42 of the stencil's mean square): differences are zero or at least 2^-453, the smoothness
// indicators zero or at least 2^-908, tau zero or at least 2^-961, tau / (b + eps) at most 2^53, candidates zero or
// at least 2^-458 and the last quotient at least 2^-570; van Leer's 2 a b is at least 2^-906. The Riemann solver
// divides by densities and pressures of at least 1e-10 and by speed differences of at least 1e-14; its contact
// speed, whose numerator may be any small number, keeps the IEEE division.
// The advanced states of MUSCL-Hancock are not reconstructed values: they move with the half step, which a caller may
// choose (fvg_residual). An admissible one has a density above 1e-10 and an energy whose product with it bounds the
// momenta, so with both at most 2^200 (state_moderate, also DevState::wide) the momenta are at most 2^201, the
// velocities 2^235, the pressure 2^220, the sound speed between 2^-117 and 2^127, the contact speed's numerator at most
// 2^672 and its quotient 2^719, so that no speed is NaN; the solver's other denominators lie between 2^-47 and 2^720
// and its numerators are zero or at least 2^-204.
__device__ __forceinline__ double rcp_refined(double b) {   // the compiler's reciprocal: two Newton steps
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
// a / b from r = rcp_refined(b): zeros of a keep their sign for b > 0
__device__ __forceinline__ double quot_rcp(double a, double b, double r) {
    const double q = a * r;
    return __builtin_fma(-__builtin_fma(q, b, -a), r, q);
}
// a / b for b > 0 or a != 0, both finite
template <bool IR> __device__ __forceinline__ double dvp(double a, double b) {
    if constexpr (IR) return quot_rcp(a, b, rcp_refined(b));
    else return a / b;
}
template <bool IR> __device__ __forceinline__ float dvp(float a, float b) { return dv(a, b); }
// a / b, any zeros, infinities and NaN
template <bool IR> __device__ __forceinline__ double dvx(double a, double b) {
    if constexpr (IR) return __builtin_amdgcn_div_fixup(quot_rcp(a, b, rcp_refined(b)), b, a);
    else return a / b;
}
template <bool IR> __device__ __forceinline__ float dvx(float a, float b) { return dv(a, b); }
// the compiler's square root without its scaling of arguments below 2^-767 (zeros, infinities and NaN as IEEE has them)
template <bool IR> __device__ __forceinline__ double sqx(double x) {
    if constexpr (IR) {
        const double y = __builtin_amdgcn_rsq(x);
        double g = x * y, h = y * 0.5;
        const double r = __builtin_fma(-h, g, 0.5);
        g = __builtin_fma(g, r, g);
        h = __builtin_fma(h, r, h);
        g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
        g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
        return __builtin_amdgcn_class(x, 0x260) ? x : g;   // +-0 and +inf are their own roots
    } else {
        return sqrt(x);
    }
}
template <bool IR> __device__ __forceinline__ float sqx(float x) { return sq(x); }
// 1 / rho for a density above the floor of c2p (or NaN): only beyond 2^1000 does the division scale
__device__ __forceinline__ double recip_rho(double rho) {
    double r = dvx<true>(1.0, rho);
    if (rho > 0x1p+1000) r = 1.0 / rho;
    return r;
}
__device__ __forceinline__ float recip_rho(float rho) { return dv(1.0f, rho); }
// x / c for a constant c > 0 with inv = RN(1 / c): Markstein's correction (with a correctly rounded
// reciprocal the corrected quotient is the IEEE one for every significand of c); FP32: the product
template <bool IR> __host__ __device__ __forceinline__ double by_const(double x, double c, double inv) {
    if constexpr (IR) {
        const double q = x * inv;
        return __builtin_fma(-__builtin_fma(q, c, -x), inv, q);
    } else {
        return x / c;
    }
}
template <bool IR> __device__ __forceinline__ float by_const(float x, float c, double) { return dv(x, c); }
// k b + c for k a power of two: the product is exact (short of overflow and underflow), so one FMA rounds as the two
// operations do. EX<IR, T>: the operands are away from both ends (in-range FP64; FP32, whose error budget a last bit
// of a subnormal does not touch).
template <bool IR, typename T> constexpr bool EX = IR || std::is_same<T, float>::value;
template <bool X> __device__ __forceinline__ double p2fma(double k, double b, double c) { return X ? __builtin_fma(k, b, c) : k * b + c; }
template <bool X> __device__ __forceinline__ float p2fma(float k, float b, float c) { return __builtin_fmaf(k, b, c); }
// smin / smax of finite values that are not zeros of opposite sign: one instruction instead of a compare and two selects
template <bool IR> __device__ __forceinline__ double nmin(double a, double b) { return IR ? __builtin_fmin(a, b) : smin(a, b); }
template <bool IR> __device__ __forceinline__ double nmax(double a, double b) { return IR ? __builtin_fmax(a, b) : smax(a, b); }
template <bool IR> __device__ __forceinline__ float nmin(float a, float b) { return smin(a, b); }
template <bool IR> __device__ __forceinline__ float nmax(float a, float b) { return smax(a, b); }
__host__ __device__ __forceinline__ bool value_in_range(double v) {
    const double m = v < 0.0 ? -v : v;
    return (v == 0.0) | ((m >= 0x1p-400) & (m <= 0x1p+100));   // no short-circuit branches
}

// an admissible conservative state of MUSCL-Hancock's face fluxes, see above
__host__ __device__ __forceinline__ bool state_moderate(const double* u) { return (u[0] <= 0x1p+200) & (u[3] <= 0x1p+200); }

// the absolute floor of the WENO regularisation: 1e-300 in FP64 (Schemes.cpp:331, 343); the smallest power of ten
// above FLT_MIN in FP32, where 1e-300 would round to zero and 0/0 would reach the weights of an all-zero stencil
template <typename T> __device__ __forceinline__ T weno_floor() { return T(1e-300); }
template <> __device__ __forceinline__ float weno_floor<float>() { return 1e-37f; }

struct Eos {
    int stiff;
    double gamma, p_inf;
    double inv_g1;   // 1 / (gamma - 1), correctly rounded
};
inline Eos make_eos(bool stiff, double gamma, double p_inf) { return Eos{stiff ? 1 : 0, gamma, stiff ? p_inf : 0.0, 1.0 / (gamma - 1.0)}; }

// primitive [rho, u, v, p, w] -> conservative (Core.hpp:209-215)
template <int NV, bool IR = false, typename T>
__device__ __forceinline__ void p2c(const Eos& e, const T* W, T* U) {
    const T g = T(e.gamma);
    const T rho = W[0], u = W[1], v = W[2], p = W[3];
    const T en = by_const<IR>(!e.stiff ? p : p + g * T(e.p_inf), g - T(1.0), e.inv_g1);
    T m2 = u * u + v * v;
    if constexpr (NV == 5) {
        const T w = W[4];
        m2 = m2 + w * w;
        U[4] = rho * w;
    }
    U[0] = rho;
    U[1] = rho * u;
    U[2] = rho * v;
    if constexpr (EX<IR, T>) U[3] = p2fma<true>(T(0.5), rho * m2, en);   // en + (0.5 rho) m2
    else U[3] = en + T(0.5) * rho * m2;
}

// conservative -> primitive with the floors of Core.hpp:219-228; *inv = 1 / rho. PLAIN: the compiler's division instead of
// recip_rho, whose rare branch splits the code around it: k_ensemble, at its register limit, runs 6 % slower with it
// (1,024 instances to t = 0.05: 3.87 s plain, 4.10 with), the other kernels faster.
template <int NV, bool IR = false, bool PLAIN = false, typename T>
__device__ __forceinline__ void c2p(const Eos& e, const T* U, T* W, T* inv_out) {
    const T g = T(e.gamma);
    const T rho = nmax<IR>(U[0], T(kEosEps));
    const T inv = IR ? dvx<IR>(T(1.0), rho) : (PLAIN ? T(1.0) / rho : recip_rho(rho));
    if (inv_out) *inv_out = inv;
    const T u = U[1] * inv, v = U[2] * inv;
    T m2 = u * u + v * v;
    if constexpr (NV == 5) {
        const T w = U[4] * inv;
        m2 = m2 + w * w;
        W[4] = w;
    }
    T rho_e;   // U[3] - (0.5 rho) m2
    if constexpr (EX<IR, T>) rho_e = p2fma<true>(T(-0.5), rho * m2, U[3]);
    else rho_e = U[3] - T(0.5) * rho * m2;
    const T p = !e.stiff ? (g - T(1.0)) * rho_e : (g - T(1.0)) * rho_e - g * T(e.p_inf);
    W[0] = rho;
    W[1] = u;
    W[2] = v;
    W[3] = nmax<IR>(p, T(kEosEps));
}

template <typename T>
__device__ __forceinline__ T sound_speed(const Eos& e, T p, T rho) {
    if (!e.stiff) return sq(dv(T(e.gamma) * smax(p, T(kEosEps)), smax(rho, T(kEosEps))));
    return sq(dv(T(e.gamma) * (p + T(e.p_inf)), smax(rho, T(kEosEps))));
}
template <bool IR = false, typename T>
__device__ __forceinline__ T sound_speed_inv(const Eos& e, T p, T inv_rho) {
    if (!e.stiff) return sqx<IR>(T(e.gamma) * nmax<IR>(p, T(kEosEps)) * inv_rho);
    return sqx<IR>(T(e.gamma) * (p + T(e.p_inf)) * inv_rho);
}

template <int NV, typename T>
__device__ __forceinline__ void roundtrip(const Eos& e, T* U) {
    T W[NV];
    c2p<NV>(e, U, W, (T*)nullptr);
    p2c<NV>(e, W, U);
}

template <bool IR = false, typename T> __device__ __forceinline__ T safe_denom(T x) { return copysign(nmax<IR>(fabs(x), T(kDenomEps)), x); }

struct RiemannParams {
    Eos eos;
    int lowmach;
    double blend;
};

// the flux of a state normal to axis, and the side's factor of its star state and that state
template <int NV, typename T>
__device__ __forceinline__ void state_flux(const T* W, T E, int axis, T* F) {
    const int mn = mom(axis);
    const T rho = W[0], p = W[3], Vn = W[mn];
    F[0] = rho * Vn;
#pragma unroll
    for (int a = 0; a < NV - 2; ++a) F[mom(a)] = rho * W[mom(a)] * Vn;
    F[mn] = F[mn] + p;
    F[3] = Vn * (rho * E + p);
}
template <int NV, bool IR, typename T>
__device__ __forceinline__ void star_state(const T* W, T E, T S, T S_M, int axis, T* Us) {
    const T rho = W[0], p = W[3], Vn = W[mom(axis)];
    const T f = dvx<IR>(rho * (S - Vn), safe_denom<IR>(S - S_M));
    Us[0] = f;
#pragma unroll
    for (int a = 0; a < NV - 2; ++a) Us[mom(a)] = f * (a == axis ? S_M : W[mom(a)]);
    Us[3] = f * (E + (S_M - Vn) * (S_M + dvx<IR>(p, rho * safe_denom<IR>(S - Vn))));
}

// HLLC with Einfeldt bounds, the contact speed of Toro (10.37) and the shock blend toward HLL
// (Schemes.cpp:116-200). vel index a = 0, 1, 2 maps to W[1], W[2], W[4].
// The flux of a face comes from one side of its contact: the side is picked first, by selecting its eleven or so
// inputs, and only that side's flux, star state and two of its quotients are computed; the reference computes both
// and picks the result. Which side its four successive conditions leave: the right one when S_R < 0 or
// S_M < 0 <= S_R, else the left one, and zero when none of them holds (NaN speeds).
// BOTH: as the reference, for k_ensemble, which waits for a face's chain of operations rather than for their number:
// all that does not need the contact speed is on its way beside its quotient (1,024 instances to t = 0.03: 2.34-2.36 s,
// 2.38-2.42 with one side; 600 of 4,000 cells, 60 steps: MUSCL at 768 threads 12.0 ms against 12.6, WENO5 at 256 32.5
// against 33.6). Its first-order faces and 1,024-thread workgroups, which spill, take one (4.5 against 4.8 ms; MUSCL 13.8
// against 14.2).
template <int NV, bool IR = false, bool BOTH = false, typename T>
__device__ __forceinline__ void hllc_core(const RiemannParams& rs, const T* WL, const T* WR, const T* UL, const T* UR, T inv_L,
                                          T inv_R, T c_L, T c_R, int axis, T* F, T& smax_out) {
    const T rho_L = WL[0], p_L = WL[3];
    const T rho_R = WR[0], p_R = WR[3];
    const int mn = mom(axis);
    const T Vn_L = WL[mn], Vn_R = WR[mn];
    const T S_L = nmin<IR>(Vn_L - c_L, Vn_R - c_R);
    const T S_R = nmax<IR>(Vn_L + c_L, Vn_R + c_R);
    const T num = rho_R * Vn_R * (S_R - Vn_R) - rho_L * Vn_L * (S_L - Vn_L) + p_L - p_R;
    const T den = rho_R * (S_R - Vn_R) - rho_L * (S_L - Vn_L);
    const T S_M = dv(num, safe_denom<IR>(den));
    T Fo[NV];
    if constexpr (BOTH) {
        T FL[NV], FR[NV], UsL[NV], UsR[NV];
        const T E_L = UL[3] * inv_L, E_R = UR[3] * inv_R;
        state_flux<NV>(WL, E_L, axis, FL);
        state_flux<NV>(WR, E_R, axis, FR);
        star_state<NV, IR>(WL, E_L, S_L, S_M, axis, UsL);
        star_state<NV, IR>(WR, E_R, S_R, S_M, axis, UsR);
#pragma unroll
        for (int q = 0; q < NV; ++q) Fo[q] = T(0);
        if (S_L >= T(0))
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = FL[q];
        if (S_L < T(0) && S_M >= T(0))
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = FL[q] + S_L * (UsL[q] - UL[q]);
        if (S_M < T(0) && S_R >= T(0))
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = FR[q] + S_R * (UsR[q] - UR[q]);
        if (S_R < T(0))
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = FR[q];
    } else {
        const bool right = (S_R < T(0)) | ((S_M < T(0)) & (S_R >= T(0)));
        const bool star = right ? S_R >= T(0) : (S_L < T(0)) & (S_M >= T(0));
        const bool none = !IR & !right & !star & !(S_L >= T(0));   // not with finite speeds
        T W[NV], U[NV], Us[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            W[q] = right ? WR[q] : WL[q];
            U[q] = right ? UR[q] : UL[q];
        }
        const T S = right ? S_R : S_L, E = U[3] * (right ? inv_R : inv_L);
        state_flux<NV>(W, E, axis, Fo);
        star_state<NV, IR>(W, E, S, S_M, axis, Us);
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const T s = Fo[q] + S * (Us[q] - U[q]);
            Fo[q] = star ? s : Fo[q];
        }
        if (none)
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = T(0);
    }
    if (rs.blend > 0.0) {
        const T blend = T(rs.blend);
        const T s = dvx<IR>(fabs(p_R - p_L), nmin<IR>(p_L, p_R));
        if (s > blend) {
            const T phi = smin(dv(s - blend, blend), T(1.0));
            T FL[NV], FR[NV];
            state_flux<NV>(WL, UL[3] * inv_L, axis, FL);
            state_flux<NV>(WR, UR[3] * inv_R, axis, FR);
            T Fh[NV];
            if (S_L >= T(0)) {
#pragma unroll
                for (int q = 0; q < NV; ++q) Fh[q] = FL[q];
            } else if (S_R <= T(0)) {
#pragma unroll
                for (int q = 0; q < NV; ++q) Fh[q] = FR[q];
            } else {
                const T inv = dv(T(1.0), S_R - S_L);
#pragma unroll
                for (int q = 0; q < NV; ++q) Fh[q] = (S_R * FL[q] - S_L * FR[q] + S_L * S_R * (UR[q] - UL[q])) * inv;
            }
#pragma unroll
            for (int q = 0; q < NV; ++q) Fo[q] = (T(1.0) - phi) * Fo[q] + phi * Fh[q];
        }
    }
    smax_out = nmax<IR>(fabs(S_L), fabs(S_R));
#pragma unroll
    for (int q = 0; q < NV; ++q) F[q] = Fo[q];
}

// RiemannSolver::face_flux (Schemes.cpp:108-113, 202-229). One hllc_core for both solvers (its code is inlined once):
// the low-Mach variant blends the velocities first.
template <int NV, bool IR = false, bool PLAIN = false, bool BOTH = false, typename T>
__device__ __forceinline__ void face_flux(const RiemannParams& rs, const T* UL0, const T* UR0, int axis, T* F, T& sm) {
    T WL[NV], WR[NV], UL[NV], UR[NV], inv_L, inv_R;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        UL[q] = UL0[q];
        UR[q] = UR0[q];
    }
    c2p<NV, IR, PLAIN>(rs.eos, UL, WL, &inv_L);
    c2p<NV, IR, PLAIN>(rs.eos, UR, WR, &inv_R);
    const T c_L = sound_speed_inv<IR>(rs.eos, WL[3], inv_L);
    const T c_R = sound_speed_inv<IR>(rs.eos, WR[3], inv_R);
    if constexpr (BOTH)
        if (!rs.lowmach) {
            hllc_core<NV, IR, true>(rs, WL, WR, UL0, UR0, inv_L, inv_R, c_L, c_R, axis, F, sm);
            return;
        }
    if (rs.lowmach) {
        T ML2 = WL[1] * WL[1] + WL[2] * WL[2], MR2 = WR[1] * WR[1] + WR[2] * WR[2];
        if constexpr (NV == 5) {
            ML2 = ML2 + WL[4] * WL[4];
            MR2 = MR2 + WR[4] * WR[4];
        }
        const T M_L = dvx<IR>(sq(ML2), c_L + T(kMachEps));
        const T M_R = dvx<IR>(sq(MR2), c_R + T(kMachEps));
        const T z = smin(smax(smax(M_L, M_R), T(1e-4)), T(1.0));
#pragma unroll
        for (int a = 0; a < NV - 2; ++a) {
            const int m = mom(a);
            const T avg = T(0.5) * (WL[m] + WR[m]);
            const T half = T(0.5) * (WL[m] - WR[m]);
            WL[m] = avg + z * half;
            WR[m] = avg - z * half;
        }
        p2c<NV, IR>(rs.eos, WL, UL);
        p2c<NV, IR>(rs.eos, WR, UR);
    }
    hllc_core<NV, IR, BOTH>(rs, WL, WR, UL, UR, inv_L, inv_R, c_L, c_R, axis, F, sm);
}

// ---- limiters (Schemes.hpp:90-117) and WENO-Z (Schemes.cpp:323-353) ----
template <typename T> __device__ __forceinline__ T sgn(T x) { return (x > T(0)) ? T(1) : ((x < T(0)) ? T(-1) : T(0)); }

template <bool IR = false, typename T>
__device__ __forceinline__ T limiter(int l, T a, T b) {
    switch (l) {
    case 0: return T(0.5) * (sgn(a) + sgn(b)) * smin(fabs(a), fabs(b));
    case 1: {
        const T ab = a * b;
        return (ab > T(0)) ? dvp<IR>(T(2.0) * ab, a + b) : T(0.0);
    }
    case 2:
        if (!(a * b > T(0))) return T(0.0);
        return smin(smin(T(2.0) * fabs(a), T(0.5) * fabs(a + b)), T(2.0) * fabs(b)) * sgn(a);
    default:
        if (!(a * b > T(0))) return T(0.0);
        return fmin(fmin(T(2.0) * fabs(a), by_const<IR>(fabs(T(2.0) * a + b), T(3.0), 1.0 / 3.0)), T(2.0) * fabs(b)) * sgn(a);
    }
}

template <typename T, bool IR = false>
__device__ __forceinline__ T weno3z(T c0, T c1, T c2, T eps_rel) {
    const T eps = eps_rel * (c0 * c0 + c1 * c1 + c2 * c2) * T(1.0 / 3.0) + weno_floor<T>();
    const T v0 = T(-0.5) * c0 + T(1.5) * c1, v1 = T(0.5) * c1 + T(0.5) * c2;
    const T b0 = (c1 - c0) * (c1 - c0), b1 = (c2 - c1) * (c2 - c1);
    const T tau = fabs(b0 - b1);
    const T a0 = T(1.0 / 3.0) * (T(1.0) + dvp<IR>(tau, b0 + eps)), a1 = T(2.0 / 3.0) * (T(1.0) + dvp<IR>(tau, b1 + eps));
    return dvp<IR>(a0 * v0 + a1 * v1, a0 + a1);
}

// the candidates' quotients by 6: the IEEE division, or quot6 (the same bits) in range
template <bool IR, typename T> __device__ __forceinline__ T by6(T x) {
    if constexpr (IR && std::is_same<T, double>::value) return quot6(x);
    else return dv(x, T(6.0));
}

// Products by 2, 4 and 1/4 are exact, so they share an FMA with the sum they enter (p2fma: the same bits): 188
// operations and 8 reciprocals for the two values of a face and variable.
template <typename T, bool IR = false>
__device__ __forceinline__ T weno5z(T c0, T c1, T c2, T c3, T c4, T eps_rel) {
    constexpr bool X = EX<IR, T>;
    const T eps = eps_rel * (c0 * c0 + c1 * c1 + c2 * c2 + c3 * c3 + c4 * c4) * T(0.2) + weno_floor<T>();
    const T p0 = by6<IR>(p2fma<X>(T(2.0), c0, -(T(7.0) * c1)) + T(11.0) * c2);
    const T p1 = by6<IR>(p2fma<X>(T(2.0), c3, T(5.0) * c2 - c1));
    const T p2 = by6<IR>(p2fma<X>(T(2.0), c2, T(5.0) * c3) - c4);
    const T s0 = p2fma<X>(T(-2.0), c1, c0) + c2, t0 = p2fma<X>(T(-4.0), c1, c0) + T(3.0) * c2;
    const T s1 = p2fma<X>(T(-2.0), c2, c1) + c3, t1 = c1 - c3;
    const T s2 = p2fma<X>(T(-2.0), c3, c2) + c4, t2 = p2fma<X>(T(-4.0), c3, T(3.0) * c2) + c4;
    T b0, b1, b2;
    if constexpr (X) {
        b0 = p2fma<X>(T(0.25), t0 * t0, T(13.0 / 12.0) * s0 * s0);
        b1 = p2fma<X>(T(0.25), t1 * t1, T(13.0 / 12.0) * s1 * s1);
        b2 = p2fma<X>(T(0.25), t2 * t2, T(13.0 / 12.0) * s2 * s2);
    } else {
        b0 = T(13.0 / 12.0) * s0 * s0 + T(0.25) * t0 * t0;
        b1 = T(13.0 / 12.0) * s1 * s1 + T(0.25) * t1 * t1;
        b2 = T(13.0 / 12.0) * s2 * s2 + T(0.25) * t2 * t2;
    }
    const T tau = fabs(b0 - b2);
    const T a0 = T(0.1) * (T(1.0) + dvp<IR>(tau, b0 + eps)), a1 = T(0.6) * (T(1.0) + dvp<IR>(tau, b1 + eps)),
            a2 = T(0.3) * (T(1.0) + dvp<IR>(tau, b2 + eps));
    return dvp<IR>(a0 * p0 + a1 * p1 + a2 * p2, a0 + a1 + a2);
}

// ---- convective ghost state (Boundaries.cpp:106-153) ----
struct BcParams {
    int bc[6];
    double u_in, v_in, p_out;
    double rho_in;                   // mass-flow inlet density
    double nrbc_sigma, nrbc_beta;    // non-reflecting outlet: relaxation towards p_out, transverse weight
    double length[3];                // domain size per axis (the non-reflecting relaxation length)
    const double* ut;                // mass-flow inlet velocity per side, set on the device each residual (or null)
};

// The boundary type of a side, without indexing the parameter array by a run-time value (that would put the
// kernel arguments in scratch memory).
__device__ __forceinline__ int bc_of(const BcParams& b, int side) {
    switch (side) {
    case 0: return b.bc[0];
    case 1: return b.bc[1];
    case 2: return b.bc[2];
    case 3: return b.bc[3];
    case 4: return b.bc[4];
    default: return b.bc[5];
    }
}

// side: 0 left, 1 right, 2 bottom, 3 top, 4 front, 5 back. Periodic and non-reflecting sides never reach here; a
// mass-flow side reads its target velocity from b.ut (set by k_sides before the residual's first pass).
template <int NV>
__device__ __forceinline__ void ghost_state(const Eos& e, const BcParams& b, int side, const double* Ui, double* Ug) {
    const int bc = bc_of(b, side);
    if (bc == 6 /* transmissive */) {
#pragma unroll
        for (int q = 0; q < NV; ++q) Ug[q] = Ui[q];
        return;
    }
    const int axis = side / 2;
    const double nxn = axis == 0 ? 1.0 : 0.0, nyn = axis == 1 ? 1.0 : 0.0, nzn = axis == 2 ? 1.0 : 0.0;
    double Wi[NV], Wg[NV];
    c2p<NV>(e, Ui, Wi, (double*)nullptr);
#pragma unroll
    for (int q = 0; q < NV; ++q) Wg[q] = Wi[q];
    const double wi4 = NV == 5 ? Wi[NV == 5 ? 4 : 0] : 0.0;
    if (bc == 0 /* wall */) {
        const double Vn = Wi[1] * nxn + Wi[2] * nyn + wi4 * nzn;
        Wg[1] = Wi[1] - 2.0 * Vn * nxn;
        Wg[2] = Wi[2] - 2.0 * Vn * nyn;
        if constexpr (NV == 5) Wg[4] = Wi[4] - 2.0 * Vn * nzn;
    } else if (bc == 1 /* no-slip */) {
        Wg[1] = -Wi[1];
        Wg[2] = -Wi[2];
        if constexpr (NV == 5) Wg[4] = -Wi[4];
    } else if (bc == 2 || bc == 3 /* moving wall, velocity inlet */) {
        Wg[1] = 2.0 * b.u_in - Wi[1];
        Wg[2] = 2.0 * b.v_in - Wi[2];
        if constexpr (NV == 5) Wg[4] = -Wi[4];
    } else if (bc == 4 /* mass-flow inlet: the side's target velocity */) {
        Wg[1] = 2.0 * b.ut[side] - Wi[1];
        Wg[2] = 2.0 * b.v_in - Wi[2];
        if constexpr (NV == 5) Wg[4] = -Wi[4];
    } else if (bc == 5 /* outlet */) {
        const double Vn = Wi[1] * nxn + Wi[2] * nyn + wi4 * nzn;
        const bool outflow = Vn >= 0;
        Wg[1] = outflow ? Wi[1] : 0.0;
        Wg[2] = outflow ? Wi[2] : 0.0;
        if constexpr (NV == 5) Wg[4] = outflow ? Wi[4] : 0.0;
        Wg[3] = smax(b.p_out, 1e-5);
    }
    p2c<NV>(e, Wg, Ug);
}

}   // namespace fvg
