// phx_numerics.hpp -- per-cell and per-face arithmetic of pyHype's second-order MUSCL scheme.
//
// Every function reproduces the reference's floating-point evaluation order exactly (left-to-right
// Python/Numba association, the COO storage order of the Roe eigen-system mat-vecs, no fused
// multiply-add).  The translation unit must be compiled with -ffp-contract=off; division and
// square root are the IEEE correctly-rounded operations.  The functions are __host__ __device__ so
// that the same source is checked against the CPU oracle on the host.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

namespace phx {

// A state or flux of 4 components.  The arithmetic below is written once for a scalar type T:
// T = double is the path every kernel runs; the tangent-linear kernels instantiate it with a
// value-and-derivative pair whose value part performs exactly the same double operations.
template <class T>
struct Q4T {
    T v[4];
};
using Q4 = Q4T<double>;

// Fluid constants, evaluated on the host exactly as the reference evaluates them:
// gm1 = gamma - 1 (states/conservative.py:110), one_over_gm1 = 1.0/(gamma - 1.0) and
// g_over_gm1 = gamma/(gamma - 1.0) (fluids/base.py:58-64).
struct Phys {
    double gamma, gm1, one_over_gm1, g_over_gm1, cfl;
    int limiter;  // PHX_LIMITER_* (0 = Venkatakrishnan)
    int prim;     // reconstruction in primitive variables (SolverConfig.reconstruction_type)
    int nq;       // Gauss points per face (SolverConfig.fvm_num_quadrature_points); 0 or 1: midpoint
    int odd_gas;  // gamma or gamma - 1 outside [2^-20, 2^20]: the in-range divisions below are not used
};

template <class T>
struct PrimT {
    T r, u, v, p;
};
using Prim = PrimT<double>;

// Whether x holds on every / on any active lane of the wave (on the host: x).  A rare case is handled by
// a branch of the whole wave, with the common path as the fall-through: on gfx950 a divergent `if`
// costs about 30 cycles of a wave's time (the compare's round trip into the execution mask and back)
// and a taken branch about 60 (14 with four waves on the SIMD), the price of 6 and 12 double
// operations.  Both evaluations give the same bits, so a lane may take the general one without need.
__host__ __device__ inline unsigned long long wave_lanes(bool x) {  // the lanes where x holds (host: 0 or 1)
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(x);
#else
    return x ? 1ull : 0ull;
#endif
}
__host__ __device__ inline bool wave_all(bool x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(!x) == 0ull;
#else
    return x;
#endif
}
__host__ __device__ inline bool wave_any(bool x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(x) != 0ull;
#else
    return x;
#endif
}
#define PHX_USUAL(x) __builtin_expect(!!(x), 1)
#define PHX_RARE(x) __builtin_expect(!!(x), 0)

__host__ __device__ inline Q4 q4zero() {
    Q4 q;
    q.v[0] = q.v[1] = q.v[2] = q.v[3] = 0.0;
    return q;
}

// IEEE division by a divisor whose magnitude, and that of the numerators, is known to be moderate.  The
// compiler's sequence for n / d scales d and n where their exponents are extreme (v_div_scale: a divisor or
// quotient that is not normal, a divisor whose reciprocal is not, quotients from 2^768, numerators below
// 2^-969), refines v_rcp_f64 by two Newton steps, forms q = n*y, the remainder r = n - d*q and q + r*y
// (v_div_fmas, which undoes the scaling), and replaces the result where an operand is zero, infinite or
// NaN or the quotient is not a normal number (v_div_fixup).  For 2^-1000 <= |d| <= 2^1000, |n| >= 2^-900 and
// |n / d| in [2^-760, 2^760] the scalings and that replacement are identities, the reciprocal and its
// refinement stay normal, and so does the remainder, a multiple of 2^-106 |n|; so the refinement
// alone gives the same bits: 8 instead of 11 instructions, no dependence on VCC between
// two divisions, and one reciprocal for all numerators of a divisor (3 instructions each, 2 for 1/d).
// A numerator of +-0 gives the zero of the right sign for d > 0 (the remainder is formed as d*q - n
// so that -0 survives); for d < 0 the sign of a zero quotient is not defined.
struct Recip {
    double d;
#if defined(__HIP_DEVICE_COMPILE__)
    double y;
#endif
    __host__ __device__ explicit Recip(double x) : d(x) {
#if defined(__HIP_DEVICE_COMPILE__)
        const double y0 = __builtin_amdgcn_rcp(x);
        const double y1 = __builtin_fma(y0, __builtin_fma(-x, y0, 1.0), y0);
        y = __builtin_fma(y1, __builtin_fma(-x, y1, 1.0), y1);
#endif
    }
    __host__ __device__ double div(double n) const {
#if defined(__HIP_DEVICE_COMPILE__)
        const double q = n * y;
        return __builtin_fma(-__builtin_fma(d, q, -n), y, q);
#else
        return n / d;
#endif
    }
    __host__ __device__ double inv() const {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_fma(-__builtin_fma(d, y, -1.0), y, y);
#else
        return 1.0 / d;
#endif
    }
};
// The divisor of a function that is written once for both cases: FAST = true is a Recip (the caller
// has established the ranges), FAST = false the plain division of any type.
template <bool FAST, class T>
struct Divisor {
    T d;
    __host__ __device__ explicit Divisor(const T& x) : d(x) {}
    template <class N>
    __host__ __device__ N div(const N& n) const { return n / d; }
    __host__ __device__ T inv() const { return 1.0 / d; }
};
template <>
struct Divisor<true, double> : Recip {
    using Recip::Recip;
};

// x is 0 or |x| >= lo (false for NaN)
__host__ __device__ inline int zero_or_from(double x, double lo) { return (fabs(x) >= lo) | (x == 0.0); }
// x is 0 or 2^-600 <= |x| <= 2^600 (false for NaN)
__host__ __device__ inline int moderate(double x) {
    const double t = fabs(x);
    return ((t >= 0x1p-600) & (t <= 0x1p600)) | (x == 0.0);
}
__host__ __device__ inline unsigned hi_word(double x) {
    return (unsigned)(__builtin_bit_cast(unsigned long long, x) >> 32);
}
// all four of a, b, c, d are positive and in [2^-100, 2^100 (1 + 2^-20)]: the high words, which order
// positive doubles, compared as unsigned integers (a negative value, an infinity or NaN is outside)
__host__ __device__ inline int positive_moderate(double a, double b, double c, double d) {
    const unsigned lo = 0x39b00000u, span = 0x46300000u - 0x39b00000u;  // high words of 2^-100 and 2^100
    const unsigned x = hi_word(a) - lo, y = hi_word(b) - lo, z = hi_word(c) - lo, w = hi_word(d) - lo;
    const unsigned m = x > y ? x : y, n = z > w ? z : w;
    return (m > n ? m : n) <= span;
}

// q[c] = n[c] / d for N numerators (in place is fine): one reciprocal where d lies in [2^-100, 2^100] and
// every numerator is 0 or moderate, plain divisions otherwise (a branch that waves without such a
// lane skip).
template <int N, class T>
__host__ __device__ inline void div_all(const T (&n)[N], const T& d, T (&q)[N]) {
    if constexpr (std::is_same<T, double>::value) {
        int in = positive_moderate(d, d, d, d);
#pragma unroll
        for (int c = 0; c < N; ++c) in &= moderate(n[c]);
        if (PHX_USUAL(wave_all(in))) {
            const Recip by(d);
#pragma unroll
            for (int c = 0; c < N; ++c) q[c] = by.div(n[c]);
            return;
        }
    }
#pragma unroll
    for (int c = 0; c < N; ++c) q[c] = n[c] / d;
}
__host__ __device__ inline double inv_area(double A) {
    if (PHX_USUAL(wave_all(positive_moderate(A, A, A, A)))) return Recip(A).inv();
    return 1.0 / A;
}

// IEEE square root of a double.  The compiler's sequence scales x by 2^256 when x < 2^-767, runs
// v_rsq_f64 and a Newton-Raphson refinement (g = x*y, h = y/2, r = 1/2 - h*g, g += g*r, h += h*r,
// then twice g += (x - g*g)*h), scales back by 2^-128, and returns x itself for +-0 and +inf.  For
// 2^-767 <= x <= DBL_MAX the scalings and that select are identities, so the refinement alone gives
// the same bits (sqrt_in_range, 10 instructions); sqrt_rn evaluates it and takes the library sqrt only
// for other x (a branch that waves skip when no lane needs it), 12 instead of 17 instructions with
// the range test.
__host__ __device__ inline double sqrt_in_range(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    double d = __builtin_fma(-g, g, x);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
#else
    return sqrt(x);
#endif
}
__host__ __device__ inline double sqrt_rn(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    double g = sqrt_in_range(x);
    if (!(x >= 0x1p-767 && x <= 0x1.fffffffffffffp+1023)) {
        // an empty volatile asm keeps this a branch: the compiler would otherwise evaluate the
        // library sqrt for every lane and select
        double xs = x;
        asm volatile("" : "+v"(xs));
        g = sqrt(xs);
    }
    return g;
#else
    return sqrt(x);
#endif
}
// sqrt of the flux arithmetic: sqrt_rn (FAST: sqrt_in_range) for doubles, the type's own sqrt otherwise
template <bool FAST, class T>
__host__ __device__ inline T sqrt_f(T x) {
    if constexpr (std::is_same<T, double>::value) return FAST ? sqrt_in_range(x) : sqrt_rn(x);
    else return sqrt(x);
}

// ConservativeConverter.to_primitive (states/converter/concrete_defs.py:85-100), with
// u = rhou/rho, v = rhov/rho (conservative.py:85-99), ek = rho*Ek, Ek = 0.5*(u*u+v*v)
// (conservative.py:118-124), p = (gamma-1)*(e - ek) (conservative.py:107-110).
template <bool FAST, class T>
__host__ __device__ inline PrimT<T> cons_to_prim_f(const Q4T<T>& q, const Phys& ph) {
    PrimT<T> w;
    const Divisor<FAST, T> by(q.v[0]);
    w.r = q.v[0];
    w.u = by.div(q.v[1]);
    w.v = by.div(q.v[2]);
    const T ek = w.r * (0.5 * (w.u * w.u + w.v * w.v));
    w.p = ph.gm1 * (q.v[3] - ek);
    return w;
}
template <class T>
__host__ __device__ inline PrimT<T> cons_to_prim(const Q4T<T>& q, const Phys& ph) {
    return cons_to_prim_f<false>(q, ph);
}
// The two states of a face: one reciprocal per state where, on the whole wave, both densities lie in
// [2^-100, 2^100] and every momentum is 0 or moderate (the quotients then lie in [2^-701, 2^701]), plain
// divisions otherwise.
template <class T>
__host__ __device__ inline void cons_to_prim2(const Q4T<T>& a, const Q4T<T>& b, const Phys& ph, PrimT<T>& L,
                                              PrimT<T>& R) {
    if constexpr (std::is_same<T, double>::value) {
        if (PHX_USUAL(wave_all(positive_moderate(a.v[0], a.v[0], b.v[0], b.v[0]) & moderate(a.v[1]) & moderate(a.v[2]) &
                               moderate(b.v[1]) & moderate(b.v[2])))) {
            L = cons_to_prim_f<true>(a, ph);
            R = cons_to_prim_f<true>(b, ph);
            return;
        }
    }
    L = cons_to_prim_f<false>(a, ph);
    R = cons_to_prim_f<false>(b, ph);
}

// rotate_JIT / unrotate_JIT (utils/utils.py:75-85,148-158) with c = cos(theta), s = sin(theta).
template <class T>
__host__ __device__ inline Q4T<T> rotate(Q4T<T> q, double c, double s) {
    const T u = q.v[1], v = q.v[2];
    q.v[1] = u * c + v * s;
    q.v[2] = v * c - u * s;
    return q;
}
template <class T>
__host__ __device__ inline Q4T<T> unrotate(Q4T<T> q, double c, double s) {
    const T u = q.v[1], v = q.v[2];
    q.v[1] = u * c - v * s;
    q.v[2] = v * c + u * s;
    return q;
}
// rotate90 / unrotate90 (utils/utils.py:88-112,161-185).
template <class T>
__host__ __device__ inline Q4T<T> rotate90(Q4T<T> q) {
    const T u = q.v[2], v = q.v[1];
    q.v[1] = u;
    q.v[2] = -v;
    return q;
}
template <class T>
__host__ __device__ inline Q4T<T> unrotate90(Q4T<T> q) {
    const T u = q.v[2], v = q.v[1];
    q.v[1] = -u;
    q.v[2] = v;
    return q;
}
// BoundaryConditionFunctions.reflection (boundary_conditions/funcs.py:27-43).
template <class T>
__host__ __device__ inline Q4T<T> reflect(Q4T<T> q, double c, double s) {
    q = rotate(q, c, s);
    q.v[1] = -q.v[1];
    return unrotate(q, c, s);
}

// Harten entropy fix on the Roe wave speeds (flux/base.py:119-146).  Inputs are the slow (u-a)
// and fast (u+a) speeds of the right, left and Roe states; l1/l4 are corrected in place.
template <class T>
__host__ __device__ inline void harten(T Rslow, T Rfast, T Lslow, T Lfast, T& l1, T& l4) {
    T tp = 2.0 * (Rslow - Lslow);
    T tm = 2.0 * (Rfast - Lfast);
    tp = (tp <= 0.0) ? T(1e-8) : tp;
    tm = (tm <= 0.0) ? T(1e-8) : tm;
    if constexpr (std::is_same<T, double>::value) {
        // few waves hold a face whose speed is that close to 0: the whole wave skips the divisions
        const bool f1 = fabs(l1) < tp, f4 = fabs(l4) < tm;
        if (PHX_RARE(wave_any(f1 | f4))) {
            const double c1 = 0.5 * ((l1 * l1) / tp + tp), c4 = 0.5 * ((l4 * l4) / tm + tm);
            l1 = f1 ? c1 : l1;
            l4 = f4 ? c4 : l4;
        }
    } else {
        if (fabs(l1) < tp) l1 = 0.5 * ((l1 * l1) / tp + tp);
        if (fabs(l4) < tm) l4 = 0.5 * ((l4 * l4) / tm + tm);
    }
}

// A face of a flat region: every jump dW = W_R - W_L is +0 (all bits zero), with a density and a
// pressure in [2^-300, 2^300] and speeds of at most 2^300.  There every intermediate of the Roe
// dissipation below is finite and each term of Rc|Lambda|Lp dW is a finite number times +0, so the
// four row sums are signed zeros: rows 0, 2 and 3 are +0 (each contains a term 1.0*z or Ek*z1 that
// is +0), and row 1's sign does not matter because 0.5*(F_L1 + F_R1) >= p > 0.  The flux is then
// exactly 0.5*(F_L + F_R), and a wave whose faces are all flat skips the square roots and divisions of
// the dissipation.
__host__ __device__ inline bool roe_flat(double dr, double du, double dv, double dp, const PrimT<double>& L) {
    const unsigned long long z = __builtin_bit_cast(unsigned long long, dr) | __builtin_bit_cast(unsigned long long, du) |
                                 __builtin_bit_cast(unsigned long long, dv) | __builtin_bit_cast(unsigned long long, dp);
    const double lo = 0x1p-300, hi = 0x1p300;
    return z == 0ull && L.r >= lo && L.r <= hi && L.p >= lo && L.p <= hi && fabs(L.u) <= hi && fabs(L.v) <= hi;
}

// What the fluxes take from the two states by division and square root: the sqrt(rho)-weighted state
// (RoePrimitiveState._roe_state_from_prim_JIT, states/primitive.py:301-320), the sound speeds of the
// three states, h = gamma/(gamma-1) p*/rho* and 1/a* (ROE), and p/(gamma-1) of both states (HLLL).
template <class T>
struct RoeAvgT {
    T r, u, v, p, aL, aR, a, h, ia, eL, eR;
};
// FAST: densities and pressures in [2^-100, 2^100] and a moderate gamma.  Every divisor is then moderate:
// sqrt(rho_L) + sqrt(rho_R) in [2^-49, 2^52], the densities, rho* in [2^-100, 2^101], gamma - 1 and
// a* = sqrt(gamma p*/rho*) in [2^-111, 2^111], and so is every numerator (1, p, gamma p,
// (gamma/(gamma-1)) p*); the square roots' arguments lie in [2^-222, 2^222].
template <bool FAST, bool HLLL, class T>
__host__ __device__ inline void roe_avg_f(const PrimT<T>& L, const PrimT<T>& R, const Phys& ph, RoeAvgT<T>& m) {
    const T sL = sqrt_f<FAST>(L.r), sR = sqrt_f<FAST>(R.r);
    const T inv = Divisor<FAST, T>(sL + sR).inv();
    m.r = sqrt_f<FAST>(L.r * R.r);
    m.u = (L.u * sL + R.u * sR) * inv;
    if (!HLLL) m.v = (L.v * sL + R.v * sR) * inv;
    m.p = (L.p * sL + R.p * sR) * inv;
    m.aL = sqrt_f<FAST>(Divisor<FAST, T>(L.r).div(ph.gamma * L.p));
    m.aR = sqrt_f<FAST>(Divisor<FAST, T>(R.r).div(ph.gamma * R.p));
    const Divisor<FAST, T> by_r(m.r);
    m.a = sqrt_f<FAST>(by_r.div(ph.gamma * m.p));
    if (HLLL) {
        const Divisor<FAST, double> by_gm1(ph.gm1);
        m.eL = by_gm1.div(L.p);
        m.eR = by_gm1.div(R.p);
    } else {
        m.h = by_r.div(ph.g_over_gm1 * m.p);
        m.ia = Divisor<FAST, T>(m.a).inv();
    }
}
template <bool HLLL = false, class T>
__host__ __device__ inline RoeAvgT<T> roe_avg(const PrimT<T>& L, const PrimT<T>& R, const Phys& ph) {
    RoeAvgT<T> m;
    if constexpr (std::is_same<T, double>::value) {
        if (PHX_USUAL(!ph.odd_gas && wave_all(positive_moderate(L.r, R.r, L.p, R.p)))) {
            roe_avg_f<true, HLLL>(L, R, ph, m);
            return m;
        }
    }
    roe_avg_f<false, HLLL>(L, R, ph, m);
    return m;
}

// FluxRoe.compute_flux (flux/Roe.py:262-304) for one face, primitive left/right states.
//  * Roe state: roe_avg -- note the sqrt(rho)-weighted pressure.
//  * F from primitives: PrimitiveState._F_from_prim_JIT (states/primitive.py:223-237).
//  * Dissipation Rc |Lambda| Lp dW with the SciPy COO accumulation order of the reference's
//    block layout (flux/eigen_system.py:115-158,205-242; values flux/Roe.py:175-260).  The
//    leading "0 +" of each COO row sum only changes the sign of a zero and is omitted.
template <class T>
__host__ __device__ inline Q4T<T> roe_flux(const PrimT<T>& L, const PrimT<T>& R, const Phys& ph) {
    const T ekL = (0.5 * L.r) * (L.u * L.u + L.v * L.v);
    const T ekR = (0.5 * R.r) * (R.u * R.u + R.v * R.v);
    const T ruL = L.r * L.u, ruR = R.r * R.u;
    const T FL0 = ruL, FL1 = ruL * L.u + L.p, FL2 = ruL * L.v;
    const T FL3 = L.u * ((ph.one_over_gm1 * L.p + ekL) + L.p);
    const T FR0 = ruR, FR1 = ruR * R.u + R.p, FR2 = ruR * R.v;
    const T FR3 = R.u * ((ph.one_over_gm1 * R.p + ekR) + R.p);
    if constexpr (std::is_same<T, double>::value) {
        // flat region: the dissipation is exactly zero (roe_flat); the derivative of the dissipation
        // is not, so the tangent-linear instantiation always evaluates it
        if (PHX_RARE(wave_all(roe_flat(R.r - L.r, R.u - L.u, R.v - L.v, R.p - L.p, L)))) {
            Q4T<T> F;
            F.v[0] = 0.5 * (FL0 + FR0);
            F.v[1] = 0.5 * (FL1 + FR1);
            F.v[2] = 0.5 * (FL2 + FR2);
            F.v[3] = 0.5 * (FL3 + FR3);
            return F;
        }
    }

    const RoeAvgT<T> m = roe_avg(L, R, ph);
    const T us = m.u, vs = m.v, as = m.a, aL = m.aL, aR = m.aR;
    T l1 = us - as, l4 = us + as;
    harten(R.u - aR, R.u + aR, L.u - aL, L.u + aL, l1, l4);

    const T Ek = 0.5 * (us * us + vs * vs);           // Ek_JIT
    const T H = m.h + Ek;                             // H_given_Ek_JIT
    const T ua = us * as;
    const T ia = m.ia;                                // compute_Lp
    const T ia2 = ia * ia;
    const T h = 0.5 * ia2;
    const T r2a = 0.5 * m.r * ia;

    const T d0 = R.r - L.r, d1 = R.u - L.u, d2 = R.v - L.v, d3 = R.p - L.p;
    // Lp * dW: rows in COO order (3,1),(1,0),(2,2),(3,3),(0,1),(1,3),(0,3)
    const T y0 = (-r2a) * d1 + h * d3;
    const T y1 = 1.0 * d0 + (-ia2) * d3;
    const T y2 = 1.0 * d2;
    const T y3 = r2a * d1 + h * d3;
    // |Lambda| (diagonal)
    const T z0 = fabs(l1) * y0, z1 = fabs(us) * y1, z2 = fabs(us) * y2, z3 = fabs(l4) * y3;
    // Rc * z: COO order (3,0),(2,0),(3,1),(1,0),(2,1),(3,2),(0,0),(1,1),(2,2),(3,3),(0,1),(2,3),(1,3),(0,3)
    const T s0 = (1.0 * z0 + 1.0 * z1) + 1.0 * z3;
    const T s1 = (l1 * z0 + us * z1) + l4 * z3;
    const T s2 = ((vs * z0 + vs * z1) + 1.0 * z2) + vs * z3;
    const T s3 = (((H - ua) * z0 + Ek * z1) + vs * z2) + (H + ua) * z3;

    Q4T<T> F;
    F.v[0] = 0.5 * (FL0 + FR0) - 0.5 * s0;
    F.v[1] = 0.5 * (FL1 + FR1) - 0.5 * s1;
    F.v[2] = 0.5 * (FL2 + FR2) - 0.5 * s2;
    F.v[3] = 0.5 * (FL3 + FR3) - 0.5 * s3;
    return F;
}

// ---- Euclidean norm of HLLL's alpha (flux/HLLL.py:86-93) ----
//
// Numba lowers np.linalg.norm of a 1-D float64 array to the BLAS routine dnrm2 of the SciPy build
// it runs against.  SciPy's OpenBLAS (0.3.28 with scipy 1.15.3) uses the x87 kernel on x86-64:
// for n < 8 it accumulates 0 + x0^2 + x1^2 + x2^2 + x3^2 in order in the x87 registers (64-bit
// significand, round to nearest even after every multiply and add), takes fsqrt in the same
// format and returns the result rounded to double.  That is 1 ulp away from the double-precision
// formula sqrt(((x0^2+x1^2)+x2^2)+x3^2) on about one vector in five, so the extended format is
// emulated exactly here with 64-bit integer arithmetic.  Non-negative operands only (squares and
// their sums); no overflow or underflow exists in the extended range for squares of doubles.

// A non-negative extended value m * 2^e: m has bit 63 set, or m = 0 for zero.
struct Ext {
    unsigned long long m;
    int e;
};

__host__ __device__ inline unsigned long long umulhi64(unsigned long long a, unsigned long long b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __umul64hi(a, b);
#else
    return (unsigned long long)(((unsigned __int128)a * b) >> 64);
#endif
}

__host__ __device__ inline int clz64(unsigned long long x) { return __builtin_clzll(x); }

__host__ __device__ inline unsigned long long dbits(double x) { return __builtin_bit_cast(unsigned long long, x); }

// Rounds the 128-bit significand (hi, lo) * 2^(e - 64), hi bit 63 set, to 64 bits, nearest even;
// `sticky` flags non-zero bits below lo.
__host__ __device__ inline Ext ext_round(unsigned long long hi, unsigned long long lo, bool sticky, int e) {
    const bool half = (lo >> 63) != 0;
    const bool rest = ((lo << 1) != 0) || sticky;
    if (half && (rest || (hi & 1ull))) {
        ++hi;
        if (hi == 0) {
            hi = 1ull << 63;
            ++e;
        }
    }
    return Ext{hi, e};
}

// x*x rounded to the extended format (x87 fmul of two doubles loaded exactly).  Finite x.
__host__ __device__ inline Ext ext_sq(double x) {
    const unsigned long long b = dbits(x) & 0x7fffffffffffffffull;
    if (b == 0) return Ext{0ull, 0};
    const int be = (int)(b >> 52);
    unsigned long long M = b & 0x000fffffffffffffull;
    int E;
    if (be == 0) {
        E = -1074;  // subnormal: M * 2^-1074
    } else {
        M |= 1ull << 52;
        E = be - 1075;
    }
    const int lz = clz64(M);
    M <<= lz;  // x = M * 2^(E - lz), M in [2^63, 2^64)
    E -= lz;
    unsigned long long hi = umulhi64(M, M), lo = M * M;  // x^2 = (hi*2^64 + lo) * 2^(2E)
    int e = 2 * E + 64;
    if ((hi >> 63) == 0) {
        hi = (hi << 1) | (lo >> 63);
        lo <<= 1;
        e -= 1;
    }
    return ext_round(hi, lo, false, e);
}

// a + b rounded to the extended format (x87 fadd), a, b >= 0.
__host__ __device__ inline Ext ext_add(Ext a, Ext b) {
    if (b.m == 0) return a;
    if (a.m == 0) return b;
    if (a.e < b.e) {
        const Ext t = a;
        a = b;
        b = t;
    }
    const int d = a.e - b.e;
    // b < 2^(b.e + 64) <= 2^(a.e - 2), below half an ulp of a: a + b rounds to a.
    if (d > 65) return a;
    // a = (a.m * 2^64) * 2^(a.e - 64); b aligned to the same unit as (bh, bl) plus a sticky bit
    unsigned long long bh, bl;
    bool sticky = false;
    if (d == 0) {
        bh = b.m;
        bl = 0;
    } else if (d < 64) {
        bh = b.m >> d;
        bl = b.m << (64 - d);
    } else if (d == 64) {
        bh = 0;
        bl = b.m;
    } else {  // d == 65
        bh = 0;
        bl = b.m >> 1;
        sticky = (b.m & 1ull) != 0;
    }
    unsigned long long lo = bl;                 // a's low word is zero
    unsigned long long hi = a.m + bh;
    int e = a.e;
    if (hi < a.m) {  // carry out of bit 127: shift the 129-bit sum right by one
        sticky = sticky || (lo & 1ull);
        lo = (lo >> 1) | (hi << 63);
        hi = (hi >> 1) | (1ull << 63);
        e += 1;
    }
    return ext_round(hi, lo, sticky, e);
}

// 128-bit helpers for the square root (value = hi * 2^64 + lo).
__host__ __device__ inline bool u128_gt(unsigned long long ah, unsigned long long al, unsigned long long bh,
                                        unsigned long long bl) {
    return ah > bh || (ah == bh && al > bl);
}

// RN_double(RN_ext(sqrt(s))) for an extended s (x87 fsqrt, then the store to double).
__host__ __device__ inline double ext_sqrt_to_double(Ext s) {
    if (s.m == 0) return 0.0;
    // N = s.m * 2^k with s.e - k even, k in {63, 64}: N in [2^126, 2^128), sqrt(N) in [2^63, 2^64)
    const int k = ((s.e - 64) & 1) ? 63 : 64;
    const unsigned long long nh = (k == 64) ? s.m : (s.m >> 1);
    const unsigned long long nl = (k == 64) ? 0ull : (s.m << 63);
    const int E = (s.e - k) / 2;  // sqrt(s) = sqrt(N) * 2^E  (s.e - k is even)
    // q = floor(sqrt(N)): a double estimate (|error| < 2^13), one Newton step, then an exact fix-up
    const double dn = (double)nh * 18446744073709551616.0 + (double)nl;
    const double sq = sqrt(dn);
    unsigned long long q = (sq >= 18446744073709551616.0) ? 0xffffffffffffffffull : (unsigned long long)sq;
    {
        // rem = N - q^2 (|rem| < 2^79, two's complement over 128 bits)
        const unsigned long long qh = umulhi64(q, q), ql = q * q;
        const unsigned long long rl = nl - ql;
        const long long rh = (long long)(nh - qh - (nl < ql ? 1ull : 0ull));
        const double drem = (double)rh * 18446744073709551616.0 + (double)rl;
        const double step = drem / (2.0 * (double)q);
        const long long dq = (long long)(step + (step >= 0.0 ? 0.5 : -0.5));  // |dq| <= 2^13
        if (dq >= 0) {
            const unsigned long long up = (unsigned long long)dq;
            q = (q > 0xffffffffffffffffull - up) ? 0xffffffffffffffffull : q + up;
        } else {
            q -= (unsigned long long)(-dq);
        }
    }
    // now |q - sqrt(N)| < 1: q^2 > N -> q - 1; (q+1)^2 <= N -> q + 1 (twice each, for margin)
    for (int it = 0; it < 2; ++it) {
        const unsigned long long qh = umulhi64(q, q), ql = q * q;
        if (u128_gt(qh, ql, nh, nl)) --q;
    }
    for (int it = 0; it < 2; ++it) {
        if (q == 0xffffffffffffffffull) break;
        const unsigned long long p = q + 1;
        const unsigned long long ph = umulhi64(p, p), pl = p * p;
        if (!u128_gt(ph, pl, nh, nl)) q = p;
    }
    // round to 64 bits: up iff N - q^2 > q (sqrt(N) is never exactly q + 1/2)
    const unsigned long long qh = umulhi64(q, q), ql = q * q;
    const unsigned long long rl = nl - ql;
    const unsigned long long rh = nh - qh - (nl < ql ? 1ull : 0ull);  // 0 <= rem <= 2q < 2^65
    int e64 = E;                                                       // r64 * 2^e64
    unsigned long long r64 = q;
    if (rh != 0 || rl > q) {
        ++r64;
        if (r64 == 0) {
            r64 = 1ull << 63;
            ++e64;
        }
    }
    // round the 64-bit significand to the double's precision (53 bits, fewer if subnormal)
    int shift = 11;
    const int top = e64 + 63;  // exponent of the leading bit
    if (top < -1022) shift += -1022 - top;
    if (shift > 64) return 0.0;  // below half the smallest subnormal
    unsigned long long r53, rem_bits, halfv;
    if (shift == 64) {
        r53 = 0;
        rem_bits = r64;
        halfv = 1ull << 63;
    } else {
        r53 = r64 >> shift;
        rem_bits = r64 & ((1ull << shift) - 1ull);
        halfv = 1ull << (shift - 1);
    }
    if (rem_bits > halfv || (rem_bits == halfv && (r53 & 1ull))) ++r53;
    // r53 * 2^(e64 + shift) is exact in double (r53 <= 2^53); ldexp only scales
    return ldexp((double)r53, e64 + shift);
}

// The extended-precision norm by the integer emulation above (finite components).
__host__ __device__ inline double nrm4_ext(double a, double b, double c, double d) {
    Ext s = ext_sq(a);
    s = ext_add(s, ext_sq(b));
    s = ext_add(s, ext_sq(c));
    s = ext_add(s, ext_sq(d));
    return ext_sqrt_to_double(s);
}

// ---- fast path: the same extended-precision arithmetic carried out in pairs of doubles ----
// A value v >= 0 with a 64-bit significand is held as hi + lo (doubles, |lo| <= ulp(hi)/2, lo on
// v's 64-bit grid).  It covers components of magnitude 0 or in [2^-400, 2^400] (the low parts of the
// squares do not underflow, nothing overflows).  Each rounding to 64 bits is decided from a pair sum
// accurate to about 2^-104 of the value; where the value lies within 2^-30 of a grid unit of a
// midpoint of the 64-bit grid (exact ties included), or the square root within one 64-bit unit of a
// midpoint between two doubles (only there can the rounding to 64 bits change the rounding to
// double), the result is reported (ok = false) and taken from the integer emulation.
struct DD {
    double hi, lo;
};

// hi + lo = a + b exactly (Knuth's TwoSum)
__host__ __device__ inline DD two_sum(double a, double b) {
    const double s = a + b;
    const double bv = s - a;
    const double av = s - bv;
    return DD{s, (a - av) + (b - bv)};
}

// RN64(hi + lo), hi > 0, |lo| <= ulp(hi)/2: lo rounded to the 64-bit grid of the value's binade,
// 2^(E-63) for 2^E <= hi < 2^(E+1) (half that when hi = 2^E and lo < 0: the value is then in the
// binade below).  Adding and subtracting C = 1.5 * 2^52 * grid rounds lo to that grid, ties to even:
// C's last place is the grid unit and C / grid is even, so the parity is that of the 64-bit
// significand.  When lo carries a rounding error (exact = false), ok is cleared where lo lies within
// 2^-30 of a grid unit of a midpoint of the grid: the side of the midpoint is then not known.
__host__ __device__ inline DD rn64(double hi, double lo, bool exact, bool& ok) {
    int ex;
    const double m = frexp(hi, &ex);  // hi = m 2^ex, m in [1/2, 1): E = ex - 1
    double C = ldexp(0.75, ex - 11);  // 1.5 * 2^(E - 11) = 1.5 * 2^52 * 2^(E - 63)
    double half = ldexp(1.0, ex - 65);  // grid / 2
    if (m == 0.5 && lo < 0.0) {
        C *= 0.5;
        half *= 0.5;
    }
    const double l = (lo + C) - C;
    if (!exact && fabs(fabs(lo - l) - half) <= half * 0x1p-29) ok = false;
    return DD{hi, l};
}

// RN64(x^2), |x| = 0 or in [2^-400, 2^400]: x^2 = p + e exactly (fma)
__host__ __device__ inline DD sq64(double x, bool& ok) {
    const double p = x * x;
    if (p == 0.0) return DD{0.0, 0.0};
    return rn64(p, fma(x, x, -p), true, ok);
}

// RN64(A + B) of two 64-bit values >= 0 (x87 fadd).  The exact sum is s.hi + s.lo + A.lo + B.lo;
// the low terms are summed with their rounding errors e1, e2 tracked, so a sum carried out exactly
// (every case where the four terms span fewer than about 50 binades) decides ties exactly.
__host__ __device__ inline DD add64(DD A, DD B, bool& ok) {
    if (B.hi == 0.0) return A;
    if (A.hi == 0.0) return B;
    const DD s = two_sum(A.hi, B.hi);
    const DD t = two_sum(s.lo, A.lo);
    const DD w = two_sum(t.hi, B.lo);
    const double h = s.hi + w.hi;  // renormalised (Fast2Sum, |s.hi| >= |w.hi|): h + (w.hi - (h - s.hi)) exact
    return rn64(h, w.hi - (h - s.hi), t.lo == 0.0 && w.lo == 0.0, ok);
}

// RN53(RN64(sqrt(S))) of a 64-bit value S > 0 (x87 fsqrt, then the store to double).  z = sqrt(S)
// lies within one double unit of y = RN53(sqrt(S.hi)); z - y is known to about 2^-100 of y.  The
// rounding to 64 bits matters only where z is within half a 64-bit unit of a midpoint between two
// doubles: it then lands on the midpoint, and the store rounds that tie to the even neighbour.
__host__ __device__ inline double sqrt64(DD S, bool& ok) {
    const double y = sqrt(S.hi);
    const double p2 = y * y, e2 = fma(y, y, -p2);
    // z^2 - y^2 for z = sqrt(S) (S.hi - p2 is exact by Sterbenz), then z - y
    const double r = ((S.hi - p2) - e2) + S.lo;
    const double dlt = r / (2.0 * y);
    int ey;
    (void)frexp(y, &ey);                   // y in [2^(ey-1), 2^ey)
    const double ulp = ldexp(1.0, ey - 53);
    const double G = ldexp(1.0, ey - 64);  // 64-bit unit of y's binade
    const bool pow2 = (y == ldexp(0.5, ey));
    const double ulp_dn = pow2 ? 0.5 * ulp : ulp;
    const double g_dn = pow2 ? 0.25 * G : 0.5 * G;  // half the 64-bit unit at the lower midpoint
    const double up = dlt - 0.5 * ulp, dn = dlt + 0.5 * ulp_dn;  // z minus the midpoints
    const double mu = fabs(up), md = fabs(dn);
    if (fabs(mu - 0.5 * G) <= G * 0x1p-20 || fabs(md - g_dn) <= G * 0x1p-20) {  // not decided
        ok = false;
        return y;
    }
    const bool odd = (dbits(y) & 1ull) != 0ull;
    if (mu < 0.5 * G) return odd ? y + ulp : y;    // RN64(z) is the upper midpoint
    if (md < g_dn) return odd ? y - ulp_dn : y;     // RN64(z) is the lower midpoint
    if (up > 0.0) return y + ulp;
    if (dn < 0.0) return y - ulp_dn;
    return y;
}

__host__ __device__ inline bool nrm4_in_range(double x) {
    const double t = fabs(x);
    return t == 0.0 || (t >= 0x1p-400 && t <= 0x1p400);
}

// The norm where the pairs or the integers decide it: components of 0 or magnitude in [2^-400, 2^400] take
// the pair-of-doubles evaluation, which decides all but about one in 10^5 of them; the rest, and components
// outside that range, take the integer emulation; non-finite components the double formula (inf or
// NaN, as the extended computation gives).
__host__ __device__ __forceinline__ double nrm4_pairs(double a, double b, double c, double d) {
    if (((dbits(a) | dbits(b) | dbits(c) | dbits(d)) & 0x7fffffffffffffffull) == 0ull) return 0.0;
    const unsigned long long ex = 0x7ff0000000000000ull;
    if ((dbits(a) & ex) == ex || (dbits(b) & ex) == ex || (dbits(c) & ex) == ex || (dbits(d) & ex) == ex)
        return sqrt(((a * a + b * b) + c * c) + d * d);
    bool ok = nrm4_in_range(a) && nrm4_in_range(b) && nrm4_in_range(c) && nrm4_in_range(d);
    if (ok) {
        DD s = sq64(a, ok);
        s = add64(s, sq64(b, ok), ok);
        s = add64(s, sq64(c, ok), ok);
        s = add64(s, sq64(d, ok), ok);
        if (ok) {
            const double r = sqrt64(s, ok);
            if (ok) return r;
        }
    }
    return nrm4_ext(a, b, c, d);
}

// n / d to about 2^-46 of itself, for d in range
__host__ __device__ inline double quotient_46(double n, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rcp(d);
    return n * __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
#else
    return n / d;
#endif
}

// Euclidean norm of a 4-vector as dnrm2 computes it (see above).  Force-inlined: the kernels make no
// device-function calls.
//
// The extended computation rounds every square, sum and the root to 64 bits: its root is within
// 3 * 2^-64 of itself of the exact one (squares and three sums 4 * 2^-64, halved by the root, whose own
// rounding adds 2^-64).  So its rounding to double is that of the exact root wherever the exact root is
// further from a midpoint of two doubles than that, at most 2^-8.4 of half a last place.  Here
// the exact sum of squares is formed as a pair of doubles (to about 2^-100), y = RN(sqrt) of its high
// part and the remainder delta = (S - y^2)/(2y), known to 2^-40 of itself, tell on which side of y's
// midpoints the root lies; about one vector in 250 lies within 2^-8 of half a last place of one (or
// y is a power of two, whose lower midpoint is nearer): a wave with such a lane, or with a sum outside
// [2^-600, 2^1000], takes nrm4_pairs.  About 65 instead of 300 instructions, the same bits.
__host__ __device__ __forceinline__ double nrm4(double a, double b, double c, double d) {
    const bool zero = ((dbits(a) | dbits(b) | dbits(c) | dbits(d)) & 0x7fffffffffffffffull) == 0ull;
    if (PHX_RARE(wave_all(zero))) return 0.0;  // the jumps across the faces of a flat region
    const double pa = a * a, pb = b * b, pc = c * c, pd = d * d;
    const double e = (fma(a, a, -pa) + fma(b, b, -pb)) + (fma(c, c, -pc) + fma(d, d, -pd));
    const DD s1 = two_sum(pa, pb), s2 = two_sum(pc, pd), s3 = two_sum(s1.hi, s2.hi);
    const double tail = (s1.lo + s2.lo) + (s3.lo + e);
    const double S = s3.hi + tail;           // renormalised: |lo| <= half a last place of S,
    const double lo = tail - (S - s3.hi);    // so the root lies within one last place of y
    const unsigned hs = hi_word(S) - 0x1a700000u;  // high word of 2^-600
    const bool in = hs <= 0x7e700000u - 0x1a700000u;
    const double y = sqrt_in_range(S);
    const double delta = quotient_46(fma(-y, y, S) + lo, 2.0 * y);  // S - y*y is exact
    const unsigned long long yb = dbits(y);
    // half of y's last place, and delta against it
    const double half = __builtin_bit_cast(double, (yb & 0x7ff0000000000000ull) - (53ull << 52));
    const double m = fabs(delta);
    const bool sure = (fabs(m - half) > half * 0x1p-8) & ((yb & 0x000fffffffffffffull) != 0ull);
    if (PHX_RARE(!wave_all(zero | (in & sure)))) return nrm4_pairs(a, b, c, d);
    double r = y;
    if (m > half) r = delta > 0.0 ? y + 2.0 * half : y - 2.0 * half;
    return zero ? 0.0 : r;
}

// FluxHLLL.compute_flux + _HLLL_flux_JIT (flux/HLLL.py:25-49,70-103) for one face.
template <class T>
__host__ __device__ inline Q4T<T> hlll_flux(const PrimT<T>& L, const PrimT<T>& R, const Phys& ph) {
    const RoeAvgT<T> m = roe_avg<true>(L, R, ph);
    const T us = m.u, as = m.a, aL = m.aL, aR = m.aR;
    const T Lslow = L.u - aL, Lfast = L.u + aL;
    const T Rslow = R.u - aR, Rfast = R.u + aR;
    T l1 = us - as, l4 = us + as;
    harten(Rslow, Rfast, Lslow, Lfast, l1, l4);
    const T Lplus = (Rfast >= l4) ? Rfast : l4;      // np.maximum(R_m, Lm)
    const T Lminus = (Lslow <= l1) ? Lslow : l1;     // np.minimum(L_p, Lp)

    // ConservativeState(state=W): PrimitiveConverter.to_conservative (concrete_defs.py:126-141)
    const T ekL = (0.5 * L.r) * (L.u * L.u + L.v * L.v);
    const T ekR = (0.5 * R.r) * (R.u * R.u + R.v * R.v);
    const T UL0 = L.r, UL1 = L.r * L.u, UL2 = L.r * L.v, UL3 = m.eL + ekL;
    const T UR0 = R.r, UR1 = R.r * R.u, UR2 = R.r * R.v, UR3 = m.eR + ekR;
    // PrimitiveState.F(U=...) (states/primitive.py:203-209)
    const T FL0 = UL1, FL1 = UL1 * L.u + L.p, FL2 = UL1 * L.v, FL3 = L.u * (UL3 + L.p);
    const T FR0 = UR1, FR1 = UR1 * R.u + R.p, FR2 = UR1 * R.v, FR3 = R.u * (UR3 + R.p);
    Q4T<T> F;
    if (Lminus >= 0.0) {
        F.v[0] = FL0; F.v[1] = FL1; F.v[2] = FL2; F.v[3] = FL3;
    } else if (Lplus <= 0.0) {
        F.v[0] = FR0; F.v[1] = FR1; F.v[2] = FR2; F.v[3] = FR3;
    } else {
        const T dU0 = UR0 - UL0, dU1 = UR1 - UL1, dU2 = UR2 - UL2, dU3 = UR3 - UL3;
        const T dF0 = FR0 - FL0, dF1 = FR1 - FL1, dF2 = FR2 - FL2, dF3 = FR3 - FL3;
        const T k = as * nrm4(dU0, dU1, dU2, dU3);
        const T n = nrm4(dF0 - us * dU0, dF1 - us * dU1, dF2 - us * dU2, dF3 - us * dU3);
        const T den = (k < 1e-16) ? T(k + 1e-14) : k;
        T alpha = 1.0 - n / den;
        alpha = (0.0 >= alpha) ? T(0.0) : alpha;              // np.maximum(0, ...)
        const T ra = us / Lminus, rb = us / Lplus;
        const T mx = (ra >= rb) ? ra : rb;            // np.maximum(u/Lm, u/Lp)
        const T coef = Lminus * Lplus * (1.0 - alpha * (1.0 - mx));
        const T w = Lplus - Lminus;
        T N[4];
        N[0] = Lplus * FL0 - Lminus * FR0 + coef * dU0;
        N[1] = Lplus * FL1 - Lminus * FR1 + coef * dU1;
        N[2] = Lplus * FL2 - Lminus * FR2 + coef * dU2;
        N[3] = Lplus * FL3 - Lminus * FR3 + coef * dU3;
        div_all(N, w, F.v);
    }
    return F;
}

template <int FLUX, class T>
__host__ __device__ inline Q4T<T> face_flux(const Q4T<T>& qL, const Q4T<T>& qR, const Phys& ph) {
    PrimT<T> L, R;
    cons_to_prim2(qL, qR, ph, L, R);
    if (FLUX == 0) return roe_flux(L, R, ph);
    return hlll_flux(L, R, ph);
}

template <class T>
__host__ __device__ inline PrimT<T> as_prim(const Q4T<T>& q) { return PrimT<T>{q.v[0], q.v[1], q.v[2], q.v[3]}; }
template <class T>
__host__ __device__ inline Q4T<T> prim_q4(const PrimT<T>& w) {
    Q4T<T> q;
    q.v[0] = w.r; q.v[1] = w.u; q.v[2] = w.v; q.v[3] = w.p;
    return q;
}

// face_flux on face states in the reconstruction variables: with PrimitiveState reconstruction the
// states are primitive already and go to the flux as they are (fvm/base.py:286-289).
template <int FLUX, class T>
__host__ __device__ inline Q4T<T> face_flux_recon(const Q4T<T>& qL, const Q4T<T>& qR, const Phys& ph) {
    if (!ph.prim) return face_flux<FLUX>(qL, qR, ph);
    if (FLUX == 0) return roe_flux(as_prim(qL), as_prim(qR), ph);
    return hlll_flux(as_prim(qL), as_prim(qR), ph);
}

// Geometry of one cell as seen by the reconstruction: GG face weights x/yl = L*n (per face),
// 1/A, and the quadrature-point offsets from the centroid (dxq = xq - xc, dyq = yq - yc).
struct CellGeo {
    double xlE, xlW, xlN, xlS, ylE, ylW, ylN, ylS;
    double ainv;
    double dxE, dxW, dxN, dxS, dyE, dyW, dyN, dyS;
    bool odd = false;  // a weight or offset beyond 2^60 (or not finite): limit_venkat takes the general path
};

template <class T>
struct ReconT {
    Q4T<T> E, W, N, S;  // limited face states (SecondOrderMUSCL.limited_solution_at_quadrature_point)
};
using Recon = ReconT<double>;

// np.minimum of two scalars: a NaN operand is returned (NaN-propagating, unlike fmin).  Written as
// three selects of plain values: nested conditionals become branches, and the compiler then moves
// the evaluation of b (a whole limiter chain) into the branch where a is not NaN, serialising the
// faces' divisions.
template <class T>
__host__ __device__ inline T np_minimum(T a, T b) {
    const bool a_nan = a != a, b_nan = b != b;
    const T lo = (a <= b) ? a : b;
    const T r = b_nan ? b : lo;
    return a_nan ? a : r;
}

// np.minimum.reduce of the four faces' limiter values in the order E, W, N, S (the first NaN if
// any).  Venkatakrishnan values (GEN = false) are never -0: the numerator s*s + 2*s is +0 where it
// sums to zero (a zero sum of two doubles rounds to +0), the denominator is positive, and the
// flat-face value is 3/4.  Without a NaN the chain's result is then the minimum, which fmin returns
// with the same bits; a lane with a NaN takes the chain (a branch that waves without one skip).
template <bool GEN, class T>
__host__ __device__ inline T limiter_min4(T pE, T pW, T pN, T pS) {
    if constexpr (!GEN && std::is_same<T, double>::value) {
        const bool any_nan = (pE != pE) | (pW != pW) | (pN != pN) | (pS != pS);
        T m = fmin(fmin(pE, pW), fmin(pN, pS));
        if (any_nan) m = np_minimum(np_minimum(np_minimum(pE, pW), pN), pS);
        return m;
    } else {
        return np_minimum(np_minimum(np_minimum(pE, pW), pN), pS);
    }
}

// Slope of one face, SlopeLimiter._compute_slope (limiters/base.py:189-221): dmax/d for d > 0,
// dmin/d for d < 0, 1 otherwise.
template <class T>
__host__ __device__ inline T face_slope(T dmax, T dmin, T d) {
    const T num = (d > 0.0) ? dmax : dmin;
    return (d > 0.0 || d < 0.0) ? num / d : T(1.0);
}

// Limiter functions of limiters/limiters.py:25-62 (slope**2 is s*s).
template <class T>
__host__ __device__ inline T venkatakrishnan_fn(T s) {
    const T s2 = s * s;
    return (s2 + 2.0 * s) / (s2 + s + 2.0);
}
template <class T>
__host__ __device__ inline T limiter_fn(int lim, T s) {
    switch (lim) {
        case 1: return np_minimum(T(1.0), s);                                 // BarthJespersen
        case 2: { const T s2 = s * s; return (s2 + s) / (s2 + 1.0); }        // VanAlbada
        case 3: return (fabs(s) + s) / (s + 1.0);                             // VanLeer
        default: return venkatakrishnan_fn(s);                                 // Venkatakrishnan
    }
}

// Limiter value of one face.  GEN = false: Venkatakrishnan (the default, compiled without the
// limiter switch); GEN = true: the limiter `lim`.
// Limiter value at the default slope s = 1 (d = 0): Venkatakrishnan 3/4, the other three 1.
__host__ __device__ inline double limiter_at_one(bool gen, int lim) {
    return (gen && lim >= 1 && lim <= 3) ? 1.0 : 0.75;
}

// Where d = 0 the slope is the default 1 and the limiter value the constant limiter_fn(lim, 1)
// (3/4 = (1 + 2)/(1 + 1 + 2) exactly, or 1), so neither division is evaluated there: a wave whose
// faces all have d = 0 (a flat region) skips both.
template <bool GEN, class T>
__host__ __device__ inline T limit_face(T dmax, T dmin, T d, int lim) {
    if (!(d > 0.0 || d < 0.0)) return T(limiter_at_one(GEN, lim));
    const T num = (d > 0.0) ? dmax : dmin;
    const T s = num / d;
    return GEN ? limiter_fn(lim, s) : venkatakrishnan_fn(s);
}

// Venkatakrishnan._venkata (limiters/limiters.py:38-49) on the slope of one face.
__host__ __device__ inline double venkat_face(double dmax, double dmin, double d) {
    return limit_face<false>(dmax, dmin, d, 0);
}

// Stencil extrema: v_max_f64 / v_min_f64 as they are.  fmax and fmin of loaded values each first pass
// every operand through a v_max_f64 x, x of its own, which only quiets signaling NaNs; a neighbour
// that holds a NaN of either kind makes the gradient and with it the limited states NaN.
__host__ __device__ inline double vmax(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmax(a, b);
#endif
}
__host__ __device__ inline double vmin(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return fmin(a, b);
#endif
}
__host__ __device__ inline double vmin_abs4(double a, double b, double c, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r, t;
    asm("v_min_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
    asm("v_min_f64 %0, |%1|, |%2|" : "=v"(t) : "v"(c), "v"(d));
    return vmin(r, t);
#else
    return fmin(fmin(fabs(a), fabs(b)), fmin(fabs(c), fabs(d)));
#endif
}
template <class T>
__host__ __device__ inline T vmax(T a, T b) { return fmax(a, b); }
template <class T>
__host__ __device__ inline T vmin(T a, T b) { return fmin(a, b); }

// Venkatakrishnan's value for a slope s that is 0 or in [2^-680, 2^496]: the divisor lies in [2, 2^993] and the
// quotient in [2^-680, 2], in Recip's range
__host__ __device__ inline double venkat_in_range(double s) {
    const double s2 = s * s;
    return Recip(s2 + s + 2.0).div(s2 + 2.0 * s);
}

// n / d for a d that is 0 or in range: NaN for d = 0 (v_rcp_f64 gives an infinity, 1 - 0*inf NaN), which
// fmin passes over
__host__ __device__ inline double slope_or_nan(double n, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
    return Recip(d).div(n);
#else
    return d == 0.0 ? __builtin_nan("") : n / d;
#endif
}

// Limiter value of one variable of a cell: max(0, minimum over the four faces of Venkatakrishnan's value
// of the face's slope) (Venkatakrishnan._venkata, limiters/limiters.py:38-49, np.minimum.reduce), from the
// high-order terms h of the faces E, W, N, S (d = (u + h) - u).  3 divisions instead of 8, the same bits.
//
// The slopes of the faces with d > 0 are dmax/d, and division rounds monotonically, so the smallest
// of them is dmax / max(d); likewise dmin / min(d) over d < 0.  phi(s) = (s^2 + 2s)/(s^2 + s + 2) rises
// on [0, 4.8] (relative slope s phi'/phi >= 1/4 on [0, 2]), passes phi(2) = 1 and stays >= 1 beyond.  Its
// computed value is within 6 units of 2^-53, so of two slopes that differ by more than 2^-40 of
// themselves the smaller one has the smaller computed value as long as it is at most 2 (at
// s = 2 exactly phi = 1 exactly, and no computed value of a larger slope is below 1).  So the value at
// the smallest slope is the minimum unless another slope lies within 2^-40 of it, or all four exceed
// 2: a wave with such a lane compares all four values.  A face with d = 0 has the slope 1, whose value
// 3/4 enters as a constant.
//
// In-range divisions: dmax - dmin <= 2^100 and 2^-340 <= |u| < 2^101 make every non-zero difference
// of the stencil and every non-zero d at least 2^-394 (each is a multiple of half the last place of
// |u|), geometry up to 2^60 makes |d| <= 2^286, so a slope is 0 or in [2^-680, 2^496] and its
// square does not overflow.  Where u is 0 the differences are tested themselves: a slope that
// overflows gives inf/inf = NaN in the general evaluation, so a tiny d must not be passed over.  A
// wave with a lane outside these ranges takes the general evaluation of all faces.
__host__ __device__ __forceinline__ double limit_venkat(double u, double dmax, double dmin, const double (&h)[4], bool odd) {
    const double dE = (u + h[0]) - u, dW = (u + h[1]) - u, dN = (u + h[2]) - u, dS = (u + h[3]) - u;
    const double a = vmax(dE, dW), b = vmin(dE, dW), c = vmax(dN, dS), e = vmin(dN, dS);
    const double P = vmax(a, c), p = vmin(a, c), M = vmin(b, e), m = vmax(b, e);  // the four d again
    if (PHX_RARE(wave_lanes(vmax(P, -M) > 0.0) == 0)) return 0.75;  // flat: no increment at any face
    const double near = 1.0 - 0x1p-40;
    const double Pc = vmax(P, 0.0), Mc = vmin(M, 0.0);
    const double sP = slope_or_nan(dmax, Pc), sM = slope_or_nan(dmin, Mc);
    const double s = vmin(sP, sM);
    const double cap = vmin_abs4(P, p, M, m) == 0.0 ? 0.75 : __builtin_inf();
    const unsigned long long close = wave_lanes(vmax(p, m) > Pc * near) | wave_lanes(vmin(p, m) < Mc * near) |
                                     wave_lanes(fabs(sP - sM) <= s * 0x1p-40) | wave_lanes(vmin(s, cap) > 2.0);
    const double phi = vmin(venkat_in_range(s), cap);
    // high words: |u| in [2^-340, 2^100 (1 + 2^-20)], the spread of the stencil at most that (a NaN is beyond)
    const unsigned size = (hi_word(u) & 0x7fffffffu) - 0x2ab00000u, spread = hi_word(dmax - dmin);
    const unsigned long long wide = wave_lanes(spread > 0x46300000u), off = wave_lanes(size > 0x46300000u - 0x2ab00000u);
    if (PHX_USUAL(!odd & ((close | wide | off) == 0))) return phi;

    double w = u;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(w));  // the increments again, not kept in registers from above
#endif
    double d[4];
    int zero = (int)(u == 0.0) & zero_or_from(dmax, 0x1p-394) & zero_or_from(dmin, 0x1p-394);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        d[f] = (w + h[f]) - w;
        zero &= zero_or_from(d[f], 0x1p-394);
    }
    if (!odd & ((wide | (off & wave_lanes(zero == 0))) == 0)) {
        if (close == 0) return phi;
        double x = cap;
#pragma unroll
        for (int f = 0; f < 4; ++f) x = vmin(x, venkat_in_range(slope_or_nan(d[f] > 0.0 ? dmax : dmin, d[f])));
        return x;
    }
    const double pE = limit_face<false>(dmax, dmin, d[0], 0), pW = limit_face<false>(dmax, dmin, d[1], 0);
    const double pN = limit_face<false>(dmax, dmin, d[2], 0), pS = limit_face<false>(dmax, dmin, d[3], 0);
    const double x = limiter_min4<false>(pE, pW, pN, pS);
    return (x < 0.0) ? 0.0 : x;
}
// Barth-Jespersen's value of one variable of a cell, as limit_venkat: min(1, slope) rises with the slope and
// division rounds monotonically, so the smallest slopes are dmax / max(d) and dmin / min(d) (2 divisions
// instead of 4, the same bits).  Values and increments of at most 2^600 leave no infinity or NaN among the
// d; with both extrema at the cell the sign of the zero depends on the faces' order.
__host__ __device__ __forceinline__ double limit_bj(double u, double dmax, double dmin, const double (&h)[4]) {
    const double dE = (u + h[0]) - u, dW = (u + h[1]) - u, dN = (u + h[2]) - u, dS = (u + h[3]) - u;
    const double P = vmax(vmax(vmax(dE, dW), vmax(dN, dS)), 0.0), M = vmin(vmin(vmin(dE, dW), vmin(dN, dS)), 0.0);
    const double size = fabs(u) + ((fabs(h[0]) + fabs(h[1])) + (fabs(h[2]) + fabs(h[3])));
    const int usual = (int)(size <= 0x1p600) & (dmax - dmin <= 0x1p600) & !((int)(dmax == 0.0) & (dmin == 0.0) & (P > M));
    if (PHX_USUAL(wave_all(usual))) {
        const double sP = (P > 0.0) ? dmax / P : 1.0, sM = (M < 0.0) ? dmin / M : 1.0;
        return vmin(vmin(sP, sM), 1.0);
    }
    const double pE = limit_face<true>(dmax, dmin, dE, 1), pW = limit_face<true>(dmax, dmin, dW, 1);
    const double pN = limit_face<true>(dmax, dmin, dN, 1), pS = limit_face<true>(dmax, dmin, dS, 1);
    const double phi = limiter_min4<true>(pE, pW, pN, pS);
    return (phi < 0.0) ? 0.0 : phi;
}
// The general form: any scalar type, with GEN the limiter `lim`.
template <bool GEN, class T>
__host__ __device__ inline T limit_cell(const T& u, const T& dmax, const T& dmin, const T (&h)[4], bool odd, int lim) {
    if constexpr (std::is_same<T, double>::value) {
        if (PHX_USUAL(!GEN || lim == 0)) return limit_venkat(u, dmax, dmin, h, odd);
        if (lim == 1) return limit_bj(u, dmax, dmin, h);
    }
    const T pE = limit_face<GEN>(dmax, dmin, (u + h[0]) - u, lim);
    const T pW = limit_face<GEN>(dmax, dmin, (u + h[1]) - u, lim);
    const T pN = limit_face<GEN>(dmax, dmin, (u + h[2]) - u, lim);
    const T pS = limit_face<GEN>(dmax, dmin, (u + h[3]) - u, lim);
    const T phi = limiter_min4<GEN>(pE, pW, pN, pS);
    return (phi < 0.0) ? T(0.0) : phi;                 // np.where(phi < 0, 0, phi)
}

// One cell of the second-order reconstruction (reconstruct_var: one conserved variable):
//  * interface averages (blocks/quad_block.py:181-218),
//  * Green-Gauss gradient (gradients/greengauss.py:134-155),
//  * high-order term gx*dx + gy*dy (blocks/base.py:282-289),
//  * slope limiter with the 5-point min/max incl. ghosts (limiters/base.py:47-187): Venkatakrishnan,
//    or with GEN the limiter `lim` (BarthJespersen, VanAlbada, VanLeer),
//  * limited face values U + phi*hot (fvm/SecondOrderMUSCL.py:106-126).
// U is the cell, Uw/Ue/Us/Un its west/east/south/north neighbours (ghost values at block edges).
template <bool GEN = false, class T>
__host__ __device__ inline void reconstruct_var(T u, T uw, T ue, T us, T un, const CellGeo& g, int lim, T& qE,
                                                T& qW, T& qN, T& qS) {
    const T e = 0.5 * (u + ue);
    const T w = 0.5 * (uw + u);
    const T n = 0.5 * (u + un);
    const T s = 0.5 * (us + u);
    const T gx = (e * g.xlE + w * g.xlW + n * g.xlN + s * g.xlS) * g.ainv;
    const T gy = (e * g.ylE + w * g.ylW + n * g.ylN + s * g.ylS) * g.ainv;
    const T h[4] = {gx * g.dxE + gy * g.dyE, gx * g.dxW + gy * g.dyW, gx * g.dxN + gy * g.dyN, gx * g.dxS + gy * g.dyS};
    // np.maximum.reduce((U, UW, UE, US, UN)) - U
    const T mx = vmax(vmax(vmax(vmax(u, uw), ue), us), un);
    const T mn = vmin(vmin(vmin(vmin(u, uw), ue), us), un);
    const T phi = limit_cell<GEN>(u, T(mx - u), T(mn - u), h, g.odd, lim);
    qE = u + phi * h[0];
    qW = u + phi * h[1];
    qN = u + phi * h[2];
    qS = u + phi * h[3];
}

template <bool GEN = false, class T>
__host__ __device__ inline ReconT<T> reconstruct(const Q4T<T>& U, const Q4T<T>& Uw, const Q4T<T>& Ue,
                                                 const Q4T<T>& Us, const Q4T<T>& Un, const CellGeo& g, int lim = 0) {
    ReconT<T> r;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        reconstruct_var<GEN>(U.v[k], Uw.v[k], Ue.v[k], Us.v[k], Un.v[k], g, lim, r.E.v[k], r.W.v[k], r.N.v[k],
                             r.S.v[k]);
    return r;
}

// ---------------------------------------------------------------------------------------------
// nq-point Gauss faces (mesh/quadratures.py:33-95, fvm/base.py:168-190)
// ---------------------------------------------------------------------------------------------
constexpr int QMAX = 3;

// Offsets of the Gauss points of one cell from its centroid, faces E, W, N, S, points in rule order.
struct QGeo {
    double dx[4][QMAX], dy[4][QMAX];
};

// Reconstruction of one cell with nq points per face: the cell value (reconstruction variables),
// the Green-Gauss gradient and the limiter value; the limited value at a point is u + phi*hot.
struct ReconQ {
    Q4 u, gx, gy, phi;
};

// Weight of point i of the nq-point rule (_QUAD_2 = {-1/sqrt(3): 1, 1/sqrt(3): 1},
// _QUAD_3 = {-sqrt(3/5): 5/9, 0: 8/9, sqrt(3/5): 5/9}).
__host__ __device__ inline double gauss_w(int nq, int i) {
    if (nq == 3) return i == 1 ? 8.0 / 9.0 : 5.0 / 9.0;
    return nq == 2 ? 1.0 : 2.0;
}

// One variable of reconstruct_var with nq points per face: interface averages, Green-Gauss, and
// phi = max(0, min over E points, W points, N points, S points of the limiter of each point's slope)
// (limiters/base.py:47-187: np.minimum.reduce over the faces' point lists in that order).
__host__ __device__ inline void reconstruct_q_var(double u, double uw, double ue, double us, double un,
                                                  const CellGeo& g, const QGeo& q, int nq, int lim, double& gx,
                                                  double& gy, double& phi) {
    const double e = 0.5 * (u + ue);
    const double w = 0.5 * (uw + u);
    const double n = 0.5 * (u + un);
    const double s = 0.5 * (us + u);
    gx = (e * g.xlE + w * g.xlW + n * g.xlN + s * g.xlS) * g.ainv;
    gy = (e * g.ylE + w * g.ylW + n * g.ylN + s * g.ylS) * g.ainv;
    const double mx = vmax(vmax(vmax(vmax(u, uw), ue), us), un);
    const double mn = vmin(vmin(vmin(vmin(u, uw), ue), us), un);
    const double dmax = mx - u;
    const double dmin = mn - u;
    if (lim == 1) {
        // Barth-Jespersen: min(1, slope) rises with the slope and division rounds monotonically, so the smallest
        // slopes are dmax / max(d) and dmin / min(d): 2 divisions instead of one per point, the same bits.
        // Values and gradient of at most 2^600 and geometry of at most 2^60 leave no infinity or NaN among
        // the d; with both extrema at the cell the sign of the zero depends on the points' order.
        double P = 0.0, M = 0.0;
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int i = 0; i < QMAX; ++i) {
                if (i >= nq) continue;
                const double d = (u + (gx * q.dx[f][i] + gy * q.dy[f][i])) - u;
                P = vmax(P, d);
                M = vmin(M, d);
            }
        const int usual = (int)(fabs(gx) <= 0x1p600) & (fabs(gy) <= 0x1p600) & (fabs(u) <= 0x1p600) & (dmax - dmin <= 0x1p600) &
                          !((int)(dmax == 0.0) & (dmin == 0.0) & (P > M));
        if (PHX_USUAL(!g.odd && wave_all(usual))) {
            const double sP = (P > 0.0) ? dmax / P : 1.0, sM = (M < 0.0) ? dmin / M : 1.0;
            phi = vmin(vmin(sP, sM), 1.0);
            return;
        }
    }
    double p = 0.0;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < QMAX; ++i) {
            if (i >= nq) continue;
            const double h = gx * q.dx[f][i] + gy * q.dy[f][i];
            const double pf = limit_face<true>(dmax, dmin, (u + h) - u, lim);
            p = (f == 0 && i == 0) ? pf : np_minimum(p, pf);
        }
    phi = (p < 0.0) ? 0.0 : p;
}

__host__ __device__ inline ReconQ reconstruct_q(const Q4& U, const Q4& Uw, const Q4& Ue, const Q4& Us, const Q4& Un,
                                                const CellGeo& g, const QGeo& q, int nq, int lim) {
    ReconQ r;
    r.u = U;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        reconstruct_q_var(U.v[k], Uw.v[k], Ue.v[k], Us.v[k], Un.v[k], g, q, nq, lim, r.gx.v[k], r.gy.v[k], r.phi.v[k]);
    return r;
}

// Limited value at point i of face f: U + phi*(gx*dxq + gy*dyq)
// (SecondOrderMUSCL.limited_solution_at_quadrature_point, fvm/SecondOrderMUSCL.py:106-126).
__host__ __device__ inline Q4 qstate(const ReconQ& r, const QGeo& q, int f, int i) {
    Q4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double h = r.gx.v[k] * q.dx[f][i] + r.gy.v[k] * q.dy[f][i];
        o.v[k] = r.u.v[k] + r.phi.v[k] * h;
    }
    return o;
}

// Ideal-gas CFL quantity min(dx/(|u|+a), dy/(|v|+a)) of one cell (blocks/quad_block.py:433-436;
// ConservativeState.u/v/p/a, states/conservative.py:85-137).
__host__ __device__ inline double cell_dt(const Q4& q, double dx, double dy, const Phys& ph) {
    const double rho = q.v[0];
    const double u = q.v[1] / rho;
    const double v = q.v[2] / rho;
    const double p = ph.gm1 * (q.v[3] - rho * (0.5 * (u * u + v * v)));
    const double a = sqrt_rn(ph.gamma * p / rho);
    const double tx = dx / (fabs(u) + a);
    const double ty = dy / (fabs(v) + a);
    return (tx <= ty) ? tx : ty;
}

}  // namespace phx
