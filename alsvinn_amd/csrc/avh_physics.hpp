// Device-side physics of the FP64 finite-volume stage: equation state
// algebra, reconstructions and numerical fluxes.  Every expression keeps the
// operation order of the reference CPU path so that results are bit-equal:
// no FMA contraction (also forced by -ffp-contract=off), IEEE divide and
// sqrt, the same association of sums and products.
#pragma once
#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace avh {

// Workgroup barrier for data exchanged through LDS alone.  __syncthreads also
// waits for the wavefront's global loads and stores in flight, which here
// would put prefetched tiles and the write-back of results on the critical
// path of every plane or layer.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Correctly rounded FP64 square root for x in [2^-767, DBL_MAX]: the
// operation sequence the compiler emits for sqrt() on gfx950 -- v_rsq_f64,
// then g = x*r, h = r/2 and two Goldschmidt / Newton corrections by fused
// multiply-adds -- without the steps that are the identity on that range
// (scaling tiny arguments by 2^256 and the result back by 2^-128, and the
// zero / infinity fix-up), so the result has the same bits as sqrt(x) there.
__device__ __forceinline__ double sqrt_core(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r;
    double h = r * 0.5;
    const double d0 = fma(-h, g, 0.5);
    g = fma(g, d0, g);
    h = fma(h, d0, h);
    const double d1 = fma(-g, g, x);
    g = fma(d1, h, g);
    const double d2 = fma(-g, g, x);
    return fma(d2, h, g);
}

// Quotients that share a denominator.  The compiler divides n/d in FP64 on
// gfx950 as
//   d' = div_scale(d), n' = div_scale(n), r = rcp(d'),
//   r = fma(r, fma(-d', r, 1), r) twice, q0 = n' * r,
//   q = div_fmas(fma(-d', q0, n'), r, q0), result div_fixup(q, d, n).
// When d > 0, d and 1/d are normal, n is zero or has |n| >= 2^-968 and the
// quotient's binary exponent lies in [-1000, 760], the scalings are the
// identity (no VCC scale), div_fmas is a plain fma and div_fixup returns q
// -- or, for n = +-0, the zero with the sign of n.  The quotient is then a
// function of the refined reciprocal r alone, so r is computed once per
// denominator (div_recip) and each numerator costs one multiply and two
// fmas (div_shared).  The residual is formed as d*q0 - n and subtracted, the
// exact negation of the compiler's n - d*q0 added: nonzero numerators give
// the same bits, and n = +-0 gives +-0 as div_fixup does.
__device__ __forceinline__ double div_recip(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    return r;
}
__device__ __forceinline__ double div_shared(double n, double d, double r) {
    const double q0 = n * r;
    return fma(-fma(d, q0, -n), r, q0);
}
// 1/d: div_shared with numerator 1, whose first product is r itself.
__device__ __forceinline__ double div_one(double d) {
    const double r = div_recip(d);
    return fma(-fma(d, r, -1.0), r, r);
}
// lo <= n <= hi (false for zero, negative values, inf and NaN)
__device__ __forceinline__ bool positive_within(double n, double lo, double hi) {
    return (n >= lo) & (n <= hi);
}
// Binary exponent e of x = f * 2^e, 0.5 <= |f| < 1 (v_frexp_exp_i32_f64):
// 0 for +-0, the true exponent (<= -1022) for subnormals.  It is also 0 for
// inf and NaN, so a check built on it must exclude those by another test.
// `x is zero or |x| >= 2^(k-1)` is `frexp_exp(x) >= k`.
__device__ __forceinline__ int frexp_exp(double x) { return __builtin_amdgcn_frexp_exp(x); }

// Arithmetic of an interface's reconstruction and flux.
//   PlainOps   the compiler's sqrt and divide everywhere.
//   SharedOps  sqrt_core and div_recip / div_shared wherever operands provably
//              lie where these give PlainOps' bits; otherwise `ok` is cleared
//              and the caller recomputes the interface with PlainOps.
// What has to be checked for that is spread so that most of it is paid once
// per cell and not once per interface (the stage is bound by the FP64 pipe,
// and a check costs the same issue slot as an addition):
//   per launch     gamma in [1 + 2^-20, 2^10]             (EQ::gamma_admitted)
//   per cell       sum of |q_v| <= 2^85, momenta zero or at least 2^-600
//                  (EQ::admitted, of every cell of the tile and its halo)
//   per interface  each side: rho >= 2^-90, gamma p >= 2^-300, momenta zero or
//                  at least 2^-390; HLL3: the two star denominators and two
//                  star numerators; HLL: the denominator and the numerators.
// Measured against per-interface checks of every operand and the compiler's
// divisions for the WENO terms and star quotients (one MI355X, same box): 16
// RK3 steps at 1024^2 2381 -> 2114 us, 4 at 256^3 13.93 -> 12.80 ms; about 55
// fewer VALU instructions and 3 fewer quarter-rate reciprocals an interface.
// The bounds the cell check leaves on the face values and everything formed
// from them (faces are combinations of three cells with weights of magnitude
// at most 11/6, so at most 2^87):
//   u = m/rho: zero or in [2^-477, 2^177]; 0.5 m.m: zero or in [2^-781, 2^176]
//   p <= 2^97, p >= 2^-310; sound speeds in [2^-194, 2^99] (squares likewise
//   far inside sqrt_core's range); the two sides' sqrt(rho) in [2^-45, 2^44].
// "Zero or at least" carries through sums because doubles of magnitude at
// least 2^-k are multiples of 2^(-k-52), and so is any rounded sum of them:
// a difference of such values is zero or at least 2^(-k-52).
// The checks feed a flag instead of branching, and combine with
// non-short-circuit '&', so that they stay lane masks and an interface stays
// one straight-line block for the scheduler.
struct PlainOps {
    static constexpr bool SHARED = false;
    __device__ __forceinline__ static double sqrt_in_range(double x) { return sqrt(x); }
};
struct SharedOps {
    static constexpr bool SHARED = true;
    // sqrt of an argument known to lie in [2^-767, DBL_MAX]
    __device__ __forceinline__ static double sqrt_in_range(double x) { return sqrt_core(x); }
};
template <bool SHARED>
struct OpsFor {
    typedef PlainOps type;
};
template <>
struct OpsFor<true> {
    typedef SharedOps type;
};

enum { RECON_NONE = 0, RECON_WENO2 = 1, RECON_ENO2 = 2, RECON_ENO3 = 3 };

// ---------------------------------------------------------------------------
// Equations.  A conserved state is NV doubles: burgers {u};
// euler<nsd> {rho, m[0..nsd-1], E}.

struct BurgersEq {
    static constexpr int NV = 1;
    static constexpr int NSD = 3;  // the flux is the same along every axis
    struct All {
        double u;
    };
    // makeAllVariables (alsfvm/include/alsfvm/equation/burgers/Burgers.hpp:220-224)
    __device__ __forceinline__ static All make_all(const double* q, double) { return All{q[0]}; }
    template <class OPS>
    __device__ __forceinline__ static All make_all_ops(const double* q, double g, bool&) { return make_all(q, g); }
    // computePointFlux: u*u/2 (Burgers.hpp:158-164)
    __device__ __forceinline__ static double point_flux(double u) { return u * u / 2; }
    // CPUCellComputer::obeysConstraints + Burgers::obeysConstraints
    // (alsfvm/src/equation/CPUCellComputer.cpp:79-125, Burgers.hpp:212-217)
    __device__ __forceinline__ static bool obeys(const double* q, double) {
        const double u = q[0];
        return !__builtin_isnan(u) && !__builtin_isinf(u);
    }
    __device__ __forceinline__ static bool obeys_fast(const double* q, double g) { return obeys(q, g); }
    // SharedOps serves the WENO2 weights alone.  They need the bounds that
    // Euler puts on the density's differences and on the momenta; the face
    // values are not divided by anything, so an interface checks nothing.
    __device__ __forceinline__ static bool gamma_admitted(double) { return true; }
    __device__ __forceinline__ static bool admitted(const double* q) {
        return (fabs(q[0]) <= 0x1p85) & (frexp_exp(q[0]) >= -599);
    }
};

template <int NSD_>
struct EulerEq {
    static constexpr int NSD = NSD_;
    static constexpr int NV = NSD_ + 2;
    struct All {
        double rho, m[NSD_], E, p, u[NSD_];
        double rinv;  // refined reciprocal of rho (div_recip), 0 when not formed
    };
    // vec::dot, left to right (alsutils/include/alsutils/vec{1,2,3}.hpp)
    __device__ __forceinline__ static double dot(const double* m) {
        double s = m[0] * m[0];
#pragma unroll
        for (int c = 1; c < NSD_; ++c) s = s + m[c] * m[c];
        return s;
    }
    // computeExtra: ie = E - 0.5*m.m/rho, u = m/rho, p = (gamma-1)*ie
    // (alsfvm/include/alsfvm/equation/euler/Euler.hpp:204-211)
    __device__ __forceinline__ static All make_all(const double* q, double gamma) {
        All a;
        a.rho = q[0];
#pragma unroll
        for (int c = 0; c < NSD_; ++c) a.m[c] = q[1 + c];
        a.E = q[NSD_ + 1];
        const double ie = a.E - 0.5 * dot(a.m) / a.rho;
#pragma unroll
        for (int c = 0; c < NSD_; ++c) a.u[c] = a.m[c] / a.rho;
        a.p = (gamma - 1) * ie;
        a.rinv = 0.0;
        return a;
    }
    // The two checks SharedOps rests on beside its own per-interface ones
    // (see SharedOps): the equation's gamma, once per launch, and a cell's
    // conserved state, once per cell of a tile.  The sum of magnitudes bounds
    // every variable, and is NaN or infinite when one of them is.  Momenta
    // below 2^-600 (products with a WENO weight, at least 2^-404, could then
    // be subnormal) are left to PlainOps, so that halving the weights instead
    // of the sums (weno2_face) loses no bit.
    __device__ __forceinline__ static bool gamma_admitted(double gamma) {
        return positive_within(gamma, 0x1.00001p0, 0x1p10);
    }
    __device__ __forceinline__ static bool admitted(const double* q) {
        double s = fabs(q[0]);
        int emin = frexp_exp(q[1]);
#pragma unroll
        for (int v = 1; v < NV; ++v) s = s + fabs(q[v]);
#pragma unroll
        for (int c = 1; c < NSD_; ++c) emin = min(emin, frexp_exp(q[1 + c]));
        return (s <= 0x1p85) & (emin >= -599);
    }
    // make_all under OPS.  SharedOps forms one reciprocal of rho for the
    // divisions by rho; rho in [2^-90, 2^87] and the momenta's bounds put
    // every quotient in [2^-868, 2^266] or at zero.  0.5 m.m / rho is formed
    // as 0.5 (m.m / rho), and subtracted in one fused step: halving is exact
    // here, so neither changes a bit.
    template <class OPS>
    __device__ __forceinline__ static All make_all_ops(const double* q, double gamma, bool& ok) {
        if constexpr (!OPS::SHARED) {
            return make_all(q, gamma);
        } else {
            All a;
            a.rho = q[0];
#pragma unroll
            for (int c = 0; c < NSD_; ++c) a.m[c] = q[1 + c];
            a.E = q[NSD_ + 1];
            const double mm = dot(a.m);
            int emin = frexp_exp(a.m[0]);
#pragma unroll
            for (int c = 1; c < NSD_; ++c) emin = min(emin, frexp_exp(a.m[c]));
            ok = ok & (a.rho >= 0x1p-90) & (emin >= -389);
            const double r = div_recip(a.rho);
            const double ie = fma(-0.5, div_shared(mm, a.rho, r), a.E);
#pragma unroll
            for (int c = 0; c < NSD_; ++c) a.u[c] = div_shared(a.m[c], a.rho, r);
            a.rinv = r;
            a.p = (gamma - 1) * ie;
            return a;
        }
    }
    // sqrt(g*p / rho) for a state a from make_all_ops<OPS> (the sound speed;
    // n = g*p).  SharedOps checks n >= 2^-300 (p is then positive, and so
    // bounded above by (gamma - 1) E): the quotient lies in [2^-387, 2^197].
    template <class OPS>
    __device__ __forceinline__ static double sqrt_div_rho(double n, const All& a, bool& ok) {
        if constexpr (!OPS::SHARED) {
            return sqrt(n / a.rho);
        } else {
            ok = ok & (n >= 0x1p-300);
            return sqrt_core(div_shared(n, a.rho, a.rinv));
        }
    }
    // (n1, n2) / (wl + wr) with wl, wr the square roots of the two sides'
    // densities: n1 = uL wl + uR wr, n2 = wl pL + wr pR.  Under SharedOps
    // wl + wr is in [2^-44, 2^45], n1 zero or in [2^-574, 2^222] and n2, a sum
    // of two positive terms, in [2^-355, 2^142].
    template <class OPS>
    __device__ __forceinline__ static void div_roe(double n1, double n2, double wl, double wr, double& q1,
                                                   double& q2) {
        if constexpr (!OPS::SHARED) {
            q1 = n1 / (wl + wr);
            q2 = n2 / (wl + wr);
        } else {
            const double den = wl + wr;
            const double r = div_recip(den);
            q1 = div_shared(n1, den, r);
            q2 = div_shared(n2, den, r);
        }
    }
    // sqrt(g*p / rho) at the Roe pressure, which lies between the two sides'
    // (up to rounding), and the mean density: under SharedOps the quotient is
    // in [2^-389, 2^198] and needs no check of its own.
    template <class OPS>
    __device__ __forceinline__ static double sqrt_roe(double n, double rho) {
        if constexpr (!OPS::SHARED) {
            return sqrt(n / rho);
        } else {
            return sqrt_core(div_shared(n, rho, div_recip(rho)));
        }
    }
    // computePointFlux along DIR (Euler.hpp:172-181)
    template <int DIR>
    __device__ __forceinline__ static void point_flux(const All& a, double* F) {
        F[0] = a.m[DIR];
#pragma unroll
        for (int c = 0; c < NSD_; ++c) F[1 + c] = a.m[c] * a.u[DIR];
        F[1 + DIR] = F[1 + DIR] + a.p;
        F[NSD_ + 1] = (a.E + a.p) * a.u[DIR];
    }
    // conserved and extra variables finite, rho > 0, p > 0
    // (alsfvm/src/equation/CPUCellComputer.cpp:79-125, Euler.hpp:269-277)
    __device__ __forceinline__ static bool obeys(const double* q, double gamma) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < NV; ++i) ok = ok && !__builtin_isnan(q[i]) && !__builtin_isinf(q[i]);
        const All a = make_all(q, gamma);
        ok = ok && !__builtin_isnan(a.p) && !__builtin_isinf(a.p);
#pragma unroll
        for (int c = 0; c < NSD_; ++c) ok = ok && !__builtin_isnan(a.u[c]) && !__builtin_isinf(a.u[c]);
        return ok && (a.rho > 0) && (a.p > 0);
    }
    // obeys() decided without a division where the answer is plain: a state
    // whose magnitudes sum to at most 2^85 has no NaN or infinity, rho >=
    // 2^-90 makes every velocity and the kinetic energy finite, and the
    // pressure is positive if E exceeds the kinetic energy by more than the
    // rounding of either form: 2 rho E - m.m > 2^-40 (2 rho E), with 2 rho E >=
    // 2^-900 so that nothing underflows, and gamma - 1 >= 2^-20.  Any other
    // state takes obeys() itself.
    __device__ __forceinline__ static bool obeys_fast(const double* q, double gamma) {
        double s = fabs(q[0]);
#pragma unroll
        for (int v = 1; v < NV; ++v) s = s + fabs(q[v]);
        const double e2 = 2 * q[0] * q[NSD_ + 1];
        const double gap = e2 - dot(q + 1);
        bool plain = (s <= 0x1p85) & (q[0] >= 0x1p-90) & (e2 >= 0x1p-900) & (gap > 0x1p-40 * e2);
        plain = plain & gamma_admitted(gamma);
        return plain ? true : obeys(q, gamma);
    }
};

// ---------------------------------------------------------------------------
// Numerical fluxes F(left, right) along DIR; each returns the interface wave
// speed used for the CFL condition.

// burgers::Godunov (alsfvm/include/alsfvm/numflux/burgers/Godunov.hpp:40-60):
// F = max(f(max(uL,0)), f(min(uR,0))), wave speed max(|uL|, |uR|).
// Only the WENO2 weights divide, so only there it has a SharedOps path (a step
// of 1024 cells, rk3: 5.5 -> 5.1 us).
template <bool FAST_>
struct GodunovFluxT {
    template <int RECON>
    using For = GodunovFluxT<RECON == RECON_WENO2>;
    static constexpr bool FAST = FAST_;
    template <int DIR, class EQ>
    __device__ __forceinline__ static double flux(const BurgersEq::All& L, const BurgersEq::All& R,
                                                  double, double* F) {
        const double fl = BurgersEq::point_flux(fmax(L.u, 0.0));
        const double fr = BurgersEq::point_flux(fmin(R.u, 0.0));
        F[0] = fmax(fl, fr);
        return fmax(fabs(L.u), fabs(R.u));
    }
    template <class OPS, int DIR, class EQ>
    __device__ __forceinline__ static double flux_ops(const BurgersEq::All& L, const BurgersEq::All& R, double g,
                                                      double* F, bool&) {
        return flux<DIR, EQ>(L, R, g, F);
    }
};
typedef GodunovFluxT<false> GodunovFlux;

// euler::HLL (alsfvm/include/alsfvm/numflux/euler/HLL.hpp).  The reference's
// if/else chain is evaluated branch-free: every candidate is computed and the
// chain's answer is selected, which gives the same value as the branch taken.
struct HLLFlux {
    template <int RECON>
    using For = HLLFlux;
    static constexpr bool FAST = true;  // the stage kernel runs flux_ops<SharedOps> first
    template <int DIR, class EQ>
    __device__ __forceinline__ static double flux(const typename EQ::All& L, const typename EQ::All& R,
                                                  double g, double* F) {
        bool ok = true;
        return flux_ops<PlainOps, DIR, EQ>(L, R, g, F, ok);
    }
    template <class OPS, int DIR, class EQ>
    __device__ __forceinline__ static double flux_ops(const typename EQ::All& L, const typename EQ::All& R,
                                                      double g, double* F, bool& ok) {
        constexpr int NSD = EQ::NSD;
        constexpr int NV = EQ::NV;
        const double wl = OPS::sqrt_in_range(L.rho);
        const double wr = OPS::sqrt_in_range(R.rho);
        const double rho = (L.rho + R.rho) / 2;
        double ud, p;
        EQ::template div_roe<OPS>(L.u[DIR] * wl + R.u[DIR] * wr, L.p * wl + R.p * wr, wl, wr, ud, p);
        const double cs = EQ::template sqrt_roe<OPS>(g * p, rho);
        const double cfl = EQ::template sqrt_div_rho<OPS>(g * L.p, L, ok);
        const double cfr = EQ::template sqrt_div_rho<OPS>(g * R.p, R, ok);
        const double sl = fmin(L.u[DIR] - cfl, ud - cs);
        const double sr = fmax(R.u[DIR] + cfr, ud + cs);
        double fl[NV], fr[NV], ul[NV], ur[NV];
        EQ::template point_flux<DIR>(L, fl);
        EQ::template point_flux<DIR>(R, fr);
        ul[0] = L.rho;
        ur[0] = R.rho;
#pragma unroll
        for (int c = 0; c < NSD; ++c) {
            ul[1 + c] = L.m[c];
            ur[1 + c] = R.m[c];
        }
        ul[NSD + 1] = L.E;
        ur[NSD + 1] = R.E;
        const double srsl = sr * sl;
        const double den = sr - sl;
        double num[NV], mid[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) num[i] = sr * fl[i] - sl * fr[i] + srsl * (ur[i] - ul[i]);
        if constexpr (OPS::SHARED) {
            // one reciprocal for the NV quotients: den in [2^-100, 2^180] (the
            // speeds are at most 2^179) and every numerator zero or in
            // [2^-701, 2^456] put them in [2^-881, 2^556] or at zero
            int emin = frexp_exp(num[0]);
#pragma unroll
            for (int i = 1; i < NV; ++i) emin = min(emin, frexp_exp(num[i]));
            ok = ok & (den >= 0x1p-100) & (emin >= -700);
            const double r = div_recip(den);
#pragma unroll
            for (int i = 0; i < NV; ++i) mid[i] = div_shared(num[i], den, r);
        } else {
#pragma unroll
            for (int i = 0; i < NV; ++i) mid[i] = num[i] / den;
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double v = mid[i];
            v = (sr < 0) ? fr[i] : v;
            v = (sl > 0) ? fl[i] : v;
            v = (sl == 0) ? 0.0 : v;
            F[i] = v;
        }
        return fmax(fabs(sl), fabs(sr));
    }
};

// euler::HLL3 (alsfvm/include/alsfvm/numflux/euler/HLL3.hpp:52-148).  The two
// star-state branches (sm >= 0 / sm < 0) share one formula on the side's
// variables, so the side is selected first and the formula evaluated once.
struct HLL3Flux {
    template <int RECON>
    using For = HLL3Flux;
    static constexpr bool FAST = true;  // the stage kernel runs flux_ops<SharedOps> first
    // The star state of side k (k = L when s_m >= 0, else R): its speed sk,
    // the star conserved state `mid`, the side's conserved state `uc` and
    // its point flux `fk`, formed from side k's values by point_flux's
    // operations (the same bits as selecting between both point fluxes).
    // The transverse momentum fluxes in the star velocities are m[c] * u[DIR].
    // SharedOps forms one reciprocal for the quotients over aa and one for
    // those over s_m - s_k.  With |speeds| <= 2^179 and |u - speed| zero or at
    // least 2^-477 (a speed is a multiple of 2^-248, and u - 0 is u):
    //   -aa in [2^-150, 2^80] (aa < 0 in any flow; checked), numerators zero or
    //   in [2^-919, 2^268]: quotients in [2^-999, 2^418] or zero.  Both are
    //   negated, because div_shared keeps the sign of a zero for a positive
    //   denominator.
    //   |s_m - s_k| in [2^-100, 2^150], numerators checked at least 2^-700 and
    //   2^-800 in magnitude and at most 2^630: quotients in [2^-950, 2^730].
    template <class OPS, int DIR, class EQ>
    __device__ __forceinline__ static void star_side(const typename EQ::All& L, const typename EQ::All& R, double sl,
                                                     double sr, double& sk, double* mid, double* uc, double* fk,
                                                     bool& ok) {
        constexpr int NSD = EQ::NSD;
        const double pl = L.p, pr = R.p;
        const double udl = L.u[DIR] - sl;
        const double udr = R.u[DIR] - sr;
        const double aa = udr * R.rho - udl * L.rho;
        const double nm = R.m[DIR] * udr - L.m[DIR] * udl + pr - pl;
        double ra = 0.0, sm;
        if constexpr (OPS::SHARED) {
            ok = ok & positive_within(-aa, 0x1p-150, 0x1p80);
            ra = div_recip(-aa);
            sm = div_shared(-nm, -aa, ra);
        } else {
            sm = nm / aa;
        }

        const bool left = sm >= 0;
        const double rk = left ? L.rho : R.rho;
        const double udk = left ? udl : udr;
        sk = left ? sl : sr;
        const double pk = left ? pl : pr;
        const double uk = left ? L.u[DIR] : R.u[DIR];
        const double ek = left ? L.E : R.E;

        const double ds = sm - sk;
        const double n0 = rk * udk;
        const double pm = pk + rk * (uk - sm) * udk;
        const double ne = udk * ek + pk * uk - pm * sm;
        if constexpr (OPS::SHARED) {
            ok = ok & (fabs(ds) >= 0x1p-100) & (fabs(ds) <= 0x1p150) & (fabs(n0) >= 0x1p-700) &
                 (fabs(ne) >= 0x1p-800);
            const double rs = div_recip(ds);
            mid[0] = div_shared(n0, ds, rs);
            mid[NSD + 1] = div_shared(ne, ds, rs);
        } else {
            mid[0] = n0 / ds;
            mid[NSD + 1] = ne / ds;
        }
#pragma unroll
        for (int c = 0; c < NSD; ++c) {
            // us = (fR.m - fL.m - sR*mR + sL*mL)/aa with us[DIR] = sm
            double us = sm;
            if (c != DIR) {
                const double nt = R.m[c] * R.u[DIR] - L.m[c] * L.u[DIR] - R.m[c] * sr + L.m[c] * sl;
                if constexpr (OPS::SHARED) us = div_shared(-nt, -aa, ra);
                else us = nt / aa;
            }
            mid[1 + c] = us * mid[0];
            uc[1 + c] = left ? L.m[c] : R.m[c];
        }
        uc[0] = rk;
        uc[NSD + 1] = ek;
        fk[0] = uc[1 + DIR];
#pragma unroll
        for (int c = 0; c < NSD; ++c) fk[1 + c] = uc[1 + c] * uk;
        fk[1 + DIR] = fk[1 + DIR] + pk;
        fk[NSD + 1] = (ek + pk) * uk;
    }
    template <int DIR, class EQ>
    __device__ __forceinline__ static double flux(const typename EQ::All& L, const typename EQ::All& R,
                                                  double g, double* F) {
        bool ok = true;
        return flux_ops<PlainOps, DIR, EQ>(L, R, g, F, ok);
    }
    template <class OPS, int DIR, class EQ>
    __device__ __forceinline__ static double flux_ops(const typename EQ::All& L, const typename EQ::All& R,
                                                      double g, double* F, bool& ok) {
        constexpr int NV = EQ::NV;
        // computeHLLSpeeds
        const double wl = OPS::sqrt_in_range(L.rho);
        const double wr = OPS::sqrt_in_range(R.rho);
        const double rho = (L.rho + R.rho) / 2;
        double ud, p;
        EQ::template div_roe<OPS>(L.u[DIR] * wl + R.u[DIR] * wr, wl * L.p + wr * R.p, wl, wr, ud, p);
        const double cfl = EQ::template sqrt_div_rho<OPS>(g * L.p, L, ok);
        const double cfr = EQ::template sqrt_div_rho<OPS>(g * R.p, R, ok);
        // correct = jump/2; halving is exact but for subnormal jumps, which a
        // velocity sum of SharedOps' range does not notice, so there it is
        // fused into the sums
        const double jump = fmax(0.0, L.u[DIR] - R.u[DIR]);
        double ul, ur;
        if constexpr (OPS::SHARED) {
            ul = fma(0.5, jump, L.u[DIR]);
            ur = fma(-0.5, jump, R.u[DIR]);
        } else {
            const double correct = 0.5 * jump;
            ul = L.u[DIR] + correct;
            ur = R.u[DIR] - correct;
        }
        const double cs = EQ::template sqrt_roe<OPS>(g * p, rho);
        const double sl = fmin(ul - cfl, ud - cs);
        const double sr = fmax(ur + cfr, ud + cs);

        // subsonic interfaces (sL < 0 < sR) take the star branch.  Under
        // SharedOps a wavefront that is subsonic throughout skips the other
        // three branches and never forms both point fluxes (fewer values
        // live across the star formulas); otherwise both point fluxes are
        // formed first, as the general branch selects between them.
        const bool star = !(sl == 0) && !(sl > 0) && !(sr < 0);
        double sk, mid[NV], uc[NV], fk[NV];
        star_side<OPS, DIR, EQ>(L, R, sl, sr, sk, mid, uc, fk, ok);
        if (__all(star)) {
#pragma unroll
            for (int i = 0; i < NV; ++i) F[i] = fk[i] + sk * (mid[i] - uc[i]);
        } else {
            double fl[NV], fr[NV];
            EQ::template point_flux<DIR>(L, fl);
            EQ::template point_flux<DIR>(R, fr);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                double v = fk[i] + sk * (mid[i] - uc[i]);
                v = (sr < 0) ? fr[i] : v;
                v = (sl > 0) ? fl[i] : v;
                v = (sl == 0) ? 0.0 : v;
                F[i] = v;
            }
        }
        return fmax(fabs(sl), fabs(sr));
    }
};

// ---------------------------------------------------------------------------
// Reconstructions on an LDS tile.  `s` points at variable 0 of the tile,
// `vs` is the per-variable stride, `i` the cell, `sd` the stride along the
// reconstruction direction.  The indicator is variable 0 (rho or u).

template <int RECON>
struct ReconTraits;
template <>
struct ReconTraits<RECON_NONE> {
    static constexpr int GHOST = 1;
};
template <>
struct ReconTraits<RECON_WENO2> {
    static constexpr int GHOST = 2;
};
template <>
struct ReconTraits<RECON_ENO2> {
    static constexpr int GHOST = 2;
};
template <>
struct ReconTraits<RECON_ENO3> {
    static constexpr int GHOST = 3;
};

// WENO2 (alsfvm/include/alsfvm/reconstruction/WENO2.hpp:31-95; epsilon 1e-8,
// WENOCoefficients.hpp:21).  RIGHT selects the value at the cell's right face
// (the reference's `right` volume), otherwise the left face.
__device__ __forceinline__ void weno2_weights(double a0, double a1, double& w0, double& w1) {
    w0 = a0 / (a0 + a1);
    w1 = a1 / (a0 + a1);
}

// Under SharedOps a face's weights come from the reciprocals r = 1/d of the
// smoothness terms d = 3 (eps + b)^2 of the differences ahead (r0) and behind
// (r1), so 2/d is 2r (doubling is exact) and one reciprocal serves both
// quotients of a face.  The weights are formed halved: the 0.5 of the face
// value is a power of two, so it commutes with the rounding of every product
// and sum (no product is subnormal unless the face is below 2^-390, which
// the interface check excludes; EQ::admitted).  For the right face
// 0.5 * 2 r0 / (2 r0 + r1) is r0 / (2 r0 + r1): no multiplication at all.
// Admitted cells give d in [2^-53, 2^348]: r, the sum, and the quotients
// (at least 2^-404) need no check.
__device__ __forceinline__ double weno2_recip(double diff) {
    const double e = 1e-8 + diff * diff;
    return div_one(3 * e * e);
}
template <bool RIGHT>
__device__ __forceinline__ void weno2_half_weights(double r0, double r1, double& h0, double& h1) {
    const double den = RIGHT ? fma(2.0, r0, r1) : fma(2.0, r1, r0);
    const double r = div_recip(den);
    h0 = div_shared(r0, den, r);
    h1 = div_shared(r1, den, r);
    if (RIGHT) h1 = 0.5 * h1;
    else h0 = 0.5 * h0;
}

// A face of cell i from the reciprocals ahead (r0) and behind (r1) of it.
template <int NV, bool RIGHT>
__device__ __forceinline__ void weno2_face_recips(const double* s, int vs, int i, int sd, double r0, double r1,
                                                  double* out) {
    double h0, h1;
    weno2_half_weights<RIGHT>(r0, r1, h0, h1);
    const double hc = RIGHT ? 3 * h1 + h0 : 3 * h0 + h1;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double* u = s + v * vs;
        out[v] = RIGHT ? h0 * u[i + sd] + hc * u[i] - h1 * u[i - sd] : h1 * u[i - sd] + hc * u[i] - h0 * u[i + sd];
    }
}

template <int NV, bool RIGHT, class OPS>
__device__ __forceinline__ void weno2_face(const double* s, int vs, int i, int sd, double* out) {
    const double eps = 1e-8;
    const double w0 = s[i];
    const double dp = s[i + sd] - w0;
    const double dm = w0 - s[i - sd];
    if constexpr (OPS::SHARED) {
        weno2_face_recips<NV, RIGHT>(s, vs, i, sd, weno2_recip(dp), weno2_recip(dm), out);
        return;
    }
    const double b0 = dp * dp;
    const double b1 = dm * dm;
    const double d0 = 3 * (eps + b0) * (eps + b0);
    const double d1 = 3 * (eps + b1) * (eps + b1);
    if (RIGHT) {
        const double a0 = 2 / d0;
        const double a1 = 1 / d1;
        double w0r, w1r;
        weno2_weights(a0, a1, w0r, w1r);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double* u = s + v * vs;
            out[v] = 0.5 * (w0r * u[i + sd] + (3 * w1r + w0r) * u[i] - w1r * u[i - sd]);
        }
    } else {
        const double a0 = 1 / d0;
        const double a1 = 2 / d1;
        double w0l, w1l;
        weno2_weights(a0, a1, w0l, w1l);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double* u = s + v * vs;
            out[v] = 0.5 * (w1l * u[i - sd] + (3 * w0l + w1l) * u[i] - w0l * u[i + sd]);
        }
    }
}

// ENO coefficient tables (alsfvm/src/reconstruction/ENOCoefficients.cpp:27-40)
template <int ORDER>
__device__ __forceinline__ double eno_coef(int r, int j);
template <>
__device__ __forceinline__ double eno_coef<2>(int r, int j) {
    const double c00 = 3.0 / 2.0, c01 = -1.0 / 2.0, c10 = 1.0 / 2.0, c11 = 1.0 / 2.0,
                 c20 = -1.0 / 2.0, c21 = 3.0 / 2.0;
    const double a = (r == 0) ? c00 : ((r == 1) ? c10 : c20);
    const double b = (r == 0) ? c01 : ((r == 1) ? c11 : c21);
    return j == 0 ? a : b;
}
template <>
__device__ __forceinline__ double eno_coef<3>(int r, int j) {
    const double t[4][3] = {{11.0 / 6.0, -7.0 / 6.0, 1.0 / 3.0},
                            {1.0 / 3.0, 5.0 / 6.0, -1.0 / 6.0},
                            {-1.0 / 6.0, 5.0 / 6.0, 1.0 / 3.0},
                            {1.0 / 3.0, -7.0 / 6.0, 11.0 / 6.0}};
    double v = t[0][j];
    v = (r == 1) ? t[1][j] : v;
    v = (r == 2) ? t[2][j] : v;
    v = (r == 3) ? t[3][j] : v;
    return v;
}

// ENO<order> (alsfvm/src/reconstruction/ENOCPU.cpp:41-187): the stencil shift
// grows by one at each divided-difference level where |dd[x-1]| < |dd[x]|;
// divided differences are plain differences of the indicator,
// dd0[y] = w[y+1]-w[y], dd1[y] = dd0[y+1]-dd0[y] (ENOCPU.cpp:205-262).
// left face uses coefficients[shift], right face coefficients[shift+1].
template <int ORDER, int NV, bool RIGHT>
__device__ __forceinline__ void eno_face(const double* s, int vs, int i, int sd, double* out) {
    int shift = 0;
    {
        const double ddr = s[i + sd] - s[i];
        const double ddl = s[i] - s[i - sd];
        if (fabs(ddl) < fabs(ddr)) shift++;
    }
    if (ORDER == 3) {
        const double d0p = s[i + 2 * sd] - s[i + sd];
        const double d00 = s[i + sd] - s[i];
        const double d0m = s[i] - s[i - sd];
        const double ddr = d0p - d00;
        const double ddl = d00 - d0m;
        if (fabs(ddl) < fabs(ddr)) shift++;
    }
    const int r = RIGHT ? shift + 1 : shift;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double* u = s + v * vs;
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < ORDER; ++j) acc += eno_coef<ORDER>(r, j) * u[i + (j - shift) * sd];
        out[v] = acc;
    }
}

template <int RECON, int NV, bool RIGHT, class OPS>
__device__ __forceinline__ void recon_face_ops(const double* s, int vs, int i, int sd, double* out) {
    if (RECON == RECON_NONE) {
#pragma unroll
        for (int v = 0; v < NV; ++v) out[v] = s[v * vs + i];
    } else if (RECON == RECON_WENO2) {
        weno2_face<NV, RIGHT, OPS>(s, vs, i, sd, out);
    } else if (RECON == RECON_ENO2) {
        eno_face<2, NV, RIGHT>(s, vs, i, sd, out);
    } else {
        eno_face<3, NV, RIGHT>(s, vs, i, sd, out);
    }
}

}  // namespace avh
