// Per-face arithmetic of the Euler update, shared by the FP64 step kernel and
// the mixed-precision kernel (T = float for reconstruction and fluxes).
//
// Every expression keeps the reference's operation order so that, compiled
// without FP contraction, the FP64 instantiation reproduces the reference's
// results bit for bit (sound speeds use sqrt where the reference calls
// pow(x, 0.5); see the per-function citations).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#define IB_HD __host__ __device__ __forceinline__

namespace ibtfo {

enum { SCH_LAX = 0, SCH_MUSCL = 1, SCH_MHM = 2, SCH_GODUNOV = 3 };
enum { RS_HLL = 0, RS_HLLC = 1, RS_PVRS = 2, RS_SW = 3 };
enum { LIM_MINMOD = 0, LIM_VANLEER = 1, LIM_VANALBADA = 2 };

// Square root. On the device, for x in [2^-767, 2^1023] (every sound speed and
// shock factor of a physical state), the rsq seed + Goldschmidt refinement +
// two residual corrections that the compiler's IEEE sqrt runs after its range
// scaling, without the scaling and special-value fixups: the same arithmetic on
// the same operands, so the same correctly rounded result. Other x (zero,
// tiny, infinite, negative, NaN) take the full IEEE sequence.
#if defined(__HIP_DEVICE_COMPILE__)
IB_HD bool sqrt_plain(double x) { return x >= 0x1p-767 && x <= 0x1.fffffffffffffp+1023; }
IB_HD double sqrt_unscaled(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}
#endif
IB_HD double ib_sqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    double g = sqrt_unscaled(x);
    if (__builtin_expect(!sqrt_plain(x), 0)) g = __builtin_sqrt(x);
    return g;
#else
    return __builtin_sqrt(x);
#endif
}
// Two roots with one test for the rare operands, so that their chains overlap.
IB_HD void ib_sqrt2(double x, double y, double& gx, double& gy) {
#if defined(__HIP_DEVICE_COMPILE__)
    gx = sqrt_unscaled(x);
    gy = sqrt_unscaled(y);
    if (__builtin_expect(!(sqrt_plain(x) && sqrt_plain(y)), 0)) {
        gx = __builtin_sqrt(x);
        gy = __builtin_sqrt(y);
    }
#else
    gx = __builtin_sqrt(x);
    gy = __builtin_sqrt(y);
#endif
}
// FP32 (mixed-precision form): the hardware square root (1 ulp)
IB_HD float ib_sqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sqrtf(x);
#else
    return __builtin_sqrtf(x);
#endif
}
IB_HD void ib_sqrt2(float x, float y, float& gx, float& gy) {
    gx = ib_sqrt(x);
    gy = ib_sqrt(y);
}
IB_HD double ib_fabs(double x) { return __builtin_fabs(x); }
IB_HD float ib_fabs(float x) { return __builtin_fabsf(x); }

// --------------------------------------------------------------- division
// Correctly rounded quotients at a fraction of the cost of the generic IEEE
// sequence (v_div_scale x2 / v_rcp / 4 fma / mul / fma / v_div_fmas / v_div_fixup):
//  * rcp_of(b): y ~ 1/b from v_rcp_f64 (relative error below 2^-24 as measured)
//    refined by one cubic step, y + y(e + e^2) with e = 1 - b y: three fma where
//    two Newton steps take four, and the same half ulp (the seed's error cubed
//    is 2^-72);
//  * dq(a, r): q0 = a*y, residual e = b*q0 - a (exact, one fma), q = q0 - e*y
//    (Markstein's final correction, also the IEEE sequence's), which is RN(a/b).
//    With the residual taken as b*q0 - a, an exact quotient's correction is
//    (-0)*y = -0 for b > 0, which leaves q0 as it is, so a zero quotient keeps
//    IEEE's sign without a copysign (for b < 0, a non-physical density, a zero
//    quotient's sign is not IEEE's);
//    Neither form differed from IEEE division in 2.1e9 random pairs and 8.1e8
//    pairs whose quotient lies next to a rounding boundary. The kernel is bound by
//    FP64 issue: with these and the exact halvings below, the 4096x2048 cut-cell
//    step went from 316 to 297 us (HLL) and from 408 to 383 us (Steger-Warming);
//  * divisions by run constants (dx, dy, gamma, gamma-1) use y = RN(1/d)
//    computed on the host, with the same correction;
//  * one reciprocal serves all quotients with the same denominator.
// The IEEE sequence's operand scaling is omitted, so the result equals IEEE
// division for operands and quotients of magnitude in [2^-1000, 2^1000]; a zero
// or non-finite denominator gives NaN (IEEE: +-inf for a finite non-zero
// numerator), which only arises once a state is already non-physical.
template <typename T> struct Rcp { T b, y; };

IB_HD Rcp<double> rcp_of(double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y, 1.0);
    y = __builtin_fma(y, __builtin_fma(e, e, e), y);
    return Rcp<double>{b, y};
#else
    return Rcp<double>{b, 1.0 / b};
#endif
}
// FP32 (mixed-precision form): the hardware reciprocal (1 ulp) and a plain
// product, about 2 ulp per quotient; no correct rounding is attempted there.
IB_HD Rcp<float> rcp_of(float b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return Rcp<float>{b, __builtin_amdgcn_rcpf(b)};
#else
    return Rcp<float>{b, 1.0f / b};
#endif
}
IB_HD double ib_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
IB_HD float ib_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
IB_HD double ib_max(double a, double b) { return __builtin_fmax(a, b); }
template <typename T> IB_HD T dq(T a, const Rcp<T>& r) {
    T q0 = a * r.y;
    T e = ib_fma(q0, r.b, -a);
    return ib_fma(-e, r.y, q0);
}
IB_HD float dq(float a, const Rcp<float>& r) { return a * r.y; }
template <typename T> IB_HD T ddiv(T a, T b) { return dq(a, rcp_of(b)); }

// minmod/Slope_limiter.H:4: (a*b > 0) ? ((a/b > 1) ? b : a) : 0.
// For a*b > 0 the rounded quotient exceeds 1 exactly when |a| > |b|: the next
// number above |b| is larger by more than |b| 2^-53 (half the spacing above 1),
// in the subnormal range too; equal infinities and NaN compare false both ways.
// So no division, and with a = b the only case in which the order of the
// arguments could matter, a cell's two slopes in one direction are one value.
template <typename T> IB_HD T lim_minmod(T a, T b) {
    const T m = ib_fabs(a) > ib_fabs(b) ? b : a;
    return a * b > T(0) ? m : T(0);
}
// VanLeer/Slope_limiter.H:4 as expanded at the call sites, whose second argument
// is the unparenthesised difference P - Q: `(r*r + r) * b / (r*r + 1)` becomes
// (r*r + r)*P - Q/(r*r + 1).
template <typename T> IB_HD T lim_vanleer_ref(T a, T P, T Q) {
    T r = ddiv(a + T(1e-7), (P - Q) + T(1e-7));
    return (r > T(0)) ? ((r * r + r) * P - ddiv(Q, r * r + T(1))) : T(0);
}
// The same limiter with its argument parenthesised (corrected mode), written
// with one division: with A = a + 1e-7, B = b + 1e-7 and r = A/B,
// (r*r + r) b / (r*r + 1) = b A (A + B) / (A*A + B*B), and r > 0 iff A*B > 0.
// lim(a, b) and lim(b, a) share the denominator, so a cell's two slopes in one
// direction cost one reciprocal (vanleer_pair).
template <typename T> IB_HD T lim_vanleer_fixed(T a, T b) {
    T A = a + T(1e-7), B = b + T(1e-7);
    return (A * B > T(0)) ? ddiv(b * (A * (A + B)), A * A + B * B) : T(0);
}
// {lim(a, b), lim(b, a)} of lim_vanleer_fixed. FLAT evaluates the quotients before
// the selects, so that the four components' chains overlap (a wave with few others
// beside it); else each component becomes a branch of its own, with far fewer
// registers (the cut-cell marching strip in FP64: 121 VGPRs instead of 141).
template <bool FLAT, typename T> IB_HD void vanleer_pair(T a, T b, T& sab, T& sba) {
    T A = a + T(1e-7), B = b + T(1e-7);
    T n = A + B;
    Rcp<T> rd = rcp_of(A * A + B * B);
    const bool pos = A * B > T(0);
    if (FLAT) {
        const T qab = dq(b * (A * n), rd), qba = dq(a * (B * n), rd);
        sab = pos ? qab : T(0);
        sba = pos ? qba : T(0);
    } else {
        sab = pos ? dq(b * (A * n), rd) : T(0);
        sba = pos ? dq(a * (B * n), rd) : T(0);
    }
}
// VanAlbada/Slope_limiter.H:4 does not compile (undeclared r); its evident
// intent, with r defined as in the sibling limiter.
template <typename T> IB_HD T lim_vanalbada(T a, T b) {
    T r = ddiv(a + T(1e-7), b + T(1e-7));
    return (r > T(0)) ? ddiv((r + ib_fabs(r)) * b, T(1) + ib_fabs(r)) : T(0);
}
template <int LIM, typename T> IB_HD T slope(T a, T P, T Q, bool quirks) {
    if (LIM == LIM_MINMOD) return lim_minmod(a, P - Q);
    if (LIM == LIM_VANLEER) return quirks ? lim_vanleer_ref(a, P, Q) : lim_vanleer_fixed(a, P - Q);
    return lim_vanalbada(a, P - Q);
}

// Both slopes of one cell from its neighbours um, u0, up (per component):
// lo = u0 + 0.5 lim(u0 - um, up - u0) is the cell's state on its upper face
// (U_L of face +1/2), hi = u0 - 0.5 lim(up - u0, u0 - um) its state on its lower
// face (U_R of face -1/2); recon() below evaluates the same expressions face by face.
template <int LIM, bool FLAT, typename T> IB_HD void slope_pair(const T* um, const T* u0, const T* up, T* lo, T* hi,
                                                                bool quirks) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        T sl, sh;
        if (LIM == LIM_MINMOD) {
            sl = sh = lim_minmod(u0[k] - um[k], up[k] - u0[k]);
        } else if (LIM == LIM_VANLEER && !quirks) {
            vanleer_pair<FLAT>(u0[k] - um[k], up[k] - u0[k], sl, sh);
        } else {
            sl = slope<LIM>(u0[k] - um[k], up[k], u0[k], quirks);
            sh = slope<LIM>(up[k] - u0[k], u0[k], um[k], quirks);
        }
        lo[k] = ib_fma(T(0.5), sl, u0[k]);  // the halving is exact, so this is the sum's own rounding
        hi[k] = ib_fma(T(-0.5), sh, u0[k]);
    }
}

// Face states from the 4 cells around face i+1/2 (MUSCL_Scheme.cpp:83-85, :99-101):
// U_L = U_i + 0.5*lim(U_i - U_{i-1}, U_{i+1} - U_i),
// U_R = U_{i+1} - 0.5*lim(U_{i+2} - U_{i+1}, U_{i+1} - U_i).
template <int LIM, typename T> IB_HD void recon(const T* u0, const T* u1, const T* u2, const T* u3, T* UL, T* UR,
                                                 bool quirks) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        UL[k] = u1[k] + T(0.5) * slope<LIM>(u1[k] - u0[k], u2[k], u1[k], quirks);
        UR[k] = u2[k] - T(0.5) * slope<LIM>(u3[k] - u2[k], u2[k], u1[k], quirks);
    }
}

// Gas and mesh constants, with the reciprocals of the constant divisors.
template <typename T> struct GasT {
    T gam, gm1, gp1, c1;  // gamma, gamma-1, gamma+1, (gamma-1)/2/gamma
    Rcp<T> r_gam, r_gm1, r_dx, r_dy;
};

// primitive view of a conserved state (rho, u, v, p), with 1/rho kept for reuse
template <typename T> struct PState {
    T rho, u, v, p, E;
    Rcp<T> ir;
};
// Conserve2Flux.cpp:66-69: u = rho u / rho, v = rho v / rho, p = (gamma-1)(E - rho(u^2+v^2)/2)
template <typename T> IB_HD PState<T> pstate(T gm1, const T* U) {
    PState<T> s;
    s.rho = U[0];
    s.ir = rcp_of(s.rho);
    s.u = dq(U[1], s.ir);
    s.v = dq(U[2], s.ir);
    // 0.5 rho (u^2 + v^2) is half of the rounded rho (u^2 + v^2), exactly
    s.p = gm1 * ib_fma(T(-0.5), s.rho * (s.u * s.u + s.v * s.v), U[3]);
    s.E = U[3];
    return s;
}
// sqrt(gamma p / rho) of both states of a face, where the reference calls pow(gamma p / rho, 0.5)
template <typename T> IB_HD void sounds(const GasT<T>& g, const PState<T>& L, const PState<T>& R, T& al, T& ah) {
    ib_sqrt2(dq(g.gam * L.p, L.ir), dq(g.gam * R.p, R.ir), al, ah);
}

// Conserve2Flux.cpp:71-74 (x) / :106-109 (y): physical flux of a conserved state.
// The tangential momentum term is rho*u*v evaluated left to right in both directions.
template <bool Y, typename T> IB_HD void phys_flux(T rho, T u, T v, T p, T E, T* F) {
    if (!Y) { F[0] = rho * u; F[1] = rho * u * u + p; F[2] = rho * u * v; F[3] = (E + p) * u; }
    else { F[0] = rho * v; F[1] = rho * u * v; F[2] = rho * v * v + p; F[3] = (E + p) * v; }
}
template <bool Y, typename T> IB_HD void phys_flux(const PState<T>& s, T* F) { phys_flux<Y>(s.rho, s.u, s.v, s.p, s.E, F); }
template <typename T> IB_HD void primitives(T gm1, const T* U, T& rho, T& u, T& v, T& p) {
    rho = U[0]; u = U[1] / rho; v = U[2] / rho;
    p = gm1 * (U[3] - T(0.5) * rho * (u * u + v * v));
}
template <bool Y, typename T> IB_HD void flux_of(T gm1, const T* U, T* F) {
    PState<T> s = pstate(gm1, U);
    phys_flux<Y>(s, F);
}

// Corrected mode only (no reference counterpart): positivity of a state, the
// per-face first-order fallback and the density/pressure floors (applied to
// updated fluid cells: rho <- max(rho, RHO_FLOOR); if p <= P_FLOOR,
// E <- P_FLOOR/(gamma-1) + kinetic energy).
template <typename T> IB_HD bool physical(const PState<T>& s) { return s.rho > T(0) && s.p > T(0); }
constexpr double RHO_FLOOR = 1e-8, P_FLOOR = 1e-8;

// HLL/Riemann_solver.cpp:131-168 (x), :202-235 (y). Returns true when the
// first branch (S_lo >= 0) is taken; F is then F(U_lo) (the y solver's caller
// decides what that branch stores).
// The reference's expressions, with their factors 1/2 moved to where an fma takes
// them: a power of two scales exactly, so every rounding is the reference's. The
// right wave speed is evaluated only where the left one leaves the choice open
// (supersonic faces end at F(U_lo): a third of the solver's work).
template <bool Y, typename T>
IB_HD bool hll_face(const GasT<T>& g, const PState<T>& L, const PState<T>& R, const T* Ulo, const T* Uhi, T* F,
                    bool quirks) {
    const T unl = Y ? L.v : L.u, unh = Y ? R.v : R.u;
    T al, ah;
    sounds(g, L, R, al, ah);
    // p* = (p_lo + p_hi)/2 + (un_lo - un_hi)/2 * (rho_bar * a_bar)
    const T x = (unl - unh) * ((L.rho + R.rho) * (al + ah));
    T p_star = ib_fma(T(0.125), x, T(0.5) * (L.p + R.p));
    // corrected estimate (Toro, Riemann Solvers, 3rd ed., eq. 10.59-10.60): p* >= 0 and
    // the shock factor only where p* exceeds the side's pressure
    if (!quirks) p_star = p_star > T(0) ? p_star : T(0);
    const T t = dq(g.gp1 * p_star, g.r_gam);
    // sqrt((gamma+1) p* / 2 / gamma / p_K + (gamma-1)/2/gamma)
    auto factor = [&](T pK) { return ib_sqrt(ib_fma(T(0.5), ddiv(t, pK), g.c1)); };
    T ql = T(1), qh = T(1);
    if (quirks || !(p_star <= L.p)) ql = factor(L.p);
    const T Sl = unl - al * ql;
    T Fl[4], Fh[4];
    phys_flux<Y>(L, Fl);
    if (Sl >= T(0)) {
#pragma unroll
        for (int k = 0; k < 4; k++) F[k] = Fl[k];
        return true;
    }
    if (quirks || !(p_star <= R.p)) qh = factor(R.p);
    const T Sh = unh + ah * qh;
    phys_flux<Y>(R, Fh);
    if (Sh <= T(0)) {
#pragma unroll
        for (int k = 0; k < 4; k++) F[k] = Fh[k];
        return false;
    }
    Rcp<T> iw = rcp_of(Sh - Sl);
#pragma unroll
    for (int k = 0; k < 4; k++) F[k] = dq(Sh * Fl[k] - Sl * Fh[k] + Sh * Sl * (Uhi[k] - Ulo[k]), iw);
    return false;
}

// StegerWarming/Riemann_solver.cpp:184-234 (x), :274-325 (y): F+(U_lo) + F-(U_hi)
// with eigenvalue smoothing delta = 1e-6. un/ut = normal/tangential velocity.
template <bool Y, typename T> IB_HD void sw_half(const GasT<T>& g, T rho, T un, T ut, T a, T h, bool plus, T* out) {
    const T d2 = T(1e-6) * T(1e-6);
    T s1 = ib_sqrt(un * un + d2);
    T m = un - a, q = un + a;
    T s3 = ib_sqrt(m * m + d2), s4 = ib_sqrt(q * q + d2);
    T l1 = plus ? T(0.5) * (un + s1) : T(0.5) * (un - s1);
    T l3 = plus ? T(0.5) * (m + s3) : T(0.5) * (m - s3);
    T l4 = plus ? T(0.5) * (q + s4) : T(0.5) * (q - s4);
    T u2 = Y ? (ut * ut + un * un) : (un * un + ut * ut);
    T twogm1 = T(2) * g.gm1;
    // rho * (...) / 2 / gamma
    out[0] = dq(rho * (twogm1 * l1 + l3 + l4) * T(0.5), g.r_gam);
    out[1] = dq(rho * (twogm1 * un * l1 + (un - a) * l3 + (un + a) * l4) * T(0.5), g.r_gam);
    out[2] = dq(rho * (twogm1 * ut * l1 + l3 * ut + l4 * ut) * T(0.5), g.r_gam);
    out[3] = dq(rho * (g.gm1 * u2 * l1 + (h - a * un) * l3 + (h + a * un) * l4) * T(0.5), g.r_gam);
}
template <bool Y, typename T> IB_HD void sw_face(const GasT<T>& g, const PState<T>& L, const PState<T>& R, T* F) {
    T al, ah;
    sounds(g, L, R, al, ah);
    // e = p / (gamma-1) / rho ; h = e + u*u/2 + v*v/2 + p/rho
    T el = dq(dq(L.p, g.r_gm1), L.ir), eh = dq(dq(R.p, g.r_gm1), R.ir);
    T hl = el + L.u * L.u * T(0.5) + L.v * L.v * T(0.5) + dq(L.p, L.ir);
    T hh = eh + R.u * R.u * T(0.5) + R.v * R.v * T(0.5) + dq(R.p, R.ir);
    T fp[4], fn[4];
    sw_half<Y>(g, L.rho, Y ? L.v : L.u, Y ? L.u : L.v, al, hl, true, fp);
    sw_half<Y>(g, R.rho, Y ? R.v : R.u, Y ? R.u : R.v, ah, hh, false, fn);
    if (!Y) {
        F[0] = fp[0] + fn[0]; F[1] = fp[1] + fn[1]; F[2] = fp[2] + fn[2]; F[3] = fp[3] + fn[3];
    } else {
        F[0] = fp[0] + fn[0]; F[1] = fp[2] + fn[2]; F[2] = fp[1] + fn[1]; F[3] = fp[3] + fn[3];
    }
}

// PVRS/Riemann_solver.cpp:308-435 (x), :463-589 (y). The y solver's stray
// store at :550 (energy flux written through the state index macro into another
// cell's record) is not reproduced: in the reference's parallel builds its
// target is raced; here that branch leaves the energy slot as the reference's
// own slot would be left (the aliased x-flux), reported through `stray`.
template <bool Y, typename T> IB_HD void pvrs_face(const GasT<T>& g, const T* Ulo, const T* Uhi, T* F, bool& stray) {
    T rl, ul, vl, pl, rh, uh, vh, ph;
    primitives(g.gm1, Ulo, rl, ul, vl, pl);
    primitives(g.gm1, Uhi, rh, uh, vh, ph);
    T unl = Y ? vl : ul, utl = Y ? ul : vl, unh = Y ? vh : uh, uth = Y ? uh : vh;
    T al = ib_sqrt(g.gam * pl / rl), ah = ib_sqrt(g.gam * ph / rh);
    T rho_bar = T(0.5) * (rl + rh);
    T a_bar = T(0.5) * (al + ah);
    T p_star = T(0.5) * (pl + ph) + T(0.5) * (unl - unh) * (rho_bar * a_bar);
    T u_star = T(0.5) * (unl + unh) + T(0.5) * (pl - ph) / (rho_bar * a_bar);
    T rl_star = rl + (p_star - pl) / al / al;
    T rh_star = rh + (p_star - ph) / ah / ah;
    T Sl = unl - al * ib_sqrt(g.gp1 * p_star / T(2) / g.gam / pl + g.c1);
    T Sh = unh + ah * ib_sqrt(g.gp1 * p_star / T(2) / g.gam / ph + g.c1);
    T S_Hl = unl - al;
    T S_Tl = u_star - pow(al * (p_star / ph), g.c1);
    T S_Hh = unh + ah;
    T S_Th = u_star + pow(ah * (p_star / ph), g.c1);
    T f[4];  // normal mass, normal momentum, tangential momentum, energy
    stray = false;
    auto side = [&](T rho, T un, T ut, T p, T E) {
        f[0] = rho * un; f[1] = rho * un * un + p; f[2] = Y ? rho * ut * un : rho * un * ut; f[3] = (E + p) * un;
    };
    auto star = [&](T rs, T ut) {
        f[0] = rs * u_star; f[1] = rs * u_star * u_star + p_star; f[2] = rs * u_star * ut;
        f[3] = (g.gam * p_star / g.gm1 + T(0.5) * rs * (u_star * u_star + ut * ut)) * u_star;
    };
    auto fan = [&](T rho, T un, T ut, T p, T as) {
        T base = T(2) / g.gp1 + g.gm1 * (rho) / g.gp1 / as;
        T rf = rho * pow(base, T(2) / g.gm1);
        T uf = T(2) * (as + g.gm1 * un / T(2)) / g.gp1;
        T pf = p * pow(base, T(2) * g.gam / g.gm1);
        f[0] = rf * uf; f[1] = rf * uf * uf + pf; f[2] = rf * uf * ut;
        f[3] = (g.gam * pf / g.gm1 + T(0.5) * rf * (uf * uf + ut * ut)) * uf;
    };
    if (u_star > T(0)) {
        if (p_star > pl) { if (Sl > T(0)) side(rl, unl, utl, pl, Ulo[3]); else star(rl_star, utl); }
        else if (S_Hl > T(0)) side(rl, unl, utl, pl, Ulo[3]);
        else if (S_Tl < T(0)) star(rl_star, utl);
        else fan(rl, unl, utl, pl, al);
    } else {
        if (p_star > ph) {
            if (Sh < T(0)) { side(rh, unh, uth, ph, Uhi[3]); stray = Y; }
            else star(rh_star, uth);
        } else if (S_Hh < T(0)) side(rh, unh, uth, ph, Uhi[3]);
        else if (S_Th > T(0)) star(rh_star, uth);
        else fan(rh, unh, uth, ph, ah);
    }
    if (!Y) { F[0] = f[0]; F[1] = f[1]; F[2] = f[2]; F[3] = f[3]; }
    else { F[0] = f[0]; F[1] = f[2]; F[2] = f[1]; F[3] = f[3]; }
}

}  // namespace ibtfo
