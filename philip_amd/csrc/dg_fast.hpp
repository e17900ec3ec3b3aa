// Cached-node point physics of the line kernels, direction K fixed at compile
// time, in the arithmetic type T: float on the mixed path, double on the FP64
// path.  Each function is an algebraic restatement of the point physics in
// dg_physics.hpp (same formula in exact arithmetic) arranged to use few
// divisions: per-node quantities (1/rho, pressure, beta, sqrt(rho), sound
// speed, enthalpy) are computed once per node and reused by every pair and
// face that touches the node.  In float the reciprocals, square roots and
// logarithms are the hardware v_rcp_f32 / v_sqrt_f32 / v_log_f32 instructions;
// in double the reciprocal is v_rcp_f64 with a third-order step, the square root v_rsq_f64 with
// Newton steps, the logarithm the library's double routine.
//
//   ec_flux_fast   Chandrashekar / Ranocha two-point flux (euler.cpp:709-807):
//                  log means from f = (a-b)/(a+b), and 1/(2 beta_ln (gamma-1))
//                  and p_hat/rho_ln expressed through F_beta, F_rho and
//                  1/(beta1+beta2), so a pair costs three reciprocals.
//   roe_fast       Roe-Pike + Harten entropy fix (convective_numerical_flux.cpp:
//                  332-480) with Roe averages from sqrt(rho) of each side.
//   num_flux_fast  baseline (central or two-point) + dissipation (LxF / Roe)
//                  (convective_numerical_flux.cpp:34-54).
//
// The FP64 path's VALU issue is what its stage kernels spend most of their time on, so its
// versions (the *64 functions) are arranged for fewer instructions than the float ones: one
// reciprocal serves both 1/(rho1+rho2) and 1/(b1+b2), 1/F_rho comes from its expansion and one
// Newton step, and |avg v|^2 - avg |v|^2 / 2 is v1.v2 / 2.  Every sum over the two sides is written so that exchanging them and turning the
// normal around gives the exact negative, so a face evaluated from either side needs no
// selection of an owner (the Kennedy-Gruber and Ismail-Roe fluxes are ordered by it).  They take a direction K or (CV) a normal / cofactor column nv.
#pragma once
#include <type_traits>

#include "dg_physics.hpp"
#include "dg_rules.hpp"

namespace dgx {

template <typename T> struct Fast;
#ifndef DGX_HOST_TEST
template <> struct Fast<float> {
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    static __device__ __forceinline__ float sqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }
    static __device__ __forceinline__ float log_(float x) { return __logf(x); }
};
template <> struct Fast<double> {
    // v_rcp_f64 (within 4.6e-8 of 1/x) refined by one third-order step r (1 + e + e^2), e = 1 - x r:
    // the remaining relative error is e^3 ~ 1e-22, so the result is rounded once, at one FMA less
    // than two Newton-Raphson steps
    static __device__ __forceinline__ double rcp(double x)
    {
        const double r = __builtin_amdgcn_rcp(x);
        const double e = __builtin_fma(-x, r, 1.0);
        const double t = __builtin_fma(e, e, e);
        return __builtin_fma(r, t, r);
    }
    // sqrt(x) and 1/sqrt(x) from v_rsq_f64 by one coupled Newton (Goldschmidt) step and one residual
    // correction each; no scaling (x is a density, a squared sound speed or a squared area).
    // x = 0 and x = inf, whose products are NaN, are returned as they are.
    static __device__ __forceinline__ void sqrt_rsqrt(double x, double *root, double *inv)
    {
        const double y = __builtin_amdgcn_rsq(x);
        double g = x * y, h = 0.5 * y;
        const double r = __builtin_fma(-h, g, 0.5);
        g = __builtin_fma(g, r, g);
        h = __builtin_fma(h, r, h);
        const double d = __builtin_fma(-g, g, x);
        g = __builtin_fma(d, h, g);
        *root = __builtin_amdgcn_class(x, 0x260) ? x : g;  // -0, +0, +inf
        const double q = __builtin_fma(-h, g, 0.5);
        *inv = 2.0 * __builtin_fma(h, q, h);
    }
    static __device__ __forceinline__ double sqrt_(double x)
    {
        double g, h;
        sqrt_rsqrt(x, &g, &h);
        return g;
    }
    static __device__ __forceinline__ double log_(double x) { return log(x); }
};
#else
// host build of the same formulas (CPU checks of the restatement)
template <typename T> struct FastHost {
    static inline T rcp(T x) { return T(1) / x; }
    static inline T sqrt_(T x) { return std::sqrt(x); }
    static inline T log_(T x) { return std::log(x); }
};
template <> struct Fast<float> : FastHost<float> {};
template <> struct Fast<double> : FastHost<double> {
    static inline void sqrt_rsqrt(double x, double *root, double *inv)
    {
        *root = std::sqrt(x);
        *inv = 1.0 / *root;
    }
};
#endif
template <typename T> __device__ __forceinline__ T frcp(T x) { return Fast<T>::rcp(x); }
template <typename T> __device__ __forceinline__ T fsqrt(T x) { return Fast<T>::sqrt_(x); }
template <typename T> __device__ __forceinline__ T flog(T x) { return Fast<T>::log_(x); }
template <typename T> __device__ __forceinline__ T fmx(T a, T b) { return a > b ? a : b; }
template <typename T> __device__ __forceinline__ T fab(T a) { return a < T(0) ? -a : a; }

// Per-node cache: conservative state and derived quantities.
template <typename T, int D> struct NodeC {
    T u[D + 2];
    T vel[D];
    T p, b, v2, sr, c, h;  // pressure, beta, |v|^2, sqrt(rho), sound speed, total enthalpy
};

template <typename T> struct FastConst {
    T gam, gamm1, inv_gamm1;
    int two_point, conv_flux;
};

template <typename T> __device__ __forceinline__ FastConst<T> fast_const(const PhysConst &pc)
{
    FastConst<T> f;
    f.gam = T(pc.gam);
    f.gamm1 = T(pc.gamm1);
    f.inv_gamm1 = T(1.0 / pc.gamm1);
    f.two_point = pc.two_point;
    f.conv_flux = pc.conv_flux;
    return f;
}

// Fills every field of q from q.u; beta is rho/(2p) (Chandrashekar) or rho/p (Ranocha).  In double
// |v|^2, which the FP64 fluxes do not use, is left out.  (One reciprocal 1/(rho e), e = rho E -
// |m|^2/2, for both 1/rho and 1/p took three operations less and left p three times further off; the
// pressure's rounding is what a residual at low Mach number is made of.)
template <typename T, int D>
__device__ __forceinline__ void node_fill(NodeC<T, D> &q, const FastConst<T> &fc)
{
    if constexpr (std::is_same<T, double>::value) {
        const double ir = frcp<double>(q.u[0]);
        double v2 = 0.0;
        for (int k = 0; k < D; ++k) {
            q.vel[k] = q.u[1 + k] * ir;
            v2 += q.vel[k] * q.vel[k];
        }
        q.p = fc.gamm1 * (q.u[D + 1] - 0.5 * q.u[0] * v2);
        const double rp = q.u[0] * frcp<double>(q.p);
        q.b = (fc.two_point == 3) ? rp : 0.5 * rp;
        q.sr = fsqrt<double>(q.u[0]);
        q.c = fsqrt<double>(fc.gam * q.p * ir);
        q.h = (q.u[D + 1] + q.p) * ir;
        return;
    }
    const T ir = frcp<T>(q.u[0]);
    T v2 = T(0);
    for (int k = 0; k < D; ++k) {
        q.vel[k] = q.u[1 + k] * ir;
        v2 += q.vel[k] * q.vel[k];
    }
    q.v2 = v2;
    q.p = fc.gamm1 * (q.u[D + 1] - T(0.5) * q.u[0] * v2);
    const T rp = q.u[0] * frcp<T>(q.p);
    q.b = (fc.two_point == 3) ? rp : T(0.5) * rp;
    q.sr = fsqrt<T>(q.u[0]);
    q.c = fsqrt<T>(fc.gam * q.p * ir);
    q.h = (q.u[D + 1] + q.p) * ir;
}

// F of the Ismail-Roe log mean  mean_ln(a, b) = (a + b) / (2 F),  f = (a - b) / (a + b)
// (series branch below 1e-2 as euler.cpp:629-647, Horner form with constant reciprocals).
template <typename T>
__device__ __forceinline__ T log_mean_F(T a, T b, T f)
{
    const T uu = f * f;
    if (uu < T(1.0e-2)) return T(1) + uu * (T(1.0 / 3.0) + uu * (T(1.0 / 5.0) + uu * T(1.0 / 7.0)));
    return T(0.5) * flog<T>(a * frcp<T>(b)) * frcp<T>(f);
}

template <typename T, int D, int K>
__device__ __forceinline__ void ec_flux_fast(const T rho1, const T *v1, const T p1, const T b1, const T q1v2,
                                             const T rho2, const T *v2, const T p2, const T b2, const T q2v2,
                                             const FastConst<T> &fc, T *f)
{
    const bool ra = (fc.two_point == 3);
    const T sr = rho1 + rho2, isr = frcp<T>(sr);
    const T Fr = log_mean_F<T>(rho1, rho2, (rho1 - rho2) * isr);
    const T sb = b1 + b2, isb = frcp<T>(sb);
    const T Fb = log_mean_F<T>(b1, b2, (b1 - b2) * isb);
    const T rho_ln = T(0.5) * sr * frcp<T>(Fr);
    T va[D], vsq = T(0);
    for (int k = 0; k < D; ++k) {
        va[k] = T(0.5) * (v1[k] + v2[k]);
        vsq += va[k] * va[k];
    }
    T p_hat, H;
    if (ra) {
        p_hat = T(0.5) * (p1 + p2);
        H = T(2) * Fb * isb * fc.inv_gamm1 + T(4) * p_hat * Fr * isr;
    } else {
        p_hat = T(0.5) * sr * isb;
        H = isb * (Fb * fc.inv_gamm1 + Fr);
    }
    H += vsq - T(0.25) * (q1v2 + q2v2);
    const T m = rho_ln * va[K];
    f[0] = m;
    for (int vd = 0; vd < D; ++vd) f[1 + vd] = m * va[vd];
    f[1 + K] += p_hat;
    f[D + 1] = m * H;
    if (ra) f[D + 1] -= T(0.5) * (p1 * v1[K] + p2 * v2[K]);
}

// The same in double (Chandrashekar / Ranocha), along e_K or (CV) contracted with nv.  1/F_rho: the
// expansion of x / atanh x to u^3 is within 1e-9 of it for u < 1e-2, one Newton step squares that.
template <int D, int K, bool CV>
__device__ __forceinline__ void ec_flux64(const NodeC<double, D> &a, const NodeC<double, D> &b, const double *nv,
                                          const FastConst<double> &fc, double *f)
{
    const bool ra = (fc.two_point == 3);
    const double sr = a.u[0] + b.u[0], sb = a.b + b.b;
    const double t = frcp<double>(sr * sb);
    // 1/(b1+b2) carries the pressure: one more Newton step takes the products' rounding out again
    const double isr = t * sb, isb0 = t * sr, isb = isb0 + isb0 * (1.0 - sb * isb0);
    const double fr = (a.u[0] - b.u[0]) * isr, fb = (a.b - b.b) * isb;
    const double ur = fr * fr, ub = fb * fb;
    double Fr = 1.0 + ur * (1.0 / 3.0 + ur * (1.0 / 5.0 + ur * (1.0 / 7.0)));
    double Fb = 1.0 + ub * (1.0 / 3.0 + ub * (1.0 / 5.0 + ub * (1.0 / 7.0)));
    const double g = 1.0 - ur * (1.0 / 3.0 + ur * (4.0 / 45.0 + ur * (44.0 / 945.0)));
    double iFr = g + g * (1.0 - Fr * g);
    if (__builtin_expect(!(ur < 1.0e-2 && ub < 1.0e-2), 0)) {
        // larger over smaller: the same bits whichever side is a
        if (!(ur < 1.0e-2)) {
            const bool gt = a.u[0] > b.u[0];
            const double hi = gt ? a.u[0] : b.u[0], lo = gt ? b.u[0] : a.u[0];
            Fr = 0.5 * flog<double>(hi * frcp<double>(lo)) * frcp<double>(fab<double>(fr));
            iFr = frcp<double>(Fr);
        }
        if (!(ub < 1.0e-2)) {
            const bool gt = a.b > b.b;
            const double hi = gt ? a.b : b.b, lo = gt ? b.b : a.b;
            Fb = 0.5 * flog<double>(hi * frcp<double>(lo)) * frcp<double>(fab<double>(fb));
        }
    }
    double w[D], dot = a.vel[0] * b.vel[0], wn = 0.0;
    for (int k = 0; k < D; ++k) w[k] = a.vel[k] + b.vel[k];
    for (int k = 1; k < D; ++k) dot += a.vel[k] * b.vel[k];
    if constexpr (CV) {
        wn = w[0] * nv[0];
        for (int k = 1; k < D; ++k) wn += w[k] * nv[k];
    } else {
        wn = w[K];
    }
    double p_hat, H;
    if (ra) {
        p_hat = 0.5 * (a.p + b.p);
        H = 2.0 * (Fb * isb * fc.inv_gamm1) + 4.0 * p_hat * (Fr * isr);
    } else {
        p_hat = 0.5 * sr * isb;
        H = isb * (Fb * fc.inv_gamm1 + Fr);
    }
    H += 0.5 * dot;
    const double m = 0.25 * sr * iFr * wn, hm = 0.5 * m;
    f[0] = m;
    if constexpr (CV) {
        for (int vd = 0; vd < D; ++vd) f[1 + vd] = hm * w[vd] + p_hat * nv[vd];
    } else {
        for (int vd = 0; vd < D; ++vd) f[1 + vd] = (vd == K) ? hm * w[vd] + p_hat : hm * w[vd];
    }
    f[D + 1] = m * H;
    if (ra) {
        double pa, pb;
        if constexpr (CV) {
            double va = a.vel[0] * nv[0], vb = b.vel[0] * nv[0];
            for (int k = 1; k < D; ++k) {
                va += a.vel[k] * nv[k];
                vb += b.vel[k] * nv[k];
            }
            pa = a.p * va;
            pb = b.p * vb;
        } else {
            pa = a.p * a.vel[K];
            pb = b.p * b.vel[K];
        }
        const double pw = pa + pb;
        f[D + 1] -= 0.5 * pw;
    }
}

// What a form keeps in two fields of a node's FP64 cache (rho, v, p, beta, H, c, sqrt(rho)): the
// conservative form the momentum in the velocity's place and 1/rho in beta's, so that the mass flux is
// the momentum itself, as it is in a trace; Kennedy-Gruber and Ismail-Roe, which have no beta, E there.
// Lax-Friedrichs dissipation, which does not read sqrt(rho), has E in that field in every form
// (energy_in_sr): read from memory by the face items instead, E was a round trip in the middle of the
// line phase (conservative rhs in small blocks, 3D p=1 20^3 12.3 -> 10.1 us, p=2 13^3 11.0 -> 8.9 us).
__device__ __forceinline__ bool energy_in_sr(int conv_flux) { return conv_flux == 0 || conv_flux == 4; }
template <int D, int FORM>
__device__ __forceinline__ void node_to_cache64(const FastConst<double> &fc, NodeC<double, D> &n)
{
    if (energy_in_sr(fc.conv_flux)) n.sr = n.u[D + 1];
    if constexpr (FORM == FORM_CONS) {
        for (int k = 0; k < D; ++k) n.vel[k] = n.u[1 + k];
        n.b = frcp<double>(n.u[0]);
    } else if constexpr (FORM == FORM_GEN) {
        n.b = n.u[D + 1];
    }
}
template <int D, int FORM> __device__ __forceinline__ void node_from_cache64(NodeC<double, D> &n)
{
    if constexpr (FORM == FORM_CONS) {
        for (int k = 0; k < D; ++k) {
            n.u[1 + k] = n.vel[k];
            n.vel[k] = n.u[1 + k] * n.b;
        }
    } else if constexpr (FORM == FORM_GEN) {
        n.u[D + 1] = n.b;
    }
}

// Kennedy-Gruber and Ismail-Roe of two nodes through the generic evaluation of dg_physics.hpp (CV:
// contracted with nv).  Kennedy-Gruber averages E / rho: E is the node's own (rebuilt as rho H - p its
// rounding makes the energy flux a fifth less accurate).
template <int D, int K, bool CV>
__device__ __forceinline__ void other_flux64(const NodeC<double, D> &a, const NodeC<double, D> &b, const double *nv,
                                             const PhysConst &pc, double *f)
{
    Prim<double, D> qa, qb;
    double ua[D + 2], ub[D + 2];
    qa.rho = ua[0] = a.u[0];
    qb.rho = ub[0] = b.u[0];
    for (int k = 0; k < D; ++k) {
        qa.vel[k] = a.vel[k];
        qb.vel[k] = b.vel[k];
        ua[1 + k] = a.u[0] * a.vel[k];
        ub[1 + k] = b.u[0] * b.vel[k];
    }
    qa.p = a.p;
    qb.p = b.p;
    ua[D + 1] = a.u[D + 1];
    ub[D + 1] = b.u[D + 1];
    if constexpr (CV) two_point_flux_vec<double, D>(ua, qa, ub, qb, nv, pc, f);
    else two_point_flux_dir<double, D>(ua, qa, ub, qb, K, pc, f);
}

// Two-point flux of two cached nodes; Kennedy-Gruber and Ismail-Roe go through
// the generic evaluation of dg_physics.hpp.
template <typename T, int D, int K>
__device__ __forceinline__ void pair_flux_fast(const NodeC<T, D> &a, const NodeC<T, D> &b, const FastConst<T> &fc,
                                               const PhysConst &pc, T *f)
{
    if constexpr (std::is_same<T, double>::value) {
        if (fc.two_point >= 2) ec_flux64<D, K, false>(a, b, nullptr, fc, f);
        else other_flux64<D, K, false>(a, b, nullptr, pc, f);
        return;
    }
    if (fc.two_point >= 2) {
        ec_flux_fast<T, D, K>(a.u[0], a.vel, a.p, a.b, a.v2, b.u[0], b.vel, b.p, b.b, b.v2, fc, f);
    } else {
        Prim<T, D> qa, qb;
        qa.rho = a.u[0];
        qb.rho = b.u[0];
        for (int k = 0; k < D; ++k) {
            qa.vel[k] = a.vel[k];
            qb.vel[k] = b.vel[k];
        }
        qa.p = a.p;
        qb.p = b.p;
        two_point_flux_dir<T, D>(a.u, qa, b.u, qb, K, pc, f);
    }
}

template <typename T, int D, int K>
__device__ __forceinline__ void roe_fast(const NodeC<T, D> &L, const NodeC<T, D> &R, T sgn, const FastConst<T> &fc,
                                         T *out)
{
    const T vnL = L.vel[K] * sgn, vnR = R.vel[K] * sgn;
    const T isum = frcp<T>(L.sr + R.sr);
    const T rho_ravg = L.sr * R.sr;
    T v_ravg[D], vel2 = T(0);
    for (int k = 0; k < D; ++k) {
        v_ravg[k] = (R.sr * R.vel[k] + L.sr * L.vel[k]) * isum;
        vel2 += v_ravg[k] * v_ravg[k];
    }
    const T h_ravg = (R.sr * R.h + L.sr * L.h) * isum;
    const T vn = v_ravg[K] * sgn;
    const T c2 = fc.gamm1 * (h_ravg - T(0.5) * vel2);
    const T c = (c2 > T(0)) ? fsqrt<T>(c2) : T(1e10);
    T eig[3] = {fab<T>(vn - c), fab<T>(vn), fab<T>(vn + c)};
    const T eL[3] = {fab<T>(vnL - L.c), fab<T>(vnL), fab<T>(vnL + L.c)};
    const T eR[3] = {fab<T>(vnR - R.c), fab<T>(vnR), fab<T>(vnR + R.c)};
    for (int e = 0; e < 3; ++e) {
        const T eps = fmx<T>(fab<T>(eig[e] - eL[e]), fab<T>(eR[e] - eig[e]));
        if (eig[e] < eps) eig[e] = T(0.5) * (eig[e] * eig[e] * frcp<T>(eps) + eps);
    }
    const T dp = R.p - L.p, drho = R.u[0] - L.u[0];
    const T dVn = vnR - vnL;
    const T hic2 = T(0.5) * frcp<T>(c2);
    const T rc = rho_ravg * c * dVn;
    const T co0 = eig[0] * (dp - rc) * hic2;
    const T co1 = eig[1] * (drho - T(2) * dp * hic2);
    const T co2 = eig[1] * rho_ravg;
    const T co3 = eig[2] * (dp + rc) * hic2;
    // tangential velocity jump: the normal component cancels exactly
    T dvt_dot = T(0);
    T A[D + 2];
    A[0] = co0 + co1 + co3;
    for (int k = 0; k < D; ++k) {
        const T dvt = (k == K) ? T(0) : (R.vel[k] - L.vel[k]);
        dvt_dot += v_ravg[k] * dvt;
        const T nk = (k == K) ? sgn : T(0);
        A[1 + k] = co0 * (v_ravg[k] - c * nk) + co1 * v_ravg[k] + co2 * dvt + co3 * (v_ravg[k] + c * nk);
    }
    A[D + 1] = co0 * (h_ravg - c * vn) + co1 * vel2 * T(0.5) + co2 * dvt_dot + co3 * (h_ravg + c * vn);
    for (int s = 0; s < D + 2; ++s) out[s] = T(-0.5) * A[s];
}

// Convective flux of a node (with its momentum) along e_K or (CV) contracted with nv.
template <int D, int K, bool CV>
__device__ __forceinline__ void convective_flux64(const NodeC<double, D> &q, const double *nv, double *f)
{
    double m;
    if constexpr (CV) {
        m = q.u[1] * nv[0];
        for (int k = 1; k < D; ++k) m += q.u[1 + k] * nv[k];
    } else {
        m = q.u[1 + K];
    }
    f[0] = m;
    for (int k = 0; k < D; ++k) {
        f[1 + k] = m * q.vel[k];
        if constexpr (CV) f[1 + k] += q.p * nv[k];
        else if (k == K) f[1 + k] += q.p;
    }
    f[D + 1] = m * q.h;
}

// Roe-Pike dissipation with Harten's entropy fix in double, -1/2 of it added to out: along the unit
// normal n (CV) or sgn e_K.  co0 + co3 and (co3 - co0) c are formed once and shared by every state.
template <int D, int K, bool CV>
__device__ __forceinline__ void roe64(const NodeC<double, D> &L, const NodeC<double, D> &R, double sgn,
                                      const double *n, double vnL, double vnR, const FastConst<double> &fc,
                                      double *out)
{
    const double isum = frcp<double>(L.sr + R.sr);
    const double wL = L.sr * isum, wR = R.sr * isum, rho = L.sr * R.sr;
    double v[D], v2 = 0.0, vn = 0.0;
    for (int k = 0; k < D; ++k) {
        const double a = wL * L.vel[k], b = wR * R.vel[k];
        v[k] = a + b;
    }
    v2 = v[0] * v[0];
    for (int k = 1; k < D; ++k) v2 += v[k] * v[k];
    if constexpr (CV) {
        vn = v[0] * n[0];
        for (int k = 1; k < D; ++k) vn += v[k] * n[k];
    } else {
        vn = v[K] * sgn;
    }
    const double ha = wL * L.h, hb = wR * R.h;
    const double h = ha + hb;
    const double c2 = fc.gamm1 * (h - 0.5 * v2);
    double c, ic;
    Fast<double>::sqrt_rsqrt(c2, &c, &ic);
    double hic2 = 0.5 * (ic * ic);
    if (__builtin_expect(!(c2 > 0.0), 0)) {
        c = 1e10;
        hic2 = 0.5 * frcp<double>(c2);
    }
    double eig[3] = {fab<double>(vn - c), fab<double>(vn), fab<double>(vn + c)};
    const double eL[3] = {fab<double>(vnL - L.c), fab<double>(vnL), fab<double>(vnL + L.c)};
    const double eR[3] = {fab<double>(vnR - R.c), fab<double>(vnR), fab<double>(vnR + R.c)};
    for (int e = 0; e < 3; ++e) {
        const double eps = fmx<double>(fab<double>(eig[e] - eL[e]), fab<double>(eR[e] - eig[e]));
        if (eig[e] < eps) eig[e] = 0.5 * (eig[e] * eig[e] * frcp<double>(eps) + eps);
    }
    const double dp = R.p - L.p, drho = R.u[0] - L.u[0], dVn = vnR - vnL;
    const double rc = rho * c * dVn;
    const double e0 = eig[0] * hic2, e2 = eig[2] * hic2;
    const double co0 = e0 * (dp - rc), co3 = e2 * (dp + rc);
    const double s = co0 + co3, dc = (co3 - co0) * c;
    const double co1 = eig[1] * (drho - 2.0 * dp * hic2), co2 = eig[1] * rho;
    const double A0 = s + co1;
    out[0] -= 0.5 * A0;
    double vt = 0.0;
    for (int k = 0; k < D; ++k) {
        double dvt = R.vel[k] - L.vel[k], Ak;
        if constexpr (CV) {
            dvt -= dVn * n[k];
            Ak = A0 * v[k] + co2 * dvt;
            Ak += dc * n[k];
        } else {
            // the normal component of the tangential jump cancels exactly
            Ak = A0 * v[k];
            if (k == K) Ak += dc * sgn;
            else Ak += co2 * dvt;
        }
        if (CV || k != K) vt += v[k] * dvt;
        out[1 + k] -= 0.5 * Ak;
    }
    double AE = s * h + dc * vn;
    AE += co1 * 0.5 * v2;
    AE += co2 * vt;
    out[D + 1] -= 0.5 * AE;
}

// Numerical flux in double along the unit normal n (CV) or sgn e_K, outward of side L; exchanging
// the sides and turning the normal around gives the exact negative.  GEN: the two-point flux is
// Kennedy-Gruber or Ismail-Roe, else Chandrashekar or Ranocha; `first` orders the sides for the
// former, which are not written that way.  Lax-Friedrichs dissipation reads the energies u[D + 1] as
// well (rebuilt from H they would leave a jump of their rounding times the sound speed).  mom(left, k): a
// side's momentum, asked for only where a flux needs it (the central flux, Lax-Friedrichs dissipation).
template <int D, int K, bool CV, bool GEN, typename Mom>
__device__ __forceinline__ void num_flux64(const NodeC<double, D> &L, const NodeC<double, D> &R, double sgn,
                                           const double *n, bool first, const FastConst<double> &fc,
                                           const PhysConst &pc, const Mom &mom, double *out)
{
    const int cf = fc.conv_flux;
    double vnL, vnR;
    if constexpr (CV) {
        vnL = L.vel[0] * n[0];
        vnR = R.vel[0] * n[0];
        for (int k = 1; k < D; ++k) {
            vnL += L.vel[k] * n[k];
            vnR += R.vel[k] * n[k];
        }
    } else {
        vnL = L.vel[K] * sgn;
        vnR = R.vel[K] * sgn;
    }
    if (cf >= 3) {
        if constexpr (!GEN) {
            ec_flux64<D, K, CV>(L, R, n, fc, out);
        } else {
            // ordered by value: a branch would run both orders in a wave that holds both
            NodeC<double, D> a, b;
            a.u[0] = first ? L.u[0] : R.u[0];
            b.u[0] = first ? R.u[0] : L.u[0];
            for (int k = 0; k < D; ++k) {
                a.vel[k] = first ? L.vel[k] : R.vel[k];
                b.vel[k] = first ? R.vel[k] : L.vel[k];
            }
            a.p = first ? L.p : R.p;
            b.p = first ? R.p : L.p;
            a.u[D + 1] = first ? L.u[D + 1] : R.u[D + 1];
            b.u[D + 1] = first ? R.u[D + 1] : L.u[D + 1];
            other_flux64<D, K, CV>(a, b, n, pc, out);
        }
        if constexpr (!CV)
            for (int s = 0; s < D + 2; ++s) out[s] *= sgn;
    } else {
        double mL, mR;
        if constexpr (CV) {
            mL = mom(true, 0) * n[0];
            mR = mom(false, 0) * n[0];
            for (int k = 1; k < D; ++k) {
                mL += mom(true, k) * n[k];
                mR += mom(false, k) * n[k];
            }
        } else {
            mL = mom(true, K) * sgn;
            mR = mom(false, K) * sgn;
        }
        const double ps = 0.5 * (L.p + R.p);
        out[0] = 0.5 * (mL + mR);
        for (int k = 0; k < D; ++k) {
            const double a = mL * L.vel[k], b = mR * R.vel[k];
            out[1 + k] = 0.5 * (a + b);
            if constexpr (CV) out[1 + k] += ps * n[k];
            else if (k == K) out[1 + k] += ps * sgn;
        }
        const double a = mL * L.h, b = mR * R.h;
        out[D + 1] = 0.5 * (a + b);
    }
    if (cf == 0 || cf == 4) {
        const double hl = 0.5 * fmx<double>(fab<double>(vnL) + L.c, fab<double>(vnR) + R.c);
        out[0] -= hl * (R.u[0] - L.u[0]);
        for (int k = 0; k < D; ++k) {
            const double a = mom(true, k), b = mom(false, k);
            out[1 + k] -= hl * (b - a);
        }
        out[D + 1] -= hl * (R.u[D + 1] - L.u[D + 1]);
    }
    if (cf == 1 || cf == 5) roe64<D, K, CV>(L, R, sgn, n, vnL, vnR, fc, out);
}

// The same with the momentum rho v.
template <int D, int K, bool CV, bool GEN>
__device__ __forceinline__ void num_flux64(const NodeC<double, D> &L, const NodeC<double, D> &R, double sgn,
                                           const double *n, bool first, const FastConst<double> &fc,
                                           const PhysConst &pc, double *out)
{
    const auto mom = [&](bool left, int k) { return left ? L.u[0] * L.vel[k] : R.u[0] * R.vel[k]; };
    num_flux64<D, K, CV, GEN>(L, R, sgn, n, first, fc, pc, mom, out);
}

// Numerical flux of a face node along the normal sgn * e_K, L the interior
// (owner) side.
template <typename T, int D, int K>
__device__ __forceinline__ void num_flux_fast(const NodeC<T, D> &L, const NodeC<T, D> &R, T sgn,
                                              const FastConst<T> &fc, const PhysConst &pc, T *out)
{
    if constexpr (std::is_same<T, double>::value) {
        if (fc.two_point >= 2) num_flux64<D, K, false, false>(L, R, sgn, nullptr, true, fc, pc, out);
        else num_flux64<D, K, false, true>(L, R, sgn, nullptr, true, fc, pc, out);
        return;
    }
    const int cf = fc.conv_flux;
    T base[D + 2];
    if (cf >= 3) {
        pair_flux_fast<T, D, K>(L, R, fc, pc, base);
        for (int s = 0; s < D + 2; ++s) base[s] *= sgn;
    } else {
        T f1[D + 2], f2[D + 2];
        convective_flux_dir<T, D>(L.u, K, fc.gamm1, f1);
        convective_flux_dir<T, D>(R.u, K, fc.gamm1, f2);
        for (int s = 0; s < D + 2; ++s) base[s] = (T(0.5) * (f1[s] + f2[s])) * sgn;
    }
    T diss[D + 2];
    for (int s = 0; s < D + 2; ++s) diss[s] = T(0);
    if (cf == 0 || cf == 4) {
        const T lam = fmx<T>(fab<T>(L.vel[K]) + L.c, fab<T>(R.vel[K]) + R.c);
        for (int s = 0; s < D + 2; ++s) diss[s] = T(-0.5) * lam * (R.u[s] - L.u[s]);
    }
    if (cf == 1 || cf == 5) roe_fast<T, D, K>(L, R, sgn, fc, diss);
    for (int s = 0; s < D + 2; ++s) out[s] = base[s] + diss[s];
}

// ---- Navier-Stokes in double ------------------------------------------------------------------
// Viscous fluxes of one node in every direction, momentum and energy components only (the density
// component is zero): f[k][a] = F_v(u, grad u) . e_k, a = 0..D-1 momentum, D energy, the formulas of
// viscous_flux_all with one reciprocal, 1/rho.
__device__ __forceinline__ double visc_mu64(const PhysConst &pc, double T_)
{
    if (pc.use_constant_viscosity) return pc.mu_const / pc.reynolds;
    const double tr = pc.temperature_ratio;
    return (1.0 + tr) * frcp<double>(T_ + tr) * (T_ * fsqrt<double>(T_)) / pc.reynolds;
}

template <int D>
__device__ __forceinline__ void viscous_flux64(const double *u, const double *g, const PhysConst &pc,
                                               double (&f)[D][D + 1])
{
    const double gm2 = pc.gam * pc.mach2;
    const double ir = frcp<double>(u[0]);
    double vel[D], v2 = 0.0;
    for (int k = 0; k < D; ++k) {
        vel[k] = u[1 + k] * ir;
        v2 += vel[k] * vel[k];
    }
    const double T_ = gm2 * pc.gamm1 * (u[D + 1] * ir - 0.5 * v2);
    const double mu = visc_mu64(pc, T_);
    const double kappa = mu / (pc.gamm1 * pc.mach2 * pc.prandtl);
    double vg[D][D], div = 0.0;
    for (int a = 0; a < D; ++a)
        for (int b = 0; b < D; ++b) vg[a][b] = (g[(1 + a) * D + b] - vel[a] * g[b]) * ir;
    for (int a = 0; a < D; ++a) div += vg[a][a];
    div *= (2.0 / 3.0) * mu;
    for (int k = 0; k < D; ++k) {
        // grad p = (gamma - 1) (grad E - v . grad m + |v|^2/2 grad rho)
        double pg = g[(D + 1) * D + k] + 0.5 * v2 * g[k];
        for (int a = 0; a < D; ++a) pg -= vel[a] * g[(1 + a) * D + k];
        const double dT = (gm2 * pc.gamm1 * pg - T_ * g[k]) * ir;
        double fe = -kappa * dT;
        for (int a = 0; a < D; ++a) {
            double tau = mu * (vg[a][k] + vg[k][a]);
            if (a == k) tau -= div;
            f[k][a] = -tau;
            fe -= vel[a] * tau;
        }
        f[k][D] = fe;
    }
}

// F_v(u, du n) . n for a unit normal n and a state jump du (the SIPG penalty flux): with the
// gradient du n the velocity gradient is w n, w = (dm - v drho)/rho.
template <int D>
__device__ __forceinline__ void viscous_jump64(const NodeC<double, D> &q, const double *du, const double *n,
                                               const PhysConst &pc, double *f)
{
    const double gm2 = pc.gam * pc.mach2;
    const double ir = frcp<double>(q.u[0]);
    const double T_ = gm2 * q.p * ir;
    const double mu = visc_mu64(pc, T_);
    const double kappa = mu / (pc.gamm1 * pc.mach2 * pc.prandtl);
    double w[D], wn = 0.0, v2 = 0.0, pg = du[D + 1];
    for (int k = 0; k < D; ++k) {
        w[k] = (du[1 + k] - q.vel[k] * du[0]) * ir;
        wn += w[k] * n[k];
        v2 += q.vel[k] * q.vel[k];
        pg -= q.vel[k] * du[1 + k];
    }
    pg += 0.5 * v2 * du[0];
    double fe = -kappa * ((gm2 * pc.gamm1 * pg - T_ * du[0]) * ir);
    for (int k = 0; k < D; ++k) {
        const double tau = mu * (w[k] + (1.0 / 3.0) * wn * n[k]);
        f[k] = -tau;
        fe -= q.vel[k] * tau;
    }
    f[D] = fe;
}

} // namespace dgx
