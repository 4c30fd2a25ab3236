// Device arithmetic policies, limiters and fluxes of the four dimensionally
// split schemes.
//
// Every function is written in "sweep order": state index 0 is the density
// (h or rho), 1 the momentum normal to the sweep, 2 the tangential momentum,
// 3 the energy (Euler).  A y sweep passes (h, hv, hu[, E]) and maps the result
// back, as computeFluxG does in GPUSimulators/cuda/SWE2D_KP07_dimsplit.cu:71-110.
//
// Two arithmetic policies share the code:
//   MathExact  IEEE division and square root, and (by the translation unit's
//              -ffp-contract=off) no fused multiply-add.  Each expression is
//              evaluated in the operand order of the CUDA source, so results
//              are bitwise equal to an IEEE float32 evaluation of the
//              reference arithmetic.
//   MathFast   hardware reciprocal / square root (v_rcp_f32, v_sqrt_f32, about
//              1 ulp) with shared reciprocals and contraction allowed.  Held
//              against the float32 oracle at relative L1 <= 1e-5.
#pragma once

#include <hip/hip_runtime.h>

namespace fvmi {

// One transcendental of several values, issued as one run: a lone one among
// other VALU instructions costs two to three times its place in a run (the two
// waves that a SIMD issues from in turn fall out of step at each change).
// s_nop: a transcendental's result may not be read by the next instruction,
// which the compiler does not see inside the block.
#define FVMI_TRANS_RUN(name, one, op)                                                                                    \
    template <int N>                                                                                                \
    __device__ __forceinline__ void name(const float (&x)[N], float (&r)[N]) {                                      \
        static_assert((N >= 1 && N <= 4) || N == 8, "runs of 1 to 4, or two of 4");                                 \
        if constexpr (N == 8) {                                                                                     \
            const float xa[4] = {x[0], x[1], x[2], x[3]}, xb[4] = {x[4], x[5], x[6], x[7]};                         \
            float ra[4], rb[4];                                                                                     \
            name<4>(xa, ra);                                                                                        \
            name<4>(xb, rb);                                                                                        \
            r[0] = ra[0], r[1] = ra[1], r[2] = ra[2], r[3] = ra[3];                                                 \
            r[4] = rb[0], r[5] = rb[1], r[6] = rb[2], r[7] = rb[3];                                                 \
        } else if constexpr (N == 1)                                                                                \
            r[0] = one(x[0]);                                                                                       \
        else if constexpr (N == 2)                                                                                  \
            asm(op " %0, %2\n\t" op " %1, %3\n\ts_nop 0" : "=&v"(r[0]), "=v"(r[1]) : "v"(x[0]), "v"(x[1]));       \
        else if constexpr (N == 3)                                                                                  \
            asm(op " %0, %3\n\t" op " %1, %4\n\t" op " %2, %5\n\ts_nop 0"                                        \
                : "=&v"(r[0]), "=&v"(r[1]), "=v"(r[2])                                                              \
                : "v"(x[0]), "v"(x[1]), "v"(x[2]));                                                                 \
        else                                                                                                        \
            asm(op " %0, %4\n\t" op " %1, %5\n\t" op " %2, %6\n\t" op " %3, %7\n\ts_nop 0"                       \
                : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=v"(r[3])                                                 \
                : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));                                                      \
    }
FVMI_TRANS_RUN(rcp_all, __builtin_amdgcn_rcpf, "v_rcp_f32")
FVMI_TRANS_RUN(rsq_all, __builtin_amdgcn_rsqf, "v_rsq_f32")
FVMI_TRANS_RUN(sqrt_all, __builtin_amdgcn_sqrtf, "v_sqrt_f32")
#undef FVMI_TRANS_RUN

// Correctly rounded float32 division and square root in fewer instructions
// than the compiler's general IEEE sequences, for operands in the normal range
// (no scaling for denormal or overflowing intermediates, no special-case
// fix-up: a zero or infinite divisor gives NaN).
//  * reciprocal: v_rcp_f32 (1 ulp) refined by one Newton step with FMA,
//    y = y0 + y0 (1 - b y0), which rounds to the correctly rounded 1/b;
//  * quotient: q0 = a y, the exact remainder r = a - b q0 by FMA, and
//    q = q0 + r y: correctly rounded when y is (Markstein's theorem).  A zero
//    quotient needs care only for its sign, which q0 has and q0 + r y may turn
//    from -0 into +0: div_rn puts it back with one v_bfi (the sign of a zero
//    reaches copysign in the WAF limiter), quot_rn leaves it (no other scheme
//    reads a zero's sign, and its values are equal either way; exact runs from
//    momenta of +0 and -0 keep the oracle's signs too);
//  * square root: v_sqrt_f32 (1 ulp) and its two neighbours, the one whose
//    residual x - s s' changes sign chosen by two FMAs (exact from x = 2^-101 on,
//    within 2 ulp below; 0 and infinity give themselves).  Newton's correction
//    s + (x - s^2) y/2 from y = v_rsq_f32(x) takes 6 instructions for 9 and equals
//    it from 2^-101 up to the largest finite number only: y is infinite at 0, the
//    residual underflows below, and infinity gives NaN.  A branch to the
//    compiler's sequence for those cost small grids more than the neighbours do
//    (a step of one simulator: WAF 1023x777 48.1 us without it, 50.3 with the
//    neighbours, 52.6 with the branch, KP07 2048x1500 68.6, 72.3 and 77.8; three
//    simulators in turn, WAF 4096^2 476, 486 and 472, Euler 8192^2 1800, 1824 and
//    1824).
// Checked against the IEEE sequences on every mantissa of [1, 2) (reciprocal)
// and [1, 4) (square root) and on random quotients, and in every exact-
// arithmetic test, which compare the fields with the float32 oracle for
// equality.  The exact kernels are bound by VALU issue, so their time follows
// the instruction count: with the quotient at 6 instructions (8 before, its sign
// chosen by a compare) and the limiter of minmod_slope, KP07_dimsplit has 358
// instructions a row (480 before).
__device__ __forceinline__ float rcp_rn(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}
// a / b with y = rcp_rn(b) known
__device__ __forceinline__ float quot_rn(float a, float b, float y) {
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float div_rn(float a, float b, float y) {
    const float q = a * y;
    return __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-b, q, a), y, q), q);
}
__device__ __forceinline__ float quot_rn(float a, float b) { return quot_rn(a, b, rcp_rn(b)); }
__device__ __forceinline__ float div_rn(float a, float b) { return div_rn(a, b, rcp_rn(b)); }
// the square root of x from s = v_sqrt_f32(x)
__device__ __forceinline__ float sqrt_rn(float x, float s) {
    const float dn = __uint_as_float(__float_as_uint(s) - 1u);
    const float up = __uint_as_float(__float_as_uint(s) + 1u);
    const float r = (__builtin_fmaf(-dn, s, x) <= 0.0f) ? dn : s;
    return (__builtin_fmaf(-up, s, x) > 0.0f) ? up : r;
}
__device__ __forceinline__ float sqrt_rn(float x) { return sqrt_rn(x, __builtin_amdgcn_sqrtf(x)); }
// the same of N values, their v_rcp / v_sqrt in one run
template <int N>
__device__ __forceinline__ void rcp_rn_all(const float (&b)[N], float (&r)[N]) {
    float y[N];
    rcp_all<N>(b, y);
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = __builtin_fmaf(__builtin_fmaf(-b[i], y[i], 1.0f), y[i], y[i]);
}
template <int N>
__device__ __forceinline__ void sqrt_rn_all(const float (&x)[N], float (&r)[N]) {
    float s[N];
    sqrt_all<N>(x, s);
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = sqrt_rn(x[i], s[i]);
}

struct MathExact {
    static constexpr bool exact = true;
    __device__ static __forceinline__ float div(float a, float b) { return div_rn(a, b); }
    __device__ static __forceinline__ float quot(float a, float b) { return quot_rn(a, b); }
    __device__ static __forceinline__ float sqrt(float x) { return sqrt_rn(x); }
    __device__ static __forceinline__ float rcp(float x) { return rcp_rn(x); }
};

struct MathFast {
    static constexpr bool exact = false;
    __device__ static __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    __device__ static __forceinline__ float div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
    __device__ static __forceinline__ float quot(float a, float b) { return div(a, b); }
    __device__ static __forceinline__ float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
};

// ---------------------------------------------------------------------------
// Limiters: GPUSimulators/cuda/limiters.h, common.h
// ---------------------------------------------------------------------------

// minmodSlope (limiters.h:31-41) in exact arithmetic, from the reference's
// backward, central and forward differences.  Its sign products 0.25 sb
// (sb + sc) (sc + sf) are the common sign or zero, so its value is the median
// form: the inner median is zero unless b and f share a sign, and then c shares
// it (the float differences keep the order of the operands).  2 instructions
// where the sign products take 10.  No factor of two is moved between the
// differences and the slope: that would round differently where they are
// denormal, as at the foot of a wave that decays into still water.
// The fast policy evaluates the same minmod in a scaled form (reconstruct_fast
// in fv_substep.h, half_slope in fv_unsplit.h).
__device__ __forceinline__ float minmod_slope(float b, float c, float f) {
    return __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(b, f, 0.0f), c, 0.0f);
}

// generalized_minmod, limiters.h:100-102
__device__ __forceinline__ float generalized_minmod(float r, float theta) {
    return fmaxf(0.0f, fminf(theta * r, fminf((1.0f + r) / 2.0f, theta)));
}

// desingularize, common.h:81-83
template <class M>
__device__ __forceinline__ float desingularize(float x, float eps) {
    return __builtin_copysignf(fmaxf(fabsf(x), fminf(M::quot(x * x, 2.0f * eps) + 0.5f * eps, eps)), x);
}

// limiterToWAFLimiter, SWECommon.h:109-111
__device__ __forceinline__ float limiter_to_waf(float r, float c) {
    return 1.0f - (1.0f - fabsf(c)) * r;
}

// ---------------------------------------------------------------------------
// Shallow water: GPUSimulators/cuda/SWECommon.h
// ---------------------------------------------------------------------------

// F_func, SWECommon.h:29-37
template <class M>
__device__ __forceinline__ void swe_F(const float q[3], float g, float F[3]) {
    if constexpr (M::exact) {
        F[0] = q[1];
        F[1] = M::quot(q[1] * q[1], q[0]) + 0.5f * g * q[0] * q[0];
        F[2] = M::quot(q[1] * q[2], q[0]);
    } else {
        const float u = q[1] * M::rcp(q[0]);
        F[0] = q[1];
        F[1] = q[1] * u + 0.5f * g * q[0] * q[0];
        F[2] = q[2] * u;
    }
}

// The fluxes below are the exact policy's (the fast one's are in fv_fast.h).

// CentralUpwindFlux, SWECommon.h:228-241.  qm = left state, qp = right state.
__device__ __forceinline__ void swe_cu_flux(const float qm[3], const float qp[3], float g, float out[3]) {
    const float h[2] = {qm[0], qp[0]}, gh[2] = {g * qm[0], g * qp[0]};
    float y[2], c[2];
    rcp_rn_all<2>(h, y);
    sqrt_rn_all<2>(gh, c);
    const float um = quot_rn(qm[1], qm[0], y[0]), up = quot_rn(qp[1], qp[0], y[1]);
    const float Fm[3] = {qm[1], quot_rn(qm[1] * qm[1], qm[0], y[0]) + 0.5f * g * qm[0] * qm[0],
                         quot_rn(qm[1] * qm[2], qm[0], y[0])};
    const float Fp[3] = {qp[1], quot_rn(qp[1] * qp[1], qp[0], y[1]) + 0.5f * g * qp[0] * qp[0],
                         quot_rn(qp[1] * qp[2], qp[0], y[1])};
    const float am = fminf(fminf(um - c[0], up - c[1]), 0.0f);
    const float ap = fmaxf(fmaxf(um + c[0], up + c[1]), 0.0f);
    const float apam = ap * am;
    const float den = ap - am, iden = rcp_rn(den);
#pragma unroll
    for (int k = 0; k < 3; ++k) out[k] = quot_rn((ap * Fm[k] - am * Fp[k]) + apam * (qp[k] - qm[k]), den, iden);
}

// HLL_flux (SWE), SWECommon.h:274-313
__device__ __forceinline__ void swe_hll_flux(const float ql[3], const float qr[3], float g, float out[3]) {
    const float h_l = ql[0], h_r = qr[0];
    const float h[2] = {h_l, h_r}, gh[2] = {g * h_l, g * h_r};
    float y[2], c[2];
    rcp_rn_all<2>(h, y);
    sqrt_rn_all<2>(gh, c);
    const float u_l = quot_rn(ql[1], h_l, y[0]), u_r = quot_rn(qr[1], h_r, y[1]);
    const float c_l = c[0], c_r = c[1];
    const float h_dag = 0.5f * (h_l + h_r) - quot_rn(0.25f * (u_r - u_l) * (h_l + h_r), c_l + c_r);
    const float q_l_tmp = sqrt_rn(0.5f * quot_rn((h_dag + h_l) * h_dag, h_l * h_l));
    const float q_r_tmp = sqrt_rn(0.5f * quot_rn((h_dag + h_r) * h_dag, h_r * h_r));
    const float q_l = (h_dag > h_l) ? q_l_tmp : 1.0f;
    const float q_r = (h_dag > h_r) ? q_r_tmp : 1.0f;
    const float S_l = u_l - c_l * q_l;
    const float S_r = u_r + c_r * q_r;
    const float F_l[3] = {ql[1], quot_rn(ql[1] * ql[1], h_l, y[0]) + 0.5f * g * h_l * h_l,
                          quot_rn(ql[1] * ql[2], h_l, y[0])};
    const float F_r[3] = {qr[1], quot_rn(qr[1] * qr[1], h_r, y[1]) + 0.5f * g * h_r * h_r,
                          quot_rn(qr[1] * qr[2], h_r, y[1])};
    const float srsl = S_r * S_l;
    const float den = S_r - S_l, iden = rcp_rn(den);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float star = quot_rn(S_r * F_l[k] - S_l * F_r[k] + srsl * (qr[k] - ql[k]), den, iden);
        out[k] = (S_l >= 0.0f) ? F_l[k] : ((S_r <= 0.0f) ? F_r[k] : star);
    }
}

// computeHStar, SWECommon.h:114-121
template <class M>
__device__ __forceinline__ float compute_h_star(float h_l, float h_r, float u_l, float u_r, float c_l, float c_r,
                                                float g) {
    (void)h_l;
    (void)h_r;
    const float h_tmp = 0.5f * (c_l + c_r) + 0.25f * (u_l - u_r);
    return M::quot(h_tmp * h_tmp, g);
}

// ---------------------------------------------------------------------------
// WAF in pieces: per-cell quantities, h* per interface, and the flux from the
// two cells at the interface plus what it needs of the outer two.  A march
// computes each cell's quantities and each interface's h* once and shares
// them between the (up to four) fluxes that use them; the values are those
// swe_waf_flux computes for itself, so the exact policy stays bitwise equal.
// ---------------------------------------------------------------------------

struct WafCell {
    float h, hu, hv;  // state in sweep order (depth, normal, tangential momentum)
    float u, v, c;    // normal and tangential velocity, sqrt(g h)
    float ih;         // 1/h
    float f1, f2;     // fluxes of the normal and tangential momentum (that of h is hu)
};

// hg = g/2
template <class M>
__device__ __forceinline__ WafCell waf_cell(const float q[3], float g, float hg, float sqrt_g) {
    WafCell p;
    p.h = q[0];
    p.hu = q[1];
    p.hv = q[2];
    if constexpr (M::exact) {
        p.ih = rcp_rn(p.h);
        p.u = div_rn(p.hu, p.h, p.ih);
        p.v = div_rn(p.hv, p.h, p.ih);
        p.c = M::sqrt(g * p.h);
        p.f1 = quot_rn(p.hu * p.hu, p.h, p.ih) + hg * p.h * p.h;
        p.f2 = div_rn(p.hu * p.hv, p.h, p.ih);
    } else {
        const float s = __builtin_amdgcn_rsqf(p.h);
        p.ih = s * s;
        p.u = p.hu * p.ih;
        p.v = p.hv * p.ih;
        p.c = sqrt_g * p.h * s;
        p.f1 = p.hu * p.u + hg * p.h * p.h;
        p.f2 = p.hv * p.u;
    }
    return p;
}

// computeHStar (SWECommon.h:114-121) of the interface between l and r
template <class M>
__device__ __forceinline__ float waf_hstar(const WafCell& l, const WafCell& r, float g, float inv_g) {
    if constexpr (M::exact) {
        return compute_h_star<M>(l.h, r.h, l.u, r.u, l.c, r.c, g);
    } else {
        const float t = 0.5f * (l.c + r.c) + 0.25f * (l.u - r.u);
        return t * t * inv_g;
    }
}

// desingularize(x, 1e-6) of the WAF limiter ratios (SWECommon.h:170-176); fast
// form: the sign of x on the magnitude max(|x|, min(x^2/(2 eps) + eps/2, eps))
template <class M>
__device__ __forceinline__ float waf_desing(float x) {
    if constexpr (M::exact) {
        return desingularize<M>(x, 1.0e-6f);
    } else {
        const float eps = 1.0e-6f, inv_2eps = 0.5e6f;
        return __builtin_copysignf(
            __builtin_fmaxf(__builtin_fabsf(x), __builtin_fminf(x * x * inv_2eps + 0.5f * eps, eps)), x);
    }
}

// The limiter denominators of the interface between cells l and r with h* hd:
// desingularize(h* - h_l), desingularize(v_r - v_l), desingularize(h_r - h*)
// (SWECommon.h:170-176).  The upwind numerators of an interface's three
// ratios are the same quantities of the interface to its left (positive
// Courant number) or to its right, with the same operands in the same order,
// so each interface computes its own once and its neighbours take them.
struct WafDen {
    float d1, d2, d3;
};

template <class M>
__device__ __forceinline__ WafDen waf_den(const WafCell& l, const WafCell& r, float hd) {
    WafDen D;
    D.d1 = waf_desing<M>(hd - l.h);
    D.d2 = waf_desing<M>(r.v - l.v);
    D.d3 = waf_desing<M>(r.h - hd);
    return D;
}

// WAF_1D_flux (SWECommon.h:131-210) between cells l (= Q_l1) and r (= Q_r1)
// with h* h_dag, given the limiter denominators of this interface (D) and of
// the interfaces to its left (Dl) and right (Dr).  dtd = dt / d (fast policy).
template <class M>
__device__ __forceinline__ void waf_flux_core(const WafCell& L, const WafCell& R, const WafDen& Dl, const WafDen& D,
                                              const WafDen& Dr, float h_dag, float d, float dt, float dtd,
                                              float out[3]) {
    const float h_l = L.h, h_r = R.h, u_l = L.u, u_r = R.u, v_l = L.v, v_r = R.v, c_l = L.c, c_r = R.c;
    const float q_l1[3] = {L.h, L.hu, L.hv};
    const float q_r1[3] = {R.h, R.hu, R.hv};
    const float F_1[3] = {L.hu, L.f1, L.f2};
    const float F_4[3] = {R.hu, R.f1, R.f2};
    if constexpr (M::exact) {
        const float q_arg[2] = {0.5f * ((h_dag + h_l) * h_dag), 0.5f * ((h_dag + h_r) * h_dag)};
        float q_tmp[2];
        sqrt_rn_all<2>(q_arg, q_tmp);
        const float q_l = (h_dag > h_l) ? quot_rn(q_tmp[0], h_l, L.ih) : 1.0f;
        const float q_r = (h_dag > h_r) ? quot_rn(q_tmp[1], h_r, R.ih) : 1.0f;
        const float S_l = u_l - c_l * q_l;
        const float S_r = u_r + c_r * q_r;
        const float dl = h_l * (u_l - S_l), dr = h_r * (u_r - S_r);
        const float S_star = M::div(S_l * h_r * (u_r - S_r) - S_r * h_l * (u_l - S_l), dr - dl);
        const float e[2] = {S_l - S_star, S_r - S_star};
        float ie[2];
        rcp_rn_all<2>(e, ie);
        const float s_l = div_rn(-dl, e[0], ie[0]);  // h_l (S_l - u_l) / (S_l - S_star)
        const float s_r = div_rn(-dr, e[1], ie[1]);
        const float Q_star_l[3] = {s_l * 1.0f, s_l * S_star, s_l * v_l};
        const float Q_star_r[3] = {s_r * 1.0f, s_r * S_star, s_r * v_r};
        float F_2[3], F_3[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            F_2[k] = F_1[k] + S_l * (Q_star_l[k] - q_l1[k]);
            F_3[k] = F_4[k] + S_r * (Q_star_r[k] - q_r1[k]);
        }
        // Courant numbers; a zero one has the sign of its numerator
        const float p_1 = S_l * dt, p_2 = S_star * dt, p_3 = S_r * dt;
        const float c_1 = M::quot(p_1, d), c_2 = M::quot(p_2, d), c_3 = M::quot(p_3, d);
        // desingularize((c_1 > 0) ? h_dag_l - h_l2 : h_dag_r - h_r) / desingularize(h_dag - h_l), ...
        const float den[3] = {D.d1, D.d2, D.d3};
        float iden[3];
        rcp_rn_all<3>(den, iden);
        const float r_1 = quot_rn((c_1 > 0.0f) ? Dl.d1 : Dr.d1, D.d1, iden[0]);
        const float r_2 = quot_rn((c_2 > 0.0f) ? Dl.d2 : Dr.d2, D.d2, iden[1]);
        const float r_3 = quot_rn((c_3 > 0.0f) ? Dl.d3 : Dr.d3, D.d3, iden[2]);
        const float A_1 = __builtin_copysignf(1.0f, p_1) * limiter_to_waf(generalized_minmod(r_1, 1.9f), c_1);
        const float A_2 = __builtin_copysignf(1.0f, p_2) * limiter_to_waf(generalized_minmod(r_2, 1.9f), c_2);
        const float A_3 = __builtin_copysignf(1.0f, p_3) * limiter_to_waf(generalized_minmod(r_3, 1.9f), c_3);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            out[k] = 0.5f * (F_1[k] + F_4[k]) -
                     0.5f * (A_1 * (F_2[k] - F_1[k]) + A_2 * (F_3[k] - F_2[k]) + A_3 * (F_4[k] - F_3[k]));
    } else {
        const float il = L.ih, ir = R.ih;
        const float q_l = (h_dag > h_l) ? M::sqrt(0.5f * ((h_dag + h_l) * h_dag)) * il : 1.0f;
        const float q_r = (h_dag > h_r) ? M::sqrt(0.5f * ((h_dag + h_r) * h_dag)) * ir : 1.0f;
        const float S_l = u_l - c_l * q_l;
        const float S_r = u_r + c_r * q_r;
        const float dl = h_l * (u_l - S_l), dr = h_r * (u_r - S_r);
        const float S_star = (S_l * dr - S_r * dl) * M::rcp(dr - dl);
        // shared reciprocal of (S_l - S_star)(S_r - S_star)
        const float el = S_l - S_star, er = S_r - S_star;
        const float ie = M::rcp(el * er);
        const float s_l = -dl * (er * ie);  // h_l (S_l - u_l) / (S_l - S_star)
        const float s_r = -dr * (el * ie);  // h_r (S_r - u_r) / (S_r - S_star)
        const float Qsl[3] = {s_l, s_l * S_star, s_l * v_l};
        const float Qsr[3] = {s_r, s_r * S_star, s_r * v_r};
        const float c_1 = S_l * dtd, c_2 = S_star * dtd, c_3 = S_r * dtd;
        auto gmm = [](float r) {
            return __builtin_fmaxf(0.0f, __builtin_fminf(1.9f * r, __builtin_fminf((1.0f + r) * 0.5f, 1.9f)));
        };
        const float r_1 = ((c_1 > 0.0f) ? Dl.d1 : Dr.d1) * M::rcp(D.d1);
        const float r_2 = ((c_2 > 0.0f) ? Dl.d2 : Dr.d2) * M::rcp(D.d2);
        const float r_3 = ((c_3 > 0.0f) ? Dl.d3 : Dr.d3) * M::rcp(D.d3);
        const float A_1 = __builtin_copysignf(1.0f, c_1) * (1.0f - (1.0f - __builtin_fabsf(c_1)) * gmm(r_1));
        const float A_2 = __builtin_copysignf(1.0f, c_2) * (1.0f - (1.0f - __builtin_fabsf(c_2)) * gmm(r_2));
        const float A_3 = __builtin_copysignf(1.0f, c_3) * (1.0f - (1.0f - __builtin_fabsf(c_3)) * gmm(r_3));
        // With a = F_2 - F_1 = S_l (Q*_l - Q_l1) and b = F_3 - F_4 = S_r (Q*_r - Q_r1),
        // A_1 (F_2 - F_1) + A_2 (F_3 - F_2) + A_3 (F_4 - F_3)
        //   = (A_1 - A_2) a + A_2 (F_4 - F_1) + (A_2 - A_3) b.
        const float w12 = 0.5f * (A_1 - A_2), w2 = 0.5f * A_2, w23 = 0.5f * (A_2 - A_3);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float a = S_l * (Qsl[k] - q_l1[k]);
            const float b = S_r * (Qsr[k] - q_r1[k]);
            out[k] = 0.5f * (F_1[k] + F_4[k]) - (w12 * a + w2 * (F_4[k] - F_1[k]) + w23 * b);
        }
    }
}

// writeCfl per-cell value, SWECommon.h:497-504
template <class M>
__device__ __forceinline__ float swe_cell_dt(const float q[3], float dx, float dy, float g) {
    if constexpr (M::exact) {
        const float h = q[0];
        const float u = M::quot(q[1], h);
        const float v = M::quot(q[2], h);
        const float max_u = M::quot(dx, fabsf(u) + M::sqrt(g * h));
        const float max_v = M::quot(dy, fabsf(v) + M::sqrt(g * h));
        return fminf(max_u, max_v);
    } else {
        const float ih = M::rcp(q[0]);
        const float c = M::sqrt(g * q[0]);
        return fminf(M::quot(dx, fabsf(q[1] * ih) + c), M::quot(dy, fabsf(q[2] * ih) + c));
    }
}

// ---------------------------------------------------------------------------
// Euler: GPUSimulators/cuda/EulerCommon.h
// ---------------------------------------------------------------------------

// F_func, EulerCommon.h:93-109.  P is a pressure.
template <class M>
__device__ __forceinline__ void euler_F(const float q[4], float P, float F[4]) {
    const float u = M::quot(q[1], q[0]);
    F[0] = q[1];
    F[1] = q[1] * u + P;
    F[2] = q[2] * u;
    F[3] = u * (q[3] + P);
}

// 1/rho, normal velocity, pressure, sound speed and flux of the two states of an
// interface (pressure EulerCommon.h:83-90, F_func :93-109)
__device__ __forceinline__ void euler_states(const float ql[4], const float qr[4], float gamma, float u[2], float c[2],
                                             float F_l[4], float F_r[4]) {
    const float rho[2] = {ql[0], qr[0]};
    float y[2], P[2], cc[2];
    rcp_rn_all<2>(rho, y);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float* q = i ? qr : ql;
        float* F = i ? F_r : F_l;
        u[i] = quot_rn(q[1], q[0], y[i]);
        P[i] = (gamma - 1.0f) * (q[3] - quot_rn(0.5f * (q[1] * q[1] + q[2] * q[2]), q[0], y[i]));
        cc[i] = quot_rn(gamma * P[i], q[0], y[i]);
        F[0] = q[1];
        F[1] = q[1] * u[i] + P[i];
        F[2] = q[2] * u[i];
        F[3] = u[i] * (q[3] + P[i]);
    }
    float s[2];
    sqrt_rn_all<2>(cc, s);
    c[0] = s[0];
    c[1] = s[1];
}

// HLL_flux (Euler), EulerCommon.h:117-160
__device__ __forceinline__ void euler_hll_flux(const float ql[4], const float qr[4], float gamma, float out[4]) {
    const float h_l = ql[0], h_r = qr[0];
    float u[2], c[2], F_l[4], F_r[4];
    euler_states(ql, qr, gamma, u, c, F_l, F_r);
    const float h_dag = 0.5f * (h_l + h_r) - quot_rn(0.25f * (u[1] - u[0]) * (h_l + h_r), c[0] + c[1]);
    const float q_l_tmp = sqrt_rn(0.5f * quot_rn((h_dag + h_l) * h_dag, h_l * h_l));
    const float q_r_tmp = sqrt_rn(0.5f * quot_rn((h_dag + h_r) * h_dag, h_r * h_r));
    const float q_l = (h_dag > h_l) ? q_l_tmp : 1.0f;
    const float q_r = (h_dag > h_r) ? q_r_tmp : 1.0f;
    const float S_l = u[0] - c[0] * q_l;
    const float S_r = u[1] + c[1] * q_r;
    const float srsl = S_r * S_l;
    const float den = S_r - S_l, iden = rcp_rn(den);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float star = quot_rn(S_r * F_l[k] - S_l * F_r[k] + srsl * (qr[k] - ql[k]), den, iden);
        out[k] = (S_l >= 0.0f) ? F_l[k] : ((S_r <= 0.0f) ? F_r[k] : star);
    }
}

// CentralUpwindFlux (Euler), EulerCommon.h:171-187
__device__ __forceinline__ void euler_cu_flux(const float qm[4], const float qp[4], float gamma, float out[4]) {
    float u[2], c[2], Fm[4], Fp[4];
    euler_states(qm, qp, gamma, u, c, Fm, Fp);
    const float am = fminf(fminf(u[0] - c[0], u[1] - c[1]), 0.0f);
    const float ap = fmaxf(fmaxf(u[0] + c[0], u[1] + c[1]), 0.0f);
    const float apam = ap * am;
    const float den = ap - am, iden = rcp_rn(den);
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = quot_rn((ap * Fm[k] - am * Fp[k]) + apam * (qp[k] - qm[k]), den, iden);
}

// writeCfl per-cell value (Euler), EulerCommon.h:41-49: sqrt(gamma*rho) as written
template <class M>
__device__ __forceinline__ float euler_cell_dt(const float q[4], float dx, float dy, float gamma) {
    const float rho = q[0];
    const float u = M::quot(q[1], rho);
    const float v = M::quot(q[2], rho);
    const float max_u = M::quot(dx, fabsf(u) + M::sqrt(gamma * rho));
    const float max_v = M::quot(dy, fabsf(v) + M::sqrt(gamma * rho));
    return fminf(max_u, max_v);
}

}  // namespace fvmi
