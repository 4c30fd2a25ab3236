// Fast-arithmetic forms of the scheme fluxes (MathFast policy).
//
// Same mathematics as fv_math.h (and the reference expressions it cites), with
// the divisions and square roots regrouped so that each state costs one
// transcendental instruction where the reference needs several:
//   * one v_rsq per state gives 1/h = s*s and sqrt(g*h) = sqrt(g)*h*s;
//   * reciprocals of a pair share one v_rcp of the product;
//   * quotients with a common denominator reuse one reciprocal.
// Rounding differs from the exact policy by a few ulp per operation; the
// results are held to relative L1 <= 1e-5 of the float32 oracle.
#pragma once

#include <hip/hip_runtime.h>

#include "fv_math.h"

namespace fvmi {
namespace fast {

__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// Predictor difference F(QL) - F(QR) of the SWE flux (SWECommon.h:29-37), one
// reciprocal r = 1/(QL0 QR0) for both faces.  The faces are h0 -/+ (theta/2) m0
// in depth, so the pressure term g/2 (QL0^2 - QR0^2) = -g theta m0 h0.
__device__ __forceinline__ void swe_pred_diff(const float QL[3], const float QR[3], float r, float h0, float m0,
                                              float g_theta, float D[3]) {
    const float uL = QL[1] * (QR[0] * r);
    const float uR = QR[1] * (QL[0] * r);
    D[0] = QL[1] - QR[1];
    D[1] = (QL[1] * uL - QR[1] * uR) - g_theta * (m0 * h0);
    D[2] = QL[2] * uL - QR[2] * uR;
}

// Weights of the HLL flux F = wl F_l - wr F_r + wq (q_r - q_l) with the
// reference's upwind selection (SWECommon.h:299-311, EulerCommon.h:146-159:
// F_l if S_l >= 0, else F_r if S_r <= 0, else the HLL average) folded into
// clamped speeds sl = min(S_l, 0) and sr = max(S_r, S_l, 1e-30):
//   wl = sr / (sr - sl), wr = sl / (sr - sl), wq = sr sl / (sr - sl).
// S_l >= 0 gives sl = 0 and sr > 0: F_l (also when S_r <= 0 <= S_l, where the
// reference tests S_l first).  S_l < 0 and S_r <= 0 give sr = 1e-30: F_r up to
// a relative 1e-30 / |S_l|.  Otherwise sl = S_l, sr = S_r: the HLL average.
__device__ __forceinline__ void hll_speeds(float S_l, float S_r, float& sl, float& sr) {
    sl = __builtin_fminf(S_l, 0.0f);
    sr = __builtin_fmaxf(__builtin_fmaxf(S_r, S_l), 1e-30f);
}

// The fluxes below take the C interfaces of a lane at once, their
// transcendentals in runs.

// Central-upwind flux (SWECommon.h:228-241),
//   (ap F(qm) - am F(qp) + ap am (qp - qm)) / (ap - am)
//     = wm (F(qm) - am qm) - wp (F(qp) - ap qp),  wm = ap/(ap-am), wp = am/(ap-am),
// where F(q) - a q = (q1 - a q0, q1 (u - a) + g/2 q0^2, q2 (u - a)).
template <int C>
__device__ __forceinline__ void swe_cu_flux(const float (&qm)[C][3], const float (&qp)[C][3], float hg, float sg,
                                            float (&out)[C][3]) {
    float h[2 * C], s[2 * C], um[C], up[C], am[C], ap[C], den[C], iden[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        h[2 * c] = qp[c][0];
        h[2 * c + 1] = qm[c][0];
    }
    rsq_all<2 * C>(h, s);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float sp = s[2 * c], sm = s[2 * c + 1];
        up[c] = qp[c][1] * (sp * sp), um[c] = qm[c][1] * (sm * sm);
        const float cp = sg * qp[c][0] * sp, cm = sg * qm[c][0] * sm;
        am[c] = __builtin_fminf(__builtin_fminf(um[c] - cm, up[c] - cp), 0.0f);
        ap[c] = __builtin_fmaxf(__builtin_fmaxf(um[c] + cm, up[c] + cp), 0.0f);
        den[c] = ap[c] - am[c];
    }
    rcp_all<C>(den, iden);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float wm = ap[c] * iden[c], wp = am[c] * iden[c];
        const float dm = um[c] - am[c], dp = up[c] - ap[c];
        const float A0 = qm[c][1] - am[c] * qm[c][0], B0 = qp[c][1] - ap[c] * qp[c][0];
        const float A1 = qm[c][1] * dm + hg * qm[c][0] * qm[c][0], B1 = qp[c][1] * dp + hg * qp[c][0] * qp[c][0];
        const float A2 = qm[c][2] * dm, B2 = qp[c][2] * dp;
        out[c][0] = wm * A0 - wp * B0;
        out[c][1] = wm * A1 - wp * B1;
        out[c][2] = wm * A2 - wp * B2;
    }
}

// HLL flux, SWE (SWECommon.h:274-313)
template <int C>
__device__ __forceinline__ void swe_hll_flux(const float (&ql)[C][3], const float (&qr)[C][3], float hg, float sg,
                                             float (&out)[C][3]) {
    float h[2 * C], s[2 * C], u_l[C], u_r[C], c_l[C], c_r[C], cs[C], ics[C], hd[C], x[2 * C], q[2 * C], S_l[C],
        S_r[C], den[C], iden[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        h[2 * c] = ql[c][0];
        h[2 * c + 1] = qr[c][0];
    }
    rsq_all<2 * C>(h, s);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float sl = s[2 * c], sr = s[2 * c + 1];
        u_l[c] = ql[c][1] * (sl * sl), u_r[c] = qr[c][1] * (sr * sr);
        c_l[c] = sg * ql[c][0] * sl, c_r[c] = sg * qr[c][0] * sr;
        cs[c] = c_l[c] + c_r[c];
    }
    rcp_all<C>(cs, ics);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float hs = ql[c][0] + qr[c][0];
        hd[c] = 0.5f * hs - 0.25f * (u_r[c] - u_l[c]) * hs * ics[c];
        x[2 * c] = 0.5f * (hd[c] + ql[c][0]) * hd[c];
        x[2 * c + 1] = 0.5f * (hd[c] + qr[c][0]) * hd[c];
    }
    sqrt_all<2 * C>(x, q);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float il = s[2 * c] * s[2 * c], ir = s[2 * c + 1] * s[2 * c + 1];
        const float q_l = (hd[c] > ql[c][0]) ? q[2 * c] * il : 1.0f;
        const float q_r = (hd[c] > qr[c][0]) ? q[2 * c + 1] * ir : 1.0f;
        S_l[c] = u_l[c] - c_l[c] * q_l;
        S_r[c] = u_r[c] + c_r[c] * q_r;
    }
    float sl[C], sr[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        hll_speeds(S_l[c], S_r[c], sl[c], sr[c]);
        den[c] = sr[c] - sl[c];
    }
    rcp_all<C>(den, iden);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float F_l[3] = {ql[c][1], ql[c][1] * u_l[c] + hg * ql[c][0] * ql[c][0], ql[c][2] * u_l[c]};
        const float F_r[3] = {qr[c][1], qr[c][1] * u_r[c] + hg * qr[c][0] * qr[c][0], qr[c][2] * u_r[c]};
        const float wl = sr[c] * iden[c], wr = sl[c] * iden[c], wq = sr[c] * sl[c] * iden[c];
#pragma unroll
        for (int k = 0; k < 3; ++k) out[c][k] = (wl * F_l[k] - wr * F_r[k]) + wq * (qr[c][k] - ql[c][k]);
    }
}

// 1 / (admissible dt) of one cell, SWE (SWECommon.h:497-504): max over the two
// directions of (|u| + sqrt(g h)) / d.
__device__ __forceinline__ float swe_cell_rate(const float q[3], float sg, float idx, float idy) {
    const float s = rsq(q[0]);
    const float ih = s * s;
    const float c = sg * q[0] * s;
    return __builtin_fmaxf((__builtin_fabsf(q[1] * ih) + c) * idx, (__builtin_fabsf(q[2] * ih) + c) * idy);
}

// ---- Euler (EulerCommon.h) -------------------------------------------------

// Predictor difference F(QL, gamma) - F(QR, gamma) (the reference's predictor
// passes gamma in the pressure slot, EE2D_KP07_dimsplit.cu:57-58).
__device__ __forceinline__ void euler_pred_diff(const float QL[4], const float QR[4], float r, float gamma,
                                                float D[4]) {
    const float uL = QL[1] * (QR[0] * r);
    const float uR = QR[1] * (QL[0] * r);
    D[0] = QL[1] - QR[1];
    D[1] = QL[1] * uL - QR[1] * uR;  // the +gamma terms cancel
    D[2] = QL[2] * uL - QR[2] * uR;
    D[3] = uL * (QL[3] + gamma) - uR * (QR[3] + gamma);
}

// 1/rho, normal velocity, pressure and sound speed of the left (even) and
// right (odd) states of C interfaces
template <int C>
__device__ __forceinline__ void euler_states(const float (&ql)[C][4], const float (&qr)[C][4], float gamma,
                                             float (&inv)[2 * C], float (&u)[2 * C], float (&P)[2 * C],
                                             float (&cs)[2 * C]) {
    float x[2 * C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        x[2 * c] = ql[c][0];
        x[2 * c + 1] = qr[c][0];
    }
    rcp_all<2 * C>(x, inv);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) {
        const float* q = (i & 1) ? qr[i / 2] : ql[i / 2];
        u[i] = q[1] * inv[i];
        P[i] = (gamma - 1.0f) * (q[3] - 0.5f * (q[1] * q[1] + q[2] * q[2]) * inv[i]);
        x[i] = gamma * P[i] * inv[i];
    }
    sqrt_all<2 * C>(x, cs);
}

// HLL flux, Euler (EulerCommon.h:117-160)
template <int C>
__device__ __forceinline__ void euler_hll_flux(const float (&ql)[C][4], const float (&qr)[C][4], float gamma,
                                               float (&out)[C][4]) {
    float inv[2 * C], u[2 * C], P[2 * C], cs[2 * C], x[C], ics[C], hd[C], y[2 * C], q[2 * C], sl[C], sr[C], iden[C];
    euler_states<C>(ql, qr, gamma, inv, u, P, cs);
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = cs[2 * c] + cs[2 * c + 1];
    rcp_all<C>(x, ics);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float hs = ql[c][0] + qr[c][0];
        hd[c] = 0.5f * hs - 0.25f * (u[2 * c + 1] - u[2 * c]) * hs * ics[c];
        y[2 * c] = 0.5f * (hd[c] + ql[c][0]) * hd[c];
        y[2 * c + 1] = 0.5f * (hd[c] + qr[c][0]) * hd[c];
    }
    sqrt_all<2 * C>(y, q);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float q_l = (hd[c] > ql[c][0]) ? q[2 * c] * inv[2 * c] : 1.0f;
        const float q_r = (hd[c] > qr[c][0]) ? q[2 * c + 1] * inv[2 * c + 1] : 1.0f;
        hll_speeds(u[2 * c] - cs[2 * c] * q_l, u[2 * c + 1] + cs[2 * c + 1] * q_r, sl[c], sr[c]);
        x[c] = sr[c] - sl[c];
    }
    rcp_all<C>(x, iden);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float ul = u[2 * c], ur = u[2 * c + 1], Pl = P[2 * c], Pr = P[2 * c + 1];
        const float F_l[4] = {ql[c][1], ql[c][1] * ul + Pl, ql[c][2] * ul, ul * (ql[c][3] + Pl)};
        const float F_r[4] = {qr[c][1], qr[c][1] * ur + Pr, qr[c][2] * ur, ur * (qr[c][3] + Pr)};
        const float wl = sr[c] * iden[c], wr = sl[c] * iden[c], wq = sr[c] * sl[c] * iden[c];
#pragma unroll
        for (int k = 0; k < 4; ++k) out[c][k] = (wl * F_l[k] - wr * F_r[k]) + wq * (qr[c][k] - ql[c][k]);
    }
}

// Central-upwind flux, Euler (EulerCommon.h:171-187)
template <int C>
__device__ __forceinline__ void euler_cu_flux(const float (&qm)[C][4], const float (&qp)[C][4], float gamma,
                                              float (&out)[C][4]) {
    float inv[2 * C], u[2 * C], P[2 * C], cs[2 * C], am[C], ap[C], x[C], iden[C];
    euler_states<C>(qm, qp, gamma, inv, u, P, cs);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int m = 2 * c, p = 2 * c + 1;
        am[c] = __builtin_fminf(__builtin_fminf(u[m] - cs[m], u[p] - cs[p]), 0.0f);
        ap[c] = __builtin_fmaxf(__builtin_fmaxf(u[m] + cs[m], u[p] + cs[p]), 0.0f);
        x[c] = ap[c] - am[c];
    }
    rcp_all<C>(x, iden);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int m = 2 * c, p = 2 * c + 1;
        const float Fp[4] = {qp[c][1], qp[c][1] * u[p] + P[p], qp[c][2] * u[p], u[p] * (qp[c][3] + P[p])};
        const float Fm[4] = {qm[c][1], qm[c][1] * u[m] + P[m], qm[c][2] * u[m], u[m] * (qm[c][3] + P[m])};
        const float wm = ap[c] * iden[c], wp = am[c] * iden[c], wq = ap[c] * am[c] * iden[c];
#pragma unroll
        for (int k = 0; k < 4; ++k) out[c][k] = (wm * Fm[k] - wp * Fp[k]) + wq * (qp[c][k] - qm[c][k]);
    }
}

// 1 / (admissible dt) of one cell, Euler (EulerCommon.h:41-49, sqrt(gamma*rho) as written)
__device__ __forceinline__ float euler_cell_rate(const float q[4], float gamma, float idx, float idy) {
    const float s = rsq(gamma * q[0]);
    const float c = gamma * q[0] * s;
    const float ih = gamma * s * s;  // 1/rho
    return __builtin_fmaxf((__builtin_fabsf(q[1] * ih) + c) * idx, (__builtin_fabsf(q[2] * ih) + c) * idy);
}

}  // namespace fast
}  // namespace fvmi
