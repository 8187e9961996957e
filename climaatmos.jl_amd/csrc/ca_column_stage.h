// ca_column_stage.h -- the implicit ARS343 stage and the explicit tendency of
// one column held in a wavefront's registers: lane l owns the R consecutive
// rows R l .. R l + R - 1 (row k = centre k and face k) of its column's W lanes, so
// a column has up to R W levels.  Face nlev carries
// u_3 = 0 and needs no row of its own.
//
// Vertical neighbours are lane exchanges (DPP wave shifts, ca_newton_pcr.hip)
// or, inside a lane's rows, register moves.  What depends on one centre alone
// (theta_v, theta_v - theta_vr, Pi^7, dp/drho) is formed once per centre and
// exchanged, not recomputed on both faces, and the centre rows of the Jacobian
// are formed on each face from the face fluxes q = I^f(rho J) g^33 and q h.
// Included by ca_newton_pcr.hip after its lane exchanges.
#pragma once
#include "ca_kernels.h"

namespace cst {

// value of the row below / above every row (row 0 / the last row receive some
// lane's value, maybe another column's: every use selects by the row index)
template <int R, class T>
__device__ __forceinline__ void prev(const T (&v)[R], T (&o)[R]) {
    const T e = pcr::up1(v[R - 1]);
#pragma unroll
    for (int r = R - 1; r > 0; --r) o[r] = v[r - 1];
    o[0] = e;
}
template <int R, class T>
__device__ __forceinline__ void next(const T (&v)[R], T (&o)[R]) {
    const T e = pcr::dn1(v[0]);
#pragma unroll
    for (int r = 0; r < R - 1; ++r) o[r] = v[r + 1];
    o[R - 1] = e;
}

// the value of the column's lane 0 in all its lanes
template <int W>
__device__ __forceinline__ float first(float v) {
    if constexpr (W == 64) return pcr::lane0(v);
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    return (threadIdx.x & 32) ? b : a;
}

// per-level tables of the lane's rows; rows beyond the column repeat the last
// centre / face so that every value stays finite
template <int R>
struct Lev {
    int k[R];
    bool hasC[R], intF[R], upF[R];  // centre k, interior face k, interior face k + 1 exist
    float is2[R], sJ[R], sJm[R], isJ[R], isJm[R];  // 1 / s^2, s^2 Jv and its reciprocal (m: centre k - 1)
    float g0[R], gp[R], gm[R];      // g^33 at faces k, k + 1, k - 1
    float Phic[R], zf[R];           // g z_c, Rayleigh profile at face k
    double Phid[R], dPhid[R];       // g z_c and the geopotential step of face k in float64
};
template <int R>
__device__ __forceinline__ void lev_load(const DevGeom &g, int lane, Lev<R> &t) {
    const int nl = g.nlev;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = R * lane + r;
        t.k[r] = k;
        t.hasC[r] = k < nl;
        t.intF[r] = k >= 1 && k < nl;
        t.upF[r] = k + 1 < nl;
        const int kc = min(k, nl - 1), km = max(kc - 1, 0), kf = min(k, nl);
        t.is2[r] = g.is2c[kc];
        t.sJ[r] = g.sc[kc] * g.sc[kc] * g.Jvc[kc];
        t.sJm[r] = g.sc[km] * g.sc[km] * g.Jvc[km];
        t.isJ[r] = g.isJc[kc];
        t.isJm[r] = g.isJc[km];
        t.g0[r] = g.g33f[kf];
        t.gp[r] = g.g33f[kc + 1];
        t.gm[r] = g.g33f[max(kf - 1, 0)];
        t.Phic[r] = g.Phic[kc];
        t.zf[r] = g.zeta_f[kf];
        t.Phid[r] = g.Phic_d[kc];
        t.dPhid[r] = g.dPhif_d[kf];
    }
}

// horizontal metric of the column and its Rayleigh coefficient
struct Met1 {
    float gu11, gu12, gu22, Jh, iJh, aw;
};
__device__ __forceinline__ Met1 met1_load(const DevGeom &g, const DevNum &n, int col) {
    Met1 m;
    m.gu11 = g.gu11[col];
    m.gu12 = g.gu12[col];
    m.gu22 = g.gu22[col];
    m.Jh = g.Jh[col];
    m.iJh = g.iJh[col];
    m.aw = !n.rayleigh ? 0.0f : (g.aw_col ? g.aw_col[col] : n.alpha_w);
    return m;
}

// 1 / d from the hardware reciprocal (1 ulp) and one Newton-Raphson step
__device__ __forceinline__ float rcp_nr(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}

// a b, with OWN rounded on its own.  The flux through a face enters the centre
// below it and leaves the one above: contracted into the two differences (one of
// two products exact, the other rounded) it is not the same value in both.  On a
// sphere the horizontal pressure gradient sees that: the winds' error against
// float64 grew by 1.5% (four steps at h_elem 16, 63 levels: 4.72e-7 against
// 4.66e-7 with OWN), for 0.3% of a step.  Independent columns show no difference
// (0.1% of the error, either way, over 1200 columns of 30 and of 63 levels) and
// contract.
template <bool OWN>
__device__ __forceinline__ float flux(float a, float b) {
    if constexpr (OWN) {
#pragma clang fp contract(off)
        return a * b;
    } else {
        return a * b;
    }
}

// Temperature in float64 from rho e_tot / rho (et), the kinetic energy and Phi
__device__ __forceinline__ double temperature(const DevNum &n, double et, float K, double Phid) {
    return fmax(n.dT_0 + (et - (double)K - Phid + n.dR_d * n.dT_0) * n.dicv_d, n.dTmin);
}

// The tridiagonal Schur system in float64 (the acoustic system is stiff:
// dtg c / dz >> 1).  With two or three rows per lane the lane's upper rows are
// eliminated first, as x_j = p_j - q_j x_0 - s_j x_0' of the lane's first row and
// that of the lane above; one row per lane is left for parallel cyclic
// reduction over the column's W lanes, and the others are substituted back.
template <int R, int W>
__device__ __forceinline__ void solve(const double (&L)[R], const double (&D)[R], const double (&U)[R],
                                      const double (&b)[R], float (&x)[R]) {
    static_assert(R >= 1 && R <= 3, "one to three rows per lane");
    double Ld = L[0], Dd = D[0], Ud = U[0], rd = b[0];
    double p1 = 0.0, q1 = 0.0, s1 = 0.0, p2 = 0.0, q2 = 0.0, s2 = 0.0;
    if constexpr (R >= 2) {
        const double i = ca_drcp(D[1]);
        if constexpr (R == 2) {
            q1 = L[1] * i;
            s1 = U[1] * i;
            p1 = b[1] * i;
        } else {
            const double f = L[2] * i, j = ca_drcp(D[2] - f * U[1]);
            q2 = -(f * L[1]) * j;
            s2 = U[2] * j;
            p2 = (b[2] - f * b[1]) * j;
            q1 = (L[1] - U[1] * q2) * i;
            s1 = -(U[1] * s2) * i;
            p1 = (b[1] - U[1] * p2) * i;
        }
        // the last row of the lane below
        const double qb = pcr::below<W>(R == 2 ? q1 : q2), sb = pcr::below<W>(R == 2 ? s1 : s2);
        const double pb = pcr::below<W>(R == 2 ? p1 : p2);
        Dd = D[0] - L[0] * sb - U[0] * q1;
        rd = b[0] - L[0] * pb - U[0] * p1;
        Ld = -L[0] * qb;
        Ud = -U[0] * s1;
    }
#pragma unroll
    for (int s = 1; s < W; s <<= 1) {
        const double iD = ca_drcp(Dd);
        const double Ln = Ld * iD, Un = Ud * iD, rn = rd * iD;
        double La, Ua, ra, Lb, Ub, rb;
        pcr::pcr_nbrs<W>(Ln, s, La, Lb);
        pcr::pcr_nbrs<W>(Un, s, Ua, Ub);
        pcr::pcr_nbrs<W>(rn, s, ra, rb);
        const double nD = Dd - Ld * Ua - Ud * Lb;
        const double nr = rd - Ld * ra - Ud * rb;
        Ld = -Ld * La;
        Ud = -Ud * Ub;
        Dd = nD;
        rd = nr;
    }
    const double xe = rd * ca_drcp(Dd);
    x[0] = (float)xe;
    if constexpr (R >= 2) {
        const double xn = pcr::above<W>(xe);
        x[1] = (float)(p1 - q1 * xe - s1 * xn);
        if constexpr (R == 3) x[2] = (float)(p2 - q2 * xe - s2 * xn);
    }
}

// correct_implicit_advection_tendency! (implicit_tendency.jl:322-339): the rho e_tot
// tendency of the upwind minus the central enthalpy flux, from u_3, h (made
// relative to the lowest cell, which cancels) and rho J of the new state
template <int R, int W>
__device__ __forceinline__ void correction(const Lev<R> &t, const Met1 &m, const DevNum &n, int nl, const float (&u3)[R],
                                           float (&hr)[R], const float (&rJn)[R], float (&corr)[R]) {
    const float href = first<W>(hr[0]);
#pragma unroll
    for (int r = 0; r < R; ++r) hr[r] -= href;
    float h1[R], h2[R], h4[R], rJm[R], dF[R], dF1[R];
    prev<R>(hr, h1);
    prev<R>(h1, h2);
    next<R>(hr, h4);
    prev<R>(rJn, rJm);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        dF[r] = 0.0f;
        if (t.intF[r]) {
            const float v = u3[r] * t.g0[r];
            const float up = upwind_product(n.upw, t.k[r], nl, v, n.dt, h2[r], h1[r], hr[r], h4[r]);
            dF[r] = 0.5f * (rJm[r] + rJn[r]) * (up - v * (0.5f * (h1[r] + hr[r])));
        }
    }
    next<R>(dF, dF1);
#pragma unroll
    for (int r = 0; r < R; ++r)
        corr[r] = t.hasC[r] ? ((t.upF[r] ? 0.0f - dF1[r] : 0.0f) + dF[r]) * (m.iJh * t.isJ[r]) : 0.0f;
}

// One implicit stage of one column: U~ (rho, u1, u2, rhoe, u3 with u3 = 0 off
// the interior faces) in, U (rho, rhoe, u3; u_h is unchanged) and F_I =
// (U - U~) / dtg (fr, fe, fu) out.  Same algorithm as k_newton_pcr: one Newton
// iteration with the manual Jacobian, the Schur complement on u_3 and the
// post-Newton upwind correction.
template <int R, int W, bool OWN>
__device__ __forceinline__ void newton(const Lev<R> &t, const Met1 &m, const DevNum &n, int nl, float dtg, float idtg,
                                       float (&rho)[R], const float (&u1)[R], const float (&u2)[R], float (&rhoe)[R],
                                       float (&u3)[R], float (&fr)[R], float (&fe)[R], float (&fu)[R]) {
    float u3m[R], u3p[R];
    prev<R>(u3, u3m);
    next<R>(u3, u3p);
    float Kh[R], h[R], dp[R], thv[R];
    double thd[R], Pid[R], Pi7[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        u3p[r] = t.upF[r] ? u3p[r] : 0.0f;
        const float c1 = t.is2[r] * (m.gu11 * u1[r] + m.gu12 * u2[r]);
        const float c2 = t.is2[r] * (m.gu12 * u1[r] + m.gu22 * u2[r]);
        Kh[r] = u1[r] * c1 + u2[r] * c2;
        const float K = 0.5f * (Kh[r] + 0.5f * (u3[r] * t.g0[r] * u3[r] + u3p[r] * t.gp[r] * u3p[r]));
        const double et = (double)rhoe[r] * ca_drcp((double)rho[r]);
        const double Td = temperature(n, et, K, t.Phid[r]);
        Pid[r] = ca_dexner(n, (double)rho[r] * n.dR_d * Td * n.dp0inv);
        h[r] = (float)(et + n.dR_d * Td);
        thv[r] = (float)Td * ca_rcp((float)Pid[r]);
        Pi7[r] = ca_dpow7(Pid[r]);
        thd[r] = (Td - (n.dTmr + (n.dTsr - n.dTmr) * Pi7[r])) * ca_drcp(Pid[r]);
        dp[r] = n.kap * (n.T_0 * n.cp_d - K - t.Phic[r]);  // d p / d rho at fixed rho e_tot
    }
    float ra[R], ha[R], dpa[R], thva[R], q[R], qh[R], qm[R], qhm[R], qp[R], qhp[R];
    double thda[R], Pia[R], Pi7a[R];
    prev<R>(rho, ra);
    prev<R>(h, ha);
    prev<R>(dp, dpa);
    prev<R>(thv, thva);
    prev<R>(thd, thda);
    prev<R>(Pid, Pia);
    prev<R>(Pi7, Pi7a);
#pragma unroll
    for (int r = 0; r < R; ++r) {  // face k: I^f(rho J) g^33 and its product with I^f(h); 0 off the interior
        const float rJf = 0.5f * (ra[r] * t.sJm[r] + rho[r] * t.sJ[r]) * m.Jh;
        q[r] = t.intF[r] ? rJf * t.g0[r] : 0.0f;
        qh[r] = t.intF[r] ? q[r] * (0.5f * (ha[r] + h[r])) : 0.0f;
    }
    prev<R>(q, qm);
    prev<R>(qh, qhm);
    next<R>(q, qp);
    next<R>(qh, qhp);
    float a0[R], a1[R], e0[R], e1[R], Rr[R], Re[R], x[R], x1[R];
    double L[R], D[R], U[R], b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        qp[r] = t.upF[r] ? qp[r] : 0.0f;
        qhp[r] = t.upF[r] ? qhp[r] : 0.0f;
        // centre k: A(rho, u3), A(rho e, u3) on faces k, k + 1 and R = dtg T_imp
        const float c = dtg * (m.iJh * t.isJ[r]);
        a0[r] = c * q[r];
        a1[r] = -c * qp[r];
        e0[r] = c * qh[r];
        e1[r] = -c * qhp[r];
        Rr[r] = -c * (flux<OWN>(qp[r], u3p[r]) - flux<OWN>(q[r], u3[r]));
        Re[r] = -c * (flux<OWN>(qhp[r], u3p[r]) - flux<OWN>(qh[r], u3[r]));
        L[r] = 0.0;
        D[r] = 1.0;
        U[r] = 0.0;
        b[r] = 0.0;
        if (t.intF[r]) {
            // centre k - 1, from the same face values
            const float cm = dtg * (m.iJh * t.isJm[r]);
            const float q0 = t.k[r] >= 2 ? qm[r] : 0.0f, qh0 = t.k[r] >= 2 ? qhm[r] : 0.0f;
            const float w0 = t.k[r] >= 2 ? u3m[r] : 0.0f;
            const float pa0 = cm * q0, pa1 = -cm * q[r], pe0 = cm * qh0, pe1 = -cm * qh[r];
            const float pRr = -cm * (flux<OWN>(q[r], u3[r]) - flux<OWN>(q0, w0)), pRe = -cm * (flux<OWN>(qh[r], u3[r]) - flux<OWN>(qh0, w0));
            // face row (manual_sparse_jacobian.jl:713-870)
            const float pg = ca_rcp(0.5f * (ra[r] + rho[r]));
            const double dPid = Pid[r] - Pia[r];
            const float buoy = n.cp_d * (0.5f * (thva[r] + thv[r])) * (float)dPid * pg;
            const float r0 = dtg * (pg * dpa[r] + 0.5f * buoy), r1 = dtg * (0.5f * buoy - pg * dp[r]);
            const float ef = dtg * (pg * n.kap);
            const float ka = -n.kap * ra[r] * pg, kb = n.kap * rho[r] * pg;
            const float beta = m.aw * t.zf[r];
            const float wf = 0.5f * u3[r] * t.g0[r];
            const float lo = dtg * (ka * (0.5f * w0 * t.gm[r]));
            const float dd = dtg * ((ka + kb) * wf - beta) - 1.0f;
            const float up = dtg * (kb * (0.5f * u3p[r] * t.gp[r]));
            // the pressure gradient and buoyancy (implicit_tendency.jl:287-293) in float64
            const double sg = dPid * ca_drcp(Pia[r] + Pid[r]), s2 = sg * sg;
            double z = 1.0 / 19.0;
#pragma unroll
            for (int j = 17; j >= 1; j -= 2) z = fma(z, s2, 1.0 / j);
            const double dPhr =
                -n.dcp_d * (n.dTmr * (2.0 * sg * z) + (n.dTsr - n.dTmr) * (1.0 / 7.0) * (Pi7[r] - Pi7a[r]));
            const float pgf = (float)(-((t.dPhid[r] - dPhr) + n.dcp_d * (0.5 * (thda[r] + thd[r])) * dPid));
            const float Ru3 = dtg * (pgf - beta * u3[r]);
            L[r] = lo + r0 * pa0 + ef * pe0;
            D[r] = dd + r0 * pa1 + ef * pe1 + r1 * a0[r] - ef * e0[r];
            U[r] = up + r1 * a1[r] - ef * e1[r];
            b[r] = Ru3 + r0 * pRr + r1 * Rr[r] + ef * pRe - ef * Re[r];
        }
    }
    solve<R, W>(L, D, U, b, x);
    next<R>(x, x1);
    float u3n[R], hr[R], rJn[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float xp = t.upF[r] ? x1[r] : 0.0f, x0 = t.intF[r] ? x[r] : 0.0f;
        const float dr = a0[r] * x0 + a1[r] * xp - Rr[r], de = e0[r] * x0 + e1[r] * xp - Re[r];
        rho[r] -= dr;
        rhoe[r] -= de;
        u3[r] -= x0;  // 0 off the interior faces
        u3n[r] = u3[r];
        fr[r] = -dr * idtg;
        fe[r] = -de * idtg;
        fu[r] = -x0 * idtg;
    }
    if (n.upw == 0) return;
    next<R>(u3n, u3p);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float w1 = t.upF[r] ? u3p[r] : 0.0f;
        const float K = 0.5f * (Kh[r] + 0.5f * (u3[r] * t.g0[r] * u3[r] + w1 * t.gp[r] * w1));
        const double et = (double)rhoe[r] * ca_drcp((double)rho[r]);
        hr[r] = (float)(et + n.dR_d * temperature(n, et, K, t.Phid[r]));
        rJn[r] = rho[r] * t.sJ[r] * m.Jh;
    }
    float corr[R];
    correction<R, W>(t, m, n, nl, u3, hr, rJn, corr);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        rhoe[r] += dtg * corr[r];
        fe[r] += corr[r];
    }
}

// ------------------------------------------------ implicit vertical diffusion
// a tridiagonal system in float32 with N right-hand sides (solved in place):
// the diffusion blocks, -I minus a diffusion operator, are diagonally dominant.
// Row elimination as in solve.
template <int R, int W, int N>
__device__ __forceinline__ void tri32(const float (&L)[R], const float (&D)[R], const float (&U)[R], float (&b)[N][R]) {
    float Ls, Ds, Us, r[N], Lo = 0.0f, Uo = 0.0f, ro[N];
    if constexpr (R == 1) {
        Ls = L[0];
        Ds = D[0];
        Us = U[0];
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = b[i][0];
    } else {
        const float iD = rcp_nr(D[1]);
        Lo = L[1] * iD;
        Uo = U[1] * iD;
        const float Lp = pcr::below<W>(Lo), Up = pcr::below<W>(Uo);
        Ds = D[0] - L[0] * Up - U[0] * Lo;
        Ls = -L[0] * Lp;
        Us = -U[0] * Uo;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            ro[i] = b[i][1] * iD;
            r[i] = b[i][0] - L[0] * pcr::below<W>(ro[i]) - U[0] * ro[i];
        }
    }
#pragma unroll
    for (int s = 1; s < W; s <<= 1) {
        const float iD = rcp_nr(Ds);
        const float Ln = Ls * iD, Un = Us * iD;
        float La, Ua, Lb, Ub;
        pcr::pcr_nbrs<W>(Ln, s, La, Lb);
        pcr::pcr_nbrs<W>(Un, s, Ua, Ub);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float ra, rb;
            pcr::pcr_nbrs<W>(r[i] * iD, s, ra, rb);
            r[i] = r[i] - Ls * ra - Us * rb;
        }
        Ds = Ds - Ls * Ua - Us * Lb;
        Ls = -Ls * La;
        Us = -Us * Ub;
    }
    const float iD = rcp_nr(Ds);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float x = r[i] * iD;
        b[i][0] = x;
        if constexpr (R == 2) b[i][1] = ro[i] - Lo * x - Uo * pcr::above<W>(x);
    }
}

// level tables of the diffusion
template <int R>
struct Dif {
    float fJ[R];         // face k: s^2 Jv g^33
    float s[R], is[R];   // centre k: s and 1 / s on a sphere, 1 on columns
    float dis[R];        // 1 / s_k - 1 / s_{k-1}
    float kdec[R];
};
template <int R>
__device__ __forceinline__ void dif_load(const DevGeom &g, const DevNum &n, int lane, Dif<R> &d) {
    const int nl = g.nlev;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = R * lane + r, kc = min(k, nl - 1), km = max(kc - 1, 0), kf = min(k, nl);
        d.fJ[r] = g.sf[kf] * g.sf[kf] * g.Jvf[kf] * g.g33f[kf];
        const float s = n.sphere ? g.sc[kc] : 1.0f, sm = n.sphere ? g.sc[km] : 1.0f;
        d.s[r] = s;
        d.is[r] = 1.0f / s;
        d.dis[r] = (sm - s) * (1.0f / s) * (1.0f / sm);
        d.kdec[r] = n.vdk == 0 ? g.kdec[kc] : 1.0f;
    }
}

// The implicit stage with implicit vertical diffusion: as newton, with the
// diffusion of rho e_tot and u_h in T_imp, its blocks in the Jacobian, and the
// approximate block-arrowhead solve (manual_sparse_jacobian.jl:538-578) of
// n.siters iterations.  U overwrites U~ in all five components.
// The momentum diffusion is formed on u_i / s: the Cartesian velocity is
// (u_1 a^1 + u_2 a^2) / s with the column's level-independent basis, and its
// flux divergence projects back with a_i, whose products with a^j are delta_ij.
template <int R, int W>
__device__ __forceinline__ void newton_idiff(const Lev<R> &t, const Dif<R> &df, const Met1 &m, const DevNum &n, int nl,
                                             float D0, float dtg, float (&rho)[R], float (&u1)[R], float (&u2)[R],
                                             float (&rhoe)[R], float (&u3)[R]) {
    float u3m[R], u3p[R];
    prev<R>(u3, u3m);
    next<R>(u3, u3p);
    float h[R], dp[R], thv[R], c1[R], c2[R], iK[R], irho[R];
    double Td[R], thd[R], Pid[R], Pi7[R];
    float spd[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        u3p[r] = t.upF[r] ? u3p[r] : 0.0f;
        c1[r] = t.is2[r] * (m.gu11 * u1[r] + m.gu12 * u2[r]);
        c2[r] = t.is2[r] * (m.gu12 * u1[r] + m.gu22 * u2[r]);
        const float uu = u1[r] * c1[r] + u2[r] * c2[r];
        spd[r] = sqrtf(uu);
        const float K = 0.5f * (uu + 0.5f * (u3[r] * t.g0[r] * u3[r] + u3p[r] * t.gp[r] * u3p[r]));
        const double et = (double)rhoe[r] * ca_drcp((double)rho[r]);
        Td[r] = temperature(n, et, K, t.Phid[r]);
        const double pd = (double)rho[r] * n.dR_d * Td[r];
        iK[r] = (float)pd;  // the pressure; becomes 1 / K_h below
        Pid[r] = ca_dexner(n, pd * n.dp0inv);
        h[r] = (float)(et + n.dR_d * Td[r]);
        thv[r] = (float)Td[r] * ca_rcp((float)Pid[r]);
        Pi7[r] = ca_dpow7(Pid[r]);
        thd[r] = (Td[r] - (n.dTmr + (n.dTsr - n.dTmr) * Pi7[r])) * ca_drcp(Pid[r]);
        dp[r] = n.kap * (n.T_0 * n.cp_d - K - t.Phic[r]);
        irho[r] = rcp_nr(rho[r]);
    }
    const float spd0 = n.vdk == 1 ? first<W>(spd[0]) : 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {  // ca_Kc
        float K = D0 * df.kdec[r];
        if (n.vdk == 1) {
            const float p = iK[r], x = (85000.0f - p) * 1.0e-4f;
            K = n.CE * spd0 * n.za * (p > 85000.0f ? 1.0f : expf(-(x * x)));
        }
        iK[r] = 1.0f / fmaxf(K, 1.1920929e-07f);
    }
    float ra[R], ha[R], dpa[R], thva[R], iKa[R], u1a[R], u2a[R], c1a[R], c2a[R], irm[R], irp[R];
    double Tda[R], thda[R], Pia[R], Pi7a[R];
    prev<R>(rho, ra);
    prev<R>(h, ha);
    prev<R>(dp, dpa);
    prev<R>(thv, thva);
    prev<R>(iK, iKa);
    prev<R>(u1, u1a);
    prev<R>(u2, u2a);
    prev<R>(c1, c1a);
    prev<R>(c2, c2a);
    prev<R>(irho, irm);
    next<R>(irho, irp);
    prev<R>(Td, Tda);
    prev<R>(thd, thda);
    prev<R>(Pid, Pia);
    prev<R>(Pi7, Pi7a);
    float q[R], qh[R], cf[R], Fs[R], F1[R], F2[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {  // faces: advective and diffusive fluxes, 0 off the interior
        q[r] = qh[r] = cf[r] = Fs[r] = F1[r] = F2[r] = 0.0f;
        if (t.intF[r]) {
            q[r] = 0.5f * (ra[r] * t.sJm[r] + rho[r] * t.sJ[r]) * m.Jh * t.g0[r];
            qh[r] = q[r] * (0.5f * (ha[r] + h[r]));
            const float rK = (0.5f * (ra[r] + rho[r])) * (1.0f / (0.5f * (iKa[r] + iK[r])));
            cf[r] = m.Jh * df.fJ[r] * rK;
            // s_d(k) - s_d(k - 1) from the float64 temperatures, u_i / s from the
            // differences plus the metric step: no difference of near equals
            Fs[r] = -cf[r] * (n.cp_d * (float)(Td[r] - Tda[r]) + (float)t.dPhid[r]);
            F1[r] = -cf[r] * ((u1[r] - u1a[r]) * df.is[r] + u1a[r] * df.dis[r]);
            F2[r] = -cf[r] * ((u2[r] - u2a[r]) * df.is[r] + u2a[r] * df.dis[r]);
        }
    }
    float qm[R], qhm[R], qp[R], qhp[R], cfp[R], Fsp[R], F1p[R], F2p[R];
    prev<R>(q, qm);
    prev<R>(qh, qhm);
    next<R>(q, qp);
    next<R>(qh, qhp);
    next<R>(cf, cfp);
    next<R>(Fs, Fsp);
    next<R>(F1, F1p);
    next<R>(F2, F2p);
    const float kcv = n.cp_d / n.cv_d;
    float a0[R], a1[R], e0[R], e1[R], Rr[R], Re[R], elo[R], ed[R], eup[R], hlo[R], hd[R], hup[R], bh[2][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool up = t.upF[r];
        qp[r] = up ? qp[r] : 0.0f;
        qhp[r] = up ? qhp[r] : 0.0f;
        const float iJ = m.iJh * t.isJ[r], c = dtg * iJ;
        a0[r] = c * q[r];
        a1[r] = -c * qp[r];
        e0[r] = c * qh[r];
        e1[r] = -c * qhp[r];
        Rr[r] = -c * (flux<true>(qp[r], u3p[r]) - flux<true>(q[r], u3[r]));
        Re[r] = -c * ((flux<true>(qhp[r], u3p[r]) - flux<true>(qh[r], u3[r])) + ((up ? Fsp[r] : 0.0f) - Fs[r]));
        const float ch = -c * df.s[r] * irho[r];
        bh[0][r] = ch * ((up ? F1p[r] : 0.0f) - F1[r]);
        bh[1][r] = ch * ((up ? F2p[r] : 0.0f) - F2[r]);
        const float dlo = cf[r] * c, dup = up ? cfp[r] * c : 0.0f, dd = -(dlo + dup);
        elo[r] = t.intF[r] ? dlo * (kcv * irm[r]) : 0.0f;
        ed[r] = dd * (kcv * irho[r]) - 1.0f;
        eup[r] = up ? dup * (kcv * irp[r]) : 0.0f;
        hlo[r] = irho[r] * dlo;
        hd[r] = irho[r] * dd - 1.0f;
        hup[r] = irho[r] * dup;
        if (!t.hasC[r]) {  // beyond the column: identity rows
            a0[r] = a1[r] = e0[r] = e1[r] = Rr[r] = Re[r] = bh[0][r] = bh[1][r] = 0.0f;
            elo[r] = eup[r] = hlo[r] = hup[r] = 0.0f;
            ed[r] = hd[r] = 1.0f;
        }
    }
    // y_e = inv(A_ee) b_e
    float ye[1][R], yea[R], eda[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ye[0][r] = Re[r];
    tri32<R, W, 1>(elo, ed, eup, ye);
    prev<R>(ye[0], yea);
    prev<R>(ed, eda);
    // face rows, b_w' = b_w - A_wrho y_rho - A_we y_e, and the preconditioner's u_3
    // block with diag(A_ee) in place of A_ee
    float r0[R], r1[R], ef[R], lo[R], dd[R], up_[R], h0a[R], h0b[R], h1a[R], h1b[R], bw[R];
    double Pl[R], Pd[R], Pu[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        r0[r] = r1[r] = ef[r] = lo[r] = up_[r] = h0a[r] = h0b[r] = h1a[r] = h1b[r] = bw[r] = 0.0f;
        dd[r] = 1.0f;
        Pl[r] = Pu[r] = 0.0;
        Pd[r] = 1.0;
        if (t.intF[r]) {
            const float cm = dtg * (m.iJh * t.isJm[r]);
            const bool two = t.k[r] >= 2;
            const float q0 = two ? qm[r] : 0.0f, qh0 = two ? qhm[r] : 0.0f, w0 = two ? u3m[r] : 0.0f;
            const float pa0 = cm * q0, pa1 = -cm * q[r], pe0 = cm * qh0, pe1 = -cm * qh[r];
            const float pRr = -cm * (flux<true>(q[r], u3[r]) - flux<true>(q0, w0));
            const float pg = ca_rcp(0.5f * (ra[r] + rho[r]));
            const double dPid = Pid[r] - Pia[r];
            const float buoy = n.cp_d * (0.5f * (thva[r] + thv[r])) * (float)dPid * pg;
            r0[r] = dtg * (pg * dpa[r] + 0.5f * buoy);
            r1[r] = dtg * (0.5f * buoy - pg * dp[r]);
            ef[r] = dtg * (pg * n.kap);
            const float ka = -dtg * n.kap * ra[r] * pg, kb = dtg * n.kap * rho[r] * pg;
            const float beta = m.aw * t.zf[r];
            lo[r] = ka * (0.5f * w0 * t.gm[r]);
            dd[r] = (ka + kb) * (0.5f * u3[r] * t.g0[r]) - dtg * beta - 1.0f;
            up_[r] = kb * (0.5f * u3p[r] * t.gp[r]);
            h0a[r] = ka * c1a[r];
            h0b[r] = ka * c2a[r];
            h1a[r] = kb * c1[r];
            h1b[r] = kb * c2[r];
            const double sg = dPid * ca_drcp(Pia[r] + Pid[r]), s2 = sg * sg;
            double z = 1.0 / 19.0;
#pragma unroll
            for (int j = 17; j >= 1; j -= 2) z = fma(z, s2, 1.0 / j);
            const double dPhr =
                -n.dcp_d * (n.dTmr * (2.0 * sg * z) + (n.dTsr - n.dTmr) * (1.0 / 7.0) * (Pi7[r] - Pi7a[r]));
            const float pgf = (float)(-((t.dPhid[r] - dPhr) + n.dcp_d * (0.5 * (thda[r] + thd[r])) * dPid));
            bw[r] = dtg * (pgf - beta * u3[r]) + r0[r] * pRr + r1[r] * Rr[r] - ef[r] * (yea[r] - ye[0][r]);
            const float ia = ef[r] * rcp_nr(eda[r]), ib = ef[r] * rcp_nr(ed[r]);
            Pl[r] = lo[r] + r0[r] * pa0 - ia * pe0;
            Pd[r] = dd[r] + r0[r] * pa1 + r1[r] * a0[r] - ia * pe1 + ib * e0[r];
            Pu[r] = up_[r] + r1[r] * a1[r] + ib * e1[r];
        }
    }
    float xh1[R], xh2[R], xw[R], xwp[R];
#pragma unroll
    for (int r = 0; r < R; ++r) xh1[r] = xh2[r] = xw[r] = 0.0f;
    for (int it = 0; it < n.siters; ++it) {
        float rh[2][R], rw[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            rh[0][r] = bh[0][r];
            rh[1][r] = bh[1][r];
            rw[r] = bw[r];
        }
        if (it > 0) {  // r = b' - S x
            float x1m[R], x1p[R], x2m[R], x2p[R], xwm[R], mm[1][R], mma[R], pA[R], pAa[R];
            prev<R>(xh1, x1m);
            next<R>(xh1, x1p);
            prev<R>(xh2, x2m);
            next<R>(xh2, x2p);
            prev<R>(xw, xwm);
            next<R>(xw, xwp);
#pragma unroll
            for (int r = 0; r < R; ++r) {  // hlo, hup and the couplings are 0 where a neighbour is missing
                const float wp = t.upF[r] ? xwp[r] : 0.0f;
                rh[0][r] -= hd[r] * xh1[r] + (t.intF[r] ? hlo[r] * x1m[r] : 0.0f) + (t.upF[r] ? hup[r] * x1p[r] : 0.0f);
                rh[1][r] -= hd[r] * xh2[r] + (t.intF[r] ? hlo[r] * x2m[r] : 0.0f) + (t.upF[r] ? hup[r] * x2p[r] : 0.0f);
                mm[0][r] = e0[r] * xw[r] + e1[r] * wp;  // A_ew x_w
                pA[r] = a0[r] * xw[r] + a1[r] * wp;     // A_rho,w x_w
            }
            tri32<R, W, 1>(elo, ed, eup, mm);
            prev<R>(mm[0], mma);
            prev<R>(pA, pAa);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (t.intF[r]) {
                    float sx = dd[r] * xw[r] + (t.k[r] >= 2 ? lo[r] * xwm[r] : 0.0f) + (t.upF[r] ? up_[r] * xwp[r] : 0.0f);
                    sx += h0a[r] * x1m[r] + h0b[r] * x2m[r] + h1a[r] * xh1[r] + h1b[r] * xh2[r];
                    sx += r0[r] * pAa[r] + r1[r] * pA[r] - ef[r] * (mma[r] - mm[0][r]);
                    rw[r] -= sx;
                }
        }
        // z_h = inv(A_hh) r_h (two components); z_w = inv(P_ww) (r_w - A_wh z_h)
        tri32<R, W, 2>(hlo, hd, hup, rh);
        float z1m[R], z2m[R], zw[R];
        double rd[R];
        prev<R>(rh[0], z1m);
        prev<R>(rh[1], z2m);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (t.intF[r]) rw[r] -= h0a[r] * z1m[r] + h0b[r] * z2m[r] + h1a[r] * rh[0][r] + h1b[r] * rh[1][r];
            rd[r] = rw[r];
        }
        solve<R, W>(Pl, Pd, Pu, rd, zw);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            xh1[r] += rh[0][r];
            xh2[r] += rh[1][r];
            xw[r] += t.intF[r] ? zw[r] : 0.0f;
        }
    }
    next<R>(xw, xwp);
    float xe[1][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        xwp[r] = t.upF[r] ? xwp[r] : 0.0f;
        xe[0][r] = Re[r] - (e0[r] * xw[r] + e1[r] * xwp[r]);
    }
    tri32<R, W, 1>(elo, ed, eup, xe);
    // Newton update
#pragma unroll
    for (int r = 0; r < R; ++r) {
        rho[r] -= a0[r] * xw[r] + a1[r] * xwp[r] - Rr[r];
        u1[r] -= xh1[r];
        u2[r] -= xh2[r];
        rhoe[r] -= xe[0][r];
        u3[r] -= xw[r];  // 0 off the interior faces
    }
    if (n.upw == 0) return;
    // post-Newton upwind correction at the new state
    float hr[R], rJn[R];
    next<R>(u3, u3p);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float w1 = t.upF[r] ? u3p[r] : 0.0f;
        const float d1 = t.is2[r] * (m.gu11 * u1[r] + m.gu12 * u2[r]);
        const float d2 = t.is2[r] * (m.gu12 * u1[r] + m.gu22 * u2[r]);
        const float K = 0.5f * ((u1[r] * d1 + u2[r] * d2) + 0.5f * (u3[r] * t.g0[r] * u3[r] + w1 * t.gp[r] * w1));
        const double et = (double)rhoe[r] * ca_drcp((double)rho[r]);
        hr[r] = (float)(et + n.dR_d * temperature(n, et, K, t.Phid[r]));
        rJn[r] = rho[r] * t.sJ[r] * m.Jh;
    }
    float corr[R];
    correction<R, W>(t, m, n, nl, u3, hr, rJn, corr);
#pragma unroll
    for (int r = 0; r < R; ++r) rhoe[r] += dtg * corr[r];
}

}  // namespace cst
