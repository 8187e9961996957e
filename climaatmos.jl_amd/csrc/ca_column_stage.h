// ca_column_stage.h -- the implicit ARS343 stage and the explicit tendency of
// one column held in a wavefront's registers: lane l owns the R consecutive
// rows R l .. R l + R - 1 (row k = centre k and face k), so R = 1 holds
// columns of up to 64 levels and R = 2 of up to 128.  Face nlev carries
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
// lane's finite value; every use selects by the row index)
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

// Temperature in float64 from rho e_tot / rho (et), the kinetic energy and Phi
__device__ __forceinline__ double temperature(const DevNum &n, double et, float K, double Phid) {
    return fmax(n.dT_0 + (et - (double)K - Phid + n.dR_d * n.dT_0) * n.dicv_d, n.dTmin);
}

// The tridiagonal Schur system in float64 (the acoustic system is stiff:
// dtg c / dz >> 1).  Two rows per lane: the odd row is eliminated into its
// even neighbours first, which leaves one row per lane for parallel cyclic
// reduction over the column's W lanes, and is substituted back.  With W = 32 the
// exchanges across lanes 31 / 32 fetch the other column's finite values, which
// meet exactly zero couplings.
template <int R, int W>
__device__ __forceinline__ void solve(const double (&L)[R], const double (&D)[R], const double (&U)[R],
                                      const double (&b)[R], float (&x)[R]) {
    double Ld, Dd, Ud, rd, Lo = 0.0, Uo = 0.0, ro = 0.0;
    if constexpr (R == 1) {
        Ld = L[0];
        Dd = D[0];
        Ud = U[0];
        rd = b[0];
    } else {
        static_assert(R == 2, "one or two rows per lane");
        const double i = ca_drcp(D[1]);
        Lo = L[1] * i;
        Uo = U[1] * i;
        ro = b[1] * i;
        const double Lp = pcr::up1(Lo), Up = pcr::up1(Uo), rp = pcr::up1(ro);  // odd row of the lane below
        Dd = D[0] - L[0] * Up - U[0] * Lo;
        rd = b[0] - L[0] * rp - U[0] * ro;
        Ld = -L[0] * Lp;
        Ud = -U[0] * Uo;
    }
#pragma unroll
    for (int s = 1; s < W; s <<= 1) {
        const double iD = ca_drcp(Dd);
        const double Ln = Ld * iD, Un = Ud * iD, rn = rd * iD;
        double La, Ua, ra, Lb, Ub, rb;
        pcr::pcr_nbrs(Ln, s, La, Lb);
        pcr::pcr_nbrs(Un, s, Ua, Ub);
        pcr::pcr_nbrs(rn, s, ra, rb);
        const double nD = Dd - Ld * Ua - Ud * Lb;
        const double nr = rd - Ld * ra - Ud * rb;
        Ld = -Ld * La;
        Ud = -Ud * Ub;
        Dd = nD;
        rd = nr;
    }
    const double xe = rd * ca_drcp(Dd);
    x[0] = (float)xe;
    if constexpr (R == 2) x[1] = (float)(ro - Lo * xe - Uo * pcr::dn1(xe));
}

// One implicit stage of one column: U~ (rho, u1, u2, rhoe, u3 with u3 = 0 off
// the interior faces) in, U (rho, rhoe, u3; u_h is unchanged) and F_I =
// (U - U~) / dtg (fr, fe, fu) out.  Same algorithm as k_newton_pcr: one Newton
// iteration with the manual Jacobian, the Schur complement on u_3 and the
// post-Newton upwind correction.
template <int R, int W>
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
        Rr[r] = -c * (qp[r] * u3p[r] - q[r] * u3[r]);
        Re[r] = -c * (qhp[r] * u3p[r] - qh[r] * u3[r]);
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
            const float pRr = -cm * (q[r] * u3[r] - q0 * w0), pRe = -cm * (qh[r] * u3[r] - qh0 * w0);
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
    for (int r = 0; r < R; ++r) {
        const float corr = t.hasC[r] ? ((t.upF[r] ? 0.0f - dF1[r] : 0.0f) + dF[r]) * (m.iJh * t.isJ[r]) : 0.0f;
        rhoe[r] += dtg * corr;
        fe[r] += corr;
    }
}

}  // namespace cst
