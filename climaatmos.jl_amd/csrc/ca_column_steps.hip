// ca_column_steps.hip -- whole ARS343 steps of independent columns in one
// launch: a wavefront per column, the column in its registers for all steps.
//
// The step is the one ca_step and ca_ensemble_step describe: explicit tendency
// (k_explicit's column form), three implicit stages (ca_column_stage.h), and
// the final combination u + dt sum_j b_j (F_E,j + F_I,j) with the impenetrability
// filter.  Lane l holds rows R l .. R l + R - 1 of the column (R = 1: up to 64
// levels, R = 2: up to 128): its state, the stage state, three explicit and two
// implicit stage tendencies and the level tables stay in registers, and the
// state is read and written once per launch.
//
// What bounds it: one column's chain of dependent instructions; columns do not
// share anything, and up to 1024 (one per SIMD) run at the speed of one.  As
// LDS phases of a workgroup per member (k_ensemble) a step took about 60
// barriers: 60 steps of 512 members of 30 to 128 levels 3350 us at 64 lanes and
// about 1600 at 256, 505 here (8.4 us per step, set by the deepest members).  As
// ca_step's kernels over a column grid it took seven launches: 49 us per step
// for one column of 30 levels, 4.8 here.  Large grids gain as well, since nothing
// goes through memory between stages: 65,536 columns of 63 levels 692 -> 317 us
// as one step per call, 608 -> 231 with ten; so every column grid takes this
// launch.
#include "ca_kernels.h"
#include "ca_column_stage.h"

// where the columns live: members[m] with their own tables (the ensembles), or
// column m of a grid
struct ColumnSet {
    const DevGeom *members;  // null: column m of g
    const int *order;        // ensembles: the member of workgroup b
    const int64_t *off;      // ensembles: offset of member m's state
};

namespace cst {

// tables of the explicit tendency
template <int R>
struct Exp {
    float Jf[R], iJf[R], isf[R], iJvf[R];  // face k: s^2 Jv and its reciprocal (without J_h), 1 / s, 1 / Jv
    float iJvc[R], zc[R], kdec[R];         // centre k: 1 / Jv, Rayleigh profile, decay of D0
};
template <int R>
__device__ __forceinline__ void exp_load(const DevGeom &g, const DevNum &n, int lane, Exp<R> &e) {
    const int nl = g.nlev;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = R * lane + r, kc = min(k, nl - 1), kf = min(k, nl);
        e.Jf[r] = g.sf[kf] * g.sf[kf] * g.Jvf[kf];
        e.iJf[r] = g.isJf[kf];
        e.isf[r] = g.isf[kf];
        e.iJvf[r] = g.iJvf[kf];
        e.iJvc[r] = g.iJvc[kc];
        e.zc[r] = g.zeta_c[kc];
        e.kdec[r] = n.vdiff && n.vdk == 0 && g.kdec ? g.kdec[kc] : 1.0f;
    }
}

// the column's Coriolis parameters and diffusivity
struct Cor {
    float f3, f12a, f12b, D0;
};

// remaining_tendency! of a column (k_explicit without horizontal terms): the
// tendencies of u_1, u_2, rho e_tot and u_3 (rho's is zero)
template <int R>
__device__ __forceinline__ void explicit_column(const Lev<R> &t, const Exp<R> &e, const Met1 &m, const Cor &f,
                                                const DevNum &n, const float (&rho)[R], const float (&u1)[R],
                                                const float (&u2)[R], const float (&rhoe)[R], const float (&u3)[R],
                                                float (&d1)[R], float (&d2)[R], float (&de)[R], float (&d3)[R]) {
    float u3p[R], c1[R], c2[R], Kh[R], Kv[R], sd[R], iK[R], irJ[R];
    next<R>(u3, u3p);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float w1 = t.upF[r] ? u3p[r] : 0.0f;
        c1[r] = t.is2[r] * (m.gu11 * u1[r] + m.gu12 * u2[r]);
        c2[r] = t.is2[r] * (m.gu12 * u1[r] + m.gu22 * u2[r]);
        Kh[r] = 0.5f * (u1[r] * c1[r] + u2[r] * c2[r]);
        Kv[r] = 0.25f * (u3[r] * t.g0[r] * u3[r] + w1 * t.gp[r] * w1);
        const float J = m.Jh * t.sJ[r], a3 = f.f3 * e.iJvc[r];
        irJ[r] = ca_rcp(rho[r] * J);
        d1[r] = J * (a3 * c2[r]);
        d2[r] = -J * (a3 * c1[r]);
        if (n.rayleigh && n.alpha_uh != 0.0f) {
            const float beta = n.alpha_uh * e.zc[r];
            d1[r] -= beta * u1[r];
            d2[r] -= beta * u2[r];
        }
        sd[r] = iK[r] = 0.0f;
    }
    if (n.vdiff) {
        const float spd0 = n.vdk == 1 ? pcr::lane0(sqrtf(2.0f * Kh[0])) : 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double et = (double)rhoe[r] * ca_drcp((double)rho[r]);
            const double Td = temperature(n, et, Kh[r] + Kv[r], t.Phid[r]);
            sd[r] = n.cp_d * ((float)Td - n.T_0) + t.Phic[r];
            float K = f.D0 * e.kdec[r];
            if (n.vdk == 1) {  // ca_Kc
                const float p = (float)((double)rho[r] * n.dR_d * Td), x = (85000.0f - p) * 1.0e-4f;
                K = n.CE * spd0 * n.za * (p > 85000.0f ? 1.0f : expf(-(x * x)));
            }
            iK[r] = 1.0f / fmaxf(K, 1.1920929e-07f);
        }
    }
    float ra[R], u1a[R], u2a[R], c1a[R], c2a[R], Kha[R], Kva[R], sda[R], iKa[R];
    prev<R>(rho, ra);
    prev<R>(u1, u1a);
    prev<R>(u2, u2a);
    prev<R>(c1, c1a);
    prev<R>(c2, c2a);
    prev<R>(Kh, Kha);
    prev<R>(Kv, Kva);
    prev<R>(sd, sda);
    prev<R>(iK, iKa);
    float G1[R], G2[R], Fs[R], F1[R], F2[R], G1p[R], G2p[R], Fsp[R], F1p[R], F2p[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        G1[r] = G2[r] = Fs[r] = F1[r] = F2[r] = d3[r] = 0.0f;
        if (t.intF[r]) {
            const float Jf = m.Jh * e.Jf[r], iJf = m.iJh * e.iJf[r];
            const float w1 = u1[r] - u1a[r], w2 = u2[r] - u2a[r];
            const float A1 = f.f12a * e.isf[r] - w2 * iJf, A2 = f.f12b * e.isf[r] + w1 * iJf;
            const float b3 = 0.5f * (ra[r] * t.sJm[r] + rho[r] * t.sJ[r]) * m.Jh * (u3[r] * t.g0[r]);
            G1[r] = Jf * (A2 * b3);
            G2[r] = -Jf * (A1 * b3);
            const float i1 = 0.5f * (c1a[r] + c1[r]), i2 = 0.5f * (c2a[r] + c2[r]);
            d3[r] = -(Jf * (A1 * i2 - A2 * i1) + ((Kh[r] - Kha[r]) + (Kv[r] - Kva[r])));
            if (n.vdiff) {
                const float rK = (0.5f * (ra[r] + rho[r])) * (1.0f / (0.5f * (iKa[r] + iK[r])));
                const float c = -Jf * e.iJvf[r] * e.iJvf[r] * rK;
                Fs[r] = c * (sd[r] - sda[r]);
                F1[r] = c * w1;
                F2[r] = c * w2;
            }
        }
    }
    next<R>(G1, G1p);
    next<R>(G2, G2p);
    next<R>(Fs, Fsp);
    next<R>(F1, F1p);
    next<R>(F2, F2p);
#pragma unroll
    for (int r = 0; r < R; ++r) {  // face nlev: zero (its row may not exist)
        d1[r] -= (0.5f * (G1[r] + (t.upF[r] ? G1p[r] : 0.0f))) * irJ[r];
        d2[r] -= (0.5f * (G2[r] + (t.upF[r] ? G2p[r] : 0.0f))) * irJ[r];
        de[r] = 0.0f;
        if (n.vdiff) {
            const float iJ = m.iJh * t.isJ[r], irho = ca_rcp(rho[r]);
            de[r] = -((t.upF[r] ? Fsp[r] : 0.0f) - Fs[r]) * iJ;
            d1[r] -= ((t.upF[r] ? F1p[r] : 0.0f) - F1[r]) * iJ * irho;
            d2[r] -= ((t.upF[r] ? F2p[r] : 0.0f) - F2[r]) * iJ * irho;
        }
    }
}

}  // namespace cst

template <int R>
__global__ void __launch_bounds__(64) k_column_steps(DevGeom gr, ColumnSet cs, DevNum n, float *__restrict__ Y,
                                                     EnsTab tab, float dt, int nsteps) {
    const int lane = threadIdx.x;
    const int m = cs.members ? cs.order[blockIdx.x] : (int)blockIdx.x;
    const DevGeom &g = cs.members ? cs.members[m] : gr;
    const int col = cs.members ? 0 : m;
    float *base = cs.members ? Y + cs.off[m] : Y + col;
    const int64_t rs = g.ncol, ps = g.nC;
    const int nl = g.nlev;
    cst::Lev<R> t;
    cst::lev_load<R>(g, lane, t);
    cst::Exp<R> e;
    cst::exp_load<R>(g, n, lane, e);
    const cst::Met1 mt = cst::met1_load(g, n, col);
    const cst::Cor f{g.f3n[col], g.f12a[col], g.f12b[col], n.vdiff && n.vdk == 0 ? g.D0_col[col] : 0.0f};
    float rho[R], u1[R], u2[R], rhoe[R], u3[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t q = (int64_t)min(t.k[r], nl - 1) * rs;
        rho[r] = base[q];
        u1[r] = base[ps + q];
        u2[r] = base[2 * ps + q];
        rhoe[r] = base[3 * ps + q];
        u3[r] = t.intF[r] ? base[4 * ps + q] : 0.0f;
    }
    for (int s = 0; s < nsteps; ++s) {
        float E1[3][R], E2[3][R], Ee[3][R], Ew[3][R];  // F_E of stages 0, 1, 2
        float Ir[2][R], Ie[2][R], Iw[2][R];            // F_I of stages 1, 2
        cst::explicit_column<R>(t, e, mt, f, n, rho, u1, u2, rhoe, u3, E1[0], E2[0], Ee[0], Ew[0]);
#pragma unroll
        for (int i = 1; i < 4; ++i) {
            float vr[R], v1[R], v2[R], ve[R], vw[R], fr[R], fe[R], fu[R];
            const float dtg = dt * tab.aI[i][i];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float sr = 0.0f, s1 = 0.0f, s2 = 0.0f, se = 0.0f, sw = 0.0f;
#pragma unroll
                for (int j = 0; j < i; ++j) {
                    s1 = fmaf(tab.aE[i][j], E1[j][r], s1);
                    s2 = fmaf(tab.aE[i][j], E2[j][r], s2);
                    se = fmaf(tab.aE[i][j], Ee[j][r], se);
                    sw = fmaf(tab.aE[i][j], Ew[j][r], sw);
                    if (j >= 1) {
                        sr = fmaf(tab.aI[i][j], Ir[j - 1][r], sr);
                        se = fmaf(tab.aI[i][j], Ie[j - 1][r], se);
                        sw = fmaf(tab.aI[i][j], Iw[j - 1][r], sw);
                    }
                }
                vr[r] = fmaf(dt, sr, rho[r]);
                v1[r] = fmaf(dt, s1, u1[r]);
                v2[r] = fmaf(dt, s2, u2[r]);
                ve[r] = fmaf(dt, se, rhoe[r]);
                vw[r] = t.intF[r] ? fmaf(dt, sw, u3[r]) : 0.0f;
            }
            cst::newton<R, 64, false>(t, mt, n, nl, dtg, 1.0f / dtg, vr, v1, v2, ve, vw, fr, fe, fu);
            float d1[R], d2[R], de[R], dw[R];
            cst::explicit_column<R>(t, e, mt, f, n, vr, v1, v2, ve, vw, d1, d2, de, dw);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (i < 3) {
                    E1[i][r] = d1[r];
                    E2[i][r] = d2[r];
                    Ee[i][r] = de[r];
                    Ew[i][r] = dw[r];
                    Ir[i - 1][r] = fr[r];
                    Ie[i - 1][r] = fe[r];
                    Iw[i - 1][r] = fu[r];
                } else {  // u + dt sum_j b_j (F_E,j + F_I,j), b_0 = 0
                    const float b1 = tab.b[1], b2 = tab.b[2], b3 = tab.b[3];
                    rho[r] = fmaf(dt, fmaf(b3, fr[r], fmaf(b2, Ir[1][r], b1 * Ir[0][r])), rho[r]);
                    u1[r] = fmaf(dt, fmaf(b3, d1[r], fmaf(b2, E1[2][r], b1 * E1[1][r])), u1[r]);
                    u2[r] = fmaf(dt, fmaf(b3, d2[r], fmaf(b2, E2[2][r], b1 * E2[1][r])), u2[r]);
                    rhoe[r] = fmaf(dt, fmaf(b3, de[r] + fe[r], fmaf(b2, Ee[2][r] + Ie[1][r], b1 * (Ee[1][r] + Ie[0][r]))),
                                   rhoe[r]);
                    u3[r] = t.intF[r] ? fmaf(dt,
                                             fmaf(b3, dw[r] + fu[r],
                                                  fmaf(b2, Ew[2][r] + Iw[1][r], b1 * (Ew[1][r] + Iw[0][r]))),
                                             u3[r])
                                      : 0.0f;
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (t.hasC[r]) {
            const int64_t q = (int64_t)t.k[r] * rs;
            base[q] = rho[r];
            base[ps + q] = u1[r];
            base[2 * ps + q] = u2[r];
            base[3 * ps + q] = rhoe[r];
            base[4 * ps + q] = u3[r];
        }
    if (lane == 0) base[4 * ps + (int64_t)nl * rs] = 0.0f;
}

template __global__ void k_column_steps<1>(DevGeom, ColumnSet, DevNum, float *, EnsTab, float, int);
template __global__ void k_column_steps<2>(DevGeom, ColumnSet, DevNum, float *, EnsTab, float, int);
