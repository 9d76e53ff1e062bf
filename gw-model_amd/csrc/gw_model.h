// gw_model.h -- the Greenstein-Winslow global model on the device (and host):
// derived constants, the per-step constant tables the SSA reads, and the
// explicit-Euler global ODE step. Every expression keeps the reference's
// operation order so that results are bit-identical to the CPU oracle.
#pragma once

#include "gw_math.h"
#include "../../include/gw_capi.h"

namespace gw {

constexpr double kFaraday = 96.5;   // src/includes/common.hpp:9
constexpr double kGasConst = 8.314; // src/includes/common.hpp:10

GW_HD double sq(double x) { return x * x; }
GW_HD double cube(double x) { return x * x * x; }

// Derived constants of GW::Constants (src/includes/GW_utils.tpp:67-116).
struct CellConsts {
    double RT_F, F_RT, CRU_factor, CSA_FVcyto, VSS_Vcyto, Vcyto_VNSR, VJSR_VNSR;
    double gamma0a, gamma0a2, gamma0a3, gamma0a4, binv, omega_b, omega_b2, omega_b3, omega_b4;
    double BSR_const, BSL_const, VSS_VJSR, CSQN_const, JLCC_const, Cao_scaled;
    double Nao3, INaCa_const, sigma, INaK_const, sqrtKo, PKv14_Csc, Ito2_const, IK1_const, ICaL_const, CMDN_const;
};

GW_HD void cell_consts_init(CellConsts &c, const gw_params_t &p, int nCRU)
{
    c.RT_F = kGasConst * p.T / kFaraday;
    c.F_RT = 1.0 / c.RT_F;
    c.CRU_factor = static_cast<double>(p.NCaRU) / static_cast<double>(nCRU);
    c.CSA_FVcyto = p.CSA / (1000 * p.Vcyto * kFaraday);
    c.VSS_Vcyto = p.VSS / p.Vcyto;
    c.Vcyto_VNSR = p.Vcyto / p.VNSR;
    c.VJSR_VNSR = p.VJSR / p.VNSR;
    c.gamma0a = p.gamma0 * p.a;
    c.gamma0a2 = c.gamma0a * p.a;
    c.gamma0a3 = c.gamma0a2 * p.a;
    c.gamma0a4 = c.gamma0a3 * p.a;
    c.binv = 1.0 / p.b;
    c.omega_b = p.omega * c.binv;
    c.omega_b2 = c.omega_b * c.binv;
    c.omega_b3 = c.omega_b2 * c.binv;
    c.omega_b4 = c.omega_b3 * c.binv;
    c.BSR_const = p.KBSR * p.BSRT;
    c.BSL_const = p.KBSL * p.BSLT;
    c.VSS_VJSR = p.VSS / p.VJSR;
    c.CSQN_const = p.KCSQN * p.CSQNT;
    c.JLCC_const = 2.0e6 * p.PCaL / p.VSS;
    c.Cao_scaled = 0.341 * p.Cao;
    c.Nao3 = p.Nao * p.Nao * p.Nao;
    c.INaCa_const = 5000.0 * p.kNaCa / ((p.KmNa * p.KmNa * p.KmNa + p.Nao * p.Nao * p.Nao) * (p.KmCa + p.Cao));
    c.sigma = (gw::exp(p.Nao / 67.3) - 1.0) / 7.0;
    c.INaK_const = p.INaKmax * p.Ko / (p.Ko + p.KmKo);
    c.sqrtKo = __builtin_sqrt(p.Ko);
    c.PKv14_Csc = p.PKv14 / p.Csc;
    c.Ito2_const = 1.0e9 * p.Pto2 * kFaraday * c.CRU_factor / p.CSA;
    c.IK1_const = p.Ko / (p.Ko + p.KmK1);
    c.ICaL_const = -1000.0 * (2.0 * kFaraday * p.VSS) * c.CRU_factor / p.CSA;
    c.CMDN_const = p.KCMDN * p.CMDNT;
}

// Independent quotients, one after another. The close forms them one per lane
// of a wave instead.
struct Serial {
    template <int N>
    GW_HD void operator()(const double (&num)[N], const double (&den)[N], double (&q)[N]) const
    {
        for (int i = 0; i < N; ++i) q[i] = num[i] / den[i];
    }
};

// Constants the SSA reads during one step (frozen inside GW_model::SSA,
// src/includes/GW.tpp:214-233). The LCC propensities of a subunit in state s
// are tabulated so that (r0 + r1) + r2 = lccP[s] + lccQ[s] * CaSS bit for bit;
// R0, R1 hold r0, r1 with the CaSS-proportional slot set to zero (r2 is
// never needed on its own: the transition scan stops before comparing it).
template <class R>
struct LccTableT {
    R P[13], Q[13], R0[13], R1[13];
};
using LccTable = LccTableT<double>;
using LccTableF = LccTableT<float>;

struct StepConsts {
    double Cai, CaNSR;
    double inact0, inact1;   // (y == 0) ? yinf/tau : (1 - yinf)/tau  (GW_utils.hpp:381)
    double JLCC_mult, JLCC_exp;
    uint32_t step_lo;
    uint32_t _pad;
    LccTable lcc;            // read per lane (indexed by the LCC state)
};

// GW::alphaLCC .. tauLCC (GW_utils.hpp:365-375)
// The exponentials of the per-step constants: alpha, beta, y_inf and tau of
// the LCC (GW_utils.hpp:365-375, as exp(arg)), then exp(-V F/RT).
enum ScSlot : int { SC_AL, SC_BE, SC_YINF, SC_TAU, SC_EXPM, SC_N };

GW_HD double sc_arg(int slot, double V, double F_RT)
{
    if (slot == SC_EXPM) return -(V * F_RT);
    const double t = V + (slot <= SC_BE ? -35.0 : slot == SC_YINF ? 12.5 : 30.0);
    const double c = slot == SC_AL ? 0.012 : slot == SC_BE ? -0.05 : slot == SC_YINF ? 5.0 : 12.0;
    return slot <= SC_BE ? c * t : t / c;
}

// Per-step constants of GW_model::SSA (GW.tpp:216-221) from the exponentials
// X[SC_*] of sc_arg's arguments, without the LCC rate table. At V == 0 the multiplier
// takes its analytic limit JLCC_const / 2 instead of 0/0.
template <class Quot>
GW_HD void step_consts_scalars(StepConsts &k, const CellConsts &c, double V, const double *X, double Cai, double CaNSR,
                               uint32_t step_lo, Quot &&quot)
{
    const double num[3] = {0.4, 340.0, 1.0}, den[3] = {1.0 + X[SC_YINF], 1.0 + X[SC_TAU], X[SC_EXPM]};
    double q[3], q2[3];
    quot(num, den, q);
    const double yinf = q[0] + 0.6;
    const double tau = q[1] + 60.0;
    k.Cai = Cai;
    k.CaNSR = CaNSR;
    k.JLCC_exp = sq(q[2]);
    const double num2[3] = {yinf, 1.0 - yinf, c.JLCC_const * V * c.F_RT}, den2[3] = {tau, tau, k.JLCC_exp - 1};
    quot(num2, den2, q2);
    k.inact0 = q2[0];
    k.inact1 = q2[1];
    k.JLCC_mult = (V == 0.0) ? c.JLCC_const / 2.0 : q2[2];
    k.step_lo = step_lo;
    k._pad = 0;
}

struct LccRow {
    double P, Q, R0, R1;
};

// Row s of the LCC rate table of update_LCC_rates (GW_utils.tpp:118-186):
// r0, r1, r2 of state s, the CaSS-proportional rate's coefficient in Q.
// State 1 carries its CaSS term in r1: (r0 + g0 CaSS) + 0 == P + Q CaSS with
// P = r0; states 2..5 carry it in r2: (r0 + r1) + Q CaSS; the others
// (r0 + r1) + r2 + 0.
GW_HD LccRow lcc_row(int s, const gw_params_t &p, const CellConsts &c, const double *X)
{
    // without a switch: on the device thirteen lanes form a row each
    const double al = 2.0 * X[SC_AL];
    const double be = 0.0882 * X[SC_BE];
    const double k = static_cast<double>(s);
    double r0 = 0, r1 = 0, r2 = 0, q = 0;
    if (s >= 1 && s <= 5) {
        r0 = s == 1 ? 4 * al : (k - 1) * be;                       // 4 al, be, 2 be, 3 be, 4 be
        r1 = s == 1 ? 0.0 : s == 5 ? p.f : (5 - k) * al;           // -, 3 al, 2 al, al, f
        q = s == 1 ? p.gamma0 : s == 2 ? c.gamma0a : s == 3 ? c.gamma0a2 : s == 4 ? c.gamma0a3 : c.gamma0a4;
    } else if (s >= 7 && s <= 11) {
        r0 = s == 7 ? p.omega : s == 8 ? c.omega_b : s == 9 ? c.omega_b2 : s == 10 ? c.omega_b3 : c.omega_b4;
        r1 = s == 7 ? 4 * al * p.a : (k - 7) * be * c.binv;        // 4 al a, be/b, 2 be/b, 3 be/b, 4 be/b
        r2 = s == 7 ? 0.0 : s == 11 ? p.f1 : (11 - k) * al * p.a;  // -, 3 al a, 2 al a, al a, f1
    } else if (s > 0) {
        r0 = s == 6 ? p.g : p.g1;
    }
    LccRow w;
    w.R0 = r0;
    w.R1 = r1;
    w.Q = q;
    if (s == 1) w.P = r0;
    else if (s >= 2 && s <= 5) w.P = r0 + r1;
    else w.P = r0 + r1 + r2;
    return w;
}

template <class R>
GW_HD void lcc_row_store(LccTableT<R> &t, int s, const LccRow &w)
{
    t.P[s] = static_cast<R>(w.P);
    t.Q[s] = static_cast<R>(w.Q);
    t.R0[s] = static_cast<R>(w.R0);
    t.R1[s] = static_cast<R>(w.R1);
}

// Per-step constants of GW_model::SSA and the LCC rate table, from the
// exponentials X[SC_*] of sc_arg's arguments.
GW_HD void step_consts_x(StepConsts &k, const gw_params_t &p, const CellConsts &c, double V, const double *X,
                         double Cai, double CaNSR, uint32_t step_lo)
{
    step_consts_scalars(k, c, V, X, Cai, CaNSR, step_lo, Serial());
    for (int s = 0; s < 13; ++s) lcc_row_store(k.lcc, s, lcc_row(s, p, c, X));
}

// step_consts_x with its exponentials evaluated in turn (exp(-V F/RT) given).
GW_HD void step_consts(StepConsts &k, const gw_params_t &p, const CellConsts &c, double V, double expmVF_RT,
                       double Cai, double CaNSR, uint32_t step_lo)
{
    double X[SC_N];
    for (int i = 0; i < SC_EXPM; ++i) X[i] = gw::exp(sc_arg(i, V, c.F_RT));
    X[SC_EXPM] = expmVF_RT;
    step_consts_x(k, p, c, V, X, Cai, CaNSR, step_lo);
}

// The SSA constants of a step rounded to FP32, for the FP32-local SSA.
struct StepConstsF {
    double Cai_d, CaNSR_d;   // kept in FP64: they enter the SSA only through differences
    float Cai, CaNSR;
    float inact0, inact1;
    float JLCC_mult, JLCC_exp;
    LccTableF lcc;
};

GW_HD void step_consts_f32_scalars(StepConstsF &f, const StepConsts &k)
{
    f.Cai_d = k.Cai;
    f.CaNSR_d = k.CaNSR;
    f.Cai = static_cast<float>(k.Cai);
    f.CaNSR = static_cast<float>(k.CaNSR);
    f.inact0 = static_cast<float>(k.inact0);
    f.inact1 = static_cast<float>(k.inact1);
    f.JLCC_mult = static_cast<float>(k.JLCC_mult);
    f.JLCC_exp = static_cast<float>(k.JLCC_exp);
}

GW_HD void step_consts_f32(StepConstsF &f, const StepConsts &k)
{
    step_consts_f32_scalars(f, k);
    for (int s = 0; s < 13; ++s) lcc_row_store(f.lcc, s, LccRow{k.lcc.P[s], k.lcc.Q[s], k.lcc.R0[s], k.lcc.R1[s]});
}

// ---------------------------------------------------------------------------
// Global ODE: update_QKr / update_QKv (GW.tpp:25-44, 64-123) and the
// derivatives of update_V_and_concentration_derivatives, update_gate_derivatives,
// update_Kr/Kv_derivatives (GW.tpp:126-212). dg receives dt * f(state) as the
// reference forms it. Returns GW_OK or GW_E_NONPOSITIVE_CONC.
// ---------------------------------------------------------------------------
struct FluxSums {
    double JLCC, Jxfer, Jtr, ClCh;
};

// The exponentials, logarithms and powers of global_derivatives whose
// arguments depend on the state alone, in a fixed slot order. gd_args forms
// each argument exactly as the formula that uses it; gd_finish reads the
// values X[slot]. The values may come from one evaluation after another
// (global_derivatives) or from many lanes at once: the same function of the
// same argument either way, so the derivatives are the same bits.
enum GdSlot : int {
    GD_EXPM,                                  // exp(-VF_RT)
    GD_NACA, GD_NAK, GD_KR_R, GD_KP,          // INaCa, INaK, IKr rectification, IKp
    GD_AM, GD_BM, GD_AH, GD_BH1, GD_BH2, GD_BH3, GD_AJ1, GD_AJ2, GD_AJ3,
    GD_BJ1, GD_BJ2, GD_BJ3, GD_BJ4, GD_XKS, GD_TXKS1, GD_TXKS2,   // gates (common.hpp:175-218)
    GD_KR0, GD_KR1, GD_KR2, GD_KR3, GD_KR4, GD_KR5, GD_KR6,       // update_QKr (GW.tpp:25-44)
    GD_KV0, GD_KV1, GD_KV2, GD_KV3, GD_KV4, GD_KV5, GD_KV6, GD_KV7,   // update_QKv (GW.tpp:64-123)
    GD_LOG0,                                  // logarithms from here
    GD_LNA = GD_LOG0, GD_LK, GD_LKS,          // log(Nao/Nai), log(Ko/Ki), the IKs reversal
    GD_POW0,                                  // powers from here (exponent py[slot - GD_POW0])
    GD_PNAK = GD_POW0, GD_PF, GD_PR,          // INaK, Jup forward and reverse
    GD_N,
    GD_IK1 = GD_N,                            // exp(1.5 (V - EK) F/RT), IK1: its argument needs X[GD_LK]
    GD_X                                      // values in all
};

GW_HD double gd_eval(int slot, double arg, double y)
{
    return slot < GD_LOG0 ? gw::exp(arg) : slot < GD_POW0 ? gw::log(arg) : gw::pow(arg, y);
}

GW_HD void gd_args(const gw_params_t &p, const gw_globals_t &g, double VF_RT, double *arg, double *py)
{
    const double V = g.V;
    arg[GD_EXPM] = -VF_RT;
    arg[GD_NACA] = p.eta * VF_RT;
    arg[GD_NAK] = -0.1 * VF_RT;
    arg[GD_KR_R] = 0.0446 * V;
    arg[GD_KP] = (7.488 - V) / 5.98;
    arg[GD_AM] = -0.1 * (V + 47.13);
    arg[GD_BM] = -V / 11.0;
    arg[GD_AH] = -(V + 80.0) / 6.8;
    arg[GD_BH1] = -(V + 10.66) / 11.1;
    arg[GD_BH2] = 0.079 * V;
    arg[GD_BH3] = 0.35 * V;
    arg[GD_AJ1] = 0.2444 * V;
    arg[GD_AJ2] = -0.04391 * V;
    arg[GD_AJ3] = 0.311 * (V + 79.23);
    arg[GD_BJ1] = -2.535e-7 * V;
    arg[GD_BJ2] = -0.1 * (V + 32.0);
    arg[GD_BJ3] = -0.01052 * V;
    arg[GD_BJ4] = -0.1378 * (V + 40.14);
    arg[GD_XKS] = -(V - 24.7) / 13.6;
    arg[GD_TXKS1] = -0.148 * (V - 10.0);
    arg[GD_TXKS2] = 0.0687 * (V - 10.0);
    arg[GD_KR0] = 0.0272 * V;
    arg[GD_KR1] = -0.0431 * V;
    arg[GD_KR2] = 0.0262 * V;
    arg[GD_KR3] = 2.71e-6 * V;
    arg[GD_KR4] = -0.0269 * V;
    arg[GD_KR5] = 0.0120 * V;
    arg[GD_KR6] = -0.0443 * V;
    arg[GD_KV0] = p.aaKv14 * V;
    arg[GD_KV1] = p.aaKv43 * V;
    arg[GD_KV2] = -p.aiKv14 * V;
    arg[GD_KV3] = -p.aiKv43 * V;
    arg[GD_KV4] = -p.baKv14 * V;
    arg[GD_KV5] = -p.baKv43 * V;
    arg[GD_KV6] = p.biKv14 * V;
    arg[GD_KV7] = p.biKv43 * V;
    arg[GD_LNA] = p.Nao / g.Nai;
    arg[GD_LK] = p.Ko / g.Ki;
    arg[GD_LKS] = (p.Ko + 0.01833 * p.Nao) / (g.Ki + 0.01833 * g.Nai);
    arg[GD_PNAK] = p.KmNai / g.Nai;
    py[0] = 1.5;
    arg[GD_PF] = g.Cai / p.Kmf;
    py[1] = p.Hf;
    arg[GD_PR] = g.CaNSR / p.Kmr;
    py[2] = p.Hr;
}

// One Kv chain (Kv1.4 or Kv4.3): generator entries of update_QKv (GW.tpp:64-123)
// and the derivatives of update_Kv_derivatives (GW.tpp:135-160), in registers.
GW_HD void kv_chain(double aa, double ai, double ba, double bi, double f1, double f2, double f3, double f4,
                    double b1, double b2, double b3, double b4, const double y[10], double dt, double d[10])
{
    const double q01 = 4 * aa, q05 = bi, q00 = -(q01 + q05);
    const double q10 = ba, q12 = 3 * aa, q16 = f1 * bi, q11 = -(q10 + q12 + q16);
    const double q21 = 2 * ba, q23 = 2 * aa, q27 = f2 * bi, q22 = -(q21 + q23 + q27);
    const double q32 = 3 * ba, q34 = aa, q38 = f3 * bi, q33 = -(q32 + q34 + q38);
    const double q43 = 4 * ba, q49 = f4 * bi, q44 = -(q43 + q49);
    const double q56 = 4 * aa * b1, q50 = ai, q55 = -(q56 + q50);
    const double q65 = ba / f1, q67 = 3 * aa * b2 / b1, q61 = ai / b1, q66 = -(q65 + q67 + q61);
    const double q76 = 2 * ba * f1 / f2, q78 = 2 * aa * b3 / b2, q72 = ai / b2, q77 = -(q76 + q78 + q72);
    const double q87 = 3 * ba * f2 / f3, q89 = aa * b4 / b3, q83 = ai / b3, q88 = -(q87 + q89 + q83);
    const double q98 = 4 * ba * f3 / f4, q94 = ai / b4, q99 = -(q98 + q94);
    d[0] = dt * (q10 * y[1] + q50 * y[5] + q00 * y[0]);
    d[1] = dt * (q01 * y[0] + q21 * y[2] + q61 * y[6] + q11 * y[1]);
    d[2] = dt * (q12 * y[1] + q32 * y[3] + q72 * y[7] + q22 * y[2]);
    d[3] = dt * (q23 * y[2] + q43 * y[4] + q83 * y[8] + q33 * y[3]);
    d[4] = dt * (q34 * y[3] + q94 * y[9] + q44 * y[4]);
    d[5] = dt * (q65 * y[6] + q05 * y[0] + q55 * y[5]);
    d[6] = dt * (q56 * y[5] + q76 * y[7] + q16 * y[1] + q66 * y[6]);
    d[7] = dt * (q67 * y[6] + q87 * y[8] + q27 * y[2] + q77 * y[7]);
    d[8] = dt * (q78 * y[7] + q98 * y[9] + q38 * y[3] + q88 * y[8]);
    d[9] = dt * (q89 * y[8] + q49 * y[4] + q99 * y[9]);
}

// Currents of one step, in the order of GW::Currents (GW.hpp:25-42).
struct Currents {
    double INa, INab, INaCa, INaK, IKr, IKs, Ito1, Ito2, IK1, IKp, ICaL, ICab, IpCa, Jup, Jtr_tot, Jxfer_tot;
};

// The same arguments one slot per lane: slot s < GD_LOG0 is (x + d) * c or
// (x + d) / c of x = V or VF_RT, with c a number or a parameter times one;
// negated and reordered forms of gd_args round alike.
enum GdArgSrc : int32_t { GA_VF = 1, GA_DIV = 2, GA_PARAM = 4 };
struct GdArg {
    double d, c;
    int32_t src, off;   // off: the parameter's word in gw_params_t
};
#define GW_GA_PARAM_(field, c, src) {0.0, c, GA_PARAM | (src), static_cast<int32_t>(offsetof(gw_params_t, field) / 8)}
__device__ __constant__ const GdArg kGdArg[GD_LOG0] = {
    {0.0, -1.0, GA_VF, 0},                                                            // EXPM
    GW_GA_PARAM_(eta, 1.0, GA_VF), {0.0, -0.1, GA_VF, 0},                             // NACA, NAK
    {0.0, 0.0446, 0, 0}, {-7.488, -5.98, GA_DIV, 0},                                  // KR_R, KP
    {47.13, -0.1, 0, 0}, {0.0, -11.0, GA_DIV, 0},                                     // AM, BM
    {80.0, -6.8, GA_DIV, 0}, {10.66, -11.1, GA_DIV, 0}, {0.0, 0.079, 0, 0}, {0.0, 0.35, 0, 0},   // AH, BH1..3
    {0.0, 0.2444, 0, 0}, {0.0, -0.04391, 0, 0}, {79.23, 0.311, 0, 0},                 // AJ1..3
    {0.0, -2.535e-7, 0, 0}, {32.0, -0.1, 0, 0}, {0.0, -0.01052, 0, 0}, {40.14, -0.1378, 0, 0},   // BJ1..4
    {-24.7, -13.6, GA_DIV, 0}, {-10.0, -0.148, 0, 0}, {-10.0, 0.0687, 0, 0},          // XKS, TXKS1..2
    {0.0, 0.0272, 0, 0}, {0.0, -0.0431, 0, 0}, {0.0, 0.0262, 0, 0}, {0.0, 2.71e-6, 0, 0},        // KR0..3
    {0.0, -0.0269, 0, 0}, {0.0, 0.0120, 0, 0}, {0.0, -0.0443, 0, 0},                  // KR4..6
    GW_GA_PARAM_(aaKv14, 1.0, 0), GW_GA_PARAM_(aaKv43, 1.0, 0), GW_GA_PARAM_(aiKv14, -1.0, 0), GW_GA_PARAM_(aiKv43, -1.0, 0),
    GW_GA_PARAM_(baKv14, -1.0, 0), GW_GA_PARAM_(baKv43, -1.0, 0), GW_GA_PARAM_(biKv14, 1.0, 0), GW_GA_PARAM_(biKv43, 1.0, 0)};
#undef GW_GA_PARAM_

__device__ __forceinline__ GdArg gd_arg_row(int slot) { return kGdArg[slot]; }
__device__ __forceinline__ double gd_arg_value(const GdArg &r, const gw_params_t &p, double V, double VF_RT)
{
    const double c = (r.src & GA_PARAM) ? r.c * reinterpret_cast<const double *>(&p)[r.off] : r.c;
    const double t = ((r.src & GA_VF) ? VF_RT : V) + r.d;
    return (r.src & GA_DIV) ? t / c : t * c;
}

// The argument of slot s >= GD_LOG0 and, for a power, its exponent (else 0).
// Every value is read before one is chosen: a choice between reads would be a branch.
GW_HD double gd_log_arg(int slot, const gw_params_t &p, const gw_globals_t &g, double &y)
{
    const double Nao = p.Nao, Ko = p.Ko, KmNai = p.KmNai, Kmf = p.Kmf, Kmr = p.Kmr, Hf = p.Hf, Hr = p.Hr;
    const double Nai = g.Nai, Ki = g.Ki, Cai = g.Cai, CaNSR = g.CaNSR;
    const double Kso = Ko + 0.01833 * Nao, Ksi = Ki + 0.01833 * Nai;
    y = slot == GD_PNAK ? 1.5 : slot == GD_PF ? Hf : slot == GD_PR ? Hr : 0.0;
    const double num = slot == GD_LNA ? Nao : slot == GD_LK ? Ko : slot == GD_LKS ? Kso : slot == GD_PNAK ? KmNai
                     : slot == GD_PF ? Cai : CaNSR;
    const double den = slot == GD_LNA ? Nai : slot == GD_LK ? Ki : slot == GD_LKS ? Ksi : slot == GD_PNAK ? Nai
                     : slot == GD_PF ? Kmf : Kmr;
    return num / den;
}

// The Kv chains one value per lane: a generator entry is m r u / v of one of
// the chain's four rates r and factors u, v (kv_chain's expressions: a factor
// left out is 1, which changes no bit), a derivative is two or three inflows
// and the diagonal, in kv_chain's order.
namespace kv {
constexpr int kEntries = 26;
// parameters of a chain, as words from its alphaa0: the rates' scales, then f1..f4, b1..b4
enum Off : uint32_t { AA = 0, BA = 2, AI = 4, BI = 6, F1 = 8, F2, F3, F4, B1, B2, B3, B4, ONE = 31 };
static_assert(offsetof(gw_params_t, b4Kv14) - offsetof(gw_params_t, alphaa0Kv14) == 15 * sizeof(double) &&
                  offsetof(gw_params_t, f1Kv14) - offsetof(gw_params_t, alphaa0Kv14) == F1 * sizeof(double) &&
                  offsetof(gw_params_t, b4Kv43) - offsetof(gw_params_t, alphaa0Kv43) == 15 * sizeof(double) &&
                  offsetof(gw_params_t, f1Kv43) - offsetof(gw_params_t, alphaa0Kv43) == F1 * sizeof(double) &&
                  offsetof(gw_params_t, betai0Kv14) - offsetof(gw_params_t, alphaa0Kv14) == BI * sizeof(double),
              "both chains' parameters lie in the same order");
constexpr uint32_t ent(uint32_t m, uint32_t r, uint32_t u = ONE, uint32_t v = ONE) { return m | r << 3 | u << 6 | v << 11; }
__device__ __constant__ const uint32_t kEntry[kEntries] = {
    ent(4, AA), ent(1, BI),                                   // 0: q01 q05
    ent(1, BA), ent(3, AA), ent(1, BI, F1),                   // 2: q10 q12 q16
    ent(2, BA), ent(2, AA), ent(1, BI, F2),                   // 5: q21 q23 q27
    ent(3, BA), ent(1, AA), ent(1, BI, F3),                   // 8: q32 q34 q38
    ent(4, BA), ent(1, BI, F4),                               // 11: q43 q49
    ent(4, AA, B1), ent(1, AI),                               // 13: q56 q50
    ent(1, BA, ONE, F1), ent(3, AA, B2, B1), ent(1, AI, ONE, B1),   // 15: q65 q67 q61
    ent(2, BA, F1, F2), ent(2, AA, B3, B2), ent(1, AI, ONE, B2),    // 18: q76 q78 q72
    ent(3, BA, F2, F3), ent(1, AA, B4, B3), ent(1, AI, ONE, B3),    // 21: q87 q89 q83
    ent(4, BA, F3, F4), ent(1, AI, ONE, B4)};                 // 24: q98 q94
// Row i: inflow k as (entry, from state); the outgoing entries are consecutive from `out`.
struct Row {
    uint8_t e[3], s[3], nin, out, nout;
};
__device__ __constant__ const Row kRow[10] = {
    {{2, 14, 0}, {1, 5, 0}, 2, 0, 2},   {{0, 5, 17}, {0, 2, 6}, 3, 2, 3},  {{3, 8, 20}, {1, 3, 7}, 3, 5, 3},
    {{6, 11, 23}, {2, 4, 8}, 3, 8, 3},  {{9, 25, 0}, {3, 9, 0}, 2, 11, 2}, {{15, 1, 0}, {6, 0, 0}, 2, 13, 2},
    {{13, 18, 4}, {5, 7, 1}, 3, 15, 3}, {{16, 21, 7}, {6, 8, 2}, 3, 18, 3}, {{19, 24, 10}, {7, 9, 3}, 3, 21, 3},
    {{22, 12, 0}, {8, 4, 0}, 2, 24, 2}};

__device__ __forceinline__ uint32_t entry(int k) { return kEntry[k]; }
__device__ __forceinline__ Row row(int i) { return kRow[i]; }
__device__ __forceinline__ double entry_value(uint32_t e, const gw_params_t &p, const double *X, int chain)
{
    const double *P = chain == 0 ? &p.alphaa0Kv14 : &p.alphaa0Kv43;
    const uint32_t r = (e >> 3) & 7, u = (e >> 6) & 31, v = (e >> 11) & 31;
    // X[GD_KV0 ..]: aa, ai, ba, bi of Kv1.4 and Kv4.3 in turn
    const int slot = GD_KV0 + (r == AA ? 0 : r == AI ? 2 : r == BA ? 4 : 6) + chain;
    const double rate = P[r] * X[slot];
    const double fu = P[u & 15], fv = P[v & 15];
    return static_cast<double>(e & 7) * rate * (u == ONE ? 1.0 : fu) / (v == ONE ? 1.0 : fv);
}
__device__ __forceinline__ double derivative(const Row &r, int i, const double *q, const double *y, double dt)
{
    double out = q[r.out] + q[r.out + 1];
    if (r.nout > 2) out += q[r.out + 2];
    double in = q[r.e[0]] * y[r.s[0]] + q[r.e[1]] * y[r.s[1]];
    if (r.nin > 2) in += q[r.e[2]] * y[r.s[2]];
    return dt * (in + -out * y[i]);
}
}  // namespace kv

// Whether every Nernst argument is positive (the reference exits where one is not, common.hpp:72-75).
GW_HD bool gd_concentrations_ok(const gw_params_t &p, const gw_globals_t &g)
{
    return !(g.Nai <= 0.0 || p.Nao <= 0.0 || g.Ki <= 0.0 || p.Ko <= 0.0);
}

// The potassium reversal potential (common.hpp:70-75) and the argument of X[GD_IK1], from lk = X[GD_LK].
GW_HD double gd_EK(const CellConsts &c, double lk) { return lk * c.RT_F / 1.0; }
GW_HD double gd_ik1_arg(const CellConsts &c, double V, double lk) { return 1.5 * (V - gd_EK(c, lk)) * c.F_RT; }

// The derivatives from the values X[slot], except the Kv chains (gd_chain_kv
// below), in three parts that share only their inputs and gd_combine, which
// joins them. A part gathers its independent quotients and has quot(num, den,
// q) form them: one after another (Serial), or one per lane.
template <class Quot>
GW_HD void gd_k_currents(const gw_params_t &p, const CellConsts &c, const gw_globals_t &g, double VF_RT,
                         const double *X, Currents &cur, Quot &&quot)
{
    const double V = g.V;
    const double e = X[GD_EXPM];
    const double EK = gd_EK(c, X[GD_LK]);
    const double num[4] = {1.0, 1.0, 1., (c.PKv14_Csc) * (kFaraday * VF_RT) * g.Kv14[4]};
    const double den[4] = {1.0 + 1.4945 * X[GD_KR_R], 2.0 + X[GD_IK1], 1. + X[GD_KP], 1 - e};
    double q[4];
    quot(num, den, q);
    const double RKr = q[0], K1inf = q[1], Kp = q[2];
    cur.IKr = p.GKr * c.sqrtKo * RKr * g.Kr[3] * (V - EK) * 0.5;               // GW_utils.hpp:273-279
    {   // GW_utils.hpp:282-291
        const double EKs = X[GD_LKS] * c.RT_F;
        cur.IKs = p.GKs * sq(g.xKs) * (V - EKs);
    }
    // GW_utils.hpp:299-303 with exp_term = exp(-VF/RT) (GW.tpp:185); limit at V == 0
    const double mm = VF_RT == 0.0 ? (c.PKv14_Csc) * kFaraday * g.Kv14[4] : q[3];
    const double IKv14 = mm * ((g.Ki - p.Ko * e) + 0.02 * (g.Nai - p.Nao * e)) * 1.0e9;
    const double IKv43 = p.GKv43 * g.Kv43[4] * (V - EK);                       // GW_utils.hpp:294-297
    cur.Ito1 = IKv14 + IKv43;
    cur.IK1 = p.GK1 * K1inf * c.IK1_const * (V - EK);                          // GW_utils.hpp:306-312
    cur.IKp = p.GKp * Kp * (V - EK);                                           // GW_utils.hpp:315-319
}

// The Na and Ca currents, SERCA uptake, the cytosolic buffering factor and the
// troponin derivatives before the factor dt (GW.tpp:201-202).
template <class Quot>
GW_HD void gd_na_ca_currents(const gw_params_t &p, const CellConsts &c, const gw_globals_t &g, const double *X,
                             Currents &cur, double &beta_cyto, double &dLTRPN, double &dHTRPN, Quot &&quot)
{
    const double V = g.V;
    const double expmVF_RT = X[GD_EXPM];
    const double e1 = X[GD_NACA];                                               // common.hpp:163-168
    const double e2 = e1 * expmVF_RT;
    const double f = X[GD_PF];                                                  // GW_utils.hpp:339-344
    const double r = X[GD_PR];
    const double x = p.KCMDN + g.Cai;                                           // GW_utils.hpp:347-351
    const double num[5] = {c.INaCa_const * (e1 * cube(g.Nai) * p.Cao - e2 * c.Nao3 * g.Cai), 1.0, g.Cai,
                           p.Vmaxf * f - p.Vmaxr * r, c.CMDN_const};
    const double den[5] = {1.0 + p.ksat * e2, 1.0 + 0.1245 * X[GD_NAK] + 0.0365 * c.sigma * expmVF_RT,
                           p.KmpCa + g.Cai, 1.0 + f + r, sq(x)};
    double q[5];
    quot(num, den, q);
    const double num2[2] = {c.INaK_const * q[1], 1.0};                          // common.hpp:121-124, 140-143
    const double den2[2] = {1.0 + X[GD_PNAK], 1.0 + q[4]};
    double q2[2];
    quot(num2, den2, q2);
    const double ENa = X[GD_LNA] * c.RT_F / 1.0;
    const double ECa = X[GD_LK] * c.RT_F / 2.0;                                 // K-based, as GW.tpp:176
    cur.INa = p.GNa * cube(g.m) * g.h * g.j * (V - ENa);                       // common.hpp:89-92
    cur.INab = p.GNab * (V - ENa);                                             // common.hpp:100-101
    cur.INaCa = q[0];
    cur.INaK = q2[0];
    cur.ICab = p.GCab * (V - ECa);
    cur.IpCa = p.IpCamax * q[2];                                                // common.hpp:109-110
    cur.Jup = q[3];
    beta_cyto = q2[1];
    dLTRPN = p.kLTRPNp * g.Cai * (p.LTRPNtot - g.CaLTRPN) - p.kLTRPNm * g.CaLTRPN;
    dHTRPN = p.kHTRPNp * g.Cai * (p.HTRPNtot - g.CaHTRPN) - p.kHTRPNm * g.CaHTRPN;
}

// The gates (m, h, j and xKs, GW.tpp:162-168), the IKr chain, and the currents
// and fluxes formed from the CRU sums. d: the derivatives of the gates and of
// the chain (gw_globals_t order).
template <class Quot>
GW_HD void gd_gates_kr_cru(const gw_params_t &p, const CellConsts &c, const gw_globals_t &g, double VF_RT,
                           const double *X, const FluxSums &S, double dt, double d[9], Currents &cur, Quot &&quot)
{
    const double V = g.V;
    const double expmVF_RT = X[GD_EXPM];
    const bool hi = V >= -40.0;
    const double q23 = 0.0218 * X[GD_KR2], q24 = 1.29e-5 * X[GD_KR3], q32 = 0.0009 * X[GD_KR4];
    const double q34 = 0.0622 * X[GD_KR5], q43 = 0.0059 * X[GD_KR6];
    const double bj = 0.3 * X[GD_BJ1], aj = (-127140.0 * X[GD_AJ1] - 3.474e-5 * X[GD_AJ2]) * (V + 37.78);
    const double bjd = 1.0 + X[GD_BJ2], ajd = 1.0 + X[GD_AJ3];
    const double num[9] = {0.32 * (V + 47.13), 1.0, hi ? bj : aj, 0.1212 * X[GD_BJ3], 1.0, 0.0000719 * (V - 10.0),
                           0.000131 * (V - 10.0), q32 * q43 * q24,
                           S.ClCh * c.Ito2_const * VF_RT * (p.Clcyto * expmVF_RT - p.Clo)};
    const double den[9] = {1.0 - X[GD_AM], 0.13 * (1.0 + X[GD_BH1]), hi ? bjd : ajd, 1.0 + X[GD_BJ4], 1.0 + X[GD_XKS],
                           1.0 - X[GD_TXKS1], X[GD_TXKS2] - 1.0, q23 * q34, expmVF_RT - 1.0};
    double q[9];
    quot(num, den, q);
    // common.hpp:175-218; the limits of 0/0
    const double am = (V == -47.13) ? 3.2 : q[0], bm = 0.08 * X[GD_BM];
    const double ah = hi ? 0.0 : 0.135 * X[GD_AH], bh = hi ? q[1] : 3.56 * X[GD_BH2] + 3.1e5 * X[GD_BH3];
    const double a_j = hi ? 0.0 : q[2], b_j = hi ? q[2] : q[3];
    const double tauXKs_inv = (V == 10.0) ? 0.0000719 / 0.148 + 0.000131 / 0.0687 : q[5] + q[6];
    d[0] = dt * (am * (1.0 - g.m) - bm * g.m);
    d[1] = dt * (ah * (1.0 - g.h) - bh * g.h);
    d[2] = dt * (a_j * (1.0 - g.j) - b_j * g.j);
    d[3] = dt * (q[4] - g.xKs) * tauXKs_inv;
    // update_QKr (GW.tpp:25-44) and update_Kr_derivatives (GW.tpp:126-133)
    const double *x = g.Kr;
    const double q12 = p.Kf, q21 = p.Kb;   // initialise_QKr (GW.hpp:75)
    const double q01 = 0.0069 * X[GD_KR0];
    const double q00 = -q01;
    const double q10 = 0.0227 * X[GD_KR1];
    const double q11 = -(q10 + q12);
    const double q22 = -(q21 + q23 + q24);
    const double q33 = -(q32 + q34);
    const double q42 = q[7];
    const double q44 = -(q42 + q43);
    d[4] = dt * (q10 * x[1] + q00 * x[0]);
    d[5] = dt * (q01 * x[0] + q21 * x[2] + q11 * x[1]);
    d[6] = dt * (q12 * x[1] + q32 * x[3] + q42 * x[4] + q22 * x[2]);
    d[7] = dt * (q23 * x[2] + q43 * x[4] + q33 * x[3]);
    d[8] = dt * (q24 * x[2] + q34 * x[3] + q44 * x[4]);
    // GW_utils.hpp:322-330 (its limit at V == 0), 354-355
    cur.Ito2 = VF_RT == 0.0 ? S.ClCh * c.Ito2_const * (p.Clo - p.Clcyto) : q[8];
    cur.ICaL = S.JLCC * c.ICaL_const;
    cur.Jtr_tot = S.Jtr * c.CRU_factor;
    cur.Jxfer_tot = S.Jxfer * c.CRU_factor;
}

// GW.tpp:201-211: the increments of V and the concentrations, into d[0..6]
// (gw_globals_t order: V, Nai, Ki, Cai, CaNSR, CaLTRPN, CaHTRPN).
GW_HD void gd_combine(const CellConsts &c, const Currents &cur, double beta_cyto, double dLTRPN, double dHTRPN, double dt,
                      double Istim, double d[7])
{
    d[1] = -dt * c.CSA_FVcyto * (cur.INa + cur.INab + 3 * cur.INaCa + 3 * cur.INaK);
    d[2] = -dt * c.CSA_FVcyto * (cur.IKr + cur.IKs + cur.Ito1 + cur.IK1 + cur.IKp - 2 * cur.INaK);
    d[3] = dt * beta_cyto *
           (-0.5 * c.CSA_FVcyto * (cur.ICab + cur.IpCa - 2 * cur.INaCa) + c.VSS_Vcyto * cur.Jxfer_tot - cur.Jup -
            (dLTRPN + dHTRPN));
    d[4] = dt * (c.Vcyto_VNSR * cur.Jup - c.VJSR_VNSR * cur.Jtr_tot);
    d[5] = dLTRPN * dt;
    d[6] = dHTRPN * dt;
    d[0] = dt * (Istim - (cur.INa + cur.ICaL + cur.IKr + cur.IKs + cur.Ito1 + cur.IK1 + cur.IKp + cur.Ito2 +
                          cur.INaK + cur.INaCa + cur.IpCa + cur.ICab + cur.INab));
}

// GW.tpp:64-123, 135-160: the derivatives of the Kv1.4 (which == 0) or Kv4.3
// (which == 1) chain.
GW_HD void gd_chain_kv(const gw_params_t &p, const double *X, const gw_globals_t &g, double dt, int which,
                       double dKv[10])
{
    if (which == 0) {
        const double aa14 = p.alphaa0Kv14 * X[GD_KV0];
        const double ai14 = p.alphai0Kv14 * X[GD_KV2];
        const double ba14 = p.betaa0Kv14 * X[GD_KV4];
        const double bi14 = p.betai0Kv14 * X[GD_KV6];
        kv_chain(aa14, ai14, ba14, bi14, p.f1Kv14, p.f2Kv14, p.f3Kv14, p.f4Kv14, p.b1Kv14, p.b2Kv14, p.b3Kv14,
                 p.b4Kv14, g.Kv14, dt, dKv);
    } else {
        const double aa43 = p.alphaa0Kv43 * X[GD_KV1];
        const double ai43 = p.alphai0Kv43 * X[GD_KV3];
        const double ba43 = p.betaa0Kv43 * X[GD_KV5];
        const double bi43 = p.betai0Kv43 * X[GD_KV7];
        kv_chain(aa43, ai43, ba43, bi43, p.f1Kv43, p.f2Kv43, p.f3Kv43, p.f4Kv43, p.b1Kv43, p.b2Kv43, p.b3Kv43,
                 p.b4Kv43, g.Kv43, dt, dKv);
    }
}

// All the derivatives from the values X[slot].
GW_HD int gd_finish(const gw_params_t &p, const CellConsts &c, const gw_globals_t &g, double VF_RT, const double *X,
                    double dt, double Istim, const FluxSums &S, gw_globals_t &dg, Currents &cur)
{
    if (!gd_concentrations_ok(p, g)) return GW_E_NONPOSITIVE_CONC;
    double beta_cyto, dLTRPN, dHTRPN, d[7], gk[9];
    const Serial quot;
    gd_k_currents(p, c, g, VF_RT, X, cur, quot);
    gd_na_ca_currents(p, c, g, X, cur, beta_cyto, dLTRPN, dHTRPN, quot);
    gd_gates_kr_cru(p, c, g, VF_RT, X, S, dt, gk, cur, quot);
    gd_combine(c, cur, beta_cyto, dLTRPN, dHTRPN, dt, Istim, d);
    dg.V = d[0];
    dg.Nai = d[1];
    dg.Ki = d[2];
    dg.Cai = d[3];
    dg.CaNSR = d[4];
    dg.CaLTRPN = d[5];
    dg.CaHTRPN = d[6];
    dg.m = gk[0];
    dg.h = gk[1];
    dg.j = gk[2];
    dg.xKs = gk[3];
    for (int i = 0; i < 5; ++i) dg.Kr[i] = gk[4 + i];
    gd_chain_kv(p, X, g, dt, 0, dg.Kv14);
    gd_chain_kv(p, X, g, dt, 1, dg.Kv43);
    return GW_OK;
}

// gd_finish with gd_args' functions evaluated one after another.
GW_HD int global_derivatives(const gw_params_t &p, const CellConsts &c, const gw_globals_t &g, double VF_RT,
                             double dt, double Istim, const FluxSums &S, gw_globals_t &dg, Currents &cur)
{
    double X[GD_X], py[GD_N - GD_POW0];
    gd_args(p, g, VF_RT, X, py);
    for (int i = 0; i < GD_N; ++i) X[i] = gd_eval(i, X[i], i >= GD_POW0 ? py[i - GD_POW0] : 0.0);
    X[GD_IK1] = gw::exp(gd_ik1_arg(c, g.V, X[GD_LK]));
    return gd_finish(p, c, g, VF_RT, X, dt, Istim, S, dg, cur);
}

}  // namespace gw
