// gw_ssa.h -- per-CRU Gillespie SSA over one global step on a quad of lanes
// (one lane per subunit), in FP64 or in the FP32-local variant.
//
// Restates SSA_single_CRU and its helpers (src/includes/SSA.tpp:10-310,
// SSA.hpp:67-71, GW_utils.tpp:118-255, GW_utils.hpp:378-391) for gfx950:
//   - lane j of a quad owns subunit j of one CRU: its CaSS, JLCC, Jrel and one
//     packed 64-bit word (six signed RyR counts, the LCC state, the y gate and
//     the ClCh state). CRU-level state (CaJSR, the xoshiro stream, the step's
//     time, the waiting time) is replicated in the four lanes and evolves
//     identically in each, so every lane draws the same uniforms;
//   - the 4-ring coupling Jiss (SSA.tpp:39-42) and the ordered sums over
//     subunits are DPP quad_perm moves; sums keep the reference order
//     ((x0 + x1) + x2) + x3 in every lane;
//   - the propensities of the chosen subunit are recomputed when an event is
//     sampled, from the inputs the reference's stored rate arrays were formed
//     from (CaSS before this iteration's update, RyR counts before any
//     threshold re-split), so every comparison sees identical values;
//   - all arithmetic keeps the reference's operation order (in FP64,
//     bit-exact with the CPU oracle when compiled with -ffp-contract=off);
//   - the FP32-local variant runs the same code with R = float: propensities,
//     fluxes, buffering factors and waiting times in FP32 with the hardware
//     reciprocal and log2; the integer channel states and the random streams
//     are unchanged. CaSS and CaJSR keep FP64 accumulators (each FP32
//     increment is added to an FP64 running value) because their per-step
//     increments near rest are below one FP32 ulp (CaJSR: about 0.6 ulp), and
//     the concentration differences that drive fluxes are formed in FP64.
#pragma once

#include "gw_model.h"

namespace gw {

// ---- packed subunit word -------------------------------------------------
// bytes 0..5: signed count of the subunit's 5 RyRs in states 1..6;
// bits 48..51: LCC state (1..12); bit 52: y (1 = available); bit 53: ClCh open.
GW_HD int ryr_get(uint64_t w, int k) { return static_cast<int>(static_cast<int8_t>((w >> (8 * k)) & 0xff)); }
GW_HD uint64_t ryr_set(uint64_t w, int k, int v)
{
    return (w & ~(0xffULL << (8 * k))) | (static_cast<uint64_t>(static_cast<uint8_t>(static_cast<int8_t>(v))) << (8 * k));
}
GW_HD int sub_lcc(uint64_t w) { return static_cast<int>((w >> 48) & 15u); }
GW_HD int sub_y(uint64_t w) { return static_cast<int>((w >> 52) & 1u); }
GW_HD int sub_cl(uint64_t w) { return static_cast<int>((w >> 53) & 1u); }
GW_HD uint64_t sub_set_lcc(uint64_t w, int s) { return (w & ~(15ULL << 48)) | (static_cast<uint64_t>(s) << 48); }
GW_HD uint64_t sub_flip_y(uint64_t w) { return w ^ (1ULL << 52); }
GW_HD uint64_t sub_flip_cl(uint64_t w) { return w ^ (1ULL << 53); }
GW_HD uint64_t sub_pack(int lcc, int y, int cl, const int *n6)
{
    uint64_t w = 0;
    for (int k = 0; k < 6; ++k) w = ryr_set(w, k, n6[k]);
    w = sub_set_lcc(w, lcc);
    if (y) w |= 1ULL << 52;
    if (cl) w |= 1ULL << 53;
    return w;
}

// New LCC state after transition `tr` from state s (the map of sample_LCC,
// src/includes/SSA.tpp:103-197): mode-normal states 1..6, mode-Ca 7..12.
GW_HD int lcc_next(int s, int tr)
{
    if (s == 6) return 5;
    if (s == 12) return 11;
    if (s == 1) return tr == 0 ? 2 : 7;
    if (s == 7) return tr == 0 ? 1 : 8;
    if (s <= 5) return tr == 0 ? s - 1 : (tr == 1 ? s + 1 : s + 6);
    return tr == 0 ? s - 6 : (tr == 1 ? s - 1 : s + 1);
}

// Per-cell parameters the SSA reads (a subset of gw_params_t and CellConsts),
// in the SSA's local arithmetic type.
template <class R>
struct SsaParamsT {
    R rRyR, rxfer, rtr, riss;
    R KBSR, KBSL, KCSQN, BSR_const, BSL_const, CSQN_const, VSS_VJSR;
    R k12, k21, k23, k32, k34, k43, k45, k54, k56, k65, k25, k52;
    R kfClCh, kbClCh, Cao_scaled;
    // rate sums and products of the FP32-local subunit total (formed in FP64)
    R k23_25, k45_43, k56_54, k45k34, k32k43, k65k52, k65k54;
};
using SsaParams = SsaParamsT<double>;
using SsaParamsF = SsaParamsT<float>;

GW_HD void ssa_params_init(SsaParams &s, const gw_params_t &p, const CellConsts &c)
{
    s.rRyR = p.rRyR; s.rxfer = p.rxfer; s.rtr = p.rtr; s.riss = p.riss;
    s.KBSR = p.KBSR; s.KBSL = p.KBSL; s.KCSQN = p.KCSQN;
    s.BSR_const = c.BSR_const; s.BSL_const = c.BSL_const; s.CSQN_const = c.CSQN_const; s.VSS_VJSR = c.VSS_VJSR;
    s.k12 = p.k12; s.k21 = p.k21; s.k23 = p.k23; s.k32 = p.k32; s.k34 = p.k34; s.k43 = p.k43;
    s.k45 = p.k45; s.k54 = p.k54; s.k56 = p.k56; s.k65 = p.k65; s.k25 = p.k25; s.k52 = p.k52;
    s.kfClCh = p.kfClCh; s.kbClCh = p.kbClCh; s.Cao_scaled = c.Cao_scaled;
    s.k23_25 = p.k23 + p.k25; s.k45_43 = p.k45 + p.k43; s.k56_54 = p.k56 + p.k54;
    s.k45k34 = p.k45 * p.k34; s.k32k43 = p.k32 * p.k43; s.k65k52 = p.k65 * p.k52; s.k65k54 = p.k65 * p.k54;
}

// Whether the numerators and denominators of the SSA's quotients (beta_ss,
// beta_jsr, the lumped RyR pairs) lie within what quot_plain asks for while the
// concentrations lie in [0, 2^100): every constant of them in [2^-100, 2^100].
GW_HD int ssa_params_plain(const SsaParams &s)
{
    const double v[] = {s.KBSR, s.KBSL, s.KCSQN, s.BSR_const, s.BSL_const, s.CSQN_const, s.k34, s.k43, s.k56, s.k65};
    int ok = 1;
    for (double x : v) ok &= x >= 0x1p-100 && x <= 0x1p100;
    return ok;
}

GW_HD void ssa_params_f32(SsaParamsF &f, const SsaParams &s)
{
    const double *src = &s.rRyR;
    float *dst = &f.rRyR;
    for (int i = 0; i < static_cast<int>(sizeof(SsaParams) / sizeof(double)); ++i) dst[i] = static_cast<float>(src[i]);
}

// The parameters of a cell's SSA through the scalar cache, into scalar
// registers (they are the same for every lane). The compiler does this by
// itself only where no store of the kernel can come before the load; where the
// kernel stores a CRU and goes on, it keeps them in vector registers, 72 in
// FP64 and 36 in FP32, which are what limits the waves in flight.
template <class T>
__device__ __forceinline__ T load_scalar(const T *p)
{
    static_assert(sizeof(T) % 4 == 0, "whole words");
    struct Words { uint32_t w[sizeof(T) / 4]; } v;
    const auto *q = (const __attribute__((address_space(4))) uint32_t *)(reinterpret_cast<uintptr_t>(p));
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) v.w[i] = q[i];
    return __builtin_bit_cast(T, v);
}

// Local arithmetic of the SSA. FP64: IEEE division and the shared log, bit-exact
// with the oracle. FP32 (the FP32-local variant): one hardware reciprocal
// (v_rcp_f32, 1 ulp) times the numerator, and the hardware log2 (v_log_f32).
// PLAIN: the operands are known to need no scaling (quot_plain).
template <bool PLAIN = false>
__device__ __forceinline__ double ldiv(double a, double b) { return PLAIN ? quot_plain(a, b) : a / b; }
template <bool PLAIN = false>
__device__ __forceinline__ float ldiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// A concentration in [0, 2^100), by its high word; with plain parameters the
// denominators formed from such ones lie within 2^+-302.
constexpr uint32_t kPlainHigh = (1023u + 100u) << 20;
__device__ __forceinline__ uint32_t high_word(double x) { return static_cast<uint32_t>(bits_of(x) >> 32); }
// A sum of rates within 2^+-250.
__device__ __forceinline__ bool plain_total(double x) { return high_word(x) - (773u << 20) < (500u << 20); }
__device__ __forceinline__ double lneglog(double u) { return -gw::log_u01(u); }
__device__ __forceinline__ float lneglog(float u) { return -(__builtin_amdgcn_logf(u) * 0.693147182f); }
__device__ __forceinline__ float sq(float x) { return x * x; }

// Rapid-buffering factors of update_CaSS (SSA.tpp:90) and update_CaJSR
// (SSA.hpp:69). FP64: the reference's expressions. FP32-local: the same
// fractions over one denominator, one reciprocal each instead of three and two.
template <bool PLAIN = false, class R>
__device__ __forceinline__ R beta_ss(const SsaParamsT<R> &P, R ca)
{
    if constexpr (sizeof(R) == 8) {
        return ldiv<PLAIN>(R(1), 1 + ldiv<PLAIN>(P.BSR_const, sq(P.KBSR + ca)) + ldiv<PLAIN>(P.BSL_const, sq(P.KBSL + ca)));
    } else {
        const R x2 = sq(P.KBSR + ca), y2 = sq(P.KBSL + ca), p = x2 * y2;
        return ldiv(p, __builtin_fmaf(P.BSL_const, x2, __builtin_fmaf(P.BSR_const, y2, p)));
    }
}
template <bool PLAIN = false, class R>
__device__ __forceinline__ R beta_jsr(const SsaParamsT<R> &P, R jsr)
{
    if constexpr (sizeof(R) == 8) {
        return ldiv<PLAIN>(R(1), 1 + ldiv<PLAIN>(P.CSQN_const, sq(P.KCSQN + jsr)));
    } else {
        const R x2 = sq(P.KCSQN + jsr);
        return ldiv(x2, x2 + P.CSQN_const);
    }
}

// The 12 RyR propensities of one subunit (update_RyR_rates, GW_utils.tpp:222-255),
// visited in storage order; `f(k, r)` receives each rate.
template <bool PLAIN = false, class R, class F>
__device__ __forceinline__ void ryr_rates(const SsaParamsT<R> &P, uint64_t w, R ca, F &&f)
{
    const R C2 = ca * ca;
    const int n1 = ryr_get(w, 0), n2 = ryr_get(w, 1), n3 = ryr_get(w, 2);
    const int n4 = ryr_get(w, 3), n5 = ryr_get(w, 4), n6 = ryr_get(w, 5);
    const bool hi34 = ca > R(3.685e-2);
    const bool hi56 = ca > R(1.15e-4);
    const R a3 = static_cast<R>(n3), a4 = static_cast<R>(n4), a5 = static_cast<R>(n5);
    R r3 = a3 * P.k34 * C2, r4 = a4 * P.k45, r7 = a3 * P.k32, r8 = a4 * P.k43;
    if (hi34) {
        const R tau34 = ldiv<PLAIN>(R(1), P.k34 * C2 + P.k43);
        const R a = static_cast<R>(n3 + n4);
        r3 = R(0);
        r4 = a * P.k45 * P.k34 * C2 * tau34;
        r7 = a * P.k32 * P.k43 * tau34;
        r8 = R(0);
    }
    R r5, r9, r10, r11;
    if (hi56) {
        const R eq56 = ldiv<PLAIN>(P.k65, P.k56 * C2 + P.k65);
        const R a = static_cast<R>(n5 + n6);
        r5 = R(0);
        r9 = a * P.k52 * eq56;
        r10 = a * P.k54 * C2 * eq56;
        r11 = R(0);
    } else {
        r5 = a5 * P.k56 * C2;
        r9 = a5 * P.k52;
        r10 = a5 * P.k54 * C2;
        r11 = static_cast<R>(n6) * P.k65;
    }
    f(0, static_cast<R>(n1) * P.k12 * C2);
    f(1, static_cast<R>(n2) * P.k23 * C2);
    f(2, static_cast<R>(n2) * P.k25 * C2);
    f(3, r3);
    f(4, r4);
    f(5, r5);
    f(6, static_cast<R>(n2) * P.k21);
    f(7, r7);
    f(8, r8);
    f(9, r9);
    f(10, r10);
    f(11, r11);
}

// The 12 RyR rates of ryr_rates summed in FP32, gathered by count (each lumped
// pair's two rates in one closed form): about half the instructions; the event
// choice still walks the individual rates (ryr_pick). Which product of a sum of
// two is rounded, and which is fused, is part of the result, so the fused
// operations are written out here as everywhere in FP32 (left to the compiler they
// move with the code around them); the quads and the lanes differ in it.
template <bool LANE>
__device__ __forceinline__ float ryr_total(const SsaParamsF &P, uint64_t w, float ca)
{
    const auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
    const float C2 = ca * ca;
    const float n1 = static_cast<float>(ryr_get(w, 0)), n2 = static_cast<float>(ryr_get(w, 1));
    const float n3 = static_cast<float>(ryr_get(w, 2)), n4 = static_cast<float>(ryr_get(w, 3));
    const float n5 = static_cast<float>(ryr_get(w, 4)), n6 = static_cast<float>(ryr_get(w, 5));
    // 1->2, 2->3, 2->5, 2->1
    float r = LANE ? fma(n2, P.k21, C2 * fma(n1, P.k12, n2 * P.k23_25)) : fma(C2, fma(n2, P.k23_25, n1 * P.k12), n2 * P.k21);
    // 3<->4 with 4->5 and 3->2: lumped, (n3 + n4)(k45 k34 C2 + k32 k43) / (k34 C2 + k43)
    if (ca > 3.685e-2f) {
        r += (n3 + n4) * ldiv(fma(P.k45k34, C2, P.k32k43), fma(P.k34, C2, P.k43));
    } else {
        const float k = fma(P.k34, C2, P.k32);
        r += LANE ? fma(n3, k, n4 * P.k45_43) : fma(n4, P.k45_43, n3 * k);
    }
    // 5<->6 with 5->2 and 5->4: lumped, (n5 + n6) k65 (k52 + k54 C2) / (k56 C2 + k65)
    if (ca > 1.15e-4f) {
        r += (n5 + n6) * ldiv(fma(P.k65k54, C2, P.k65k52), fma(P.k56, C2, P.k65));
    } else {
        const float k = fma(P.k56_54, C2, P.k52);
        r += LANE ? fma(n5, k, n6 * P.k65) : fma(n6, P.k65, n5 * k);
    }
    return r;
}

// Subunit total. FP64: in the reference accumulation order (SSA.tpp:48-56),
// 0 + LCC sum, + inactivation, + RyR[0..11], + ClCh, which bit-exact replay
// needs. FP32-local: the same sum with ryr_total; LANE: for one lane per CRU.
template <bool PLAIN = false, bool LANE = false, class R, class KT>
__device__ __forceinline__ R subunit_total(const SsaParamsT<R> &P, const KT &K, const LccTableT<R> &T, uint64_t w, R ca)
{
    const int L = sub_lcc(w);
    R s = T.P[L] + T.Q[L] * ca;
    s += sub_y(w) ? K.inact1 : K.inact0;
    if constexpr (sizeof(R) == 8) {
        ryr_rates<PLAIN>(P, w, ca, [&](int, R r) { s += r; });
        s += sub_cl(w) ? P.kbClCh : P.kfClCh * ca;
        return s;
    } else {
        s += sub_cl(w) ? P.kbClCh : P.kfClCh * ca;
        return s + ryr_total<LANE>(P, w, ca);
    }
}

// Rest-state sampler of one CRU: initialise_LCC / _LCC_i / _RyR / _ClCh
// (src/includes/GW_utils.tpp:5-64) and the CRUState constants (GW_utils.tpp:212-213),
// drawing from a stream keyed by the complement of the CRU's SSA stream key.
// Per CRU the draws are LCC[0..3], y[0..3], RyR[0..3][0..4], ClCh[0..3].
template <int PRNG>
GW_HD void sample_rest_cru(uint64_t seed, int64_t i, double ca[4], double &jsr, uint64_t sub[4])
{
    uint64_t s[4];
    rng_seed(PRNG, s, ~stream_key(seed, i));
    auto u = [&]() { return u01(rng_next<PRNG>(s[0], s[1], s[2], s[3])); };
    for (int j = 0; j < 4; ++j) {
        const double v = u();  // sample_weights over {0.958, 0.038, 0.004} -> LCC 1, 2, 7
        const bool b1 = 0.958 < v, b2 = b1 && 0.958 + 0.038 < v;
        sub[j] = sub_set_lcc(0, b2 ? 7 : b1 ? 2 : 1);
    }
    for (int j = 0; j < 4; ++j) {
        const double v = u();  // {0.9425, 0.0575} -> y = 1, 0
        if (!(0.9425 < v)) sub[j] = sub_flip_y(sub[j]);
    }
    for (int j = 0; j < 4; ++j) {
        for (int k = 0; k < 5; ++k) {
            const double v = u();  // {0.609, 0.1955, 0.1955} -> RyR states 1, 5, 6
            const bool b1 = 0.609 < v, b2 = b1 && 0.609 + 0.5 * 0.391 < v;
            sub[j] += 1ULL << (b2 ? 40 : b1 ? 32 : 0);   // counts of at most 5: no carry
        }
    }
    for (int j = 0; j < 4; ++j) {
        const double v = u();  // {0.998, 0.002} -> ClCh 0, 1
        if (0.998 < v) sub[j] = sub_flip_cl(sub[j]);
    }
    for (int j = 0; j < 4; ++j) ca[j] = 1.45370e-4;
    jsr = 0.908408;
}

GW_HD void sample_rest_cru_any(int prng, uint64_t seed, int64_t i, double ca[4], double &jsr, uint64_t sub[4])
{
    switch (prng) {
    case 0: sample_rest_cru<0>(seed, i, ca, jsr, sub); break;
    case 1: sample_rest_cru<1>(seed, i, ca, jsr, sub); break;
    case 2: sample_rest_cru<2>(seed, i, ca, jsr, sub); break;
    case 3: sample_rest_cru<3>(seed, i, ca, jsr, sub); break;
    case 4: sample_rest_cru<4>(seed, i, ca, jsr, sub); break;
    default: sample_rest_cru<5>(seed, i, ca, jsr, sub); break;
    }
}

struct Digest {
    uint64_t count, hash;
};

GW_HD void digest_event(Digest &d, uint32_t step_lo, int j, int kind, int detail)
{
    const uint32_t code = static_cast<uint32_t>(j) | (static_cast<uint32_t>(kind) << 2) |
                          ((static_cast<uint32_t>(detail) & 15u) << 5) | (step_lo << 16);
    d.count++;
    d.hash = (d.hash ^ code) * 0x100000001b3ULL;
}

constexpr uint32_t kMaxItersPerStep = 1u << 22;

// ---------------------------------------------------------------------------
// Quad helpers: DPP quad_perm moves within each group of 4 lanes. Every call
// sits in quad-uniform control flow, so the source lanes are active.
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ uint32_t qmov32(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ uint64_t qmov64(uint64_t u)
{
    return (static_cast<uint64_t>(qmov32<CTRL>(static_cast<uint32_t>(u >> 32))) << 32) |
           qmov32<CTRL>(static_cast<uint32_t>(u));
}
template <int CTRL>
__device__ __forceinline__ double qmov(double v) { return double_of(qmov64<CTRL>(bits_of(v))); }
template <int CTRL>
__device__ __forceinline__ float qmov(float v) { return __builtin_bit_cast(float, qmov32<CTRL>(__builtin_bit_cast(uint32_t, v))); }
template <int CTRL>
__device__ __forceinline__ int qmovi(int v) { return static_cast<int>(qmov32<CTRL>(static_cast<uint32_t>(v))); }

template <int K, class R>
__device__ __forceinline__ R qget(R v) { return qmov<K * 0x55>(v); }          // lane K of the quad
template <int K>
__device__ __forceinline__ int qgeti(int v) { return qmovi<K * 0x55>(v); }
template <class R>
__device__ __forceinline__ R qnext(R v) { return qmov<0x39>(v); }             // lane (j + 1) & 3
template <class R>
__device__ __forceinline__ R qprev(R v) { return qmov<0x93>(v); }             // lane (j + 3) & 3
__device__ __forceinline__ int qseli(int v, int k)                             // lane k (quad-uniform k)
{
    const int a = qgeti<0>(v), b = qgeti<1>(v), c = qgeti<2>(v), d = qgeti<3>(v);
    return k == 0 ? a : k == 1 ? b : k == 2 ? c : d;
}
__device__ __forceinline__ uint64_t qselu(uint64_t v, int k)
{
    const uint64_t a = qmov64<0x00>(v), b = qmov64<0x55>(v), c = qmov64<0xAA>(v), d = qmov64<0xFF>(v);
    return k == 0 ? a : k == 1 ? b : k == 2 ? c : d;
}
__device__ __forceinline__ double qsel(double v, int k) { return double_of(qselu(bits_of(v), k)); }
__device__ __forceinline__ float qsel(float v, int k)
{
    return __builtin_bit_cast(float, static_cast<uint32_t>(qseli(static_cast<int>(__builtin_bit_cast(uint32_t, v)), k)));
}
template <class R>
__device__ __forceinline__ R qsum4(R v) { return qget<0>(v) + qget<1>(v) + qget<2>(v) + qget<3>(v); }
__device__ __forceinline__ int qsum4i(int v) { return qgeti<0>(v) + qgeti<1>(v) + qgeti<2>(v) + qgeti<3>(v); }

// Replicated CRU-level state of a quad (CaJSR accumulates in FP64 in both forms).
// sample_RyR's choice (SSA.tpp:200-259): the first of the 12 transitions
// whose cumulative rate reaches uu. In FP64 this is the reference's rule as
// it stands. In FP32 the scaled uniform can exceed the cumulative sum by
// rounding, which would take the last transition whatever its rate; there
// only transitions with a positive rate are taken (the last of them on such
// an excess, none (-1) if no rate is positive), so no RyR leaves an empty
// state.
template <class R>
__device__ __forceinline__ int ryr_pick(const SsaParamsT<R> &P, uint64_t w, R ca, R uu)
{
    // without branches: `live` falls at the first cumulative rate that reaches uu
    int tr = sizeof(R) == 8 ? 0 : -1;
    R cum = R(0);
    bool live = true;
    ryr_rates(P, w, ca, [&](int k, R r) {
        if (k > 0) live = live & (cum < uu);
        if (sizeof(R) == 8) tr += (k > 0 && live) ? 1 : 0;
        else tr = (live & (r > R(0))) ? k : tr;
        cum = k == 0 ? r : cum + r;
    });
    return tr;
}

// Source and target states (0..5) of RyR transition tr (0..11, in
// sample_RyR's order, SSA.tpp:200-259).
// One octal digit per transition.
GW_HD int ryr_from(int tr) { return static_cast<int>(0544321432110ULL >> (3 * tr)) & 7; }
GW_HD int ryr_to(int tr) { return static_cast<int>(0431210543421ULL >> (3 * tr)) & 7; }

// FP32-local only: whether transition tr may be applied to word w at the
// subspace Ca the step has just reached. The transition is chosen from the
// propensities before the Ca update (as in the reference); when that update
// re-split a lumped pair, a transition chosen at a pair-sum rate can take a
// member below zero outside lumped mode, and negative counts make negative
// propensities (a negative waiting time runs the Euler updates backwards).
// Such a transition is not applied: a member leaves only while it holds a
// RyR, or while its pair is lumped and the pair holds one.
GW_HD bool ryr_allowed(uint64_t w, int tr, double ca)
{
    const int from = ryr_from(tr);
    if ((from == 2 || from == 3) && ca > 0.03685) return ryr_get(w, 2) + ryr_get(w, 3) > 0;
    if ((from == 4 || from == 5) && ca > 1.15e-4) return ryr_get(w, 4) + ryr_get(w, 5) > 0;
    return ryr_get(w, from) > 0;
}

// Re-splits due in update_CaSS (SSA.tpp:93-96) as a mask: 1 for the (5,6)
// pair, 2 for the (3,4) pair. The reference re-splits at most one pair per
// update (the (5,6) pair when Ca falls through both thresholds at once); the
// FP32-local form re-splits both then, so no lumped pair is left unsplit
// below its threshold.
template <class R>
GW_HD int split_mask(double oldA, double tmp)
{
    const int m56 = (oldA > 1.15e-4 && tmp <= 1.15e-4) ? 1 : 0;
    const int m34 = (oldA > 0.03685 && tmp <= 0.03685) ? 2 : 0;
    if (sizeof(R) == 8) return m56 ? m56 : m34;
    return m56 | m34;
}

// Whether transition tr keeps both counts it changes within the signed byte
// a subunit word holds them in. Lumped-pair members drift (a transition at a
// pair-sum rate moves one named member), and nothing bounds the drift; the
// reference counts in int, so a count leaving [-128, 127] is reported
// (GW_E_RANGE) instead of wrapping.
GW_HD bool ryr_in_range(uint64_t w, int tr)
{
    return ryr_get(w, ryr_from(tr)) > -128 && ryr_get(w, ryr_to(tr)) < 127;
}

// Apply RyR transition tr (0..11, in sample_RyR's order) to a subunit word:
// one RyR from one count to another. With 128 added to each count no byte
// borrows or carries (ryr_in_range).
GW_HD uint64_t ryr_apply(uint64_t w, int tr)
{
    constexpr uint64_t kBias = 0x808080808080ULL;
    return ((w ^ kBias) + (1ULL << (8 * ryr_to(tr))) - (1ULL << (8 * ryr_from(tr)))) ^ kBias;
}

struct CruQ {
    double jsr;
    uint64_t r0, r1, r2, r3;
};

// The step's constants a quad reads beside the LCC table, in registers (in
// scalar ones where they come through load_scalar): chosen where they lie in
// memory, each choice is a load with the whole latency in every iteration.
// Cai and CaNSR at the accumulator precision.
template <class R>
struct QuadConsts {
    double Cai, CaNSR;
    R inact0, inact1, JLCC_mult, JLCC_exp;
};
GW_HD QuadConsts<double> quad_consts(const StepConsts &k)
{
    return {k.Cai, k.CaNSR, k.inact0, k.inact1, k.JLCC_mult, k.JLCC_exp};
}
GW_HD QuadConsts<float> quad_consts(const StepConstsF &k)
{
    return {k.Cai_d, k.CaNSR_d, k.inact0, k.inact1, k.JLCC_mult, k.JLCC_exp};
}
// The same from memory that no block of the launch writes.
__device__ __forceinline__ QuadConsts<double> quad_consts_scalar(const StepConsts &k)
{
    struct Head { double v[6]; };
    const Head h = load_scalar(reinterpret_cast<const Head *>(&k));
    return {h.v[0], h.v[1], h.v[2], h.v[3], h.v[4], h.v[5]};
}
__device__ __forceinline__ QuadConsts<float> quad_consts_scalar(const StepConstsF &k)
{
    struct Head { double Cai_d, CaNSR_d; float Cai, CaNSR, inact0, inact1, JLCC_mult, JLCC_exp; };
    const Head h = load_scalar(reinterpret_cast<const Head *>(&k));
    return {h.Cai_d, h.CaNSR_d, h.inact0, h.inact1, h.JLCC_mult, h.JLCC_exp};
}

// Per-CRU outputs of one step for the reductions (identical in the 4 lanes).
struct QuadOut {
    double Jxfer;    // ((Jxfer0 + Jxfer1) + Jxfer2) + Jxfer3 of the last iteration
    double Jtr;      // Jtr of the last iteration
    double JLCC;     // ((JLCC0 + JLCC1) + JLCC2) + JLCC3 after the step
    double Jrel;     // sum of Jrel after the step
    int open;        // open RyRs (states 3 + 4) after the step
    int clch;        // open ClCh after the step
    uint32_t iters;  // SSA loop iterations
    int err;         // nonzero if the iteration cap was hit
    int changed;     // nonzero if this lane's subunit word or JLCC changed (an event or a re-split)
};

// Uniform draws: FP64 uses the reference's 64-bit map; FP32 the top 24 bits.
template <int PRNG, class R>
__device__ __forceinline__ R qdraw(CruQ &q)
{
    if constexpr (sizeof(R) == 8) {
        return u01(rng_next<PRNG>(q.r0, q.r1, q.r2, q.r3));
    } else {
        return static_cast<float>(static_cast<uint32_t>(rng_next<PRNG>(q.r0, q.r1, q.r2, q.r3) >> 40)) * 0x1p-24f;
    }
}

// Two uniforms from one 64-bit draw, bits 40..63 and 16..39 (the one-lane
// FP32-local layout, built for xoshiro256** only, whose scrambled output has
// no weak bit): an event iteration then advances the engine twice, not four
// times.
__device__ __forceinline__ void split2(uint64_t x, float &hi, float &mid)
{
    hi = static_cast<float>(static_cast<uint32_t>(x >> 40)) * 0x1p-24f;
    mid = static_cast<float>(static_cast<uint32_t>(x >> 16) & 0xffffffu) * 0x1p-24f;
}
template <int PRNG>
__device__ __forceinline__ void draw2(CruQ &q, float &hi, float &mid)
{
    split2(rng_next<PRNG>(q.r0, q.r1, q.r2, q.r3), hi, mid);
}

// One global step of SSA_single_CRU (SSA.tpp:286-310); lane j holds subunit j.
// R is the local arithmetic type (double: the reference path; float: the
// FP32-local variant); KT the step constants of that type. CaSS (`ca`) and
// CaJSR accumulate in FP64 in both; with R = double every expression below is
// the reference's, in its order.
template <class R>
struct QuadState {
    double ca;      // this lane's subunit CaSS (FP64 accumulator in both forms)
    R jl;           // this lane's subunit JLCC
    uint64_t w;     // this lane's subunit word
    CruQ q;         // CaJSR and the CRU's engine (the same in the four lanes)
    Digest dig;     // replay digest (the same in the four lanes)
    int open;
    R Jrel, t, Jtr, Jxfer;
    uint32_t iters;
    int err, changed;
};

// copy_from_CRUState (SSA.tpp:10-33): the step's starting fluxes.
template <class R>
__device__ __forceinline__ void quad_begin(QuadState<R> &S, const SsaParamsT<R> &P)
{
    S.iters = 0;
    S.err = 0;
    S.changed = 0;
    S.open = ryr_get(S.w, 2) + ryr_get(S.w, 3);
    S.Jrel = P.rRyR * static_cast<R>(S.open) * static_cast<R>(S.q.jsr - S.ca);
    S.t = R(0);
    S.Jtr = R(0);
    S.Jxfer = R(0);
}

// One iteration of SSA_single_CRU's loop (SSA.tpp:290-309) for a quad; true
// when the step is finished (the same in the four lanes).
template <int PRNG, bool DIGEST, class R>
__device__ __forceinline__ bool quad_iterate(QuadState<R> &S, const SsaParamsT<R> &P, const QuadConsts<R> &K,
                                             const LccTableT<R> &T, R dt, uint32_t step_lo, int j)
{
    const double Cai = K.Cai, CaNSR = K.CaNSR;
    S.iters++;
    // update_fluxes + update_rates (SSA.tpp:37-56)
    const double oldA = S.ca;
    const R old = static_cast<R>(oldA);
    const double o_next = qnext(oldA);
    const double o_prev = qprev(oldA);
    S.Jtr = P.rtr * static_cast<R>(CaNSR - S.q.jsr);
    const R s_me = subunit_total(P, K, T, S.w, old);
    const R s0 = qget<0>(s_me), s1 = qget<1>(s_me), s2 = qget<2>(s_me), s3 = qget<3>(s_me);
    const R total = s0 + s1 + s2 + s3;
    const R jump = ldiv(lneglog(qdraw<PRNG, R>(S.q)), total);
    const bool last = !(S.t + jump < dt);
    const R h = last ? dt - S.t : jump;
    const uint64_t w_pre = S.w;
    // update_CaSS (SSA.tpp:87-99) for this lane's subunit
    const R Jiss = P.riss * static_cast<R>(o_next + o_prev - 2 * oldA);
    S.Jxfer = P.rxfer * static_cast<R>(oldA - Cai);
    const R betaSS = beta_ss(P, old);
    const R dCaSS = h * (S.jl + S.Jrel - S.Jxfer + Jiss) * betaSS;
    const double tmp = oldA + static_cast<double>(dCaSS);
    const int split = split_mask<R>(oldA, tmp);
    const int splits = qgeti<0>(split) | qgeti<1>(split) << 2 | qgeti<2>(split) << 4 | qgeti<3>(split) << 6;
    // sample_RyR56 / sample_RyR34 (SSA.tpp:59-84), in subunit order (a
    // subunit's (5,6) pair first): every lane of the quad draws the same
    // Bernoulli uniforms and the owner applies them
#pragma unroll 1
    for (int m = splits; m != 0; m &= m - 1) {
        const int bit = __builtin_ctz(m), jj = bit >> 1;
        const int sh = (bit & 1) ? 16 : 32;   // the (3,4) or the (5,6) pair's bytes
        const int n_me = static_cast<int8_t>(S.w >> sh) + static_cast<int8_t>(S.w >> (sh + 8));
        const R kb = (bit & 1) ? P.k43 : P.k65, kf = (bit & 1) ? P.k34 : P.k56;
        const R pr = qsel(ldiv(kb, kb + kf * sq(old)), jj);
        const int n = qseli(n_me, jj);
        int X = 0;
        for (int i = 0; i < n; ++i)
            if (qdraw<PRNG, R>(S.q) < pr) X++;
        const int na = (n > 0) ? X : 0;
        if (j == jj) {
            const uint64_t pair = n > 0 ? static_cast<uint64_t>(X & 0xff) | static_cast<uint64_t>((n - X) & 0xff) << 8 : 0;
            S.w = (S.w & ~(0xffffULL << sh)) | pair << sh;
            S.changed = 1;
        }
        if (DIGEST) digest_event(S.dig, step_lo, jj, (bit & 1) ? 5 : 4, na);
    }
    S.ca = tmp;
    // update_CaJSR (SSA.hpp:67-71), replicated
    {
        const R Jsum = qsum4(S.Jrel);
        const R betaJSR = beta_jsr(P, static_cast<R>(S.q.jsr));
        S.q.jsr += static_cast<double>(h * betaJSR * (S.Jtr - P.VSS_VJSR * Jsum));
    }
    if (last) return true;
    if (S.iters >= kMaxItersPerStep) {   // no physical state gets here; stop instead of spinning
        S.err = 1;
        return true;
    }
    S.t += jump;
    // sample_weights over the subunits (common.hpp:49-59)
    int js;
    {
        const R u = qdraw<PRNG, R>(S.q) * total;
        R cum = s0;
        js = 0;
        if (cum < u) { js = 1; cum += s1;
            if (cum < u) { js = 2; cum += s2;
                if (cum < u) { js = 3; } } }
    }
    // sample_new_state (SSA.tpp:262-283): every lane classifies its own
    // subunit; the chosen lane's class is broadcast to the quad
    const R u3 = qdraw<PRNG, R>(S.q);
    const int L = sub_lcc(S.w);
    const int y = sub_y(S.w);
    const int cl = sub_cl(S.w);
    const R Q = T.Q[L], r0 = T.R0[L], R1 = T.R1[L];
    const R sum_LCC = T.P[L] + Q * old;
    const R inact = y ? K.inact1 : K.inact0;
    const R clr = cl ? P.kbClCh : P.kfClCh * old;
    const R sum_RyR = s_me - (sum_LCC + inact + clr);
    const R u = u3 * s_me;
    const int cls = (u < sum_LCC) ? 0 : (u < (sum_LCC + inact)) ? 1 : (u < (sum_LCC + inact + sum_RyR)) ? 2 : 3;
    const int cls_q = qseli(cls, js);
    const R u4 = (cls_q == 0 || cls_q == 2) ? qdraw<PRNG, R>(S.q) : R(0);
    int detail = 0;
    if (j == js) {
        S.changed = 1;
        const R J = K.JLCC_mult * (P.Cao_scaled - K.JLCC_exp * static_cast<R>(S.ca));   // the flux of a channel that opens now
        if (cls == 0) {
            // sample_LCC (SSA.tpp:103-197); the scan never compares after adding r2
            const R uu = u4 * sum_LCC;
            const R r01 = r0 + ((L == 1) ? Q * old : R1);
            const int tr = r0 < uu ? (r01 < uu ? 2 : 1) : 0;
            const int Ln = lcc_next(L, tr);
            if ((L == 5 && Ln == 6) || (L == 11 && Ln == 12))
                S.jl = (y == 1) ? J : R(0);
            else if (L == 6 || L == 12)
                S.jl = R(0);
            S.w = sub_set_lcc(S.w, Ln);
            detail = Ln;
        } else if (cls == 1) {
            const int yn = 1 - y;
            S.w = sub_flip_y(S.w);
            if (yn == 0) S.jl = R(0);
            else if (L == 6 || L == 12) S.jl = J;
            detail = yn;
        } else if (cls == 2) {
            // sample_RyR (SSA.tpp:200-259) over the propensities before this iteration's update
            int tr = ryr_pick(P, w_pre, old, u4 * sum_RyR);
            if (sizeof(R) == 4 && tr >= 0 && !ryr_allowed(S.w, tr, S.ca)) tr = -1;
            if (tr >= 0) {
                if (!ryr_in_range(S.w, tr)) S.err = 1;
                S.w = ryr_apply(S.w, tr);
            }
            if (tr == 1 || tr == 10) S.open += 1;
            else if (tr == 4 || tr == 7) S.open -= 1;
            S.Jrel = P.rRyR * static_cast<R>(S.open) * static_cast<R>(S.q.jsr - S.ca);
            detail = tr;
        } else {
            S.w = sub_flip_cl(S.w);
            detail = 1 - cl;
        }
    }
    if (DIGEST) digest_event(S.dig, step_lo, js, cls_q, qseli(detail, js));
    return false;
}

// outputs of update_CRUstate_from_temp (GW.tpp:47-62) for the reductions;
// FP32 values enter the FP64 sums exactly
template <class R>
__device__ __forceinline__ QuadOut quad_outputs(const QuadState<R> &S)
{
    QuadOut out;
    out.Jxfer = qsum4(static_cast<double>(S.Jxfer));
    out.Jtr = static_cast<double>(S.Jtr);
    out.JLCC = qsum4(static_cast<double>(S.jl));
    out.Jrel = qsum4(static_cast<double>(S.Jrel));
    out.open = qsum4i(ryr_get(S.w, 2) + ryr_get(S.w, 3));
    out.clch = qsum4i(sub_cl(S.w));
    out.iters = S.iters;
    out.err = S.err;
    out.changed = S.changed;
    return out;
}

template <int PRNG, bool DIGEST, class R>
__device__ QuadOut ssa_step_quad(double &ca, R &jl, uint64_t &w, CruQ &q, const SsaParamsT<R> &P,
                                 const QuadConsts<R> &K, const LccTableT<R> &T, R dt, Digest &dig, uint32_t step_lo, int j)
{
    QuadState<R> S;
    S.ca = ca;
    S.jl = jl;
    S.w = w;
    S.q = q;
    S.dig = dig;
    quad_begin(S, P);
    while (!quad_iterate<PRNG, DIGEST>(S, P, K, T, dt, step_lo, j)) {
    }
    ca = S.ca;
    jl = S.jl;
    w = S.w;
    q = S.q;
    dig = S.dig;
    return quad_outputs(S);
}

// ---------------------------------------------------------------------------
// One lane per CRU (FP32-local variant). The lane visits its four subunits in
// order, as SSA_single_CRU itself does (SSA.tpp:37-99, 262-283); the sampled
// subunit's values are read and written through selects, so no register array
// is indexed with a run-time index.
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ T sel4(const T (&v)[4], int k) { return k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3]; }
template <class T>
__device__ __forceinline__ void put4(T (&v)[4], int k, T x)
{
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (k == j) v[j] = x;
}

// The working state of one CRU during one global step.
struct LaneState {
    double ca[4];
    uint64_t w[4];
    CruQ q;
    float jl[4];
    float Jrel[4];
    uint64_t open;   // open RyRs of the four subunits, 16 signed bits each
    float t;
    uint32_t iters;
    int changed;     // the subunit words or JLCC changed since the CRU was loaded (an event or a re-split)
};

// A subunit's open RyRs are the sum of two counts that each fill a signed byte.
GW_HD uint64_t open_field(int j, int v) { return static_cast<uint64_t>(static_cast<uint16_t>(v)) << (16 * j); }
GW_HD int open_get(uint64_t o, int j) { return static_cast<int16_t>(o >> (16 * j)); }
GW_HD void open_put(uint64_t &o, int j, int v) { o = (o & ~(0xffffULL << (16 * j))) | open_field(j, v); }

// copy_from_CRUState (SSA.tpp:10-33): the step's starting fluxes.
__device__ __forceinline__ void lane_begin(LaneState &S, float rRyR)
{
    S.open = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int open = ryr_get(S.w[j], 2) + ryr_get(S.w[j], 3);
        S.open |= open_field(j, open);
        S.Jrel[j] = rRyR * static_cast<float>(open) * static_cast<float>(S.q.jsr - S.ca[j]);
    }
    S.t = 0.0f;
    S.iters = 0;
}

// An iteration of SSA_single_CRU's loop (SSA.tpp:290-309) comes in two parts,
// so that a wave can let its events wait: lane_try forms the rates, the
// waiting time and the increments without storing any of them (a lane whose
// event has to wait runs the same iteration again), lane_commit stores them
// with the re-splits of the update and, where the iteration ends in one,
// chooses and applies the event. The event (subunit, class, transition) is chosen from the
// propensities before this iteration's Ca update, as in the reference, but
// its uniforms are drawn before the re-split Bernoulli draws of that update
// rather than after them: the draws are independent, so the joint law of the
// choice and the re-splits is the same, and only the choice (not the
// pre-update channel words and totals) has to be kept across the update.
// The four uniforms of an event iteration (waiting time, subunit, class,
// transition) and the Bernoulli trials of a re-split come two per engine draw.
struct LaneTry {
    float s[4];        // subunit totals
    float d[4], dj;    // the increments of CaSS and CaJSR
    float total, jump, u_sub, Jtr;
    double Jxfer;      // summed over the subunits in order
    int split;         // split_mask of subunit j at bits 2j, 2j + 1
    bool last;
};

// The step's constants an iteration reads, out of LDS once: chosen where they lie, each choice is a branch.
struct LaneConsts {
    double Cai, CaNSR;
    float inact0, inact1;
};

template <int PRNG>
__device__ __forceinline__ void lane_try(const LaneState &S, LaneTry &X, const SsaParamsF &P, const LaneConsts &K,
                                         const LccTableF &T, float dt)
{
    // update_fluxes + update_rates (SSA.tpp:37-56)
    X.Jtr = P.rtr * static_cast<float>(K.CaNSR - S.q.jsr);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        X.s[j] = subunit_total<false, true>(P, K, T, S.w[j], static_cast<float>(S.ca[j]));
        asm volatile("" : "+v"(X.s[j]));   // one subunit after another: interleaved, they need twice the registers
    }
    X.total = X.s[0] + X.s[1] + X.s[2] + X.s[3];
    float u_jump;
    split2(rng_output<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3), u_jump, X.u_sub);
    X.jump = ldiv(lneglog(u_jump), X.total);
    X.last = !(S.t + X.jump < dt);
    const float h = X.last ? dt - S.t : X.jump;
    // update_CaSS (SSA.tpp:87-99)
    X.split = 0;
    X.Jxfer = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double oldA = S.ca[j];
        const float ring = static_cast<float>(S.ca[(j + 1) & 3] + S.ca[(j + 3) & 3] - 2 * oldA);
        const float out = static_cast<float>(oldA - K.Cai);
        const float Jxfer = P.rxfer * out;
        const float betaSS = beta_ss(P, static_cast<float>(oldA));
        X.d[j] = h * __builtin_fmaf(P.riss, ring, __builtin_fmaf(-P.rxfer, out, S.jl[j] + S.Jrel[j])) * betaSS;
        asm volatile("" : "+v"(X.d[j]));
        X.split |= split_mask<float>(oldA, oldA + static_cast<double>(X.d[j])) << (2 * j);
        X.Jxfer = j == 0 ? static_cast<double>(Jxfer) : X.Jxfer + Jxfer;
    }
    // update_CaJSR (SSA.hpp:67-71)
    const float Jsum = S.Jrel[0] + S.Jrel[1] + S.Jrel[2] + S.Jrel[3];
    const float betaJSR = beta_jsr(P, static_cast<float>(S.q.jsr));
    X.dj = h * betaJSR * __builtin_fmaf(-P.VSS_VJSR, Jsum, X.Jtr);
}

// ev: the iteration ends in an event; false if the iteration cap was hit or a
// count left the range its byte holds. K: the step's constants in LDS.
template <int PRNG>
__device__ __forceinline__ bool lane_commit(LaneState &S, const LaneTry &X, const SsaParamsF &P, const StepConstsF &K, bool ev)
{
    const LccTableF &T = K.lcc;
    rng_advance<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3);   // past the waiting time's draw
    int js = 0, cls = 0, tr = 0;
    if (ev) {
        // sample_weights over the subunits (common.hpp:49-59)
        const float u = X.u_sub * X.total;
        float cum = X.s[0];
        if (cum < u) { js = 1; cum += X.s[1];
            if (cum < u) { js = 2; cum += X.s[2];
                if (cum < u) { js = 3; } } }
        // the class and transition of sample_new_state (SSA.tpp:262-283) on subunit js
        const uint64_t wj = sel4(S.w, js);
        const float oldj = static_cast<float>(sel4(S.ca, js));
        const float sj = sel4(X.s, js);
        const int L = sub_lcc(wj);
        const float Q = T.Q[L], r0 = T.R0[L], R1 = T.R1[L], i0 = K.inact0, i1 = K.inact1;
        const float sum_LCC = __builtin_fmaf(Q, oldj, T.P[L]);
        const float inact = sub_y(wj) ? i1 : i0;
        const float clr = sub_cl(wj) ? P.kbClCh : P.kfClCh * oldj;
        const float sum_RyR = sj - (sum_LCC + inact + clr);
        float u_cls, u_tr;
        draw2<PRNG>(S.q, u_cls, u_tr);
        const float u3 = u_cls * sj;
        cls = (u3 < sum_LCC) ? 0 : (u3 < (sum_LCC + inact)) ? 1 : (u3 < (sum_LCC + inact + sum_RyR)) ? 2 : 3;
        if (cls == 0) {
            // sample_LCC (SSA.tpp:103-197)
            const float uu = u_tr * sum_LCC;
            const float r01 = r0 + ((L == 1) ? Q * oldj : R1);
            tr = r0 < uu ? (r01 < uu ? 2 : 1) : 0;
        } else if (cls == 2) {
            tr = ryr_pick(P, wj, oldj, u_tr * sum_RyR);
        }
    }
    // sample_RyR56 / sample_RyR34 (SSA.tpp:59-84), in subunit order, a subunit's (5,6) pair first
#pragma unroll 1
    for (int m = X.split; m != 0; m &= m - 1) {
        const int bit = __builtin_ctz(m), j = bit >> 1;
        const int sh = (bit & 1) ? 16 : 32;   // the (3,4) or the (5,6) pair's bytes
        uint64_t w = sel4(S.w, j);
        const float C2 = sq(static_cast<float>(sel4(S.ca, j)));
        const float kb = (bit & 1) ? P.k43 : P.k65, kf = (bit & 1) ? P.k34 : P.k56;
        const float pr = ldiv(kb, __builtin_fmaf(kf, C2, kb));
        const int n = static_cast<int8_t>(w >> sh) + static_cast<int8_t>(w >> (sh + 8));
        int c = 0;
        for (int i = 0; i < n; i += 2) {   // two Bernoulli trials per engine draw
            float b0, b1;
            draw2<PRNG>(S.q, b0, b1);
            c += (b0 < pr) ? 1 : 0;
            c += (i + 1 < n && b1 < pr) ? 1 : 0;
        }
        const uint64_t pair = n > 0 ? static_cast<uint64_t>(c & 0xff) | static_cast<uint64_t>((n - c) & 0xff) << 8 : 0;
        w = (w & ~(0xffffULL << sh)) | pair << sh;
        put4(S.w, j, w);
        S.changed = 1;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) S.ca[j] += static_cast<double>(X.d[j]);
    S.q.jsr += static_cast<double>(X.dj);
    S.iters++;
    if (!ev) return true;
    if (S.iters >= kMaxItersPerStep) return false;   // no physical state gets here; stop instead of spinning
    S.t += X.jump;
    S.changed = 1;
    bool ok = true;
    // apply the chosen event to subunit js after the update (SSA.tpp:262-283)
    uint64_t wj = sel4(S.w, js);
    const double caj_d = sel4(S.ca, js);
    const float caj = static_cast<float>(caj_d);
    float jlj = sel4(S.jl, js);
    const int L = sub_lcc(wj);
    const int y = sub_y(wj);
    const float J = K.JLCC_mult * __builtin_fmaf(-K.JLCC_exp, caj, P.Cao_scaled);   // the flux of a channel that opens now
    if (cls == 0) {
        const int Ln = lcc_next(L, tr);
        if ((L == 5 && Ln == 6) || (L == 11 && Ln == 12))
            jlj = (y == 1) ? J : 0.0f;
        else if (L == 6 || L == 12)
            jlj = 0.0f;
        wj = sub_set_lcc(wj, Ln);
    } else if (cls == 1) {
        wj = sub_flip_y(wj);
        if (y == 1) jlj = 0.0f;
        else if (L == 6 || L == 12) jlj = J;
    } else if (cls == 2) {
        // sample_RyR (SSA.tpp:200-259): the transition chosen above, unless it
        // would take a RyR out of an empty state (ryr_allowed)
        int open = open_get(S.open, js);
        if (tr >= 0 && ryr_allowed(wj, tr, caj_d)) {
            ok = ryr_in_range(wj, tr);
            wj = ryr_apply(wj, tr);
            open += (tr == 1 || tr == 10) ? 1 : (tr == 4 || tr == 7) ? -1 : 0;
            open_put(S.open, js, open);
        }
        put4(S.Jrel, js, P.rRyR * static_cast<float>(open) * static_cast<float>(S.q.jsr - caj_d));
    } else {
        wj = sub_flip_cl(wj);
    }
    put4(S.w, js, wj);
    put4(S.jl, js, jlj);
    return ok;
}

// ---------------------------------------------------------------------------
// One lane per CRU in FP64: the operations of quad_iterate, in its order and
// with its draws, so the results are the same bits. The quad spends a wave
// instruction on 16 CRUs for everything that belongs to a CRU and not to a
// subunit (the draws, the waiting time's logarithm, CaJSR) and moves the rest
// between its lanes; one lane per CRU spends it on 64.
// An iteration comes in three parts, so that a wave can let its events wait:
//   lane64_try     rates, waiting time and the updated concentrations, none of
//                  them stored: a lane whose event has to wait runs the same
//                  iteration again;
//   lane64_commit  stores them, with the re-splits of the update;
//   lane64_event   chooses and applies the event that ends the iteration.
// ---------------------------------------------------------------------------
struct Lane64State {
    double ca[4];
    double jl[4];
    double Jrel[4];
    uint64_t w[4];
    CruQ q;
    double t;
    uint64_t open;    // open RyRs of the four subunits, 16 signed bits each
    uint32_t iters;
    int changed;      // the subunit words or JLCC changed since the CRU was loaded
};

struct Lane64Consts {
    double Cai, CaNSR, inact0, inact1;
};

struct Lane64Try {
    double ca[4];     // CaSS after the update
    double s[4];      // subunit totals
    double total, h, jump, jsr, Jxfer, Jtr;
    int split;        // split_mask of subunit j at bits 2j, 2j + 1
    bool last;
};

__device__ __forceinline__ void lane64_begin(Lane64State &S, double rRyR)
{
    S.open = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int open = ryr_get(S.w[j], 2) + ryr_get(S.w[j], 3);
        S.open |= open_field(j, open);
        S.Jrel[j] = rRyR * static_cast<double>(open) * (S.q.jsr - S.ca[j]);
    }
    S.t = 0.0;
    S.iters = 0;
}

// The waiting time's quotient; a draw of zero has an infinite logarithm.
__device__ __forceinline__ double plain_quotient(double neglog, double total)
{
    return __ballot(!plain_total(total) || neglog > 0x1p10) == 0 ? quot_plain(neglog, total) : neglog / total;
}

template <int PRNG, bool PLAIN>
__device__ __forceinline__ void lane64_try_form(const Lane64State &S, Lane64Try &X, const SsaParams &P, const StepConsts &K,
                                           const LccTable &T, double dt)
{
    const Lane64Consts k{K.Cai, K.CaNSR, K.inact0, K.inact1};   // read once: chosen where they lie, each choice is a branch
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        X.s[j] = subunit_total<PLAIN>(P, k, T, S.w[j], S.ca[j]);
        asm volatile("" : "+v"(X.s[j]));   // one subunit after another: interleaved, they need twice the registers
    }
    X.total = X.s[0] + X.s[1] + X.s[2] + X.s[3];
    X.jump = plain_quotient(lneglog(u01(rng_output<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3))), X.total);
    X.last = !(S.t + X.jump < dt);
    X.h = X.last ? dt - S.t : X.jump;
    X.split = 0;
    double Jx[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // update_CaSS (SSA.tpp:87-99)
        const double old = S.ca[j];
        const double Jiss = P.riss * (S.ca[(j + 1) & 3] + S.ca[(j + 3) & 3] - 2 * old);
        Jx[j] = P.rxfer * (old - k.Cai);
        const double d = X.h * (S.jl[j] + S.Jrel[j] - Jx[j] + Jiss) * beta_ss<PLAIN>(P, old);
        X.ca[j] = old + d;
        asm volatile("" : "+v"(X.ca[j]));
        X.split |= split_mask<double>(old, X.ca[j]) << (2 * j);
    }
    X.Jxfer = Jx[0] + Jx[1] + Jx[2] + Jx[3];
    // update_CaJSR (SSA.hpp:67-71)
    X.Jtr = P.rtr * (k.CaNSR - S.q.jsr);
    const double Jsum = S.Jrel[0] + S.Jrel[1] + S.Jrel[2] + S.Jrel[3];
    X.jsr = S.q.jsr + X.h * beta_jsr<PLAIN>(P, S.q.jsr) * (X.Jtr - P.VSS_VJSR * Jsum);
}

// Plain quotients where all lanes' concentrations allow it: 60 instructions less
// of an iteration's 1,165 (12.8 M CRUs 479 and 463 us per step; the quads, whose
// waves have the vector unit for themselves less of the time, lose 2% by the
// choice and divide in full).
template <int PRNG>
__device__ __forceinline__ void lane64_try(const Lane64State &S, Lane64Try &X, const SsaParams &P, const StepConsts &K,
                                           const LccTable &T, double dt, bool plain_cell)
{
    const uint32_t hi = max(max(max(high_word(S.ca[0]), high_word(S.ca[1])), max(high_word(S.ca[2]), high_word(S.ca[3]))),
                            high_word(S.q.jsr));
    if (plain_cell && __ballot(hi >= kPlainHigh) == 0) lane64_try_form<PRNG, true>(S, X, P, K, T, dt);
    else lane64_try_form<PRNG, false>(S, X, P, K, T, dt);
}

// old: the concentrations the iteration started from; w_pre: the words before the re-splits.
template <int PRNG>
__device__ __forceinline__ void lane64_commit(Lane64State &S, const Lane64Try &X, const SsaParams &P, double (&old)[4],
                                              uint64_t (&w_pre)[4])
{
    rng_advance<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        old[j] = S.ca[j];
        w_pre[j] = S.w[j];
    }
    // sample_RyR56 / sample_RyR34 (SSA.tpp:59-84), in subunit order
#pragma unroll 1
    for (int m = X.split; m != 0; m &= m - 1) {
        const int bit = __builtin_ctz(m), j = bit >> 1;
        const int sh = (bit & 1) ? 16 : 32;   // the (3,4) or the (5,6) pair's bytes
        uint64_t w = sel4(S.w, j);
        const double C2 = sq(sel4(old, j));
        const double kb = (bit & 1) ? P.k43 : P.k65, kf = (bit & 1) ? P.k34 : P.k56;
        const double pr = kb / (kb + kf * C2);
        const int n = static_cast<int8_t>(w >> sh) + static_cast<int8_t>(w >> (sh + 8));
        int c = 0;
        for (int i = 0; i < n; ++i)
            if (u01(rng_next<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3)) < pr) c++;
        const uint64_t pair = n > 0 ? static_cast<uint64_t>(c & 0xff) | static_cast<uint64_t>((n - c) & 0xff) << 8 : 0;
        w = (w & ~(0xffffULL << sh)) | pair << sh;
        put4(S.w, j, w);
        S.changed = 1;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) S.ca[j] = X.ca[j];
    S.q.jsr = X.jsr;
    S.iters++;
}

// sample_weights over the subunits (common.hpp:49-59) and sample_new_state
// (SSA.tpp:262-283) on the chosen one; false if a count left the range its
// byte holds.
template <int PRNG>
__device__ __forceinline__ bool lane64_event(Lane64State &S, const Lane64Try &X, const SsaParams &P, const StepConsts &K,
                                             const LccTable &T, const double (&old)[4], const uint64_t (&w_pre)[4])
{
    S.t += X.jump;
    S.changed = 1;
    int js = 0;
    {
        const double u = u01(rng_next<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3)) * X.total;
        double cum = X.s[0];
        if (cum < u) { js = 1; cum += X.s[1];
            if (cum < u) { js = 2; cum += X.s[2];
                if (cum < u) { js = 3; } } }
    }
    const double u3 = u01(rng_next<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3));
    uint64_t w = sel4(S.w, js);
    const double o = sel4(old, js), s_me = sel4(X.s, js), ca = sel4(S.ca, js);
    double jl = sel4(S.jl, js);
    const int L = sub_lcc(w), y = sub_y(w), cl = sub_cl(w);
    const double Q = T.Q[L], r0 = T.R0[L], R1 = T.R1[L], i0 = K.inact0, i1 = K.inact1;
    const double J = K.JLCC_mult * (P.Cao_scaled - K.JLCC_exp * ca);   // the flux of a channel that opens now
    const double sum_LCC = T.P[L] + Q * o;
    const double inact = y ? i1 : i0;
    const double clr = cl ? P.kbClCh : P.kfClCh * o;
    const double sum_RyR = s_me - (sum_LCC + inact + clr);
    const double u = u3 * s_me;
    const int cls = (u < sum_LCC) ? 0 : (u < (sum_LCC + inact)) ? 1 : (u < (sum_LCC + inact + sum_RyR)) ? 2 : 3;
    const double u4 = (cls == 0 || cls == 2) ? u01(rng_next<PRNG>(S.q.r0, S.q.r1, S.q.r2, S.q.r3)) : 0.0;
    bool ok = true;
    if (cls == 0) {
        // sample_LCC (SSA.tpp:103-197); the scan never compares after adding r2
        const double uu = u4 * sum_LCC;
        const double r01 = r0 + ((L == 1) ? Q * o : R1);
        const int tr = r0 < uu ? (r01 < uu ? 2 : 1) : 0;
        const int Ln = lcc_next(L, tr);
        if ((L == 5 && Ln == 6) || (L == 11 && Ln == 12))
            jl = (y == 1) ? J : 0.0;
        else if (L == 6 || L == 12)
            jl = 0.0;
        w = sub_set_lcc(w, Ln);
    } else if (cls == 1) {
        w = sub_flip_y(w);
        if (y == 1) jl = 0.0;
        else if (L == 6 || L == 12) jl = J;
    } else if (cls == 2) {
        // sample_RyR (SSA.tpp:200-259) over the propensities before this iteration's update
        const int tr = ryr_pick(P, sel4(w_pre, js), o, u4 * sum_RyR);
        ok = ryr_in_range(w, tr);
        w = ryr_apply(w, tr);
        int open = open_get(S.open, js);
        open += (tr == 1 || tr == 10) ? 1 : (tr == 4 || tr == 7) ? -1 : 0;
        open_put(S.open, js, open);
        put4(S.Jrel, js, P.rRyR * static_cast<double>(open) * (S.q.jsr - ca));
    } else {
        w = sub_flip_cl(w);
    }
    put4(S.w, js, w);
    put4(S.jl, js, jl);
    return ok;
}

}  // namespace gw
