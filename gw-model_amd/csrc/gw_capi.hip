// gw_capi.hip -- kernels of the MI355X Greenstein-Winslow integrator and the
// C-ABI of include/gw_capi.h.
//
// Device layout: every CRU of every cell owns one slot. Per-subunit words are
// stored [slot][4] (CaSS, JLCC, the packed subunit word holding the six RyR
// counts, LCC state, y gate and ClCh); CaJSR is [slot]; the engine state is
// [slot][4] words and the replay digest [slot][2]. A CRU is advanced by a quad
// of lanes (lane j owns subunit j) or, in FP32-local shapes that ask for it and
// in large FP64 batches, by one lane; a block's CRUs belong to one cell.
//
// One Euler step (GW_model::euler_step, src/includes/GW.tpp:236-272) is one
// launch of k_step (or half a launch, where CRUs stay in registers over two
// steps). Its SSA blocks advance every CRU through SSA(dt) with the
// cell's frozen constants and reduce the flux sums exactly (128-bit fixed
// point) into one partial per block. Its first blocks, one per cell, close
// the previous step at the same time: they sum that step's partials, apply
// globals += dGlobals, form the derivatives of the new step and the SSA
// constants of the step after it. This works because SSA(n+1) needs only the
// globals of step n+1 = globals(n) + dGlobals(n), and dGlobals(n) was formed
// from the sums of step n-1; the sums of step n enter dGlobals(n+1) only.
// Step constants and block partials are double-buffered by step parity.
#include "gw_kernels.h"
#include "gw_route.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <iterator>
#include <mutex>
#include <random>
#include <string>
#include <vector>

using namespace gw;

namespace {

// ===========================================================================
// device helpers
// ===========================================================================
__device__ double protocol_istim(const DevCell &C, double t, int64_t step)
{
    switch (C.proto.kind) {
    case GW_PROTO_TABLE:
        return (C.istim && step < C.istim_len) ? C.istim[step] : 0.0;
    case GW_PROTO_PACE: {
        const double x = t - C.proto.start;
        if (x < 0.0) return 0.0;
        const double ph = (C.proto.period > 0.0 && C.proto.period < 1e300) ? fmod(x, C.proto.period) : x;
        return ph < C.proto.duration ? C.proto.amplitude : 0.0;
    }
    default:
        return 0.0;
    }
}

__device__ double protocol_vclamp(const DevCell &C, double t)
{
    return (t >= C.proto.t_on && t < C.proto.t_off) ? C.proto.step : C.proto.hold;
}

__device__ void obs_update(gw_cell_obs_t &o, double V_old, double V, double t_old, double dt, double Cai, double ICaL,
                           double open_frac, double jrel_scaled)
{
    o.peak_V = fmax(o.peak_V, V);
    o.min_V = fmin(o.min_V, V);
    o.peak_Cai = fmax(o.peak_Cai, Cai);
    o.peak_ICaL_neg = fmin(o.peak_ICaL_neg, ICaL);
    o.sum_open_RyR_frac += open_frac;
    o.int_Jrel += jrel_scaled * dt;
    o.n_steps += 1.0;
    // APD90: upstroke = upward crossing of -40 mV; end = downward crossing of
    // V_rest + 0.1 (V_peak - V_rest), both linearly interpolated between steps.
    if (o.apd_t_up < 0.0) {
        o.apd_v_rest = fmin(o.apd_v_rest, V);
        if (V_old < -40.0 && V >= -40.0) {
            o.apd_t_up = t_old + dt * (-40.0 - V_old) / (V - V_old);
            o.apd_v_peak = V;
        }
    } else {
        o.apd_v_peak = fmax(o.apd_v_peak, V);
        const double thr = o.apd_v_rest + 0.1 * (o.apd_v_peak - o.apd_v_rest);
        if (V_old > thr && V <= thr && V < o.apd_v_peak - 10.0) {
            const double tx = t_old + dt * (V_old - thr) / (V_old - V);
            const double apd = tx - o.apd_t_up;
            o.apd90_prev = o.apd90_last;
            o.apd90_last = apd;
            if (o.beats_done >= 1.0) {
                o.alt_sum += fabs(apd - o.apd90_prev);
                o.alt_count += 1.0;
            }
            o.beats_done += 1.0;
            o.apd_t_up = -1.0;
            o.apd_v_rest = V;
        }
    }
    o.v_prev = V;
}

// Derivatives of the step d.step at state d.g (the part of euler_step before
// SSA(dt), GW.tpp:238-247) and, when kslot >= 0, that step's SSA constants
// (GW.tpp:216-221) into d.k[kslot]. Works on register copies of the cell's
// globals and constants; the results are written back to the cell's state once.
__device__ void prepare_step(const DevCell &C, CellDyn &d, const FluxSums &S, double dt, Currents &cur, int kslot)
{
    const gw_params_t &p = C.p;
    const CellConsts &c = C.c;
    gw_globals_t g = d.g;
    gw_globals_t dg;
    const double Istim = protocol_istim(C, d.t, d.step);
    if (d.clamp) g.V = protocol_vclamp(C, d.t);
    const double VF_RT = g.V * c.F_RT;
    const double expm = gw::exp(-VF_RT);
    const int rc = global_derivatives(p, c, g, VF_RT, dt, Istim, S, dg, cur);
    if (rc != GW_OK && d.status == 0) d.status = rc;
    d.Istim = Istim;
    d.g = g;
    d.dg = dg;
    if (kslot >= 0) {
        step_consts(d.k[kslot], p, c, g.V, expm, g.Cai, g.CaNSR, static_cast<uint32_t>(d.step & 0xffff));
        step_consts_f32(d.kf[kslot], d.k[kslot]);
    }
}

// SSA constants of the step after d.step, into d.k[(d.step + 1) & 1]: the
// potential and concentrations that step will start from (globals + dGlobals
// unless frozen; the clamp potential at t + dt under a clamp protocol), formed
// with the same operations prepare_step will apply at that step.
__device__ void lookahead_consts(const DevCell &C, CellDyn &d, double dt, bool frozen)
{
    double V = d.g.V, Cai = d.g.Cai, CaNSR = d.g.CaNSR;
    if (!frozen) {
        if (!d.clamp) V += d.dg.V;
        Cai += d.dg.Cai;
        CaNSR += d.dg.CaNSR;
    }
    if (d.clamp) V = protocol_vclamp(C, d.t + dt);
    const double VF_RT = V * C.c.F_RT;
    const double expm = gw::exp(-VF_RT);
    const int slot = static_cast<int>((d.step + 1) & 1);
    step_consts(d.k[slot], C.p, C.c, V, expm, Cai, CaNSR, static_cast<uint32_t>((d.step + 1) & 0xffff));
    step_consts_f32(d.kf[slot], d.k[slot]);
}

// Exact sums over a cell's CRUs.
struct FluxTotals {
    Fx jlcc, jxfer, jtr, jrel;
    int64_t clch, open;
    int32_t err;
};

__device__ __forceinline__ void totals_zero(FluxTotals &m)
{
    fx_zero(m.jlcc); fx_zero(m.jxfer); fx_zero(m.jtr); fx_zero(m.jrel);
    m.clch = 0; m.open = 0; m.err = 0;
}

__device__ void totals_add(FluxTotals &a, const FluxTotals &b)
{
    fx_add(a.jlcc, b.jlcc);
    fx_add(a.jxfer, b.jxfer);
    fx_add(a.jtr, b.jtr);
    fx_add(a.jrel, b.jrel);
    a.clch += b.clch;
    a.open += b.open;
    a.err |= b.err;
}

// The 128-bit value of three (signed) limb sums.
__device__ __forceinline__ Fx limbs_fx(uint64_t S0, uint64_t S1, uint64_t S2)
{
    Fx f;
    f.lo = S0;
    f.hi = static_cast<uint64_t>(static_cast<int64_t>(S0) >> 63);
    fx_add_raw(f, S1 << 43, static_cast<uint64_t>(static_cast<int64_t>(S1) >> 21));
    fx_add_raw(f, 0, S2 << 22);
    return f;
}

// The three 43-bit limbs of v, whole numbers in FP64 (all of v's sign): the
// 128-bit value fx_add forms, truncated at 2^-80, without its shifts. Where v
// is not below 2^24 in magnitude they are zero and the answer is false.
__device__ __forceinline__ bool limb_split(double v, double &lo, double &mid, double &hi)
{
    const bool ok = __builtin_fabs(v) < 0x1p24;
    v = ok ? v : 0.0;
    hi = __builtin_trunc(v * 0x1p-6);
    const double r = __builtin_fma(hi, -0x1p6, v);
    mid = __builtin_trunc(r * 0x1p37);
    const double r2 = __builtin_fma(mid, -0x1p-37, r);
    lo = __builtin_trunc(r2 * 0x1p80);
    return ok;
}

// Exact per-block sums of the SSA outputs. Each flux is added in its three
// limbs, whole numbers in FP64, into LDS; no block's CRUs reach 2^53 in a limb
// sum, so the order does not matter. The integer outputs (iterations, open
// RyRs, open ClCh, error flags) are added the same way, lane j of each quad
// adding output j, so that no atomic address is shared by the whole wave
// (which would make the compiler scan the active lanes one by one); four copies,
// by quad, leave four lanes of a wave to an address.
constexpr int kCopies = 4;
struct BlockAcc {
    double limb[PW_ITERS][kCopies];   // Jxfer, Jtr, JLCC, Jrel, three limbs each
    unsigned long long ints[PW_N - PW_ITERS][kCopies];   // iterations, open RyRs, open ClCh, error flags
};

__device__ __forceinline__ void acc_zero(BlockAcc &A)
{
    const int t = threadIdx.x;
    static_assert(sizeof(BlockAcc) == 64 * 8, "one word per thread of the smallest block");
    if (t < 64) reinterpret_cast<unsigned long long *>(&A)[t] = 0;
}

// Adds v to flux q's sum; false if it left the range (limb_split).
__device__ __forceinline__ bool acc_add(BlockAcc &A, int q, int copy, double v)
{
    double lo, mid, hi;
    const bool ok = limb_split(v, lo, mid, hi);
    unsafeAtomicAdd(&A.limb[3 * q][copy], lo);
    unsafeAtomicAdd(&A.limb[3 * q + 1][copy], mid);
    unsafeAtomicAdd(&A.limb[3 * q + 2][copy], hi);
    return ok;
}

// The outputs of a quad's CRU: lane j adds output j (update_CRUstate_from_temp, GW.tpp:47-62).
__device__ __forceinline__ void quad_add(BlockAcc &A, int j, const QuadOut &o, uint64_t iters)
{
    const int copy = (threadIdx.x >> 2) & (kCopies - 1);
    const int fl = acc_add(A, j, copy, j == 0 ? o.Jxfer : j == 1 ? o.Jtr : j == 2 ? o.JLCC : o.Jrel) ? 0 : 1;
    // error flags of the three summed fluxes (the range of Jrel is not checked)
    const int e = (qgeti<0>(fl) | qgeti<1>(fl) | qgeti<2>(fl)) | (o.err ? 4 : 0);
    const int64_t iv = j == 0 ? static_cast<int64_t>(iters) : j == 1 ? o.open : j == 2 ? o.clch : e;
    atomicAdd(&A.ints[j][copy], static_cast<unsigned long long>(iv));
}

// Word t of the block's partial.
__device__ __forceinline__ uint64_t acc_word(const BlockAcc &A, int t)
{
    if (t < PW_ITERS) {
        double d = A.limb[t][0];
        for (int k = 1; k < kCopies; ++k) d += A.limb[t][k];
        return static_cast<uint64_t>(static_cast<int64_t>(d));
    }
    uint64_t v = A.ints[t - PW_ITERS][0];
    for (int k = 1; k < kCopies; ++k) v += A.ints[t - PW_ITERS][k];
    return t == PW_ERR ? (v != 0) : v;
}

// The block's partial of one step, one word per thread.
__device__ __forceinline__ void write_partial(const KArgs &a, const BlockAcc &A, int64_t index)
{
    const int t = threadIdx.x;
    if (t < PW_N) a.partials[index].w[t] = acc_word(A, t);
}

template <int NT>
__device__ void block_reduce(FluxTotals *red, FluxTotals mine)
{
    const int tid = threadIdx.x;
    red[tid] = mine;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (tid < s) totals_add(red[tid], red[tid + s]);
        __syncthreads();
    }
}

// ===========================================================================
// kernels
// ===========================================================================
// Thread t of an SSA-shaped block handles subunit (t & 3) of CRU (t >> 2).

// The blocks of every cell in every shape (grid: cells, shapes).
__global__ void k_block_info(const DevCell *cells, BlockInfo *out)
{
    const DevCell &C = cells[blockIdx.x];
    const int sh = blockIdx.y;
    const int per = crus_per_block(sh);
    for (int b = threadIdx.x; b < C.nblk[sh]; b += blockDim.x)
        out[C.blk_all[sh] + b] = BlockInfo{static_cast<int32_t>(blockIdx.x), min(per, C.n_cru - b * per),
                                           C.slot0 + static_cast<int64_t>(b) * per};
}

// A CRU's engine, replay digest and rest state (src/includes/GW_utils.tpp:5-64),
// one lane per CRU; padding slots get an inert state. One kernel with every
// lane at work: 12.8 M CRUs take 454 us (seeding apart from sampling, with one
// lane of four at work in the sampler and its counts in scratch, took 2,550),
// which writes the state at 3.8 TB/s.
constexpr int kInitMap = shape_of_crus(kBlock);
template <int PRNG>
__global__ __launch_bounds__(kBlock) void k_init_crus(KArgs a, const BlockInfo *blocks)
{
    const BlockInfo bi = blocks[blockIdx.x];
    const DevCell &C = a.cells[bi.cell];
    const int t = threadIdx.x;
    const int64_t slot = bi.slot + t;
    const int64_t i = slot - C.slot0;
    if (i >= (C.n_cru + kSlotAlign - 1) / kSlotAlign * kSlotAlign) return;
    uint64_t s[4];
    rng_seed(PRNG, s, stream_key(C.seed, i));
    double ca[4] = {}, jsr = 0.0;
    uint64_t sub[4];
    if (t < bi.n) sample_rest_cru<PRNG>(C.seed, i, ca, jsr, sub);
    else
        for (int j = 0; j < 4; ++j) sub[j] = sub_set_lcc(0, 1);
    double2 *pc = reinterpret_cast<double2 *>(a.CaSS + slot * 4);
    pc[0] = make_double2(ca[0], ca[1]);
    pc[1] = make_double2(ca[2], ca[3]);
    ulonglong2 *pw = reinterpret_cast<ulonglong2 *>(a.sub + slot * 4);
    pw[0] = make_ulonglong2(sub[0], sub[1]);
    pw[1] = make_ulonglong2(sub[2], sub[3]);
    ulonglong2 *pr = reinterpret_cast<ulonglong2 *>(a.rng + slot * 4);
    pr[0] = make_ulonglong2(s[0], s[1]);
    pr[1] = make_ulonglong2(s[2], s[3]);
    if (a.JLCCf) {
        *reinterpret_cast<float4 *>(a.JLCCf + slot * 4) = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
        double2 *pj = reinterpret_cast<double2 *>(a.JLCC + slot * 4);
        pj[0] = pj[1] = make_double2(0.0, 0.0);
    }
    a.CaJSR[slot] = jsr;
    if (a.dig) {
        a.dig[slot * 2] = 0;
        a.dig[slot * 2 + 1] = 0xcbf29ce484222325ULL;
    }
}

// x added n times: the fixed-point term times n.
__device__ __forceinline__ int fx_add_times(Fx &acc, double x, uint64_t n)
{
    Fx one;
    fx_zero(one);
    const int err = fx_add(one, x);
    fx_add_raw(acc, one.lo * n, one.hi * n + __umul64hi(one.lo, n));
    return err;
}

// Step-0 preparation of every cell (one block per cell; 36 cells of 12,500 CRUs
// 57 us, 80 with one CRU's reads in flight per lane): the flux sums the
// reference's first euler_step reads -- JLCC of the given state, Jxfer and Jtr
// of the constructor's default CRU state and default globals (GW.hpp:104-113),
// ClCh of the given state -- then derivatives and SSA constants.
__global__ void k_init_cells(KArgs a)
{
    __shared__ FluxTotals red[kBlock];
    const int cell = blockIdx.x;
    const DevCell &C = a.cells[cell];
    CellDyn &D = a.dyn[cell];
    FluxTotals mine;
    totals_zero(mine);
    const double X = C.p.rxfer * (1.45370e-4 - 1.45273e-4);
    const double X4 = X + X + X + X;
    const double Y = C.p.rtr * (0.908882 - 0.908408);
    constexpr int kAhead = 4;   // CRUs whose reads are in flight per lane
    uint64_t count = 0;
    for (int64_t i0 = threadIdx.x; i0 < C.n_cru; i0 += kAhead * kBlock) {
        double jl[kAhead][4];
        uint64_t w[kAhead][4];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int64_t slot = C.slot0 + min(i0 + u * kBlock, static_cast<int64_t>(C.n_cru) - 1);
            for (int j = 0; j < 4; ++j) jl[u][j] = ld_jlcc(a, slot * 4 + j);
            for (int j = 0; j < 4; ++j) w[u][j] = a.sub[slot * 4 + j];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (i0 + u * kBlock >= C.n_cru) break;
            ++count;
            mine.err |= fx_add(mine.jlcc, jl[u][0] + jl[u][1] + jl[u][2] + jl[u][3]);
            for (int j = 0; j < 4; ++j) {
                mine.clch += sub_cl(w[u][j]);
                mine.open += ryr_get(w[u][j], 2) + ryr_get(w[u][j], 3);
            }
        }
    }
    if (count > 0) {   // as often as the lane has CRUs
        mine.err |= fx_add_times(mine.jxfer, X4, count);
        mine.err |= fx_add_times(mine.jtr, Y, count);
    }
    block_reduce<kBlock>(red, mine);
    if (threadIdx.x == 0) {
        const FluxTotals &t = red[0];
        FluxSums S{fx_to_double(t.jlcc), fx_to_double(t.jxfer), fx_to_double(t.jtr), static_cast<double>(t.clch)};
        D.sums[0] = S.JLCC; D.sums[1] = S.Jxfer; D.sums[2] = S.Jtr; D.sums[3] = S.ClCh;
        D.sums[4] = static_cast<double>(t.open); D.sums[5] = 0.0;
        D.t = 0.0;
        D.step = 0;
        D.status = t.err ? GW_E_RANGE : 0;
        D.stop_step = kNoStop;
        Currents cur;
        prepare_step(C, D, S, a.dt, cur, 0);
        lookahead_consts(C, D, a.dt, a.frozen != 0);
        if (D.status != 0) D.stop_step = 0;
        D.obs.v_prev = D.g.V;
    }
}

// Copy a step's LCC rate table into LDS (it is read with a per-lane index;
// the cell's other constants are wave-uniform and are read as scalars).
template <class KT, class TT>
__device__ __forceinline__ void load_lcc_table(const KT &K, TT &T)
{
    const uint32_t *src = reinterpret_cast<const uint32_t *>(&K.lcc);
    uint32_t *dst = reinterpret_cast<uint32_t *>(&T);
    for (int w = threadIdx.x; w < static_cast<int>(sizeof(TT) / 4); w += blockDim.x) dst[w] = src[w];
}


// SSA(dt) of `nsteps` steps (GW_model::SSA, src/includes/GW.tpp:214-234) for
// the CRUs of SSA block b, with the constants of step step0 (nsteps > 1
// only in frozen-globals replay, where they do not change). The block's flux
// partial of the last step goes to partials[step0 & 1][b]. R is the CRU-local arithmetic (double, or float for the
// FP32-local variant); CaSS and CaJSR are FP64 in both.
template <class R> struct LocalState;
template <> struct LocalState<double> {
    using Consts = StepConsts;
    static __device__ __forceinline__ double *jlcc(const KArgs &a) { return a.JLCC; }
    static __device__ __forceinline__ const SsaParams &params(const DevCell &C) { return C.sp; }
    static __device__ __forceinline__ const StepConsts &consts(const CellDyn &D, int ks) { return D.k[ks]; }
};
template <> struct LocalState<float> {
    using Consts = StepConstsF;
    static __device__ __forceinline__ float *jlcc(const KArgs &a) { return a.JLCCf; }
    static __device__ __forceinline__ const SsaParamsF &params(const DevCell &C) { return C.spf; }
    static __device__ __forceinline__ const StepConstsF &consts(const CellDyn &D, int ks) { return D.kf[ks]; }
};

// SSA block b's CRUs. Among cells of one size they follow from b, and no read
// stands before those of the cell (a launch starts with cold caches). With the
// same for the close, in us per step: 1,250 CRUs 6.52 and 6.40, 12,500 7.10 and
// 7.01, 256 cells of 7,250 91.6 and 90.1.
__device__ __forceinline__ BlockInfo block_info(const KArgs &a, int b, int per)
{
    if (a.uni_n == 0) return load_scalar(&a.blocks[b]);
    const int cell = static_cast<int>(static_cast<uint64_t>(b) * a.uni_magic >> 32);
    const int at = (b - cell * a.uni_nblk) * per;
    return BlockInfo{cell, min(per, a.uni_n - at), static_cast<int64_t>(cell) * a.uni_slots + at};
}

template <int PRNG, bool DIGEST, class R, int BLOCK>
__device__ __forceinline__ void ssa_block(const KArgs &a, int b, int64_t step0, int64_t nsteps, LccTableT<R> &T, BlockAcc &acc)
{
    using LS = LocalState<R>;
    const int tid = threadIdx.x;
    const int j = tid & 3;
    const BlockInfo bi = block_info(a, b, BLOCK / 4);
    const int ks = static_cast<int>(step0 & 1);
    const DevCell &C = a.cells[bi.cell];
    const CellDyn &D = a.dyn[bi.cell];
    // the CRU's state, in flight with the cell's parameters and constants and with the LCC table on its way into LDS
    const int i = tid >> 2;
    R *const JLCC = LS::jlcc(a);
    const int64_t slot = bi.slot + min(i, bi.n - 1);
    double ca = a.CaSS[slot * 4 + j];
    R jl = JLCC[slot * 4 + j];
    uint64_t w = a.sub[slot * 4 + j];
    CruQ q;
    q.jsr = a.CaJSR[slot];
    q.r0 = a.rng[slot * 4];
    q.r1 = a.rng[slot * 4 + 1];
    q.r2 = a.rng[slot * 4 + 2];
    q.r3 = a.rng[slot * 4 + 3];
    const auto sp = load_scalar(&LS::params(C));
    const QuadConsts<R> kk = quad_consts_scalar(LS::consts(D, ks));
    load_lcc_table(LS::consts(D, ks), T);
    acc_zero(acc);
    __syncthreads();
    const bool active = i < bi.n && step0 < D.stop_step;
    if (active) {
        Digest dg{0, 0};
        if (DIGEST) {
            dg.count = a.dig[slot * 2];
            dg.hash = a.dig[slot * 2 + 1];
        }
        QuadOut o{};
        uint64_t iters = 0;
        int changed = 0;
        const R dt = static_cast<R>(a.dt);
        for (int64_t s = 0; s < nsteps; ++s) {
            o = ssa_step_quad<PRNG, DIGEST>(ca, jl, w, q, sp, kk, T, dt, dg, static_cast<uint32_t>((step0 + s) & 0xffff), j);
            iters += o.iters;
            changed |= o.changed;
            if (o.err) break;
        }
        a.CaSS[slot * 4 + j] = ca;
        if (changed) {   // the channel word and JLCC change only at events and re-splits
            JLCC[slot * 4 + j] = jl;
            a.sub[slot * 4 + j] = w;
        }
        if (j == 0) {
            a.CaJSR[slot] = q.jsr;
            a.rng[slot * 4] = q.r0;
            a.rng[slot * 4 + 1] = q.r1;
            a.rng[slot * 4 + 2] = q.r2;
            a.rng[slot * 4 + 3] = q.r3;
            if (DIGEST) {
                a.dig[slot * 2] = dg.count;
                a.dig[slot * 2 + 1] = dg.hash;
            }
        }
        quad_add(acc, j, o, iters);
    }
    __syncthreads();
    write_partial(a, acc, ks * a.nblocks + b);
}

// ---------------------------------------------------------------------------
// The close of one cell's step, a block's work. A step of a small batch lasts
// as long as this chain of dependent FP64 arithmetic, so it is cut into four
// roles that run on the block's waves side by side (in turn where the block
// has fewer waves) between three barriers, and within a role one value per
// lane wherever the same operations serve many values:
//   1. load:    parameters, globals and block partials, all in flight at once;
//   2. values:  role 0 the exponentials of the derivatives, one per lane;
//               role 1 the logarithms, the powers and the IK1 exponential, one
//               per lane; role 2 the stimulus; role 3 the sums of the partials;
//   3. terms:   role 0 the K currents; role 1 the Na and Ca currents and
//               the uptake; role 2 the Kv chains, one generator entry, then one
//               derivative per lane; role 3 the gates, the IKr chain and
//               the currents formed from the sums;
//   4. joining: roles 0 and 1 the increments and the next step's constants
//               (its exponentials, then the rows of its LCC table, one per
//               lane); role 2 observables and trace; role 3 the stores.
// Each value is formed by the operations of the serial gd_finish and
// step_consts, in their order, so the results are the same bits. Timed in one
// cell of 12,500 CRUs: 11,700 cycles, where the form that ran the sums as a
// butterfly of 128-bit adds and the terms on single lanes took 26,500. Issue
// bounds it: a dependent FP64 operation takes the 4 cycles of its issue.
// ---------------------------------------------------------------------------
constexpr int kGd0 = 7;   // V, Nai, Ki, Cai, CaNSR, CaLTRPN, CaHTRPN: the globals gd_combine derives
constexpr int kSumLanes = PW_N / 2;   // lanes that read one partial, two words each

template <int NT>
struct CloseLds {
    static constexpr int kWaves = NT / kWave;
    static constexpr int kGroups = NT / kSumLanes;
    uint64_t red[kGroups][PW_N];  // partial sums by group of lanes
    double g[36];            // the globals the derivatives start from (gw_globals_t order)
    double x[GD_X];          // the values of the transcendentals
    double ch[29];           // the derivatives of the gates m, h, j, xKs and of the IKr, Kv4.3 and
                             // Kv1.4 chains (the last 29 globals, gw_globals_t order)
    double q[2][kv::kEntries];   // the generator entries of the Kv1.4 and Kv4.3 chains
    double beta_cyto, dLTRPN, dHTRPN;
    double Istim;            // the stimulus of the new time
    double S[4];             // JLCC, Jxfer, Jtr and ClCh of the step's SSA
    double jrel;
    int64_t open;
    int32_t err;
    Currents cur;
    gw_params_t p;           // the cell's parameters, derived constants and observables, staged
    CellConsts c;            // once (each would otherwise be waited on load by load)
    gw_cell_obs_t obs;
};
static_assert(sizeof(gw_globals_t) == 36 * sizeof(double), "globals are 36 doubles");
static_assert(sizeof(gw_params_t) % 8 == 0 && sizeof(CellConsts) % 8 == 0, "staged as 8-byte words");
static_assert(offsetof(gw_globals_t, h) == offsetof(gw_globals_t, m) + sizeof(double) &&
                  offsetof(gw_globals_t, xKs) == offsetof(gw_globals_t, m) + 3 * sizeof(double) &&
                  offsetof(gw_globals_t, Kr) == offsetof(gw_globals_t, m) + 4 * sizeof(double) &&
                  offsetof(gw_globals_t, Kv43) == offsetof(gw_globals_t, Kr) + 5 * sizeof(double) &&
                  offsetof(gw_globals_t, Kv14) == offsetof(gw_globals_t, Kr) + 15 * sizeof(double) &&
                  sizeof(gw_globals_t) == offsetof(gw_globals_t, m) + 29 * sizeof(double) &&
                  offsetof(gw_globals_t, m) == kGd0 * sizeof(double),
              "the gates and the three chains are the last 29 globals: m, h, j, xKs, Kr, Kv4.3, Kv1.4");

// Two adjacent words of a partial; COH reads them past the caches (the
// persistent kernel's SSA blocks write them that way within the launch).
template <bool COH>
__device__ __forceinline__ void partial_pair(const uint64_t *p, uint64_t &x, uint64_t &y)
{
    if constexpr (COH) {
        const unsigned long long *q = reinterpret_cast<const unsigned long long *>(p);
        x = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        y = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        const ulonglong2 v = *reinterpret_cast<const ulonglong2 *>(p);
        x = v.x;
        y = v.y;
    }
}

__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int lane)
{
    return static_cast<uint64_t>(__shfl(static_cast<unsigned long long>(v), lane));
}
__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m)
{
    return static_cast<uint64_t>(__shfl_xor(static_cast<unsigned long long>(v), m));
}

__device__ __forceinline__ double read_lane(double v, int lane)
{
    const uint64_t u = bits_of(v);
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(u), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(u >> 32), lane);
    return double_of(static_cast<uint64_t>(hi) << 32 | lo);
}

// The quotients of a wave-uniform part, one per lane: a correctly rounded FP64
// division is eleven instructions, spent once for all of them.
struct LaneQuot {
    int lane;
    template <int N>
    __device__ __forceinline__ void operator()(const double (&num)[N], const double (&den)[N], double (&q)[N]) const
    {
        double n = num[0], d = den[0];
#pragma unroll
        for (int i = 1; i < N; ++i) {
            n = lane == i ? num[i] : n;
            d = lane == i ? den[i] : d;
        }
        const double r = n / d;
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = read_lane(r, i);
    }
};

// Close step n = D.step of one cell: the exact sum of the cell's block
// partials of step n, globals += dGlobals (GW.tpp:252-271), t += dt, the
// derivatives of step n+1, observables and trace, and the SSA constants of
// step n+2 (those of step n+1 were formed one close earlier and are in use by
// the SSA blocks running beside this one). Every thread of the block (NT)
// takes part. D is the cell's dynamic state: a.dyn[cell], or in the persistent
// kernel a copy the close block keeps in LDS for the whole launch. closing: the
// step, where the launch knows it. With it, and among cells of one size, the
// partials' addresses wait for no read of the cell.
template <int NT, bool COH = false>
__device__ __forceinline__ void close_cell(const KArgs &a, int cell, CellDyn &D, CloseLds<NT> &L, int64_t closing = -1)
{
    constexpr int kWaves = NT / kWave;
    const DevCell &C = a.cells[cell];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = kWaves > 1 ? __builtin_amdgcn_readfirstlane(tid / kWave) : 0;
    auto role = [&](int r) { return wave == (r & (kWaves - 1)); };
    // ---- 1. load
    const int status = D.status;
    const bool clamp = D.clamp != 0;
    const int64_t step_new = D.step + 1;
    const int ks = static_cast<int>((step_new - 1) & 1);
    const double t_old = D.t;
    const double V_old = D.g.V;
    const double t_new = t_old + a.dt;
    double g_in = 0.0, dg_in = 0.0;
    if (tid < 36) {
        g_in = reinterpret_cast<const double *>(&D.g)[tid];
        dg_in = reinterpret_cast<const double *>(&D.dg)[tid];
    }
    constexpr int kPW = sizeof(gw_params_t) / 8, kCW = sizeof(CellConsts) / 8, kOW = sizeof(gw_cell_obs_t) / 8;
    constexpr int kStage = (kPW + kCW + kOW + NT - 1) / NT;
    unsigned long long stage[kStage];
#pragma unroll
    for (int r = 0; r < kStage; ++r) {
        const int w = tid + r * NT;
        stage[r] = 0;
        if (w < kPW) stage[r] = reinterpret_cast<const unsigned long long *>(&C.p)[w];
        else if (w < kPW + kCW) stage[r] = reinterpret_cast<const unsigned long long *>(&C.c)[w - kPW];
        else if (w < kPW + kCW + kOW) stage[r] = reinterpret_cast<const unsigned long long *>(&D.obs)[w - kPW - kCW];
    }
    const GdArg arg = gd_arg_row(role(0) && lane < GD_LOG0 ? lane : 0);
    const uint32_t kv_entry = kv::entry(lane < 2 * kv::kEntries ? lane % kv::kEntries : 0);
    const kv::Row kv_row = kv::row(lane < 20 ? lane % 10 : 0);
    {
        const int64_t par = closing >= 0 ? closing & 1 : ks;
        const Partial *src = a.partials + par * a.nblocks + (a.uni_n ? static_cast<int64_t>(cell) * a.uni_nblk : C.blk0[a.shape]);
        const int nb = a.uni_n ? a.uni_nblk : C.nblk[a.shape];
        constexpr int kG = CloseLds<NT>::kGroups;
        const int w2 = 2 * (tid & (kSumLanes - 1)), grp = tid / kSumLanes;
        uint64_t s0 = 0, s1 = 0;
        constexpr int kAhead = COH ? 1 : 8;   // reads in flight per lane
        for (int q = grp; q < nb; q += kAhead * kG) {
            uint64_t x[kAhead], y[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) partial_pair<COH>(src[min(q + u * kG, nb - 1)].w + w2, x[u], y[u]);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const bool in = q + u * kG < nb;
                s0 += in ? x[u] : 0;
                s1 += in ? y[u] : 0;
            }
        }
        L.red[grp][w2] = s0;
        L.red[grp][w2 + 1] = s1;
    }
    // globals += dGlobals (GW.tpp:252-271), one global per thread; V is held under a
    // clamp and then set to the clamp potential of the new time (prepare_step)
    if (tid < 36) {
        double v = g_in;
        if (!a.frozen && !(tid == 0 && clamp)) v += dg_in;
        if (tid == 0 && clamp) v = protocol_vclamp(C, t_new);
        L.g[tid] = v;
    }
#pragma unroll
    for (int r = 0; r < kStage; ++r) {
        const int w = tid + r * NT;
        if (w < kPW) reinterpret_cast<unsigned long long *>(&L.p)[w] = stage[r];
        else if (w < kPW + kCW) reinterpret_cast<unsigned long long *>(&L.c)[w - kPW] = stage[r];
        else if (w < kPW + kCW + kOW) reinterpret_cast<unsigned long long *>(&L.obs)[w - kPW - kCW] = stage[r];
    }
    __syncthreads();
    // ---- 2. values
    const gw_globals_t &g = *reinterpret_cast<const gw_globals_t *>(L.g);
    const gw_params_t &p = L.p;
    const CellConsts &c = L.c;
    const double VF_RT = g.V * c.F_RT;
    if (role(0) && lane < GD_LOG0) L.x[lane] = gw::exp(gd_arg_value(arg, p, g.V, VF_RT));
    if (role(1) && lane < GD_N - GD_LOG0) {
        const int slot = GD_LOG0 + lane;
        double y;
        const double arg1 = gd_log_arg(slot, p, g, y);
        const double lg = gw::log(arg1);
        // the powers, and on LK's lane the IK1 exponential, are an exponential of the logarithm
        const double e = gw::exp(slot == GD_LK ? gd_ik1_arg(c, g.V, lg) : y * lg);
        L.x[slot] = slot < GD_POW0 ? lg : pow_special(arg1, y, e);
        if (slot == GD_LK) L.x[GD_IK1] = e;
    }
    if (role(2) && lane == 0) L.Istim = status == 0 ? protocol_istim(C, t_new, step_new) : 0.0;
    if (role(3)) {
        const int w = lane & (PW_N - 1);
        uint64_t v = 0;
        for (int k = lane / PW_N; k < CloseLds<NT>::kGroups; k += kWave / PW_N) v += L.red[k][w];
        for (int m = PW_N; m < kWave; m <<= 1) v += shfl_xor_u64(v, m);
        // lane q < 4 recombines flux q; JLCC, Jxfer, Jtr, ClCh into S[0..3]
        const int q3 = 3 * (lane & 3);
        const double f = fx_to_double(limbs_fx(shfl_u64(v, q3), shfl_u64(v, q3 + 1), shfl_u64(v, q3 + 2)));
        if (lane < 3) L.S[lane == 2 ? 0 : lane + 1] = f;
        else if (lane == 3) L.jrel = f;
        else if (lane == PW_CLCH) L.S[3] = static_cast<double>(static_cast<int64_t>(v));
        else if (lane == PW_OPEN) L.open = static_cast<int64_t>(v);
        else if (lane == PW_ERR) L.err = static_cast<uint32_t>(v) != 0;
        else if (lane == PW_ITERS && a.iters_total) atomicAdd(a.iters_total, static_cast<unsigned long long>(v));
    }
    __syncthreads();
    if (status != 0) return;
    if (L.err) {
        if (tid == 0) {
            D.status = GW_E_RANGE;
            D.stop_step = step_new + 1;   // SSA(step_new) runs beside this close; none after it
        }
        return;
    }
    // ---- 3. terms
    const FluxSums S{L.S[0], L.S[1], L.S[2], L.S[3]};
    if (role(0)) {
        Currents k;
        gd_k_currents(p, c, g, VF_RT, L.x, k, LaneQuot{lane});
        if (lane == 0) {
            L.cur.IKr = k.IKr; L.cur.IKs = k.IKs; L.cur.Ito1 = k.Ito1; L.cur.IK1 = k.IK1; L.cur.IKp = k.IKp;
        }
    }
    if (role(1)) {
        Currents k;
        double beta_cyto, dLTRPN, dHTRPN;
        gd_na_ca_currents(p, c, g, L.x, k, beta_cyto, dLTRPN, dHTRPN, LaneQuot{lane});
        if (lane == 0) {
            L.cur.INa = k.INa; L.cur.INab = k.INab; L.cur.INaCa = k.INaCa; L.cur.INaK = k.INaK;
            L.cur.ICab = k.ICab; L.cur.IpCa = k.IpCa; L.cur.Jup = k.Jup;
            L.beta_cyto = beta_cyto; L.dLTRPN = dLTRPN; L.dHTRPN = dHTRPN;
        }
    }
    if (role(2)) {
        if (lane < 2 * kv::kEntries) {
            const int chain = lane / kv::kEntries;
            L.q[chain][lane % kv::kEntries] = kv::entry_value(kv_entry, p, L.x, chain);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the entries pass between lanes of this wave
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < 20) {
            const int chain = lane / 10;
            L.ch[(chain == 0 ? 19 : 9) + lane % 10] =
                kv::derivative(kv_row, lane % 10, L.q[chain], chain == 0 ? g.Kv14 : g.Kv43, a.dt);
        }
    }
    if (role(3)) {
        Currents k;
        double d[9];
        gd_gates_kr_cru(p, c, g, VF_RT, L.x, S, a.dt, d, k, LaneQuot{lane});
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 9; ++i) L.ch[i] = d[i];
            L.cur.Ito2 = k.Ito2; L.cur.ICaL = k.ICaL; L.cur.Jtr_tot = k.Jtr_tot; L.cur.Jxfer_tot = k.Jxfer_tot;
        }
    }
    __syncthreads();
    // ---- 4. joining
    const int slot = static_cast<int>((step_new + 1) & 1);
    if (role(0) || role(1)) {
        double d[kGd0];
        gd_combine(c, L.cur, L.beta_cyto, L.dLTRPN, L.dHTRPN, a.dt, L.Istim, d);
        // lookahead_consts: the potential and concentrations the step after starts from
        double V = g.V, Cai = g.Cai, CaNSR = g.CaNSR;
        if (!a.frozen) {
            if (!clamp) V += d[0];
            Cai += d[3];
            CaNSR += d[4];
        }
        if (clamp) V = protocol_vclamp(C, t_new + a.dt);
        const double e = gw::exp(sc_arg(lane < SC_N ? lane : 0, V, c.F_RT));
        double X[SC_N];
#pragma unroll
        for (int i = 0; i < SC_N; ++i) X[i] = read_lane(e, i);
        if (role(0)) {
            if (lane < kGd0) {
                double v = d[0];
#pragma unroll
                for (int i = 1; i < kGd0; ++i)
                    if (lane == i) v = d[i];
                reinterpret_cast<double *>(&D.dg)[lane] = v;
            }
            StepConsts k;
            step_consts_scalars(k, c, V, X, Cai, CaNSR, static_cast<uint32_t>((step_new + 1) & 0xffff), LaneQuot{lane});
            if (lane == 0) {
                StepConsts &K = D.k[slot];
                K.Cai = k.Cai;
                K.CaNSR = k.CaNSR;
                K.inact0 = k.inact0;
                K.inact1 = k.inact1;
                K.JLCC_mult = k.JLCC_mult;
                K.JLCC_exp = k.JLCC_exp;
                K.step_lo = k.step_lo;
                K._pad = 0;
                step_consts_f32_scalars(D.kf[slot], k);
            }
        }
        if (role(1) && lane < 13) {
            const LccRow w = lcc_row(lane, p, c, X);
            lcc_row_store(D.k[slot].lcc, lane, w);
            lcc_row_store(D.kf[slot].lcc, lane, w);
        }
    }
    if (role(2) && lane == 0) {
        const double open_frac = static_cast<double>(L.open) / (20.0 * C.n_cru);
        gw_cell_obs_t o = L.obs;
        obs_update(o, V_old, g.V, t_old, a.dt, g.Cai, L.cur.ICaL, open_frac, L.jrel * c.CRU_factor);
        D.obs = o;
        if (a.trace_every > 0 && (step_new % a.trace_every) == 0 && D.trace_rows < a.trace_cap) {
            double *row = a.trace + (D.trace_rows * a.ncells + cell) * 4;
            row[0] = g.V;
            row[1] = g.Cai;
            row[2] = L.cur.ICaL;
            row[3] = open_frac;
            D.trace_rows += 1;
        }
    }
    if (role(3)) {
        if (lane < 36) reinterpret_cast<double *>(&D.g)[lane] = L.g[lane];
        if (lane >= kGd0 && lane < 36) reinterpret_cast<double *>(&D.dg)[lane] = L.ch[lane - kGd0];
        if (lane == 0) {
            D.Istim = L.Istim;
            D.sums[0] = S.JLCC; D.sums[1] = S.Jxfer; D.sums[2] = S.Jtr; D.sums[3] = S.ClCh;
            D.sums[4] = static_cast<double>(L.open); D.sums[5] = L.jrel;
            D.t = t_new;
            D.step = step_new;
            int st = 0;
            if (!gd_concentrations_ok(p, g)) st = GW_E_NONPOSITIVE_CONC;
            else if (!(g.V == g.V) || !(g.Cai == g.Cai)) st = GW_E_NAN;
            // A cell that fails here stops after the SSA of step_new, which runs beside
            // this close in the same launch: the SSA blocks read stop_step, which only
            // changes from a value above step_new to step_new + 1, so every block of
            // that launch runs the step and none runs a later one.
            if (st != 0) {
                D.status = st;
                D.stop_step = step_new + 1;
            }
        }
    }
}

// One launch per Euler step: the first `nclose` blocks close step ssa_step-1
// of every cell while the remaining blocks run SSA(ssa_step). The two halves
// share no data: the SSA reads the constants of its step (formed by the close
// one launch earlier) and writes the other partials buffer. ssa_step < 0
// launches the closes alone (the last close of a sequence).
// Resident waves per SIMD the SSA kernels are compiled for: FP64 needs about
// 128 VGPRs; the FP32-local SSA fits 80, where the close in the first blocks
// spills up to 36 bytes.
template <class R> constexpr int kWavesPerSimd = sizeof(R) == 4 ? 6 : 4;

// ssa_step is relative to *base when base is given (replayed graphs of steps).
template <int PRNG, bool DIGEST, class R, int BLOCK>
__global__ __launch_bounds__(BLOCK, kWavesPerSimd<R>) void k_step(KArgs a, int64_t ssa_step, int32_t nclose,
                                                                   const int64_t *base)
{
    __shared__ LccTableT<R> T;
    __shared__ CloseLds<BLOCK> csh;
    __shared__ BlockAcc acc;
    const int bid = blockIdx.x;
    const int64_t step = base ? *base + ssa_step : ssa_step;
    if (bid < nclose) {
        close_cell<BLOCK>(a, bid, a.dyn[bid], csh, ssa_step < 0 ? -1 : step - 1);
        return;
    }
    ssa_block<PRNG, DIGEST, R, BLOCK>(a, bid - nclose, step, 1, T, acc);
}

// The SSA of block b with a quad of lanes per CRU and CPT CRUs per quad: wave
// w of the block owns 16 * CPT consecutive CRUs of the block's cell; a quad
// whose CRU has finished the step takes the next CRU not yet taken (the
// finishing quads in quad order, by a ballot of their first lanes). Lane j
// adds output j of each CRU it finishes to the exact block sums, so the
// results do not depend on which quad ran which CRU. No replay digests.
template <int PRNG, class R, int BLOCK, int CPT>
__device__ __forceinline__ void ssa_block_refill(const KArgs &a, int b, int64_t step0, LccTableT<R> &T, BlockAcc &acc)
{
    constexpr int kQuads = kWave / 4;
    constexpr int kMap = shape_of_crus(BLOCK / 4 * CPT);
    static_assert(crus_per_block(kMap) == BLOCK / 4 * CPT, "CRUs per block must be 16 << map");
    using LS = LocalState<R>;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int j = tid & 3;
    const int qd = lane >> 2;
    const BlockInfo bi = block_info(a, b, BLOCK / 4 * CPT);
    const int ks = static_cast<int>(step0 & 1);
    const DevCell &C = a.cells[bi.cell];
    const CellDyn &D = a.dyn[bi.cell];
    const auto sp = load_scalar(&LS::params(C));
    const QuadConsts<R> kk = quad_consts_scalar(LS::consts(D, ks));
    load_lcc_table(LS::consts(D, ks), T);
    acc_zero(acc);
    __syncthreads();
    const int start = wave * (kQuads * CPT);
    const int64_t slot0 = bi.slot + start;
    const int w1 = min(kQuads * CPT, bi.n - start);   // CRUs of the wave's range
    int i = qd;
    int next = kQuads;   // first CRU of the range not yet taken (wave-uniform)
    bool have = (i < w1) && (step0 < D.stop_step);
    R *const JLCC = LS::jlcc(a);
    const R dt = static_cast<R>(a.dt);
    const uint32_t step_lo = static_cast<uint32_t>(step0 & 0xffff);
    QuadState<R> S;
    auto load = [&](int64_t slot) {
        S.ca = a.CaSS[slot * 4 + j];
        S.jl = JLCC[slot * 4 + j];
        S.w = a.sub[slot * 4 + j];
        S.q.jsr = a.CaJSR[slot];
        S.q.r0 = a.rng[slot * 4];
        S.q.r1 = a.rng[slot * 4 + 1];
        S.q.r2 = a.rng[slot * 4 + 2];
        S.q.r3 = a.rng[slot * 4 + 3];
        S.dig = Digest{0, 0};
        quad_begin(S, sp);
    };
    if (have) load(slot0 + i);
    while (__ballot(have)) {
        bool fin = false;
        if (have) {
            fin = quad_iterate<PRNG, false>(S, sp, kk, T, dt, step_lo, j);
            if (fin) {
                const int64_t slot = slot0 + i;
                a.CaSS[slot * 4 + j] = S.ca;
                if (S.changed) {   // the channel word and JLCC change only at events and re-splits
                    JLCC[slot * 4 + j] = S.jl;
                    a.sub[slot * 4 + j] = S.w;
                }
                if (j == 0) {
                    a.CaJSR[slot] = S.q.jsr;
                    a.rng[slot * 4] = S.q.r0;
                    a.rng[slot * 4 + 1] = S.q.r1;
                    a.rng[slot * 4 + 2] = S.q.r2;
                    a.rng[slot * 4 + 3] = S.q.r3;
                }
                const QuadOut o = quad_outputs(S);
                quad_add(acc, j, o, o.iters);
            }
        }
        const uint64_t m = __ballot(fin && j == 0);
        if (fin) {
            i = next + static_cast<int>(__popcll(m & ((1ULL << (4 * qd)) - 1)));
            have = i < w1;
            if (have) load(slot0 + i);
        }
        next += __popcll(m);
    }
    __syncthreads();
    write_partial(a, acc, ks * a.nblocks + b);
}

// The refill loop keeps a CRU's addresses and the next CRU's index live beside
// the quad state: 127 to 131 VGPRs, which 3 waves per SIMD leave room for.
template <int PRNG, class R, int BLOCK, int CPT>
__global__ __launch_bounds__(BLOCK, 3) void k_step_refill(KArgs a, int64_t ssa_step, int32_t nclose,
                                                           const int64_t *base)
{
    __shared__ LccTableT<R> T;
    __shared__ CloseLds<BLOCK> csh;
    __shared__ BlockAcc acc;
    const int bid = blockIdx.x;
    const int64_t step = base ? *base + ssa_step : ssa_step;
    if (bid < nclose) {
        close_cell<BLOCK>(a, bid, a.dyn[bid], csh, ssa_step < 0 ? -1 : step - 1);
        return;
    }
    ssa_block_refill<PRNG, R, BLOCK, CPT>(a, bid - nclose, step, T, acc);
}

// Sum over the 64 lanes of a wave by a fixed xor butterfly (the same value,
// bit for bit, in every lane).
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v += __shfl_xor(v, m, kWave);
    return v;
}
__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

__device__ __forceinline__ void lane_load(const KArgs &a, int64_t slot, LaneState &S)
{
    const double2 *pc = reinterpret_cast<const double2 *>(a.CaSS + slot * 4);
    const double2 c01 = pc[0], c23 = pc[1];
    S.ca[0] = c01.x; S.ca[1] = c01.y; S.ca[2] = c23.x; S.ca[3] = c23.y;
    const float4 j4 = *reinterpret_cast<const float4 *>(a.JLCCf + slot * 4);
    S.jl[0] = j4.x; S.jl[1] = j4.y; S.jl[2] = j4.z; S.jl[3] = j4.w;
    const ulonglong2 *pw = reinterpret_cast<const ulonglong2 *>(a.sub + slot * 4);
    const ulonglong2 w01 = pw[0], w23 = pw[1];
    S.w[0] = w01.x; S.w[1] = w01.y; S.w[2] = w23.x; S.w[3] = w23.y;
    const ulonglong2 *pr = reinterpret_cast<const ulonglong2 *>(a.rng + slot * 4);
    const ulonglong2 r01 = pr[0], r23 = pr[1];
    S.q.r0 = r01.x; S.q.r1 = r01.y; S.q.r2 = r23.x; S.q.r3 = r23.y;
    S.q.jsr = a.CaJSR[slot];
    S.changed = 0;
}

__device__ __forceinline__ void lane_store(const KArgs &a, int64_t slot, const LaneState &S)
{
    double2 *qc = reinterpret_cast<double2 *>(a.CaSS + slot * 4);
    qc[0] = make_double2(S.ca[0], S.ca[1]);
    qc[1] = make_double2(S.ca[2], S.ca[3]);
    if (S.changed) {   // the channel words and JLCC change only at events and re-splits
        *reinterpret_cast<float4 *>(a.JLCCf + slot * 4) = make_float4(S.jl[0], S.jl[1], S.jl[2], S.jl[3]);
        ulonglong2 *qw = reinterpret_cast<ulonglong2 *>(a.sub + slot * 4);
        qw[0] = make_ulonglong2(S.w[0], S.w[1]);
        qw[1] = make_ulonglong2(S.w[2], S.w[3]);
    }
    ulonglong2 *qr = reinterpret_cast<ulonglong2 *>(a.rng + slot * 4);
    qr[0] = make_ulonglong2(S.q.r0, S.q.r1);
    qr[1] = make_ulonglong2(S.q.r2, S.q.r3);
    a.CaJSR[slot] = S.q.jsr;
}

// Running FP64 sums of the outputs of the CRUs each lane finishes, in
// finishing order, one LDS slot per thread (kept out of the registers the SSA
// needs), added by LDS atomics that no one waits for.
template <int BLOCK>
struct LaneSums {
    double Jxfer[BLOCK], Jtr[BLOCK], JLCC[BLOCK], Jrel[BLOCK];
    // iterations, open RyRs in 20 signed bits from bit 32 and open ClCh from bit 52: a wave owns at most
    // 512 CRUs, and a lane whose neighbours are busy takes nearly all of them
    unsigned long long ints[BLOCK];
    int err;
    __device__ __forceinline__ void zero(int t)
    {
        Jxfer[t] = Jtr[t] = JLCC[t] = Jrel[t] = 0.0;
        ints[t] = 0;
        if (t == 0) err = 0;
    }
    // outputs of update_CRUstate_from_temp (GW.tpp:47-62), summed in subunit order in FP64
    __device__ __forceinline__ void add(int t, const LaneState &S, const LaneTry &X)
    {
        unsafeAtomicAdd(&Jxfer[t], X.Jxfer);
        unsafeAtomicAdd(&Jtr[t], static_cast<double>(X.Jtr));
        unsafeAtomicAdd(&JLCC[t], ((static_cast<double>(S.jl[0]) + S.jl[1]) + S.jl[2]) + S.jl[3]);
        unsafeAtomicAdd(&Jrel[t], ((static_cast<double>(S.Jrel[0]) + S.Jrel[1]) + S.Jrel[2]) + S.Jrel[3]);
        int open = 0, clch = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            open += ryr_get(S.w[j], 2) + ryr_get(S.w[j], 3);
            clch += sub_cl(S.w[j]);
        }
        const int64_t v = (static_cast<int64_t>(clch) << 52) + (static_cast<int64_t>(open) << 32) + S.iters;
        atomicAdd(&ints[t], static_cast<unsigned long long>(v));
    }
};

// Per-wave sums of the lanes' output sums (a fixed FP64 xor butterfly, the
// same in every lane), added exactly into the block accumulators by lanes 0..3.
template <int BLOCK>
__device__ __forceinline__ void lane_accumulate(BlockAcc &acc, const LaneSums<BLOCK> &Ls, int t)
{
    const int lane = t & (kWave - 1);
    const double sx = wave_sum(Ls.Jxfer[t]), st = wave_sum(Ls.Jtr[t]), sl = wave_sum(Ls.JLCC[t]), sr = wave_sum(Ls.Jrel[t]);
    const int64_t v64 = static_cast<int64_t>(Ls.ints[t]);
    const int iters = static_cast<int>(v64 & 0xffffffff);
    const int open = static_cast<int>(static_cast<int64_t>(Ls.ints[t] << 12) >> 44);
    const int clch = static_cast<int>((v64 - (static_cast<int64_t>(open) << 32)) >> 52);
    const int n_it = wave_sum(iters), n_open = wave_sum(open), n_cl = wave_sum(clch);
    const int k = lane & 3;
    const double v = k == 0 ? sx : k == 1 ? st : k == 2 ? sl : sr;
    const bool bad = __ballot(lane < 3 && !(__builtin_fabs(v) < 0x1p24)) != 0 || Ls.err != 0;
    if (lane < 4) {
        acc_add(acc, lane, 0, v);
        const int64_t iv = lane == 0 ? n_it : lane == 1 ? n_open : lane == 2 ? n_cl : (bad ? 1 : 0);
        atomicAdd(&acc.ints[lane][0], static_cast<unsigned long long>(iv));
    }
}

// The SSA of block b with one lane per CRU (FP32-local variant), steps m ..
// m + nss - 1 (nss <= NSS). Wave w of the block owns kWave * CPT consecutive
// CRUs of the block's cell. Its lanes start on the first kWave of them; a lane
// whose CRU has finished its steps takes the next CRU of the range not yet
// taken (the finishing lanes in lane order, by a ballot), so the wave makes
// about (iterations of its range) / kWave trips rather than CPT times the most
// iterations of any one CRU. Which lane runs which CRU depends only on the
// CRUs' own iterations, the same on every run. Each lane sums the outputs of
// its CRUs in FP64 as it finishes them; the per-wave sums are a fixed xor
// butterfly, added exactly across waves and blocks.
//
// Events wait: in nearly every trip a lane or two of the 64 end their
// iteration in an event, whose code is nearly as long as the rest of the
// trip. Such a lane leaves its CRU as it was and runs the same iteration again
// (it would idle otherwise), until event_batch lanes of the wave hold an
// event, or no other lane made progress, or no fresh CRU is left. Early in an
// action potential (1.9% of the iterations end in an event), two steps per
// launch, batches of 1 and 8: 256 x 7,000 CRUs, 4 per lane, 51.1 and 49.2 us
// per step, 64 x 12,500 32.6 and 31.3; 2 per lane 49.2 and 52.5: too few
// iterations per lane to wait for, so there an event is applied at once.
template <int BLOCK, int NSS>
struct LaneLds {
    StepConstsF K[NSS];
    BlockAcc acc[NSS];
    LaneSums<BLOCK> Ls[NSS];
};

constexpr int event_batch(int cpt) { return cpt >= 4 ? 8 : 1; }

template <int PRNG, int BLOCK, int CPT, int NSS>
__device__ __forceinline__ void ssa_block_lane(const KArgs &a, int b, int64_t m, int nss, LaneLds<BLOCK, NSS> &L)
{
    constexpr int kMap = shape_of_crus(BLOCK * CPT);
    static_assert(crus_per_block(kMap) == BLOCK * CPT, "CRUs per block must be 16 << map");
    constexpr int kWords = sizeof(StepConstsF) / 4;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const BlockInfo bi = block_info(a, b, BLOCK * CPT);
    const DevCell &C = a.cells[bi.cell];
    const CellDyn &D = a.dyn[bi.cell];
    const float rRyR = C.spf.rRyR;
    const float dt = static_cast<float>(a.dt);
#pragma unroll
    for (int s = 0; s < NSS; ++s) {
        if (s < nss)
            for (int t = tid; t < kWords; t += BLOCK)
                reinterpret_cast<uint32_t *>(&L.K[s])[t] = reinterpret_cast<const uint32_t *>(&D.kf[(m + s) & 1])[t];
        acc_zero(L.acc[s]);
        L.Ls[s].zero(tid);
    }
    __syncthreads();
    const int64_t stop = D.stop_step;
    const bool run1 = nss > 1 && m + 1 < stop;
    const int start = wave * (kWave * CPT);
    const int w1 = min(kWave * CPT, bi.n - start);   // CRUs of the wave's range
    const int64_t slot0 = bi.slot + start;
    int i = lane;
    int next = kWave;   // first CRU of the range not yet taken (wave-uniform)
    bool have = i < w1 && m < stop;
    int sidx = 0;       // the step (0: m, 1: m + 1) this lane's CRU is in
    LaneState S;
    if (have) {
        lane_load(a, slot0 + i, S);
        lane_begin(S, rRyR);
    }
    while (__ballot(have)) {
        const SsaParamsF *spp = &C.spf;
        asm volatile("" : "+s"(spp));   // read again in each trip: held over the loop they push others out
        const SsaParamsF sp = load_scalar(spp);
        LaneTry X;
        bool ev = false;
        const StepConstsF &K = L.K[NSS > 1 ? sidx : 0];
        if (have) {
            lane_try<PRNG>(S, X, sp, LaneConsts{K.Cai_d, K.CaNSR_d, K.inact0, K.inact1}, K.lcc, dt);
            ev = !X.last;
        }
        const uint64_t m_ev = __ballot(ev);
        const uint64_t m_last = __ballot(have && !ev);
        const bool go = __popcll(m_ev) >= event_batch(CPT) || m_last == 0 || next >= w1;   // wave-uniform
        bool fin = have && !ev;
        if (have && (go || !ev)) {
            if (!lane_commit<PRNG>(S, X, sp, K, ev && go)) {
                L.Ls[sidx].err = 1;
                fin = fin || S.iters >= kMaxItersPerStep;
            }
        }
        if (fin) {
            L.Ls[NSS > 1 ? sidx : 0].add(tid, S, X);
            if (NSS > 1 && sidx == 0 && run1) {   // the same CRU, next step
                sidx = 1;
                lane_begin(S, rRyR);
                fin = false;
            } else {
                sidx = 0;
                lane_store(a, slot0 + i, S);
            }
        }
        const uint64_t msk = __ballot(fin);
        if (fin) {
            if constexpr (CPT > 1) {
                i = next + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(msk >> 32),
                                            __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(msk), 0u)));
                have = i < w1;
                if (have) {
                    lane_load(a, slot0 + i, S);
                    lane_begin(S, rRyR);
                }
            } else {
                have = false;
            }
        }
        next += __popcll(msk);
    }
    for (int s = 0; s < nss; ++s) lane_accumulate(L.acc[s], L.Ls[s], tid);
    __syncthreads();
    for (int s = 0; s < nss; ++s) write_partial(a, L.acc[s], ((m + s) & 1) * a.nblocks + b);
}

// One lane per CRU needs about 100 VGPRs; 4 waves per SIMD keep it, and the
// close in its first blocks, free of spills.
template <int PRNG, int BLOCK, int CPT>
__global__ __launch_bounds__(BLOCK, 4) void k_step_lane(KArgs a, int64_t ssa_step, int32_t nclose, const int64_t *base)
{
    __shared__ union {
        LaneLds<BLOCK, 1> ssa;
        CloseLds<BLOCK> close;
    } sh;
    const int bid = blockIdx.x;
    const int64_t step = base ? *base + ssa_step : ssa_step;
    if (bid < nclose) {
        close_cell<BLOCK>(a, bid, a.dyn[bid], sh.close, ssa_step < 0 ? -1 : step - 1);
        return;
    }
    ssa_block_lane<PRNG, BLOCK, CPT, 1>(a, bid - nclose, step, 1, sh.ssa);
}

// ---------------------------------------------------------------------------
// Persistent stepping of a batch whose SSA blocks can all be resident at once
// (a few cells of up to tens of thousands of CRUs, where a step is short and a
// launch per step leaves the chip waiting on launch latency). One launch runs
// nsteps Euler steps with the cells' CRUs held in registers. The order of the
// work is that of the launch-per-step form: SSA(n) of a cell runs with the
// constants formed by the close of step n - 2, beside the close of step n - 1,
// and the close of step n sums the block partials of SSA(n). Within the
// launch the kernel boundaries are replaced by tags and a counter: each SSA
// block writes its partial and then the partial's tag (the step index + 1);
// the cell's close block waits until every partial of the cell carries the
// tag of the step it closes, and after forming the constants of step n + 2
// it publishes them and raises the cell's `kready` to n + 3, which the SSA
// blocks wait for before step n + 2. (A counter that every SSA block
// incremented would serialise hundreds of same-address atomics per step.)

// Everything that crosses blocks (partials, constants, counters) is written
// and read with device-coherent atomic accesses, and each writer waits for its
// data stores to complete before it moves a counter, so no cache-wide
// writeback or invalidation is issued. The last close runs in the same launch,
// so every step is closed when it returns. The results are bit-identical to
// the launch-per-step form (the same arithmetic, exact flux sums). Every wait
// is bounded: after a.spin_limit polls the waiter sets `timeout`, which every
// other waiter also sees, and all blocks leave.
// ---------------------------------------------------------------------------
constexpr int64_t kSpinLimit = int64_t(1) << 21;   // polls of about 1 us: a wait gives up after seconds

__device__ bool wait_at_least(unsigned long long *p, unsigned long long v, int32_t *timeout, int64_t limit)
{
    for (int64_t it = 0;; ++it) {
        if (ld_coh(p) >= v) return true;
        if (__hip_atomic_load(timeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        if (it >= limit) {
            __hip_atomic_store(timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Counter, published constants and partial tags of every cell before a
// persistent launch from the fully closed state at step step0, whose
// constants of steps step0 and step0 + 1 are in the cell's parity slots. One
// block per cell.
template <class R>
__global__ void k_sync_init(KArgs a, int64_t step0)
{
    using KT = typename LocalState<R>::Consts;
    constexpr int kWords = sizeof(KT) / 8;
    const int c = blockIdx.x;
    if (c == 0 && threadIdx.x == 0) *a.timeout = 0;
    if (c >= a.ncells) return;
    CellSync &X = a.sync[c];
    const CellDyn &D = a.dyn[c];
    for (int t = threadIdx.x; t < 2 * kXchgWords; t += blockDim.x) {
        const int par = t / kXchgWords, w = t % kXchgWords;
        unsigned long long v = 0;
        if (w < kWords) v = reinterpret_cast<const unsigned long long *>(&LocalState<R>::consts(D, par))[w];
        else if (w == kXchgWords - 1) v = static_cast<unsigned long long>(D.stop_step);
        X.k[par][w] = v;
    }
    if (threadIdx.x == 0) X.kready = static_cast<unsigned long long>(step0 + 2);
    const DevCell &C = a.cells[c];
    for (int q = threadIdx.x; q < 2 * C.nblk[kShapeDefault]; q += blockDim.x) {
        const int par = q & 1, blk = q >> 1;
        a.partials[par * a.nblocks + C.blk0[kShapeDefault] + blk].w[PW_ERR] = 0;
    }
}

template <int PRNG, bool DIGEST, class R>
__device__ __forceinline__ void ssa_block_persist(const KArgs &a, int b, int64_t step0, int64_t nsteps,
                                                  LccTableT<R> &T, BlockAcc &acc,
                                                  typename LocalState<R>::Consts &K, int64_t &stop, int &leave)
{
    using LS = LocalState<R>;
    using KT = typename LS::Consts;
    constexpr int kWords = sizeof(KT) / 8;
    static_assert(sizeof(KT) % 8 == 0 && kWords < kXchgWords, "step constants fit the exchange slot");
    const int tid = threadIdx.x;
    const int j = tid & 3;
    const BlockInfo bi = block_info(a, b, kBlock / 4);
    const DevCell &C = a.cells[bi.cell];
    CellSync &X = a.sync[bi.cell];
    const auto sp = load_scalar(&LS::params(C));
    const bool mine = (tid >> 2) < bi.n;
    const int64_t slot = bi.slot + (mine ? tid >> 2 : 0);
    R *const JLCC = LS::jlcc(a);
    double ca = 0.0;
    R jl = R(0);
    uint64_t w = 0;
    CruQ q{};
    Digest dg{0, 0};
    if (mine) {
        ca = a.CaSS[slot * 4 + j];
        jl = JLCC[slot * 4 + j];
        w = a.sub[slot * 4 + j];
        q.jsr = a.CaJSR[slot];
        q.r0 = a.rng[slot * 4];
        q.r1 = a.rng[slot * 4 + 1];
        q.r2 = a.rng[slot * 4 + 2];
        q.r3 = a.rng[slot * 4 + 3];
        if (DIGEST) {
            dg.count = a.dig[slot * 2];
            dg.hash = a.dig[slot * 2 + 1];
        }
    }
    int changed = 0;
    const R dt = static_cast<R>(a.dt);
    for (int64_t k = 0; k < nsteps; ++k) {
        const int64_t n = step0 + k;
        const int ks = static_cast<int>(n & 1);
        if (tid == 0)
            leave = wait_at_least(&X.kready, static_cast<unsigned long long>(n + 1), a.timeout, a.spin_limit) ? 0 : 1;
        __syncthreads();
        if (leave) break;
        // the step's constants and the cell's stop step, published by its close
        for (int t = tid; t < kWords; t += kBlock) reinterpret_cast<unsigned long long *>(&K)[t] = ld_coh(&X.k[ks][t]);
        if (tid == 0) stop = static_cast<int64_t>(ld_coh(&X.k[ks][kXchgWords - 1]));
        acc_zero(acc);
        __syncthreads();
        load_lcc_table(K, T);
        __syncthreads();
        if (mine && n < stop) {
            const QuadOut o = ssa_step_quad<PRNG, DIGEST>(ca, jl, w, q, sp, quad_consts(K), T, dt, dg, static_cast<uint32_t>(n & 0xffff), j);
            changed |= o.changed;
            quad_add(acc, j, o, o.iters);
        }
        __syncthreads();
        post_partial(a.partials[ks * a.nblocks + b], tid, tid < PW_N ? acc_word(acc, tid) : 0, n);
    }
    if (mine) {
        a.CaSS[slot * 4 + j] = ca;
        if (changed) {
            JLCC[slot * 4 + j] = jl;
            a.sub[slot * 4 + j] = w;
        }
        if (j == 0) {
            a.CaJSR[slot] = q.jsr;
            a.rng[slot * 4] = q.r0;
            a.rng[slot * 4 + 1] = q.r1;
            a.rng[slot * 4 + 2] = q.r2;
            a.rng[slot * 4 + 3] = q.r3;
            if (DIGEST) {
                a.dig[slot * 2] = dg.count;
                a.dig[slot * 2 + 1] = dg.hash;
            }
        }
    }
}

// After the close of step n: publish the constants of step n + 2 it formed
// (the cell's parity slot (n + 2) & 1) and the cell's stop step, then raise
// the cell's counter to n + 3. The counter moves after the other stores have
// completed. A cell that had already stopped publishes its unchanged slot,
// so that every waiter goes on (and finds the stop step). Every thread of the
// block takes part.
template <class R>
__device__ __forceinline__ void publish_consts(CellSync &X, const CellDyn &D, int64_t n)
{
    using KT = typename LocalState<R>::Consts;
    constexpr int kWords = sizeof(KT) / 8;
    const int par = static_cast<int>((n + 2) & 1);
    for (int t = threadIdx.x; t < kWords; t += blockDim.x)
        st_coh(&X.k[par][t], reinterpret_cast<const unsigned long long *>(&LocalState<R>::consts(D, par))[t]);
    if (threadIdx.x == 0) st_coh(&X.k[par][kXchgWords - 1], static_cast<unsigned long long>(D.stop_step));
    stores_done();
    __syncthreads();
    if (threadIdx.x == 0) st_coh(&X.kready, static_cast<unsigned long long>(n + 3));
}

// Wave 0 of a close block waits until every partial of the cell for step n
// carries the tag n + 1 (each lane polls its share, the wave votes). The
// partials of a parity are cleared before the launch (k_sync_init), and
// SSA(n + 2), which writes the same slots, waits for the close of step n.
__device__ bool wait_partials(const KArgs &a, const DevCell &C, int64_t n, int32_t *timeout, int64_t limit)
{
    const int nblk = C.nblk[kShapeDefault];
    const unsigned long long *base =
        reinterpret_cast<const unsigned long long *>(a.partials + (n & 1) * a.nblocks + C.blk0[kShapeDefault]);
    const int32_t want = static_cast<int32_t>(n + 1);
    for (int64_t it = 0;; ++it) {
        bool ok = true;
        for (int q = threadIdx.x; q < nblk; q += kWave)
            ok = ok && static_cast<int32_t>(ld_coh(base + q * PW_N + PW_ERR) >> 32) == want;
        if (__all(ok)) return true;
        if (__hip_atomic_load(timeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        if (it >= limit) {
            if (threadIdx.x == 0) __hip_atomic_store(timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// The close block of one cell in the persistent kernel: keeps the cell's
// dynamic state in LDS for the launch (it is its only writer), closes steps
// step0 .. step0 + nsteps - 1 in turn, each once every SSA block of the cell
// has written its partial of that step, and publishes the constants it
// formed.
template <class R>
__device__ __forceinline__ void close_persist(const KArgs &a, int cell, int64_t step0, int64_t nsteps, CellDyn &Dl,
                                              CloseLds<kBlock> &sh, int &leave)
{
    static_assert(sizeof(CellDyn) % 8 == 0, "the dynamic state is whole 8-byte words");
    constexpr int kDynWords = sizeof(CellDyn) / 8;
    const DevCell &C = a.cells[cell];
    CellSync &X = a.sync[cell];
    unsigned long long *g = reinterpret_cast<unsigned long long *>(&a.dyn[cell]);
    unsigned long long *l = reinterpret_cast<unsigned long long *>(&Dl);
    for (int t = threadIdx.x; t < kDynWords; t += blockDim.x) l[t] = g[t];
    __syncthreads();
    for (int64_t k = 0; k < nsteps; ++k) {
        const int64_t n = step0 + k;
        if (threadIdx.x < kWave) {
            const bool ok = wait_partials(a, C, n, a.timeout, a.spin_limit);
            if (threadIdx.x == 0) leave = ok ? 0 : 1;
        }
        __syncthreads();
        if (leave) break;
        close_cell<kBlock, true>(a, cell, Dl, sh);
        __syncthreads();
        publish_consts<R>(X, Dl, n);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kDynWords; t += blockDim.x) g[t] = l[t];
}

// The first ncells blocks close (four waves, one for each role), the others are
// the SSA blocks of the default shape (64 CRUs, a quad of lanes per CRU). At the
// waves per SIMD of k_step the two kinds in one loop each spill: 80 to 85 VGPRs
// in FP64, 123 FP32-local.
template <int PRNG, bool DIGEST, class R>
__global__ __launch_bounds__(kBlock, kWavesPerSimd<R>) void k_persist(KArgs a, int64_t step0, int64_t nsteps)
{
    __shared__ LccTableT<R> T;
    __shared__ CloseLds<kBlock> csh;
    __shared__ BlockAcc acc;
    __shared__ typename LocalState<R>::Consts K;
    __shared__ CellDyn Dl;
    __shared__ int64_t stop;
    __shared__ int leave;
    const int bid = blockIdx.x;
    if (bid < a.ncells) {
        close_persist<R>(a, bid, step0, nsteps, Dl, csh, leave);
        return;
    }
    ssa_block_persist<PRNG, DIGEST, R>(a, bid - a.ncells, step0, nsteps, T, acc, K, stop, leave);
}

// ---------------------------------------------------------------------------
// Two Euler steps per launch, one lane per CRU (FP32-local). A launch runs
// SSA(m) and SSA(m + 1) for every CRU with its state held in registers
// between them, so the state crosses HBM once per two steps. SSA(m) needs the
// constants formed by the close of step m - 2 and SSA(m + 1) those of the
// close of step m - 1; neither close can run before every SSA block of the
// previous launch has written its partial, so both run just before the
// launch, in their own kernel (k_close_cells, one block of four waves per cell,
// a wave for each role of the close).
// A lane that has finished step m of its CRU goes on to step m + 1 of the
// same CRU (reading that step's constants from its LDS slot), and only then
// stores the CRU and takes the next one of its wave's range. Each lane sums
// the outputs of each step separately in finishing order; the per-wave sums
// are added exactly into one block partial per step. The launch sequence of a
// call (host, launch_steps_pair): SSA(step0), SSA(step0 + 1) with no closes
// before them (the call starts with every step closed); then the closes of
// the two steps before each later pair; an odd last step runs alone after one
// close; a last close kernel closes the rest. A cell that fails in either
// close stops as with one step per launch: SSA(s) runs while s < stop_step,
// which the closes before the launch have set. With one CRU per lane (CPT =
// 1) a lane's sums are its CRU's own outputs, so the results are bit-identical
// to one step per launch; with refilled lanes the order of a lane's FP64 sums
// depends on which CRUs it ran, which can change their rounding.
// ---------------------------------------------------------------------------
// What bounds it on 12.8 M CRUs is HBM: the state in and out, 207 B per CRU
// measured, at 4.4 TB/s (a copy of this size reaches 4.9), 318 us per step.
// Before its parameters lay in scalar registers and the step's constants were
// read at the top of a trip (chosen in LDS, each choice was a branch) it took
// 418. 98 VGPRs with four or more CRUs per lane, where a fifth wave per SIMD
// changes nothing (321); with one or two it does (1 per lane 372 and 327, 2
// per lane 335 and 311 us).
template <int PRNG, int BLOCK, int CPT>
__global__ __launch_bounds__(BLOCK, CPT <= 2 ? 5 : 4) void k_step_lane2(KArgs a, int64_t m, int32_t nss)
{
    __shared__ LaneLds<BLOCK, 2> sh;
    ssa_block_lane<PRNG, BLOCK, CPT, 2>(a, blockIdx.x, m, nss, sh);
}

// One or two (ncl) consecutive closes of every cell, one block of four waves per cell (the
// two-steps-per-launch sequence), one wave for each of the close's roles. At
// 4 waves per SIMD the blocks of 1,024 cells are resident at once, and share the
// issue of their compute units: two closes of 64 cells take 10.4 us, of 256
// 12.2, of 512 19.5, of 1,024 33.
__global__ __launch_bounds__(kBlock, 4) void k_close_cells(KArgs a, int32_t ncl)
{
    __shared__ CloseLds<kBlock> sh;
    const int cell = blockIdx.x;
    close_cell<kBlock>(a, cell, a.dyn[cell], sh);
    if (ncl < 2) return;
    __syncthreads();   // written out, not a loop: a loop keeps the close's constants in registers across its turns and spills
    close_cell<kBlock>(a, cell, a.dyn[cell], sh);
}

// ---------------------------------------------------------------------------
// FP64 with one lane per CRU (gw_ssa.h, lane64_*), one or two Euler steps per
// launch, refilled from CPT CRUs per lane as in the FP32-local kernels. It
// replaces the quads where a launch has more CRUs than the GPU can hold in
// quads several times over (run_config): there a wave's instructions count,
// and this form needs about half as many per CRU and step.
//
// Events wait: about 3% of the iterations end in an event, so in nearly every
// trip of a wave of 64 CRUs one or two lanes would take the event path, a
// third as long as the rest of the trip. A lane whose iteration ends in an event
// leaves its CRU as it was and runs the same iteration again (it would idle
// otherwise), until event_batch lanes of the wave hold an event, or no other
// lane made progress, or no fresh CRU is left to keep the others busy; then
// all of them commit at once. 12.8 M CRUs, 4 per lane: 552, 551, 542 and 543
// us per step with batches of 1, 4, 8 and 16 events (479 and then 463 since).
//
// Flux sums: a CRU's four outputs are split into three 43-bit limbs in FP64
// arithmetic, truncated at 2^-80 like fx_add, and added as whole numbers into
// sixteen copies of the block accumulators in LDS (below 2^53, so exact in
// FP64, whatever the order).
// ---------------------------------------------------------------------------
constexpr int kAccCopies = 16;

struct Lane64Acc {
    double limb[12][kAccCopies];
    unsigned long long ints[kAccCopies];   // iterations in the low 40 bits, open ClCh above
    int open[kAccCopies];
    int err;
};

template <int NSS>
struct Lane64Lds {
    StepConsts K[NSS];
    Lane64Acc acc[NSS];
};

// Adds v in limbs; false if it is not below 2^24 in magnitude (then it adds nothing).
__device__ __forceinline__ bool lane64_add(Lane64Acc &A, int q, int copy, double v)
{
    double lo, mid, hi;
    const bool ok = limb_split(v, lo, mid, hi);
    unsafeAtomicAdd(&A.limb[3 * q][copy], lo);
    unsafeAtomicAdd(&A.limb[3 * q + 1][copy], mid);
    unsafeAtomicAdd(&A.limb[3 * q + 2][copy], hi);
    return ok;
}

__device__ __forceinline__ void lane64_output(Lane64Acc &A, const Lane64State &S, double Jxfer, double Jtr, bool ok)
{
    const int copy = threadIdx.x & (kAccCopies - 1);
    ok &= lane64_add(A, 0, copy, Jxfer);
    ok &= lane64_add(A, 1, copy, Jtr);
    ok &= lane64_add(A, 2, copy, S.jl[0] + S.jl[1] + S.jl[2] + S.jl[3]);
    lane64_add(A, 3, copy, S.Jrel[0] + S.Jrel[1] + S.Jrel[2] + S.Jrel[3]);   // the range of Jrel is not checked
    int open = 0, clch = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        open += ryr_get(S.w[j], 2) + ryr_get(S.w[j], 3);
        clch += sub_cl(S.w[j]);
    }
    atomicAdd(&A.ints[copy], static_cast<unsigned long long>(clch) << 40 | S.iters);
    atomicAdd(&A.open[copy], open);
    if (!ok) A.err = 1;
}

__device__ __forceinline__ void lane64_load(const KArgs &a, int64_t slot, Lane64State &S)
{
    const double2 *pc = reinterpret_cast<const double2 *>(a.CaSS + slot * 4);
    const double2 c01 = pc[0], c23 = pc[1];
    const double2 *pj = reinterpret_cast<const double2 *>(a.JLCC + slot * 4);
    const double2 j01 = pj[0], j23 = pj[1];
    const ulonglong2 *pw = reinterpret_cast<const ulonglong2 *>(a.sub + slot * 4);
    const ulonglong2 w01 = pw[0], w23 = pw[1];
    const ulonglong2 *pr = reinterpret_cast<const ulonglong2 *>(a.rng + slot * 4);
    const ulonglong2 r01 = pr[0], r23 = pr[1];
    S.q.jsr = a.CaJSR[slot];
    S.ca[0] = c01.x; S.ca[1] = c01.y; S.ca[2] = c23.x; S.ca[3] = c23.y;
    S.jl[0] = j01.x; S.jl[1] = j01.y; S.jl[2] = j23.x; S.jl[3] = j23.y;
    S.w[0] = w01.x; S.w[1] = w01.y; S.w[2] = w23.x; S.w[3] = w23.y;
    S.q.r0 = r01.x; S.q.r1 = r01.y; S.q.r2 = r23.x; S.q.r3 = r23.y;
    S.changed = 0;
}

__device__ __forceinline__ void lane64_store(const KArgs &a, int64_t slot, const Lane64State &S)
{
    double2 *qc = reinterpret_cast<double2 *>(a.CaSS + slot * 4);
    qc[0] = make_double2(S.ca[0], S.ca[1]);
    qc[1] = make_double2(S.ca[2], S.ca[3]);
    if (S.changed) {   // the channel words and JLCC change only at events and re-splits
        double2 *qj = reinterpret_cast<double2 *>(a.JLCC + slot * 4);
        qj[0] = make_double2(S.jl[0], S.jl[1]);
        qj[1] = make_double2(S.jl[2], S.jl[3]);
        ulonglong2 *qw = reinterpret_cast<ulonglong2 *>(a.sub + slot * 4);
        qw[0] = make_ulonglong2(S.w[0], S.w[1]);
        qw[1] = make_ulonglong2(S.w[2], S.w[3]);
    }
    ulonglong2 *qr = reinterpret_cast<ulonglong2 *>(a.rng + slot * 4);
    qr[0] = make_ulonglong2(S.q.r0, S.q.r1);
    qr[1] = make_ulonglong2(S.q.r2, S.q.r3);
    a.CaJSR[slot] = S.q.jsr;
}

// SSA(m .. m + nss - 1) of block b (one wave, 64 * CPT CRUs of one cell), nss <= NSS.
template <int PRNG, int CPT, int NSS>
__device__ __forceinline__ void ssa_block_lane64(const KArgs &a, int b, int64_t m, int nss, Lane64Lds<NSS> &P)
{
    constexpr int kMap = shape_of_crus(kWave * CPT);
    static_assert(crus_per_block(kMap) == kWave * CPT, "CRUs per block must be 16 << map");
    constexpr int kWords = sizeof(StepConsts) / 4;
    const int lane = threadIdx.x;
    const BlockInfo bi = block_info(a, b, kWave * CPT);
    const DevCell &C = a.cells[bi.cell];
    const CellDyn &D = a.dyn[bi.cell];
#pragma unroll
    for (int s = 0; s < NSS; ++s) {
        if (s < nss)
            for (int t = lane; t < kWords; t += kWave)
                reinterpret_cast<uint32_t *>(&P.K[s])[t] = reinterpret_cast<const uint32_t *>(&D.k[(m + s) & 1])[t];
        for (int t = lane; t < static_cast<int>(sizeof(Lane64Acc) / 4); t += kWave) reinterpret_cast<uint32_t *>(&P.acc[s])[t] = 0;
    }
    __syncthreads();
    const double dt = a.dt;
    const double rRyR = C.sp.rRyR;
    const bool plain = load_scalar(&C.plain) != 0;
    const int64_t stop = D.stop_step;
    const bool run1 = nss > 1 && m + 1 < stop;
    const int w1 = bi.n;   // CRUs of the range
    const int64_t slot0 = bi.slot;
    int i = lane;
    int next = kWave;   // first CRU of the range not yet taken (wave-uniform)
    bool have = i < w1 && m < stop;
    int sidx = 0;       // the step (0: m, 1: m + 1) this lane's CRU is in
    Lane64State S;
    if (have) {
        lane64_load(a, slot0 + i, S);
        lane64_begin(S, rRyR);
    }
    while (__ballot(have)) {
        const SsaParams *spp = &C.sp;
        asm volatile("" : "+s"(spp));   // read again in each trip: held over the loop they would not fit
        const SsaParams sp = load_scalar(spp);
        Lane64Try X;
        bool ev = false;
        if (have) {
            lane64_try<PRNG>(S, X, sp, P.K[sidx], P.K[sidx].lcc, dt, plain);
            ev = !X.last;
        }
        const uint64_t m_ev = __ballot(ev);
        const uint64_t m_last = __ballot(have && !ev);
        const bool go = __popcll(m_ev) >= event_batch(CPT) || m_last == 0 || next >= w1;   // wave-uniform
        bool fin = have && !ev;
        bool ok = true;
        if (have && (go || !ev)) {
            double old[4];
            uint64_t w_pre[4];
            lane64_commit<PRNG>(S, X, sp, old, w_pre);
            if (ev && go) {
                if (S.iters >= kMaxItersPerStep) {   // no physical state gets here; stop instead of spinning
                    ok = false;
                    fin = true;
                } else if (!lane64_event<PRNG>(S, X, sp, P.K[sidx], P.K[sidx].lcc, old, w_pre)) {
                    P.acc[sidx].err = 1;
                }
            }
        }
        if (fin) {
            lane64_output(P.acc[sidx], S, X.Jxfer, X.Jtr, ok);
            if (NSS > 1 && sidx == 0 && run1) {   // the same CRU, next step
                sidx = 1;
                lane64_begin(S, rRyR);
                fin = false;
            } else {
                sidx = 0;
                lane64_store(a, slot0 + i, S);
            }
        }
        const uint64_t msk = __ballot(fin);
        if (fin) {
            if constexpr (CPT > 1) {
                i = next + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(msk >> 32),
                                            __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(msk), 0u)));
                have = i < w1;
                if (have) {
                    lane64_load(a, slot0 + i, S);
                    lane64_begin(S, rRyR);
                }
            } else {
                have = false;
            }
        }
        next += __popcll(msk);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NSS; ++s) {
        if (s >= nss || lane >= PW_N) continue;
        const Lane64Acc &A = P.acc[s];
        uint64_t v = 0;
        if (lane < PW_ITERS) {
            double d = 0.0;
            for (int k = 0; k < kAccCopies; ++k) d += A.limb[lane][k];   // whole numbers below 2^53
            v = static_cast<uint64_t>(static_cast<int64_t>(d));
        } else if (lane == PW_ERR) {
            v = A.err != 0;
        } else {
            for (int k = 0; k < kAccCopies; ++k)
                v += lane == PW_OPEN ? static_cast<uint64_t>(static_cast<int64_t>(A.open[k]))
                   : lane == PW_CLCH ? A.ints[k] >> 40 : A.ints[k] & ((1ULL << 40) - 1);
        }
        a.partials[((m + s) & 1) * a.nblocks + b].w[lane] = v;
    }
}

// One step, the closes of the step before in the first blocks (as k_step).
// 147 VGPRs (149 with two steps per launch): three waves per SIMD (at four, 23 spilled and 12.8 M CRUs took 649
// us per step against 542 then). Issue of vector instructions bounds them: 17.2
// per CRU and step, 78% of the time (the quads: 50.7, 87%).
template <int PRNG, int CPT>
__global__ __launch_bounds__(kWave, 3) void k_step_lane64(KArgs a, int64_t ssa_step, int32_t nclose, const int64_t *base)
{
    __shared__ union {
        Lane64Lds<1> ssa;
        CloseLds<kWave> close;
    } sh;
    const int bid = blockIdx.x;
    const int64_t step = base ? *base + ssa_step : ssa_step;
    if (bid < nclose) {
        close_cell<kWave>(a, bid, a.dyn[bid], sh.close, ssa_step < 0 ? -1 : step - 1);
        return;
    }
    ssa_block_lane64<PRNG, CPT, 1>(a, bid - nclose, step, 1, sh.ssa);
}

// One or two (nss) steps, their closes before them in k_close_cells.
template <int PRNG, int CPT>
__global__ __launch_bounds__(kWave, 3) void k_step2_lane64(KArgs a, int64_t m, int32_t nss)
{
    __shared__ Lane64Lds<2> sh;
    ssa_block_lane64<PRNG, CPT, 2>(a, blockIdx.x, m, nss, sh);
}

// Graph bookkeeping: the step index a replayed chunk starts at.
__global__ void k_set_base(int64_t *base, int64_t v) { *base = v; }
__global__ void k_advance_base(int64_t *base, int64_t k) { *base += k; }

// Frozen-globals replay: nsteps SSA steps in one launch.
template <int PRNG, bool DIGEST, class R>
__global__ __launch_bounds__(kBlock, kWavesPerSimd<R>) void k_ssa(KArgs a, int64_t step0, int64_t nsteps)
{
    __shared__ LccTableT<R> T;
    __shared__ BlockAcc acc;
    ssa_block<PRNG, DIGEST, R, kBlock>(a, blockIdx.x, step0, nsteps, T, acc);
}

// Close a frozen replay of nsteps: sums of the last step, clock advanced as
// t += dt per step (src/pyGW.hpp:116).
__global__ void k_frozen_close(KArgs a, int64_t step0, int64_t nsteps)
{
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= a.ncells) return;
    const DevCell &C = a.cells[cell];
    CellDyn &D = a.dyn[cell];
    const Partial *src = a.partials + (step0 & 1) * a.nblocks + C.blk0[a.shape];
    uint64_t w[PW_N] = {};
    for (int b = 0; b < C.nblk[a.shape]; ++b)
        for (int k = 0; k < PW_N; ++k) w[k] += src[b].w[k];
    auto flux = [&](int q) { return fx_to_double(limbs_fx(w[3 * q], w[3 * q + 1], w[3 * q + 2])); };
    if (a.iters_total) atomicAdd(a.iters_total, static_cast<unsigned long long>(w[PW_ITERS]));
    if (w[PW_ERR] && D.status == 0) D.status = GW_E_RANGE;
    D.sums[0] = flux(2); D.sums[1] = flux(0); D.sums[2] = flux(1);
    D.sums[3] = static_cast<double>(static_cast<int64_t>(w[PW_CLCH]));
    D.sums[4] = static_cast<double>(static_cast<int64_t>(w[PW_OPEN])); D.sums[5] = flux(3);
    for (int64_t s = 0; s < nsteps; ++s) D.t += a.dt;
    D.step += nsteps;
    if (D.status != 0 && D.stop_step > D.step) D.stop_step = D.step;
}

// A piece of one cell's state on its way between device and host, in pinned
// host memory that the kernels below write and read themselves: the CRU state
// as the device packs it, 72 bytes per CRU, and JLCC where it is asked for,
// with the cell's status and globals in front. The host expands it to the
// row-major layout (GWCRUState, src/pyGW.cpp:78-87).
struct PieceHead {
    int64_t status;
    gw_globals_t g;
};
constexpr size_t kPieceHead = 512;
static_assert(sizeof(PieceHead) <= kPieceHead && sizeof(gw_globals_t) % 8 == 0, "the head of a piece");

struct PieceView {
    PieceHead *head;
    double *CaSS;
    uint64_t *sub;
    double *CaJSR;
    void *JLCC;   // doubles, floats where an FP32-local batch writes it
};

__host__ __device__ inline PieceView piece_view(void *base, int64_t m)
{
    PieceView v;
    char *p = static_cast<char *>(base);
    v.head = reinterpret_cast<PieceHead *>(p); p += kPieceHead;
    v.CaSS = reinterpret_cast<double *>(p); p += 4 * m * 8;
    v.sub = reinterpret_cast<uint64_t *>(p); p += 4 * m * 8;
    v.CaJSR = reinterpret_cast<double *>(p); p += (m + 1) / 2 * 16;
    v.JLCC = p;
    return v;
}
constexpr size_t piece_bytes(int64_t m) { return kPieceHead + static_cast<size_t>(m) * 104 + 8; }

// The status and globals of a cell, by the first block of a piece's kernel.
__device__ __forceinline__ void write_head(const CellDyn &D, PieceHead *head)
{
    static_assert(sizeof(gw_globals_t) / 8 <= kBlock, "a lane per word");
    if (blockIdx.x != 0) return;
    const uint64_t *g = reinterpret_cast<const uint64_t *>(&D.g);
    if (threadIdx.x < sizeof(gw_globals_t) / 8) reinterpret_cast<uint64_t *>(&head->g)[threadIdx.x] = g[threadIdx.x];
    if (threadIdx.x == 0) head->status = D.status;
}

// CRUs i0 .. i0 + m - 1 of a cell (i0 even), one 16-byte word per lane: whole
// lines go over the link, which bounds it.
int64_t piece_words(int64_t m, int jlcc, bool f32)
{
    return 4 * m + (m + 1) / 2 + (jlcc ? (f32 ? m : 2 * m) : 0);
}
__global__ __launch_bounds__(kBlock) void k_get_piece(KArgs a, int cell, int64_t i0, int64_t m, int jlcc, void *base)
{
    const DevCell &C = a.cells[cell];
    const PieceView v = piece_view(base, m);
    const int64_t slot = C.slot0 + i0;
    write_head(a.dyn[cell], v.head);
    auto put = [](void *dst, const void *src, int64_t w) {
        static_cast<ulonglong2 *>(dst)[w] = static_cast<const ulonglong2 *>(src)[w];
    };
    int64_t w = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (w < 2 * m) return put(v.CaSS, a.CaSS + slot * 4, w);
    if ((w -= 2 * m) < 2 * m) return put(v.sub, a.sub + slot * 4, w);
    if ((w -= 2 * m) < (m + 1) / 2) return put(v.CaJSR, a.CaJSR + slot, w);   // an odd last one with its padding slot
    w -= (m + 1) / 2;
    if (!jlcc) return;
    if (a.JLCCf) {
        if (w < m) put(v.JLCC, a.JLCCf + slot * 4, w);
    } else if (w < 2 * m) {
        put(v.JLCC, a.JLCC + slot * 4, w);
    }
}

// The same CRUs from a piece whose JLCC, where there is one, is in doubles.
__global__ __launch_bounds__(kBlock) void k_put_piece(KArgs a, int cell, int64_t i0, int64_t m, int has_jlcc, void *base)
{
    const DevCell &C = a.cells[cell];
    const PieceView v = piece_view(base, m);
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;   // a subunit
    if (i >= 4 * m) return;
    const int64_t slot = C.slot0 + i0;
    a.CaSS[slot * 4 + i] = v.CaSS[i];
    a.sub[slot * 4 + i] = v.sub[i];
    st_jlcc(a, slot * 4 + i, has_jlcc ? static_cast<const double *>(v.JLCC)[i] : 0.0);
    if (i < m) a.CaJSR[slot + i] = v.CaJSR[i];
}

// One cell's CRU state in the reduced record encoding (gw_cru_state_reduced_t),
// 40 bytes per CRU.
struct ReducedView {
    PieceHead *head;
    float *CaSS, *CaJSR;
    int16_t *RyR;
    int8_t *LCC;
    uint8_t *LCCi, *ClCh;
};

__host__ __device__ inline ReducedView reduced_view(void *base, int64_t m)
{
    ReducedView v;
    char *p = static_cast<char *>(base);
    v.head = reinterpret_cast<PieceHead *>(p); p += kPieceHead;
    v.CaSS = reinterpret_cast<float *>(p); p += 4 * m * 4;
    v.RyR = reinterpret_cast<int16_t *>(p); p += 4 * m * 2;
    v.CaJSR = reinterpret_cast<float *>(p); p += m * 4;
    v.LCC = reinterpret_cast<int8_t *>(p); p += 4 * m;
    v.LCCi = reinterpret_cast<uint8_t *>(p); p += 4 * m;
    v.ClCh = reinterpret_cast<uint8_t *>(p);
    return v;
}

// RyR_state_to_int16 (src/utils.py:8-22) of one subunit word: a lumped pair
// with a negative member counts as its sum in the pair's first member.
__device__ __forceinline__ int16_t ryr_code(uint64_t w)
{
    const int r1 = ryr_get(w, 0), r2 = ryr_get(w, 1), r3 = ryr_get(w, 2), r4 = ryr_get(w, 3);
    const int r5 = ryr_get(w, 4), r6 = ryr_get(w, 5);
    const bool neg34 = r3 < 0 || r4 < 0, neg56 = r5 < 0 || r6 < 0;
    const int s3 = neg34 ? r3 + r4 : r3, s4 = neg34 ? 0 : r4, s5 = neg56 ? r5 + r6 : r5;
    return static_cast<int16_t>(r1 + 6 * r2 + 36 * s3 + 216 * s4 + 1296 * s5);
}

__global__ __launch_bounds__(kBlock) void k_get_piece_reduced(KArgs a, int cell, int64_t i0, int64_t m, void *base)
{
    const DevCell &C = a.cells[cell];
    const ReducedView v = reduced_view(base, m);
    write_head(a.dyn[cell], v.head);
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= m) return;
    const int64_t slot = C.slot0 + i0 + i;
    float ca[4];
    short ry[4];
    signed char lcc[4];
    unsigned char y[4], cl[4];
    for (int j = 0; j < 4; ++j) {
        ca[j] = static_cast<float>(ld_cass(a, slot * 4 + j));
        const uint64_t w = a.sub[slot * 4 + j];
        lcc[j] = static_cast<int8_t>(sub_lcc(w));
        y[j] = static_cast<uint8_t>(sub_y(w));
        cl[j] = static_cast<uint8_t>(sub_cl(w));
        ry[j] = ryr_code(w);
    }
    reinterpret_cast<float4 *>(v.CaSS)[i] = make_float4(ca[0], ca[1], ca[2], ca[3]);
    reinterpret_cast<short4 *>(v.RyR)[i] = make_short4(ry[0], ry[1], ry[2], ry[3]);
    reinterpret_cast<char4 *>(v.LCC)[i] = make_char4(lcc[0], lcc[1], lcc[2], lcc[3]);
    reinterpret_cast<uchar4 *>(v.LCCi)[i] = make_uchar4(y[0], y[1], y[2], y[3]);
    reinterpret_cast<uchar4 *>(v.ClCh)[i] = make_uchar4(cl[0], cl[1], cl[2], cl[3]);
    v.CaJSR[i] = static_cast<float>(ld_cajsr(a, slot));
}

__global__ void k_reset_obs(CellDyn *dyn, int ncells)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    gw_cell_obs_t &o = dyn[c].obs;
    const double V = dyn[c].g.V;
    o.peak_V = -1e300; o.min_V = 1e300; o.peak_Cai = -1e300; o.peak_ICaL_neg = 1e300;
    o.sum_open_RyR_frac = 0; o.int_Jrel = 0; o.n_steps = 0;
    o.v_prev = V; o.apd_v_rest = V; o.apd_v_peak = V; o.apd_t_up = -1.0;
    o.apd90_last = -1.0; o.apd90_prev = -1.0; o.alt_sum = 0; o.alt_count = 0; o.beats_done = 0;
}

// The post-hoc L-type Ca and Ca-activated Cl currents of src/model.py:414-481
// at each cell's current state (one block per cell): ICaL from the open LCCs
// (state 6 or 12 with the y gate open) at the instantaneous V and CaSS,
//   ICaL = CRU_factor PCaL/CSA 4F (VF/RT)/(e^{2VF/RT} - 1) sum_open (CaSS e^{2VF/RT} - 0.341 Cao) 1e9,
// and Ito2 from the open ClCh,
//   Ito2 = CRU_factor Pto2/CSA F (VF/RT)/(e^{-VF/RT} - 1) n_open (Clcyto e^{-VF/RT} - Clo) 1e9.
// The sum of CaSS over open channels is exact (fixed point), so the result
// does not depend on the launch. At V = 0 the factors take their limits,
// 1/2 and -1, where the reference divides 0/0 (deviation D4). out[2c] = ICaL,
// out[2c + 1] = Ito2 of cell c.
__global__ void k_posthoc_currents(KArgs a, double *out)
{
    __shared__ FluxTotals red[kBlock];
    const int cell = blockIdx.x;
    const DevCell &C = a.cells[cell];
    const CellDyn &D = a.dyn[cell];
    FluxTotals mine;
    totals_zero(mine);
    for (int64_t i = threadIdx.x; i < C.n_cru; i += kBlock) {
        const int64_t slot = C.slot0 + i;
        double s = 0.0;
        for (int j = 0; j < 4; ++j) {
            const uint64_t w = a.sub[slot * 4 + j];
            const int L = sub_lcc(w);
            if ((L == 6 || L == 12) && sub_y(w)) {
                s += ld_cass(a, slot * 4 + j);
                mine.open += 1;
            }
            mine.clch += sub_cl(w);
        }
        mine.err |= fx_add(mine.jlcc, s);
    }
    block_reduce<kBlock>(red, mine);
    if (threadIdx.x != 0) return;
    const FluxTotals &t = red[0];
    const gw_params_t &p = C.p;
    const double V = D.g.V;
    const double x = V * C.c.F_RT;
    const double e2 = gw::exp(2.0 * x), em = gw::exp(-x);
    const double f2 = (V == 0.0) ? 0.5 : x / (e2 - 1.0);
    const double fm = (V == 0.0) ? -1.0 : x / (em - 1.0);
    const double n_open = static_cast<double>(t.open);
    out[2 * cell] = C.c.CRU_factor * (p.PCaL / p.CSA) * (4.0 * kFaraday) * f2 *
                    (fx_to_double(t.jlcc) * e2 - 0.341 * p.Cao * n_open) * 1e9;
    out[2 * cell + 1] = C.c.CRU_factor * (p.Pto2 / p.CSA) * kFaraday * fm *
                        static_cast<double>(t.clch) * (p.Clcyto * em - p.Clo) * 1e9;
}

// Status and trace row count of every cell into out[0..n) and out[n..2n),
// and the persistent kernel's timeout flag into out[2n] (pinned host memory).
__global__ void k_gather_dyn(const CellDyn *dyn, int ncells, const int32_t *timeout, int64_t *out)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c == 0) out[2 * ncells] = *timeout;
    if (c >= ncells) return;
    out[c] = dyn[c].status;
    out[ncells + c] = dyn[c].trace_rows;
}

// Words w0 .. w0 + n - 1 of every cell's dynamic state (pinned host memory).
__global__ void k_export_dyn(const CellDyn *dyn, int ncells, int w0, int n, uint64_t *out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<int64_t>(ncells) * n) return;
    const int64_t c = i / n;
    out[i] = reinterpret_cast<const uint64_t *>(dyn + c)[w0 + static_cast<int>(i - c * n)];
}

__global__ void k_zero_trace_rows(CellDyn *dyn, int ncells)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < ncells) dyn[c].trace_rows = 0;
}

// One cell whose globals, CRU state or stimulus changed after it has been
// stepped: the derivatives and SSA constants of its current step are formed
// again from its state (prepare_step + lookahead_consts, as the constructor
// does at step 0), keeping its clock, step index and observables; no other
// cell is touched. With resum != 0 (a new CRU state) the sums read from the
// CRU state -- JLCC, ClCh, open RyRs -- are formed again from it, while Jxfer
// and Jtr keep the values of the cell's last SSA: in the reference those are
// per-CRU arrays only the SSA writes (GW.tpp:47-62), not part of GWCRUState.
__global__ void k_refresh_cell(KArgs a, int cell, int resum)
{
    __shared__ FluxTotals red[kBlock];
    const DevCell &C = a.cells[cell];
    CellDyn &D = a.dyn[cell];
    if (resum) {
        FluxTotals mine;
        totals_zero(mine);
        for (int64_t i = threadIdx.x; i < C.n_cru; i += kBlock) {
            const int64_t slot = C.slot0 + i;
            double jl[4];
            for (int j = 0; j < 4; ++j) jl[j] = ld_jlcc(a, slot * 4 + j);
            mine.err |= fx_add(mine.jlcc, jl[0] + jl[1] + jl[2] + jl[3]);
            for (int j = 0; j < 4; ++j) {
                const uint64_t w = a.sub[slot * 4 + j];
                mine.clch += sub_cl(w);
                mine.open += ryr_get(w, 2) + ryr_get(w, 3);
            }
        }
        block_reduce<kBlock>(red, mine);
    }
    if (threadIdx.x != 0) return;
    if (resum) {
        D.sums[0] = fx_to_double(red[0].jlcc);
        D.sums[3] = static_cast<double>(red[0].clch);
        D.sums[4] = static_cast<double>(red[0].open);
        if (red[0].err && D.status == 0) D.status = GW_E_RANGE;
    }
    const FluxSums S{D.sums[0], D.sums[1], D.sums[2], D.sums[3]};
    Currents cur;
    prepare_step(C, D, S, a.dt, cur, static_cast<int>(D.step & 1));
    lookahead_consts(C, D, a.dt, a.frozen != 0);
    if (D.status != 0 && D.stop_step > D.step) D.stop_step = D.step;
}
// ===========================================================================
// host side
// ===========================================================================
void set_err(char *err, size_t errlen, const char *fmt, ...)
{
    if (!err || errlen == 0) return;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(err, errlen, fmt, ap);
    va_end(ap);
}

#define HIP_TRY(expr)                                                                               \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) {                                                                     \
            set_err(err, errlen, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
            return GW_E_HIP;                                                                        \
        }                                                                                           \
    } while (0)

gw_params_t default_params()
{
    gw_params_t p;
#define GW_SET_DEFAULT_(type, name, dflt) p.name = static_cast<type>(dflt);
    GW_PARAMETER_FIELDS(GW_SET_DEFAULT_)
#undef GW_SET_DEFAULT_
    return p;
}

gw_globals_t default_globals()
{
    gw_globals_t g;
    g.V = -91.382; g.Nai = 10.0; g.Ki = 131.84; g.Cai = 1.45273e-4; g.CaNSR = 0.908882;
    g.CaLTRPN = 8.98282e-3; g.CaHTRPN = 0.137617; g.m = 5.33837e-4; g.h = 0.996345; g.j = 0.997315;
    g.xKs = 2.04171e-4;
    const double Kr[5] = {0.999503, 4.13720e-4, 7.27568e-5, 8.73984e-6, 1.36159e-6};
    const double Kv43[10] = {0.953060, 0.0253906, 2.53848e-4, 1.12796e-6, 1.87950e-9,
                             0.0151370, 0.00517622, 8.96600e-4, 8.17569e-5, 2.24032e-6};
    const double Kv14[10] = {0.722328, 0.101971, 0.00539932, 1.27081e-4, 1.82742e-6,
                             0.152769, 0.00962328, 0.00439043, 0.00195348, 0.00143629};
    for (int i = 0; i < 5; ++i) g.Kr[i] = Kr[i];
    for (int i = 0; i < 10; ++i) { g.Kv43[i] = Kv43[i]; g.Kv14[i] = Kv14[i]; }
    return g;
}

}  // namespace

// Device memory of the allocation-free entry point (gw_run_noalloc): one
// static array, which every GPU the library runs on holds until the process
// ends. Host code never passes the array's name to a kernel or a copy: it
// uses the address hipGetSymbolAddress gives on each device (gw_ctx_create).
constexpr size_t kScratchBytes = size_t(64) << 20;
__device__ __align__(256) unsigned char scratch[kScratchBytes];
// The pinned host memory a context holds for that entry point from its
// creation on: two pieces of a cell's state (allocating 4 MB takes 0.35 ms once).
constexpr int64_t kFixedPieceCrus = 16384;
constexpr size_t kFixedPin = 2 * ((piece_bytes(kFixedPieceCrus) + 255) & ~size_t(255));
constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

struct gw_ctx {
    int device = 0;
    int cus = kRouteCus;              // its compute units
    hipStream_t stream = nullptr;
    void *scratch = nullptr;          // this device's address of `scratch`
    void *fixed_pin = nullptr;        // pinned memory and events of the allocation-free runs (kFixedPin bytes)
    hipEvent_t fixed_ev[2] = {};
    std::mutex pin_mu;                // a pinned buffer no batch holds, of at most kPinKeep bytes
    void *pin = nullptr;
    size_t pin_bytes = 0;
    std::vector<gw_batch *> batches;  // live batches; released by gw_ctx_destroy
};

struct gw_batch {
    gw_ctx *ctx = nullptr;
    int32_t ncells = 0, precision = 0, prng = 0;
    double dt = 1e-3;
    int64_t ntot = 0, nblocks = 0;
    bool digest = true;
    bool frozen = false;
    bool prepared = false;
    int64_t steps_done = 0;
    int32_t trace_every = 0;
    int64_t trace_cap = 0;
    int32_t shape = kShapeDefault;   // block -> cell map in use (16 << shape CRUs per block)
    int32_t persist_mode = 0;        // persistent step kernel: 0 off (default), 1 on, 2 when every block fits at once
    int32_t persist_fit = -1;        // whether every block of the persistent kernel fits at once (-1: not known)
    int32_t steps_per_launch = 0;    // SSA steps per plain launch where the kernel can run two: 1, 2, 0 automatic
    int32_t cfg = 2;                 // launch configuration (kConfigs) asked for, 4 x 256 by default
    int32_t run_cfg = 2;             // the one the batch's shape arrays are set for (apply_shape)
    int64_t ncrus = 0;               // CRUs of all cells
    bool uniform = true;             // all cells have the same number
    // replayed graphs of step chunks (0 = plain launches)
    int32_t graph_steps = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    int32_t graph_steps_built = 0, graph_cfg = -1;   // graph_cfg: the configuration that ran (run_cfg)
    bool graph_digest = false;
    KArgs graph_args{};
    int64_t *d_step_base = nullptr;
    int64_t nblocks_shape[kNumShapes] = {};
    int64_t bc_off[kNumShapes] = {};   // offset of each map's block -> cell table
    int64_t max_nblocks = 0;
    std::vector<DevCell> cells_h;
    std::vector<double *> istim_dev;
    KArgs a{};
    DevCell *d_cells = nullptr;
    CellDyn *d_dyn = nullptr;
    BlockInfo *d_blocks = nullptr;
    // pinned host memory that kernels write results to: leased from the context
    // or allocated when first needed, handed back with the batch
    void *pin = nullptr;
    size_t pin_bytes = 0;
    hipEvent_t pin_ev[2] = {};
    // the device memory of a batch, one allocation (own_arena) or, for an
    // allocation-free batch (noalloc), a part of the scratch array; its pinned
    // memory and events are then the context's
    bool noalloc = false;
    bool own_arena = false;
    char *arena = nullptr;
    size_t arena_size = 0, arena_used = 0;
    double *arena_table = nullptr;   // the stimulus table of cell 0
    int64_t arena_table_cap = 0;
};

namespace {

// The next 256-byte aligned piece of a batch's device memory. Before there is
// any, the pieces are only counted (arena_used).
int carve(gw_batch *B, void **p, size_t bytes, char *err, size_t errlen)
{
    const size_t at = (B->arena_used + 255) & ~size_t(255);
    if (B->arena && at + bytes > B->arena_size) {
        set_err(err, errlen, "the allocation-free path holds at most %zu bytes of device state (%zu MiB of static "
                "scratch per GPU); this run needs more: use fewer CRUs or fewer steps, or gw_run",
                B->arena_size, B->arena_size >> 20);
        return GW_E_INVALID_ARG;
    }
    *p = B->arena ? B->arena + at : nullptr;
    B->arena_used = at + bytes;
    return GW_OK;
}

template <class T>
int dmalloc(gw_batch *B, T **p, size_t n, char *err, size_t errlen)
{
    *p = nullptr;
    if (n == 0) return GW_OK;
    void *q = nullptr;
    const int rc = carve(B, &q, n * sizeof(T), err, errlen);
    *p = static_cast<T *>(q);
    return rc;
}

// At least `bytes` of pinned host memory for the batch: the buffer the context
// keeps, if it is large enough, or a new one. (A buffer costs some 100 us and
// up to allocate, as much as 15 steps of a small cell.)
constexpr size_t kPinLeast = size_t(256) << 10, kPinKeep = size_t(16) << 20;

void release_pin(gw_batch *B)
{
    gw_ctx *ctx = B->ctx;
    if (B->noalloc) return;
    if (B->pin && B->pin_bytes <= kPinKeep) {
        std::lock_guard<std::mutex> lock(ctx->pin_mu);
        if (B->pin_bytes > ctx->pin_bytes) {
            std::swap(B->pin, ctx->pin);
            std::swap(B->pin_bytes, ctx->pin_bytes);
        }
    }
    if (B->pin) (void)hipHostFree(B->pin);
    B->pin = nullptr;
    B->pin_bytes = 0;
}

int ensure_pin(gw_batch *B, size_t bytes, char *err, size_t errlen)
{
    if (B->pin_bytes >= bytes) return GW_OK;
    if (B->noalloc) {   // pieces of kFixedPieceCrus CRUs fit, and so does what one cell's state and status take
        set_err(err, errlen, "allocation-free batch: %zu bytes of pinned host memory exceed the context's %zu", bytes, B->pin_bytes);
        return GW_E_INVALID_ARG;
    }
    gw_ctx *ctx = B->ctx;
    if (B->pin) HIP_TRY(hipHostFree(B->pin));
    B->pin = nullptr;
    B->pin_bytes = 0;
    {
        std::lock_guard<std::mutex> lock(ctx->pin_mu);
        if (ctx->pin_bytes >= bytes) {
            std::swap(B->pin, ctx->pin);
            std::swap(B->pin_bytes, ctx->pin_bytes);
            return GW_OK;
        }
    }
    const size_t n = std::max(bytes, kPinLeast);
    HIP_TRY(hipHostMalloc(&B->pin, n, hipHostMallocDefault));
    B->pin_bytes = n;
    return GW_OK;
}

__global__ void k_fill_u64(unsigned long long *p, int64_t n, unsigned long long v)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_zero_i32(int32_t *p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

int batch_create(gw_ctx *ctx, int32_t ncells, const gw_cell_desc_t *cells, int32_t precision, int32_t prng_id,
                 double dt, const gw_globals_t *g0, void *arena, size_t arena_size, int64_t table_cap,
                 gw_batch **out, char *err, size_t errlen);

int validate_params(const gw_params_t &p, char *err, size_t errlen)
{
    if (!(p.T > 0 && p.CSA > 0 && p.Vcyto > 0 && p.VNSR > 0 && p.VJSR > 0 && p.VSS > 0 && p.NCaRU > 0 && p.Ko > 0 &&
          p.Nao > 0 && p.Cao > 0 && p.b > 0)) {
        set_err(err, errlen, "parameters: temperatures, volumes, NCaRU, b and external concentrations must be > 0");
        return GW_E_INVALID_ARG;
    }
    return GW_OK;
}

int launch_cfg_check(gw_batch *B, char *err, size_t errlen)
{
    if (B->nblocks <= 0 || B->nblocks > (1LL << 31) - 1) {
        set_err(err, errlen, "invalid number of SSA blocks %lld", static_cast<long long>(B->nblocks));
        return GW_E_INVALID_ARG;
    }
    return GW_OK;
}

constexpr int config_shape(int c)
{
    return shape_of_crus(kConfigs[c].threads / kConfigs[c].lanes * kConfigs[c].cpl);
}
static_assert(config_shape(kConfigDefault) == kShapeDefault, "the default configuration uses the setup map");
static_assert(config_shape(kNumConfigs - 1) < kNumShapes, "block -> cell maps cover every configuration");

// The launch configuration asked for; run_config chooses the one that runs.
void set_shape(gw_batch *B, int c) { B->cfg = c; }

void apply_shape(gw_batch *B, int c)
{
    B->run_cfg = c;
    B->shape = config_shape(c);
    B->nblocks = B->nblocks_shape[B->shape];
    B->a.shape = B->shape;
    B->a.nblocks = B->nblocks;
    B->a.blocks = B->d_blocks + B->bc_off[B->shape];
    // block_info's arithmetic, where the product with the rounded reciprocal is exact for every block
    const DevCell &C = B->cells_h[0];
    const uint64_t nb = static_cast<uint64_t>(C.nblk[B->shape]), magic = ((uint64_t(1) << 32) + nb - 1) / nb;
    const bool exact = B->uniform && static_cast<uint64_t>(B->nblocks) * (magic * nb - (uint64_t(1) << 32)) < uint64_t(1) << 32;
    B->a.uni_n = exact ? C.n_cru : 0;
    B->a.uni_nblk = C.nblk[B->shape];
    B->a.uni_slots = static_cast<int32_t>(B->ntot / B->ncells);
    B->a.uni_magic = magic;
}

// Configurations other than the default are built for the fast path only:
// FP64 without replay digests or FP32-local, xoshiro256**, free-running
// globals; one lane per CRU is FP32-local only.
bool shape_allowed(const gw_batch *B, int c)
{
    const bool fast = B->prng == GW_PRNG_XOSHIRO256SS && !B->frozen;
    if (kConfigs[c].lanes == 1) return fast && B->precision == GW_PREC_FP32_LOCAL;
    if (kConfigs[c].cpl > 1) return fast && B->precision == GW_PREC_FP64 && !B->digest;   // refilled quads
    return c == kConfigDefault || (fast && (B->precision == GW_PREC_FP32_LOCAL || !B->digest));
}

constexpr int kAutotuneGraphSteps = 64;   // steps per captured graph the autotuner tries
constexpr int kAutotuneWarm = kAutotuneGraphSteps + 2;   // untimed steps before every trial

int prepare(gw_batch *B, char *err, size_t errlen)
{
    if (B->prepared) return GW_OK;
    hipLaunchKernelGGL(k_init_cells, dim3(B->ncells), dim3(kBlock), 0, B->ctx->stream, B->a);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_reset_obs, dim3((B->ncells + 255) / 256), dim3(256), 0, B->ctx->stream, B->d_dyn, B->ncells);
    HIP_TRY(hipGetLastError());
    B->prepared = true;
    B->steps_done = 0;
    return GW_OK;
}

template <int PRNG>
void launch_frozen(gw_batch *B, int64_t step0, int64_t n)
{
    if (B->precision == GW_PREC_FP32_LOCAL)
        hipLaunchKernelGGL((k_ssa<PRNG, false, float>), dim3(B->nblocks), dim3(kBlock), 0, B->ctx->stream, B->a, step0, n);
    else if (B->digest)
        hipLaunchKernelGGL((k_ssa<PRNG, true, double>), dim3(B->nblocks), dim3(kBlock), 0, B->ctx->stream, B->a, step0, n);
    else
        hipLaunchKernelGGL((k_ssa<PRNG, false, double>), dim3(B->nblocks), dim3(kBlock), 0, B->ctx->stream, B->a, step0, n);
    hipLaunchKernelGGL(k_frozen_close, dim3((B->ncells + 63) / 64), dim3(64), 0, B->ctx->stream, B->a, step0, n);
}

void launch_frozen_steps(gw_batch *B, int64_t step0, int64_t n)
{
    apply_shape(B, kConfigDefault);
    switch (B->prng) {
    case 0: launch_frozen<0>(B, step0, n); break;
    case 1: launch_frozen<1>(B, step0, n); break;
    case 2: launch_frozen<2>(B, step0, n); break;
    case 3: launch_frozen<3>(B, step0, n); break;
    case 4: launch_frozen<4>(B, step0, n); break;
    default: launch_frozen<5>(B, step0, n); break;
    }
}

// Grid of one launch: the closes, then one block per SSA tile.
unsigned step_grid(const gw_batch *B, int64_t ssa_step, int32_t nclose)
{
    return static_cast<unsigned>(nclose + (ssa_step >= 0 ? B->nblocks : 0));
}

// A step launch: with timing events through the dispatch packet, without them
// as a plain launch (the form stream capture records into a graph).
template <class K>
void dispatch(K kernel, unsigned grid, int threads, gw_batch *B, hipEvent_t e0, hipEvent_t e1, int64_t ssa_step,
              int32_t nclose, const int64_t *base)
{
    if (e0)
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, B->ctx->stream, e0, e1, 0u, B->a, ssa_step, nclose, base);
    else
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, B->ctx->stream, B->a, ssa_step, nclose, base);
}

// One launch of k_step: SSA(ssa_step) (none if ssa_step < 0) beside the
// closes of the previous step (when nclose > 0). When e0/e1 are given, the
// dispatch itself records them (its start and end, no extra queue packets).
template <int PRNG, int BLOCK>
void launch_k_step_shape(gw_batch *B, int64_t ssa_step, int32_t nclose, hipEvent_t e0, hipEvent_t e1, const int64_t *base)
{
    const unsigned grid = step_grid(B, ssa_step, nclose);
    if (B->precision == GW_PREC_FP32_LOCAL) {
        dispatch(k_step<PRNG, false, float, BLOCK>, grid, BLOCK, B, e0, e1, ssa_step, nclose, base);
        return;
    }
    if constexpr (BLOCK == kBlock) {
        if (B->digest) {
            dispatch(k_step<PRNG, true, double, BLOCK>, grid, BLOCK, B, e0, e1, ssa_step, nclose, base);
            return;
        }
    }
    dispatch(k_step<PRNG, false, double, BLOCK>, grid, BLOCK, B, e0, e1, ssa_step, nclose, base);
}

// Shapes that a caller can ask for beside the default are built for xoshiro256**
// only (the engine of the production path; shape_allowed() keeps the others off
// them), the ones that run_config chooses by itself for every engine.
template <int PRNG>
void launch_k_step(gw_batch *B, int64_t ssa_step, int32_t nclose, hipEvent_t e0, hipEvent_t e1, const int64_t *base)
{
    if (B->run_cfg >= kLane64) {
        const unsigned grid = step_grid(B, ssa_step, nclose);
        switch (B->run_cfg) {
        case kLane64: dispatch(k_step_lane64<PRNG, 2>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
        case kLane64 + 1: dispatch(k_step_lane64<PRNG, 4>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
        default: dispatch(k_step_lane64<PRNG, 8>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
        }
        return;
    }
    if constexpr (PRNG == GW_PRNG_XOSHIRO256SS) {
        if (kConfigs[B->run_cfg].lanes == 1) {
            const unsigned grid = step_grid(B, ssa_step, nclose);
            switch (B->run_cfg) {
            case 4: dispatch(k_step_lane<PRNG, 64, 1>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 5: dispatch(k_step_lane<PRNG, 128, 1>, grid, 128, B, e0, e1, ssa_step, nclose, base); break;
            case 6: dispatch(k_step_lane<PRNG, 256, 1>, grid, 256, B, e0, e1, ssa_step, nclose, base); break;
            case 7: dispatch(k_step_lane<PRNG, 64, 2>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 8: dispatch(k_step_lane<PRNG, 128, 2>, grid, 128, B, e0, e1, ssa_step, nclose, base); break;
            case 9: dispatch(k_step_lane<PRNG, 256, 2>, grid, 256, B, e0, e1, ssa_step, nclose, base); break;
            case 10: dispatch(k_step_lane<PRNG, 64, 4>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 11: dispatch(k_step_lane<PRNG, 128, 4>, grid, 128, B, e0, e1, ssa_step, nclose, base); break;
            case 12: dispatch(k_step_lane<PRNG, 256, 4>, grid, 256, B, e0, e1, ssa_step, nclose, base); break;
            case 13: dispatch(k_step_lane<PRNG, 64, 8>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 14: dispatch(k_step_lane<PRNG, 128, 8>, grid, 128, B, e0, e1, ssa_step, nclose, base); break;
            default: dispatch(k_step_lane<PRNG, 256, 8>, grid, 256, B, e0, e1, ssa_step, nclose, base); break;
            }
            return;
        }
        if (kConfigs[B->run_cfg].cpl > 1) {
            const unsigned grid = step_grid(B, ssa_step, nclose);
            switch (B->run_cfg) {   // FP64 only (shape_allowed)
            case 16: dispatch(k_step_refill<PRNG, double, 64, 2>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 17: dispatch(k_step_refill<PRNG, double, 64, 4>, grid, 64, B, e0, e1, ssa_step, nclose, base); break;
            case 18: dispatch(k_step_refill<PRNG, double, 128, 4>, grid, 128, B, e0, e1, ssa_step, nclose, base); break;
            default: dispatch(k_step_refill<PRNG, double, 256, 4>, grid, 256, B, e0, e1, ssa_step, nclose, base); break;
            }
            return;
        }
    }
    if (B->shape == 0) {   // plain quads run with 64 threads or the default's 256 (run_config)
        launch_k_step_shape<PRNG, 64>(B, ssa_step, nclose, e0, e1, base);
        return;
    }
    launch_k_step_shape<PRNG, kBlock>(B, ssa_step, nclose, e0, e1, base);
}

void launch_one(gw_batch *B, int64_t ssa_step, int32_t nclose, hipEvent_t e0, hipEvent_t e1,
                const int64_t *base = nullptr)
{
    switch (B->prng) {
    case 0: launch_k_step<0>(B, ssa_step, nclose, e0, e1, base); break;
    case 1: launch_k_step<1>(B, ssa_step, nclose, e0, e1, base); break;
    case 2: launch_k_step<2>(B, ssa_step, nclose, e0, e1, base); break;
    case 3: launch_k_step<3>(B, ssa_step, nclose, e0, e1, base); break;
    case 4: launch_k_step<4>(B, ssa_step, nclose, e0, e1, base); break;
    default: launch_k_step<5>(B, ssa_step, nclose, e0, e1, base); break;
    }
}

// The replayable graph of graph_steps step launches (each SSA(base + k) beside
// the close of the step before) and the launch that advances base. It is
// captured again whenever the launch arguments or shape change.
bool graph_current(const gw_batch *B)
{
    return B->graph_exec && B->graph_steps_built == B->graph_steps && B->graph_cfg == B->run_cfg &&
           B->graph_digest == B->digest &&
           std::memcmp(&B->graph_args, &B->a, sizeof(KArgs)) == 0;
}

void graph_release(gw_batch *B)
{
    if (B->graph_exec) (void)hipGraphExecDestroy(B->graph_exec);
    if (B->graph) (void)hipGraphDestroy(B->graph);
    B->graph_exec = nullptr;
    B->graph = nullptr;
}

hipError_t graph_build(gw_batch *B)
{
    graph_release(B);
    hipStream_t st = B->ctx->stream;
    hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    for (int k = 0; k < B->graph_steps; ++k) launch_one(B, k, B->ncells, nullptr, nullptr, B->d_step_base);
    hipLaunchKernelGGL(k_advance_base, dim3(1), dim3(1), 0, st, B->d_step_base, static_cast<int64_t>(B->graph_steps));
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(st, &g);
    if (e != hipSuccess) return e;
    B->graph = g;
    e = hipGraphInstantiate(&B->graph_exec, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        graph_release(B);
        return e;
    }
    B->graph_steps_built = B->graph_steps;
    B->graph_cfg = B->run_cfg;
    B->graph_digest = B->digest;
    B->graph_args = B->a;
    return hipSuccess;
}

// The persistent step kernel of a batch's engine and precision.
template <int PRNG>
const void *persist_fn_prng(const gw_batch *B)
{
    if (B->precision == GW_PREC_FP32_LOCAL) return reinterpret_cast<const void *>(&k_persist<PRNG, false, float>);
    if (B->digest) return reinterpret_cast<const void *>(&k_persist<PRNG, true, double>);
    return reinterpret_cast<const void *>(&k_persist<PRNG, false, double>);
}

const void *persist_fn(const gw_batch *B)
{
    switch (B->prng) {
    case 0: return persist_fn_prng<0>(B);
    case 1: return persist_fn_prng<1>(B);
    case 2: return persist_fn_prng<2>(B);
    case 3: return persist_fn_prng<3>(B);
    case 4: return persist_fn_prng<4>(B);
    default: return persist_fn_prng<5>(B);
    }
}

// Whether every block of the persistent kernel (the closes and the SSA blocks
// of the default shape) can be resident at once on the batch's device.
bool persist_fits(gw_batch *B)
{
    if (B->persist_fit >= 0) return B->persist_fit != 0;
    int per_cu = 0, cus = 0;
    const int64_t grid = B->ncells + B->nblocks_shape[kShapeDefault];
    B->persist_fit = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, persist_fn(B), kBlock, 0) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, B->ctx->device) == hipSuccess)
        B->persist_fit = static_cast<int64_t>(per_cu) * cus >= grid ? 1 : 0;
    return B->persist_fit != 0;
}

// The persistent kernel runs the default shape's free-running steps.
bool use_persist(gw_batch *B)
{
    return B->persist_mode != 0 && !B->frozen && B->cfg == kConfigDefault && persist_fits(B);
}

// What the next steps run in (gw_route.h), except where only the kernels of the
// shape asked for are built.
BatchSize batch_size(const gw_batch *B)
{
    return {B->precision == GW_PREC_FP32_LOCAL, B->ncrus, B->ncells, B->ctx->cus};
}

int run_config(gw_batch *B)
{
    if (B->frozen || (B->precision == GW_PREC_FP64 && B->digest) || use_persist(B)) return B->cfg;
    return route(B->cfg, batch_size(B));
}

// Steps step0 .. step0+n-1 in one cooperative launch of the persistent kernel
// (which closes every step itself), after its counters are set for step0.
hipError_t launch_persist(gw_batch *B, int64_t step0, int64_t n)
{
    if (B->precision == GW_PREC_FP32_LOCAL)
        hipLaunchKernelGGL(k_sync_init<float>, dim3(B->ncells), dim3(64), 0, B->ctx->stream, B->a, step0);
    else
        hipLaunchKernelGGL(k_sync_init<double>, dim3(B->ncells), dim3(64), 0, B->ctx->stream, B->a, step0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t grid = B->ncells + B->nblocks_shape[kShapeDefault];
    void *args[] = {&B->a, &step0, &n};
    e = hipLaunchCooperativeKernel(persist_fn(B), dim3(static_cast<unsigned>(grid)), dim3(kBlock), args, 0,
                                   B->ctx->stream);
    return e;
}

// Whether the batch's plain launches can run two SSA steps each: FP32-local
// free-running steps on a one-lane shape of 64 threads (k_step_lane2;
// xoshiro256**, as every shape a caller can ask for), or FP64 steps that
// run_config gives to the one-lane kernels (k_step2_lane64); not persistent,
// no replayed graphs.
bool pair_capable(gw_batch *B)
{
    if (B->frozen || B->graph_steps > 0 || use_persist(B)) return false;
    const int c = run_config(B);
    const LaunchCfg &L = kConfigs[c];
    if (c >= kLane64) return true;
    return B->precision == GW_PREC_FP32_LOCAL && L.lanes == 1 && L.threads == 64 && B->prng == GW_PRNG_XOSHIRO256SS;
}

// Two steps per launch where asked for, or by the batch's size (gw_route.h).
bool use_pair(gw_batch *B)
{
    if (B->steps_per_launch == 1 || !pair_capable(B)) return false;
    return B->steps_per_launch == 2 || route_pair(run_config(B), batch_size(B));
}

// One launch of the two-step kernel: SSA(m .. m + nss - 1); with e0/e1 the
// dispatch records its own start and end.
template <class K>
void dispatch_pair(K kernel, gw_batch *B, int64_t m, int32_t nss, hipEvent_t e0, hipEvent_t e1)
{
    const dim3 grid(static_cast<unsigned>(B->nblocks)), block(64);
    if (e0)
        hipExtLaunchKernelGGL(kernel, grid, block, 0, B->ctx->stream, e0, e1, 0u, B->a, m, nss);
    else
        hipLaunchKernelGGL(kernel, grid, block, 0, B->ctx->stream, B->a, m, nss);
}

template <int P>
void launch_pair_lane64(gw_batch *B, int64_t m, int32_t nss, hipEvent_t e0, hipEvent_t e1)
{
    switch (B->run_cfg) {
    case kLane64: dispatch_pair(k_step2_lane64<P, 2>, B, m, nss, e0, e1); break;
    case kLane64 + 1: dispatch_pair(k_step2_lane64<P, 4>, B, m, nss, e0, e1); break;
    default: dispatch_pair(k_step2_lane64<P, 8>, B, m, nss, e0, e1); break;
    }
}

void launch_pair(gw_batch *B, int64_t m, int32_t nss, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr)
{
    constexpr int P = GW_PRNG_XOSHIRO256SS;
    if (B->run_cfg >= kLane64) {
        switch (B->prng) {
        case 0: launch_pair_lane64<0>(B, m, nss, e0, e1); break;
        case 1: launch_pair_lane64<1>(B, m, nss, e0, e1); break;
        case 2: launch_pair_lane64<2>(B, m, nss, e0, e1); break;
        case 3: launch_pair_lane64<3>(B, m, nss, e0, e1); break;
        case 4: launch_pair_lane64<4>(B, m, nss, e0, e1); break;
        default: launch_pair_lane64<5>(B, m, nss, e0, e1); break;
        }
        return;
    }
    switch (kConfigs[B->run_cfg].cpl) {
    case 1: dispatch_pair(k_step_lane2<P, 64, 1>, B, m, nss, e0, e1); break;
    case 2: dispatch_pair(k_step_lane2<P, 64, 2>, B, m, nss, e0, e1); break;
    case 4: dispatch_pair(k_step_lane2<P, 64, 4>, B, m, nss, e0, e1); break;
    default: dispatch_pair(k_step_lane2<P, 64, 8>, B, m, nss, e0, e1); break;
    }
}

void launch_closes(gw_batch *B, int32_t ncl)
{
    hipLaunchKernelGGL(k_close_cells, dim3(B->ncells), dim3(kBlock), 0, B->ctx->stream, B->a, ncl);
}

// Steps step0 .. step0+n-1 two per launch: the first launch runs SSA(step0)
// and SSA(step0+1) with no closes before it (the call starts with every step
// closed); each later launch is preceded by the closes its SSA steps need (up
// to two), an odd last step runs alone, and a last close kernel closes the
// rest. Returns the number of SSA launches through *launches. With ssa_ms,
// every SSA dispatch records its own start and end through a ring of event
// pairs (the host waits for the dispatch that last used a pair before reusing
// it, kRing launches back, so the queue never runs dry), and *ssa_ms is the
// sum of their durations: the SSA kernel's time without the close kernels.
hipError_t launch_steps_pair(gw_batch *B, int64_t step0, int64_t n, int64_t *launches, double *ssa_ms = nullptr)
{
    constexpr int kRing = 256;
    std::vector<hipEvent_t> ev(ssa_ms ? 2 * kRing : 0, nullptr);
    hipError_t e = hipSuccess;
    for (auto &x : ev)
        if ((e = hipEventCreate(&x)) != hipSuccess) break;
    double acc = 0.0;
    auto harvest = [&](int r) {
        float f = 0.f;
        hipError_t h = hipEventSynchronize(ev[2 * r + 1]);
        if (h == hipSuccess) h = hipEventElapsedTime(&f, ev[2 * r], ev[2 * r + 1]);
        acc += f;
        return h;
    };
    int64_t m = step0, c = step0, count = 0;   // next SSA step, first step not closed
    const int64_t end = step0 + n;
    while (e == hipSuccess && m < end) {
        const int32_t nss = end - m >= 2 ? 2 : 1;
        const int32_t ncl = static_cast<int32_t>(std::max<int64_t>(0, m + nss - 2 - c));   // closes up to m+nss-3
        if (ncl > 0) launch_closes(B, ncl);
        if (ssa_ms) {
            const int r = static_cast<int>(count % kRing);
            if (count >= kRing && (e = harvest(r)) != hipSuccess) break;
            launch_pair(B, m, nss, ev[2 * r], ev[2 * r + 1]);
        } else {
            launch_pair(B, m, nss);
        }
        c += ncl;
        m += nss;
        ++count;
    }
    if (e == hipSuccess && c < end) launch_closes(B, static_cast<int32_t>(end - c));
    for (int64_t k = std::max<int64_t>(0, count - kRing); ssa_ms && e == hipSuccess && k < count; ++k)
        e = harvest(static_cast<int>(k % kRing));
    for (auto &x : ev)
        if (x) (void)hipEventDestroy(x);
    if (ssa_ms) *ssa_ms = acc;
    if (launches) *launches = count;
    if (e != hipSuccess) return e;
    return hipGetLastError();
}

// Steps step0 .. step0+n-1: n launches, launch k running SSA(step0+k) beside
// close(step0+k-1), then one launch with the last closes. Between calls every
// step is closed, so the cell state read by the host is that of step0+n.
// With graphs enabled, the middle launches are replays of the captured chunk.
hipError_t launch_steps(gw_batch *B, int64_t step0, int64_t n, int64_t *launches = nullptr)
{
    if (launches) *launches = 0;
    if (n <= 0) return hipSuccess;
    apply_shape(B, run_config(B));
    if (use_persist(B)) {
        if (launches) *launches = 1;
        return launch_persist(B, step0, n);
    }
    if (use_pair(B)) return launch_steps_pair(B, step0, n, launches);
    if (launches) *launches = n;
    launch_one(B, step0, 0, nullptr, nullptr);
    int64_t k = 1;
    if (B->graph_steps > 0 && n - 1 >= B->graph_steps) {
        hipError_t e = hipSuccess;
        if (!graph_current(B)) e = graph_build(B);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_set_base, dim3(1), dim3(1), 0, B->ctx->stream, B->d_step_base, step0 + 1);
        for (; k + B->graph_steps <= n; k += B->graph_steps)
            if ((e = hipGraphLaunch(B->graph_exec, B->ctx->stream)) != hipSuccess) return e;
    }
    for (; k < n; ++k) launch_one(B, step0 + k, B->ncells, nullptr, nullptr);
    launch_one(B, -1, B->ncells, nullptr, nullptr);
    return hipGetLastError();
}

// launch_steps with every step's dispatch timed through a ring of event pairs:
// before a pair is reused, the host waits for the dispatch that last recorded
// it (kRing steps back), so the queue never runs dry. The final close-only
// launch is not timed.
int launch_steps_timed(gw_batch *B, int64_t step0, int64_t n, double *ssa_ms, char *err, size_t errlen)
{
    constexpr int kRing = 512;
    std::vector<hipEvent_t> ev(2 * kRing, nullptr);
    int rc = GW_OK;
    double acc = 0.0;
    for (auto &e : ev)
        if (hipEventCreate(&e) != hipSuccess) {
            set_err(err, errlen, "hipEventCreate failed");
            rc = GW_E_HIP;
            break;
        }
    auto harvest = [&](int r) {
        float f = 0.f;
        if (hipEventSynchronize(ev[2 * r + 1]) != hipSuccess || hipEventElapsedTime(&f, ev[2 * r], ev[2 * r + 1]) != hipSuccess)
            return false;
        acc += f;
        return true;
    };
    for (int64_t k = 0; rc == GW_OK && k < n; ++k) {
        const int r = static_cast<int>(k % kRing);
        if (k >= kRing && !harvest(r)) {
            set_err(err, errlen, "event timing failed");
            rc = GW_E_HIP;
            break;
        }
        launch_one(B, step0 + k, k == 0 ? 0 : B->ncells, ev[2 * r], ev[2 * r + 1]);
    }
    if (rc == GW_OK && n > 0) launch_one(B, -1, B->ncells, nullptr, nullptr);
    for (int64_t k = std::max<int64_t>(0, n - kRing); rc == GW_OK && k < n; ++k)
        if (!harvest(static_cast<int>(k % kRing))) {
            set_err(err, errlen, "event timing failed");
            rc = GW_E_HIP;
        }
    for (auto &e : ev)
        if (e) (void)hipEventDestroy(e);
    if (ssa_ms) *ssa_ms = acc;
    return rc;
}

// Status and trace row count of every cell (k_gather_dyn); *out stays valid
// until the batch's pinned memory is used again.
int gather_dyn(gw_batch *B, const int64_t **out, char *err, size_t errlen)
{
    const int rc = ensure_pin(B, (2 * static_cast<size_t>(B->ncells) + 1) * sizeof(int64_t), err, errlen);
    if (rc) return rc;
    hipLaunchKernelGGL(k_gather_dyn, dim3((B->ncells + 255) / 256), dim3(256), 0, B->ctx->stream, B->d_dyn, B->ncells,
                       B->a.timeout, static_cast<int64_t *>(B->pin));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    *out = static_cast<const int64_t *>(B->pin);
    return GW_OK;
}

// `bytes` bytes at offset `at` of every cell's dynamic state, cell after cell.
int read_dyn(gw_batch *B, size_t at, size_t bytes, const void **out, char *err, size_t errlen)
{
    const int rc = ensure_pin(B, bytes * static_cast<size_t>(B->ncells), err, errlen);
    if (rc) return rc;
    const int n = static_cast<int>(bytes / 8);
    const int64_t words = static_cast<int64_t>(B->ncells) * n;
    hipLaunchKernelGGL(k_export_dyn, dim3(static_cast<unsigned>((words + 255) / 256)), dim3(256), 0, B->ctx->stream,
                       B->d_dyn, B->ncells, static_cast<int>(at / 8), n, static_cast<uint64_t *>(B->pin));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    *out = B->pin;
    return GW_OK;
}

int cell_error(int cell, int32_t st, char *err, size_t errlen)
{
    const char *what = st == GW_E_NONPOSITIVE_CONC ? "a Nernst potential received a non-positive concentration"
                     : st == GW_E_NAN ? "a global state variable became NaN"
                     : st == GW_E_RANGE ? "a CRU flux, a RyR count or the SSA iteration count left the supported range"
                                        : "device error";
    set_err(err, errlen, "cell %d: %s (status %d)", cell, what, st);
    return st;
}

int check_status(gw_batch *B, char *err, size_t errlen)
{
    const int64_t *v = nullptr;
    const int rc = gather_dyn(B, &v, err, errlen);
    if (rc) return rc;
    if (v[2 * static_cast<size_t>(B->ncells)] != 0) {
        set_err(err, errlen, "a bounded wait of the persistent step kernel expired; the steps of this call are incomplete");
        return GW_E_TIMEOUT;
    }
    for (int c = 0; c < B->ncells; ++c)
        if (v[c] != 0) return cell_error(c, static_cast<int32_t>(v[c]), err, errlen);
    return GW_OK;
}

// After a per-cell override: before the first step the whole batch is
// prepared afresh at step 0 (nothing has run); after it only this cell's
// current step is formed again (k_refresh_cell).
int refresh_cell(gw_batch *B, int cell, int resum, char *err, size_t errlen)
{
    if (!B->prepared || B->steps_done == 0) {
        B->prepared = false;
        return GW_OK;
    }
    hipLaunchKernelGGL(k_refresh_cell, dim3(1), dim3(kBlock), 0, B->ctx->stream, B->a, cell, resum);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    return GW_OK;
}

template <int PRNG>
void launch_init_crus(gw_batch *B)
{
    hipLaunchKernelGGL(k_init_crus<PRNG>, dim3(static_cast<unsigned>(B->nblocks_shape[kInitMap])), dim3(kBlock), 0,
                       B->ctx->stream, B->a, B->d_blocks + B->bc_off[kInitMap]);
}

hipError_t init_crus(gw_batch *B)
{
    switch (B->prng) {
    case 0: launch_init_crus<0>(B); break;
    case 1: launch_init_crus<1>(B); break;
    case 2: launch_init_crus<2>(B); break;
    case 3: launch_init_crus<3>(B); break;
    case 4: launch_init_crus<4>(B); break;
    default: launch_init_crus<5>(B); break;
    }
    return hipGetLastError();
}

// Pieces of one cell's state read through pinned memory, two at a time, so
// that the host expands one while the stream goes on (another piece, or the
// steps after a record). A cell of up to piece_crus CRUs is one piece.
constexpr int64_t kPieceCrus = 65536;
static_assert(kPieceCrus % 2 == 0 && 2 * piece_bytes(kPieceCrus) <= kPinKeep, "a context keeps two pieces");
static_assert(kFixedPieceCrus % 2 == 0, "a piece starts at an even CRU");
int64_t piece_crus(const gw_batch *B) { return B->noalloc ? kFixedPieceCrus : kPieceCrus; }

enum PieceForm : int { PIECE_CRUS, PIECE_CRUS_JLCC, PIECE_REDUCED };
struct PieceQueue {
    struct Piece {
        int64_t record, i0, m;
        double t;
    };
    gw_batch *B;
    int cell, form;
    size_t stride;
    Piece piece[2];
    int first = 0, live = 0;
};

int pieces_open(PieceQueue &q, gw_batch *B, int cell, int form, char *err, size_t errlen)
{
    q.B = B;
    q.cell = cell;
    q.form = form;
    q.stride = (piece_bytes(std::min<int64_t>(B->cells_h[cell].n_cru, piece_crus(B))) + 255) & ~size_t(255);
    const int rc = ensure_pin(B, 2 * q.stride, err, errlen);
    if (rc) return rc;
    for (hipEvent_t &e : B->pin_ev)
        if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return GW_OK;
}

// The oldest piece into sink(piece, base), which returns a status.
template <class Sink>
int pieces_pop(PieceQueue &q, Sink &&sink, char *err, size_t errlen)
{
    HIP_TRY(hipEventSynchronize(q.B->pin_ev[q.first]));
    const int rc = sink(q.piece[q.first], static_cast<char *>(q.B->pin) + q.first * q.stride);
    q.first ^= 1;
    --q.live;
    return rc;
}

// The cell's state after the steps launched so far; one piece is left under way.
template <class Sink>
int pieces_push(PieceQueue &q, int64_t record, double t, Sink &&sink, char *err, size_t errlen)
{
    gw_batch *B = q.B;
    const int64_t n = B->cells_h[q.cell].n_cru, most = piece_crus(B);
    hipStream_t s = B->ctx->stream;
    for (int64_t i0 = 0; i0 < n; i0 += most) {
        const int64_t m = std::min(most, n - i0);
        const int k = q.first ^ q.live;   // live is 0 or 1 here
        void *base = static_cast<char *>(B->pin) + k * q.stride;
        if (q.form == PIECE_REDUCED) {
            hipLaunchKernelGGL(k_get_piece_reduced, dim3(static_cast<unsigned>((m + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                               B->a, q.cell, i0, m, base);
        } else {
            const int jlcc = q.form == PIECE_CRUS_JLCC;
            const int64_t w = piece_words(m, jlcc, B->a.JLCCf != nullptr);
            hipLaunchKernelGGL(k_get_piece, dim3(static_cast<unsigned>((w + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, B->a,
                               q.cell, i0, m, jlcc, base);
        }
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(B->pin_ev[k], s));
        q.piece[k] = {record, i0, m, t};
        if (++q.live == 2) {
            const int rc = pieces_pop(q, sink, err, errlen);
            if (rc) return rc;
        }
    }
    return GW_OK;
}

template <class Sink>
int pieces_drain(PieceQueue &q, Sink &&sink, char *err, size_t errlen)
{
    while (q.live > 0) {
        const int rc = pieces_pop(q, sink, err, errlen);
        if (rc) return rc;
    }
    return GW_OK;
}

// CRUs i0 .. i0 + m - 1 of a piece into the rows of c (any of which may be null).
void expand_piece(void *base, int64_t i0, int64_t m, bool f32, const gw_cru_state_t &c)
{
    const PieceView v = piece_view(base, m);
    const int64_t n = 4 * m;
    if (c.CaSS) std::memcpy(c.CaSS + 4 * i0, v.CaSS, n * 8);
    if (c.CaJSR) std::memcpy(c.CaJSR + i0, v.CaJSR, m * 8);
    if (c.JLCC) {
        if (f32)
            for (int64_t k = 0; k < n; ++k) c.JLCC[4 * i0 + k] = static_cast<double>(static_cast<const float *>(v.JLCC)[k]);
        else
            std::memcpy(c.JLCC + 4 * i0, v.JLCC, n * 8);
    }
    if (c.LCC) for (int64_t k = 0; k < n; ++k) c.LCC[4 * i0 + k] = sub_lcc(v.sub[k]);
    if (c.LCC_inactivation) for (int64_t k = 0; k < n; ++k) c.LCC_inactivation[4 * i0 + k] = sub_y(v.sub[k]);
    if (c.ClCh) for (int64_t k = 0; k < n; ++k) c.ClCh[4 * i0 + k] = sub_cl(v.sub[k]);
    if (c.RyR)
        for (int64_t k = 0; k < n; ++k)
            for (int r = 0; r < 6; ++r) c.RyR[(4 * i0 + k) * 6 + r] = ryr_get(v.sub[k], r);
}

void expand_reduced(void *base, int64_t i0, int64_t m, const gw_cru_state_reduced_t &c)
{
    const ReducedView v = reduced_view(base, m);
    if (c.CaSS) std::memcpy(c.CaSS + 4 * i0, v.CaSS, 4 * m * 4);
    if (c.CaJSR) std::memcpy(c.CaJSR + i0, v.CaJSR, m * 4);
    if (c.RyR) std::memcpy(c.RyR + 4 * i0, v.RyR, 4 * m * 2);
    if (c.LCC) std::memcpy(c.LCC + 4 * i0, v.LCC, 4 * m);
    if (c.LCC_inactivation) std::memcpy(c.LCC_inactivation + 4 * i0, v.LCCi, 4 * m);
    if (c.ClCh) std::memcpy(c.ClCh + 4 * i0, v.ClCh, 4 * m);
}

}  // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
extern "C" {

void gw_params_default(gw_params_t *p)
{
    if (p) *p = default_params();
}

void gw_globals_default(gw_globals_t *g)
{
    if (g) *g = default_globals();
}

int gw_prng_from_name(const char *name)
{
    if (!name) return -1;
    static const char *names[GW_PRNG_COUNT] = {"xoshiro256**", "xoshiro256++", "xoshiro256+",
                                               "xoroshiro128**", "xoroshiro128++", "xoroshiro128+"};
    for (int i = 0; i < GW_PRNG_COUNT; ++i)
        if (std::strcmp(name, names[i]) == 0) return i;
    return -1;
}

int gw_version(void) { return GW_CAPI_VERSION; }

int gw_rest_state(int32_t n_cru, uint64_t seed, int32_t prng_id, gw_cru_state_t *out)
{
    if (n_cru <= 0 || !out || prng_id < 0 || prng_id >= GW_PRNG_COUNT) return GW_E_INVALID_ARG;
    for (int64_t i = 0; i < n_cru; ++i) {
        double ca[4], jsr;
        uint64_t sub[4];
        sample_rest_cru_any(prng_id, seed, i, ca, jsr, sub);
        for (int j = 0; j < 4; ++j) {
            if (out->CaSS) out->CaSS[i * 4 + j] = ca[j];
            if (out->JLCC) out->JLCC[i * 4 + j] = 0.0;
            if (out->LCC) out->LCC[i * 4 + j] = sub_lcc(sub[j]);
            if (out->LCC_inactivation) out->LCC_inactivation[i * 4 + j] = sub_y(sub[j]);
            if (out->ClCh) out->ClCh[i * 4 + j] = sub_cl(sub[j]);
            if (out->RyR)
                for (int k = 0; k < 6; ++k) out->RyR[(i * 4 + j) * 6 + k] = ryr_get(sub[j], k);
        }
        if (out->CaJSR) out->CaJSR[i] = jsr;
    }
    return GW_OK;
}

int gw_ctx_create(gw_ctx **out, int device, char *err, size_t errlen)
{
    if (!out) {
        set_err(err, errlen, "out is null");
        return GW_E_INVALID_ARG;
    }
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
        set_err(err, errlen, "no HIP device is visible");
        return GW_E_NO_DEVICE;
    }
    if (device < 0 || device >= n) {
        set_err(err, errlen, "device %d out of range (%d devices)", device, n);
        return GW_E_INVALID_ARG;
    }
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        set_err(err, errlen, "device %d is %s; this library is built for gfx950", device, prop.gcnArchName);
        return GW_E_NO_DEVICE;
    }
    HIP_TRY(hipSetDevice(device));
    if (device < kMaxDevices) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_ptr[device]) {
            void *ptr = nullptr;
            const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !ptr) {
                set_err(err, errlen, "hipGetSymbolAddress(scratch) failed on device %d: %s", device, hipGetErrorString(e));
                return GW_E_HIP;
            }
            g_scratch_ptr[device] = ptr;
        }
    }
    gw_ctx *c = new gw_ctx;
    c->device = device;
    c->cus = prop.multiProcessorCount;
    c->scratch = device < kMaxDevices ? g_scratch_ptr[device] : nullptr;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        set_err(err, errlen, "hipStreamCreate failed");
        return GW_E_HIP;
    }
    hipError_t e = hipHostMalloc(&c->fixed_pin, kFixedPin, hipHostMallocDefault);
    for (hipEvent_t &ev : c->fixed_ev)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e != hipSuccess) {
        set_err(err, errlen, "allocating the context's pinned host memory: %s", hipGetErrorString(e));
        gw_ctx_destroy(c);
        return GW_E_HIP;
    }
    *out = c;
    return GW_OK;
}

int gw_ctx_destroy(gw_ctx *ctx)
{
    if (!ctx) return GW_OK;
    while (!ctx->batches.empty()) gw_batch_destroy(ctx->batches.back());
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipStreamDestroy(ctx->stream);
    if (ctx->pin) (void)hipHostFree(ctx->pin);
    if (ctx->fixed_pin) (void)hipHostFree(ctx->fixed_pin);
    for (hipEvent_t e : ctx->fixed_ev)
        if (e) (void)hipEventDestroy(e);
    delete ctx;
    return GW_OK;
}

int gw_batch_destroy(gw_batch *B)
{
    if (!B) return GW_OK;
    auto &live = B->ctx->batches;
    live.erase(std::remove(live.begin(), live.end(), B), live.end());
    (void)hipSetDevice(B->ctx->device);
    (void)hipStreamSynchronize(B->ctx->stream);
    graph_release(B);
    release_pin(B);
    for (hipEvent_t e : B->pin_ev)
        if (e && !B->noalloc) (void)hipEventDestroy(e);
    if (B->own_arena) (void)hipFree(B->arena);
    if (B->a.trace) (void)hipFree(B->a.trace);
    for (double *p : B->istim_dev)
        if (p) (void)hipFree(p);
    delete B;
    return GW_OK;
}

int gw_batch_create(gw_ctx *ctx, int32_t ncells, const gw_cell_desc_t *cells, int32_t precision, int32_t prng_id,
                    double dt, const gw_globals_t *g0, gw_batch **out, char *err, size_t errlen)
{
    return batch_create(ctx, ncells, cells, precision, prng_id, dt, g0, nullptr, 0, 0, out, err, errlen);
}

}  // extern "C"

namespace {

constexpr size_t kArenaReserve = 210;   // bytes per CRU

// gw_batch_create, or with arena != null an allocation-free batch whose device
// memory is carved from arena[0, arena_size); a stimulus table of table_cap
// steps is carved with the rest.
int batch_create(gw_ctx *ctx, int32_t ncells, const gw_cell_desc_t *cells, int32_t precision, int32_t prng_id,
                 double dt, const gw_globals_t *g0, void *arena, size_t arena_size, int64_t table_cap,
                 gw_batch **out, char *err, size_t errlen)
{
    if (!ctx || !cells || !out || ncells <= 0) {
        set_err(err, errlen, "gw_batch_create: null argument or ncells <= 0");
        return GW_E_INVALID_ARG;
    }
    *out = nullptr;
    if (!(dt > 0.0) || !std::isfinite(dt)) {
        set_err(err, errlen, "step size must be > 0");
        return GW_E_INVALID_ARG;
    }
    if (prng_id < 0 || prng_id >= GW_PRNG_COUNT) {
        set_err(err, errlen, "unknown PRNG id %d", prng_id);
        return GW_E_INVALID_ARG;
    }
    if (precision != GW_PREC_FP64 && precision != GW_PREC_FP32_LOCAL) {
        set_err(err, errlen, "unknown precision %d", precision);
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    gw_batch *B = new gw_batch;
    B->ctx = ctx;
    B->arena = static_cast<char *>(arena);
    B->arena_size = arena ? arena_size : 0;
    if (arena) {
        B->noalloc = true;
        B->pin = ctx->fixed_pin;
        B->pin_bytes = kFixedPin;
        std::copy(std::begin(ctx->fixed_ev), std::end(ctx->fixed_ev), std::begin(B->pin_ev));
    }
    B->ncells = ncells;
    B->precision = precision;
    B->prng = prng_id;
    B->dt = dt;
    B->cells_h.resize(ncells);
    B->istim_dev.assign(ncells, nullptr);
    int64_t slot = 0;
    for (int c = 0; c < ncells; ++c) {
        const gw_cell_desc_t &d = cells[c];
        if (d.n_cru <= 0 || d.n_cru > (1 << 20)) {
            set_err(err, errlen, "cell %d: n_cru must be in 1..%d", c, 1 << 20);
            delete B;
            return GW_E_INVALID_ARG;
        }
        int rc = validate_params(d.params, err, errlen);
        if (rc != GW_OK) {
            delete B;
            return rc;
        }
        if (d.protocol.kind < GW_PROTO_TABLE || d.protocol.kind > GW_PROTO_CLAMP) {
            set_err(err, errlen, "cell %d: unknown protocol kind %d", c, d.protocol.kind);
            delete B;
            return GW_E_INVALID_ARG;
        }
        DevCell &C = B->cells_h[c];
        std::memset(&C, 0, sizeof(C));
        C.p = d.params;
        cell_consts_init(C.c, C.p, d.n_cru);
        ssa_params_init(C.sp, C.p, C.c);
        C.plain = ssa_params_plain(C.sp);
        ssa_params_f32(C.spf, C.sp);
        C.proto = d.protocol;
        C.seed = d.seed;
        C.n_cru = d.n_cru;
        C.slot0 = slot;
        for (int sh = 0; sh < kNumShapes; ++sh) {
            const int per = crus_per_block(sh);
            C.nblk[sh] = (d.n_cru + per - 1) / per;
        }
        slot += static_cast<int64_t>((d.n_cru + kSlotAlign - 1) / kSlotAlign) * kSlotAlign;
    }
    int64_t nblocks_all = 0;
    for (int sh = 0; sh < kNumShapes; ++sh) {
        B->bc_off[sh] = nblocks_all;
        int64_t blk = 0;
        for (int c = 0; c < ncells; ++c) {
            DevCell &C = B->cells_h[c];
            C.blk0[sh] = blk;
            C.blk_all[sh] = nblocks_all + blk;
            blk += C.nblk[sh];
        }
        B->nblocks_shape[sh] = blk;
        nblocks_all += blk;
        B->max_nblocks = std::max(B->max_nblocks, blk);
    }
    B->ntot = slot;
    for (int c = 0; c < ncells; ++c) {
        B->ncrus += cells[c].n_cru;
        B->uniform = B->uniform && cells[c].n_cru == cells[0].n_cru;
    }
    B->nblocks = B->nblocks_shape[kShapeDefault];
    const int64_t N = B->ntot;
    KArgs &a = B->a;
    int rc = GW_OK;
    const bool f32 = precision == GW_PREC_FP32_LOCAL;
    auto lay_out = [&]() {
        int r = dmalloc(B, &a.CaSS, 4 * N, err, errlen);
        if (r || (r = dmalloc(B, &a.CaJSR, N, err, errlen)) ||
            (!f32 && (r = dmalloc(B, &a.JLCC, 4 * N, err, errlen))) ||
            (f32 && (r = dmalloc(B, &a.JLCCf, 4 * N, err, errlen))) ||
            (r = dmalloc(B, &a.sub, 4 * N, err, errlen)) ||
            (r = dmalloc(B, &a.rng, 4 * N, err, errlen)) ||
            (!f32 && (r = dmalloc(B, &a.dig, 2 * N, err, errlen))) ||
            (r = dmalloc(B, &a.partials, 2 * B->max_nblocks, err, errlen)) ||
            (r = dmalloc(B, &a.iters_total, 1, err, errlen)) || (r = dmalloc(B, &B->d_step_base, 1, err, errlen)) ||
            (r = dmalloc(B, &B->d_cells, ncells, err, errlen)) || (r = dmalloc(B, &B->d_dyn, ncells, err, errlen)) ||
            (r = dmalloc(B, &a.sync, static_cast<size_t>(ncells), err, errlen)) ||
            (r = dmalloc(B, &a.timeout, 1, err, errlen)) ||
            (r = dmalloc(B, &B->d_blocks, static_cast<size_t>(nblocks_all), err, errlen)) ||
            (r = dmalloc(B, &B->arena_table, static_cast<size_t>(table_cap), err, errlen)))
            return r;
        return static_cast<int>(GW_OK);
    };
    if (!B->arena) {   // count, then one allocation for all of them
        void *mem = nullptr;
        hipError_t he = hipSuccess;
        if ((rc = lay_out()) == GW_OK && (he = hipMalloc(&mem, B->arena_used)) != hipSuccess) {
            set_err(err, errlen, "allocating %zu bytes of device memory: %s", B->arena_used, hipGetErrorString(he));
            rc = GW_E_HIP;
        }
        if (rc == GW_OK) {
            B->arena = static_cast<char *>(mem);
            B->own_arena = true;
            B->arena_size = B->arena_used;
            B->arena_used = 0;
        }
    } else {
        // a run's limit of CRUs and steps counts this much beside the batch
        void *reserved = nullptr;
        rc = carve(B, &reserved, kArenaReserve * static_cast<size_t>(B->cells_h[0].n_cru), err, errlen);
    }
    if (rc == GW_OK) rc = lay_out();
    if (rc != GW_OK) {
        gw_batch_destroy(B);
        return rc;
    }
    B->arena_table_cap = table_cap;
    a.cells = B->d_cells;
    a.dyn = B->d_dyn;
    a.blocks = B->d_blocks + B->bc_off[kShapeDefault];
    a.shape = kShapeDefault;
    a.ntot = N;
    a.nblocks = B->nblocks;
    a.dt = dt;
    a.ncells = ncells;
    a.frozen = 0;
    a.trace_every = 0;
    a.trace_cap = 0;
    a.trace = nullptr;
    a.prng = prng_id;
    a.precision = precision;
    a.spin_limit = kSpinLimit;
    // per-cell stimulus tables are attached later; globals start at g0 or the defaults
    std::vector<CellDyn> dyn(ncells);
    for (int c = 0; c < ncells; ++c) {
        std::memset(&dyn[c], 0, sizeof(CellDyn));
        dyn[c].g = g0 ? *g0 : default_globals();
        dyn[c].clamp = (cells[c].protocol.kind == GW_PROTO_CLAMP) ? 1 : 0;
    }
    auto fail = [&](hipError_t e) {
        set_err(err, errlen, "HIP error during batch creation: %s", hipGetErrorString(e));
        gw_batch_destroy(B);
        return GW_E_HIP;
    };
    hipError_t e;
    if ((e = hipMemcpyAsync(B->d_cells, B->cells_h.data(), ncells * sizeof(DevCell), hipMemcpyHostToDevice, ctx->stream)) != hipSuccess) return fail(e);
    if ((e = hipMemcpyAsync(B->d_dyn, dyn.data(), ncells * sizeof(CellDyn), hipMemcpyHostToDevice, ctx->stream)) != hipSuccess) return fail(e);
    hipLaunchKernelGGL(k_block_info, dim3(ncells, kNumShapes), dim3(kBlock), 0, ctx->stream, B->d_cells, B->d_blocks);
    if ((e = hipGetLastError()) != hipSuccess) return fail(e);
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, ctx->stream, a.iters_total, int64_t(1), 0ull);
    if ((e = hipGetLastError()) != hipSuccess) return fail(e);
    hipLaunchKernelGGL(k_fill_u64, dim3((ncells * (sizeof(CellSync) / 8) + 255) / 256), dim3(256), 0, ctx->stream,
                       reinterpret_cast<unsigned long long *>(a.sync), int64_t(ncells) * int64_t(sizeof(CellSync) / 8),
                       0ull);
    if ((e = hipGetLastError()) != hipSuccess) return fail(e);
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(64), 0, ctx->stream, a.timeout, int64_t(1));
    if ((e = hipGetLastError()) != hipSuccess) return fail(e);
    if ((e = init_crus(B)) != hipSuccess) return fail(e);
    if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return fail(e);
    ctx->batches.push_back(B);
    *out = B;
    return GW_OK;
}

}  // namespace

extern "C" {

int gw_batch_set_cru_state(gw_batch *B, int32_t cell, const gw_cru_state_t *c, char *err, size_t errlen)
{
    if (!B || !c || cell < 0 || cell >= B->ncells || !c->CaSS || !c->CaJSR || !c->LCC || !c->LCC_inactivation ||
        !c->RyR || !c->ClCh) {
        set_err(err, errlen, "gw_batch_set_cru_state: bad arguments");
        return GW_E_INVALID_ARG;
    }
    const int64_t n = B->cells_h[cell].n_cru;
    // whether any value is out of range, without a branch per value; then which
    uint32_t bad = 0;
    for (int64_t i = 0; i < 4 * n; ++i)
        bad |= (static_cast<uint32_t>(c->LCC[i]) - 1u > 11u) | ((c->LCC_inactivation[i] | c->ClCh[i]) & ~1) |
               !(std::fabs(c->CaSS[i]) <= DBL_MAX);
    for (int64_t i = 0; i < 24 * n; ++i) bad |= static_cast<uint32_t>(c->RyR[i]) + 100u > 200u;
    for (int64_t i = 0; i < n; ++i) bad |= !(std::fabs(c->CaJSR[i]) <= DBL_MAX);
    if (bad) {
        for (int64_t i = 0; i < 4 * n; ++i) {
            if (c->LCC[i] < 1 || c->LCC[i] > 12) {
                set_err(err, errlen, "LCC states must be integers in 1..12 (got %d at flat index %lld)", c->LCC[i], static_cast<long long>(i));
                return GW_E_INVALID_ARG;
            }
            if ((c->LCC_inactivation[i] & ~1) || (c->ClCh[i] & ~1)) {
                set_err(err, errlen, "LCC_inactivation and ClCh must be 0 or 1 (flat index %lld)", static_cast<long long>(i));
                return GW_E_INVALID_ARG;
            }
            if (!std::isfinite(c->CaSS[i])) {
                set_err(err, errlen, "CaSS must be finite");
                return GW_E_INVALID_ARG;
            }
        }
        for (int64_t i = 0; i < 24 * n; ++i)
            if (c->RyR[i] < -100 || c->RyR[i] > 100) {
                set_err(err, errlen, "RyR counts must lie in -100..100");
                return GW_E_INVALID_ARG;
            }
        for (int64_t i = 0; i < n; ++i)
            if (!std::isfinite(c->CaJSR[i])) {
                set_err(err, errlen, "CaJSR must be finite");
                return GW_E_INVALID_ARG;
            }
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    const int64_t most = piece_crus(B);
    int rc = ensure_pin(B, piece_bytes(std::min(n, most)), err, errlen);
    if (rc) return rc;
    hipStream_t s = B->ctx->stream;
    for (int64_t i0 = 0; i0 < n; i0 += most) {
        const int64_t m = std::min(most, n - i0);
        const PieceView v = piece_view(B->pin, m);
        std::memcpy(v.CaSS, c->CaSS + 4 * i0, 4 * m * 8);
        std::memcpy(v.CaJSR, c->CaJSR + i0, m * 8);
        if (c->JLCC) std::memcpy(v.JLCC, c->JLCC + 4 * i0, 4 * m * 8);
        for (int64_t k = 0; k < 4 * m; ++k) {
            const int64_t q = 4 * i0 + k;
            v.sub[k] = sub_pack(c->LCC[q], c->LCC_inactivation[q], c->ClCh[q], c->RyR + q * 6);
        }
        hipLaunchKernelGGL(k_put_piece, dim3(static_cast<unsigned>((4 * m + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, B->a,
                           cell, i0, m, c->JLCC ? 1 : 0, B->pin);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(s));
    }
    return refresh_cell(B, cell, 1, err, errlen);
}

int gw_batch_get_cru_state(gw_batch *B, int32_t cell, gw_cru_state_t *c, char *err, size_t errlen)
{
    if (!B || !c || cell < 0 || cell >= B->ncells) {
        set_err(err, errlen, "gw_batch_get_cru_state: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    PieceQueue q;
    int rc = pieces_open(q, B, cell, c->JLCC ? PIECE_CRUS_JLCC : PIECE_CRUS, err, errlen);
    if (rc) return rc;
    const bool f32 = B->a.JLCCf != nullptr;
    auto sink = [&](const PieceQueue::Piece &p, void *base) {
        expand_piece(base, p.i0, p.m, f32, *c);
        return GW_OK;
    };
    rc = pieces_push(q, 0, 0.0, sink, err, errlen);
    return rc ? rc : pieces_drain(q, sink, err, errlen);
}

int gw_batch_get_cru_state_reduced(gw_batch *B, int32_t cell, gw_cru_state_reduced_t *c, char *err, size_t errlen)
{
    if (!B || !c || cell < 0 || cell >= B->ncells) {
        set_err(err, errlen, "gw_batch_get_cru_state_reduced: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    PieceQueue q;
    int rc = pieces_open(q, B, cell, PIECE_REDUCED, err, errlen);
    if (rc) return rc;
    auto sink = [&](const PieceQueue::Piece &p, void *base) {
        expand_reduced(base, p.i0, p.m, *c);
        return GW_OK;
    };
    rc = pieces_push(q, 0, 0.0, sink, err, errlen);
    return rc ? rc : pieces_drain(q, sink, err, errlen);
}

int gw_batch_set_globals(gw_batch *B, int32_t cell, const gw_globals_t *g, char *err, size_t errlen)
{
    if (!B || !g || cell < 0 || cell >= B->ncells) {
        set_err(err, errlen, "gw_batch_set_globals: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    HIP_TRY(hipMemcpyAsync(&B->d_dyn[cell].g, g, sizeof(gw_globals_t), hipMemcpyHostToDevice, B->ctx->stream));
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    return refresh_cell(B, cell, 0, err, errlen);
}

int gw_batch_get_globals(gw_batch *B, gw_globals_t *g_out, char *err, size_t errlen)
{
    if (!B || !g_out) {
        set_err(err, errlen, "gw_batch_get_globals: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    const void *d = nullptr;
    const int rc = read_dyn(B, offsetof(CellDyn, g), sizeof(gw_globals_t), &d, err, errlen);
    if (rc) return rc;
    std::memcpy(g_out, d, static_cast<size_t>(B->ncells) * sizeof(gw_globals_t));
    return GW_OK;
}

int gw_batch_set_stimulus_table(gw_batch *B, int32_t cell, const double *istim, int64_t n, char *err, size_t errlen)
{
    if (!B || cell < 0 || cell >= B->ncells || (n > 0 && !istim) || n < 0) {
        set_err(err, errlen, "gw_batch_set_stimulus_table: bad arguments");
        return GW_E_INVALID_ARG;
    }
    if (B->cells_h[cell].proto.kind == GW_PROTO_CLAMP) {
        set_err(err, errlen, "gw_batch_set_stimulus_table: cell %d is voltage-clamped; a stimulus table has no effect on it",
                cell);
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    double *d = nullptr;
    const bool carved = cell == 0 && n <= B->arena_table_cap;
    if (!B->own_arena || (carved && n > 0)) {   // the table carved at creation (cell 0 only)
        if (!carved) {
            set_err(err, errlen, "allocation-free batch: a stimulus table of %lld steps exceeds the %lld carved",
                    static_cast<long long>(n), static_cast<long long>(B->arena_table_cap));
            return GW_E_INVALID_ARG;
        }
        if (n > 0) {
            d = B->arena_table;
            HIP_TRY(hipMemcpyAsync(d, istim, n * sizeof(double), hipMemcpyHostToDevice, B->ctx->stream));
        }
    } else {
        if (B->istim_dev[cell]) HIP_TRY(hipFree(B->istim_dev[cell]));
        B->istim_dev[cell] = nullptr;
        if (n > 0) {
            HIP_TRY(hipMalloc(&d, n * sizeof(double)));
            HIP_TRY(hipMemcpyAsync(d, istim, n * sizeof(double), hipMemcpyHostToDevice, B->ctx->stream));
        }
        B->istim_dev[cell] = d;
    }
    B->cells_h[cell].istim = d;
    B->cells_h[cell].istim_len = n;
    B->cells_h[cell].proto.kind = GW_PROTO_TABLE;
    HIP_TRY(hipMemcpyAsync(&B->d_cells[cell], &B->cells_h[cell], sizeof(DevCell), hipMemcpyHostToDevice, B->ctx->stream));
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    return refresh_cell(B, cell, 0, err, errlen);
}

int gw_batch_step(gw_batch *B, int64_t nsteps, char *err, size_t errlen)
{
    if (!B || nsteps < 0) {
        set_err(err, errlen, "gw_batch_step: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    int rc = launch_cfg_check(B, err, errlen);
    if (rc) return rc;
    rc = prepare(B, err, errlen);
    if (rc) return rc;
    if (B->frozen) {
        // one launch per chunk; a chunk is at most ~2^26 CRU-steps of work
        const int64_t chunk = std::max<int64_t>(1, std::min<int64_t>(1 << 18, (1LL << 26) / std::max<int64_t>(1, B->ntot)));
        for (int64_t done = 0; done < nsteps;) {
            const int64_t n = std::min(chunk, nsteps - done);
            launch_frozen_steps(B, B->steps_done, n);
            HIP_TRY(hipGetLastError());
            done += n;
            B->steps_done += n;
            rc = check_status(B, err, errlen);
            if (rc) return rc;
        }
        return GW_OK;
    }
    const int64_t chunk = 4096;
    for (int64_t done = 0; done < nsteps;) {
        const int64_t n = std::min(chunk, nsteps - done);
        HIP_TRY(launch_steps(B, B->steps_done, n));
        done += n;
        B->steps_done += n;
        rc = check_status(B, err, errlen);
        if (rc) return rc;
    }
    return GW_OK;
}

int gw_batch_get_time(gw_batch *B, double *t, int64_t *steps_done)
{
    if (!B) return GW_E_INVALID_ARG;
    (void)hipSetDevice(B->ctx->device);
    if (!B->prepared) {
        if (t) *t = 0.0;
        if (steps_done) *steps_done = 0;
        return GW_OK;
    }
    // every running cell shares the clock; a cell that failed stopped its own
    constexpr size_t t0 = offsetof(CellDyn, t), len = offsetof(CellDyn, obs) - t0;
    const void *mem = nullptr;
    if (read_dyn(B, t0, len, &mem, nullptr, 0) != GW_OK) return GW_E_HIP;
    struct {
        double t;
        int64_t step;
        int32_t status;
    } x;
    std::vector<decltype(x)> d(static_cast<size_t>(B->ncells));
    for (int c = 0; c < B->ncells; ++c) {
        const char *w = static_cast<const char *>(mem) + c * len;
        std::memcpy(&d[c].t, w, sizeof(x.t));
        std::memcpy(&d[c].step, w + offsetof(CellDyn, step) - t0, sizeof(x.step));
        std::memcpy(&d[c].status, w + offsetof(CellDyn, status) - t0, sizeof(x.status));
    }
    int pick = -1;
    for (int c = 0; c < B->ncells && pick < 0; ++c)
        if (d[c].status == 0) pick = c;
    if (pick < 0) {
        pick = 0;
        for (int c = 1; c < B->ncells; ++c)
            if (d[c].step > d[pick].step) pick = c;
    }
    if (t) *t = d[pick].t;
    if (steps_done) *steps_done = d[pick].step;
    return GW_OK;
}

int gw_batch_get_obs(gw_batch *B, gw_cell_obs_t *obs, char *err, size_t errlen)
{
    if (!B || !obs) {
        set_err(err, errlen, "gw_batch_get_obs: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    const void *d = nullptr;
    const int rc = read_dyn(B, offsetof(CellDyn, obs), sizeof(gw_cell_obs_t), &d, err, errlen);
    if (rc) return rc;
    std::memcpy(obs, d, static_cast<size_t>(B->ncells) * sizeof(gw_cell_obs_t));
    return GW_OK;
}

int gw_batch_reset_obs(gw_batch *B, char *err, size_t errlen)
{
    if (!B) return GW_E_INVALID_ARG;
    HIP_TRY(hipSetDevice(B->ctx->device));
    int rc = prepare(B, err, errlen);
    if (rc) return rc;
    hipLaunchKernelGGL(k_reset_obs, dim3((B->ncells + 255) / 256), dim3(256), 0, B->ctx->stream, B->d_dyn, B->ncells);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    return GW_OK;
}

int gw_batch_enable_trace(gw_batch *B, int32_t every, int64_t capacity, char *err, size_t errlen)
{
    if (!B || every < 0 || capacity < 0) {
        set_err(err, errlen, "gw_batch_enable_trace: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    if (B->a.trace) HIP_TRY(hipFree(B->a.trace));
    B->a.trace = nullptr;
    B->a.trace_every = 0;
    B->a.trace_cap = 0;
    if (every > 0 && capacity > 0) {
        HIP_TRY(hipMalloc(&B->a.trace, static_cast<size_t>(capacity) * B->ncells * 4 * sizeof(double)));
        B->a.trace_every = every;
        B->a.trace_cap = capacity;
    }
    hipLaunchKernelGGL(k_zero_trace_rows, dim3((B->ncells + 255) / 256), dim3(256), 0, B->ctx->stream, B->d_dyn, B->ncells);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    return GW_OK;
}

int gw_batch_get_trace(gw_batch *B, double *out, int64_t max_rows, int64_t *rows, char *err, size_t errlen)
{
    if (!B || !rows) {
        set_err(err, errlen, "gw_batch_get_trace: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    const int64_t *v = nullptr;
    int rc = gather_dyn(B, &v, err, errlen);
    if (rc) return rc;
    const int n = B->ncells;
    int64_t r = 0;
    for (int c = 0; c < n; ++c) r = std::max(r, v[n + c]);
    r = std::min(r, max_rows);
    if (r > 0 && out) {
        HIP_TRY(hipMemcpyAsync(out, B->a.trace, static_cast<size_t>(r) * n * 4 * sizeof(double), hipMemcpyDeviceToHost, B->ctx->stream));
        HIP_TRY(hipStreamSynchronize(B->ctx->stream));
        // a cell that stopped early (non-zero status) wrote fewer rows: its later rows read NaN
        for (int c = 0; c < n; ++c)
            for (int64_t k = std::max<int64_t>(0, v[n + c]); k < r; ++k)
                for (int q = 0; q < 4; ++q) out[(k * n + c) * 4 + q] = std::nan("");
    }
    hipLaunchKernelGGL(k_zero_trace_rows, dim3((n + 255) / 256), dim3(256), 0, B->ctx->stream, B->d_dyn, n);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    *rows = r;
    return GW_OK;
}

int gw_batch_get_event_digest(gw_batch *B, int32_t cell, uint64_t *count, uint64_t *hash, char *err, size_t errlen)
{
    if (!B || cell < 0 || cell >= B->ncells || !count || !hash) {
        set_err(err, errlen, "gw_batch_get_event_digest: bad arguments");
        return GW_E_INVALID_ARG;
    }
    if (!B->a.dig) {
        set_err(err, errlen, "event digests are not kept by this batch");
        return GW_E_INVALID_ARG;
    }
    const DevCell &C = B->cells_h[cell];
    HIP_TRY(hipSetDevice(B->ctx->device));
    std::vector<uint64_t> pairs(2 * static_cast<size_t>(C.n_cru));
    HIP_TRY(hipMemcpyAsync(pairs.data(), B->a.dig + 2 * C.slot0, pairs.size() * sizeof(uint64_t), hipMemcpyDeviceToHost, B->ctx->stream));
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    for (int64_t i = 0; i < C.n_cru; ++i) {
        count[i] = pairs[2 * i];
        hash[i] = pairs[2 * i + 1];
    }
    return GW_OK;
}

int gw_batch_get_iterations(gw_batch *B, uint64_t *iters)
{
    if (!B || !iters) return GW_E_INVALID_ARG;
    (void)hipSetDevice(B->ctx->device);
    unsigned long long v = 0;
    (void)hipMemcpyAsync(&v, B->a.iters_total, sizeof(v), hipMemcpyDeviceToHost, B->ctx->stream);
    if (hipStreamSynchronize(B->ctx->stream) != hipSuccess) return GW_E_HIP;
    *iters = v;
    return GW_OK;
}

int gw_launch_config(int32_t index, int32_t *lanes_per_cru, int32_t *block, int32_t *crus_per_lane)
{
    if (index < 0 || index >= kNumConfigs) return GW_E_INVALID_ARG;
    if (lanes_per_cru) *lanes_per_cru = kConfigs[index].lanes;
    if (block) *block = kConfigs[index].threads;
    if (crus_per_lane) *crus_per_lane = kConfigs[index].cpl;
    return GW_OK;
}

int gw_batch_set_launch(gw_batch *B, int32_t lanes_per_cru, int32_t block, int32_t crus_per_lane, char *err,
                        size_t errlen)
{
    if (!B) return GW_E_INVALID_ARG;
    const int lanes = lanes_per_cru ? lanes_per_cru : 4;
    const int threads = block ? block : (lanes == 4 ? kBlock : 64);
    const int cpl = crus_per_lane ? crus_per_lane : 1;
    int c = -1;
    for (int k = 0; k < kNumConfigs; ++k)
        if (kConfigs[k].lanes == lanes && kConfigs[k].threads == threads && kConfigs[k].cpl == cpl) c = k;
    if (c < 0) {
        set_err(err, errlen, "launch shape of %d lanes per CRU x %d threads x %d CRUs per lane is not available "
                "(4 lanes: 64, 128, 256 or 512 threads with 1 CRU per quad, 64 with 2, 64, 128 or 256 with 4; "
                "1 lane: 64, 128 or 256 threads, 1, 2, 4 or 8 CRUs per lane)", lanes_per_cru, block, crus_per_lane);
        return GW_E_INVALID_ARG;
    }
    if (!shape_allowed(B, c)) {
        set_err(err, errlen, "launch shape of %d lanes per CRU x %d threads is not available for this batch (other "
                "shapes than 4 x 256 need xoshiro256** without replay digests or frozen globals; 1 lane per CRU needs "
                "FP32-local; refilled quads need FP64)", lanes, threads);
        return GW_E_INVALID_ARG;
    }
    set_shape(B, c);
    return GW_OK;
}

int gw_batch_get_launch(gw_batch *B, int32_t *lanes_per_cru, int32_t *block, int32_t *crus_per_lane)
{
    if (!B) return GW_E_INVALID_ARG;
    return gw_launch_config(B->cfg, lanes_per_cru, block, crus_per_lane);
}

int gw_batch_get_running(gw_batch *B, int32_t *lanes_per_cru, int32_t *block, int32_t *crus_per_lane)
{
    if (!B) return GW_E_INVALID_ARG;
    (void)hipSetDevice(B->ctx->device);
    const LaunchCfg &L = kConfigs[run_config(B)];
    if (lanes_per_cru) *lanes_per_cru = L.lanes;
    if (block) *block = L.threads;
    if (crus_per_lane) *crus_per_lane = L.cpl;
    return GW_OK;
}

int gw_batch_autotune(gw_batch *B, int64_t trial_steps, int32_t *lanes_out, int32_t *block_out, int32_t *cpl_out,
                      int32_t *graph_out, double *ms_per_step, char *err, size_t errlen)
{
    if (!B || trial_steps <= 0) {
        set_err(err, errlen, "gw_batch_autotune: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    int rc = prepare(B, err, errlen);
    if (rc) return rc;
    hipStream_t st = B->ctx->stream;
    const int64_t N = B->ntot;
    KArgs &a = B->a;
    // everything a step changes; restored after every trial
    struct Piece {
        void *p;
        size_t n;
    };
    std::vector<Piece> pieces = {{a.CaSS, 32 * static_cast<size_t>(N)},
                                 {a.CaJSR, 8 * static_cast<size_t>(N)},
                                 {a.JLCC ? static_cast<void *>(a.JLCC) : static_cast<void *>(a.JLCCf),
                                  (a.JLCC ? 32 : 16) * static_cast<size_t>(N)},
                                 {a.sub, 32 * static_cast<size_t>(N)},
                                 {a.rng, 32 * static_cast<size_t>(N)},
                                 {B->d_dyn, sizeof(CellDyn) * static_cast<size_t>(B->ncells)},
                                 {a.iters_total, sizeof(unsigned long long)}};
    if (a.dig) pieces.push_back({a.dig, 16 * static_cast<size_t>(N)});
    size_t total = 0;
    for (const Piece &q : pieces) total += (q.n + 255) & ~static_cast<size_t>(255);
    char *snap = nullptr;
    HIP_TRY(hipMalloc(&snap, total));
    auto copy_all = [&](bool save) {
        size_t off = 0;
        for (const Piece &q : pieces) {
            const hipError_t e = save ? hipMemcpyAsync(snap + off, q.p, q.n, hipMemcpyDeviceToDevice, st)
                                      : hipMemcpyAsync(q.p, snap + off, q.n, hipMemcpyDeviceToDevice, st);
            if (e != hipSuccess) return e;
            off += (q.n + 255) & ~static_cast<size_t>(255);
        }
        return hipSuccess;
    };
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t he = copy_all(true);
    if (he == hipSuccess) he = hipEventCreate(&e0);
    if (he == hipSuccess) he = hipEventCreate(&e1);
    const int64_t steps0 = B->steps_done;
    int best_cfg = B->cfg;
    double best_ms = 1e300;
    double ran_ms[kNumConfigs + 4];   // of what a shape runs as (run_config; last, the persistent kernel): timed once
    std::fill(std::begin(ran_ms), std::end(ran_ms), -1.0);
    // of shapes that run alike, the one that runs as itself
    auto consider = [&](int c, double ms, bool itself) {
        if (ms_per_step) ms_per_step[c] = ms;
        if (ms < best_ms || (ms == best_ms && itself)) {
            best_ms = ms;
            best_cfg = c;
        }
    };
    for (int c = 0; c < kNumConfigs && he == hipSuccess; ++c) {
        if (ms_per_step) ms_per_step[c] = -1.0;
        if (!shape_allowed(B, c)) continue;
        set_shape(B, c);
        const int ran = use_persist(B) ? kNumConfigs + 3 : run_config(B);
        if (ran_ms[ran] >= 0.0) {
            consider(c, ran_ms[ran], ran == c);
            continue;
        }
        if ((he = launch_steps(B, B->steps_done, kAutotuneWarm)) != hipSuccess) break;
        B->steps_done += kAutotuneWarm;
        if ((he = hipEventRecord(e0, st)) != hipSuccess) break;
        if ((he = launch_steps(B, B->steps_done, trial_steps)) != hipSuccess) break;
        if ((he = hipEventRecord(e1, st)) != hipSuccess) break;
        if ((he = hipEventSynchronize(e1)) != hipSuccess) break;
        float f = 0.f;
        if ((he = hipEventElapsedTime(&f, e0, e1)) != hipSuccess) break;
        ran_ms[ran] = f / static_cast<double>(trial_steps);
        consider(c, ran_ms[ran], ran == c);
        he = copy_all(false);
        B->steps_done = steps0;
    }
    // the fastest shape with the other number of SSA steps per launch, where
    // it can run both (the CRU state kept in registers across two steps, or
    // streamed through HBM every step)
    const int32_t spl0 = B->steps_per_launch;
    int32_t best_spl = spl0;
    set_shape(B, best_cfg);
    if (he == hipSuccess && pair_capable(B)) {
        const int32_t used = use_pair(B) ? 2 : 1;   // the choice the trials above ran with
        best_spl = used;
        B->steps_per_launch = 3 - used;
        if ((he = launch_steps(B, B->steps_done, kAutotuneWarm)) == hipSuccess) {
            B->steps_done += kAutotuneWarm;
            if ((he = hipEventRecord(e0, st)) == hipSuccess && (he = launch_steps(B, B->steps_done, trial_steps)) == hipSuccess &&
                (he = hipEventRecord(e1, st)) == hipSuccess && (he = hipEventSynchronize(e1)) == hipSuccess) {
                float f = 0.f;
                if ((he = hipEventElapsedTime(&f, e0, e1)) == hipSuccess) {
                    const double ms = f / static_cast<double>(trial_steps);
                    if (ms < best_ms) {
                        best_ms = ms;
                        best_spl = B->steps_per_launch;
                    }
                }
            }
        }
        if (he == hipSuccess) he = copy_all(false);
        B->steps_done = steps0;
        B->steps_per_launch = best_spl;
    }
    // the fastest shape once more with its steps replayed as captured graphs
    const int32_t graph0 = B->graph_steps;
    int32_t best_graph = 0;
    if (ms_per_step) ms_per_step[kNumConfigs] = -1.0;
    if (he == hipSuccess && trial_steps > kAutotuneGraphSteps) {
        set_shape(B, best_cfg);
        B->graph_steps = kAutotuneGraphSteps;
        // the warm-up captures and replays the graph once, outside the timed window
        if ((he = launch_steps(B, B->steps_done, kAutotuneWarm)) == hipSuccess) {
            B->steps_done += kAutotuneWarm;
            if ((he = hipEventRecord(e0, st)) == hipSuccess && (he = launch_steps(B, B->steps_done, trial_steps)) == hipSuccess &&
                (he = hipEventRecord(e1, st)) == hipSuccess && (he = hipEventSynchronize(e1)) == hipSuccess) {
                float f = 0.f;
                if ((he = hipEventElapsedTime(&f, e0, e1)) == hipSuccess) {
                    const double ms = f / static_cast<double>(trial_steps);
                    if (ms_per_step) ms_per_step[kNumConfigs] = ms;
                    // graphs only when they save more than noise (launch-bound batches)
                    if (ms < 0.98 * best_ms) best_graph = kAutotuneGraphSteps;
                }
            }
        }
        if (he == hipSuccess) he = copy_all(false);
        B->steps_done = steps0;
    }
    B->graph_steps = (he == hipSuccess) ? best_graph : graph0;
    B->steps_per_launch = (he == hipSuccess) ? best_spl : spl0;
    if (he == hipSuccess) he = copy_all(false);
    if (he == hipSuccess) he = hipStreamSynchronize(st);
    B->steps_done = steps0;
    set_shape(B, best_cfg);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(snap);
    if (he != hipSuccess) {
        set_err(err, errlen, "autotune: %s", hipGetErrorString(he));
        return GW_E_HIP;
    }
    gw_batch_get_launch(B, lanes_out, block_out, cpl_out);
    if (graph_out) *graph_out = B->graph_steps;
    return check_status(B, err, errlen);
}

int gw_batch_time_steps(gw_batch *B, int64_t nsteps, double *ms, double *ssa_ms, int64_t *launches, char *err,
                        size_t errlen)
{
    if (!B || nsteps <= 0 || !ms) {
        set_err(err, errlen, "gw_batch_time_steps: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    int rc = prepare(B, err, errlen);
    if (rc) return rc;
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    HIP_TRY(hipEventRecord(e0, B->ctx->stream));
    apply_shape(B, run_config(B));
    const bool persist = use_persist(B);
    int64_t nlaunch = nsteps;   // SSA launches
    if (ssa_ms && use_pair(B)) {   // two steps per launch, each SSA dispatch timed
        HIP_TRY(launch_steps_pair(B, B->steps_done, nsteps, &nlaunch, ssa_ms));
    } else if (ssa_ms && !persist) {   // one step per launch, each dispatch timed
        rc = launch_steps_timed(B, B->steps_done, nsteps, ssa_ms, err, errlen);
        if (rc) return rc;
    } else {
        HIP_TRY(launch_steps(B, B->steps_done, nsteps, &nlaunch));
    }
    HIP_TRY(hipGetLastError());
    B->steps_done += nsteps;
    HIP_TRY(hipEventRecord(e1, B->ctx->stream));
    HIP_TRY(hipEventSynchronize(e1));
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = f;
    if (ssa_ms && persist) *ssa_ms = f;   // one launch runs every step
    if (launches) *launches = nlaunch;
    return check_status(B, err, errlen);
}

int gw_batch_set_persistent(gw_batch *B, int32_t mode, char *err, size_t errlen)
{
    if (!B || mode < 0 || mode > 2) {
        set_err(err, errlen, "gw_batch_set_persistent: mode must be 0 (off), 1 (on) or 2 (when it fits)");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    if (mode == 1 && !persist_fits(B)) {
        set_err(err, errlen, "gw_batch_set_persistent: the batch's %lld SSA blocks and %d close blocks cannot all be "
                "resident at once", static_cast<long long>(B->nblocks_shape[kShapeDefault]), B->ncells);
        return GW_E_INVALID_ARG;
    }
    B->persist_mode = mode;
    return GW_OK;
}

int gw_batch_get_currents(gw_batch *B, double *ICaL, double *Ito2, char *err, size_t errlen)
{
    if (!B || (!ICaL && !Ito2)) {
        set_err(err, errlen, "gw_batch_get_currents: bad arguments");
        return GW_E_INVALID_ARG;
    }
    HIP_TRY(hipSetDevice(B->ctx->device));
    int rc = prepare(B, err, errlen);
    if (rc) return rc;
    const size_t bytes = 2 * sizeof(double) * static_cast<size_t>(B->ncells);
    rc = ensure_pin(B, bytes, err, errlen);
    if (rc) return rc;
    double *h = static_cast<double *>(B->pin);
    hipLaunchKernelGGL(k_posthoc_currents, dim3(B->ncells), dim3(kBlock), 0, B->ctx->stream, B->a, h);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(B->ctx->stream));
    for (int c = 0; c < B->ncells; ++c) {
        if (ICaL) ICaL[c] = h[2 * c];
        if (Ito2) Ito2[c] = h[2 * c + 1];
    }
    return GW_OK;
}

int gw_batch_set_spin_limit(gw_batch *B, int64_t polls, char *err, size_t errlen)
{
    if (!B || polls < 0) {
        set_err(err, errlen, "gw_batch_set_spin_limit: polls must be >= 0");
        return GW_E_INVALID_ARG;
    }
    B->a.spin_limit = polls > 0 ? polls : kSpinLimit;
    return GW_OK;
}

int gw_batch_get_persistent(gw_batch *B, int32_t *active)
{
    if (!B || !active) return GW_E_INVALID_ARG;
    (void)hipSetDevice(B->ctx->device);
    *active = use_persist(B) ? 1 : 0;
    return GW_OK;
}

int gw_batch_set_steps_per_launch(gw_batch *B, int32_t steps, char *err, size_t errlen)
{
    if (!B || steps < 0 || steps > 2) {
        set_err(err, errlen, "gw_batch_set_steps_per_launch: steps must be 1, 2 or 0 (automatic)");
        return GW_E_INVALID_ARG;
    }
    B->steps_per_launch = steps;
    return GW_OK;
}

int gw_batch_get_steps_per_launch(gw_batch *B, int32_t *steps)
{
    if (!B || !steps) return GW_E_INVALID_ARG;
    (void)hipSetDevice(B->ctx->device);
    *steps = use_pair(B) ? 2 : 1;
    return GW_OK;
}

int gw_batch_set_graph(gw_batch *B, int32_t steps_per_graph, char *err, size_t errlen)
{
    if (!B || steps_per_graph < 0 || steps_per_graph > 4096) {
        set_err(err, errlen, "gw_batch_set_graph: steps_per_graph must be in 0..4096");
        return GW_E_INVALID_ARG;
    }
    B->graph_steps = steps_per_graph;
    return GW_OK;
}

// Internal switches used by gw_run and the replay tests.
int gw_batch_set_mode(gw_batch *B, int32_t frozen, int32_t digest)
{
    if (!B) return GW_E_INVALID_ARG;
    B->frozen = frozen != 0;
    B->a.frozen = frozen != 0;
    B->digest = digest != 0;
    if (!shape_allowed(B, B->cfg)) set_shape(B, kConfigDefault);
    return GW_OK;
}

}  // extern "C"

namespace {

// The loop of run<PRNG> (src/pyGW.hpp:102-122) on a one-cell batch: the state
// after each step i with i % record_every == 0 goes to sink(piece, base) while
// its number, piece.record, is below num_records. A record is on its way and
// expanded by the host while the stream runs the steps after it. Every 10 steps
// of a cell of 64 CRUs one costs 11 us beside them (waiting for it, and a copy
// to pageable memory for each field, cost 127); of 12,500 CRUs, 190 us, the
// host's expansion into fresh pages (395).
template <class Sink>
int run_records(gw_batch *B, double dt, int64_t num_steps, int32_t record_every, int64_t num_records, int form,
                Sink &&sink_piece, char *err, size_t errlen)
{
    if (num_steps == 0) return GW_OK;
    int rc = launch_cfg_check(B, err, errlen);
    if (rc || (rc = prepare(B, err, errlen))) return rc;
    PieceQueue q;
    if ((rc = pieces_open(q, B, 0, form, err, errlen))) return rc;
    auto sink = [&](const PieceQueue::Piece &p, void *base) {   // a head stands first in either form
        const int64_t st = static_cast<const PieceHead *>(base)->status;
        if (st != 0) return cell_error(0, static_cast<int32_t>(st), err, errlen);
        sink_piece(p, base);
        return static_cast<int>(GW_OK);
    };
    constexpr int64_t kUnchecked = 4096;   // steps launched beyond the last whose status is or will be read
    double t = 0.0;
    int64_t counter = 0, unchecked = 0;
    for (int64_t i = 0; i < num_steps;) {
        // next record after step i_rec (i_rec % record_every == 0, i_rec >= i)
        const int64_t i_rec = ((i + record_every - 1) / record_every) * record_every;
        const int64_t upto = std::min(num_steps, i_rec + 1);
        while (i < upto) {
            const int64_t n = std::min(upto - i, kUnchecked - unchecked);
            HIP_TRY(launch_steps(B, B->steps_done, n));
            B->steps_done += n;
            for (int64_t k = 0; k < n; ++k) t += dt;
            i += n;
            unchecked += n;
            if (unchecked == kUnchecked) {
                if ((rc = pieces_drain(q, sink, err, errlen)) || (rc = check_status(B, err, errlen))) return rc;
                unchecked = 0;
            }
        }
        if (i == i_rec + 1) {
            if (counter < num_records) {
                if ((rc = pieces_push(q, counter, t, sink, err, errlen))) return rc;
                unchecked = 0;
            }
            ++counter;
        }
    }
    if ((rc = pieces_drain(q, sink, err, errlen))) return rc;
    return unchecked > 0 ? check_status(B, err, errlen) : GW_OK;
}

template <class Sink>
int run_loop(gw_ctx *ctx, const gw_params_t *p, int32_t n_cru, double dt, int64_t num_steps, const double *istim,
             int32_t record_every, const gw_globals_t *g0, const gw_cru_state_t *c0, uint64_t seed, int32_t prng_id,
             int32_t precision, int64_t num_records, int form, Sink &&sink_piece, char *err, size_t errlen,
             bool noalloc = false)
{
    if (!ctx || !p || n_cru <= 0 || num_steps < 0 || record_every <= 0) {
        set_err(err, errlen, "gw_run: invalid arguments (n_cru > 0, num_steps >= 0, record_every > 0 required)");
        return GW_E_INVALID_ARG;
    }
    gw_cell_desc_t d;
    std::memset(&d, 0, sizeof(d));
    d.n_cru = n_cru;
    d.seed = seed;
    d.params = *p;
    d.protocol.kind = GW_PROTO_TABLE;
    gw_batch *B = nullptr;
    int rc;
    if (noalloc) {
        if (!ctx->scratch) {
            set_err(err, errlen, "gw_run_noalloc: no scratch address for device %d", ctx->device);
            return GW_E_INVALID_ARG;
        }
        rc = batch_create(ctx, 1, &d, precision, prng_id, dt, g0, ctx->scratch, kScratchBytes,
                          istim ? num_steps : 0, &B, err, errlen);
    } else {
        rc = batch_create(ctx, 1, &d, precision, prng_id, dt, g0, nullptr, 0, istim ? num_steps : 0, &B, err, errlen);
    }
    if (rc) return rc;
    gw_batch_set_mode(B, 0, 0);
    if (c0) {
        gw_cru_state_t c = *c0;
        c.JLCC = nullptr;  // a reference run starts with JLCC = 0 (GW.hpp:104-113)
        rc = gw_batch_set_cru_state(B, 0, &c, err, errlen);
        if (rc) { gw_batch_destroy(B); return rc; }
    }
    if (num_steps > 0 && istim) {
        rc = gw_batch_set_stimulus_table(B, 0, istim, num_steps, err, errlen);
        if (rc) { gw_batch_destroy(B); return rc; }
    }
    rc = run_records(B, dt, num_steps, record_every, num_records, form, sink_piece, err, errlen);
    gw_batch_destroy(B);
    return rc;
}

// gw_run and gw_run_noalloc: the same run, records in the full layout.
int run_full(gw_ctx *ctx, const gw_params_t *p, int32_t n_cru, double dt, int64_t num_steps, const double *istim,
             int32_t record_every, const gw_globals_t *g0, const gw_cru_state_t *c0, uint64_t seed, int32_t prng_id,
             int32_t precision, gw_record_t *out, char *err, size_t errlen, bool noalloc)
{
    const int64_t n = n_cru;
    auto scalars = [&](int64_t k, double t, const gw_globals_t &g) {
#define PUT(f, v) if (out->f) out->f[k] = (v)
        PUT(t, t); PUT(V, g.V); PUT(m, g.m); PUT(h, g.h); PUT(j, g.j); PUT(Nai, g.Nai); PUT(Ki, g.Ki);
        PUT(Cai, g.Cai); PUT(CaNSR, g.CaNSR); PUT(CaLTRPN, g.CaLTRPN); PUT(CaHTRPN, g.CaHTRPN); PUT(xKs, g.xKs);
#undef PUT
        if (out->XKr) for (int q = 0; q < 5; ++q) out->XKr[k * 5 + q] = g.Kr[q];
        if (out->XKv14) for (int q = 0; q < 10; ++q) out->XKv14[k * 10 + q] = g.Kv14[q];
        if (out->XKv43) for (int q = 0; q < 10; ++q) out->XKv43[k * 10 + q] = g.Kv43[q];
    };
    const bool f32 = precision == GW_PREC_FP32_LOCAL;
    auto record = [&](const PieceQueue::Piece &p, void *base) {
        const int64_t k = p.record;
        if (p.i0 == 0) scalars(k, p.t, static_cast<const PieceHead *>(base)->g);
        gw_cru_state_t c;
        c.CaSS = out->CaSS ? out->CaSS + k * n * 4 : nullptr;
        c.CaJSR = out->CaJSR ? out->CaJSR + k * n : nullptr;
        c.LCC = out->LCC ? out->LCC + k * n * 4 : nullptr;
        c.LCC_inactivation = out->LCC_inactivation ? out->LCC_inactivation + k * n * 4 : nullptr;
        c.ClCh = out->ClCh ? out->ClCh + k * n * 4 : nullptr;
        c.RyR = out->RyR ? out->RyR + k * n * 24 : nullptr;
        c.JLCC = nullptr;
        expand_piece(base, p.i0, p.m, f32, c);
    };
    return run_loop(ctx, p, n_cru, dt, num_steps, istim, record_every, g0, c0, seed, prng_id, precision,
                    out ? out->num_records : 0, PIECE_CRUS, record, err, errlen, noalloc);
}

}  // namespace

extern "C" {

int gw_run(gw_ctx *ctx, const gw_params_t *p, int32_t n_cru, double dt, int64_t num_steps, const double *istim,
           int32_t record_every, const gw_globals_t *g0, const gw_cru_state_t *c0, uint64_t seed, int32_t prng_id,
           int32_t precision, gw_record_t *out, char *err, size_t errlen)
{
    return run_full(ctx, p, n_cru, dt, num_steps, istim, record_every, g0, c0, seed, prng_id, precision, out, err,
                    errlen, false);
}

int gw_run_noalloc(gw_ctx *ctx, const gw_params_t *p, int32_t n_cru, double dt, int64_t num_steps,
                   const double *istim, int32_t record_every, const gw_globals_t *g0, const gw_cru_state_t *c0,
                   uint64_t seed, int32_t prng_id, int32_t precision, gw_record_t *out, char *err, size_t errlen)
{
    return run_full(ctx, p, n_cru, dt, num_steps, istim, record_every, g0, c0, seed, prng_id, precision, out, err,
                    errlen, true);
}

int gw_run_reduced(gw_ctx *ctx, const gw_params_t *p, int32_t n_cru, double dt, int64_t num_steps,
                   const double *istim, int32_t record_every, const gw_globals_t *g0, const gw_cru_state_t *c0,
                   uint64_t seed, int32_t prng_id, int32_t precision, gw_record_reduced_t *out, char *err,
                   size_t errlen)
{
    const int64_t n = n_cru;
    auto scalars = [&](int64_t k, double t, const gw_globals_t &g) {
#define PUT(f, v) if (out->f) out->f[k] = static_cast<float>(v)
        PUT(t, t); PUT(V, g.V); PUT(m, g.m); PUT(h, g.h); PUT(j, g.j); PUT(Nai, g.Nai); PUT(Ki, g.Ki);
        PUT(Cai, g.Cai); PUT(CaNSR, g.CaNSR); PUT(CaLTRPN, g.CaLTRPN); PUT(CaHTRPN, g.CaHTRPN); PUT(xKs, g.xKs);
#undef PUT
        if (out->XKr) for (int q = 0; q < 4; ++q) out->XKr[k * 4 + q] = static_cast<float>(g.Kr[q]);
        if (out->XKv14) for (int q = 0; q < 9; ++q) out->XKv14[k * 9 + q] = static_cast<float>(g.Kv14[q]);
        if (out->XKv43) for (int q = 0; q < 9; ++q) out->XKv43[k * 9 + q] = static_cast<float>(g.Kv43[q]);
    };
    auto record = [&](const PieceQueue::Piece &p, void *base) {
        const int64_t k = p.record;
        if (p.i0 == 0) scalars(k, p.t, static_cast<const PieceHead *>(base)->g);
        gw_cru_state_reduced_t c;
        c.CaSS = out->CaSS ? out->CaSS + k * n * 4 : nullptr;
        c.CaJSR = out->CaJSR ? out->CaJSR + k * n : nullptr;
        c.LCC = out->LCC ? out->LCC + k * n * 4 : nullptr;
        c.LCC_inactivation = out->LCC_inactivation ? out->LCC_inactivation + k * n * 4 : nullptr;
        c.ClCh = out->ClCh ? out->ClCh + k * n * 4 : nullptr;
        c.RyR = out->RyR ? out->RyR + k * n * 4 : nullptr;
        expand_reduced(base, p.i0, p.m, c);
    };
    return run_loop(ctx, p, n_cru, dt, num_steps, istim, record_every, g0, c0, seed, prng_id, precision,
                    out ? out->num_records : 0, PIECE_REDUCED, record, err, errlen);
}

int gw_run_batch(gw_ctx *ctx, int32_t ncells, const gw_cell_desc_t *cells, int32_t precision, double dt, int64_t nsteps,
                 gw_globals_t *g_out, gw_cell_obs_t *obs_out, char *err, size_t errlen)
{
    gw_batch *B = nullptr;
    int rc = gw_batch_create(ctx, ncells, cells, precision, GW_PRNG_XOSHIRO256SS, dt, nullptr, &B, err, errlen);
    if (rc) return rc;
    gw_batch_set_mode(B, 0, 0);
    rc = gw_batch_step(B, nsteps, err, errlen);
    if (!rc && g_out) rc = gw_batch_get_globals(B, g_out, err, errlen);
    if (!rc && obs_out) rc = gw_batch_get_obs(B, obs_out, err, errlen);
    gw_batch_destroy(B);
    return rc;
}

}  // extern "C"
