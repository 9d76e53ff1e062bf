// gw_route.h -- which launch configuration a batch's steps run in, as a function
// of the shape asked for, the batch's size and the device's compute units.
// Nothing of it needs a GPU or the HIP headers.
#pragma once

#include "../../include/gw_capi.h"

#include <stdint.h>

namespace gw {

// The launch configurations: lanes per CRU (4: a quad per CRU, FP64 or
// FP32-local; 1: one lane per CRU, FP32-local), threads per block, and CRUs
// per lane (lane kernels only: each wave owns 64 x that many CRUs and refills
// its lanes as CRUs finish their step).
struct LaunchCfg {
    int lanes, threads, cpl;
};
constexpr int kNumConfigs = GW_LAUNCH_CONFIGS;
constexpr int kConfigDefault = 2;
constexpr int kLane1 = 4;   // one CRU per lane; the shapes after it repeat its 64, 128 and 256 threads
constexpr int kLane64 = kNumConfigs;   // the FP64 one-lane kernels of 2, 4 and 8 CRUs per lane, which route chooses
constexpr LaunchCfg kConfigs[kNumConfigs + 3] = {
    {4, 64, 1},  {4, 128, 1}, {4, 256, 1}, {4, 512, 1},                 // quads: 16..128 CRUs per block
    {1, 64, 1},  {1, 128, 1}, {1, 256, 1},                               // one lane per CRU
    {1, 64, 2},  {1, 128, 2}, {1, 256, 2},                               // two CRUs per lane, refilled
    {1, 64, 4},  {1, 128, 4}, {1, 256, 4},                               // four
    {1, 64, 8},  {1, 128, 8}, {1, 256, 8},                               // eight (up to 2048 CRUs per block)
    {4, 64, 2},  {4, 64, 4},  {4, 128, 4}, {4, 256, 4},                  // quads refilled from 2 or 4 CRUs each
    {1, 64, 2},  {1, 64, 4},  {1, 64, 8}};                               // FP64, one lane per CRU

static_assert(kConfigs[0].lanes == 4 && kConfigs[0].threads == 64 && kConfigs[0].cpl == 1 &&
                  kConfigs[kConfigDefault].lanes == 4 && kConfigs[kConfigDefault].threads == 256 &&
                  kConfigs[kConfigDefault].cpl == 1,
              "the two quad shapes that run");
constexpr bool refill_shapes_in_order()
{
    for (int c = kLane1; c < kLane1 + 12; ++c)
        if (kConfigs[c].lanes != 1 || kConfigs[c].threads != 64 << (c - kLane1) % 3 || (kConfigs[c].cpl == 1) != (c < kLane1 + 3))
            return false;
    return true;
}
static_assert(refill_shapes_in_order(), "route's arithmetic on the one-lane shapes");

struct BatchSize {
    bool f32;        // FP32-local
    int64_t crus;    // of all cells
    int32_t cells;
    int32_t cus;     // compute units of the device
};

// A crossing measured on 256 compute units: it is a number of rounds that the
// batch's waves make of the device's slots (of closes per compute unit, for the
// cells), so on a part of the device it lies in proportion.
constexpr int kRouteCus = 256;
constexpr int64_t crossing(int64_t measured, const BatchSize &b) { return measured * b.cus / kRouteCus; }

// The configuration that runs for one asked for: that one, except where another
// gives the same results faster (the same bits, but for refilled FP32-local lanes,
// whose FP64 sums are in another order than one CRU per lane's; equal in every
// run compared).
//
// Plain quads (FP64 or FP32-local) run with 256 threads per block, whose close
// has four waves, while the close is the longer half of a step, and with 64,
// whose blocks wait on fewer waves, where the SSA is. In us per step with 256
// and 64 threads: FP64, 12,500 CRUs 7.4 and 16.8; 150,000 18.5 and 19.1;
// 200,000 22.2 and 21.6; 450,000 44 and 40; 300 cells of 200 CRUs 14.5 and
// 13.6; FP32-local, 300,000 CRUs 19.9 and 20.7; 400,000 24.8 and 23.1; 300
// cells of 200 CRUs 11.3 and 13.5. (128 and 512 lie between or behind.)
//
// Large FP64 batches run one lane per CRU. In us per step early in an action
// potential, the lanes with two steps per launch (4 x 64 quads; one lane with
// 2, 4 and 8 CRUs per lane; - not run): 300,000 CRUs 29.1, 31.2, 36.0, -;
// 350,000 32.3, 31.2, -, -; 390,000 35.0, 31.7, -, -; 525,000 44.4, 39.9, 42.7, -; 800,000
// 65.3, 51.2, 53.2, -; 900,000 70.5, 54.1, 54.9, -; 1.0 M 77.4, 58.3, 55.5,
// -; 2.5 M -, 125, 116, -; 12.8 M 1,182, -, 526, 463. Below, a batch is a few
// rounds of quads and one round of lanes, whose trips are longer. Cells of
// fewer CRUs than a wave has lanes stay with the quads (20,000 cells of 33
// CRUs 300 and 317 us, of 66 CRUs 178 and 173).
//
// FP32-local shapes of several CRUs per lane run one per lane, on as many
// threads, below 300,000 CRUs: there all of them fit the wave slots at once, and
// a wave's chain of CRUs is what a step waits for. In us per step with 4 and 1
// per lane, 64 threads: 12,500 CRUs 17.2 and 10.0; 200 cells of 333 20.3 and
// 12.3; 90,000 19.4 and 12.0; 200,000 20.7 and 14.9; 300,000 23.0 and 19.0;
// 440,000 25.8 and 25.0; 3,000 cells of 140 60.4 and 62.5.
constexpr int64_t kRefillCrus = 300000;
constexpr int64_t kLane64Crus = 340000, kLane64Crus4 = 950000, kLane64Crus8 = 2500000;
constexpr int64_t kQuad64Crus = 180000, kQuad64CrusF32 = 350000, kQuad64Cells = 256;

constexpr int route(int cfg, const BatchSize &b)
{
    if (!b.f32 && b.crus >= crossing(kLane64Crus, b) && b.crus >= int64_t(64) * b.cells)
        return kLane64 + (b.crus < crossing(kLane64Crus4, b) ? 0 : b.crus < crossing(kLane64Crus8, b) ? 1 : 2);
    const LaunchCfg &L = kConfigs[cfg];
    if (L.lanes == 1 && L.cpl > 1 && b.crus < crossing(kRefillCrus, b)) return kLane1 + (cfg - kLane1) % 3;
    if (L.lanes != 4 || L.cpl != 1) return cfg;
    const bool narrow = b.f32 ? b.crus >= crossing(kQuad64CrusF32, b)
                              : b.crus >= crossing(kQuad64Crus, b) || b.cells >= crossing(kQuad64Cells, b);
    return narrow ? 0 : kConfigDefault;
}

// Whether a running configuration that can do either runs two steps per launch:
// batches of 450,000 CRUs and more, where the state's HBM traffic is worth more
// than the separate close kernel costs, 10 us per two steps. FP32-local, one and
// two steps per launch, in us per step: 400,000 CRUs 25.2 and 25.0 (four CRUs per
// lane), 24.7 and 24.0 (one); 600,000 31.5 and 27.9, 30.8 and 28.5; 200,000 20.7
// and 21.6, 15.1 and 17.3. The FP64 one-lane kernels always do: 390,000 CRUs 33.6
// and 31.7; 450,000 41.0 and 37.5; 600,000 47.4 and 43.4.
constexpr int64_t kPairCrus = 450000;

constexpr bool route_pair(int running, const BatchSize &b)
{
    return running >= kLane64 || b.crus >= crossing(kPairCrus, b);
}

}  // namespace gw
