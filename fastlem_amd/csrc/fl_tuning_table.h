// fl_tuning_table.h -- launch tunings by workload class.  Rows are tried in
// order; the first whose max_sites and terrain kind match a solve gives its
// tuning.  A tuning shapes launches only: every row gives the same results.
//
// The rows are set by hand from timings of each class (named beside it, with the
// workgroup sizes' times).  The autotuner (fastlem_amd/autotune.py, which calls
// fl_autotune on each class and can write this file) starts from them and takes
// another value only where it is faster by more than one percent: it keeps the
// 65k and 1M terrains' rows and both batches', and would take two others that gain
// 1.6 and 1.5 percent on its own terrain and lose on the next.
//
// Workgroup sizes of the per-site kernels: smaller ones spread a small terrain
// over more compute units (fewer wavefronts of a workgroup wait for its slowest
// row); at hundreds of thousands of sites the sizes differ by under one percent.
#pragma once

#include <stdint.h>

struct fl_tuning_row {
  uint64_t max_sites;  // union sites up to this many
  uint32_t batch;      // 0: one terrain, 1: several
  uint32_t site_block, long_chain, tail_units, pipelining, compact_min_idle;
};

static const fl_tuning_row fl_tuning_table[] = {
    // two terrains of 10k sites: 256 4.94, 128 4.74, 64 4.68 ms.  (long_chain 6: 16k
    // sites 1.63 instead of 1.66 ms, 30k with max slopes 10.17 instead of 10.10)
    {32768ull, 0, 64, 16, 32, 1, 65536u},
    // two of 80k: 256 8.12, 128 7.90, 64 7.85 ms
    {131072ull, 0, 64, 16, 32, 1, 65536u},
    // two of 400k: 256 29.94, 128 29.72, 64 29.91, 512 30.78 ms.  (64: 262k sites 10.20
    // instead of 10.35 ms, a strip of as many 38.45 instead of 38.15)
    {524288ull, 0, 128, 16, 32, 1, 65536u},
    // two of 1M: 256 59.45, 128 59.03, 64 59.24, 512 60.85 ms
    {UINT64_MAX, 0, 128, 16, 16, 1, 65536u},
    // two batches of 48 terrains, 1000..32768: 256 16.82, 128 16.74 ms
    {1317794ull, 1, 128, 16, 16, 1, 65536u},
    // batch of 64 terrains, 1000..262144 sites: 137.6 ms, no other value of a parameter
    // faster by one percent
    {UINT64_MAX, 1, 256, 16, 16, 1, 65536u},
};
