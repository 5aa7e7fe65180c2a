// launch_rules.hpp -- how a walk is launched, as rules on its sizes: whether its spins
// are visited sorted, how many a wave carries, which loop walks them, and whether the
// waves on a SIMD are capped.  None changes a result.  Plain C++.
#pragma once
#include <math.h>
#include <stdint.h>

#include <algorithm>

namespace sw {

constexpr uint64_t kWaveSpins = 64 * 1024;               // a wave on each of the 1024 SIMDs

// Spins per wave of a single walk.  A wave takes as long as the slowest of its lanes,
// the one that meets the most vessel walls and redraws, and a SIMD with one wave waits
// out every latency of it.  So where waves of half as many spins still find a SIMD
// each, half the lanes stay empty, 64 lanes against 32: 64^3, GRE of 400 steps, 1e3
// spins 260 -> 238 us, 3.2e4 302 -> 275; 256^3, 3e2 spins 182 -> 184 us, 2e3 219 -> 214,
// 3.2e4 288 -> 263; bSSFP of 20 dummies 1.38 -> 1.25 ms at 8e3; replayed spin echo of
// 2e4 spins 1.26 -> 0.93 ms.  Shorter waves lose again below 2 blocks a CU (8 lanes: 0.6 to
// 0.75 of the rate of 64 at 1e3 spins), and above the line the waves share issue slots
// (32 lanes 1.00 of the rate at 6.5e4 spins, 0.86 at 1e5).
inline uint32_t single_lanes(uint32_t n_local) { return n_local <= 32u * 1024 ? 32 : 64; }

// Whether a single walk that asks for spatial order gets it.  Sorted spins share
// lines with their neighbours, which pays when more lines are in use than the L2s hold
// (8 of 4 MiB in 128-byte lines: 262144).  Below that every spin keeps its lines by
// itself, and order only costs: its launches, and waves of neighbours, some of which all
// meet vessel walls and redraw while others are long done.  The same when the records
// fit each L2.  A spin uses the more lines the longer its step (in voxels, the standard
// deviation of one axis): sorted time over unsorted, 200 steps, FP32, 8-voxel blocks of
// two permeable tissues,
//                    step 0.16   0.32   0.63   1.26   2.5
//   256^3, 6.5e4 spins   1.14    1.15   1.13   1.12   1.06
//          1.3e5         1.15    1.14   1.11   0.87   0.85
//          2e5           1.14    1.11   0.85   0.82   0.84
//   400^3, 1.3e5         1.16    1.11   1.11   0.97   0.96
//          2e5           1.12    1.09   1.02   0.95   0.94
//   128^3, 2e5           1.05    1.02   0.89   0.73   0.73
// so the line falls as 1 / (1 + 2 step), down to 90000 spins, below which steps longer
// still cost no more lines (every step meets another).  It stands at 212992 spins for
// steps up to 0.31:
// 800 steps of 0.32, 256^3 0.98 to 1.10 at 2e5 spins, 0.74 to 0.94 at 3e5; 600^3 1.10 at
// 2.1e5; int16 records of 200^3 1.04 at 2.4e5, 0.84 at 3e5; 64^3, whose records fit, 1.35 at
// 1.3e5 and 1.25 at 5e5.
constexpr uint64_t kUnsortedBytes = 4ull << 20;
inline uint32_t unsorted_spins(double step) {
    return (uint32_t)std::min(212992., std::max(90000., 346000. / (1. + 2. * step)));
}
inline bool order_pays(uint32_t n_local, uint64_t rec_bytes, double step) {
    return n_local > unsorted_spins(step) && rec_bytes >= kUnsortedBytes;
}

// Whether a single walk of one TR in single precision takes the general loop and not that
// of walk_prod.hpp, whose rare blocks (walls, crossings) are the longer ones where a wave
// has a SIMD to itself.  That shows between the half-filled waves and two waves a SIMD
// where a wave meets such a block at nearly every step: long steps, or crossings that read
// their probability from global memory (more tissues than the LDS tables take).  General
// loop over production loop, 400 steps:
//                                      1e3 spins  3e4    3.3e4  6.5e4  1e5    1.4e5  4e5
//   2 tissues, 128^3, step 0.2          1.09      1.05   1.00   0.99   1.01   1.04   1.04
//                          0.63         1.02      0.99   0.95   0.95   0.96   0.97   1.01
//   20 tissues, permeable, step 0.32    1.1 (2e3)        0.92   0.92   0.94   0.96   1.0 (5e5)
// In double precision the production loop is the faster by 1.04 to 1.14 throughout.
inline bool general_loop(uint32_t n_local, bool f64, double step, bool global_crossings) {
    return !f64 && n_local > 32u * 1024 && n_local <= 128u * 1024 && (step >= 0.5 || global_crossings);
}

// Whether the waves on a SIMD are held to kCapWaves (4) in a single walk, or a batch's to
// 4 and not 5.  Each spin in flight comes back to the lines it last read; the waves that
// fit a SIMD (8) hold more lines than an L2, so fewer waves wait less.  What they wait
// for grows with
//  - the records that the spins in flight on an XCD meet: of the whole phantom when
//    unsorted, of an eighth when sorted (an XCD's part), of it the share of its spins
//    that 8 waves are, and around it what spins drift over the walk;
//  - the step (in voxels): how often a spin needs another line, and of how many.
// cap_reach is the product, MiB voxel^2.  The lines are where uncapped and capped time
// cross over 80^3 to 500^3, steps of 0.1 to 2.5, 160 to 5100 time points, float32 and int16
// records, 4e5 to 2e6 spins.  Uncapped time over capped (for a batch, 5 waves over 4),
// nine tenths of the measurements below and above the line:
//                       line   below          above
//   one TR              0.85   0.92 to 1.12   0.98 to 1.49   (FP32 256^3, step 0.32, 800 points: 1.26 at 4e5 spins)
//   dummy TRs           1.1    0.92 to 1.02   0.96 to 1.49
//   two attempts        1.85   0.92 to 1.00   0.99 to 1.11   (a trip of the loop: records above 256 MiB; 500^3, 1e6
//                                                             spins of a spin echo of 2000 points 1.02)
//     with dummy TRs    2.5    0.93 to 0.98   0.98 to 1.14
//   batch, dummy TRs    8      0.88 to 1.01   0.95 to 1.23
//   fused, one TR       1.2    0.91 to 1.06   0.99 to 1.34
//   fused, dummy TRs    2.1    0.89 to 1.03   0.96 to 1.35   (1000^3 with 2e6 spins 117.4 -> 109.0 ms)
// A batch of scans with one TR goes by the records alone (kCapWindow, without drift): its
// tiles of one phantom meet in the same lines where few are in flight.  The FoV sweep's 64
// tiles, whose reach is 0 to 8, run 95.3 ms at 4 waves and 104.2 at 5; six tiles of one scale
// 0.90 to 0.97 below a reach of 2, 0.94 to 1.16 above.
// Only from 6 waves a SIMD on, so that the last round is not a fraction of the others: 3e5
// spins (4.6 waves) 0.82 to 0.88 on 256^3.
enum CapKind : int { CAP_SINGLE = 0, CAP_PAIRS = 1, CAP_BATCH = 2, CAP_FUSED = 3 };
constexpr double kCapWindow = 2.8;
// The records in reach, MiB; drift: how far spins spread over the walk, in voxels.
inline double cap_window(uint64_t rec_bytes, double voxels, uint64_t n_tile, bool sorted, double drift) {
    const double part = sorted ? std::min(1., 8. * (double)kWaveSpins / (double)n_tile) / 8 : 1.;
    const double side = cbrt(voxels * part) + 0.7 * drift;           // 0.35 standard deviations each way
    return (double)rec_bytes / (1 << 20) * std::min(1., side * side * side / voxels);
}
inline double cap_reach(uint64_t rec_bytes, double voxels, uint64_t n_tile, bool sorted, double step, double n_steps) {
    const double often = std::min(step, 0.65);           // longer steps meet another line every time
    return cap_window(rec_bytes, voxels, n_tile, sorted, step * sqrt(n_steps)) * often * often;
}
inline bool cap_pays(CapKind kind, bool one_tr, double reach, double window, uint64_t n_all) {
    constexpr double kLine[4][2] = {{1.1, 0.85}, {2.5, 1.85}, {8., 0.}, {2.1, 1.2}};
    if (n_all < 6 * kWaveSpins) return false;
    return kind == CAP_BATCH && one_tr ? window > kCapWindow : reach > kLine[kind][one_tr];
}

}  // namespace sw
