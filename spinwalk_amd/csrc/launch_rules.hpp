// launch_rules.hpp -- how a walk is launched, as rules on its sizes: whether its spins
// are visited sorted and how many a wave carries.  None changes a result.  Plain C++.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace sw {

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

}  // namespace sw
