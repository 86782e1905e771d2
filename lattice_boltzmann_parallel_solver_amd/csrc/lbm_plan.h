// Which of the kernels with the same results a run takes: times of their
// launches, from measurements on MI355X, compared.  Plain C++ (no HIP), so that
// the rules can be tested on the host.
#pragma once

#include <stdint.h>

#include "lbm_types.h"

namespace lbm {

// Time of a one-step launch among others, us.  Fitted to 1600 lattices of up to 8
// million nodes (within 5 % on nine of ten, 12 % at most below): the launch, 3 to 4
// us, and the planes read and written at 7.9 TB/s (FP64), 7.8 to 10 (FP32, faster
// below 36 MB) and 6.5 (FP16, whose arithmetic is that of FP32), a third slower
// out of the last-level cache, and up to 1.5 times in rows of 64 columns or fewer.
double step_us(int storage, const Geom &g, bool program);

// Time of a two-step launch of whole rows or column tiles, us: rounds of
// `resident` row ranges of `rows` rows each.  A block walks its rows one after
// another, so a range costs its rows and three or four more (the halo rows and the
// first loads), 3.7 to 4.9 us each whatever the storage, by the waves and columns
// per thread of the block, less without an outlet and half to 0.7 of it without a
// boundary program.  Of blocks of five and of ten waves a CU holds one less than the
// runtime says (five waves: two, not three, in FP64 and five, not six, else; ten:
// two, not three), and the ranges left over start late: rows of 300 columns in
// FP16 take 3.7 us each with 1250 ranges on 1536 places and 4.9 with 1397.
double sweep2_us(int storage, const Geom &g, bool program, bool outlet, const SweepShape &sh, int rows, int resident);

// Whether the library's own choice is two steps per launch, with extra_us a
// launch on top (the rows that a pressure fix reaches).  us a step, one step per
// launch / two, channels: FP16 400x1030 6.8 / 10.4, 1600x1030 15.0 / 19.6,
// 520x640 6.3 / 8.1, 1332x284 6.9 / 8.2, 3300x400 14.9 / 12.6; FP32 300x1100 6.6 /
// 8.1, 400x900 6.7 / 6.6, 1100x1800 22.6 / 21.1; FP64 270x1030 9.4 / 10.9, 1200x514
// 16.1 / 15.2.  Over 753 lattices measured both ways this rule loses 3 % on one and
// nothing on the others, and leaves 7 to 15 % on 7.
bool two_steps_pay(int storage, const Geom &g, bool program, bool outlet, const SweepShape &sh, int rows, int resident,
                   double extra_us);

// Most threads of a block of the tile kernel (its registers).
constexpr int tile_threads(size_t elem, bool pressure) { return elem == 8 ? (pressure ? 512 : 768) : (pressure ? 768 : 1024); }

// Time of a launch of k steps of the tile kernel among others, us: the launch and
// its last stores, each further round of blocks, for every step of a round a barrier
// and LDS part and one for every wave that a SIMD holds, and the bytes that the
// blocks load, halos included, at 6 to 12 TB/s.  Fitted to 5200 runs of 400 to 2^18
// nodes, all storages and kinds of boundary: launches of all of a tiling's steps
// within 5 % on nine of ten.
double tile_us(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k);

// The tiling of a lattice, or K = 0 where it does not pay (tile_pays; above 2^18
// nodes in FP64, 3 * 2^16 in FP32 and FP16, it never did).  The tilings are compared by
// 3.3 us a round and, for each step, 0.35 us and one part for every wave that a SIMD
// holds, 0.4 us in FP64 and 0.12 in FP32 and FP16: shorter than the launches are, but
// in their order.  us a step, single steps / tiles: FP64 channels 300x300 6.0 / 2.3,
// 203x494 6.1 / 3.8, with the pressure fix 551x412 8.2 / 13.3, 1403x170 9.1 / 12.2,
// 56x838 5.3 / 3.8; FP32 652x294 with the fix 5.9 / 5.3; FP16 1656x115 5.8 / 6.6.
// Takes 10 to 40 us.
TileShape pick_tile(int storage, const Geom &g, bool program, bool pressure, int cus, double other_us);

// Whether a launch of k <= sh.K steps of a tiling beats the kernel that would run
// otherwise, with other_us a step (the launch's halos are those of k steps, its rounds of blocks those of the tiling: FP32 67x2897, us a
// step with 2, 3 and 4: 7.3, 5.6 and 4.7, single steps 5.7).
bool tile_pays(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int k,
               double other_us);

// Whether a run of `steps` steps goes through tiles: its last steps, too few for a
// launch of their own, run on the other kernel, which finds the state in other L2
// caches than it would write it to (0.25 us a MB of state, 0.65 without a boundary
// program).  FP64 62x2261, periodic, two steps a launch, us a step in runs of 2, 3, 5
// and 7: 4.2, 7.0, 5.8 and 5.3, single steps 5.4.
bool tile_run_pays(int storage, const Geom &g, bool program, bool pressure, int cus, const TileShape &sh, int64_t steps,
                   double other_us);

}  // namespace lbm
