// Which kind of products the per-XCD LSTM kernel multiplies with, and where its h lies in LDS (lstm_xcd_kernels.h): plain arithmetic,
// so that both can be checked without a GPU.
#pragma once

#include <stdint.h>

#include "xproj_plan.h"

namespace pimhip
{
// Whether the launches of a layer's two steps make its projection too, in place of a launch for both rows (a launch per step, the layer
// alone or in both directions; a stack of one direction stays with the projection's launch, two layers of 1024 15.3 / 16.7 us).  W_ih is
// then read twice and a launch saved.  What that is worth depends on the kernel that makes the projection of two rows otherwise: the
// split-K kernel, for up to 127 tiles of 128 gate rows, costs nearly always more than a second read, the tiles' kernel of more rows streams
// W_ih as fast as the steps do (us a call, the projection's launch / in the steps, with the same weights again and with plans in turn that
// do not fit the caches; megabytes of W_ih).
//   split-K: one layer of 1024 over 2048 18.9 / 10.0 and 22.7 / 12.8, over 16384 (134) 86 / 46 and 114 / 50; of 1536 over 8192 (101) 54 / 43 and 68 / 46; of 2056 over 2056
//     32.0 / 27.1 and 35.5 / 31.2, over 8192 (135) 64 / 63 and 77 / 67; of 3072 over 3072 (75) 48.1 / 45.9 and 54.4 / 49.5, over 6144 (151) 65.1 / 71.2 and 79.5 / 74.7; two
//     directions of 1024 over 1024 15.5 / 12.5 and 19.0 / 14.9, of 1536 over 4096 (101) 43.3 / 42.7 and 51.4 / 46.4, over 6144 (151) 55.2 / 59.7 and 68.6 / 63.1
//   tiles: one layer of 4096 over 256 (8) 52.9 / 50.3 and 56.1 / 55.6, over 1024 (34) 59.4 / 55.9 and 59.6 / 60.7, over 4096 (134) 72.6 / 92.8 and 86.7 / 97.9; two directions of
//     2056 over 256 (8) 31.8 / 28.1 and 34.6 / 32.6, over 1024 (34) 37.7 / 35.1 and 38.4 / 39.7, over 2056 (68) 43.1 / 47.2 and 50.4 / 51.7, over 4096 (135) 52.9 / 73.5
//     and 62.9 / 77.8
inline bool lstm_two_steps_project(int dirs, int layers, int64_t H, int64_t in_w, int num_cus)
{
    if (dirs == 1 && layers > 1) return false;
    const bool tiles = xproj_tile_rows(2, 4 * H, dirs, false, num_cus) != 0;
    const double megabytes = 8.0 * (double)dirs * (double)H * (double)in_w / (1 << 20);  // of W_ih, 2^20 bytes each
    return tiles ? megabytes <= 32.0 : megabytes <= 96.0 || 4 * H * dirs < 10240;
}

// v_dot2 instead of sparse matrix instructions.  The latter's weights pass through LDS first (1 to 1.6 us per launch), and they take
// whole fragments of 64 columns in groups of four: v_dot2 is better for a few steps of more than 256 units, and longest for 513 to 656, of
// whose second and third group the sparse fragments are half empty.  From 65 to 256 units one group holds the row and there is nothing to
// win.  `chained`: the layers a launch runs as a pipeline, 1 for recurrences that are fed by none other; the more there are, the more steps
// the launch has beside its sequence's.
// The lines were drawn at these figures (MI355X, graph replays, time on v_dot2 over time on sparse instructions), which had v_dot2 ahead
// for fewer than 64 units at any length too:
//   one layer, at 2 / 4 / 6 / 8 / 10 / 16 steps: 64 units 1.00 / 0.95 / 0.99 / 0.99 / 1.01 / 1.01, 128 0.95 / 0.97 / 1.00 / 1.00 / 1.02 / 1.02, 192 1.01 / 1.01 /
//     1.06 / 1.04 / 1.07 / 1.08, 320 0.97 / 0.97 / 0.99 / 1.02 / 1.04 / 1.06, 512 0.94 / 0.97 / 0.99 / 1.02 / 1.04 / 1.07, 640 0.90 / 0.93 / 0.95 / 0.97 / 0.98 / 1.01,
//     768 0.94 / 0.97 / 0.99 / 1.02 / 1.02 / 1.05, 1024 0.95 / 0.98 / 1.00 / 1.02 / 1.04 / 1.08; two directions within 0.02 of these
//   one layer, at 24 / 80 / 200 steps: 8 units 0.97 / 0.95 / 0.95, 32 0.96 / 0.96 / 0.96, 48 0.95 / 0.95 / 0.94, 64 1.00 / 1.01 / 1.01, 128 1.02 / 1.04 / 1.04
//   two layers, at 2 / 3 / 4 / 6 / 8 steps: 128 1.00 / 1.00 / 1.00 / 0.99 / 1.01, 256 1.01 / 1.02 / 1.03 / 1.04 / 1.05, 512 0.96 / 0.98 / 1.00 / 1.02 / 1.03, 640 0.94 /
//     0.96 / 0.97 / 0.98 / 1.00, 768 0.98 / 1.00 / 1.00 / 1.01 / 1.03, 1024 0.97 / 0.99 / 1.01 / 1.03 / 1.05; at 24 / 80 / 200: 8 0.97 / 0.98 / 0.98, 48 0.98 / 0.97 /
//     0.97, 64 1.01 / 1.02 / 1.03
//   three layers, at 2 / 3 / 4: 512 1.01 / 1.01 / 1.02, 640 0.97 / 1.00 / 1.00, 1024 1.00 / 1.02 / 1.03; at 24 / 80 / 200: 16 0.97 / 0.98 / 0.98, 32 1.06 / 1.13 / 1.15;
//     four layers, at 2 / 4 / 8: 16 0.98 .. 1.00, 640 1.00 / 1.01 / 1.03
// What stands around the products on a step's path has been shortened since, for the sparse kind by more (same layout as above): one layer, at 2 / 4 / 6 / 8 / 10 / 16 / 80 steps:
//     8 1.05 / 1.02 / 1.01 / 1.04 / 1.04 / 1.02 / 1.01, 64 1.02 / 1.02 / 1.03 / 1.02 / 1.04 / 1.04 / 1.05, 128 1.00 / 1.01 / 1.01 / 1.02 / 1.04 / 1.06 / 1.09, 512 0.91 / 0.96 / 1.00 /
//     1.03 / 1.05 / 1.12 / 1.26, 640 0.89 / 0.92 / 1.00 / 1.04 / 1.06 / 1.10 / 1.26, 1024 0.93 / 0.97 / 1.01 / 1.05 / 1.09 / 1.16 / 1.38; two layers at 2 / 3 / 4 / 80: 48 1.04 / 1.03 /
//     1.04 / 1.05, 512 0.98 / 1.01 / 1.02 / 1.28, 1024 0.98 / 1.01 / 1.03 / 1.41.
// By these v_dot2 is the slower kind now for all of fewer than 64 units (1 to 5 %), for 64 and 128 (0 to 4 %) and in the last steps in front of the other
// lines (up to 6 %), though no call is slower than it was when the lines were drawn.  A move of the lines changes which sums such calls make,
// and with them last bits of their results.
inline bool xcd_on_dot(int64_t H, int64_t T, int chained)
{
    const bool half_empty = H > 512 && H <= 656;
    if (chained == 1) {
        if (H <= 64) return H < 64 || T < 24;
        return H <= 128 ? T < 8 : H > 256 && T < (half_empty ? 11 : 7);
    }
    if (chained == 2) return H < 64 || (H > 256 && T < (half_empty ? 7 : 4));
    return chained == 3 && (H <= 16 || (half_empty && T < 3));
}

// Where the 16-byte piece p of h lies in LDS.  A read of 8 bytes per lane takes from eight rows of 128 bytes (the row pairs of A) two
// of four pieces; in their own order four of the rows share their banks, and the eight wavefronts' reads of a step took 512 cycles of
// the LDS where 128 do.  Rows 2 q, 2 q + 1 have their pieces exchanged by 0, 1, 4 or 5 instead: every half wavefront reads all banks
// once.  Two layers of 1024, 341 steps 480.6 -> 428.8 us, two directions, 50 steps 82.4 -> 75.0.
constexpr int xcd_h_place(int p) { return p ^ ((p >> 4 & 1) | (p >> 5 & 1) << 2); }

// The first of the two neighbouring pieces of which a lane takes half each for the sparse operand's register set s: the first half for
// even lanes, the second for odd ones.
constexpr int xcd_h_operand_piece(int s, int lane) { return 8 * (8 * s + ((lane & 15) >> 1)) + 2 * (lane >> 4); }
}  // namespace pimhip
