// Which kernel makes an input projection of many time steps: host arithmetic only.
#pragma once

#include <stdint.h>

namespace pimhip
{
static constexpr int kXprojTileCols = 128;  // columns of a tile of input_projection_tile_f16_kernel

inline int xproj_tiles(int64_t T, int64_t N, int rows) { return (int)((T + rows - 1) / rows * ((N + kXprojTileCols - 1) / kXprojTileCols)); }

// The row tiles per wavefront (MT) of the kernel for many time steps, or 0: the split-K kernels.  Measured on MI355X (256 CUs) over
// T = 50 .. 2048, K = 240 .. 2048, N = 1024 .. 4096 (us, split-K kernel / 64-row / 128-row tiles, plain weights):
//   64-row tiles in all   128 (T 200, K 1024, N 4096) 9.7 / 8.7 / -    130 (800, 1024, 1280) 10.6 / 9.2 / 12.4   104 (800, 512, 1024) 6.5 / 7.1 / 8.7
//                         192 (341, 1024, 4096) 12.5 / 9.8 / 13.2      416 (800, 1024, 4096) 24.6 / 17.7 / 14.5  1024 (2048, 1024, 4096) 56 / 37 / 29
// A block fills a CU, so what counts is how many tiles the busiest CU runs one after another, a 128-row tile taking 1.5 times as
// long as a 64-row one.  From half as many 64-row tiles as CUs on they win; against packed weights, whose split-K kernel moves
// half the LDS bytes, from five eighths (128: 8.3 / 8.7, 192: 10.7 / 9.6).
inline int xproj_tile_rows(int64_t T, int64_t N, int count, bool packed, int num_cus)
{
    if ((double)T * (double)N > 1e12) return 0;  // (counts below stay within an int)
    const int t64 = count * xproj_tiles(T, N, 64), t128 = count * xproj_tiles(T, N, 128);
    if (t64 < (packed ? num_cus * 5 / 8 : num_cus / 2)) return 0;
    const int r64 = (t64 + num_cus - 1) / num_cus, r128 = (t128 + num_cus - 1) / num_cus;
    return 2 * r64 <= 3 * r128 ? 2 : 4;
}
}  // namespace pimhip
