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

// The most encoder positions for which the context columns of `layers` layers are made by one launch with the weights in registers
// (context_projection_f16_kernel) instead of a launch per layer: it reads enc from the caches once per 32 weight rows, 16 positions
// at a time, so a block's time grows with the positions, and with one layer there is no launch to save.  Measured on MI355X (us of
// set_encoder, launch per layer / one launch):
//   one layer     256 wide at 48 / 80 positions 4.4 / 4.0, 4.5 / 5.2   512 5.6 / 4.9, 5.7 / 6.5   704 at 80 / 117 8.6 / 7.6, 9.0 / 10.3   1024 11.6 / 10.3, 13.7 / 14.0
//   two layers    256 at 160 / 200 8.5 / 8.3, 8.8 / 9.9   1024 at 128 / 160 26.4 / 15.0, 18.2 / 17.9
//   three layers  256 at 160 12.6 / 8.4   1024 at 128 / 160 / 200 39.4 / 21.9, 27.0 / 25.6, 30.0 / 30.7
inline int64_t context_most_positions(int layers, int64_t K) { return layers >= 2 ? 160 : K <= 512 ? 48 : 80; }
}  // namespace pimhip
