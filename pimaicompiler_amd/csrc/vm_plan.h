// How an I_X_W product (gemv_vm_f16_kernel) is cut into column blocks and slices of the reduction: host arithmetic only, so that
// its bounds can be checked without a GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace pimhip
{
static constexpr int kVmWaves = 8;                                        // wavefronts of a block
static constexpr int64_t kVmLargeWeightBytes = 16ll << 20;                // past it the weight's stream is the bound (kKeepCachedBytes)

struct VmPlan {
    int lanes_per_row;    // 8: blocks of 64 columns, 16: of 128
    int col_blocks;
    int by_xcd;           // neighbouring column blocks go to one XCD
    int slices;           // of the reduction; the partial sums of all but the last are exchanged in (slices - 1) * N words
    int rows_per_slice;
    // The product's partial sums never meet those of another caller: it has words of its own where the stream has a region for
    // it, and runs without any elsewhere (vm_needs_no_workspace).
    bool needs_no_workspace;
};

// Weights of at most this many bytes, and operands of no whole 16-byte pieces, touch no workspace a caller would have to order
// replays of a graph, or calls of the static entry point, against.
static constexpr int64_t kVmSmallWeightBytes = 256 * 1024;
inline bool vm_whole_pieces(int64_t N, int64_t lda, uintptr_t weight, uintptr_t results)
{
    return N % 8 == 0 && lda % 8 == 0 && (weight & 15u) == 0 && (results & 15u) == 0;
}
inline bool vm_needs_no_workspace(int64_t K, int64_t N, int64_t lda, uintptr_t weight, uintptr_t results)
{
    return K * N * 2 <= kVmSmallWeightBytes || !vm_whole_pieces(N, lda, weight, results);
}

// The most words the partial sums of any product take: below, (slices - 1) * col_blocks is less than the target, which is at
// most num_cus, and a column block has at most 128 columns.  A workspace of this size never has to grow.
inline size_t vm_max_partials(int num_cus) { return (size_t)num_cus * 128; }

// N >= 8 outputs, K rows of pitch lda at address `weight`; `results`: the addresses of all destinations, or-ed.
inline VmPlan vm_plan(int64_t K, int64_t N, int64_t lda, uintptr_t weight, uintptr_t results, int num_cus)
{
    VmPlan p;
    p.needs_no_workspace = vm_needs_no_workspace(K, N, lda, weight, results);
    // Block width: 64 columns (8 lanes per weight row) while the weight is small, so that more blocks share it: 2048 x 2048
    // 3.5 us against 4.2 with 128 columns, 12896 x 84 4.0 against 6.7.  128 columns for a weight past kVmLargeWeightBytes, whose
    // stream is the bound: 4096 x 4096 7.7 us against 8.2 with 64, 1024 x 32000 11.2 against 13.7.
    const int64_t weight_bytes = K * N * 2;
    p.lanes_per_row = weight_bytes > kVmLargeWeightBytes ? 16 : 8;
    const int cols = 8 * p.lanes_per_row;
    p.col_blocks = (int)((N + cols - 1) / cols);
    // Rows that do not start on a 128-byte line make neighbouring column blocks share lines: they go to one XCD then, whose
    // L2 hands the shared line to both (1024 x 31999: 11.6 us against 16.4), and the weight is read with plain loads.  Where
    // no line is shared the same order costs (4096 x 4096 7.9 -> 9.9 us: eight fronts instead of one).
    p.by_xcd = p.col_blocks >= 16 && (lda % 64 != 0 || (weight & 127u) != 0);
    // Slices of K: about a block per CU for a large weight, 64 blocks for a small one, but a cross-block sum costs 1 to 2 us
    // and grows with the slices: none up to 512 rows (272 x 2357: 3.1 us, two slices 3.6) and at most sqrt(K / 40) of them
    // (12896 rows, 84 columns: 4.0 us with 17, 4.9 with 64), for a large weight, which needs the blocks, sqrt(K / 10) (16384 x 1000
    // 9.9 us with 32, 12.8 with 20; 12000 x 1024 7.7 and 8.9; no limit at all is no faster up to 24000 rows).
    int64_t target = weight_bytes / 65536;
    if (target < 64) target = 64;
    if (target > num_cus) target = num_cus;
    int slices = (int)((target + p.col_blocks / 2) / p.col_blocks);  // rounded: 250 column blocks on 256 CUs are not sliced
    if (K <= 512) slices = 1;
    while (slices > 1 && (int64_t)slices * slices * (weight_bytes > kVmLargeWeightBytes ? 10 : 40) > K) --slices;
    if (slices < 1) slices = 1;
    const int row_groups = kVmWaves * 64 / p.lanes_per_row;
    int64_t rows = (K + slices - 1) / slices;
    rows = (rows + row_groups - 1) / row_groups * row_groups;
    if (rows < row_groups) rows = row_groups;  // K == 0: one empty slice, y = act(bias)
    p.rows_per_slice = (int)rows;
    p.slices = (int)((K + rows - 1) / rows);
    if (p.slices < 1) p.slices = 1;
    return p;
}
}  // namespace pimhip
