// Input projection of one LSTM layer over all time steps, on the gfx950 matrix cores:
//   out[T, N] (fp32) = x[T, K] (fp16) . w[N, K]^T (fp16) + bias[N] (fp32)
// with N = 4H gate rows and K the layer's input width.  Both operands are contiguous along K, which is
// the natural operand layout of v_mfma_f32_16x16x32_f16: lane l of a wavefront supplies 8 consecutive K
// values of row (l % 16), starting at K offset 8 * (l / 16), for A (x) and for B (w) alike, and
// receives out rows 4 * (l / 16) .. + 3 of column (l % 16).
//
// Grid (1-D): one block of 256 lanes per 16 * NT output columns and 64 time steps, 8 * ceil(column tiles / 8) * row
// blocks per projection.  Requirements checked by the launcher:
// K % 8 == 0, 16-byte aligned x and w, row pitches % 8 == 0.
#pragma once

#include "device_common.h"
#include "xproj_plan.h"

namespace pimhip
{
// A fragment-shaped load straight from global memory (16 lanes on 16 different rows) makes the vector cache look up one
// line per lane, which caps a CU at about 16 bytes per clock (measured: ~35 GB/s per CU, whatever the unrolling).  So
// the operands go through LDS, which only serves as a layout converter: the block reads 128-column slabs of its 64 x rows
// and 16 * NT w rows with row-contiguous 16-byte loads (16 adjacent lanes = 256 contiguous bytes), keeps the next slab in
// registers while the current one is multiplied, and every wavefront reads its fragments from LDS with ds_read_b128 (row
// pitch 272 bytes: 16 lanes x 16 bytes fall into 64 distinct banks).  The four wavefronts split K inside a slab (one
// 32-wide MFMA step each) and each accumulates the whole 64 x 16 * NT tile; the four partial tiles are added through LDS
// in a fixed order at the end.
static constexpr int kXprojTile = 64;    // time steps per block
static constexpr int kXprojKSplit = 4;   // wavefronts per block = MFMA K steps per slab
static constexpr int kXprojSlab = 32 * kXprojKSplit;  // K values per slab (128)
static constexpr int kXprojPitch = kXprojSlab + 8;    // LDS row pitch in halves (272 bytes)

// Up to two projections of the same x in one launch (the two directions of a bidirectional layer): blocks
// [p * blocks_per_problem, (p + 1) * blocks_per_problem) work on weight / bias / output set p.
struct XprojProblems {
    const half_t* w[2];
    const float* bias[2];
    float* out[2];
    int blocks_per_problem;
};

// NT: column tiles of 16 per block (2, or 1 when a single row block would leave CUs without work).
template <int NT>
__global__ __launch_bounds__(256) void input_projection_f16_kernel(const half_t* __restrict__ x, XprojProblems problems,
                                                                  int T, int K, int N, long ldx, long ldw, int row_blocks)
{
    const int problem = blockIdx.x >= (unsigned)problems.blocks_per_problem ? 1 : 0;
    const int block = blockIdx.x - problem * problems.blocks_per_problem;
    const half_t* __restrict__ w = problems.w[problem];
    const float* __restrict__ bias = problems.bias[problem];
    float* __restrict__ out = problems.out[problem];
    constexpr int ROWS = kXprojTile + 16 * NT;            // LDS rows per slab: x rows first, then w rows
    constexpr int CHUNKS = ROWS * (kXprojSlab / 8);       // 16-byte pieces per slab
    constexpr int PER_LANE = CHUNKS / 256;                // 5, 6 or 8
    static_assert(CHUNKS % 256 == 0, "slab must divide evenly over the block");
    constexpr int SLAB_BYTES = ROWS * kXprojPitch * 2;
    constexpr int RED_BYTES = kXprojKSplit * 4 * NT * 64 * 16;
    constexpr int LDS_BYTES = 2 * SLAB_BYTES > RED_BYTES ? 2 * SLAB_BYTES : RED_BYTES;
    __shared__ __align__(16) unsigned char lds[LDS_BYTES];  // two slabs while multiplying, the partial tiles afterwards

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int ks = tid >> 6;  // this wavefront's MFMA step inside a slab
    const int r16 = lane & 15;
    const int kq = lane >> 4;  // which 8-wide K slice of a 32-wide MFMA step this lane feeds
    // Workgroups go to the eight XCDs round-robin by linear id, and each XCD has its own L2.  All row blocks of a column
    // tile are therefore given ids that are equal modulo 8: the tile's slice of w is then pulled into one L2 once and
    // shared by its row blocks, instead of crossing the fabric once per row block and XCD.
    const int xcd = block & 7;
    const int local = block >> 3;
    const int col_tile = (local / row_blocks) * 8 + xcd;
    if (col_tile * (16 * NT) >= N) return;  // whole block, before any barrier
    const int n_base = col_tile * (16 * NT);
    const int t_base = (local % row_blocks) * kXprojTile;

    // Global side of the slab copy: piece i of this lane is row (tid + 256 i) / 16, 8-wide column (tid + 256 i) % 16.
    const half_t* src[PER_LANE];
    int dst[PER_LANE];  // LDS offset in halves within a slab
    const int kcol = (tid & 15) * 8;
#pragma unroll
    for (int i = 0; i < PER_LANE; ++i) {
        const int row = (tid >> 4) + 16 * i;
        // rows past T or N duplicate the last row; their results are never stored
        src[i] = row < kXprojTile ? x + (long)min(t_base + row, T - 1) * ldx
                                  : w + (long)min(n_base + row - kXprojTile, N - 1) * ldw;
        dst[i] = row * kXprojPitch + kcol;
    }

    half8_t zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
    float4_t acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int slabs = (K + kXprojSlab - 1) / kXprojSlab;
    // One register stage: the loads of slab s + 1 are issued before slab s is multiplied and written to the other LDS
    // buffer after it.  (A second register stage, with a barrier that does not wait for global loads, measured slower.)
    half8_t stage[PER_LANE];
    auto fetch = [&](int slab) {
        const int k = slab * kXprojSlab + kcol;
        const bool ok = k < K;  // K % 8 == 0: an 8-wide piece is entirely in or out of range
        const int kc = ok ? k : 0;
#pragma unroll
        for (int i = 0; i < PER_LANE; ++i) {
            const half8_t v = *reinterpret_cast<const half8_t*>(src[i] + kc);
            stage[i] = ok ? v : zero;
        }
    };
    auto deposit = [&](int buf) {
        half_t* base = reinterpret_cast<half_t*>(lds + buf * SLAB_BYTES);
#pragma unroll
        for (int i = 0; i < PER_LANE; ++i) *reinterpret_cast<half8_t*>(base + dst[i]) = stage[i];
    };

    fetch(0);
    deposit(0);
    __syncthreads();
    for (int s = 0; s < slabs; ++s) {
        if (s + 1 < slabs) fetch(s + 1);
        const half_t* base = reinterpret_cast<const half_t*>(lds + (s & 1) * SLAB_BYTES) + ks * 32 + kq * 8;
        half8_t a[4], b[NT];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = *reinterpret_cast<const half8_t*>(base + (m * 16 + r16) * kXprojPitch);
#pragma unroll
        for (int n = 0; n < NT; ++n) b[n] = *reinterpret_cast<const half8_t*>(base + (kXprojTile + n * 16 + r16) * kXprojPitch);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b[n], acc[m][n], 0, 0, 0);
        // Slab s + 1 goes into the other buffer, which every wavefront stopped reading before the previous barrier.
        if (s + 1 < slabs) deposit((s + 1) & 1);
        __syncthreads();
    }

    float(*red)[4 * NT][64][4] = reinterpret_cast<float(*)[4 * NT][64][4]>(lds);  // [K split][tile][lane][4 rows]
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) *reinterpret_cast<float4_t*>(&red[ks][m * NT + n][lane][0]) = acc[m][n];
    __syncthreads();

    // Wavefront `ks` now finishes the row tile m = ks: lane (r16, kq) holds rows 4 * kq .. + 3 of column r16 of a tile.
    const int m = ks;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        float4_t v = *reinterpret_cast<const float4_t*>(&red[0][m * NT + n][lane][0]);
#pragma unroll
        for (int q = 1; q < kXprojKSplit; ++q) {
            const float4_t p = *reinterpret_cast<const float4_t*>(&red[q][m * NT + n][lane][0]);
            v[0] += p[0];
            v[1] += p[1];
            v[2] += p[2];
            v[3] += p[3];
        }
        const int col = n_base + n * 16 + r16;
        if (col < N) {
            const float bv = bias ? bias[col] : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = t_base + m * 16 + kq * 4 + i;
                if (t < T) out[(long)t * N + col] = v[i] + bv;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The same product with w re-laid out once (at plan creation) in MFMA fragment order, so that w never passes through
// LDS: a wavefront's B fragment of a (16-row tile j, 32-wide K step s) is the 1 KB at ((j * ksteps + s) * 64 + lane) * 8
// halves, lane = kq * 16 + r16 holding w[16 j + r16][32 s + 8 kq .. + 7]; rows past N and columns past K are zero;
// ksteps = padded K / 32 with K padded to a multiple of kXprojSlab.  Only x goes through LDS, which halves the LDS
// traffic per MFMA (the bound of the kernel above).
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_w_fragments_kernel(const half_t* __restrict__ w, half_t* __restrict__ wp, int N, int K,
                                                               long ldw, int ntiles, int ksteps)
{
    const long chunk = (long)blockIdx.x * 256 + threadIdx.x;  // one 16-byte piece of the packed matrix
    const long total = (long)ntiles * ksteps * 64;
    if (chunk >= total) return;
    const int lane = (int)(chunk & 63);
    const long frag = chunk >> 6;
    const int s = (int)(frag % ksteps);
    const int j = (int)(frag / ksteps);
    const int row = j * 16 + (lane & 15);
    const int k = s * 32 + (lane >> 4) * 8;
    half8_t v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (half_t)0.0f;
    if (row < N && k < K) v = *reinterpret_cast<const half8_t*>(w + (long)row * ldw + k);  // K % 8 == 0
    reinterpret_cast<half8_t*>(wp)[chunk] = v;
}

struct XprojPackedProblems {
    const half_t* wp[2];
    const float* bias[2];
    float* out[2];
    int blocks_per_problem;
};

// Ranges of 16-byte words that the blocks behind the projection's own set to all-ones bytes: the hand-over slots of the
// pipeline launch that follows (lstm_xcd_kernels.h), marked "not written yet" beside the projection instead of by a launch
// of their own between the two.
struct XprojFill {
    unsigned int* ptr[6];
    unsigned int words16[6];
    int count;        // ranges; 0: the launch has no such blocks
    int first_block;  // the first block that fills
    int blocks;       // how many do
};

__device__ __forceinline__ void xproj_fill_ones(const XprojFill& f, int fb, int n_threads)
{
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 ones = {~0u, ~0u, ~0u, ~0u};
    for (int r = 0; r < f.count; ++r) {
        u32x4* p = reinterpret_cast<u32x4*>(f.ptr[r]);
        const size_t n = f.words16[r];
        for (size_t i = (size_t)fb * n_threads + threadIdx.x; i < n; i += (size_t)f.blocks * n_threads) p[i] = ones;
    }
}

// KS wavefronts per block, one 32-wide K step of a (32 * KS)-wide slab each.
template <int NT, int KS = kXprojKSplit>
__global__ __launch_bounds__(64 * KS) void input_projection_packed_f16_kernel(const half_t* __restrict__ x, XprojPackedProblems problems,
                                                                         int T, int K, int N, long ldx, int ksteps,
                                                                         int row_blocks, XprojFill fill)
{
    if (fill.count > 0 && (int)blockIdx.x >= fill.first_block) {
        xproj_fill_ones(fill, (int)blockIdx.x - fill.first_block, 64 * KS);
        return;
    }
    constexpr int SLAB = 32 * KS;                          // K values per slab
    constexpr int PITCH = SLAB + 8;                        // LDS row pitch in halves
    constexpr int CPR = SLAB / 8;                          // 16-byte pieces per x row and slab
    constexpr int CHUNKS = kXprojTile * CPR;               // 16-byte pieces of an x slab
    constexpr int PER_LANE = CHUNKS / (64 * KS);           // 4
    constexpr int SLAB_BYTES = kXprojTile * PITCH * 2;
    constexpr int RED_BYTES = KS * 4 * NT * 64 * 16;
    constexpr int LDS_BYTES = 2 * SLAB_BYTES > RED_BYTES ? 2 * SLAB_BYTES : RED_BYTES;
    __shared__ __align__(16) unsigned char lds[LDS_BYTES];

    const int problem = blockIdx.x >= (unsigned)problems.blocks_per_problem ? 1 : 0;
    const int block = blockIdx.x - problem * problems.blocks_per_problem;
    const half_t* __restrict__ wp = problems.wp[problem];
    const float* __restrict__ bias = problems.bias[problem];
    float* __restrict__ out = problems.out[problem];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int ks = tid >> 6;
    const int r16 = lane & 15;
    const int kq = lane >> 4;
    const int xcd = block & 7;  // column tiles pinned to one XCD, as above
    const int local = block >> 3;
    const int col_tile = (local / row_blocks) * 8 + xcd;
    if (col_tile * (16 * NT) >= N) return;
    const int n_base = col_tile * (16 * NT);
    const int t_base = (local % row_blocks) * kXprojTile;

    const half_t* src[PER_LANE];
    int dst[PER_LANE];
    const int kcol = (tid % CPR) * 8;
#pragma unroll
    for (int i = 0; i < PER_LANE; ++i) {
        const int row = tid / CPR + (64 * KS / CPR) * i;
        src[i] = x + (long)min(t_base + row, T - 1) * ldx;
        dst[i] = row * PITCH + kcol;
    }
    // This wavefront's B fragments: tile (col_tile * NT + n), K step 4 * slab + ks.
    const half8_t* wfrag[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wfrag[n] = reinterpret_cast<const half8_t*>(wp) + ((long)(col_tile * NT + n) * ksteps + ks) * 64 + lane;

    half8_t zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
    float4_t acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int slabs = (ksteps + KS - 1) / KS;
    half8_t stage[PER_LANE];
    half8_t b_next[NT];
    auto fetch = [&](int slab) {
        const int k = slab * SLAB + kcol;
        const bool ok = k < K;
        const int kc = ok ? k : 0;
#pragma unroll
        for (int i = 0; i < PER_LANE; ++i) {
            const half8_t v = *reinterpret_cast<const half8_t*>(src[i] + kc);
            stage[i] = ok ? v : zero;
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) b_next[n] = (slab * KS + ks < ksteps) ? wfrag[n][(long)slab * KS * 64] : zero;
    };
    auto deposit = [&](int buf) {
        half_t* base = reinterpret_cast<half_t*>(lds + buf * SLAB_BYTES);
#pragma unroll
        for (int i = 0; i < PER_LANE; ++i) *reinterpret_cast<half8_t*>(base + dst[i]) = stage[i];
    };

    fetch(0);
    deposit(0);
    __syncthreads();
    for (int s = 0; s < slabs; ++s) {
        half8_t b[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) b[n] = b_next[n];
        if (s + 1 < slabs) fetch(s + 1);
        const half_t* base = reinterpret_cast<const half_t*>(lds + (s & 1) * SLAB_BYTES) + ks * 32 + kq * 8;
        half8_t a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = *reinterpret_cast<const half8_t*>(base + (m * 16 + r16) * PITCH);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[m], b[n], acc[m][n], 0, 0, 0);
        if (s + 1 < slabs) deposit((s + 1) & 1);
        __syncthreads();
    }

    float(*red)[4 * NT][64][4] = reinterpret_cast<float(*)[4 * NT][64][4]>(lds);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) *reinterpret_cast<float4_t*>(&red[ks][m * NT + n][lane][0]) = acc[m][n];
    __syncthreads();
    if (ks >= 4) return;  // four row tiles, finished by the first four wavefronts
    const int m = ks;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        float4_t v = *reinterpret_cast<const float4_t*>(&red[0][m * NT + n][lane][0]);
#pragma unroll
        for (int q = 1; q < KS; ++q) {
            const float4_t p = *reinterpret_cast<const float4_t*>(&red[q][m * NT + n][lane][0]);
            v[0] += p[0];
            v[1] += p[1];
            v[2] += p[2];
            v[3] += p[3];
        }
        const int col = n_base + n * 16 + r16;
        if (col < N) {
            const float bv = bias ? bias[col] : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = t_base + m * 16 + kq * 4 + i;
                if (t < T) out[(long)t * N + col] = v[i] + bv;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Many time steps.  The kernels above split K over the wavefronts of a 64 x 32 tile: 12 KB pass through LDS (6 KB PACKED), written
// and read, for 16 matrix instructions, and a load has one slab of time to arrive; they level off at 13 % of the matrix cores' rate.  Here a block of
// eight wavefronts owns BM = 32 * MT time steps x 128 columns, a wavefront 16 * MT x 64 of them over half of a slab's 64 columns (two
// wavefronts per SIMD, and a chain of sums half as long): 4 + MT fragments read for 4 * MT matrix instructions.
//   - Loads go from memory straight into LDS, four slabs deep, and are counted, not drained (vmcnt): a slab has the time of two
//     others to arrive.  Staged through registers one slab ahead (two blocks per CU) a slab took 1.0 us, this way 0.53.
//   - The fragments of the next slab are asked for while this one is multiplied: 0.43 us.  What is left is the 0.21 us of matrix
//     instructions and the latency of the reads: nothing holds their order, and as compiled most of a slab's products stand in front of
//     the next slab's reads (matrix cores busy 30 %, LDS reads 18 % of a busy CU's time).
//   - An LDS row is 128 bytes, its 16-byte piece c in place c ^ (row & 7), so that eight rows of one piece fall on all banks.  The
//     weights are the first operand: a lane's four results are neighbours in a row of out (one 16-byte store).
//   - PACKED: the weights' fragments (pack_w_fragments_kernel) pass through LDS as they are; the same products in the same order.
//   - Two slabs' products are one chain of sums in the matrix cores and are then added to the total on the vector units: as far
//     from the exact sum as the kernels above at 64 columns, closer from there on (relative 0.84e-7 against 1.12e-7 at 1024).
// 800 x 1024 -> 4096, MI355X: 24.6 -> 14.5 us (packed 19.4 -> 14.4), 2048 x 1024 -> 4096 56.2 -> 32.8 (305 -> 520 TFLOP/s).
// ---------------------------------------------------------------------------------------------
static constexpr int kXprojTileSlab = 64;
static constexpr int kXprojTileBufs = 4;

struct XprojTileProblems {
    const half_t* w[2];  // PACKED: in fragment order
    const float* bias[2];
    float* out[2];
    int blocks_per_problem;
};

// 16 bytes per lane from memory straight into LDS: lane l's at `lds_base` + 16 l (lds_base: the same in all lanes).  Counted by
// vmcnt; nothing but an explicit wait orders it.  (The compiler allocates m0 to nothing and sets it in front of each use of its
// own, but it joins equal settings of m0 where it sees none in between: it is told of this one, and warns that m0 is reserved.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds16(const half_t* src, unsigned int lds_base)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_base), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int N>
__device__ __forceinline__ void wait_loads_and_barrier()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

template <bool PACKED, int MT>
__global__ __launch_bounds__(512) void input_projection_tile_f16_kernel(const half_t* __restrict__ x, XprojTileProblems problems, int T, int K,
                                                                        int N, long ldx, long ldw, int ksteps, int row_blocks, XprojFill fill)
{
    if (fill.count > 0 && (int)blockIdx.x >= fill.first_block) {
        xproj_fill_ones(fill, (int)blockIdx.x - fill.first_block, 512);
        return;
    }
    typedef float float4_any_t __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int BM = 32 * MT;
    constexpr int XP = BM / 64;                   // 16-byte pieces of x per lane and slab
    constexpr int WP = kXprojTileCols / 64;       // of w
    constexpr int PER_SLAB = XP + WP;
    constexpr int W_AT = BM * kXprojTileSlab;     // halves: x rows first, then w
    constexpr int SLAB_HALVES = (BM + kXprojTileCols) * kXprojTileSlab;
    constexpr int LDS_HALVES = kXprojTileBufs * SLAB_HALVES;
    static_assert(LDS_HALVES * 2 >= 8 * (MT / 2) * 4 * 64 * 16, "the partial tiles of the K halves pass through the same memory");
    __shared__ __align__(16) half_t lds[LDS_HALVES];

    const int problem = blockIdx.x >= (unsigned)problems.blocks_per_problem ? 1 : 0;
    const int block = blockIdx.x - problem * problems.blocks_per_problem;
    const half_t* __restrict__ w = problems.w[problem];
    const float* __restrict__ bias = problems.bias[problem];
    float* __restrict__ out = problems.out[problem];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = (wave >> 1) & 1, ks = wave >> 2;
    const int r16 = lane & 15;
    const int kq = lane >> 4;
    // Workgroups go to the eight XCDs round-robin by linear id; each XCD takes one contiguous eighth of the tiles, counted down the
    // columns: its L2 holds the weights of few column tiles, and no XCD has more tiles than the others (column tiles dealt whole to
    // the XCDs: 13.7 against 9.9 us at 1300 x 1024 -> 1280, 19 against 17 at 2048 x 240 -> 4096, the same where eight divides them).
    const int col_tiles = (N + kXprojTileCols - 1) / kXprojTileCols;
    const int tile = (block & 7) * (problems.blocks_per_problem >> 3) + (block >> 3);
    if (tile >= row_blocks * col_tiles) return;  // whole block, before any barrier
    const int n_base = tile / row_blocks * kXprojTileCols;
    const int t_base = tile % row_blocks * BM;

    // Loads: instruction i of this wavefront brings rows 64 i + 8 wave .. + 7 of the slab, lane l piece (l & 7) ^ (row & 7) of row
    // 8 wave + (l >> 3).  Rows past T or N duplicate the last one; their results are never stored.
    const int lrow = 8 * wave + (lane >> 3);
    const int kpiece = ((lane & 7) ^ (lrow & 7)) * 8;
    const half_t* src[PER_SLAB];
#pragma unroll
    for (int i = 0; i < XP; ++i) src[i] = x + (long)min(t_base + lrow + 64 * i, T - 1) * ldx;
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        if constexpr (PACKED) {  // one fragment (16 rows, 32 columns) per instruction: fragment 8 i + wave of the slab's sixteen, [tile][step]
            const int ntiles = (N + 63) / 64 * 4;
            const int f = 8 * i + wave;
            src[XP + i] = w + (((long)min(n_base / 16 + (f >> 1), ntiles - 1) * ksteps + (f & 1)) * 64 + lane) * 8;
        } else {
            src[XP + i] = w + (long)min(n_base + lrow + 64 * i, N - 1) * ldw;
        }
    }
    const int slabs = (K + kXprojTileSlab - 1) / kXprojTileSlab;
    const unsigned int lds0 = (unsigned int)(size_t)(__attribute__((address_space(3))) half_t*)lds;
    auto fetch = [&](int slab) __attribute__((always_inline)) {
        const unsigned int base = lds0 + (unsigned int)((slab % kXprojTileBufs) * SLAB_HALVES * 2) + (unsigned int)wave * 1024u;
        const int k = slab * kXprojTileSlab + kpiece;
        const int kc = k < K ? k : 0;  // (what lies past K is replaced by zeros when it is read; slabs past the last one are never read)
        const int wslab = min(slab, slabs - 1);
#pragma unroll
        for (int i = 0; i < XP; ++i) load_lds16(src[i] + kc, base + (unsigned int)(i * 8192));
#pragma unroll
        for (int i = 0; i < WP; ++i) load_lds16(src[XP + i] + (PACKED ? (long)wslab * 1024 : (long)kc), base + (unsigned int)(W_AT * 2 + i * 8192));
    };

    float4_t total[MT][4], part[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) total[m][n] = part[m][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    half8_t zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;

    // The fragments of slab s + 1 are read while slab s is multiplied (reads and matrix instructions behind one barrier, all
    // wavefronts in step, would take turns).
    half8_t a[2][MT], b[2][4];
    auto read = [&](int s, int set) __attribute__((always_inline)) {
        const half_t* base = lds + (s % kXprojTileBufs) * SLAB_HALVES;
        const int place = ((ks * 4 + kq) ^ (r16 & 7)) * 8;
#pragma unroll
        for (int m = 0; m < MT; ++m) a[set][m] = *reinterpret_cast<const half8_t*>(base + ((wm * MT + m) * 16 + r16) * kXprojTileSlab + place);
#pragma unroll
        for (int n = 0; n < 4; ++n)
            b[set][n] = *reinterpret_cast<const half8_t*>(base + W_AT + (PACKED ? ((wn * 4 + n) * 2 + ks) * 512 + lane * 8
                                                                               : ((wn * 4 + n) * 16 + r16) * kXprojTileSlab + place));
    };
    auto mask = [&](int s, int set) __attribute__((always_inline)) {  // K % 8 == 0: a piece is entirely in or out of range
        const bool ok = s * kXprojTileSlab + (ks * 4 + kq) * 8 < K;
#pragma unroll
        for (int m = 0; m < MT; ++m) a[set][m] = ok ? a[set][m] : zero;
#pragma unroll
        for (int n = 0; n < 4; ++n) b[set][n] = ok ? b[set][n] : zero;
    };
    auto multiply = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) part[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[set][n], a[set][m], part[m][n], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < kXprojTileBufs - 1; ++s) fetch(s);
    wait_loads_and_barrier<(kXprojTileBufs - 2) * PER_SLAB>();
    fetch(kXprojTileBufs - 1);
    read(0, 0);
    auto add_up = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                total[m][n] += part[m][n];
                part[m][n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };
    auto advance = [&](int s) __attribute__((always_inline)) {  // slab s is there; everybody has read slab s - 1
        wait_loads_and_barrier<(kXprojTileBufs - 2) * PER_SLAB>();
        fetch(s + kXprojTileBufs - 1);
    };
    int s = 0;
    for (; s + 2 < slabs; s += 2) {  // (no condition inside: a wait would be sized for the path with the fewest reads in flight)
        advance(s + 1);
        read(s + 1, 1);
        multiply(0);
        advance(s + 2);
        read(s + 2, 0);
        multiply(1);
        add_up();
    }
    const bool ragged = slabs * kXprojTileSlab != K;
    if (s + 1 < slabs) {
        advance(s + 1);
        read(s + 1, 1);
        multiply(0);
        if (ragged) mask(s + 1, 1);
        multiply(1);
    } else {
        if (ragged) mask(s, 0);
        multiply(0);
    }
    add_up();

    // The two K halves of a tile: each wavefront hands the other half of its row tiles over and finishes its own.
    wait_loads_and_barrier<0>();
    float4_t* red = reinterpret_cast<float4_t*>(lds);  // [wave][MT / 2][4][64]
#pragma unroll
    for (int m = 0; m < MT / 2; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) red[((wave * (MT / 2) + m) * 4 + n) * 64 + lane] = ks ? total[m][n] : total[m + MT / 2][n];
    __syncthreads();

    // Lane (r16, kq) holds columns 4 kq .. + 3 of time step r16 of every 16 x 16 tile.
    const bool whole = n_base + kXprojTileCols <= N;
    float4_t bv[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int col = n_base + (wn * 4 + n) * 16 + kq * 4;
        bv[n] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (bias && whole) bv[n] = *reinterpret_cast<const float4_any_t*>(bias + col);
        else if (bias) bv[n] = float4_t{bias[min(col, N - 1)], bias[min(col + 1, N - 1)], bias[min(col + 2, N - 1)], bias[min(col + 3, N - 1)]};
    }
#pragma unroll
    for (int m = 0; m < MT / 2; ++m) {
        const int t = t_base + (wm * MT + ks * (MT / 2) + m) * 16 + r16;
        float* o = out + (long)t * N + n_base + wn * 64 + kq * 4;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const float4_t mine = ks ? total[m + MT / 2][n] : total[m][n];
            const float4_t v = (mine + red[(((wave ^ 4) * (MT / 2) + m) * 4 + n) * 64 + lane]) + bv[n];
            if (whole && t_base + BM <= T) {
                *reinterpret_cast<float4_any_t*>(o + n * 16) = v;
            } else if (whole) {
                if (t < T) *reinterpret_cast<float4_any_t*>(o + n * 16) = v;
            } else if (t < T) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n_base + (wn * 4 + n) * 16 + kq * 4 + i < N) o[n * 16 + i] = v[i];
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Few columns, many weight rows, several weights at once: out_l[row][s] = sum_k w_l[row][k] . enc[s][k], the context columns of a
// decoder's layers over the S encoder positions of a sentence.  25 MB of weights against 24 KB of enc: a stream, which the kernel
// at the top of this file ran on the 64 workgroups its 64 x 32 tiles gave it, one launch per layer (3 x 11 us).  Here a block
// takes 32 rows of one layer, its four wavefronts a quarter of K each (every fourth 32-wide step); a wavefront asks for all
// its weights at once, straight in fragment order (16 lanes on 16 rows: slow on one CU, but with every CU at it faster than
// the memory), keeps them in 64 registers and runs over the columns 16 at a time.  Sums in the order of the kernel at the top.
// ---------------------------------------------------------------------------------------------
static constexpr int kCtxRows = 32;                        // weight rows per block
static constexpr int kCtxMaxK = 1024;
static constexpr int kCtxSteps = kCtxMaxK / 32 / kXprojKSplit;  // 32-wide steps per wavefront
static constexpr int kCtxMaxLayers = 4;

struct CtxProjProblems {
    const half_t* w[kCtxMaxLayers];
    float* out[kCtxMaxLayers];
};

__global__ __launch_bounds__(256) void context_projection_f16_kernel(const half_t* __restrict__ enc, int S, int K, int N, long ldw,
                                                                     CtxProjProblems problems)
{
    typedef float float4_any_t __attribute__((ext_vector_type(4), aligned(4)));
    __shared__ __align__(16) float4_t red[2][kXprojKSplit][kCtxRows / 16][64];
    const int lane = threadIdx.x & 63;
    const int ks = threadIdx.x >> 6;
    const int r16 = lane & 15;
    const int kq = lane >> 4;
    const int row0 = blockIdx.x * kCtxRows;
    const half_t* __restrict__ w = problems.w[blockIdx.y];
    float* __restrict__ out = problems.out[blockIdx.y];

    half8_t zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
    // K % 8 == 0: a piece is entirely in or out of range; rows past N duplicate the last one and are not stored
    half8_t wf[kCtxRows / 16][kCtxSteps];
#pragma unroll
    for (int i = 0; i < kCtxSteps; ++i) {
        const int k = (i * kXprojKSplit + ks) * 32 + kq * 8;
#pragma unroll
        for (int m = 0; m < kCtxRows / 16; ++m)
            wf[m][i] = k < K ? *reinterpret_cast<const half8_t*>(w + (long)min(row0 + m * 16 + r16, N - 1) * ldw + k) : zero;
    }
    for (int s0 = 0, buf = 0; s0 < S; s0 += 16, buf ^= 1) {
        const half_t* e = enc + (long)min(s0 + r16, S - 1) * K;
        half8_t ef[kCtxSteps];
#pragma unroll
        for (int i = 0; i < kCtxSteps; ++i) {
            const int k = (i * kXprojKSplit + ks) * 32 + kq * 8;
            ef[i] = k < K ? *reinterpret_cast<const half8_t*>(e + k) : zero;
        }
        float4_t acc[kCtxRows / 16];
#pragma unroll
        for (int m = 0; m < kCtxRows / 16; ++m) {
            acc[m] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < kCtxSteps; ++i) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ef[i], wf[m][i], acc[m], 0, 0, 0);
            red[buf][ks][m][lane] = acc[m];
        }
        __syncthreads();  // (the other buffer was last read in front of the previous barrier)
        if (ks < kCtxRows / 16) {
            // lane (r16, kq) holds positions s0 + 4 kq .. + 3 of weight row r16 of the tile
            float4_t v = red[buf][0][ks][lane];
#pragma unroll
            for (int q = 1; q < kXprojKSplit; ++q) v += red[buf][q][ks][lane];
            const int row = row0 + ks * 16 + r16, s = s0 + kq * 4;
            if (row < N && s < S) {
                float* o = out + (long)row * S + s;
                if (s + 3 < S) {
                    *reinterpret_cast<float4_any_t*>(o) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (s + i < S) o[i] = v[i];
                }
            }
        }
    }
}

// bsum[i] = b_ih[i] + b_hh[i] in fp32 (either may be null, meaning zero).
__global__ void lstm_bias_sum_kernel(const half_t* __restrict__ b_ih, const half_t* __restrict__ b_hh,
                                     float* __restrict__ bsum, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) bsum[i] = (b_ih ? (float)b_ih[i] : 0.0f) + (b_hh ? (float)b_hh[i] : 0.0f);
}

}  // namespace pimhip
