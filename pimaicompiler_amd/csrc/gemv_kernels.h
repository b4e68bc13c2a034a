// fp16 batch-1 GEMV kernels for gfx950 (fp16 storage, fp32 accumulation, one rounding at the store).
//
// Two weight orders exist on this path, named after the operand order of the product:
//   MV ("W_X_I"): y[out] = W[out,in] . x[in]   -- weight rows contiguous along the reduction
//   VM ("I_X_W"): y[out] = x[in] . A[in,out]   -- weight rows contiguous along the outputs
// plus VV, the dot product of two vectors.  Every kernel takes the fused epilogue
// y = act(acc + bias) that the reference's addmv kernels define
// (runtime/include/executor/op_executor/custom_ops.h:216-381: bias added after the alpha/beta
// combination, ReLU applied last).
//
// All of them are HBM-bound: each weight element is read from memory exactly once per launch
// through 16-byte non-temporal loads, x stays cache resident, and the only cross-lane traffic is
// the final reduction.
#pragma once

#include <type_traits>

#include "device_common.h"
#include "vm_plan.h"

namespace pimhip
{
// ---------------------------------------------------------------------------------------------
// MV order, vector path.  Requirements checked by the launcher: K % 8 == 0, ldw % 8 == 0,
// W / x 16-byte aligned.
//
// A block holds WAVES wavefronts.  KS consecutive wavefronts share one group of R rows and split
// the reduction dimension between them in an interleaved fashion (wave ks takes 16-byte chunks
// ks*64 + lane, then strides by 64*KS), so one block covers (WAVES / KS) * R rows.  Each lane
// keeps U chunks per row in flight: R*U independent 16-byte weight loads per lane per iteration.
// ---------------------------------------------------------------------------------------------
// SPLIT: x is the concatenation of two vectors that lie apart (x: the first split_chunks 16-byte pieces, x2: the rest);
// compiled out of every other instance.  KEEP: the weight is read with plain loads (load_weight).  ANY: rows, x and K need
// not be multiples of 16 bytes; the same 16-byte loads at whatever address the row has, and the K % 8 columns behind the
// last whole piece one per lane.
template <int R, int U, int WAVES, int KS, bool SPLIT = false, bool KEEP = false, bool ANY = false>
__device__ __forceinline__ void gemv_mv_f16_body(const half_t* __restrict__ W, const half_t* __restrict__ x,
                                                 const half_t* __restrict__ bias, half_t* __restrict__ y, int N,
                                                 int K, long ldw, int relu, int block,
                                                 const half_t* __restrict__ x2 = nullptr, int split_chunks = 0)
{
    static_assert(WAVES % KS == 0, "KS must divide WAVES");
    constexpr int RG = WAVES / KS;  // row groups per block
    __shared__ float red[WAVES][R];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int rg = wave / KS;
    const int ks = wave % KS;
    const long row0 = ((long)block * RG + rg) * R;

    float acc[R];
    const half_t* wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        acc[r] = 0.0f;
        long row = row0 + r;
        if (row > N - 1) row = N - 1;  // out-of-range rows re-read the last row and are never stored
        wrow[r] = W + row * ldw;
        if constexpr (ANY) {
            const int k = (K & ~7) + lane;
            if (ks == 0 && k < K) acc[r] = (float)wrow[r][k] * (float)x[k];
        }
    }
    const half8_t* xv = reinterpret_cast<const half8_t*>(x);
    const half8_t* xv2 = SPLIT ? reinterpret_cast<const half8_t*>(x2) - split_chunks : nullptr;  // (indexed from split_chunks on)
    auto x_at = [&](int c) -> half8_t {
        if constexpr (ANY) return load_weight_any<true>(x + 8 * (long)c);
        return (SPLIT && c >= split_chunks) ? xv2[c] : xv[c];
    };
    auto w_at = [&](const half_t* row, int c) -> half8_t {
        if constexpr (ANY) return load_weight_any<KEEP>(row + 8 * (long)c);
        return load_weight<KEEP>(reinterpret_cast<const half8_t*>(row) + c);
    };
    const int nchunks = K >> 3;
    constexpr int STEP = 64 * KS;

    int c = ks * 64 + lane;
    // Main loop: U chunks per row in flight, all of them in range.
    for (; c + (U - 1) * STEP < nchunks; c += U * STEP) {
        half8_t xr[U];
        half8_t wr[R][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int r = 0; r < R; ++r) wr[r][u] = w_at(wrow[r], c + u * STEP);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) xr[u] = x_at(c + u * STEP);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = dot8(wr[r][u], xr[u], acc[r]);
        }
    }
    // Tail: one chunk per row at a time.
    for (; c < nchunks; c += STEP) {
        half8_t wr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) wr[r] = w_at(wrow[r], c);
        const half8_t xr = x_at(c);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = dot8(wr[r], xr, acc[r]);
    }

#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);

    if (KS > 1) {
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) red[wave][r] = acc[r];
        }
        __syncthreads();
        if (ks == 0 && lane < R) {
            float v = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) v += red[rg * KS + s][lane];
            const long row = row0 + lane;
            if (row < N) {
                if (bias) v += (float)bias[row];
                if (relu) v = relu_f32(v);
                y[row] = (half_t)v;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long row = row0 + r;
            if (lane == r && row < N) {
                float v = acc[r];
                if (bias) v += (float)bias[row];
                if (relu) v = relu_f32(v);
                y[row] = (half_t)v;
            }
        }
    }
}

template <int R, int U, int WAVES, int KS>
__global__ __launch_bounds__(WAVES * 64) void gemv_mv_f16_kernel(const half_t* __restrict__ W,
                                                                 const half_t* __restrict__ x,
                                                                 const half_t* __restrict__ bias,
                                                                 half_t* __restrict__ y, int N, int K, long ldw,
                                                                 int relu)
{
    gemv_mv_f16_body<R, U, WAVES, KS>(W, x, bias, y, N, K, ldw, relu, blockIdx.x);
}

// The same for a small matrix that is used again and again between other work: plain loads (load_weight).  A kernel of its
// own, chosen on the host, so that the streaming kernel stays as it is.
template <int R, int U, int WAVES, int KS>
__global__ __launch_bounds__(WAVES * 64) void gemv_mv_keep_f16_kernel(const half_t* __restrict__ W,
                                                                      const half_t* __restrict__ x,
                                                                      const half_t* __restrict__ bias,
                                                                      half_t* __restrict__ y, int N, int K, long ldw,
                                                                      int relu)
{
    gemv_mv_f16_body<R, U, WAVES, KS, false, true>(W, x, bias, y, N, K, ldw, relu, blockIdx.x);
}

// The same for rows at any address and of any length (K % 8, the row pitch % 8 or an operand's address not those of whole
// 16-byte pieces).  A straddling load touches one line in eight more than an aligned one, which is what is left to the
// aligned kernel's rate: 11624 x 4967 21.3 us (5.4 TB/s; with one wavefront per row and 2-byte loads 76 us), 2049 x 2055
// 8.8 -> 3.0 us, 512 x 1345 4.0 -> 2.1, 40 x 14833 27 -> 2.9.
template <int R, int U, int WAVES, int KS, bool KEEP>
__global__ __launch_bounds__(WAVES * 64) void gemv_mv_any_f16_kernel(const half_t* __restrict__ W,
                                                                     const half_t* __restrict__ x,
                                                                     const half_t* __restrict__ bias,
                                                                     half_t* __restrict__ y, int N, int K, long ldw,
                                                                     int relu)
{
    gemv_mv_f16_body<R, U, WAVES, KS, false, KEEP, true>(W, x, bias, y, N, K, ldw, relu, blockIdx.x);
}

// The same for rows of at most 128 columns: one wavefront per row, 2-byte loads.  A row is two loads per lane here, and a whole
// piece, a tail and a sum over two wavefronts in the kernel above: 32001 x 17 4.3 us against 6.2 (one wavefront per two rows: 4.9),
// 12000 x 129 3.3 / 3.9 (3.4), 1025 x 17 2.34 / 2.6; at 257 columns 7.3 / 8.4 (6.4).
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemv_mv_short_f16_kernel(const half_t* __restrict__ W, const half_t* __restrict__ x,
                                                                    const half_t* __restrict__ bias, half_t* __restrict__ y, int N,
                                                                    int K, long ldw, int relu)
{
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * WAVES + (threadIdx.x >> 6);
    if (row >= N) return;
    const half_t* w = W + row * ldw;
    float acc = 0.0f;
    for (int k = lane; k < K; k += 64) acc = fmaf((float)w[k], (float)x[k], acc);
    acc = wave_sum(acc);
    if (lane == 0) {
        if (bias) acc += (float)bias[row];
        if (relu) acc = relu_f32(acc);
        y[row] = (half_t)acc;
    }
}

// y = act(W . cat(x1, x2) + bias) without the concatenation: the second operand of the RNNT joint network's first layer
// is cat(encoder frame, prediction), which the reference either materialises or splits the product over
// (compiler/source/frontend/optimizer/remove_cat_for_addmm.cpp:46-191: two dependent launches).
template <int R, int U, int WAVES, int KS, bool KEEP>
__global__ __launch_bounds__(WAVES * 64) void gemv_mv_cat2_f16_kernel(const half_t* __restrict__ W,
                                                                      const half_t* __restrict__ x1,
                                                                      const half_t* __restrict__ x2, int split_chunks,
                                                                      const half_t* __restrict__ bias,
                                                                      half_t* __restrict__ y, int N, int K, long ldw,
                                                                      int relu)
{
    gemv_mv_f16_body<R, U, WAVES, KS, true, KEEP>(W, x1, bias, y, N, K, ldw, relu, blockIdx.x, x2, split_chunks);
}

// Several independent MV GEMVs in one launch (sibling projections that the reference issues on separate
// streams, runtime/source/executor/op_executor/stream_ops_executor.cpp:36-47).  Blocks
// [block_begin[i], block_begin[i+1]) work on problem i.
// MAX: as many problems as the arguments have room for.  Arguments for 32 are 1.5 KB, which the host writes and a block's first
// loads fetch from all over: q, k, v and o of 768 with room for 4 instead: 5.3 -> 5.1 us a call,
// 6.2 -> 5.75 on a slower host core.
static constexpr int kGemvGroupMax = 32;
template <int MAX>
struct GemvGroupArgs {
    const half_t* W[MAX];
    const half_t* x[MAX];
    const half_t* bias[MAX];
    half_t* y[MAX];
    int N[MAX];
    int K[MAX];
    int block_begin[MAX];  // (INT_MAX past the last problem)
    unsigned int relu;     // a bit per problem
};

// Each problem runs with the block shape a launch of its own would use for its row length (long rows: the four
// wavefronts of a block split the reduction of two rows; shorter rows: two wavefronts per pair of rows).
static constexpr int kGemvGroupThreads = 256;
static constexpr int kGemvGroupLongRow = 4096;
__host__ __device__ inline int gemv_group_rows_per_block(int K) { return K >= kGemvGroupLongRow ? 2 : 4; }

template <bool KEEP, int MAX>  // KEEP: the group's weights together are small: plain loads (load_weight)
__global__ __launch_bounds__(kGemvGroupThreads) void gemv_mv_f16_group_kernel(GemvGroupArgs<MAX> g)
{
    // All entries at once: a loop that looks at one after the other waits for each, which every block of a large group pays (us, MI355X, such
    // a loop / now: 8 of 768 x 768 3.85 / 3.25, 16 7.3 / 5.45, 32 16.2 / 9.8, 32 of 2048 x 1024 36.4 / 22.6; 9 of 300 x 4096 5.05 / 5.15).
    int i = 0;
#pragma unroll
    for (int j = 1; j < MAX; ++j) i += (int)blockIdx.x >= g.block_begin[j] ? 1 : 0;
    const int block = (int)blockIdx.x - g.block_begin[i];
    if (g.K[i] >= kGemvGroupLongRow)
        gemv_mv_f16_body<2, 4, 4, 4, false, KEEP>(g.W[i], g.x[i], g.bias[i], g.y[i], g.N[i], g.K[i], (long)g.K[i], (int)(g.relu >> i & 1u), block);
    else
        gemv_mv_f16_body<2, 2, 4, 2, false, KEEP>(g.W[i], g.x[i], g.bias[i], g.y[i], g.N[i], g.K[i], (long)g.K[i], (int)(g.relu >> i & 1u), block);
}

// ---------------------------------------------------------------------------------------------
// VM order, N >= 8.  A block owns 8 * LPR adjacent outputs and a slice [k_begin, k_end) of the reduction.  LPR lanes (8
// columns, one 16-byte load each) cover the block's part of one weight row, so a wavefront reads 64 / LPR rows per load
// instruction and the block's eight wavefronts interleave over the rows of the slice, four loads in flight per lane.  The row
// groups' sums meet in LDS; from there on a thread stands for one column, 512 / (8 LPR) threads ("parts") per column.
// gridDim.y slices cover K.  With one slice the block finishes the outputs itself.  With several, the blocks of all
// slices but the last store their partial sums (fp32) in `partial[slice][N]` and exit; the blocks of the LAST slice add
// them to their own sums, in an order that depends on the slice index only (so the result is the same in every run), and
// apply the epilogue.
//
// Rows may lie at any address: a 16-byte load takes what address the row has, and the lane with the last N % 8 columns reads
// the row's last eight and keeps its own.
//
// What bounds it: the stream for a large weight (bytes in flight: eight wavefronts of four loads beat four of eight by 15 %,
// blocks of 16 wavefronts and 8 loads lose again), for a small one the chain launch, rows, LDS, cross-block words, store.  The
// group sums are spread over all threads (one thread per column adding all of them took 0.2-0.4 us more).  Measured on
// MI355X in graph replays against one block of 256 threads per 128 columns, records of 32 bytes and a kernel of 2-byte loads
// for everything not aligned: 4096 x 4096 9.3 -> 7.7 us, 4096 x 16384 22.4 -> 21.2, 16384 x 4096 24.4 -> 22.7, 1024 x 32000
// 12.0 -> 11.2, 1024 x 1024 4.7 -> 3.2; odd sizes: 1024 x 31999 22.1 -> 11.6 us, 4046 x 9937 27.3 -> 14.9, 4951 x 1301
// 30 -> 6.7, 12896 x 84 71 -> 4.0, 1252 x 54 6.5 -> 3.2.
//
// A word that has not arrived yet holds kVmEmpty (the bit pattern 0xffffffff: a NaN that no sum of products of fp16 values
// can be, since arithmetic yields the canonical NaN or the widened payload of an fp16 NaN), so a reducing thread polls
// each of its column's words until it is something else, adds it and writes kVmEmpty back for the next launch.  Words travel
// with device-scope (sc1) stores and loads; there is no fence (a device-scope fence writes back and invalidates the XCD's
// whole L2, once per block) and no ticket counter (store, acknowledgement, atomic, loads would be three trips through the
// memory side after the last block's arithmetic; polling is one).
//
// What the scheme assumes of the dispatcher, and what it does not: the producers never wait for anything, so each of
// them finishes whatever else occupies the GPU, in any dispatch order; results never depend on the order.  That the
// reducing blocks seldom wait long does: workgroups are dealt to the eight XCDs round-robin by linear id and each
// XCD starts its share in that order, so within every XCD the producers (slices 0..last-1) are started before that
// XCD's reducing blocks (the last slice), and a reducing block on one XCD waits at most for the other XCDs to get
// through the producers dealt to them.  When other work holds CUs of one XCD (a resident sequence kernel on another
// stream) that wait grows by as much as that XCD is held up.  It is bounded all the same: after `spin_limit` polls
// of one word (none at all with a limit of 0, which is how a test forces the condition from the host), or one second,
// the thread gives up on the word and computes that slice's sum for its column itself, with the producer's own
// order of operations, so the result has the bits it would have had.  The word may still arrive later and would then
// sit in the workspace as if it belonged to the next launch: the thread raises *poison (a device word the reducing blocks
// of every launch look at) and *status (for the host), and until the host has refilled the words and cleared both,
// reducing blocks do not look at them at all and compute every slice themselves: slow, but right.
// ---------------------------------------------------------------------------------------------
// Destinations of a VM product: the same result is stored to `count` buffers (the GNMT attention context goes
// straight into three concatenation buffers, runtime/source/executor/op_executor/aten_ops_executor.cpp:694-737).
static constexpr int kGemvMaxOuts = 4;
struct GemvOuts {
    half_t* y[kGemvMaxOuts];
    int count;
};

// The sliced kernel's: with the count among the flags, all its arguments are 112 bytes (what more costs a launch: launch_kernel),
// and with them at the end what the first instructions need arrives in scalar registers.
struct VmDests {
    half_t* y[kGemvMaxOuts];
};
static constexpr unsigned int kVmRelu = 1u, kVmByXcd = 2u;
static constexpr int kVmOutsShift = 2;

static constexpr int kVmLoads = 4;  // 16-byte loads in flight per lane

// acc[j] += A[k][j] * x[k] for k, k + GROUPS, .. < k_end, `a` at the lane's eight columns of row 0.
template <bool KEEP, int GROUPS>
__device__ __forceinline__ void vm_sum_rows(float (&acc)[8], const half_t* a, long lda, const half_t* __restrict__ x, int k, int k_end)
{
    constexpr int U = kVmLoads;
    auto take = [&](int k, auto last) __attribute__((always_inline)) {
        half8_t ar[U];
        float xr[U];
        // (rows past the slice re-read its last one and count as zeros: all of a trip's loads are in flight together)
        auto row = [&](int u) { return last ? min(k + u * GROUPS, k_end - 1) : k + u * GROUPS; };
#pragma unroll
        for (int u = 0; u < U; ++u) ar[u] = load_weight_any<KEEP>(a + (long)row(u) * lda);
#pragma unroll
        for (int u = 0; u < U; ++u) xr[u] = (float)x[row(u)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (last && k + u * GROUPS >= k_end) {
                xr[u] = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; ++j) ar[u][j] = (half_t)0.0f;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = fmaf((float)ar[u][j], xr[u], acc[j]);
        }
    };
    for (; k + (U - 1) * GROUPS < k_end; k += U * GROUPS) take(k, std::false_type{});
    if (k < k_end) take(k, std::true_type{});
}

// A row group's eight sums into its row of LDS; the lane with the last N % 8 columns has read the eight before N.
__device__ __forceinline__ void vm_put_sums(float* row, const float (&acc)[8], int cg, long base, int N)
{
    const long col0 = base + cg * 8;
    if (col0 + 8 <= N || col0 >= N) {
        *reinterpret_cast<float4_t*>(row + cg * 8) = float4_t{acc[0], acc[1], acc[2], acc[3]};
        *reinterpret_cast<float4_t*>(row + cg * 8 + 4) = float4_t{acc[4], acc[5], acc[6], acc[7]};
    } else {
        const int first = (int)(N - 8 - base);  // where the loaded columns lie in the block (before its start if it has fewer than eight)
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (first + j >= cg * 8) row[first + j] = acc[j];
    }
}

// LPR: lanes per weight row.  KEEP: the weight is read with plain loads (load_weight).
template <int LPR, bool KEEP>
__global__ __launch_bounds__(kVmWaves * 64) void gemv_vm_f16_kernel(const half_t* __restrict__ x,
                                                                 const half_t* __restrict__ A,
                                                                 const half_t* __restrict__ bias, long lda, int K, int N,
                                                                 int k_per_slice, unsigned int flags, float* partial,
                                                                 unsigned int* status, unsigned int* poison,
                                                                 unsigned int spin_limit, int nslices, VmDests outs)
{
    const bool relu = flags & kVmRelu, by_xcd = flags & kVmByXcd;
    const int out_count = (int)(flags >> kVmOutsShift);
    constexpr int kVmCols = 8 * LPR;
    constexpr int GROUPS = kVmWaves * (64 / LPR);     // row groups per block = LDS rows of the reduction = rows between loads of a lane
    constexpr int PARTS = kVmWaves * 64 / kVmCols;    // threads per column when the slices' sums are collected
    __shared__ __align__(16) float red[GROUPS][kVmCols];
    __shared__ float parts[PARTS][kVmCols];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int cg = lane % LPR;             // which 8 columns of the block
    const int grp = tid / LPR;
    // (The launch's own size would come with 256 bytes of further arguments: it is counted here, the slices are an argument.)
    const int per_xcd = ((N + kVmCols - 1) / kVmCols + 7) >> 3;
    const int bx = by_xcd ? (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const long base = (long)bx * kVmCols;
    if (base >= N) return;  // (a grid that goes by XCD is rounded up to whole eights)
    const long col0 = base + cg * 8;
    const int k_begin = blockIdx.y * k_per_slice;
    const int k_end = min(K, k_begin + k_per_slice);

    // (asked for now by the blocks that will reduce, needed when they start to: it travels behind the block's own rows)
    unsigned int poisoned = 0u;
    if (nslices > 1 && (int)blockIdx.y == nslices - 1) poisoned = __hip_atomic_load(poison, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;

    if (col0 < N) vm_sum_rows<KEEP, GROUPS>(acc, A + (col0 + 8 <= N ? col0 : (long)N - 8), lda, x, k_begin + grp, k_end);
    vm_put_sums(red[grp], acc, cg, base, N);
    __syncthreads();

    // From here on a thread stands for one column.
    const int c = tid % kVmCols;
    const int part = tid / kVmCols;
    const long col = base + c;
    const bool mine = col < N;
    // Part p adds the groups p, p + PARTS, .. in that order, then the parts are added in order.
    {
        float v = red[part][c];
#pragma unroll
        for (int i = 1; i < GROUPS / PARTS; ++i) v += red[part + i * PARTS][c];
        parts[part][c] = v;
    }
    __syncthreads();
    auto total = [&]() {
        float v = parts[0][c];
#pragma unroll
        for (int q = 1; q < PARTS; ++q) v += parts[q][c];
        return v;
    };
    const float own = part == 0 ? total() : 0.0f;
    auto finish = [&](float r) {
        if (bias) r += (float)bias[col];
        if (relu) r = relu_f32(r);
        const half_t out = (half_t)r;
        for (int o = 0; o < out_count; ++o) outs.y[o][col] = out;
    };

    if (nslices == 1) {
        if (part == 0 && mine) finish(own);
        return;
    }
    const int last = nslices - 1;
    if ((int)blockIdx.y != last) {
        if (part == 0 && mine)
            __hip_atomic_store(reinterpret_cast<unsigned int*>(partial) + (long)blockIdx.y * N + col, __builtin_bit_cast(unsigned int, own),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // Part p adds the words of slices p, p + PARTS, ... < last in that order, kVmAhead of them asked for together.
    constexpr int kVmAhead = 4;
    float sum = 0.0f;
    if (mine) {
        unsigned int* words = reinterpret_cast<unsigned int*>(partial) + col;
        for (int s0 = part; s0 < last; s0 += kVmAhead * PARTS) {
            unsigned int w[kVmAhead];
#pragma unroll
            for (int q = 0; q < kVmAhead; ++q) {
                w[q] = kVmEmpty;
                const int sl = s0 + q * PARTS;
                if (sl < last && poisoned == 0u && spin_limit > 0u)
                    w[q] = __hip_atomic_load(words + (long)sl * N, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (int q = 0; q < kVmAhead; ++q) {
                const int sl = s0 + q * PARTS;
                if (sl >= last) break;
                unsigned int spins = 0;
                unsigned long long t_first = 0ull;
                while (w[q] == kVmEmpty && poisoned == 0u) {
                    if (spins > 0u && (spins & 255u) == 0u && wait_clock_expired(spins, t_first)) spins = 0xffffffffu;  // gives up below
                    if (spins++ >= spin_limit) {
                        __hip_atomic_store(poison, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        break;
                    }
                    w[q] = __hip_atomic_load(words + (long)sl * N, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                float v;
                if (w[q] != kVmEmpty) {
                    v = __builtin_bit_cast(float, w[q]);
                    __hip_atomic_store(words + (long)sl * N, kVmEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    // Slice sl's sum for this column, as its own block makes it: every row group's rows in ascending order, the
                    // groups of a part in order, then the parts.
                    const int ks_begin = sl * k_per_slice, ks_end = min(K, ks_begin + k_per_slice);
                    v = 0.0f;
#pragma unroll 1
                    for (int q2 = 0; q2 < PARTS; ++q2) {
                        float pv = 0.0f;
#pragma unroll 1
                        for (int g = q2; g < GROUPS; g += PARTS) {
                            float gv = 0.0f;
#pragma unroll 1
                            for (int k = ks_begin + g; k < ks_end; k += GROUPS) gv = fmaf((float)A[(long)k * lda + col], (float)x[k], gv);
                            pv = g == q2 ? gv : pv + gv;
                        }
                        v = q2 == 0 ? pv : v + pv;
                    }
                }
                sum += v;
            }
        }
    }
    __syncthreads();  // `parts` has been read above before it is written again
    parts[part][c] = sum;
    __syncthreads();
    if (part == 0 && mine) finish(total() + own);
}

// The product of gemv_vm_f16_kernel<LPR> in the same slices, with the same sums in the same order (the same bits), by blocks that
// exchange nothing: a block owns 8 LPR / NS columns and takes NS slices at a time, NS * GROUPS row groups of LPR / NS lanes.  For
// products that use no workspace where another caller could be using it too (vm_plan.h): recorded into a graph, through the
// static entry point, on a stream without a region.  What bounds it: a block reads a line of every row, however few of its
// columns it owns, and the lines of one CU do not come faster than one in 2 to 4 clocks.  MI355X, us, sliced / this one (and with
// the whole width in a block): VM_ALONE_FIGURES
template <int LPR, int NS>
__global__ __launch_bounds__(kVmWaves * 64) void gemv_vm_alone_f16_kernel(const half_t* __restrict__ x, const half_t* __restrict__ A,
                                                                       const half_t* __restrict__ bias, GemvOuts outs, int K, int N, long lda,
                                                                       int relu, int k_per_slice, int nslices, int by_xcd)
{
    constexpr int GROUPS = kVmWaves * (64 / LPR);
    constexpr int PARTS = kVmWaves * 8 / LPR;
    constexpr int LANES = LPR / NS;
    constexpr int COLS = 8 * LANES;
    static_assert(NS * PARTS * COLS == kVmWaves * 64, "one thread per slice, part and column");
    __shared__ __align__(16) float red[NS][GROUPS][COLS];
    __shared__ float parts[NS][PARTS][COLS];
    __shared__ float sums[PARTS][COLS];  // of the slices p, p + PARTS, ..: kept by the thread that finishes the column

    const int tid = threadIdx.x;
    const int cg = tid % LANES, worker = tid / LANES;
    const int bx = by_xcd ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
    const long base = (long)bx * COLS;
    if (base >= N) return;  // (whole blocks)
    const long col0 = base + cg * 8;
    const half_t* a = A + (col0 + 8 <= N ? col0 : (long)N - 8);
    const int c = tid % COLS, part = tid / COLS % PARTS, ps = tid / (COLS * PARTS);
    if (tid < COLS) {
#pragma unroll
        for (int p = 0; p < PARTS; ++p) sums[p][c] = 0.0f;
    }
    float own = 0.0f;  // the last slice's sum
    for (int s0 = 0; s0 < nslices; s0 += NS) {
        const int s = s0 + worker / GROUPS, grp = worker % GROUPS;
        float acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
        if (s < nslices && col0 < N) vm_sum_rows<true, GROUPS>(acc, a, lda, x, s * k_per_slice + grp, min(K, (s + 1) * k_per_slice));
        vm_put_sums(red[worker / GROUPS][grp], acc, cg, base, N);
        __syncthreads();
        float v = red[ps][part][c];
#pragma unroll
        for (int i = 1; i < GROUPS / PARTS; ++i) v += red[ps][part + i * PARTS][c];
        parts[ps][part][c] = v;
        __syncthreads();  // (`parts` is read below before the next trip's first barrier, and written again behind it)
        if (tid < COLS) {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                float t = parts[i][0][c];
#pragma unroll
                for (int q = 1; q < PARTS; ++q) t += parts[i][q][c];
                if (s0 + i == nslices - 1) own = t;
                else if (s0 + i < nslices) sums[(s0 + i) % PARTS][c] += t;
            }
        }
    }
    if (tid < COLS && base + c < N) {
        float r = sums[0][c];
#pragma unroll
        for (int q = 1; q < PARTS; ++q) r += sums[q][c];
        r += own;
        if (bias) r += (float)bias[base + c];
        if (relu) r = relu_f32(r);
        for (int o = 0; o < outs.count; ++o) outs.y[o][base + c] = (half_t)r;
    }
}

// VM order, fewer than eight columns, very few weights, or few rows of no whole pieces: 2-byte loads.  A block of 16 wavefronts owns 64 adjacent output
// columns (one per lane); wavefront g takes the rows g, g + 16, ... and the sixteen partial sums meet in LDS.
static constexpr int kVmGenericWaves = 16;
__global__ __launch_bounds__(64 * kVmGenericWaves) void gemv_vm_f16_generic_kernel(const half_t* __restrict__ x,
                                                                                   const half_t* __restrict__ A,
                                                                                   const half_t* __restrict__ bias,
                                                                                   GemvOuts outs, int K, int N, long lda,
                                                                                   int relu)
{
    __shared__ float red[kVmGenericWaves][64];
    const int lane = threadIdx.x & 63;
    const int g = threadIdx.x >> 6;
    const long col = (long)blockIdx.x * 64 + lane;
    float acc = 0.0f;
    if (col < N) {
        int k = g;
        for (; k + 3 * kVmGenericWaves < K; k += 4 * kVmGenericWaves) {
            half_t a[4], xv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a[u] = A[(long)(k + u * kVmGenericWaves) * lda + col];
                xv[u] = x[k + u * kVmGenericWaves];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = fmaf((float)a[u], (float)xv[u], acc);
        }
        for (; k < K; k += kVmGenericWaves) acc = fmaf((float)A[(long)k * lda + col], (float)x[k], acc);
    }
    red[g][lane] = acc;
    __syncthreads();
    if (g == 0 && col < N) {
        float v = red[0][lane];
#pragma unroll
        for (int w = 1; w < kVmGenericWaves; ++w) v += red[w][lane];
        if (bias) v += (float)bias[col];
        if (relu) v = relu_f32(v);
        for (int o = 0; o < outs.count; ++o) outs.y[o][col] = (half_t)v;
    }
}

// ---------------------------------------------------------------------------------------------
// C[m][n] = A[m][n] + B, B either [m][n] or one row [n] added to every row (the reference's custom_add,
// runtime/include/executor/op_executor/custom_ops.h:383-433).  The exact sum of two fp16 values rounded once to
// fp16, which is also what the reference's half2 addition yields.  C may alias A or B.  HBM-bound: 6 bytes per element.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void add_f16_vec_kernel(const half_t* A, const half_t* B, half_t* C, long total8,
                                                          long row8, int b_broadcast)
{
    // Units of 8 halves (16 bytes); row8 = n / 8.
    const long stride = (long)gridDim.x * 256;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total8; i += stride) {
        const half8_t a = reinterpret_cast<const half8_t*>(A)[i];
        const half8_t b = reinterpret_cast<const half8_t*>(B)[b_broadcast ? (i % row8) : i];
        half8_t c;
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = (half_t)((float)a[e] + (float)b[e]);
        reinterpret_cast<half8_t*>(C)[i] = c;
    }
}

__global__ __launch_bounds__(256) void add_f16_generic_kernel(const half_t* A, const half_t* B, half_t* C, long total,
                                                              long n, int b_broadcast)
{
    const long stride = (long)gridDim.x * 256;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += stride)
        C[i] = (half_t)((float)A[i] + (float)B[b_broadcast ? (i % n) : i]);
}

// ---------------------------------------------------------------------------------------------
// Measurement aid: reads n16 16-byte pieces with the same streaming loads the GEMV kernels use and keeps nothing
// (the sum only exists so that the loads are not removed; `sink` is written if it equals an impossible value).  What
// a launch of this kernel takes is the floor for any kernel that has to read the same bytes once.
// ---------------------------------------------------------------------------------------------
typedef float float4_probe_t __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void stream_read_probe_kernel(const float4_probe_t* __restrict__ data, long n16, float* sink)
{
    constexpr int U = 8;
    float s = 0.0f;
    const long stride = (long)gridDim.x * 256 * U;
    for (long base = (long)blockIdx.x * 256 * U + threadIdx.x; base < n16; base += stride) {
        float4_probe_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(data + min(base + (long)u * 256, n16 - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) s += v[u][0] + v[u][3];
    }
    if (s == 1234.5f && sink) sink[0] = s;
}

// ---------------------------------------------------------------------------------------------
// VV: y[0] = sum_k a[k] * b[k].  One block of 1024 lanes; any K and alignment.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void dot_f16_kernel(const half_t* __restrict__ a, const half_t* __restrict__ b,
                                                       half_t* __restrict__ y, long K)
{
    __shared__ float red[16];
    float acc = 0.0f;
    for (long k = threadIdx.x; k < K; k += 1024) acc = fmaf((float)a[k], (float)b[k], acc);
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 16; ++w) v += red[w];
        y[0] = (half_t)v;
    }
}

}  // namespace pimhip
