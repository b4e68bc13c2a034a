// One launch for a token's pass through a top-1 mixture-of-experts feed-forward block (gfx950, batch 1, fp16 storage,
// fp32 sums):
//
//     logits = W_r . x (+ b_r)          e = argmax(logits)          (the first maximum, on the logits rounded to fp16)
//     hidden = act(W1[e] . x + b1[e])                               (rounded to fp16, as the tensor between the two products is)
//     y      = W2[e] . hidden + b2[e]   (optionally times softmax(logits)[e])
//
// The reference runs this as separate operators (the router and the two products through customAtenAddmm / atenLinear,
// runtime/source/executor/op_executor/aten_ops.cpp:609-758 and :304-307) with the choice of the expert made on the host
// in between, which costs a stream synchronisation and a read-back per token.  Here the choice never leaves the GPU:
// every block computes the router's few rows itself, reads its rows of the chosen expert's first matrix, publishes its
// slice of `hidden` and, once it has everybody's, multiplies its rows of the second matrix, which are already in
// registers by then.
//
// Grid: `blocks` blocks of eight wavefronts, all resident at once.  `hidden` travels as 16-byte words of eight values;
// block b makes words [b * wpb, (b + 1) * wpb) (wpb = 1 or 2: at most 256 blocks make the at most 512 words), i.e.
// rows 8 * wpb * b .. of W1, wavefront w the rows w * wpb .. of those.  Of W2 block b owns rows [b * rpb2, (b + 1) * rpb2),
// rpb2 <= 8, one row per wavefront.
//
// What bounds the step is not bandwidth (9.4 MB) but a chain of dependent round trips: token and router rows, the expert's
// W1 rows, the all-to-all of `hidden`, the store of y.  So nothing else may stand in that chain: the launch count (which
// says which set of exchange slots this launch uses) is a device-scope load and is asked for behind the router's cached
// loads, not in front of them; the rows of W2 are asked for once the block's own word is stored, and the hidden values by wavefronts
// that hold no row of W2 as far as there are enough (a wavefront's loads return in order: a poll behind W2's rows waits for them, 0.7 us
// where another expert's were cached); what is not waited for, the caller's view of the choice, the slots of the next launch, goes
// out behind the word too, but not at the end: a launch lasts until its last store is acknowledged.
// Measured on MI355X (8 experts, 13 tokens in a row from a graph, us a step; in brackets with the rows of W2 right behind those of W1,
// where the word, which everybody waits for, queues behind up to 64 KB): 256 / 4096 4.57 (4.67), 768 / 1024 4.53 (4.95), 768 / 3072 5.23
// (5.37), 1024 / 4096 6.41 (6.91), 1792 / 2048 6.64 (7.15), 2048 / 4096 8.91 (9.73).  With every wavefront loading a row of W2, its own or
// one to drop, and polling behind it: 7.14, 5.38, 6.39, 7.97, 6.99, 9.46.
//
// Exchange: hx[2][blocks] entries of 64 bytes, a block's words in the first 16 * wpb bytes.  An empty 8-byte half is all
// ones, which no four fp16 values written here can be (a NaN is written as 0x7e00).  The two sets alternate by the launch
// count g (a device word read at the start): a launch uses set g & 1 and marks its own entry of the other set empty for the
// launch after it.  Where every block publishes a word, block 0 advances the count behind its wait for them: everybody
// has read the count by then.  A block that publishes nothing could start so late that it reads the count
// after block 0 has advanced it, and would look into the wrong set; grids with such blocks (d_model > d_ff / 2) keep one copy
// of the count per block, each in a line of its own, read and advanced by its block (0.3 us slower per step).
//
// A wait that gives up does not leave the result undefined.  Every wait is bounded (`spin_limit` polls, one second); a block
// in which a lane gave up computes every hidden value itself from W1[e] (no other block is needed for that: it is only
// slower, a few tens of microseconds) and goes on.  It raises the plan's abort word, which stays up: every later launch
// starts in that self-sufficient mode (the exchange slots may hold values of the launch that was cut short) until the
// host has refilled the slots and cleared the word.
#pragma once

#include "device_common.h"

namespace pimhip
{

constexpr int kMoeThreads = 512;
constexpr int kMoeWaves = kMoeThreads / 64;
constexpr int kMoeMaxBlocks = 256;
constexpr int kMoeMaxExperts = 64;
constexpr int kMoeMaxModel = 2048;                    // d_model: at most four 16-byte pieces of a row per lane
constexpr int kMoeMaxFf = 4096;                       // d_ff: at most 512 words of eight hidden values
constexpr int kMoeXC = kMoeMaxModel / 8 / 64;         // 16-byte pieces of a W1 row per lane
constexpr int kMoeFC = kMoeMaxFf / 8 / 64;            // 16-byte pieces of a W2 row per lane
constexpr int kMoeMaxWordsPerBlock = 2;               // wpb
constexpr int kMoeMaxRows2 = kMoeWaves;               // W2 rows per block: one per wavefront
constexpr int kMoeEntryWords = 8;                     // 8-byte words per entry (64 bytes); the first 2 * wpb carry values
constexpr unsigned long long kMoeEmpty = ~0ull;
constexpr int kMoeCounterStride = 16;                // 32-bit words between the blocks' copies of the launch count: a 64-byte line each
// Threads [moe_first_poller(rows, words), kMoeThreads) of a block poll up to two words each: the wavefronts without a row of W2, and as
// many more as two words to a thread need.
__host__ __device__ constexpr int moe_first_poller(int rows2, int words)
{
    const int needed = (words + 127) / 128, without_row = kMoeWaves - rows2;
    return 64 * (kMoeWaves - (without_row > needed ? without_row : needed));
}
static_assert(2 * (kMoeThreads - moe_first_poller(kMoeMaxRows2, kMoeMaxFf / 8)) >= kMoeMaxFf / 8, "every word is polled");
static_assert(kMoeMaxWordsPerBlock * kMoeMaxBlocks * 8 >= kMoeMaxFf, "every hidden value has a producer");
static_assert(2 * kMoeMaxWordsPerBlock <= kMoeEntryWords, "a block's words fit its entry");

struct MoeStepArgs {
    const half_t* x;                 // [d_model]
    const half_t* router_w;          // [E, d_model]
    const half_t* router_b;          // [E] or null
    const half_t* const* tables;     // device array [4][E]: W1[e] ([d_ff, d_model]), b1[e] or null, W2[e] ([d_model, d_ff]), b2[e] or null
    half_t* y;                       // [d_model]
    half_t* router_logits;           // [E] or null
    int* expert;                     // [1] or null
    unsigned long long* hx;          // [2][blocks][kMoeEntryWords]
    unsigned int* g_counter;         // [blocks][kMoeCounterStride]: every block's copy of the launch count in word 0 of its line
    unsigned int* abort_flag;        // device word: non-zero from the first wait that gave up until the host clears it
    unsigned int* abort_host;        // the same event for the host to see
    int d_model, d_ff, E, act, scale_by_prob;
    int wpb;                         // 16-byte words of hidden values per producing block
    int rpb2;                        // rows of W2 per block
    unsigned int spin_limit;
    int alone;                       // non-zero: every block computes all hidden values itself, nothing is exchanged
    int count_stride;                // 0: one launch count, advanced by block 0; kMoeCounterStride: one per block
};

// The barrier between the phases: this wavefront's LDS traffic done, then s_barrier.  __syncthreads() would also wait until the rows
// of W2 have arrived and the stores in front of them are acknowledged.
__device__ __forceinline__ void moe_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The maximum over the four rows of 16 lanes (wave_sum_rows' exchanges).
__device__ __forceinline__ float wave_max_rows(float v)
{
    {
        float a = v, b = v;
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
        v = fmaxf(a, b);
    }
    {
        float a = v, b = v;
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
        v = fmaxf(a, b);
    }
    return v;
}

// Two 16-byte device-scope loads in flight together (load16_device_scope).
__device__ __forceinline__ void load16_twice_device_scope(const void* p, const void* q, unsigned long long (&v)[4])
{
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    u32x4 a, b;
    asm volatile("global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b) : "v"(p), "v"(q) : "memory");
    v[0] = (unsigned long long)a[0] | ((unsigned long long)a[1] << 32);
    v[1] = (unsigned long long)a[2] | ((unsigned long long)a[3] << 32);
    v[2] = (unsigned long long)b[0] | ((unsigned long long)b[1] << 32);
    v[3] = (unsigned long long)b[2] | ((unsigned long long)b[3] << 32);
}

// What the kernel's first instructions need comes as plain arguments in front of the struct: those arrive in scalar
// registers with the wavefront (kernel-argument preload) instead of through a load at its start.
// XC, FC: 16-byte pieces of a W1 / W2 row per lane.
template <int XC, int FC>
__global__ __launch_bounds__(kMoeThreads) void moe_ffn_step_f16_kernel(const half_t* x_, const half_t* router_w_, const half_t* router_b_,
                                                                       const half_t* const* tables_, int d_model_, int d_ff_, int E_, int act_,
                                                                       MoeStepArgs p)
{
    p.x = x_;
    p.router_w = router_w_;
    p.router_b = router_b_;
    p.tables = tables_;
    p.d_model = d_model_;
    p.d_ff = d_ff_;
    p.E = E_;
    p.act = act_;
    __shared__ __align__(16) half_t hidden[kMoeMaxFf];
    __shared__ float logit_s[kMoeMaxExperts];
    __shared__ const half_t* table_s[4][kMoeMaxExperts];
    __shared__ __align__(16) unsigned short mine[8 * kMoeMaxWordsPerBlock];  // this block's hidden values (bits)
    __shared__ int someone_gave_up;
    __shared__ int block_poisoned;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b = blockIdx.x, nb = gridDim.x;
    const int nx = p.d_model >> 3, nf = p.d_ff >> 3;  // 16-byte pieces of a W1 / W2 row; nf is also the number of hidden words
    half8_t zero8;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero8[e] = (half_t)0.0f;

    if (tid == 0) {
        someone_gave_up = 0;
        block_poisoned = 0;
    }
    // the experts' pointers, while the router's rows travel
    for (int i = tid; i < 4 * p.E; i += kMoeThreads) table_s[i / p.E][i % p.E] = p.tables[i];

    // ---- the token, then the router: every block computes all E logits ----
    half8_t xr[XC];
    const half8_t* x8 = reinterpret_cast<const half8_t*>(p.x);
#pragma unroll
    for (int k = 0; k < XC; ++k) xr[k] = (lane + 64 * k < nx) ? x8[lane + 64 * k] : zero8;
    // (two experts per wavefront and pass: all their loads are in flight together, one round trip for E <= 16)
    for (int e0 = wave; e0 < p.E; e0 += 2 * kMoeWaves) {
        const int e1 = e0 + kMoeWaves;
        const half8_t* w8a = reinterpret_cast<const half8_t*>(p.router_w) + (long)e0 * nx;
        const half8_t* w8b = reinterpret_cast<const half8_t*>(p.router_w) + (long)(e1 < p.E ? e1 : e0) * nx;
        half8_t ra[XC], rb[XC];
#pragma unroll
        for (int k = 0; k < XC; ++k) {
            if (64 * k >= nx) break;  // (uniform) pieces past the row for every lane
            const int c = min(lane + 64 * k, nx - 1);
            ra[k] = w8a[c];
            rb[k] = w8b[c];
        }
        float sa = 0.0f, sb = 0.0f;
#pragma unroll
        for (int k = 0; k < XC; ++k) {
            if (lane + 64 * k < nx) {
                sa = dot8(ra[k], xr[k], sa);
                sb = dot8(rb[k], xr[k], sb);
            }
        }
        sa = wave_sum(sa);
        sb = wave_sum(sb);
        if (lane == 0) {
            if (p.router_b) sa += (float)p.router_b[e0];
            logit_s[e0] = (float)(half_t)sa;
            if (e1 < p.E) {
                if (p.router_b) sb += (float)p.router_b[e1];
                logit_s[e1] = (float)(half_t)sb;
            }
        }
    }
    moe_barrier();
    // argmax over the E <= 64 logits, one per lane: the first maximum; a NaN counts as the largest value, as in at::argmax
    const float mine_l = lane < p.E ? logit_s[lane] : -INFINITY;
    const bool is_nan = mine_l != mine_l;
    const unsigned long long nan_mask = __ballot(is_nan);
    float bv = is_nan ? -INFINITY : mine_l;
    bv = fmaxf(bv, dpp_f32<kDppQuadXor1>(bv));
    bv = fmaxf(bv, dpp_f32<kDppQuadXor2>(bv));
    bv = fmaxf(bv, dpp_f32<kDppRowHalfMirror>(bv));
    bv = fmaxf(bv, dpp_f32<kDppRowMirror>(bv));
    bv = wave_max_rows(bv);
    const unsigned long long max_mask = __ballot(lane < p.E && mine_l == bv);
    const int best = nan_mask ? __builtin_ctzll(nan_mask) : __builtin_ctzll(max_mask);
    float scale = 1.0f;
    if (p.scale_by_prob) {
        const float ex = lane < p.E ? __expf(mine_l - bv) : 0.0f;
        scale = 1.0f / wave_sum(ex);
    }
    const half8_t* w1 = reinterpret_cast<const half8_t*>(table_s[0][best]);
    const half_t* b1 = table_s[1][best];
    const half8_t* w2 = reinterpret_cast<const half8_t*>(table_s[2][best]);
    const half_t* b2 = table_s[3][best];

    // One row of W1[e] times the token, bias and activation, as the bits `hidden` holds; a NaN in its canonical form.
    auto hidden_bits = [&](float a, int r) {
        if (b1) a += (float)b1[r];
        if (p.act == 1) a = relu_f32(a);
        unsigned short bits = __builtin_bit_cast(unsigned short, (half_t)a);
        if (a != a) bits = 0x7e00u;
        return bits;
    };
    // This wavefront's row of W2[e]: asked for behind the block's word, consumed at the end.
    half8_t w2r[FC];
    const int r2 = b * p.rpb2 + wave;
    const bool has_row2 = wave < p.rpb2 && r2 < p.d_model;
    auto ask_for_w2 = [&]() {
        if (!has_row2) return;
#pragma unroll
        for (int k = 0; k < FC; ++k) w2r[k] = load_weight<true>(w2 + (long)r2 * nf + min(lane + 64 * k, nf - 1));
    };

    // The launch count (which set of slots this launch uses) and the abort word are device-scope loads, which take longer
    // than the cached ones above and would hold those up if they stood in front of them (a wavefront's loads return in
    // order).  Asked for here, they travel with the rows of W1 and are needed when the block publishes.
    const unsigned int g = __hip_atomic_load(p.g_counter + p.count_stride * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned int poisoned = __hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // ---- hidden = act(W1[e] . x + b1[e]): this block's words (asked for whether or not they will be published) ----
    const int row0 = 8 * p.wpb * b + wave * p.wpb;  // this wavefront's first row
    half8_t w1r[kMoeMaxWordsPerBlock][XC];
#pragma unroll
    for (int s = 0; s < kMoeMaxWordsPerBlock; ++s) {
        const int r = min(row0 + min(s, p.wpb - 1), p.d_ff - 1);
#pragma unroll
        for (int k = 0; k < XC; ++k) w1r[s][k] = load_weight<true>(w1 + (long)r * nx + min(lane + 64 * k, nx - 1));
    }
    if (poisoned != 0u) block_poisoned = 1;
#pragma unroll
    for (int s = 0; s < kMoeMaxWordsPerBlock; ++s) {
        const int r = row0 + s;
        float a = 0.0f;
#pragma unroll
        for (int k = 0; k < XC; ++k)
            if (lane + 64 * k < nx) a = dot8(w1r[s][k], xr[k], a);
        a = wave_sum(a);
        if (lane == 0 && s < p.wpb) mine[wave * p.wpb + s] = r < p.d_ff ? hidden_bits(a, r) : (unsigned short)0;
    }
    const unsigned int set = __builtin_amdgcn_readfirstlane(g) & 1u;
    // Whether the abort word is up is decided for the block as a whole, through LDS: wavefronts look at it at slightly
    // different times and can see different values when it is raised while the launch starts; they would then disagree
    // about the barriers that follow.  (The flags were set to 0 in front of the barrier behind the router.)
    moe_barrier();
    const bool alone = p.alone != 0 || block_poisoned != 0;
    // This block's entry of the other set is empty for the next launch (nobody reads that set during this one).  Stored here and
    // below by wavefronts that do not poll, not at the end: a launch lasts until its last store has been acknowledged, a
    // microsecond for a device-scope one.
    auto empty_other_set = [&]() {
        if (tid < 2 * kMoeMaxWordsPerBlock)
            __hip_atomic_store(p.hx + ((long)(set ^ 1u) * nb + b) * kMoeEntryWords + tid, kMoeEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // What the caller sees of the choice (behind the words the others wait for).
    auto report_choice = [&]() {
        if (b != 0) return;
        if (tid == 0 && p.expert) p.expert[0] = best;
        if (tid < p.E && p.router_logits) p.router_logits[tid] = (half_t)logit_s[tid];
    };
    if (!alone) {
        if (tid < p.wpb && b * p.wpb + tid < nf) {
            const unsigned long long* src = reinterpret_cast<const unsigned long long*>(&mine[8 * tid]);
            store16_device_scope(p.hx + ((long)set * nb + b) * kMoeEntryWords + 2 * tid, src[0], src[1]);
        }
        empty_other_set();
        report_choice();
        ask_for_w2();
        // ---- everybody's hidden values: word t and word t + n_poll by the threads behind the wavefronts that wait for a row of W2 ----
        const int poll0 = moe_first_poller(p.rpb2, nf);
        const int n_poll = kMoeThreads - poll0, t0 = tid - poll0;
        if (t0 >= 0 && t0 < nf) {
            const bool two = t0 + n_poll < nf;
            const int t1 = two ? t0 + n_poll : t0;
            const unsigned long long* slot0 = p.hx + ((long)set * nb + t0 / p.wpb) * kMoeEntryWords + 2 * (t0 % p.wpb);
            const unsigned long long* slot1 = p.hx + ((long)set * nb + t1 / p.wpb) * kMoeEntryWords + 2 * (t1 % p.wpb);
            unsigned long long v[4];
            unsigned int spins = 0;
            unsigned long long t_first = 0ull;
            bool gave_up = false;
            while (true) {
                load16_twice_device_scope(slot0, slot1, v);
                if (v[0] != kMoeEmpty && v[1] != kMoeEmpty && v[2] != kMoeEmpty && v[3] != kMoeEmpty) break;
                if (spins > 0u && (spins & 255u) == 0u) {
                    if (__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) gave_up = true;
                    if (wait_clock_expired(spins, t_first)) spins = 0xffffffffu;  // gives up below
                }
                if (spins >= p.spin_limit) {  // (with a limit of 0 a lane whose first look failed gives up without another)
                    __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    gave_up = true;
                }
                if (gave_up) break;
                if (spins != 0xffffffffu) ++spins;
            }
            if (gave_up) someone_gave_up = 1;
            typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<u64x2*>(&hidden[8 * t0]) = u64x2{v[0], v[1]};
            if (two) *reinterpret_cast<u64x2*>(&hidden[8 * t1]) = u64x2{v[2], v[3]};
        }
        moe_barrier();
    } else {
        empty_other_set();
        report_choice();
        ask_for_w2();
    }
    // (With one count for all: block 0 has seen everybody's word by now, or makes it late, when it has computed by itself.)
    auto advance_count = [&]() {
        if (tid == kMoeThreads - 1 && (b == 0 || p.count_stride != 0))  // (the last wavefront seldom has a row of W2 left to finish)
            __hip_atomic_store(p.g_counter + p.count_stride * b, g + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const bool by_itself = alone || someone_gave_up != 0;
    if (!by_itself) advance_count();
    if (by_itself) {
        // ---- self-sufficient: every hidden value from W1[e], by this block alone ----
        for (int r = wave; r < p.d_ff; r += kMoeWaves) {
            float a = 0.0f;
#pragma unroll
            for (int k = 0; k < XC; ++k)
                if (lane + 64 * k < nx) a = dot8(w1[(long)r * nx + lane + 64 * k], xr[k], a);
            a = wave_sum(a);
            if (lane == 0) hidden[r] = __builtin_bit_cast(half_t, hidden_bits(a, r));
        }
        __syncthreads();
        advance_count();
    }

    // ---- y = W2[e] . hidden + b2[e] ----
    if (has_row2) {
        float a = 0.0f;
#pragma unroll
        for (int k = 0; k < FC; ++k) {
            const int c = lane + 64 * k;
            if (c < nf) a = dot8(w2r[k], *reinterpret_cast<const half8_t*>(&hidden[c * 8]), a);
        }
        a = wave_sum(a);
        if (lane == 0) {
            if (b2) a += (float)b2[r2];
            p.y[r2] = (half_t)(a * scale);
        }
    }
}

}  // namespace pimhip
