// LSTM sequences with each recurrence confined to ONE XCD of the gfx950 part.
//
// lstm_seq_f16_kernel spreads a recurrence over every CU, so each step ends in an exchange of h between all eight
// XCDs, which has to go through the memory side (device scope): 1.4-1.8 us per step for 256 blocks, whatever the
// arithmetic.  The CUs of one XCD share an L2, and data that stays below it travels much faster: an all-to-all
// round among the 32 workgroups of one XCD takes 0.43 us when the polls are served by that L2 (measured; 0.85-1.5
// us with device-scope accesses between the same workgroups).  One XCD's registers hold one layer's W_hh
// (8.4 MB at H = 1024 against 16 MB of VGPRs), so here a recurrence is a GROUP of up to 32 workgroups on one XCD,
// 32 hidden units (one 64-byte entry) each, and different recurrences (the two directions of a layer; the layers of a
// stack, each fed by the one below through memory) run on different XCDs at the same time.
//
// Placement: the dispatcher deals the workgroups of a launch to the XCDs round-robin, workgroup b to XCD (b + o) % 8
// with a start o that belongs to the hardware queue and changes over a process's life (measured: 0 on a fresh queue, 6
// and 7 later).  So a workgroup asks the hardware where it is (XCC_ID): the group it joins is the one of that XCD, and
// its rank in the group is b / 8, which under any rotation gives every XCD ranks 0 .. grid / 8 - 1 exactly once.  A
// placement that is not a rotation leaves some rank of some group empty, and that group's first exchange times out
// (every wait is bounded); a rank that is taken twice is noticed at once through a claim word per (XCD, rank).
//
// Exchange inside a group: as in lstm_seq_f16_kernel every fp16 of an entry carries a flag in bit 14 (|h| <= 1 keeps
// it free) that tells the values of super-step g from those of g - 2 in the same slot, so every piece a reader gets
// validates itself.  That is what makes the cheap accesses safe: entries are written with plain stores (the per-CU
// cache is write-through, so they land in the XCD's L2) and read with non-temporal loads (a line read that way is
// dropped from the per-CU cache at once, so the next poll goes to the L2 again).  Nothing in the results depends on
// that cache behaviour: a stale piece fails its flag check and is polled again; only the time a poll takes does.
// Every wait is bounded (spin_limit polls, then the abort flag, as in lstm_seq_f16_kernel), and as there a workgroup one
// of whose waits gave up publishes nothing from then on and computes its units of the recurrence by itself at the end.
//
// A stack of unidirectional layers runs as a pipeline over the XCDs: layer k's recurrence (group R_k) on one XCD, and for
// k >= 1 a second group P_k on another XCD that holds W_ih of layer k and turns every h of layer k - 1 into layer k's
// input-projection row as soon as it exists.  R_{k-1} hands its h_t to P_k, and P_k its row to R_k, through buffers in
// memory with one slot per time step (device-scope stores and loads; a slot is written once per launch, so there is no
// flow control): the host fills them with all-ones bytes before the launch, a pattern that neither an fp16 h (a NaN is
// stored in its canonical form there) nor an fp32 sum can be, and a reader polls a slot until none of its elements is
// that pattern.  Those hand-overs cross XCDs and take about a microsecond, but they are not on the recurrences' critical
// path: P_k looks one step ahead while it multiplies, R_k starts a few steps late and from then on finds its rows
// waiting.  All groups then advance at the rate of one group, L layers in about the time of one.
//
// A workgroup has eight wavefronts; wavefront w owns hidden units 32 * rank + 4 * w .. + 3, whose 16 gate rows it keeps in 128
// registers per lane for the whole sequence.  Per step: the first wavefronts fetch the group's entries into LDS (16 bytes per lane),
// one barrier, the 16 rows' products with h, the gate arithmetic, and one 8-byte store of the wavefront's four new h values into the
// workgroup's entry.  What bounds a step: the store becoming visible in the L2 and the poll that finds it, 0.43 us at best
// for such a round, and a chain of dependent instructions between two rounds.  Everybody waits for the slowest wavefront's way from the
// barrier to its store, so nothing stands on it that can be done before or after: the reads behind the barrier are all issued at once from
// addresses made in front of it, the store's place and flag are known, y is packed and stored behind it, and no wait on it covers memory
// operations (two layers of 1024, 341 steps, MI355X: 432 us -> 338; two directions, 50 steps 75.6 -> 63.4; one layer of 256, 200 steps
// 173 -> 144).
// The products come in two kinds:
//   XcdSparse  16 fragments of 64 columns for v_smfmac_f32_16x16x64_f16: 0.21 us of matrix instructions at H = 1024 (4 up to 256
//              units); a step 0.93 us for a single layer, 0.95 in pipelines (v_dot2 1.3, 1.4)
//   XcdDot     v_dot2 and a transposing reduction over 16 lanes: nothing passes through LDS at the start of a launch, which short
//              sequences notice, and few units leave less of it idle (xcd_on_dot in lstm_plan.h has the lines and the figures)
// Against 64 bits the sums are equally far off (rms error over the sum of the products' magnitudes, 64 .. 1024 columns, MI355X): signs
// mixed 4.7e-9 .. 9.7e-9 on v_dot2 and 3.2e-9 .. 7.9e-9 sparse, all of one sign 3.4e-8 .. 5.2e-8 and 3.5e-8 .. 4.9e-8; an h made
// from the same previous h differs from its 64-bit value by 2.07e-4 relative with either, the rounding to fp16.
#pragma once

#include <type_traits>

#include "lstm_kernels.h"
#include "lstm_plan.h"
#include "lstm_solo.h"

namespace pimhip
{
static constexpr int kXcdCount = 8;                                   // XCDs of the part
static constexpr int kXcdMembers = 32;                                // workgroups of a group (CUs of an XCD)
static constexpr int kXcdWaves = 8;
static constexpr int kXcdThreads = 64 * kXcdWaves;
static constexpr int kXcdUnitsPerWave = 4;
static constexpr int kXcdUnitsPerBlock = kXcdWaves * kXcdUnitsPerWave;  // 32 units: one 64-byte entry
static constexpr int kXcdMaxH = 1024;                                 // 64 lanes x 16 columns = 32 members x 32 units
static constexpr int kXcdEntryWords = 16;                             // 32-bit words per entry
static constexpr int kXcdMaxChains = 4;
static constexpr int kXcdRegionWords = 2 * kXcdMembers * kXcdEntryWords;  // one chain's two slots

struct XcdChain {
    const half_t* w_hh;   // [4H, H]
    const float* xproj;   // [T, 4H] fp32 with biases: computed before the launch, or filled during it by the layer's P group
    const half_t* h0;     // [H]
    const half_t* c0;     // [H]
    half_t* y;            // row t at y + t * y_stride; null for an inner layer of a pipeline
    half_t* hn;           // [H]
    half_t* cn;           // [H]
    half_t* seq_out;      // [T][H], one slot per step, read by the P group of the layer above; null for the last layer
    int reverse;          // 1: t = T-1 .. 0
    int xproj_polled;     // 1: the rows of xproj are written during this launch (all-ones bytes = not yet)
    const half_t* res_in; // [T][H]: the layer's own input, added to its output (y and seq_out get h + in); null: no residual sum
    int res_polled;       // 1: res_in is the seq_out of the layer below, written during this launch (all-ones fp16 = not yet)
};

struct XcdProj {
    const half_t* w_ih;    // [4H, H] of the layer this group feeds
    const float* bsum;     // [4H] fp32 b_ih + b_hh
    const half_t* seq_in;  // [T][H]: the h of the layer below, slot t filled during this launch
    float* xp_out;         // [T][4H]: the xproj of the layer this group feeds
};

static constexpr int kXcdRoleProj = 9;  // role values: 0 none, 1 + k recurrence of chain k, kXcdRoleProj + j projection j
static constexpr unsigned long long kXcdWaitTicks = 100000000ull;  // one second of the 100 MHz clock
// The wavefront that makes the residual sums: one that does not poll and is, of the two on its SIMD, the first through its products
// (sums around the upper layers, by wavefront 4 / by this one: three layers of 1024, 50 steps 103 / 99 us, three of 512, 100 steps
// 148 / 135, two of 136, 100 steps 123 / 118).
static constexpr int kXcdSumWave = 2;
static_assert(kXcdSumWave >= 2 && kXcdSumWave < kXcdWaves, "wavefronts 0 and 1 poll for h");
static constexpr float kXcdLog2 = -1.4426950408889634f;  // exp(-v) = exp2(kXcdLog2 v)
static constexpr int kXcdLag = 2;       // steps a recurrence fed by a P group lets that group get ahead before it starts

struct LstmXcdArgs {
    XcdChain chain[kXcdMaxChains];
    XcdProj proj[kXcdMaxChains - 1];  // proj[j] feeds chain[j + 1]
    int role[kXcdCount];       // what the group on the XCD with this hardware index runs
    unsigned int* claims;      // [kXcdCount][kXcdMembers]: the launch (a counter value of the plan) that last took (XCD, rank)
    unsigned int* hx;          // [kXcdMaxChains] regions of kXcdRegionWords; zero when the chain's counter is 2
    unsigned int* g_counter;   // [kXcdMaxChains] device words: super-steps a chain's region has seen so far, plus 2
    unsigned int* abort_flag;
    unsigned int* abort_host;
    long y_stride;
    int H;
    int T;
    unsigned int spin_limit;
};

// The barrier of a step: LDS traffic of this wavefront done, then s_barrier.  __syncthreads() would also wait for every
// global store and load the wavefront has in flight (its release semantics cover global memory), and some of those cross
// to another XCD and back; nothing that passes between the wavefronts of a workgroup here goes through global memory.
__device__ __forceinline__ void lds_barrier() { lds_only_barrier(); }

typedef unsigned int xcd_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ xcd_u32x4 load16_nt(const void* p)
{
    xcd_u32x4 v;
    asm volatile("global_load_dwordx4 %0, %1, off nt\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(p) : "memory");
    return v;
}

__device__ __forceinline__ void store8_plain(void* p, unsigned long long v)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 w = {(unsigned int)v, (unsigned int)(v >> 32)};
    asm volatile("global_store_dwordx2 %0, %1, off" : : "v"(p), "v"(w) : "memory");
}

// ---- the step's matrix-vector product on v_dot2 ----
// Row l >> 4 of 16 lanes has the wavefront's unit l >> 4: its lanes keep, of the four gate rows, the 8-wide column pieces
// 16 c + (l & 15), c = 0 .. 7.  Four dot products of up to 64 columns per lane, then a transposing reduction over the 16 lanes.
struct XcdDot {
    half8_t w[4][8];

    static __device__ __forceinline__ int unit(int lane) { return lane >> 4; }
    static __device__ __forceinline__ int gate(int lane) { return (lane >> 2) & 3; }
    static __device__ __forceinline__ bool first_of_gate(int lane) { return (lane & 3) == 0; }
    static __device__ __forceinline__ bool first_of_unit(int lane) { return (lane & 15) == 0; }

    __device__ __forceinline__ void load(const half_t* src, int u0, int, int lane, int H, bool ok)
    {
        half8_t zero;
#pragma unroll
        for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int col = (16 * c + (lane & 15)) * 8;  // H % 8 == 0: a piece is entirely in or out of range
                w[g][c] = (ok && col < H) ? *reinterpret_cast<const half8_t*>(src + ((long)g * H + u0 + (lane >> 4)) * H + col) : zero;
            }
        }
    }

    struct Sums {
        __device__ __forceinline__ void clear() {}
    };

    // What is read of h as soon as it is there: nothing (pieces are read as they are used).
    struct Operands {
    };
    struct At {
    };
    static __device__ __forceinline__ At operands_at(const half_t*, int) { return {}; }
    static __device__ __forceinline__ void keep(At&) {}
    static __device__ __forceinline__ Operands operands(At) { return {}; }

    // In every lane: the dot product of its unit's gate row gate(lane) with hb[0 .. H).
    __device__ __forceinline__ float matvec(const half_t* hb, const Operands&, Sums&, int H, int lane) const
    {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c * 128 >= H) break;  // (uniform) column pieces 16 c .. 16 c + 15 lie past the hidden state
            const half8_t hv = *reinterpret_cast<const half8_t*>(hb + (16 * c + (lane & 15)) * 8);
#pragma unroll
            for (int g = 0; g < 4; ++g) acc[g] = dot8(w[g][c], hv, acc[g]);
        }
        // Each stage halves the number of values a lane holds and doubles the lanes they are summed over: mirrored lanes of
        // the row (l ^ 15), mirrored lanes of half a row (l ^ 7), the quad.
        const bool b3 = lane & 8, b2 = lane & 4;
        float v2[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) v2[r] = (b3 ? acc[2 + r] : acc[r]) + dpp_mov_f32<kDppRowMirror>(b3 ? acc[r] : acc[2 + r]);
        float v = (b2 ? v2[1] : v2[0]) + dpp_mov_f32<kDppRowHalfMirror>(b2 ? v2[0] : v2[1]);
        v += dpp_mov_f32<kDppQuadXor1>(v);
        v += dpp_mov_f32<kDppQuadXor2>(v);
        return v;
    }

    // The activated gates of a unit, right in the lanes of gate 0: f in the mirror within half the row (l ^ 7), o in the mirror
    // within the row (l ^ 15), g in the mirror of that one (l ^ 8).  (What the other lanes make of them is never used.)
    static __device__ __forceinline__ void share(float act, float& i, float& f, float& g, float& o)
    {
        i = act;
        f = dpp_mov_f32<kDppRowHalfMirror>(act);
        o = dpp_mov_f32<kDppRowMirror>(act);
        g = dpp_mov_f32<kDppRowMirror>(f);
    }

    // The four units' 16-bit values, which lanes 0, 16, 32 and 48 hold, as one word in lane 0 (other lanes: unspecified).
    // v_permlane16_swap with both operands alike leaves lane 16's value beside lane 0's and lane 48's beside lane 32's;
    // v_permlane32_swap then brings the upper pair down.  (v_readlane and scalar shifts: 1-5 % of a step more.)
    static __device__ __forceinline__ unsigned long long pack(unsigned int v16)
    {
        unsigned int a = v16, b = v16;
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
        const unsigned int x = a | (b << 16);
        unsigned int c = x, d = x;
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(c), "+v"(d));
        return (unsigned long long)c | ((unsigned long long)d << 32);
    }

    static __device__ __forceinline__ int place(int piece) { return piece; }  // where a 16-byte piece of h lies in LDS
};

// ---- the step's matrix-vector product on v_smfmac_f32_16x16x64_f16 ----
// D[16 x 16] += A[16 x 64, two of every four columns present] . B[64 x 16]: the weights are the dense operand, 64 columns of
// the wavefront's 16 gate rows per instruction, and h is the sparse one.  A row of A holds only half of the 64 columns, but
// which half is the row's own choice: even rows name columns 0, 1 of every four, odd rows columns 2, 3, so the two rows of a
// pair together multiply all 64 columns by h, and their two results add up to the dot product.  A matrix instruction thus
// takes 1024 weights in 16 cycles where v_dot2 takes 512 and a dense MFMA with h as one of its rows as many (batch 1).
// One register set of A (eight halves per lane) has eight row pairs and holds 512 values of h; instruction m of the eight
// that use it reads the weights of pair m's 64 columns, and of its result only rows 2m, 2m + 1 mean anything: eight
// accumulators, of which each row of 16 lanes keeps the two row pairs it holds.  No sum across the 16 lanes is left to do
// (column n of D is lane n & 15), and a wavefront reads h from LDS once, 2 KB instead of 8.
typedef _Float16 half16_t __attribute__((ext_vector_type(16)));
static constexpr int kXcdFrags = kXcdMaxH / 64;  // 64-column weight fragments of a wavefront's 16 gate rows

// The lanes of the operands (checked on the hardware): lane l of A holds, of row l & 15, the eight present columns among columns
// 16 (l >> 4) .. + 15; lane l of B holds, of column l & 15, rows 8 (l >> 4) .. + 7 and 32 + 8 (l >> 4) .. + 7.  Which columns of
// the weight matrix the 64 are is free as long as both operands agree.  A lane of B takes two whole 16-byte pieces of its gate
// row, 8 m + (l >> 4) and four pieces further; halves 0..3 of a piece then meet the even row of A, halves 4..7 the odd one.

// Lane l's eight values of h in a register set of A: two 8-byte halves of neighbouring pieces, at these two LDS addresses for the first set
// and 1 KB further for the second.  Addresses, because a lane has them ready in front of the barrier that it reads behind.
struct XcdOperandAt {
    unsigned int lo, hi;
};
typedef __attribute__((address_space(3))) const half4_t* xcd_lds_half4;
__device__ __forceinline__ unsigned int xcd_lds_address(const void* p)
{
    return (unsigned int)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
__device__ __forceinline__ XcdOperandAt xcd_h_operand_at(const half_t* hb, int lane)
{
    const int lo = xcd_h_place(xcd_h_operand_piece(0, lane));
    return {xcd_lds_address(hb + lo * 8 + 4 * (lane & 1)), xcd_lds_address(hb + (lo ^ 1) * 8 + 4 * (lane & 1))};
}
static constexpr unsigned int kXcdSecondOperand = 64 * 16;   // bytes
__device__ __forceinline__ half8_t xcd_h_operand(XcdOperandAt at)
{
    return __builtin_shufflevector(*(xcd_lds_half4)(uintptr_t)at.lo, *(xcd_lds_half4)(uintptr_t)at.hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// FRAGS: four (up to 256 units) or sixteen of them.  Four have a kernel of their own: half the sums and no second operand, and with both in one
// kernel the accumulators were copied on a step's path.
static constexpr int kXcdFewUnits = 256;
template <int FRAGS>
struct XcdSparse {
    static_assert(FRAGS == kXcdFewUnits / 64 || FRAGS == kXcdFrags, "up to 256 units, or any number");
    static constexpr bool kFew = FRAGS < kXcdFrags;
    half16_t w[FRAGS];

    // Lane l holds gate l & 3 of unit (l >> 2) & 3, in all four rows of 16 lanes.
    static __device__ __forceinline__ int unit(int lane) { return (lane >> 2) & 3; }
    static __device__ __forceinline__ int gate(int lane) { return lane & 3; }
    static __device__ __forceinline__ bool first_of_gate(int lane) { return lane < 16; }
    static __device__ __forceinline__ bool first_of_unit(int lane) { return lane < 16 && (lane & 3) == 0; }

    // A wavefront's fragments.  16 lanes on 16 rows, 64 bytes of each, is what a fragment would ask of memory: 3 us per launch slower
    // than whole 256-byte pieces of rows.  So all loads are issued that way (instruction 4 i + j: rows 4 j .. + 3, columns 128 i .. + 127)
    // and each 16 rows x 128 columns then change lanes through 4 KB of LDS of the wavefront's own, 16-byte piece p of row r in place
    // p ^ r.  Row n: gate n & 3 of unit u0 + (n >> 2).
    __device__ __forceinline__ void load(const half_t* src, int u0, int wave, int lane, int H, bool ok)
    {
        __shared__ __align__(16) half_t staged[kXcdWaves][16 * 128];
        half_t* stage = staged[wave];
        half8_t zero;
#pragma unroll
        for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
        half8_t raw[FRAGS / 2][4];
#pragma unroll
        for (int i = 0; i < FRAGS / 2; ++i) {
            if (128 * i >= H) break;  // (uniform)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = 4 * j + (lane >> 4), col = 128 * i + 8 * (lane & 15);  // H % 8 == 0: a piece is entirely in or out of range
                raw[i][j] = (ok && col < H) ? *reinterpret_cast<const half8_t*>(src + ((long)(n & 3) * H + u0 + (n >> 2)) * H + col) : zero;
            }
        }
        const int n = lane & 15, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < FRAGS / 2; ++i) {
            if (128 * i >= H) {  // (uniform) nothing but zeros: 64 KB per CU and i that need not pass through LDS
#pragma unroll
                for (int m = 0; m < 2; ++m) w[2 * i + m] = __builtin_shufflevector(zero, zero, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
                continue;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 4 * j + (lane >> 4);
                *reinterpret_cast<half8_t*>(stage + r * 128 + ((lane & 15) ^ r) * 8) = raw[i][j];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (one wavefront's LDS accesses stay in order; this keeps the compiler's too)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const half8_t lo = *reinterpret_cast<const half8_t*>(stage + n * 128 + ((8 * m + g) ^ n) * 8);
                const half8_t hi = *reinterpret_cast<const half8_t*>(stage + n * 128 + ((8 * m + 4 + g) ^ n) * 8);
                w[2 * i + m] = __builtin_shufflevector(lo, hi, 0, 1, 4, 5, 2, 3, 6, 7, 8, 9, 12, 13, 10, 11, 14, 15);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    }

    // The accumulators of a step, cleared where the wavefront has nothing else to do (in front of its wait for h).
    struct Sums {
        float4_t d[kFew ? 4 : 8];
        __device__ __forceinline__ void clear()
        {
#pragma unroll
            for (int j = 0; j < (kFew ? 4 : 8); ++j) {
                d[j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                asm volatile("" : "+v"(d[j]));
            }
        }
    };

    // Both register sets of h, asked for together right behind the step's barrier (past the hidden state hb holds zeros).  Asked for
    // behind the first set's instructions, the second came 100 cycles after the last of them.
    struct Operands {
        half8_t h0, h1;
    };
    struct At {
        XcdOperandAt h0, h1;
    };
    static __device__ __forceinline__ At operands_at(const half_t* hb, int lane)
    {
        const XcdOperandAt h0 = xcd_h_operand_at(hb, lane);
        return {h0, {h0.lo + kXcdSecondOperand, h0.hi + kXcdSecondOperand}};
    }
    // (all four addresses: with an offset for the second set the reads become two of 16 bytes, whose halves then have to change places)
    static __device__ __forceinline__ void keep(At& at)
    {
        asm volatile("" : "+v"(at.h0.lo), "+v"(at.h0.hi));
        if constexpr (!kFew) asm volatile("" : "+v"(at.h1.lo), "+v"(at.h1.hi));
    }
    static __device__ __forceinline__ Operands operands(At at)
    {
        Operands o;
        o.h0 = xcd_h_operand(at.h0);
        o.h1 = kFew ? o.h0 : xcd_h_operand(at.h1);
        return o;
    }

    // In every lane l: the dot product of gate row l & 15 of the wavefront with hb[0 .. H).
    __device__ __forceinline__ float matvec(const half_t*, const Operands& h, Sums& acc, int H, int lane) const
    {
        const int index = (lane & 1) ? 0xeeeeeeee : 0x44444444;  // columns 2, 3 / 0, 1 of every four
        if constexpr (kFew) {
#pragma unroll
            for (int m = 0; m < 4; ++m) acc.d[m] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(h.h0, w[m], acc.d[m], index, 0, 0);
            const float f0 = (acc.d[0][0] + acc.d[0][1]) + (acc.d[1][2] + acc.d[1][3]);
            const float f1 = (acc.d[2][0] + acc.d[2][1]) + (acc.d[3][2] + acc.d[3][3]);
            return wave_sum_rows((lane & 32) ? 0.0f : (lane & 16) ? f1 : f0);
        } else {
#pragma unroll
        for (int m = 0; m < FRAGS; ++m) {
            if (m >= 8 && (m & 3) == 0 && m * 64 >= H) break;  // (uniform) whole fragments past the hidden state are zeros
            acc.d[m & 7] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(m < 8 ? h.h0 : h.h1, w[m], acc.d[m & 7], index, 0, 0);
            if (m == 7) asm volatile("" : : "v"(h.h1));  // (read for it behind the barrier, not behind the next line's branch)
        }
        // Row r of D lies in register r & 3 of lanes 16 (r >> 2) .. + 15: row group q keeps pairs 2 q (registers 0, 1) and 2 q + 1.
        float f[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) f[q] = (acc.d[2 * q][0] + acc.d[2 * q][1]) + (acc.d[2 * q + 1][2] + acc.d[2 * q + 1][3]);
        const float lo = (lane & 16) ? f[1] : f[0], hi = (lane & 16) ? f[3] : f[2];
        return wave_sum_rows((lane & 32) ? hi : lo);
        }
    }

    // The activated gates of a unit: the quad's four lanes share them.
    static __device__ __forceinline__ void share(float act, float& i, float& f, float& g, float& o)
    {
        i = dpp_mov_f32<0x00>(act);  // quad_perm broadcasts of lanes 0, 1, 2, 3 of the quad
        f = dpp_mov_f32<0x55>(act);
        g = dpp_mov_f32<0xAA>(act);
        o = dpp_mov_f32<0xFF>(act);
    }

    // The four units' 16-bit values, one per quad of a row of 16 lanes, as one word in lane 0 of the row: quad 1 is quad 0's mirror
    // within half the row, quads 2 and 3 lie half a row further.
    static __device__ __forceinline__ unsigned long long pack(unsigned int v16)
    {
        const unsigned int lo = v16 | (dpp_u32<kDppRowHalfMirror>(v16) << 16);
        return (unsigned long long)lo | ((unsigned long long)dpp_u32<kDppRowRor8>(lo) << 32);
    }

    static __device__ __forceinline__ int place(int piece) { return xcd_h_place(piece); }
};

// PIPE = false: groups that neither feed nor are fed across XCDs (a single layer, the two directions of one); everything
// that concerns P groups and the hand-overs is compiled out, which is worth 10 % of a step.
// RES = true: layers with a residual sum (out_t = h_t + in_t).  The sum is made where h leaves the workgroup: the wavefront
// that hands the previous step's 32 h values to the layer above adds the layer's own input of that step, which it asked
// for a step earlier, and stores y from there too (one step late; hn stays h).  Compiled in only for stacks that have such
// layers.
template <bool PIPE, bool RES, class Product>
__device__ __forceinline__ void lstm_xcd_body(const LstmXcdArgs& p)
{
    __shared__ __align__(16) half_t hbuf[2][kXcdMaxH];  // h of the previous step, double buffered by step parity
    __shared__ __align__(16) float xring[kXcdWaves][32][4][4];  // per wavefront: [step & 31][gate][unit] projection terms
    __shared__ __align__(16) unsigned long long hout[2][kXcdWaves];  // the workgroup's 32 new h values, for the layer above
    __shared__ unsigned short in_ring[2][kXcdUnitsPerBlock];        // RES: the layer's own input of the last two steps, for the sums
    // Raised by a wavefront one of whose waits gave up, always in front of a step's barrier, and read by all right behind
    // it: the workgroup then leaves the loop of steps together, publishes nothing more and computes its units by itself.
    __shared__ int block_gave_up;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (in a scalar register: what goes by it is a branch, not a mask)
    const int xcd = (int)hw_xcc_id();  // the XCD this workgroup runs on
    const int rank = blockIdx.x >> 3;
    if (xcd >= kXcdCount) {
        // An id outside 0..7: not the part this kernel is laid out for (the host checks the placement of a probe launch
        // before it chooses this kernel).  Reported like a rank taken twice; every other workgroup's waits are bounded.
        if (tid == 0) {
            __hip_atomic_store(p.abort_host + 1, (unsigned int)blockIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(p.abort_host + 2, (unsigned int)xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(p.abort_host, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        return;
    }
    const int role = p.role[xcd];
    const int H = p.H;
    const int T = p.T;
    const int members = (H + kXcdUnitsPerBlock - 1) / kXcdUnitsPerBlock;
    if (role == 0 || rank >= members) return;  // whole workgroups, before any barrier
    const bool is_proj = PIPE && role >= kXcdRoleProj;
    const int k = is_proj ? role - kXcdRoleProj + 1 : role - 1;  // the chain this group runs or feeds
    const XcdChain& ch = p.chain[k];
    const XcdProj& pj = p.proj[is_proj ? k - 1 : 0];

    bool gave_up = false;
    const unsigned int g_base = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(p.g_counter + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    // A wait of an earlier launch gave up and the host has not re-initialised the exchange since: nothing is exchanged in
    // this launch, every workgroup of a recurrence computes its units by itself.
    const bool poisoned = __builtin_amdgcn_readfirstlane(__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u;
    if (tid == 0) block_gave_up = poisoned ? 1 : 0;
    unsigned int* region = p.hx + (long)k * kXcdRegionWords;
    // This launch's mark on (XCD, rank): the counter value is new in every launch of the plan.  Found already there, two
    // workgroups of this launch share the rank, so another rank of the group is empty: not a rotation.
    unsigned int claimed_before = 0u;
    if (tid == 0)
        claimed_before = __hip_atomic_exchange(p.claims + xcd * kXcdMembers + rank, g_base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // ---- weights into registers
    const int u0 = rank * kXcdUnitsPerBlock + wave * kXcdUnitsPerWave;
    const bool units_ok = u0 < H;  // H % 8 == 0: the four units of a wavefront are all inside or all outside
    const int unit = Product::unit(lane);  // of the wavefront's four
    const int my_unit = u0 + unit;
    const int my_gate = Product::gate(lane);  // (LibTorch order i, f, g, o)
    Product weights;
    weights.load(is_proj ? pj.w_ih : ch.w_hh, u0, wave, lane, H, units_ok);
    {
        half8_t zero;
#pragma unroll
        for (int e = 0; e < 8; ++e) zero[e] = (half_t)0.0f;
        for (int i = tid; i < 2 * kXcdMaxH / 8; i += kXcdThreads) reinterpret_cast<half8_t*>(&hbuf[0][0])[i] = zero;
    }
    if (tid == 0 && claimed_before == g_base) {
        __hip_atomic_store(p.abort_host + 1, (unsigned int)blockIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(p.abort_host + 2, (unsigned int)xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p.abort_host, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();

    const int uc = units_ok ? my_unit : H - 1;
    // All lanes of the first two wavefronts fetch one piece of an h vector each: 8 fp16 = columns 8 q .. 8 q + 7.  Spread over eight
    // wavefronts of 16 lanes a step of 1024 units took 1.42 us, over four of 32 1.32, over two 1.31.  (The wavefronts that talk
    // to other XCDs, 4 .. 7 and the one that makes the residual sums, never poll for h: a wavefront's loads come back in order.)
    // Whole wavefronts poll: a lane past the hidden state looks at the last piece beside the others and keeps nothing.
    const bool polls = wave < 2 && wave * 64 * 8 < H;
    const bool in_range = (wave * 64 + lane) * 8 < H;
    const int piece = min(wave * 64 + lane, H / 8 - 1);

    // One bounded wait of the wavefront's active lanes: `again` loads and tests, a lane each; gives up like every wait of this kernel,
    // after spin_limit polls, and also after kXcdWaitTicks of the constant 100 MHz clock, however long a poll takes in the
    // environment the kernel finds itself in (a wait that succeeds does so within microseconds).  The lanes leave together: with lanes
    // that leave by themselves the way out of the loop was ten instructions of mask arithmetic, on every step's path.
    auto bounded_wait = [&](bool& gave_up_here, auto again) __attribute__((always_inline)) {
        unsigned int spins = 0;
        unsigned long long t_first = 0ull;
        while (true) {
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!again()) == 0ull, 1)) return;
            if (gave_up_here) return;
            ++spins;
            if ((spins & 255u) == 0u) {
                if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u) gave_up_here = true;
                const unsigned long long now = __builtin_amdgcn_s_memrealtime();
                if (spins == 256u) t_first = now;
                else if (now - t_first > kXcdWaitTicks) spins = 0xffffffffu;  // gives up below
            }
            if (spins >= p.spin_limit) {
                __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                gave_up_here = true;
            }
        }
    };
    // true if none of the four fp16 of the word is the all-ones pattern
    auto filled16 = [](unsigned long long v) {
        const unsigned long long x = ~v;  // an all-ones fp16 becomes zero
        return ((x & 0xffffull) != 0ull) && ((x & 0xffff0000ull) != 0ull) && ((x & 0xffff00000000ull) != 0ull) && ((x >> 48) != 0ull);
    };

    if (is_proj) {
        // ================= P group: xproj rows of layer k from the h of layer k - 1, step by step =================
        if (poisoned) return;  // (the recurrence it feeds makes its own rows then)
        const float bias = pj.bsum[(long)my_gate * H + uc];
        float* dst = pj.xp_out + (long)my_gate * H + uc;
        unsigned long long lo = 0ull, hi = 0ull;  // this lane's piece of the step ahead
        if (polls) {
            lo = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(pj.seq_in + piece * 8), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            hi = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(pj.seq_in + piece * 8) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int t = 0; t < T; ++t) {
            half_t* hb = hbuf[t & 1];
            typename Product::At operands_at = Product::operands_at(hb, lane);
            Product::keep(operands_at);
            typename Product::Sums acc;
            acc.clear();
            if (polls) {
                const unsigned long long* src = reinterpret_cast<const unsigned long long*>(pj.seq_in + (long)t * H + piece * 8);
                if (__builtin_amdgcn_ballot_w64(!(filled16(lo) && filled16(hi))) != 0ull) {
                    bounded_wait(gave_up, [&]() {
                        load16_device_scope(src, lo, hi);
                        return filled16(lo) && filled16(hi);
                    });
                }
                typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
                const u64x2 both = {lo, hi};
                if (in_range) *reinterpret_cast<half8_t*>(hb + Product::place(piece) * 8) = __builtin_bit_cast(half8_t, both);
            }
            if (gave_up) block_gave_up = 1;
            lds_barrier();
            const int dead = __builtin_amdgcn_readfirstlane(block_gave_up);  // (asked for with the reads of h, looked at where the row would leave)
            if (polls && t + 1 < T) {
                // the step ahead, in flight while this one is multiplied (tested at the top of the next iteration)
                const unsigned long long* nxt = reinterpret_cast<const unsigned long long*>(pj.seq_in + (long)(t + 1) * H + piece * 8);
                lo = __hip_atomic_load(nxt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                hi = __hip_atomic_load(nxt + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            const float v = weights.matvec(hb, Product::operands(operands_at), acc, H, lane) + bias;
            if (dead) return;  // rows made from a stale h must not reach the recurrence: it will make its own
            if (units_ok && Product::first_of_gate(lane))
                __hip_atomic_store(reinterpret_cast<unsigned int*>(dst + (long)t * 4 * H), __builtin_bit_cast(unsigned int, v), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }

    // ================= R group: the recurrence of chain k =================
    // Compiled once per combination of "its projection rows arrive during the launch" and "its h goes to a layer above":
    // a step is sensitive to every instruction on its path, and the plain combination should not carry the others'.
    auto recurrence = [&](auto polled_c, auto feeds_c, auto res_c) __attribute__((always_inline)) {
    constexpr bool polled = decltype(polled_c)::value;
    constexpr bool feeds = decltype(feeds_c)::value;
    constexpr bool res = decltype(res_c)::value;
    constexpr bool emits = feeds || res;  // the workgroup's h values leave through hout, one step late
    // Without a residual sum: lanes 0..3 of wavefront 4 hand step se's 32 h values to the layer above, 16 bytes each.
    auto emit = [&](int se) __attribute__((always_inline)) {
        const unsigned long long* src = &hout[se & 1][2 * lane];
        store16_device_scope(ch.seq_out + (long)se * H + rank * kXcdUnitsPerBlock + lane * 8, src[0], src[1]);
    };
    // With one: lanes 0..31 of the wavefront that makes the sums, one value each: a handful of instructions per step (eight values in each of
    // four lanes took 0.1 us per step more).
    const int eu = rank * kXcdUnitsPerBlock + (lane & 31);  // the unit an emitting lane handles
    const bool sums = res && wave == kXcdSumWave && lane < 32 && eu < H;
    // The input of step s is asked for right after that step's barrier, together with the projection rows two steps ahead
    // (it exists: the projection row made from it is in use), parked in LDS at the top of step s + 1 and added after
    // that step's barrier.  Parking it waits for the load, so what matters is that the load leaves early in the step: issued
    // behind the sum of the step before, it cost 0.23 us per step.
    unsigned short in_ahead = 0xffffu;
    bool sum_gave_up = false;  // (a lane's: not every lane makes sums)
    auto emit_sum = [&](int se) __attribute__((always_inline)) {
        unsigned short in_bits = in_ring[se & 1][lane & 31];
        if (ch.res_polled && in_bits == 0xffffu) {
            const unsigned short* rin = reinterpret_cast<const unsigned short*>(ch.res_in) + (long)se * H + eu;
            bounded_wait(sum_gave_up, [&]() {
                in_bits = __hip_atomic_load(rin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return in_bits != 0xffffu;
            });
        }
        const unsigned short hbits = reinterpret_cast<const unsigned short*>(&hout[se & 1][0])[lane & 31];
        const float v = (float)__builtin_bit_cast(half_t, hbits) + (float)__builtin_bit_cast(half_t, in_bits);
        const unsigned short ob = (v == v) ? __builtin_bit_cast(unsigned short, (half_t)v) : (unsigned short)0x7e00u;
        if (ch.y) reinterpret_cast<unsigned short*>(ch.y)[(long)se * p.y_stride + eu] = ob;
        if (feeds)
            __hip_atomic_store(reinterpret_cast<unsigned short*>(ch.seq_out) + (long)se * H + eu, ob, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    float c_reg = (float)ch.c0[uc];
    const bool rev = ch.reverse != 0;

    // The input-projection term does not depend on h and must stay off the step's critical path: a wavefront's loads
    // return in order, so a poll issued behind a load that misses the L2 would wait for it.  Each wavefront keeps the
    // terms of its 16 rows for up to 32 steps in LDS.  Rows that exist before the launch are fetched 16 steps at a time,
    // ONE 16-byte load per lane every 16 steps (lane l: gate l & 3 of the wavefront's four units, adjacent in a row of
    // xproj, for step offset l >> 2).  Rows that a P group writes during the launch are fetched one element per lane two
    // steps ahead, right after the step's barrier so that the load travels while the step is computed, and tested when
    // they are used; the wavefronts that poll for h leave that to wavefronts 4..7, which fetch the elements of wavefront
    // w - 4 beside their own (a poll would have to wait for such a load to come back from the other XCD first).
    const int u0c = units_ok ? u0 : H - 4;
    auto fetch_xp = [&](int s0) {
        const int sx = min(s0 + (lane >> 2), T - 1);
        const int t = rev ? (T - 1 - sx) : sx;
        return *reinterpret_cast<const float4_t*>(ch.xproj + (long)t * 4 * H + (long)(lane & 3) * H + u0c);
    };
    auto deposit_xp = [&](int half, const float4_t v) {
        *reinterpret_cast<float4_t*>(&xring[wave][half * 16 + (lane >> 2)][lane & 3][0]) = v;
    };
    const unsigned int* xp_mine = reinterpret_cast<const unsigned int*>(ch.xproj + (long)my_gate * H + uc);  // + t * 4H
    const bool fetcher = wave >= 4;
    const unsigned int* xp_other =
        reinterpret_cast<const unsigned int*>(ch.xproj + (long)my_gate * H + min(max(u0 - 16, 0) + unit, H - 1));  // wavefront w - 4's
    auto xp_bits_at = [&](int t) { return __hip_atomic_load(xp_mine + (long)t * 4 * H, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto wait_xp = [&](int t, unsigned int bits = 0xffffffffu) {
        bounded_wait(gave_up, [&]() {
            if (bits == 0xffffffffu) bits = xp_bits_at(t);
            return bits != 0xffffffffu;
        });
        return bits;
    };
    float4_t xp_next = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    unsigned int xp_ahead = 0xffffffffu, xp_ahead_other = 0xffffffffu;  // polled rows: the elements of step s + 2, loaded during step s
    if (!polled) {
        deposit_xp(0, fetch_xp(0));
        deposit_xp(1, fetch_xp(16));
    } else {
        // Let the P group get kXcdLag steps ahead, then take the first two rows.
        (void)wait_xp(min(kXcdLag, T - 1));
        reinterpret_cast<unsigned int&>(xring[wave][0][my_gate][unit]) = wait_xp(0);
        reinterpret_cast<unsigned int&>(xring[wave][1][my_gate][unit]) = wait_xp(min(1, T - 1));
    }

    // Where this wavefront publishes its four values, alternating by the count; what stands between a step's gates and that store is
    // waited for by the whole group, so nothing of it is computed there.
    unsigned char* publish_at = reinterpret_cast<unsigned char*>(region + ((long)(g_base & 1u) * kXcdMembers + rank) * kXcdEntryWords) + wave * 8;
    long publish_step = (g_base & 1u) ? -(long)sizeof(unsigned int) * kXcdMembers * kXcdEntryWords : (long)sizeof(unsigned int) * kXcdMembers * kXcdEntryWords;
    unsigned int published32 = units_ok ? 0xffffffffu : 0u;
    asm volatile("" : "+v"(published32));
    const unsigned long long published = ((unsigned long long)published32 << 32) | published32;
    const bool publishes = lane == 0;
    const bool stores_y = lane == 0 && !res && units_ok && ch.y != nullptr;
    unsigned char* y_at = reinterpret_cast<unsigned char*>(ch.y + (rev ? (long)(T - 1) * p.y_stride : 0l) + u0);
    const long y_step = (long)sizeof(half_t) * (rev ? -p.y_stride : p.y_stride);
    const float gate_scale = my_gate == 2 ? 2.0f * kXcdLog2 : kXcdLog2, gate_mul = my_gate == 2 ? 2.0f : 1.0f, gate_add = my_gate == 2 ? -1.0f : 0.0f;

    for (int s = 0; s < T; ++s) {
        half_t* hb = hbuf[s & 1];
        typename Product::At operands_at = Product::operands_at(hb, lane);
        unsigned int xp_at = xcd_lds_address(&xring[wave][s & 31][my_gate][unit]);
        Product::keep(operands_at);
        asm volatile("" : "+v"(xp_at));  // (made here, not behind the barrier)
        typename Product::Sums acc;
        acc.clear();
        unsigned int flag32 = (((g_base + (unsigned int)s) >> 1) & 1u) ? 0x40004000u : 0u;
        asm volatile("" : "+v"(flag32));  // (made here, not in front of the store)
        const unsigned long long flag = ((unsigned long long)flag32 << 32) | flag32;
        if (!polled) {
            // steps s + 16 .. s + 31 are fetched when step s starts a half, and written over the half that has just been
            // used up one step later (in a polling wavefront the poll in between has waited for them)
            if ((s & 15) == 0 && s > 0) xp_next = fetch_xp(s + 16);
            if ((s & 15) == 1 && s > 1) deposit_xp(((s >> 4) & 1) ^ 1, xp_next);
        } else if (fetcher && s >= 1 && s + 1 < T) {
            // loaded during step s - 1; read (by this wavefront and by wavefront w - 4) after the barrier of step s + 1
            reinterpret_cast<unsigned int&>(xring[wave][(s + 1) & 31][my_gate][unit]) = xp_ahead;
            reinterpret_cast<unsigned int&>(xring[wave - 4][(s + 1) & 31][my_gate][unit]) = xp_ahead_other;
        }
        if (sums && s > 0) in_ring[(s - 1) & 1][lane & 31] = in_ahead;  // read after this step's barrier
        // ---- 1. h of the previous step into LDS
        if (polls) {
            half8_t hv;
            if (s == 0) {
                hv = __builtin_bit_cast(half8_t, load16_nt(ch.h0 + piece * 8));  // (waited for here: left to the compiler it is a wait for all memory in every step)
            } else {
                const unsigned int gp = g_base + (unsigned int)s - 1u;
                const unsigned int want = ((gp >> 1) & 1u) ? 0x40004000u : 0u;
                const unsigned char* src = reinterpret_cast<const unsigned char*>(region + (long)(gp & 1u) * kXcdMembers * kXcdEntryWords) + piece * 16;
                xcd_u32x4 v;
                bounded_wait(gave_up, [&]() {
                    v = load16_nt(src) ^ want;   // what has its flags is h, without them, by that
                    return ((v[0] | v[1] | v[2] | v[3]) & 0x40004000u) == 0u;
                });
                hv = __builtin_bit_cast(half8_t, v);
            }
            if (in_range) *reinterpret_cast<half8_t*>(hb + Product::place(piece) * 8) = hv;
        }
        if (gave_up) block_gave_up = 1;
        lds_barrier();
        // (the same value in every thread: it is written in front of barriers only.  Asked for here, with the reads of h,
        // and looked at where values would leave the workgroup: the step's arithmetic does not wait for it)
        // The operands of the product and the projection terms are asked for here too, in front of everything that is not on
        // the step's path: the terms behind the sums came an LDS round trip (100 cycles) later.
        const int dead_lds = block_gave_up;
        const typename Product::Operands operands = Product::operands(operands_at);
        unsigned int xp_bits = *(__attribute__((address_space(3))) const unsigned int*)(uintptr_t)xp_at;
        __builtin_amdgcn_sched_barrier(0);
        const int dead = __builtin_amdgcn_readfirstlane(dead_lds);
        if (polled && fetcher && s + 2 < T) {
            xp_ahead = xp_bits_at(s + 2);
            xp_ahead_other = __hip_atomic_load(xp_other + (long)(s + 2) * 4 * H, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // The previous step's h of the whole workgroup (gathered in LDS before the barrier) goes to the layer above, from a
        // wavefront that does not poll.
        if (!res && feeds && s > 0 && wave == 4 && lane < 4 && rank * kXcdUnitsPerBlock + lane * 8 < H && !dead) emit(s - 1);
        if (sums) {
            in_ahead = __hip_atomic_load(reinterpret_cast<const unsigned short*>(ch.res_in) + (long)s * H + eu, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            if (s > 0 && !dead) emit_sum(s - 1);
        }
        if (res) gave_up = gave_up || __builtin_amdgcn_ballot_w64(sum_gave_up) != 0ull;

        // (a wavefront one of whose waits gave up after this step's barrier makes its h from stale values: it keeps them
        // to itself, and the group's other members stop at their next wait)
        bool stop = dead || gave_up;

        // ---- 2. the wavefront's 16 gate rows
        const float dot = weights.matvec(hb, operands, acc, H, lane);
        if (polled && __builtin_amdgcn_ballot_w64(xp_bits == 0xffffffffu) != 0ull) {  // the P group had not got there when it was fetched
            xp_bits = wait_xp(s, xp_bits);
            stop = stop || gave_up;
        }
        const float a = dot + __builtin_bit_cast(float, xp_bits);
        // Every lane activates its own gate; the lanes of a unit then share them.
        // sigmoid(a), or tanh(a) = 2 sigmoid(2a) - 1 for g: the factors are the lane's (exact: powers of two, one and zero).
        const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gate_scale * a));
        const float act = __builtin_fmaf(sg, gate_mul, gate_add);
        float g_i, g_f, g_g, g_o;
        Product::share(act, g_i, g_f, g_g, g_o);
        const float c_new = g_f * c_reg + g_i * g_g;
        const bool h_is_number = (c_new == c_new) && (g_o == g_o);
        const half_t h = (half_t)(g_o * __builtin_fmaf(__builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.0f * kXcdLog2 * c_new)), 2.0f, -1.0f));
        c_reg = c_new;

        // ---- 3. the wavefront's four h values: lane 0 publishes, then stores y (whose place in front of the publishing store
        // nothing may take: everybody waits for that one)
        const unsigned int hb16 = (unsigned int)__builtin_bit_cast(unsigned short, h);
        const unsigned int pb16 = h_is_number ? hb16 : 0u;       // a NaN cannot carry the flag: it is exchanged as 0, y keeps it
        const unsigned int sb16 = h_is_number ? hb16 : 0x7e00u;  // and goes to the layer above in its canonical form
        const unsigned long long pw = Product::pack(pb16);
        // units past H publish zeros with the flag, so that every piece of a member's entry validates
        if (publishes && !stop) store8_plain(publish_at, (pw & published) | flag);
        publish_at += publish_step;
        publish_step = -publish_step;
        const unsigned long long yw = Product::pack(hb16);
        const unsigned long long sw = emits ? Product::pack(sb16) : 0ull;
        if (stores_y) *reinterpret_cast<unsigned long long*>(y_at) = yw;
        y_at += y_step;
        if (emits && lane == 0) hout[s & 1][wave] = sw;
        if (s == T - 1 && units_ok && Product::first_of_unit(lane)) {
            ch.hn[my_unit] = h;
            ch.cn[my_unit] = (half_t)c_new;
        }
        if (dead) break;  // (a step made on stale values: nothing of it has left the workgroup)
    }
    if (emits && sums) in_ring[(T - 1) & 1][lane & 31] = in_ahead;
    if (gave_up) block_gave_up = 1;
    lds_barrier();
    if (emits && !block_gave_up) {
        if (!res && wave == 4 && lane < 4 && rank * kXcdUnitsPerBlock + lane * 8 < H) emit(T - 1);
        if (sums) emit_sum(T - 1);
        if (res && __builtin_amdgcn_ballot_w64(sum_gave_up) != 0ull) block_gave_up = 1;  // (the last sum's own wait)
    }
    lds_barrier();
    };
    const bool polled_rt = PIPE && ch.xproj_polled != 0;
    const bool feeds_rt = PIPE && ch.seq_out != nullptr;
    const bool res_rt = RES && ch.res_in != nullptr;
    if (poisoned) {
        // (nothing is exchanged)
    } else if (RES && res_rt) {
        if (!polled_rt && !feeds_rt) recurrence(std::false_type{}, std::false_type{}, std::true_type{});
        else if (!polled_rt) recurrence(std::false_type{}, std::true_type{}, std::true_type{});
        else if (!feeds_rt) recurrence(std::true_type{}, std::false_type{}, std::true_type{});
        else recurrence(std::true_type{}, std::true_type{}, std::true_type{});
    } else if (!PIPE || (!polled_rt && !feeds_rt)) recurrence(std::false_type{}, std::false_type{}, std::false_type{});
    else if (!polled_rt) recurrence(std::false_type{}, std::true_type{}, std::false_type{});
    else if (!feeds_rt) recurrence(std::true_type{}, std::false_type{}, std::false_type{});
    else recurrence(std::true_type{}, std::true_type{}, std::false_type{});
    if (block_gave_up) {
        // ---- self-sufficient: this workgroup's units of chain k, from the call's inputs, by this workgroup alone: the layers
        // below it in the launch are recomputed on the way (lstm_solo.h) ----
        SoloStack st;
        st.y_stride = p.y_stride;
        st.H = H;
        st.T = T;
        const int first = PIPE ? 0 : k;  // independent chains (the two directions of a layer) have their own projection rows
        st.n = k - first + 1;
        st.xproj = p.chain[first].xproj;
        st.res_in0 = RES ? p.chain[first].res_in : nullptr;
        st.reverse = ch.reverse;
#pragma unroll
        for (int j = 0; j < kXcdMaxChains; ++j) {
            if (first + j > k) break;
            const XcdChain& cj = p.chain[first + j];
            SoloLayer& ly = st.layer[j];
            ly.w_hh = cj.w_hh;
            ly.w_ih = j > 0 ? p.proj[first + j - 1].w_ih : nullptr;
            ly.bsum = j > 0 ? p.proj[first + j - 1].bsum : nullptr;
            ly.h0 = cj.h0;
            ly.c0 = cj.c0;
            ly.residual = (RES && cj.res_in != nullptr) ? 1 : 0;
            const bool mine = first + j == k;
            ly.y = mine ? cj.y : nullptr;
            ly.hn = cj.hn;
            ly.cn = cj.cn;
            ly.u_begin = mine ? min(rank * kXcdUnitsPerBlock, H) : 0;
            ly.u_end = mine ? min((rank + 1) * kXcdUnitsPerBlock, H) : 0;
        }
        lstm_solo_stack<kXcdThreads, PIPE ? kXcdMaxChains : 1, kXcdMaxH>(st);
        return;
    }
    // Rank 0 has finished its last step, for which (T >= 2) it needed what every member published one step earlier:
    // every member has read the counter by now.
    if (rank == 0 && tid == 0)
        __hip_atomic_store(p.g_counter + k, g_base + (unsigned int)T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// FRAGS: four up to kXcdFewUnits, otherwise sixteen.
template <bool PIPE, int FRAGS>
__global__ __launch_bounds__(kXcdThreads) void lstm_xcd_f16_kernel(LstmXcdArgs p)
{
    lstm_xcd_body<PIPE, false, XcdSparse<FRAGS>>(p);
}

template <bool PIPE>
__global__ __launch_bounds__(kXcdThreads) void lstm_xcd_dot_f16_kernel(LstmXcdArgs p)
{
    lstm_xcd_body<PIPE, false, XcdDot>(p);
}

// The pipeline for stacks that have layers with a residual sum.
template <int FRAGS>
__global__ __launch_bounds__(kXcdThreads) void lstm_xcd_res_f16_kernel(LstmXcdArgs p)
{
    lstm_xcd_body<true, true, XcdSparse<FRAGS>>(p);
}

}  // namespace pimhip
