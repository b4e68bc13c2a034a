// An RNN-transducer's whole greedy decoding loop over one utterance in one launch (gfx950, batch 1, fp16 storage, fp32 sums).
//
//     t = 0, last = start of sequence, state = (h0, c0); g, state = prediction(last, state)
//     while t < T and fewer than max_symbols emitted:
//         k = argmax(joint(enc[t], g))
//         if k == blank:  t += 1
//         else:           emit k; g, state = prediction(embedding[k], state); after max_per_frame symbols of one frame t += 1
//
// The reference interprets this loop operator by operator (prim::Loop,
// runtime/source/executor/op_executor/prim_ops_executor.cpp:820-875; per iteration executeAtenLSTM1 with seq_len == 1,
// aten_ops_executor.cpp:2135-2307, the joint network's products, aten_ops_executor.cpp:181-216, and executeAtenArgmax,
// aten_ops_executor.cpp:520-560, whose result the host reads before the next iteration): launches, gaps and a device-to-host
// round trip per step, far more than the 4.7 MB of weights cost.  rnnt_step_f16_kernel makes an iteration one launch; here
// the loop itself runs on the device:
//
//   * the same roles as the step kernel (blocks of eight hidden units per layer, of eight joint rows, of eight symbols),
//     but every workgroup stays for the whole utterance with its rows of the weights in registers: nothing is read again;
//   * the argmax is taken by every workgroup for itself from the logits that the symbol blocks publish, so the decision
//     travels with the hand-over that ends the step and every workgroup keeps the same loop state (t, symbols so far, ..);
//   * a layer's blocks also collect their own layer's h (what W_hh multiplies at the next symbol) and sum W_hh . h right
//     then, long before the next symbol is known;
//   * the first layer does not wait for the decision either (rnnt_greedy_every in rnnt_plan.h): its blocks keep the gates' sums over
//     every symbol's embedding row, make h for every symbol as soon as the h before it is known, a symbol to a lane, and publish them
//     all; who needs the first layer's h reads the decided symbol's words, which are there already.  A symbol's chain loses a cell (0.7 us) and
//     the way of a store (0.4 us);
//   * most steps of a real utterance are blanks, after which only the frame changes: the joint blocks do not wait for the
//     decision but publish the hidden vectors of the next steps as well, up to twelve ahead, as if every decision in
//     between were a blank, and the symbol blocks turn every hidden vector that arrives into logits.  When a symbol is emitted, g gets
//     a new version and what was computed ahead under the old one is simply never looked at.  A row's sum over the frame and its
//     sum over g are made apart: the frames' ahead of their turn, a frame to a wavefront with all of the block's rows, and g's once per version, so
//     that the words of all steps ahead are sums of two values each and one store;
//   * the symbol blocks exist several times over, as TEAMS: a symbol block's round (a look at 64 entries, a barrier, its sums, the
//     publish) takes 2 us however few rows it has, so one set of blocks handles a run of blanks one or two steps a round.  The
//     CUs that no other role needs hold up to eleven further copies of W2's rows, team q takes the steps that are q modulo the
//     number of teams, and the steps published ahead become logits side by side;
//   * the decision behind a symbol, which everybody waits for while nothing else is there, is not waited for from the symbol blocks: with
//     up to 64 symbols (rnnt_greedy_own_rows) the blocks of layers and joint network read the hidden vector and make it themselves (decided_alone).
//
// Measured on MI355X, us an utterance of 341 frames (2 x 320 units, 512 joint units, 29 symbols) with 74 / 114 symbols emitted: 739 /
// 996 with a hand-over of the first layer's h and of the logits per symbol, 667 / 905 without the first, 618 / 814 without both, 581 / 784
// with the sums over frames and g apart; 200 frames of 100 symbols with 34 emitted 395 / 387 / 382 / 344, of 300 symbols with 44 emitted 510 -> 481.  What bounds it
// now: of a symbol's 5 us two hand-overs of 1.1 and the look at the first layer's words of 0.95, then the cell 0.5, a joint row 0.4,
// logits and decision 0.9; in a run of blanks the steps ahead over the two hand-overs and the symbol blocks' rounds (steps ahead / teams: 8 / 8
// 605 and 366, 12 / 8 595 and 343, 16 / 8 605 and 339, 12 / 12 581 and 344 in the first and the 100-symbol case).  Not kept: all logits made by
// every block, without symbol blocks (a run of blanks 0.6 -> 0.85 us a step, eight steps' logits take every block 1.9 us); the first layer's words of
// all symbols collected ahead of the decision (28 KB a block and symbol, 2.8 us); fewer steps ahead behind a symbol (0, 2, 4 instead of 8: 705, 669, 632
// against 606).
//
// Exchange: 8-byte words of three fp16 values and a 16-bit tag, three words per producing block in a 128-byte entry of its
// own, written and read with device-scope accesses.  The tag says what the word belongs to: h of a layer carries the
// version of g (the count of the prediction network's runs), so do its words for every symbol, in entries of their own; hidden vectors and logits carry the step and the version they
// were computed under; a word with another tag is "not there yet", so nothing is ever cleared and a stale word cannot be
// taken for a fresh one.  h lives in four sets by version, hidden vectors in a ring of 32 by step, logits in one of 64.  A
// producer may overwrite what is a ring old: for the joint blocks' entries that follows from the order of things where all decisions
// come from the symbol blocks (they run at most twelve steps ahead of decisions that the symbol blocks have already published); where
// blocks decide for themselves, and for the symbol blocks' entries, a slow reader could fall a ring behind (nobody waits for the symbol blocks
// during a run of symbols, nor for the layers' blocks during a run of blanks): the producers look at a count that every block keeps of the
// decisions it has taken in (`seen`) before they reuse an entry.
//
// Waiting: a block looks at everything it waits for in one round ("pass"): the words of a vector by the first six
// wavefronts, the logits of the next steps by the last ones (of four steps by one wavefront with up to 40 symbols, one step by
// each beyond).  What the block cannot go on without is polled until it is there, the rest is looked at once; one barrier ends the round, and
// a pass can take several decisions at once: a run of blanks is a run of ones in a ballot.
//
// Sums run in the order of the step kernel, c is rounded to fp16 after every run of the prediction network as it is when
// the state travels between launches: symbols and final state equal, bit for bit, those of a loop of pimhip_rnnt_step
// driven from the host.
//
// Every wait is bounded.  A workgroup whose wait gives up raises the abort word; every workgroup then leaves the loop at its
// next wait, and the first to claim `solo_owner` decodes the whole utterance again from its start by itself (slower, tens
// of microseconds per step, the same sums): a wait that gives up costs time, not the result.
#pragma once

#include <type_traits>

#include "rnnt_kernels.h"
#include "rnnt_plan.h"

namespace pimhip
{

constexpr int kRnntGreedyVersions = 4;             // h of a layer: one entry per block and version of g, modulo this
constexpr int kRnntGreedyRing = 32;                // hidden vectors: one entry per block and step, modulo this
constexpr int kRnntGreedyLogitRing = 64;           // logits: the same
constexpr int kRnntGreedyAhead = 12;                // steps the joint network runs ahead of the decisions
constexpr int kRnntGreedyLook = 8;                 // steps whose logits one pass looks at, at most
constexpr int kRnntGreedyTeams = 12;               // at most this many teams of symbol blocks, each with the steps of one residue
constexpr int kRnntGreedyBatch = 2;                // steps' logits a symbol block publishes behind one barrier
constexpr int kRnntGreedyFrames = 64;              // frames whose sums a joint block keeps, by frame modulo this
constexpr int kRnntGreedyFramesAhead = 48;         // frames ahead of the current one that it sums at most
static_assert(kRnntGreedyAhead + 1 + kRnntWaves <= kRnntGreedyFramesAhead && kRnntGreedyFramesAhead <= kRnntGreedyFrames, "what a publish needs is kept, and nothing it needs is overwritten");
static_assert(3 * (kRnntGreedyAhead + 1) <= 64, "a joint block's words of all steps it publishes are one store of a wavefront");
static_assert(kRnntGreedyAhead < kRnntGreedyRing && (kRnntGreedyRing & (kRnntGreedyRing - 1)) == 0, "ring");
static_assert((kRnntGreedyLogitRing & (kRnntGreedyLogitRing - 1)) == 0 && kRnntGreedyLogitRing <= 128, "a ring's steps differ in their 8-bit tags");
static_assert(kRnntGreedyLook + kRnntGreedyAhead < kRnntGreedyLogitRing, "a look and what is published ahead of it lie in one ring");
static_assert(kRnntGreedyLook == kRnntWaves && kRnntGreedyLook == 8, "a wavefront per step");
static_assert(kRnntGreedyBatch <= kRnntWaves, "a wavefront stores one step's word of a batch");
constexpr int kRnntGreedyMaxVocab = 512;           // symbols
constexpr int kRnntGreedyRows = 4;                 // steps that a pass looks at where a step's logits are a row of 16 lanes'
constexpr int kRnntGreedyLaneWords = 3;            // at most this many words of a step's logits to a lane where a wavefront takes them
static_assert(3 * (kRnntGreedyMaxVocab / 8) <= 64 * kRnntGreedyLaneWords, "a wavefront takes a step's logits");
constexpr int kRnntGreedyEmbHalfs = 16384;         // embedding rows kept in LDS by the first layer's blocks (32 KB)
// 8-byte words that a block of the first layer publishes its units' h after every symbol in: three a symbol, whole 128-byte lines.
__host__ __device__ inline int rnnt_every_words(int vocab) { return (3 * vocab + 15) & ~15; }
constexpr int kRnntSeenStride = 16;                // 32-bit words between the blocks' `seen` counts

struct RnntGreedyArgs {
    RnntLayer layer[kRnntMaxLayers];
    const half_t* w1;          // [J, F + H]
    const half_t* b1;          // [J] or null
    const half_t* w2;          // [V, J]
    const half_t* b2;          // [V] or null
    const half_t* enc;         // [T, F]
    const half_t* embedding;   // [emb_rows, in_w of layer 0]: row k is the prediction network's input after symbol k
    const half_t* x0;          // [in_w of layer 0]: its input before any symbol
    const half_t* h0;          // [L, H] or null (zeros)
    const half_t* c0;
    half_t* hn;                // [L, H] or null
    half_t* cn;
    int* symbols;              // [max_symbols]
    int* result;               // [8]: symbols emitted, frames consumed, steps taken, 1 if one workgroup decoded alone, whether the
                               // last symbol is still to be fed to the prediction network, the last symbol (-1: none), 0, 0
    // Entries of kRnntEntryWords words, all ones at the start: h [kRnntGreedyVersions][the layers' blocks], hidden vectors
    // [kRnntGreedyRing][joint blocks], logits [kRnntGreedyLogitRing][symbol blocks of one team] (h_entry, hid_entry, lg_entry).
    unsigned long long* hx;
    unsigned long long* every; // [kRnntGreedyVersions][blocks of the first layer][rnnt_every_words]: h of the first layer after every symbol (EVERY)
    unsigned int* seen;        // [gridDim.x][kRnntSeenStride], the blocks of all teams, zero at the start
    unsigned int* solo_owner;  // zero at the start
    unsigned int* abort_flag;
    unsigned int* abort_host;
    int L, H, F, J, V, T;
    int emb_rows, emb_in_lds;
    int blank, max_symbols, max_per_frame;
    int run_pred_first;        // 0: the first step takes g = h0 of the last layer as it is (decoding goes on after a blank)
    int teams;                 // teams of symbol blocks: team q has the steps that are q modulo `teams`
    unsigned int spin_limit;
    int alone;                 // the launch is one workgroup that decodes by itself
};

struct RnntGreedyState {
    int t, emitted, frame_syms, label, run_pred;
};

// What symbol k does to the loop; returns whether k was emitted.
__device__ __forceinline__ bool rnnt_greedy_advance(RnntGreedyState& s, int k, int blank, int max_per_frame)
{
    if (k == blank) {
        s.t += 1;
        s.frame_syms = 0;
        s.run_pred = 0;
        return false;
    }
    s.label = k;
    s.emitted += 1;
    s.frame_syms += 1;
    s.run_pred = 1;
    if (s.frame_syms >= max_per_frame) {
        s.t += 1;
        s.frame_syms = 0;
    }
    return true;
}

template <int CTRL>
__device__ __forceinline__ unsigned int rnnt_dpp_u32(unsigned int v)
{
    return (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}

// The maximum over the 64 lanes; every lane returns it.
__device__ __forceinline__ unsigned int rnnt_max_u32(unsigned int v)
{
    v = max(v, rnnt_dpp_u32<kDppQuadXor1>(v));
    v = max(v, rnnt_dpp_u32<kDppQuadXor2>(v));
    v = max(v, rnnt_dpp_u32<0x124>(v));
    v = max(v, rnnt_dpp_u32<0x128>(v));
    {
        unsigned int a = v, b = v;
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
        v = max(a, b);
    }
    {
        unsigned int a = v, b = v;
        asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
        v = max(a, b);
    }
    return v;
}

// torch.argmax over fp16 values: the first maximum, a NaN counting as the largest.  One integer maximum over keys: the value's
// bits made monotonic (-0 as +0, a NaN above everything) in front of the index counted from the top, so that of equal
// values the first wins.  A key is never 0.
__device__ __forceinline__ unsigned int rnnt_key(unsigned int bits, int i)
{
    if (bits == 0x8000u) bits = 0u;
    unsigned int order = (bits & 0x8000u) ? (~bits & 0xffffu) : (bits | 0x8000u);
    if ((bits & 0x7fffu) > 0x7c00u) order = 0xffffu;
    return (order << 16) | (unsigned int)(0xffff - i);
}

__device__ __forceinline__ int rnnt_key_index(unsigned int key) { return 0xffff - (int)(key & 0xffffu); }

// The argmax of lg[0 .. V); every lane returns it.  A lane takes the values lane, lane + 64, ..
__device__ __forceinline__ int rnnt_argmax(const half_t* lg, int V, int lane)
{
    unsigned int key = 0u;
    for (int i = lane; i < V; i += 64) key = max(key, rnnt_key(__builtin_bit_cast(unsigned short, lg[i]), i));
    return rnnt_key_index(rnnt_max_u32(key));
}

// The largest key of a word of logits: values 8 prod + 3 part .. + 2 (the third word of a block has two).
__device__ __forceinline__ unsigned int rnnt_word_key(unsigned long long w, int prod, int part)
{
    const int i = 8 * prod + 3 * part;
    unsigned int key = max(rnnt_key((unsigned int)w & 0xffffu, i), rnnt_key((unsigned int)(w >> 16) & 0xffffu, i + 1));
    if (part < 2) key = max(key, rnnt_key((unsigned int)(w >> 32) & 0xffffu, i + 2));
    return key;
}

// The maximum over a row of 16 lanes; every lane of the row returns it.
__device__ __forceinline__ unsigned int rnnt_max_row(unsigned int v)
{
    v = max(v, rnnt_dpp_u32<kDppQuadXor1>(v));
    v = max(v, rnnt_dpp_u32<kDppQuadXor2>(v));
    v = max(v, rnnt_dpp_u32<0x124>(v));
    return max(v, rnnt_dpp_u32<0x128>(v));
}

// The whole loop by one workgroup.  LDS: hs [L * H] (h of every layer), cs [L * H], tmp [max(H, J)], lg [V].
__device__ __forceinline__ void rnnt_greedy_solo(const RnntGreedyArgs& p, half_t* hs, half_t* cs, half_t* tmp, half_t* lg)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int H = p.H, nhp = H >> 3, nfp = p.F >> 3, njp = p.J >> 3;
    __syncthreads();
    for (int i = tid; i < p.L * H; i += kRnntThreads) {
        hs[i] = p.h0 ? p.h0[i] : (half_t)0.0f;
        cs[i] = p.c0 ? p.c0[i] : (half_t)0.0f;
    }
    __syncthreads();
    RnntGreedyState s = {0, 0, 0, -1, p.run_pred_first};
    int steps = 0;
    while (s.t < p.T && s.emitted < p.max_symbols) {
        if (s.run_pred) {
            const half_t* x = s.label < 0 ? p.x0 : p.embedding + (long)s.label * p.layer[0].in_w;
            for (int l = 0; l < p.L; ++l) {
                const RnntLayer ly = p.layer[l];
                const int nxp = ly.in_w >> 3;
                const half8_t* in = reinterpret_cast<const half8_t*>(l == 0 ? x : hs + (long)(l - 1) * H);
                const half8_t* hv = reinterpret_cast<const half8_t*>(hs + (long)l * H);
                for (int u = wave; u < H; u += kRnntWaves) {
                    float a[4], ah[4];
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const long r = (long)g * H + u;
                        ah[g] = rnnt_row_dot(reinterpret_cast<const half8_t*>(ly.w_hh + r * H), hv, nhp, lane, 0.0f);
                        a[g] = rnnt_row_dot(reinterpret_cast<const half8_t*>(ly.w_ih + r * ly.in_w), in, nxp, lane, 0.0f);
                    }
                    float c_new;
                    half_t h_new;
                    const float hidden = rnnt_gate_sum(ah, lane) + (ly.bsum ? ly.bsum[(long)(lane & 3) * H + u] : 0.0f);
                    rnnt_unit(rnnt_gate_sum(a, lane) + hidden, (float)cs[(long)l * H + u], lane, c_new, h_new);
                    if (lane == 0) {
                        tmp[u] = __builtin_bit_cast(half_t, rnnt_bits((float)h_new));
                        cs[(long)l * H + u] = rnnt_round(c_new);
                    }
                }
                __syncthreads();
                for (int i = tid; i < H; i += kRnntThreads) hs[(long)l * H + i] = tmp[i];
                __syncthreads();
            }
        }
        const half8_t* fv = reinterpret_cast<const half8_t*>(p.enc + (long)s.t * p.F);
        const half8_t* gv = reinterpret_cast<const half8_t*>(hs + (long)(p.L - 1) * H);
        for (int r = wave; r < p.J; r += kRnntWaves) {
            const half8_t* row = reinterpret_cast<const half8_t*>(p.w1 + (long)r * (p.F + H));
            const float f = rnnt_sum(rnnt_row_dot(row, fv, nfp, lane, 0.0f));
            const float g = rnnt_sum(rnnt_row_dot(row + nfp, gv, nhp, lane, 0.0f));
            if (lane == 0) tmp[r] = __builtin_bit_cast(half_t, rnnt_bits(relu_f32(f + (g + (p.b1 ? (float)p.b1[r] : 0.0f)))));
        }
        __syncthreads();
        for (int v = wave; v < p.V; v += kRnntWaves) {
            float a = rnnt_row_dot(reinterpret_cast<const half8_t*>(p.w2 + (long)v * p.J), reinterpret_cast<const half8_t*>(tmp), njp, lane, 0.0f);
            a = rnnt_sum(a);
            if (lane == 0) lg[v] = __builtin_bit_cast(half_t, rnnt_bits(a + (p.b2 ? (float)p.b2[v] : 0.0f)));
        }
        __syncthreads();
        const int k = rnnt_argmax(lg, p.V, lane);
        const int at = s.emitted;
        if (rnnt_greedy_advance(s, k, p.blank, p.max_per_frame) && tid == 0) p.symbols[at] = k;
        ++steps;
        __syncthreads();
    }
    for (int i = tid; i < p.L * H; i += kRnntThreads) {
        if (p.hn) p.hn[i] = hs[i];
        if (p.cn) p.cn[i] = cs[i];
    }
    if (tid == 0) {
        p.result[0] = s.emitted;
        p.result[1] = s.t;
        p.result[2] = steps;
        p.result[3] = 1;
        p.result[4] = s.run_pred;
        p.result[5] = s.label;
    }
}

// LANE_WORDS: rnnt_greedy_lane_words.  The loop that polls for logits stands in every hand-over of a decision, so it is compiled for the
// number of words and nothing else: with three for every vocabulary past 40 symbols and a branch between it and the row's, a
// transcript of symbols alone took (2 x 320 units, 512 joint units, us a step) 7.29 with 41, 7.54 with 100, 7.58 with 169 and 7.74 with 512
// symbols, 6.95, 7.21, 7.49 and 7.71 as it is; a run of blanks 1.07, 1.09, 1.11 and 1.28, now 0.94, 0.96, 1.02 and 1.27.
// EVERY: rnnt_greedy_every.  OWN_ROWS: rnnt_greedy_own_rows, of OWN_PIECES 16-byte pieces a lane (512 joint units each).
template <int LANE_WORDS, bool EVERY, int OWN_ROWS, int OWN_PIECES>
__global__ __launch_bounds__(kRnntThreads) void rnnt_greedy_f16_kernel(const RnntGreedyArgs p)
{
    typedef unsigned long long u64;
    __shared__ __align__(16) half_t buf0[kRnntMaxVec];                              // the vector a role waits for
    __shared__ __align__(16) half_t own[kRnntMaxH];                                 // a layer's blocks: h of their layer; joint blocks: g
    __shared__ unsigned int keys[2][kRnntGreedyLook];                               // per pass (alternating): the best key of the next steps' logits, 0: not there
    __shared__ __align__(16) half_t emb[kRnntGreedyEmbHalfs];                       // first layer: the embedding rows and x0 behind them
    __shared__ __align__(16) unsigned short mine[2][kRnntGreedyBatch][12];          // this block's eight values (a symbol block's of two steps), alternating per publish
    __shared__ __align__(16) float4_t ih_of[EVERY ? kRnntWaves : 1][EVERY ? kRnntGreedyEveryVocab : 1];  // first layer: a unit's gate sums over every symbol's row
    __shared__ __align__(16) unsigned short every_mine[EVERY ? kRnntGreedyEveryVocab : 1][12];           // ... and this block's values of h after it
    __shared__ unsigned int own_keys[OWN_ROWS ? kRnntWaves * OWN_ROWS / 4 : 1];     // the best key among a wavefront's rows of W2
    __shared__ int missing[3][3];                                                   // per pass (rotating): something of the vector is not there yet; a
                                                                                    // wait has given up; something of a second vector is not there
    __shared__ int someone_gave_up;
    __shared__ int i_decode_alone;
    __shared__ int min_seen_lds;
    __shared__ int seen_lds[2];                                                     // joint blocks: the same, made beside their rounds (alternating)

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = gridDim.x, b = blockIdx.x;
    const int H = p.H, nhp = H >> 3, nwh = H >> 3, nwj = p.J >> 3, nwv = (p.V + 7) >> 3;
    const int n_lstm = p.L * nwh;

    // The solo decoder's arrays lie where the embedding rows lay (the team's loop is over by then).
    half_t* solo_hs = emb;
    half_t* solo_cs = emb + kRnntMaxLayers * kRnntMaxH;
    static_assert(2 * kRnntMaxLayers * kRnntMaxH <= kRnntGreedyEmbHalfs, "the solo decoder's state fits where the embedding rows lay");

    if (tid == 0) {
        someone_gave_up = (p.alone || __hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) ? 1 : 0;
        i_decode_alone = 0;
    }
    if (tid < 9) (&missing[0][0])[tid] = 0;
    if (tid < 2 * kRnntGreedyBatch * 12) (&mine[0][0][0])[tid] = 0;
    if constexpr (EVERY)
        for (int i = tid; i < kRnntGreedyEveryVocab * 12; i += kRnntThreads) (&every_mine[0][0])[i] = 0;
    __syncthreads();

    RnntGreedyState s = {0, 0, 0, -1, p.run_pred_first};
    int n_pred = 0, step = 0;          // runs of the prediction network and steps so far
    unsigned int n_pass = 0, n_publish = 0, waited = 0;
    bool dead = false;                 // a wait of this block has given up (the same in every thread)
    unsigned long long t_first = 0ull;

    auto running = [&]() __attribute__((always_inline)) { return s.t < p.T && s.emitted < p.max_symbols; };
    // The version of g that the current step's joint network sees: runs of the prediction network started, less one.
    auto g_version = [&]() __attribute__((always_inline)) { return n_pred + s.run_pred - 1; };
    auto h_tag = [](int version) { return (unsigned int)(version & 0x7fff); };
    auto step_tag = [](int st, int version) { return (unsigned int)(((version & 0x7f) << 8) | (st & 0xff)); };
    auto h_entry = [&](int version, int block) __attribute__((always_inline)) { return p.hx + ((long)(version & (kRnntGreedyVersions - 1)) * n_lstm + block) * kRnntEntryWords; };
    auto hid_entry = [&](int st, int j) __attribute__((always_inline)) {
        return p.hx + ((long)kRnntGreedyVersions * n_lstm + (long)(st & (kRnntGreedyRing - 1)) * nwj + j) * kRnntEntryWords;
    };
    auto lg_entry = [&](int st, int j) __attribute__((always_inline)) {
        return p.hx + ((long)kRnntGreedyVersions * n_lstm + (long)kRnntGreedyRing * nwj + (long)(st & (kRnntGreedyLogitRing - 1)) * nwv + j) * kRnntEntryWords;
    };

    // mine[which] of this publish goes out as three 8-byte words of three values and the tag each, from one wavefront (several
    // steps of a joint or symbol block: one wavefront each behind the same barrier).
    auto store_words = [&](int which, u64* entry, unsigned int tag) __attribute__((always_inline)) {
        if (lane < 3) {
            const unsigned short* m = mine[n_publish & 1u][which] + 3 * lane;
            const u64 w = (u64)m[0] | ((u64)m[1] << 16) | ((u64)m[2] << 32) | ((u64)tag << 48);
            __hip_atomic_store(entry + lane, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    auto my_value = [&](int which) __attribute__((always_inline)) -> unsigned short& { return mine[n_publish & 1u][which][wave]; };

    // One 8-byte word: looked at once, or (blocks) polled until it carries `tag` or the wait's limits are reached, in which
    // case the thread raises the abort words and this pass's "gave up" flag.  Returns whether the tag is there.
    auto fetch = [&](const u64* slot, unsigned int tag, bool blocks, int* miss, u64& w) __attribute__((always_inline)) {
        unsigned int spins = 0;
        unsigned long long first = 0ull;
        while (true) {
            w = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((unsigned int)(w >> 48) == tag) return true;
            if (!blocks) return false;
            bool give_up = false;
            if (spins > 0u && (spins & 255u) == 0u) {
                if (__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) give_up = true;
                if (wait_clock_expired(spins, first)) spins = 0xffffffffu;
            }
            if (spins >= p.spin_limit) {
                __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                give_up = true;
            }
            if (give_up) {
                miss[1] = 1;
                someone_gave_up = 1;
                return false;
            }
            if (spins != 0xffffffffu) ++spins;
        }
    };
    auto unpack = [&](u64 w, half_t* dst, int prod, int part) __attribute__((always_inline)) {
        unsigned short* d = reinterpret_cast<unsigned short*>(dst) + 8 * prod + 3 * part;
        d[0] = (unsigned short)w;
        d[1] = (unsigned short)(w >> 16);
        if (part < 2) d[2] = (unsigned short)(w >> 32);
    };
    // One round over everything this block waits for: the 8-byte words of a vector (n_vec producers from `vec`, tagged
    // vec_tag, values to vec_dst) by the first six wavefronts, and with look_waves the logits of the steps from `step` on under
    // the current version by as many of the last wavefronts: one step each, or, where a step's words fit a row of 16 lanes, four
    // steps by the last one.  The wavefront that takes a step's words makes the argmax of them (its key) right there, so that behind
    // the barrier nothing but a few keys is left to read.  What the block cannot go on without is polled until it is there
    // (vec_blocks; step_blocks: the logits of `step`), the rest is looked at once.  Returns bit 0: the vector is complete.
    // A second vector (vec2, looked at once) is taken along where the first leaves threads free; bit 1 says it is complete.
    // my_key, n_there: the key of step + lane % 8 in every lane, and how many steps from `step` on are there.
    // (The wavefronts that poll what a step is waited for with are not those that store: a wavefront's memory operations return
    // in order, and a device-scope store's acknowledgement takes longer than a poll.)
    unsigned int my_key = 0u;
    int n_there = 0;
    constexpr bool row_per_step = LANE_WORDS == 0;
    auto pass = [&](const u64* vec, int n_vec, unsigned int vec_tag, half_t* vec_dst, bool vec_blocks, int look_waves, bool step_blocks, int vec_stride = kRnntEntryWords,
                    const u64* vec2 = nullptr, int n_vec2 = 0, unsigned int vec2_tag = 0u, half_t* vec2_dst = nullptr) __attribute__((always_inline)) -> int {
        int* miss = missing[n_pass % 3u];
        u64 w;
        const int look = kRnntWaves - 1 - wave;
        if (look >= look_waves) {
            if (tid < 384) {
                // Where a symbol is on its way and this team's hidden vector is not the next one, one word of it is looked at first.
                const bool there_yet = !s.run_pred || vec_blocks || n_vec == 0 ||
                                       (unsigned int)(__hip_atomic_load(vec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 48) == vec_tag;
                if (!there_yet) miss[0] = miss[2] = 1;
                for (int i = tid; there_yet && i < 3 * (n_vec + n_vec2); i += 384) {
                    const bool second = i >= 3 * n_vec;
                    const int i2 = second ? i - 3 * n_vec : i;
                    const int prod = i2 / 3, part = i2 - 3 * prod;
                    if (!second) {
                        if (fetch(vec + (long)prod * vec_stride + part, vec_tag, vec_blocks, miss, w))
                            unpack(w, vec_dst, prod, part);
                        else
                            miss[0] = 1;
                    } else {
                        if (fetch(vec2 + (long)prod * kRnntEntryWords + part, vec2_tag, false, miss, w))
                            unpack(w, vec2_dst, prod, part);
                        else
                            miss[2] = 1;
                    }
                }
            }
        } else if (!row_per_step || look == 0) {
            // A lane's words: the one of its place in a row of 16 lanes (of step + row), or those of its place in the wavefront (of
            // step + look).  Addresses and tags in front of the polls: every instruction of them counts.
            constexpr bool kRow = row_per_step;
            constexpr int kN = kRow ? 1 : LANE_WORDS;
            const int st = step + (kRow ? lane >> 4 : look);
            const unsigned int tag = step_tag(st, g_version());
            const bool blocks = step_blocks && look == 0;
            const u64* slot[kN];
            int prod[kN], part[kN];
            bool has[kN];
            u64 v[kN];
#pragma unroll
            for (int n = 0; n < kN; ++n) {
                const int i = kRow ? (lane & 15) : lane + 64 * n;
                has[n] = i < 3 * nwv;
                prod[n] = has[n] ? i / 3 : 0;   // (a lane without a word looks at the first one)
                part[n] = has[n] ? i - 3 * prod[n] : 0;
                slot[n] = lg_entry(st, prod[n]) + part[n];
            }
            unsigned int spins = 0;
            unsigned long long first = 0ull;
            bool there;
            while (true) {
                there = true;
#pragma unroll
                for (int n = 0; n < kN; ++n) v[n] = __hip_atomic_load(slot[n], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int n = 0; n < kN; ++n) there = there && (unsigned int)(v[n] >> 48) == tag;
                if (!blocks || __all(there || (kRow && lane >= 16))) break;
                bool give_up = false;
                if (spins > 0u && (spins & 255u) == 0u) {
                    if (__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) give_up = true;
                    if (wait_clock_expired(spins, first)) spins = 0xffffffffu;
                }
                if (spins >= p.spin_limit) {
                    __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    give_up = true;
                }
                if (__any(give_up)) {
                    miss[1] = 1;
                    someone_gave_up = 1;
                    break;
                }
                if (spins != 0xffffffffu) ++spins;
            }
            unsigned int key = 0u;
#pragma unroll
            for (int n = 0; n < kN; ++n) key = max(key, rnnt_word_key(v[n], prod[n], part[n]));
            if (kRow) {
                const unsigned long long m = __ballot(there);
                const bool whole = ((m >> (lane & 48)) & 0xffffull) == 0xffffull;
                key = rnnt_max_row(key);
                if ((lane & 15) == 0) keys[n_pass & 1u][lane >> 4] = whole ? key : 0u;
            } else {
                key = rnnt_max_u32(key);
                if (!__all(there)) key = 0u;
                if (lane == 0) keys[n_pass & 1u][look] = key;
            }
        }
        rnnt_barrier();
        int r = (n_vec > 0 && miss[0] == 0) ? 1 : 0;
        if (n_vec2 > 0 && miss[2] == 0) r |= 2;
        n_there = 0;
        if (look_waves) {
            const int looked = row_per_step ? kRnntGreedyRows : look_waves;
            my_key = keys[n_pass & 1u][lane & (kRnntGreedyLook - 1)];
            const unsigned int there = (unsigned int)__ballot(my_key != 0u) & ((1u << looked) - 1u);
            n_there = __builtin_ctz(~there);
        }
        if (miss[1] != 0) dead = true;
        // the flags of the pass after the next are cleared now: their last readers passed this barrier, their next
        // writers come after the next one
        if (tid < 3) missing[(n_pass + 2u) % 3u][tid] = 0;
        ++n_pass;
        return r;
    };
    // After a pass that brought nothing: counts, and gives up when the limits are reached.  Everybody learns of it behind the
    // next pass's barrier, through that pass's flags (a word that thread 0 wrote now could be read by some threads of this
    // round and not by others).
    auto nothing_came = [&]() __attribute__((always_inline)) {
        if (tid == 0) {
            bool give_up = false;
            if (waited > 0u && (waited & 255u) == 0u) {
                if (__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) give_up = true;
                if (wait_clock_expired(waited, t_first)) waited = 0xffffffffu;
            }
            if (waited >= p.spin_limit) {
                __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                give_up = true;
            }
            if (give_up) {
                someone_gave_up = 1;
                missing[n_pass % 3u][1] = 1;
            }
            if (waited != 0xffffffffu) ++waited;
        }
    };
    auto something_came = [&]() __attribute__((always_inline)) {
        if (tid == 0) waited = 0u;
    };
    // Takes the decisions whose logits a pass found, in order, up to and including the first that emits a symbol (what lies
    // behind it was computed for a g that is no longer the current one); a run of blanks in one go.  Returns how many.
    auto take_decisions = [&]() __attribute__((always_inline)) {
        if (n_there == 0) return 0;
        const unsigned int blanks = (unsigned int)__ballot(rnnt_key_index(my_key) == p.blank) & ((1u << kRnntGreedyLook) - 1u);
        int taken = min(min(n_there, __builtin_ctz(~blanks)), p.T - s.t);
        if (taken > 0) {
            n_pred += s.run_pred;
            s.run_pred = 0;
            s.frame_syms = 0;
            s.t += taken;
            step += taken;
        }
        if (taken < n_there && s.t < p.T) {
            const int k = rnnt_key_index(__builtin_amdgcn_readlane(my_key, taken));
            const int at = s.emitted;
            n_pred += s.run_pred;
            ++step;
            ++taken;
            rnnt_greedy_advance(s, k, p.blank, p.max_per_frame);
            if (b == 0 && tid == 0) p.symbols[at] = k;
        }
        if (tid == 384) __hip_atomic_store(p.seen + (long)kRnntSeenStride * b, (unsigned int)step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return taken;
    };
    // Waits for a vector.  Returns false when the block has to leave the loop.
    auto wait_for_vector = [&](const u64* vec, int n_vec, unsigned int tag, half_t* dst, int stride = kRnntEntryWords) __attribute__((always_inline)) {
        pass(vec, n_vec, tag, dst, true, 0, false, stride);
        return !dead;
    };
    // ---- the decision behind a symbol, by every block of a layer or of the joint network for itself ----
    // The first decision under a new g is waited for by everybody and nothing else is there yet, so those blocks do not wait for the
    // symbol blocks' round and the logits' way (1.9 us): they read the hidden vector too, multiply it by W2 (rows wave,
    // wave + 8, .. in each wavefront's registers) and take the argmax, 1.1 us from the vector's arrival.  The sums are in rnnt_sum's order:
    // the symbol blocks' logits have the same bits.  The steps ahead come from the symbol blocks: eight steps' logits by every block
    // would take it 1.9 us a round.
    constexpr int kSets = OWN_ROWS ? OWN_ROWS / 4 : 1;          // of four rows
    constexpr int kOwnPieces = OWN_ROWS ? OWN_PIECES : 1;
    half8_t w2[4 * kSets][kOwnPieces];
    float own_bias = 0.0f;
    // Rows of 16 lanes take the sets in turn, the lanes of a quad the rows of a set.
    const int own_row = kRnntWaves * (4 * ((lane >> 4) & (kSets - 1)) + (lane & 3)) + wave;
    auto ask_for_w2 = [&]() __attribute__((always_inline)) {
        if constexpr (OWN_ROWS > 0) {
#pragma unroll
            for (int q = 0; q < OWN_ROWS; ++q) {
                const half8_t* row = reinterpret_cast<const half8_t*>(p.w2 + (long)min(kRnntWaves * q + wave, p.V - 1) * p.J);
#pragma unroll
                for (int k = 0; k < kOwnPieces; ++k) w2[q][k] = row[min(lane + 64 * k, nwj - 1)];
            }
            own_bias = p.b2 ? (float)p.b2[min(own_row, p.V - 1)] : 0.0f;
        }
    };
    // (The joint blocks do not use its entry again before every block has counted that decision: `seen`.)
    auto decided_alone = [&]() __attribute__((always_inline)) {
        if constexpr (OWN_ROWS > 0) {
            pass(hid_entry(step, 0), nwj, step_tag(step, g_version()), buf0, true, 0, false);
            if (dead) return false;
            const half8_t* in = reinterpret_cast<const half8_t*>(buf0);
            float x[4];
#pragma unroll
            for (int set = 0; set < kSets; ++set) {
                float a[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    a[q] = 0.0f;
#pragma unroll
                    for (int k = 0; k < kOwnPieces; ++k)
                        if (lane + 64 * k < nwj) a[q] = dot8(w2[4 * set + q][k], in[lane + 64 * k], a[q]);
                }
                x[set] = rnnt_fold4(a, lane);
            }
            static_assert(kSets <= 2, "up to 64 symbols");
            const float pair = rnnt_join16(x[0], x[kSets - 1]);
            const float sum = rnnt_join32(pair, pair);
            unsigned int key = rnnt_key(own_row < p.V ? rnnt_bits(sum + own_bias) : (unsigned short)0xfc00u, own_row);   // (-inf past the last symbol)
            key = max(key, rnnt_dpp_u32<kDppQuadXor1>(key));
            key = max(key, rnnt_dpp_u32<kDppQuadXor2>(key));
            // (a row of 16 lanes has its sums in lanes 0 .. 3)
            if ((lane & 15) == 0 && lane < 16 * kSets) own_keys[wave + kRnntWaves * (lane >> 4)] = key;
            rnnt_barrier();
            my_key = rnnt_max_u32(own_keys[lane & (kRnntWaves * kSets - 1)]);
            n_there = 1;
            take_decisions();
            return true;
        } else {
            return false;
        }
    };
    // Waits until the decision of `step` can be taken, and takes those behind it too if their logits are there already.
    // Returns false when the block has to leave the loop.
    auto wait_for_decisions = [&]() __attribute__((always_inline)) {
        if (OWN_ROWS > 0 && s.run_pred) return decided_alone();
        pass(nullptr, 0, 0u, nullptr, false, kRnntWaves, true);
        if (dead) return false;
        take_decisions();
        return true;
    };

    const int every_words = rnnt_every_words(p.V);
    auto every_entry = [&](int version, int block) __attribute__((always_inline)) { return p.every + ((long)(version & (kRnntGreedyVersions - 1)) * nwh + block) * every_words; };
    // Waits for the first layer's h of a version whose symbol has been decided.  With EVERY it was published for all symbols before the
    // decision (but for a first run with x0): the words of that symbol are picked out.
    auto wait_for_first_layer = [&](int version, half_t* dst) __attribute__((always_inline)) {
        if (EVERY && s.label >= 0) return wait_for_vector(every_entry(version, 0) + 3 * s.label, nwh, h_tag(version), dst, every_words);
        return wait_for_vector(h_entry(version, 0), nwh, h_tag(version), dst);
    };

    if (someone_gave_up == 0 && b < n_lstm) {
        // ---- a layer of the prediction network: unit u, gate rows u, H + u, 2H + u, 3H + u ----
        const int l = b / nwh, u = 8 * (b % nwh) + wave;
        const RnntLayer ly = p.layer[l];
        const int nxp = ly.in_w >> 3;
        half8_t whh[4][kRnntHC], wih[4][kRnntXC];
#pragma unroll
        for (int gt = 0; gt < 4; ++gt) {
            const half8_t* row = reinterpret_cast<const half8_t*>(ly.w_hh + ((long)gt * H + u) * H);
#pragma unroll
            for (int k = 0; k < kRnntHC; ++k) {
                if (64 * k >= nhp) break;
                whh[gt][k] = row[min(lane + 64 * k, nhp - 1)];
            }
        }
#pragma unroll
        for (int gt = 0; gt < 4; ++gt) {
            const half8_t* row = reinterpret_cast<const half8_t*>(ly.w_ih + ((long)gt * H + u) * ly.in_w);
#pragma unroll
            for (int k = 0; k < kRnntXC; ++k) {
                if (64 * k >= nxp) break;
                wih[gt][k] = row[min(lane + 64 * k, nxp - 1)];
            }
        }
        ask_for_w2();
        const float bias = ly.bsum ? ly.bsum[(long)(lane & 3) * H + u] : 0.0f;
        half_t c_half = p.c0 ? p.c0[(long)l * H + u] : (half_t)0.0f;
        half_t h_last = p.h0 ? p.h0[(long)l * H + u] : (half_t)0.0f;
        for (int i = tid; i < H; i += kRnntThreads) own[i] = p.h0 ? p.h0[(long)l * H + i] : (half_t)0.0f;
        if (l == 0 && p.emb_in_lds) {
            // the rows the first layer will be asked for: embedding[0 .. emb_rows) and, behind them, x0
            const half8_t* e8 = reinterpret_cast<const half8_t*>(p.embedding);
            half8_t* d8 = reinterpret_cast<half8_t*>(emb);
            const int n8 = p.emb_rows * nxp;
            for (int i = tid; i < n8; i += kRnntThreads) d8[i] = e8[i];
            const half8_t* x8 = reinterpret_cast<const half8_t*>(p.x0);
            if (x8)  // (null when the first step does not run the prediction network: never asked for then)
                for (int i = tid; i < nxp; i += kRnntThreads) d8[n8 + i] = x8[i];
        }
        __syncthreads();
        // W_hh . h of the layer and the bias, summed as soon as h is known
        float hidden = 0.0f;
        auto sum_hh = [&](const half_t* h) __attribute__((always_inline)) {
            const half8_t* hv = reinterpret_cast<const half8_t*>(h);
            float a_hh[4];
#pragma unroll
            for (int gt = 0; gt < 4; ++gt) {
                a_hh[gt] = 0.0f;
#pragma unroll
                for (int k = 0; k < kRnntHC; ++k)
                    if (lane + 64 * k < nhp) a_hh[gt] = dot8(whh[gt][k], hv[lane + 64 * k], a_hh[gt]);
            }
            hidden = rnnt_gate_sum(a_hh, lane) + bias;
        };
        auto sum_ih = [&](const half8_t* in, float (&a)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int gt = 0; gt < 4; ++gt) {
                a[gt] = 0.0f;
#pragma unroll
                for (int k = 0; k < kRnntXC; ++k)
                    if (lane + 64 * k < nxp) a[gt] = dot8(wih[gt][k], in[lane + 64 * k], a[gt]);
            }
        };
        // The first layer ahead of the decision: W_ih . embedding[k] once for every symbol (four symbols to a fold), then, whenever h is
        // known, this block's units of the next h after every symbol, a symbol or two to a lane.
        constexpr int kEach = EVERY ? kRnntGreedyEveryVocab / 64 : 1;
        half_t c_every[kEach];
        unsigned short h_every[kEach];
        auto sum_every_rows = [&](auto pieces, auto how_many) __attribute__((always_inline)) {
            constexpr int kP = decltype(pieces)::value, kRows = decltype(how_many)::value;   // rows asked for together: the trips to them are most of this
            const half8_t* rows = p.emb_in_lds ? reinterpret_cast<const half8_t*>(emb) : reinterpret_cast<const half8_t*>(p.embedding);
#pragma unroll 1
            for (int k0 = 0; k0 < p.V; k0 += kRows) {
                half8_t in[kRows][kP];
#pragma unroll
                for (int q = 0; q < kRows; ++q) {
                    const half8_t* row = rows + (long)min(k0 + q, p.V - 1) * nxp;
#pragma unroll
                    for (int k = 0; k < kP; ++k) in[q][k] = row[min(lane + 64 * k, nxp - 1)];
                }
                float x[kRows];
#pragma unroll
                for (int q = 0; q < kRows; ++q) {
                    float a[4];
#pragma unroll
                    for (int gt = 0; gt < 4; ++gt) {
                        a[gt] = 0.0f;
#pragma unroll
                        for (int k = 0; k < kP; ++k)
                            if (lane + 64 * k < nxp) a[gt] = dot8(wih[gt][k], in[q][k], a[gt]);
                    }
                    x[q] = rnnt_fold4(a, lane);
                }
#pragma unroll
                for (int q = 0; q < kRows; q += 4) {
                    const float sum = rnnt_join32(rnnt_join16(x[q], x[q + 1]), rnnt_join16(x[q + 2], x[q + 3]));
                    if ((lane & 12) == 0) reinterpret_cast<float*>(&ih_of[wave][k0 + q + (lane >> 4)])[lane & 3] = sum;
                }
            }
        };
        auto sum_every_ih = [&]() __attribute__((always_inline)) {
            static_assert(kRnntXC == 2, "rows of one piece to a lane or of two");
            if (nxp <= 64) sum_every_rows(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{});
            else sum_every_rows(std::integral_constant<int, 2>{}, std::integral_constant<int, 4>{});
        };
        static_assert(kRnntGreedyEveryVocab % 8 == 0, "eight symbols a round");
        auto publish_every = [&](int version) __attribute__((always_inline)) {
            float hidden_of[4];
#pragma unroll
            for (int gt = 0; gt < 4; ++gt) hidden_of[gt] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, hidden), gt));
            const float c_prev = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)c_half)));
#pragma unroll
            for (int n = 0; n < kEach; ++n) {
                if (64 * n >= p.V) break;
                const float4_t ih = ih_of[wave][min(lane + 64 * n, p.V - 1)];
                float act[4];   // as rnnt_unit does it
#pragma unroll
                for (int gt = 0; gt < 4; ++gt) {
                    const float a = ih[gt] + hidden_of[gt];
                    const float sg = fast_sigmoid_f32(gt == 2 ? 2.0f * a : a);
                    act[gt] = gt == 2 ? 2.0f * sg - 1.0f : sg;
                }
                const float c_new = __builtin_fmaf(act[1], c_prev, act[0] * act[2]);
                const half_t h_new = rnnt_round(act[3] * (2.0f * fast_sigmoid_f32(2.0f * c_new) - 1.0f));
                c_every[n] = rnnt_round(c_new);
                h_every[n] = rnnt_bits((float)h_new);
                if (lane + 64 * n < p.V) every_mine[lane + 64 * n][wave] = h_every[n];
            }
            rnnt_barrier();
            if (tid < 3 * p.V) {
                const int k = tid / 3, part = tid - 3 * k;
                const unsigned short* m = every_mine[k] + 3 * part;
                const u64 w = (u64)m[0] | ((u64)m[1] << 16) | ((u64)m[2] << 32) | ((u64)h_tag(version) << 48);
                __hip_atomic_store(every_entry(version, b) + tid, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        static_assert(3 * kRnntGreedyEveryVocab <= kRnntThreads, "a thread per word");
        sum_hh(own);
        if constexpr (EVERY) {
            if (l == 0 && !s.run_pred) {  // (a first step with x0 stands in front of the first decision otherwise)
                sum_every_ih();
                publish_every(0);
            }
        }
        bool ok = true;
        while (ok && running()) {
            if (EVERY && l == 0 && s.run_pred && s.label >= 0) {
                // this version's h is one of those made ahead
                const int version = n_pred;
                const int from = s.label & 63;
                unsigned int c_bits = (unsigned int)__builtin_amdgcn_readlane((int)__builtin_bit_cast(unsigned short, c_every[0]), from);
                unsigned int h_bits = (unsigned int)__builtin_amdgcn_readlane((int)h_every[0], from);
                if constexpr (kEach > 1) {
                    if (s.label >= 64) {
                        c_bits = (unsigned int)__builtin_amdgcn_readlane((int)__builtin_bit_cast(unsigned short, c_every[kEach - 1]), from);
                        h_bits = (unsigned int)__builtin_amdgcn_readlane((int)h_every[kEach - 1], from);
                    }
                }
                c_half = __builtin_bit_cast(half_t, (unsigned short)c_bits);
                h_last = __builtin_bit_cast(half_t, (unsigned short)h_bits);
                if (!wait_for_first_layer(version, own)) {
                    ok = false;
                    break;
                }
                sum_hh(own);
                publish_every(version + 1);
            } else if (s.run_pred) {
                const int version = n_pred;
                const half8_t* in;
                if (l == 0) {
                    const int row = s.label < 0 ? p.emb_rows : s.label;
                    in = p.emb_in_lds ? reinterpret_cast<const half8_t*>(emb) + (long)row * nxp
                                      : reinterpret_cast<const half8_t*>(s.label < 0 ? p.x0 : p.embedding + (long)s.label * ly.in_w);
                } else {
                    if (!(l == 1 ? wait_for_first_layer(version, buf0) : wait_for_vector(h_entry(version, (l - 1) * nwh), nwh, h_tag(version), buf0))) {
                        ok = false;
                        break;
                    }
                    in = reinterpret_cast<const half8_t*>(buf0);
                }
                float a[4];
                sum_ih(in, a);
                float c_new;
                half_t h_new;
                rnnt_unit(rnnt_gate_sum(a, lane) + hidden, (float)c_half, lane, c_new, h_new);
                c_half = rnnt_round(c_new);
                const unsigned short bits = rnnt_bits((float)h_new);
                h_last = __builtin_bit_cast(half_t, bits);
                if (lane == 0) my_value(0) = bits;
                rnnt_barrier();
                if (wave == 6) store_words(0, h_entry(version, b), h_tag(version));
                ++n_publish;
                // h of this layer, for W_hh at the next symbol
                if (!wait_for_vector(h_entry(version, l * nwh), nwh, h_tag(version), own)) {
                    ok = false;
                    break;
                }
                sum_hh(own);
                if constexpr (EVERY) {
                    if (l == 0) {  // (the first run, with x0)
                        sum_every_ih();
                        publish_every(version + 1);
                    }
                }
            }
            ok = wait_for_decisions();
        }
        if (ok && lane == 0) {
            if (p.hn) p.hn[(long)l * H + u] = h_last;
            if (p.cn) p.cn[(long)l * H + u] = c_half;
        }
    } else if (someone_gave_up == 0 && b < n_lstm + nwj) {
        // ---- the joint network's first layer: rows 8 jb .. + 7 of W1 over cat(f, g), for the current step and the steps behind it should
        // they all be blanks.  The sums over f and over g are made apart: the frames' sums are made ahead, eight a round, and kept, and g's
        // once per version, so that a step's eight values are a sum of two each and all steps' words leave in one store ----
        const int jb = b - n_lstm;
        const int nfp = p.F >> 3;
        const half8_t* rows = reinterpret_cast<const half8_t*>(p.w1 + (long)8 * jb * (p.F + H));
        const long row_step = (long)(nfp + nhp);
        // Frames of up to two pieces a lane (1024 wide): a wavefront takes a frame, with all eight rows in registers (every wavefront
        // reading every frame for a row of its own is 128 KB a round through the CU's 64 bytes a clock).  Longer ones: a row each, and so
        // where there are no more frames than such a round asks for, and the eight rows to a wavefront would be the 128 KB (us a call of
        // 1 / 2 / 3 frames, two layers of 320, 29 symbols, no first run, a frame / a row each: 13.4 / 12.4, 14.0 / 13.8, 14.1 / 13.5; at six 15.1 / 16.0).
        constexpr int kShort = 2, kLongAsk = 4;
        const bool short_frames = nfp <= 64 * kShort && p.T > kLongAsk;
        // One array for both kinds: eight short rows and a short frame's pieces behind them, or a long row and four long frames'.
        constexpr int kColShort = 8 * kShort, kColLong = kRnntFC, kRegs = (1 + kLongAsk) * kRnntFC;
        static_assert(kColShort + kShort <= kRegs, "both fit");
        half8_t reg[kRegs], wg[kRnntHC];
        if (short_frames) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
#pragma unroll
                for (int k = 0; k < kShort; ++k) reg[r * kShort + k] = rows[r * row_step + min(lane + 64 * k, nfp - 1)];
            }
        } else {
#pragma unroll
            for (int k = 0; k < kRnntFC; ++k) {
                if (64 * k >= nfp) break;
                reg[k] = rows[wave * row_step + min(lane + 64 * k, nfp - 1)];
            }
        }
#pragma unroll
        for (int k = 0; k < kRnntHC; ++k) {
            if (64 * k >= nhp) break;
            wg[k] = rows[wave * row_step + nfp + min(lane + 64 * k, nhp - 1)];
        }
        ask_for_w2();
        const float bias = p.b1 ? (float)p.b1[8 * jb + wave] : 0.0f;
        float* const over_f = reinterpret_cast<float*>(emb);           // [kRnntGreedyFrames][8]: sums over frames f_lo .. af_hi (where the first layer's blocks have the embedding rows)
        float* const over_g = over_f + kRnntGreedyFrames * 8;          // [8]: over g, with the bias
        int af_hi = 0, af_seen = 0;                                    // frames summed so far; those whose sums every wavefront sees
        // The next frames are asked for in front of a wait and summed behind it (their columns travel while the symbol blocks work).
        int n_ask = 0;
        auto ask = [&]() __attribute__((always_inline)) {
            n_ask = max(0, min(min(short_frames ? kRnntWaves : kLongAsk, p.T - af_hi), s.t + kRnntGreedyFramesAhead - af_hi));
            if (n_ask == 0) return;
            if (short_frames) {
                const half8_t* f8 = reinterpret_cast<const half8_t*>(p.enc + (long)(af_hi + min(wave, n_ask - 1)) * p.F);
#pragma unroll
                for (int k = 0; k < kShort; ++k) reg[kColShort + k] = f8[min(lane + 64 * k, nfp - 1)];   // (a lane past the frame's end keeps nothing of it)
            } else {
#pragma unroll
                for (int q = 0; q < kLongAsk; ++q) {
                    if (q >= n_ask) break;
                    const half8_t* f8 = reinterpret_cast<const half8_t*>(p.enc + (long)(af_hi + q) * p.F);
#pragma unroll
                    for (int k = 0; k < kRnntFC; ++k) {
                        if (64 * k >= nfp) break;
                        reg[kColLong + q * kRnntFC + k] = f8[min(lane + 64 * k, nfp - 1)];
                    }
                }
            }
        };
        auto keep = [&]() __attribute__((always_inline)) {
            if (n_ask == 0) return;
            float lo[4], hi[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (short_frames) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    lo[r] = hi[r] = 0.0f;
#pragma unroll
                    for (int k = 0; k < kShort; ++k)
                        if (lane + 64 * k < nfp) {
                            lo[r] = dot8(reg[r * kShort + k], reg[kColShort + k], lo[r]);
                            hi[r] = dot8(reg[(r + 4) * kShort + k], reg[kColShort + k], hi[r]);
                        }
                }
            } else {
#pragma unroll
                for (int q = 0; q < kLongAsk; ++q) {
                    lo[q] = 0.0f;
                    if (q >= n_ask) continue;
#pragma unroll
                    for (int k = 0; k < kRnntFC; ++k)
                        if (lane + 64 * k < nfp) lo[q] = dot8(reg[k], reg[kColLong + q * kRnntFC + k], lo[q]);
                }
            }
            // lane 16 i + j, j < 4, of the first 32: the sum of lo[j], or of hi[j]
            const float both = rnnt_join16(rnnt_fold4(lo, lane), rnnt_fold4(hi, lane));
            const float sum = rnnt_join32(both, both);
            const int i = 4 * (lane >> 4) + (lane & 3);
            if ((lane & 12) == 0 && lane < 32) {
                if (short_frames) {
                    if (wave < n_ask) over_f[((af_hi + wave) & (kRnntGreedyFrames - 1)) * 8 + i] = sum;
                } else {
                    if (i < n_ask) over_f[((af_hi + i) & (kRnntGreedyFrames - 1)) * 8 + wave] = sum;
                }
            }
            af_hi += n_ask;
            n_ask = 0;
        };
        ask();                    // (the first frames travel with the weights)
        for (int i = tid; i < H; i += kRnntThreads) own[i] = p.h0 ? p.h0[(long)(p.L - 1) * H + i] : (half_t)0.0f;  // g before the first run
        __syncthreads();
        keep();
        int have_g = -1;          // the version of g whose sums are in over_g
        int pub = 0;              // the next step to publish a hidden vector for
        // (barriers between the sums' writers and their readers: this one, and those of the waits)
        auto sum_g = [&]() __attribute__((always_inline)) {
            const half8_t* gv = reinterpret_cast<const half8_t*>(own);
            float a = 0.0f;
#pragma unroll
            for (int k = 0; k < kRnntHC; ++k)
                if (lane + 64 * k < nhp) a = dot8(wg[k], gv[lane + 64 * k], a);
            a = rnnt_sum(a);
            if (lane == 0) over_g[wave] = a + bias;
            rnnt_barrier();
            af_seen = af_hi;
        };
        sum_g();
        // With decisions that the symbol blocks have no part in (a run of symbols), nothing else keeps the joint blocks from running a ring
        // ahead of them or of a layer's block: they look at everybody's count until the entry of `step` may be used again.  What the
        // slowest block needs is there, so the wait ends.
        int min_seen = 0;         // no block has taken in fewer decisions than this
        int seen_stage = 0, seen_slot = 0, seen_here = 0x7fffffff;
        auto wait_for_the_slowest = [&]() __attribute__((always_inline)) {
            unsigned int spins = 0;
            unsigned long long first = 0ull;
            do {
                int* miss = missing[n_pass % 3u];
                if (tid == 0) min_seen_lds = 0x7fffffff;
                rnnt_barrier();
                if (tid < nb)
                    atomicMin(&min_seen_lds, (int)__hip_atomic_load(p.seen + (long)kRnntSeenStride * tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                rnnt_barrier();
                min_seen = min_seen_lds;
                if (tid == 0 && step - kRnntGreedyRing >= min_seen) {
                    bool give_up = false;
                    if (spins > 0u && (spins & 255u) == 0u) {
                        if (__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) give_up = true;
                        if (wait_clock_expired(spins, first)) spins = 0xffffffffu;
                    }
                    if (spins >= p.spin_limit) {
                        __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        give_up = true;
                    }
                    if (give_up) {
                        miss[1] = 1;
                        someone_gave_up = 1;
                    }
                    if (spins != 0xffffffffu) ++spins;
                }
                rnnt_barrier();
                if (miss[1] != 0) dead = true;
                if (tid < 3) missing[(n_pass + 2u) % 3u][tid] = 0;
                ++n_pass;
            } while (!dead && step - kRnntGreedyRing >= min_seen);
            return !dead;
        };
        const int word_step = lane / 3, word_part = lane - 3 * word_step;   // a lane's word when all steps are published
        bool ok = true;
        while (ok && running()) {
            const int version = g_version();
            int end = min(step + kRnntGreedyAhead + 1, step + (p.T - s.t));
            while (af_hi < s.t + (end - step)) {  // (the first frames, and what was not asked for in time)
                ask();
                keep();
            }
            if (version != have_g) {
                if (!(p.L == 1 ? wait_for_first_layer(version, own) : wait_for_vector(h_entry(version, (p.L - 1) * nwh), nwh, h_tag(version), own))) {
                    ok = false;
                    break;
                }
                sum_g();
                have_g = version;
                pub = step;
            }
            if (pub < step) pub = step;
            if (OWN_ROWS > 0 && end - 1 - kRnntGreedyRing >= min_seen) {
                if (!wait_for_the_slowest()) {
                    ok = false;
                    break;
                }
                end = min(end, min_seen + kRnntGreedyRing);
            }
            // the current step and up to kRnntGreedyAhead behind it
            if (af_seen < s.t + (end - step)) {
                rnnt_barrier();
                af_seen = af_hi;
            }
            if (wave == 6 && pub < end) {
                auto store = [&]() __attribute__((always_inline)) {
                    const float* f = over_f + ((s.t + (pub + word_step - step)) & (kRnntGreedyFrames - 1)) * 8 + 3 * word_part;
                    const float* g = over_g + 3 * word_part;
                    const u64 w0 = rnnt_bits(relu_f32(f[0] + g[0])), w1 = rnnt_bits(relu_f32(f[1] + g[1])), w2 = word_part < 2 ? rnnt_bits(relu_f32(f[2] + g[2])) : (unsigned short)0;
                    return w0 | (w1 << 16) | (w2 << 32) | ((u64)step_tag(pub + word_step, version) << 48);
                };
                if (lane < 3 * (end - pub)) {
                    const u64 w = store();
                    u64* const entry = hid_entry(pub + word_step, jb) + word_part;
                    if (pub == step && lane < 3) __hip_atomic_store(entry, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (everybody waits for this one)
                    if (pub != step || lane >= 3) __hip_atomic_store(entry, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            pub = max(pub, end);
            // Everybody's count of decisions, asked for when half the ring has been used: it is there two rounds later.
            const bool look_now = OWN_ROWS > 0 && seen_stage == 0 && end - 1 - kRnntGreedyRing / 2 >= min_seen;
            if (look_now) {
                if (tid == 0) seen_lds[seen_slot] = 0x7fffffff;
                if (tid < nb) seen_here = (int)__hip_atomic_load(p.seen + (long)kRnntSeenStride * tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            ask();
            const int summed = af_hi;
            ok = wait_for_decisions();
            af_seen = summed;
            if (seen_stage == 2) {
                min_seen = max(min_seen, seen_lds[seen_slot]);
                seen_slot ^= 1;
                seen_stage = 0;
            } else if (look_now) {
                if (tid < nb) atomicMin(&seen_lds[seen_slot], seen_here);
                seen_stage = 2;
            }
            keep();
        }
    } else if (someone_gave_up == 0) {
        // ---- the joint network's second layer: row v of W2, for every hidden vector that arrives ----
        const int team = (b - n_lstm - nwj) / nwv, vb = (b - n_lstm - nwj) - team * nwv, v = 8 * vb + wave;
        const int njp = p.J >> 3;
        const half8_t* row = reinterpret_cast<const half8_t*>(p.w2 + (long)min(v, p.V - 1) * p.J);
        half8_t wv[kRnntJC];
#pragma unroll
        for (int k = 0; k < kRnntJC; ++k) {
            if (64 * k >= njp) break;
            wv[k] = row[min(lane + 64 * k, njp - 1)];
        }
        const float bias = (lane == 0 && p.b2 && v < p.V) ? (float)p.b2[v] : 0.0f;
        auto own_step = [&](int st) __attribute__((always_inline)) { return st + (team + p.teams - st % p.teams) % p.teams; };  // the first of this team's from st on
        int pub = team;           // the next step to publish logits for
        int have_version = g_version();
        int min_seen = 0;         // no block has taken in fewer decisions than this
        bool ok = true;
        while (ok && running()) {
            const int version = g_version();
            if (version != have_version) {
                have_version = version;
                pub = own_step(step);
            }
            if (pub < step) pub = own_step(step);
            const int frame = s.t + (pub - step);
            bool want = frame < p.T && pub <= step + kRnntGreedyAhead;
            if (want && pub - kRnntGreedyLogitRing >= min_seen) {
                // The entry for step `pub` still holds step pub - ring: has everybody taken that decision in?
                if (tid == 0) min_seen_lds = 0x7fffffff;
                rnnt_barrier();
                if (tid < nb)
                    atomicMin(&min_seen_lds, (int)__hip_atomic_load(p.seen + (long)kRnntSeenStride * tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                rnnt_barrier();
                min_seen = min_seen_lds;
                want = pub - kRnntGreedyLogitRing < min_seen;
            }
            // the hidden vector of `step` itself is what everybody waits for (no decision can come before it): polled; one
            // of a later step is looked for once per round, between looks at the decisions
            // and the team's next one is taken along (to the LDS that the first layer's blocks use for the embedding rows)
            const int pub2 = pub + p.teams;
            const bool want2 = want && frame + p.teams < p.T && pub2 <= step + kRnntGreedyAhead && pub2 - kRnntGreedyLogitRing < min_seen;
            const int r = pass(hid_entry(pub, 0), want ? nwj : 0, step_tag(pub, version), buf0, pub == step, kRnntWaves - 6, false, kRnntEntryWords,
                               hid_entry(pub2, 0), want2 ? nwj : 0, step_tag(pub2, version), emb);
            if (dead) {
                ok = false;
                break;
            }
            if (r & 1) {
                const bool two = (r & 2) != 0;
                const half8_t* in0 = reinterpret_cast<const half8_t*>(buf0);
                const half8_t* in1 = reinterpret_cast<const half8_t*>(emb);
                float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
                for (int k = 0; k < kRnntJC; ++k) {
                    if (lane + 64 * k < njp) {
                        a0 = dot8(wv[k], in0[lane + 64 * k], a0);
                        if (two) a1 = dot8(wv[k], in1[lane + 64 * k], a1);
                    }
                }
                a0 = rnnt_sum(a0);
                if (two) a1 = rnnt_sum(a1);
                if (lane == 0) {  // (-inf past the last symbol)
                    my_value(0) = v < p.V ? rnnt_bits(a0 + bias) : (unsigned short)0xfc00u;
                    if (two) my_value(1) = v < p.V ? rnnt_bits(a1 + bias) : (unsigned short)0xfc00u;
                }
                rnnt_barrier();
                const int which = 6 - wave;
                if (which >= 0 && which < (two ? 2 : 1)) store_words(which, lg_entry(pub + which * p.teams, vb), step_tag(pub + which * p.teams, version));
                ++n_publish;
                pub += (two ? 2 : 1) * p.teams;
            }
            const int taken = take_decisions();
            if ((r & 1) || taken > 0)
                something_came();
            else
                nothing_came();
        }
    }

    // ---- the end: the team's result, or one workgroup decodes the utterance by itself ----
    __syncthreads();
    if (someone_gave_up != 0) {
        if (tid == 0) i_decode_alone = (p.alone || atomicCAS(p.solo_owner, 0u, 1u) == 0u) ? 1 : 0;
        __syncthreads();
        if (i_decode_alone) rnnt_greedy_solo(p, solo_hs, solo_cs, buf0, own);
        return;
    }
    if (b == 0 && tid == 0) {
        p.result[0] = s.emitted;
        p.result[1] = s.t;
        p.result[2] = step;
        p.result[3] = 0;
        p.result[4] = s.run_pred;
        p.result[5] = s.label;
    }
}

}  // namespace pimhip
