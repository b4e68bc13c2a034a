// Which kernel the greedy decoding loop runs (rnnt_greedy_kernels.h): host arithmetic only.
#pragma once

#include <stdint.h>

namespace pimhip
{
static constexpr int kRnntGreedyRowVocab = 5;      // up to this many symbol blocks to a team (15 words) a step's logits are a row of 16 lanes'
static constexpr int kRnntGreedyEveryVocab = 128;  // symbols that the first layer may run for ahead of the decision

// The kernel for a vocabulary: 0 where a step's words fit a row of 16 lanes, else how many of them a lane of a wavefront takes.
inline int rnnt_greedy_lane_words(int64_t vocab)
{
    const int64_t blocks = (vocab + 7) / 8;
    return blocks <= kRnntGreedyRowVocab ? 0 : (int)((3 * blocks + 63) / 64);
}

// Whether the first layer may run for every symbol ahead of the decision.  It takes the layer's cell and the store's way off a symbol's
// chain (start -> now, us an utterance; 512 joint units, 200 frames unless said): two layers of 320, 29 symbols, 341 frames with 74 and 114
// symbols emitted 739 -> 667 and 996 -> 905; 64 symbols 536 -> 491; 100 symbols 533 -> 491 and, with 34 emitted, 395 -> 387.  With one
// layer the chain is too short for the cells of more than a symbol a lane: 29 symbols 406 -> 377, one layer of 512 and 128
// symbols 458 -> 449 and, with 27 emitted, 316 -> 325.
inline bool rnnt_greedy_every_fits(int64_t vocab, int64_t layers) { return vocab <= (layers == 1 ? 64 : kRnntGreedyEveryVocab); }

// Whether it does in a call of so many frames.  The sums over all embedding rows (and the rows of W2 that every block then holds) are a
// start that the launch does not end before: 2 us of 29 symbols, 6.5 of 64, 13 of 100, 16 of 128, and all of it in front of the first decision
// where a first run with x0 precedes it.  Frames without a symbol hide it only slowly, a symbol emitted wins 1 to 2 us of it back, and how many
// there will be is not known: the line lies where a call that emits none is no slower than one of the kernel without any of this was before its
// steps ahead were doubled.  (us a call, that kernel / without as it is now / with; two layers of 320, 512 joint units, a first decision
// without the prediction network, [symbols emitted].  29 symbols: 1 frame [0] 12.0 / 13.7 / 16.1, 8 [0] 15.9 / 14.9 / 16.3, 12 [0] 19.5 / 17.1 / 18.2 and
// [9] 84.7 / 84.1 / 70.9.  64: 1 [0] 12.1 / 13.7 / 21.3, 16 [0] 22.6 / 21.8 / 23.4, [13] 116 / 115 / 99 and, with a first run, [1] 33.5 / 31.8 / 37.6, 32 [0] 35.2 /
// 29.9 / 32.1 and [29] 227 / 228 / 186.  128: 1 [0] 12.7 / 14.4 / 31.1, 32 [0] 35.6 / 31.0 / 34.2 and [9] 97 / 96 / 94, 64 [0] 61 / 49 / 50 and [16]
// 169 / 161 / 153.)
inline bool rnnt_greedy_every(int64_t vocab, int64_t layers, int64_t frames)
{
    return rnnt_greedy_every_fits(vocab, layers) && frames >= 12 && 2 * frames >= vocab;
}

// Rows of W2 that a wavefront of every block holds, for the decision behind a symbol; 0: that decision waits for the symbol blocks.  (us
// an utterance, without -> with: two layers of 320, 512 joint units, 29 symbols, 341 frames with 74 and 114 symbols emitted 660 -> 618
// and 905 -> 814, 200 frames with 64 symbols 480 -> 462.  One layer 347 -> 354: there the decision is not what the next symbol waits
// for.  640 joint units and 64 symbols, 64 more registers: 449 -> 442 with 47 symbols emitted and 283 -> 292 with 20.)  Where the first layer
// does not run ahead there are none.
inline int rnnt_greedy_own_rows(int64_t vocab, int64_t joint, int64_t layers, int64_t frames)
{
    if (layers < 2 || !rnnt_greedy_every(vocab, layers, frames)) return 0;
    return vocab <= 32 && joint <= 1024 ? 4 : vocab <= 64 && joint <= 512 ? 8 : 0;
}
}  // namespace pimhip
