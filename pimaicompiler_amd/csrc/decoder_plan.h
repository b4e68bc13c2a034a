// How a decoder step (decoder_step_f16_kernel) reads the rows of its layers: host arithmetic only, so that the rule can be checked
// without a GPU.
#pragma once

#include <stdint.h>

namespace pimhip
{
// A loop of steps reads the same weights every step.  Plain loads leave them in the caches until then as long as they fit;
// non-temporal ones leave the room to what is read with plain loads.  Measured on MI355X, us a step; MB are 2^20 bytes.
// All plain as long as all fits the 256 MB Infinity Cache, with the L2s in front of it.  Layers' rows non-temporal / plain, the classifier's
// plain:
//   mostly classifier, 1024 units, four layers with 72000 / 88000 / 96000 / 104000 / 120000 rows (205, 236, 252, 267, 298 MB):
//     38.4 / 37.5, 42.7 / 42.7, 44.5 / 44.9, 47.2 / 49.2, 51.8 / 56.4; with the context given and 72000 / 88000 / 96000 rows (229, 260, 276 MB):
//     42.2 / 41.3, 46.6 / 47.3, 48.3 / 52.1
//   mostly layers (a wide first one): one layer over 24576 / 32768 / 36864 inputs (200, 264, 296 MB) 34.5 / 30.2, 48.2 / 41.4, 50.4 / 51.7; two
//     over 32768 / 36864 (280, 312 MB) 52.8 / 47.4, 55.0 / 59.9; two over 24576 / 28672 with 32000 rows (278, 310 MB) 49.4 / 45.0, 55.0 / 61.3
static constexpr int64_t kDecKeptBytes = 240ll << 20;         // most of them the classifier's
static constexpr int64_t kDecKeptLayerBytes = 288ll << 20;    // most of them the layers'
// Somewhat more than the eight L2s of 4 MB hold, read by a block on every CU, turns them over step by step: the layers or the
// classifier, whichever fits, keeps them to itself.  1024 units, layers + classifier in MB, as a loop of calls: all non-temporal / all plain /
// as chosen:
//   layers non-temporal: 48 + 0 12.4 / 13.0 / 12.4, 64 + 0 17.2 / 17.6 / 17.2 (72 + 0 12.7 / 12.4 with it 12.7), 16 + 31 12.2 / 12.0 / 10.4, 32 + 31 15.5 /
//     16.0 / 14.9, 48 + 16 17.5 / 17.9 / 17.1, 64 + 16 21.6 / 21.8 / 20.4 (72 + 16 19.7 / 18.2 with it 18.3)
//   classifier non-temporal: 16 + 47 13.5 / 14.7 / 13.3, 16 + 62 15.8 / 16.9 / 16.0; 904 units 12 + 41 13.0 / 13.4 / 12.2, 12 + 55 16.7 / 16.5 / 15.9
//   (Neither fits, or all is more: plain is better or as good, 48 + 47 20.5 / 20.8, 48 + 62 22.2 / 21.5, 64 + 62 26.0 / 25.7; steps replayed from a
//   graph are 2 to 5 % slower with plain loads from 32 + 62 to 48 + 62.  Both nearly fit: 32 + 16 14.3 / 12.9, layers non-temporal 13.4.)  Fewer units leave CUs without a block: 640 units 19 + 39 20.6 / 17.9, classifier
//   non-temporal 19.4; 776 18 + 47 17.8 / 15.7 and 16.0.
static constexpr int64_t kDecL2Bytes = 32ll << 20;
static constexpr int64_t kDecNearlyFitLayers = 34ll << 20, kDecNearlyFitClassifier = 24ll << 20;
// From all these bytes, and to these: without a classifier, with one that fits, with layers that fit.
static constexpr int64_t kDecTurnsOverFrom = 40ll << 20, kDecTurnsOverAlone = 68ll << 20, kDecTurnsOverByLayers = 82ll << 20, kDecTurnsOverByClassifier = 80ll << 20;
static constexpr int64_t kDecTurnsOverUnits = 896;

struct DecPlain {
    bool layers, classifier;  // rows read with plain loads
};

// x_w: columns of layer 0's input; ctx_layers: layers that take the context, whose columns are streamed (ctx_streamed) or whose
// products with enc_len encoder outputs are read, fp32, in their place.
inline DecPlain dec_plain_loads(int layers, int64_t H, int64_t x_w, int ctx_layers, bool ctx_streamed, int64_t enc_len, int64_t vocab)
{
    const int64_t columns = layers * H + x_w + (layers - 1) * H;   // of W_hh, and of W_ih without the context's
    const int64_t layer_bytes = 4 * H * (2 * columns + ctx_layers * (ctx_streamed ? 2 * H : 4 * enc_len));
    const int64_t classifier_bytes = 2 * vocab * H, all = layer_bytes + classifier_bytes;
    if (H > kDecTurnsOverUnits && all > kDecTurnsOverFrom && (layer_bytes > kDecNearlyFitLayers || classifier_bytes > kDecNearlyFitClassifier)) {
        if (classifier_bytes <= kDecL2Bytes) {
            if (all <= (vocab ? kDecTurnsOverByLayers : kDecTurnsOverAlone)) return {false, true};
        } else if (layer_bytes <= kDecL2Bytes && all <= kDecTurnsOverByClassifier) {
            return {true, false};
        }
    }
    return {all <= (layer_bytes >= classifier_bytes ? kDecKeptLayerBytes : kDecKeptBytes), true};
}
}  // namespace pimhip
