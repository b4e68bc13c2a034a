// How a decoder step (decoder_step_f16_kernel) reads the rows of its layers: host arithmetic only, so that the rule can be checked
// without a GPU.
#pragma once

#include <stdint.h>

namespace pimhip
{
// A loop of steps reads the same weights every step.  Plain loads leave them in the caches until then as long as they fit;
// non-temporal ones leave the room to the classifier's rows, which are always read with plain loads.  Measured on MI355X, us a step,
// layers' rows non-temporal / plain:
//   mostly classifier, 1024 units, four layers with 72000 / 88000 / 96000 / 104000 / 120000 rows (205, 236, 252, 267, 298 MB of 2^20 bytes):
//     38.4 / 37.5, 42.7 / 42.7, 44.5 / 44.9, 47.2 / 49.2, 51.8 / 56.4; with the context given and 72000 / 88000 / 96000 rows (229, 260, 276 MB):
//     42.2 / 41.3, 46.6 / 47.3, 48.3 / 52.1
//   mostly layers (a wide first one): one layer over 24576 / 32768 / 36864 inputs (200, 264, 296 MB) 34.5 / 30.2, 48.2 / 41.4, 50.4 / 51.7; two
//     over 32768 / 36864 (280, 312 MB) 52.8 / 47.4, 55.0 / 59.9; two over 24576 / 28672 with 32000 rows (278, 310 MB) 49.4 / 45.0, 55.0 / 61.3
static constexpr int64_t kDecKeptBytes = 240ll << 20;         // most of them the classifier's
static constexpr int64_t kDecKeptLayerBytes = 288ll << 20;    // most of them the layers'

// x_w: columns of layer 0's input; ctx_layers: layers that take the context, whose columns are streamed (ctx_streamed) or whose
// products with enc_len encoder outputs are read, fp32, in their place.
inline bool dec_rows_stay(int layers, int64_t H, int64_t x_w, int ctx_layers, bool ctx_streamed, int64_t enc_len, int64_t vocab)
{
    const int64_t columns = layers * H + x_w + (layers - 1) * H;   // of W_hh, and of W_ih without the context's
    const int64_t layer_bytes = 4 * H * (2 * columns + ctx_layers * (ctx_streamed ? 2 * H : 4 * enc_len));
    const int64_t classifier_bytes = 2 * vocab * H;
    return layer_bytes + classifier_bytes <= (layer_bytes >= classifier_bytes ? kDecKeptLayerBytes : kDecKeptBytes);
}
}  // namespace pimhip
