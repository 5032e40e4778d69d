// Internal entry point of the forward kernel that takes a row or a few per workgroup (mlp_row.hip).
#pragma once
#include "common.h"

constexpr int RLT_MLP_ROW_MAX_BATCH = 2048;
// Whether it is the faster way for a network that the tiles of mlp_wide_kernel take too. Up to four rows per workgroup (1,024 rows) at every width and input (here / there, evaluate(): 17-256-256-6 7.7 / 11.3 us,
// 60-128-128-8 8.2 / 9.2, 64-192-192-6 10.1 / 10.9); eight for the 256-wide networks of up to 32 inputs (2,048 rows 11.2 / 12.6), not for more inputs, whose weights leave no registers for it (33-256-256-6
// 16.1 / 12.8, 60-128-128-8 11.1 / 9.2, 64-192-192-6 13.8 / 11.1). Narrower networks of up to 32 inputs stay on the tiles there, though they would be served here in 7.9 / 8.9 us (17-128-128-6) and 9.9 / 10.7 (17-192-192-6).
inline bool rlt_mlp_row_first(const rlt_rocm_device* device, const rlt_dense_layer* layers, int batch) {
    const int units = device->compute_units > 0 ? device->compute_units : 256;
    return batch <= 4 * units || (layers[0].out_dim == 256 && layers[0].in_dim <= 32);
}
// in -> hid -> hid -> out (in <= 128, hid <= 256 and a multiple of four, out <= 16) in one launch, the weights read as they lie (the second and third layer's 16 bytes
// at a time). keep: the layers' pre_activations / output buffers are written (forward); y (optional when keep is set) receives the last layer's output.
// RLT_E_UNSUPPORTED: the caller takes another path.
int rlt_mlp_row_forward(rlt_rocm_device* device, const rlt_dense_layer* layers, int n_layers, const float* x, int ldx, float* y, int ldy, int batch, bool keep);
