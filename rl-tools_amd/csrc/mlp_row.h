// Internal entry point of the forward kernel that takes a row or a few per workgroup (mlp_row.hip).
#pragma once
#include "common.h"

constexpr int RLT_MLP_ROW_MAX_BATCH = 2048;
// Whether it is the faster way for a network that the sixteen-row tiles take too. Up to four rows per workgroup (1,024 rows) at every width and input; eight only for the
// 256-wide networks of up to 32 inputs, whose weights leave registers for it: evaluate() / forward() of 2,048 rows here against the tiles, 17-256-256-6 14.8 / 16.1 us against
// 15.5 / 16.4, but 17-128-128-6 11.4 / 12.4 against 11.5 / 12.0, 33-256-256-6 16.8 / 18.1 against 16.1 / 17.1, 64-192-192-6 15.8 / 17.4 against 14.1 / 14.9.
inline bool rlt_mlp_row_first(const rlt_rocm_device* device, const rlt_dense_layer* layers, int batch) {
    const int units = device->compute_units > 0 ? device->compute_units : 256;
    return batch <= 4 * units || (layers[0].out_dim == 256 && layers[0].in_dim <= 32);
}
// in -> hid -> hid -> out (in <= 128, hid <= 256 and a multiple of four, out <= 16) in one launch, the weights read as they lie (the second and third layer's 16 bytes
// at a time). keep: the layers' pre_activations / output buffers are written (forward); y (optional when keep is set) receives the last layer's output.
// RLT_E_UNSUPPORTED: the caller takes another path.
int rlt_mlp_row_forward(rlt_rocm_device* device, const rlt_dense_layer* layers, int n_layers, const float* x, int ldx, float* y, int ldy, int batch, bool keep);
