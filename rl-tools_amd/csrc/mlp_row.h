// Internal entry point of the forward kernel that takes a row or a few per workgroup (mlp_row.hip).
#pragma once
#include "common.h"

constexpr int RLT_MLP_ROW_MAX_BATCH = 2048;
// in -> hid -> hid -> out (in <= 128, hid <= 256 and a multiple of four, out <= 16) in one launch, the weights read as they lie (the second and third layer's 16 bytes
// at a time). keep: the layers' pre_activations / output buffers are written (forward); y (optional when keep is set) receives the last layer's output.
// RLT_E_UNSUPPORTED: the caller takes another path.
int rlt_mlp_row_forward(rlt_rocm_device* device, const rlt_dense_layer* layers, int n_layers, const float* x, int ldx, float* y, int ldy, int batch, bool keep);
