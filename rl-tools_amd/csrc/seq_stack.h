// Internal entry points of seq_stack.hip: whole passes of the reference's recurrent approximators (dense, two GRU layers, dense) in one launch.
#pragma once
#include "common.h"

// true if the model's shape is the one that these passes take, whatever its buffers: a program may size a workspace before it has them
bool rlt_seq_stack_shape(const rlt_seq_layer* layers, int n);

// true if the model is dense (any activation but the output's, which is the identity) -> GRU -> GRU -> dense with one hidden width of 16 or 32 throughout, at most 16
// inputs and outputs, and a sequence short enough that a batch row's inputs fit the LDS
bool rlt_seq_stack_supported(const rlt_seq_layer* layers, int n, int steps);

// forward() of up to three such models in one launch (rlt_rocm_seq_forward for each; `also`: the output is stored there as well)
struct rlt_stack_forward { const rlt_seq_layer* layers; const float* x; int ldx; const uint8_t* reset; int steps, batch; float* also; };
int rlt_seq_stack_forward(rlt_rocm_device* device, const rlt_stack_forward* passes, int n);

// backward() of up to two of them in one launch (rlt_rocm_seq_backward for each), with want_w followed by the weight gradients' two launches for both. overwrite: the
// gradients are stored instead of added on. workspace: rlt_seq_stack_workspace_bytes each; reset as the GRU layers shall see it
struct rlt_stack_backward { const rlt_seq_layer* layers; const float* x; int ldx; const float* d_output; float* d_input; const uint8_t* reset; int steps, batch, want_w, overwrite; void* workspace; };
size_t rlt_seq_stack_workspace_bytes(const rlt_seq_layer* layers, int steps, int batch);
int rlt_seq_stack_backward(rlt_rocm_device* device, const rlt_stack_backward* passes, int n);
