// Internal entry points of seq_stack.hip: whole passes of the reference's recurrent approximators (dense, two GRU layers, dense) in one launch.
#pragma once
#include "common.h"

// true if the model's shape is the one that these passes take, whatever its buffers: a program may size a workspace before it has them
bool rlt_seq_stack_shape(const rlt_seq_layer* layers, int n);

// true if the model is dense (any activation but the output's, which is the identity) -> GRU -> GRU -> dense with one hidden width of 16 or 32 throughout, at most 16
// inputs and outputs, and a sequence short enough that a batch row's inputs fit the LDS
bool rlt_seq_stack_supported(const rlt_seq_layer* layers, int n, int steps);

// Whether these passes are the faster way for a batch. A workgroup of five or six wavefronts takes one row, and the chip holds 700 to 800 of them at once: a pass takes its
// steps' time for every so many rows, while the launches per layer carry two or four rows per wavefront and project on the matrix cores. Measured, launches per layer / these
// passes, widths 16 and 32, inputs and outputs 4 and 1 or 16 and 16. Forward, or backward to the input: 1,024 rows 1.09 to 2.3 at every length from 1 to 300; 2,048 rows 1.16 to
// 1.7 up to 10 steps, 0.95 to 1.3 at 30, 0.78 to 1.1 at 100; 4,096 rows 0.8 to 1.15 up to 10 steps. Backward with weight gradients (all of them in one launch): 16,384 rows of 1 to 10 steps 1.06
// to 1.3, 3,072 of 100 steps 1.04 to 1.14. A SAC update set, whose passes share launches: 4,800 rows of 3 to 10 steps 1.34 to 1.5, of 30 steps 1.11 to 1.2; 1,600 of 100 steps
// 1.11 to 1.13, 2,400 0.97 to 1.08.
enum rlt_stack_work { RLT_STACK_PASS, RLT_STACK_WEIGHT_GRADIENTS, RLT_STACK_UPDATE };
inline bool rlt_seq_stack_faster(rlt_stack_work work, int steps, int batch) {
    const long long rows = (long long)steps * batch;
    if (work == RLT_STACK_WEIGHT_GRADIENTS) return batch <= 16384 && rows <= 262144;
    if (work == RLT_STACK_UPDATE) return batch <= 4800 && rows <= 163840;
    return batch <= (steps <= 16 ? 2048 : 1024);
}

// forward() of up to three such models in one launch (rlt_rocm_seq_forward for each; `also`: the output is stored there as well)
struct rlt_stack_forward { const rlt_seq_layer* layers; const float* x; int ldx; const uint8_t* reset; int steps, batch; float* also; };
int rlt_seq_stack_forward(rlt_rocm_device* device, const rlt_stack_forward* passes, int n);

// backward() of up to two of them in one launch (rlt_rocm_seq_backward for each), with want_w followed by the weight gradients' two launches for both. overwrite: the
// gradients are stored instead of added on. workspace: rlt_seq_stack_workspace_bytes each; reset as the GRU layers shall see it
struct rlt_stack_backward { const rlt_seq_layer* layers; const float* x; int ldx; const float* d_output; float* d_input; const uint8_t* reset; int steps, batch, want_w, overwrite; void* workspace; };
size_t rlt_seq_stack_workspace_bytes(const rlt_seq_layer* layers, int steps, int batch);
int rlt_seq_stack_backward(rlt_rocm_device* device, const rlt_stack_backward* passes, int n);
