// Weight gradients of three-layer networks in -> h -> h -> out from the activations and pre-activation gradients of a whole batch, and the optimiser's step on them.
#pragma once
#include "common.h"

struct rlt_gradient_net {
    // row-major over the batch: inputs x [ldx], hidden activations h1, h2 [hid], gradients at the pre-activations d1, d2 [hid], d3 [ld3]
    const float *x, *h1, *h2, *d1, *d2, *d3;
    int ldx, ld3, in, hid, out;
    float* gradient[6];          // dW1, db1, dW2, db2, dW3, db3
    // step = 0: the sums are added onto the gradients; step = 1: they are stored there and Adam's step follows, with the soft update of a target where one is named
    int step;
    float *parameter[6], *first_moment[6], *second_moment[6], *target[6];
    uint32_t flags[6];
    rlt_adam_parameters adam; const uint32_t* age;      // the age before the step (advancing it is the caller's: a launch before this one can, and nothing has to be waited for here)
};
// one more optimiser (log_alpha's): a scalar whose gradient is `scale` times the sum of `n` values (n <= 128)
struct rlt_gradient_scalar { const float* values; int n; float scale; rlt_adam_tensor tensor; rlt_adam_parameters adam; const uint32_t* age; };

// What the launch before may have left undone: its kernel gave up waiting (*fault set: the gradients are not those of the batch). Then the sums are stored, but no step is
// taken and the ages, which that launch has advanced, get their values back. age[k]: of the networks' optimisers, then the scalar's; before: the values, in that order.
struct rlt_gradient_guard { const unsigned* fault; uint32_t* age[3]; const uint32_t* before; };

// floats that `partial` needs for these networks (0: none)
size_t rlt_batch_gradients_partial_floats(const rlt_gradient_net* nets, int n_nets, int batch);
// up to two networks on batches of the same size; one launch, or two where the batch is shared out (see batch_gradient.hip)
int rlt_batch_gradients(rlt_rocm_device* device, const rlt_gradient_net* nets, int n_nets, int batch, float polyak, const rlt_gradient_scalar* scalar, float* partial,
                        const rlt_gradient_guard* guard = nullptr);
