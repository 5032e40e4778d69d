// SAC-specific kernels: tanh-Gaussian head (sample_and_squash) forward/backward, TD target, min-Q gradient routing,
// masks, MSE gradient -- and train_critic / train_actor / update_critic_targets assembled from them.
// reference: nn/layers/sample_and_squash/operations_generic.h:148-398 (CUDA :17-115),
//            rl/algorithms/sac/operations_generic.h:133-527 (CUDA :12-128), nn/loss_functions/mse/operations_generic.h:9-97,
//            random/operations_generic.h:72-105.
#include "seq_stack.h"
#include "optim.h"
#include "common.h"
#include "sac_update.h"
#include "mlp_rows.h"
#include <algorithm>

namespace {

__device__ __forceinline__ float clampf(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }
// log N(value; mean, exp(log_std))
__device__ __forceinline__ float normal_log_prob(float mean, float log_std, float sd, float value) {
    const float neg_log_sqrt_2pi = -0.9189385332046727f;
    float z = (value - mean) / sd;
    return neg_log_sqrt_2pi - log_std - 0.5f * z * z;
}

// one action: sampled, squashed; returns its log-probability
__device__ __forceinline__ float sas_forward_element(const rlt_sas_parameters& p, float mean, float log_std_raw, const float* noise, float& sample, float& action) {
    const float log_std = clampf(log_std_raw, p.log_std_lower_bound, p.log_std_upper_bound), sd = expf(log_std);
    sample = noise ? mean + *noise * sd : mean;
    action = tanhf(sample);
    return normal_log_prob(mean, log_std, sd, sample) - logf(1.0f - action * action + p.log_probability_epsilon);
}
// the gradients at one action's mean and log standard deviation from the gradient at the action; returns the action's log-probability
__device__ __forceinline__ float sas_backward_element(const rlt_sas_parameters& p, float action, float d_action, float eps, float mu, float log_std_raw, float sample,
                                                      float alpha_over_b, float& d_mu, float& d_ls) {
    const float g = d_action * (1.0f - action * action);
    const float log_std = clampf(log_std_raw, p.log_std_lower_bound, p.log_std_upper_bound), sd = expf(log_std);
    const float z = (sample - mu) / sd;
    const float dlp_dmean = z / sd, dlp_dsample = -z / sd, dlp_dlogstd = z * z - 1.0f;
    d_mu = g + alpha_over_b * (dlp_dmean + dlp_dsample + 2.0f * action);
    d_ls = sd * (g * eps) + alpha_over_b * (dlp_dlogstd + dlp_dsample * eps * sd + 2.0f * action * eps * sd);
    if (log_std_raw < p.log_std_lower_bound || log_std_raw > p.log_std_upper_bound) d_ls = 0.0f;
    return normal_log_prob(mu, log_std, sd, sample) - logf(1.0f - action * action + p.log_probability_epsilon);
}

__global__ __launch_bounds__(256) void sas_forward_kernel(rlt_sas_parameters p, const float* __restrict__ input, int ldin, const float* __restrict__ noise, int ldn,
                                                          float* __restrict__ actions, int lda, float* __restrict__ pre_squashing, int ldp,
                                                          float* __restrict__ log_probabilities, int batch, int dim) {
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < batch; r += gridDim.x * blockDim.x) {
        float log_prob = 0.0f;
        for (int c = 0; c < dim; c++) {
            float sample, a;
            log_prob += sas_forward_element(p, input[(size_t)r * ldin + c], input[(size_t)r * ldin + dim + c], noise ? noise + (size_t)r * ldn + c : nullptr, sample, a);
            if (pre_squashing) pre_squashing[(size_t)r * ldp + c] = sample;
            actions[(size_t)r * lda + c] = a;
        }
        log_probabilities[r] = log_prob;
    }
}

// one workgroup of 1024 lanes; d_log_alpha += scale_num / count(reset) * sum_b alpha * (entropy_b - target_entropy)
__global__ __launch_bounds__(1024) void sas_backward_kernel(rlt_sas_parameters p, const float* __restrict__ input, int ldin, const float* __restrict__ noise, int ldn,
                                                            const float* __restrict__ actions, int lda, const float* __restrict__ pre_squashing, int ldp,
                                                            const float* __restrict__ d_output, int lddo, float* __restrict__ d_input, int lddi,
                                                            const float* __restrict__ log_alpha, float* __restrict__ d_log_alpha,
                                                            const uint8_t* __restrict__ reset, int batch, int dim) {
    __shared__ float partial[16];
    __shared__ float partial_n[16];
    const float alpha = expf(*log_alpha);
    const float alpha_over_b = alpha / (float)batch;
    float acc = 0.0f, nreset = 0.0f;
    for (int b = threadIdx.x; b < batch; b += blockDim.x) {
        float entropy = 0.0f;
        for (int a = 0; a < dim; a++) {
            float d_mu, d_ls;
            entropy -= sas_backward_element(p, actions[(size_t)b * lda + a], d_output[(size_t)b * lddo + a], noise[(size_t)b * ldn + a], input[(size_t)b * ldin + a],
                                            input[(size_t)b * ldin + dim + a], pre_squashing[(size_t)b * ldp + a], alpha_over_b, d_mu, d_ls);
            d_input[(size_t)b * lddi + a] = d_mu;
            d_input[(size_t)b * lddi + dim + a] = d_ls;
        }
        acc += alpha * (entropy - p.target_entropy);
        nreset += reset ? (float)(reset[b] != 0) : 1.0f;
    }
    acc = rlt_wave_sum(acc); nreset = rlt_wave_sum(nreset);
    if ((threadIdx.x & 63) == 0) { partial[threadIdx.x >> 6] = acc; partial_n[threadIdx.x >> 6] = nreset; }
    __syncthreads();
    if (threadIdx.x == 0 && d_log_alpha) {
        float s = 0.0f, n = 0.0f;
        for (int i = 0; i < 16; i++) { s += partial[i]; n += partial_n[i]; }
        *d_log_alpha += s / n;
    }
}

__device__ __forceinline__ float target_value(float q1, float q2, float reward, bool terminated, float next_log_prob, float alpha, float gamma) {
    const float min_q = fminf(q1, q2) - alpha * next_log_prob;
    const float future = !terminated ? gamma * min_q : 0.0f;
    return reward + future;
}
__global__ __launch_bounds__(256) void target_q_kernel(const float* __restrict__ q1, const float* __restrict__ q2, const float* __restrict__ rewards,
                                                       const uint8_t* __restrict__ terminated, const float* __restrict__ next_log_probs,
                                                       const float* __restrict__ log_alpha, float gamma, int ignore_termination, float* __restrict__ target, int batch) {
    const float alpha = expf(*log_alpha);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < batch; i += gridDim.x * blockDim.x) {
        target[i] = target_value(q1[i], q2[i], rewards[i], !ignore_termination && terminated[i], next_log_probs[i], alpha, gamma);
    }
}
__global__ __launch_bounds__(256) void min_q_kernel(const float* __restrict__ q1, const float* __restrict__ q2, const float* __restrict__ d1, const float* __restrict__ d2,
                                                    int ld, int cdim, int adim, float* __restrict__ out, int ldo, int batch) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < batch * adim; i += gridDim.x * blockDim.x) {
        int b = i / adim, a = i % adim;
        const float* d = (q1[b] < q2[b]) ? d1 : d2;
        out[(size_t)b * ldo + a] = d[(size_t)b * ld + cdim - adim + a];
    }
}
__global__ __launch_bounds__(256) void mask_copy_kernel(const float* __restrict__ src, int lds, float* __restrict__ dst, int ldt, const uint8_t* __restrict__ mask,
                                                        int invert, int rows, int cols) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * cols; i += gridDim.x * blockDim.x) {
        int r = i / cols, c = i % cols;
        bool m = (mask[r] != 0) != (invert != 0);
        if (m) dst[(size_t)r * ldt + c] = src[(size_t)r * lds + c];
    }
}
__global__ __launch_bounds__(256) void mask_zero_kernel(float* __restrict__ g, int ld, const uint8_t* __restrict__ mask, int invert, int rows, int cols) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * cols; i += gridDim.x * blockDim.x) {
        int r = i / cols, c = i % cols;
        bool m = (mask[r] != 0) != (invert != 0);
        if (m) g[(size_t)r * ld + c] = 0.0f;
    }
}
__global__ __launch_bounds__(256) void mse_gradient_kernel(const float* __restrict__ a, int lda, const float* __restrict__ b, int ldb, float* __restrict__ d, int ldd,
                                                           int rows, int cols, float w, const float* __restrict__ w_dev) {
    const float weight = w_dev ? *w_dev : w;
    const float constant = 2.0f / ((float)rows * (float)cols) * weight;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * cols; i += gridDim.x * blockDim.x) {
        int r = i / cols, c = i % cols;
        d[(size_t)r * ldd + c] = (a[(size_t)r * lda + c] - b[(size_t)r * ldb + c]) * constant;
    }
}
__global__ __launch_bounds__(1024) void mse_evaluate_kernel(const float* __restrict__ a, int lda, const float* __restrict__ b, int ldb, int rows, int cols, float w, float* out) {
    __shared__ float partial[16];
    float acc = 0.0f;
    for (int i = threadIdx.x; i < rows * cols; i += blockDim.x) {
        int r = i / cols, c = i % cols;
        float diff = a[(size_t)r * lda + c] - b[(size_t)r * ldb + c];
        acc += diff * diff;
    }
    acc = rlt_wave_sum(acc);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) { float s = 0.0f; for (int i = 0; i < 16; i++) s += partial[i]; *out = s * w / (float)(rows * cols); }
}
// strided row copy: dst[r][0:cols] = src[r][0:cols]
__global__ __launch_bounds__(256) void copy2d_kernel(const float* __restrict__ src, int lds, float* __restrict__ dst, int ldd, int rows, int cols) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * cols; i += gridDim.x * blockDim.x) {
        int r = i / cols, c = i % cols;
        dst[(size_t)r * ldd + c] = src[(size_t)r * lds + c];
    }
}
// loss_weight handling of train_critic/train_actor in one launch: n = count(mask) (or rows);
//   critic: d[r] = (q[r] - y[r]) * 2/rows * (rows*0.5/n), zeroed where !mask   (sac/operations_generic.h:298-316)
//   actor : d[r] = -1/n, zeroed where !mask                                   (:437-453)
__global__ __launch_bounds__(1024) void sac_d_output_kernel(const float* __restrict__ q, const float* __restrict__ y, const uint8_t* __restrict__ mask,
                                                            float* __restrict__ d, int rows, int actor) {
    __shared__ float partial[16];
    __shared__ float n_final;
    float cnt = 0.0f;
    for (int i = threadIdx.x; i < rows; i += blockDim.x) cnt += mask ? (float)(mask[i] != 0) : 1.0f;
    cnt = rlt_wave_sum(cnt);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) { float s = 0.0f; for (int i = 0; i < 16; i++) s += partial[i]; n_final = s; }
    __syncthreads();
    // scale(loss_weight, s, reciprocal) is (1 / n) * s in the reference (containers/tensor/operations_generic.h:437-443): two roundings when n is no power of two
    const float loss_weight = (1.0f / n_final) * (actor ? -1.0f : (float)rows * 0.5f);
    const float constant = 2.0f / (float)rows * loss_weight;
    for (int i = threadIdx.x; i < rows; i += blockDim.x) {
        bool m = mask ? (mask[i] != 0) : true;
        float v = actor ? loss_weight : (q[i] - y[i]) * constant;
        d[i] = m ? v : 0.0f;
    }
}

// ---- The steps between the passes of a sequence update, over S x B rows of one time step each. What bounds them is the launch (4.5 us each while the values are a few hundred
// kilobytes) and, where a sum over the rows is wanted, that one workgroup cannot ask for them all at once (9 and 15 us at 10,000 rows): each step is one launch of a row
// per thread, and the sums are formed per workgroup (the number of masked rows by every workgroup for itself, the entropy term's partial sums by the last one through).

// rows whose mask is set (all without one), the same in every thread of a workgroup of 256
__device__ __forceinline__ float count_rows(const uint8_t* __restrict__ mask, int rows) {
    if (!mask) return (float)rows;
    __shared__ int partial[4];
    int n = 0, head = (int)((4 - (reinterpret_cast<uintptr_t>(mask) & 3)) & 3);      // bytes before the first whole word
    if (head > rows) head = rows;
    const int words = (rows - head) / 4, tail = head + 4 * words;
    const uint32_t* w = reinterpret_cast<const uint32_t*>(mask + head);
    for (int i0 = threadIdx.x; i0 < words; i0 += 256 * 8) {
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) { const int i = i0 + 256 * u; v[u] = i < words ? w[i] : 0u; }
#pragma unroll
        for (int u = 0; u < 8; u++) n += __popc((((v[u] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | v[u]) & 0x80808080u);
    }
    if ((int)threadIdx.x < head) n += mask[threadIdx.x] != 0;
    if ((int)threadIdx.x < rows - tail) n += mask[tail + threadIdx.x] != 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = n;
    __syncthreads();
    return (float)(partial[0] + partial[1] + partial[2] + partial[3]);
}

// The critics' input rows: observations and, where the row's step is a final one, the policy's action, elsewhere the action taken (sac/operations_generic.h:266-278, 427-431).
// The actor's update also keeps the actions and their samples, and has the gradient at the critics' outputs filled in (:437-453).
struct SequenceActions {
    rlt_sas_parameters sas; const float* policy; const float* noise; const float* base; const uint8_t* final_step;
    float* critic_input; float* log_probabilities; float* actions; float* pre_squashing; float* d_output;      // the last three may be NULL
    int rows, obs, act;
};
__global__ __launch_bounds__(256) void sequence_actions_kernel(SequenceActions A) {
    const int D = A.obs + A.act;
    const float d = A.d_output ? (1.0f / count_rows(A.final_step, A.rows)) * -1.0f : 0.0f;
    for (int r = blockIdx.x * 256 + threadIdx.x; r < A.rows; r += gridDim.x * 256) {
        const bool last = A.final_step[r] != 0;
        const float* base = A.base + (size_t)r * D;
        float* row = A.critic_input + (size_t)r * D;
        float log_probability = 0.0f;
        for (int c = 0; c < A.act; c++) {
            float sample, action;
            const float* policy = A.policy + (size_t)r * 2 * A.act;
            log_probability += sas_forward_element(A.sas, policy[c], policy[A.act + c], A.noise + (size_t)r * A.act + c, sample, action);
            row[A.obs + c] = last ? action : base[A.obs + c];
            if (A.actions) { A.actions[(size_t)r * A.act + c] = action; A.pre_squashing[(size_t)r * A.act + c] = sample; }
        }
        A.log_probabilities[r] = log_probability;
        for (int c = 0; c < A.obs; c++) row[c] = base[c];
        if (A.d_output) A.d_output[r] = last ? d : 0.0f;
    }
}

// the target values and, for one or two critics, the gradient at the output (:144-154, 289-316)
struct SequenceTargets {
    const float* next_q[2]; const float* rewards; const uint8_t* terminated; const float* next_log_probabilities; const float* log_alpha; const uint8_t* final_step;
    const float* q[2]; float* d_output[2]; float* target; float gamma; int rows, count;
};
__global__ __launch_bounds__(256) void sequence_targets_kernel(SequenceTargets A) {
    const float alpha = expf(*A.log_alpha);
    const float constant = 2.0f / (float)A.rows * ((1.0f / count_rows(A.final_step, A.rows)) * ((float)A.rows * 0.5f));
    for (int r = blockIdx.x * 256 + threadIdx.x; r < A.rows; r += gridDim.x * 256) {
        const float target = target_value(A.next_q[0][r], A.next_q[1][r], A.rewards[r], A.terminated[r] != 0, A.next_log_probabilities[r], alpha, A.gamma);
        A.target[r] = target;
        const bool last = A.final_step[r] != 0;
        for (int k = 0; k < A.count; k++) A.d_output[k][r] = last ? (A.q[k][r] - target) * constant : 0.0f;
    }
}

// the gradient at the policy's action from the critic that values it lower (zero where the row's step is not a final one), through the squashed sample to the policy's outputs,
// and d log_alpha (:456-464)
struct SequenceActorGradient {
    rlt_sas_parameters sas; const float* q[2]; const float* d_critic_input[2]; const uint8_t* final_step; const uint8_t* reset;
    const float* policy; const float* noise; const float* actions; const float* pre_squashing; const float* log_alpha;
    float* d_action; float* d_policy; float* d_log_alpha; float* partial; uint32_t* tickets;
    int rows, obs, act;
};
__global__ __launch_bounds__(256) void sequence_actor_gradient_kernel(SequenceActorGradient A) {
    __shared__ float sums[2][4];
    const int D = A.obs + A.act;
    const float alpha = expf(*A.log_alpha), alpha_over_b = alpha / (float)A.rows;
    float acc = 0.0f, resets = 0.0f;
    for (int r = blockIdx.x * 256 + threadIdx.x; r < A.rows; r += gridDim.x * 256) {
        const float* d = (A.q[0][r] < A.q[1][r] ? A.d_critic_input[0] : A.d_critic_input[1]) + (size_t)r * D + A.obs;
        const bool last = A.final_step[r] != 0;
        float entropy = 0.0f;
        for (int c = 0; c < A.act; c++) {
            const size_t i = (size_t)r * A.act + c;
            const float* policy = A.policy + (size_t)r * 2 * A.act;
            const float d_action = last ? d[c] : 0.0f;
            A.d_action[i] = d_action;
            float d_mu, d_ls;
            entropy -= sas_backward_element(A.sas, A.actions[i], d_action, A.noise[i], policy[c], policy[A.act + c], A.pre_squashing[i], alpha_over_b, d_mu, d_ls);
            A.d_policy[(size_t)r * 2 * A.act + c] = d_mu;
            A.d_policy[(size_t)r * 2 * A.act + A.act + c] = d_ls;
        }
        acc += alpha * (entropy - A.sas.target_entropy);
        resets += (float)(A.reset[r] != 0);
    }
    acc = rlt_wave_sum(acc); resets = rlt_wave_sum(resets);
    if ((threadIdx.x & 63) == 0) { sums[0][threadIdx.x >> 6] = acc; sums[1][threadIdx.x >> 6] = resets; }
    __syncthreads();
    if (threadIdx.x < 64) {
        bool last = false;
        if (threadIdx.x == 0) {
            A.partial[2 * blockIdx.x] = (sums[0][0] + sums[0][1]) + (sums[0][2] + sums[0][3]);
            A.partial[2 * blockIdx.x + 1] = (sums[1][0] + sums[1][1]) + (sums[1][2] + sums[1][3]);
            __threadfence();
            last = rlt_last_through(A.tickets, blockIdx.x, gridDim.x);
        }
        if (__any(last)) {      // this workgroup's first wavefront sees what every other one has written
            __threadfence();
            float s = 0.0f, n = 0.0f;
            for (uint32_t b = threadIdx.x; b < gridDim.x; b += 64) { s += ((volatile float*)A.partial)[2 * b]; n += ((volatile float*)A.partial)[2 * b + 1]; }
            s = rlt_wave_sum(s); n = rlt_wave_sum(n);
            if (threadIdx.x == 0) *A.d_log_alpha = s / n;
        }
    }
}
constexpr int MAX_PARTIALS = 448;      // workgroups whose two sums fit the counters block
int sequence_grid(int rows) { const int b = (rows + 255) / 256; return b > MAX_PARTIALS ? MAX_PARTIALS : b; }

int grid1(int n) { int b = (n + 255) / 256; return b > 1024 ? 1024 : (b < 1 ? 1 : b); }

}  // namespace

extern "C" {

int rlt_rocm_mse_gradient(rlt_rocm_device* device, const float* a, int lda, const float* b, int ldb, float* d_a, int ldda, int rows, int cols,
                          float loss_weight, const float* loss_weight_device) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(a && b && d_a && rows > 0 && cols > 0 && lda >= cols && ldb >= cols && ldda >= cols);
    hipLaunchKernelGGL(mse_gradient_kernel, dim3(grid1(rows * cols)), dim3(256), 0, device->stream, a, lda, b, ldb, d_a, ldda, rows, cols, loss_weight, loss_weight_device);
    return rlt_launch_status(device);
}
int rlt_rocm_mse_evaluate(rlt_rocm_device* device, const float* a, int lda, const float* b, int ldb, int rows, int cols, float loss_weight, float* out_loss) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(a && b && out_loss && rows > 0 && cols > 0 && lda >= cols && ldb >= cols);
    hipLaunchKernelGGL(mse_evaluate_kernel, dim3(1), dim3(1024), 0, device->stream, a, lda, b, ldb, rows, cols, loss_weight, out_loss);
    return rlt_launch_status(device);
}
int rlt_rocm_sas_forward(rlt_rocm_device* device, const rlt_sas_parameters* p, const float* input, int ldin, const float* noise, int ldn,
                         float* actions, int lda, float* pre_squashing, int ldp, float* log_probabilities, int batch, int dim) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(p && input && actions && log_probabilities && batch > 0 && dim > 0 && ldin >= 2 * dim && lda >= dim);
    RLT_REQUIRE((!noise || ldn >= dim) && (!pre_squashing || ldp >= dim));
    hipLaunchKernelGGL(sas_forward_kernel, dim3(grid1(batch)), dim3(256), 0, device->stream, *p, input, ldin, noise, ldn, actions, lda, pre_squashing, ldp,
                       log_probabilities, batch, dim);
    return rlt_launch_status(device);
}
static int sas_backward_impl(rlt_rocm_device* device, const rlt_sas_parameters* p, const float* input, int ldin, const float* noise, int ldn,
                             const float* actions, int lda, const float* pre_squashing, int ldp, const float* d_output, int lddo, float* d_input, int lddi,
                             const float* log_alpha, float* d_log_alpha, const uint8_t* reset, int batch, int dim) {
    RLT_REQUIRE(p && input && noise && actions && pre_squashing && d_output && d_input && log_alpha && batch > 0 && dim > 0);
    RLT_REQUIRE(ldin >= 2 * dim && ldn >= dim && lda >= dim && ldp >= dim && lddo >= dim && lddi >= 2 * dim);
    hipLaunchKernelGGL(sas_backward_kernel, dim3(1), dim3(1024), 0, device->stream, *p, input, ldin, noise, ldn, actions, lda, pre_squashing, ldp,
                       d_output, lddo, d_input, lddi, log_alpha, d_log_alpha, reset, batch, dim);
    return rlt_launch_status(device);
}
int rlt_rocm_sas_backward(rlt_rocm_device* device, const rlt_sas_parameters* p, const float* input, int ldin, const float* noise, int ldn,
                          const float* actions, int lda, const float* pre_squashing, int ldp, const float* d_output, int lddo, float* d_input, int lddi,
                          const float* log_alpha, float* d_log_alpha, int batch, int dim) {
    if (!device) return RLT_E_NOT_INITIALISED;
    return sas_backward_impl(device, p, input, ldin, noise, ldn, actions, lda, pre_squashing, ldp, d_output, lddo, d_input, lddi, log_alpha, d_log_alpha, nullptr, batch, dim);
}
int rlt_rocm_sac_target_action_values(rlt_rocm_device* device, const float* q1_next, const float* q2_next, const float* rewards, const uint8_t* terminated,
                                      const float* next_log_probabilities, const float* log_alpha, float gamma, int ignore_termination, float* target, int batch) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(q1_next && q2_next && rewards && terminated && next_log_probabilities && log_alpha && target && batch > 0);
    hipLaunchKernelGGL(target_q_kernel, dim3(grid1(batch)), dim3(256), 0, device->stream, q1_next, q2_next, rewards, terminated, next_log_probabilities, log_alpha,
                       gamma, ignore_termination, target, batch);
    return rlt_launch_status(device);
}
int rlt_rocm_sac_min_value_d_output(rlt_rocm_device* device, const float* q1, const float* q2, const float* d1, const float* d2, int ld, int cdim, int adim,
                                    float* d_actor_output, int ldo, int batch) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(q1 && q2 && d1 && d2 && d_actor_output && batch > 0 && adim > 0 && cdim >= adim && ld >= cdim && ldo >= adim);
    hipLaunchKernelGGL(min_q_kernel, dim3(grid1(batch * adim)), dim3(256), 0, device->stream, q1, q2, d1, d2, ld, cdim, adim, d_actor_output, ldo, batch);
    return rlt_launch_status(device);
}
int rlt_rocm_mask_copy(rlt_rocm_device* device, const float* source, int lds, float* target, int ldt, const uint8_t* mask, int invert, int rows, int cols) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(source && target && mask && rows > 0 && cols > 0 && lds >= cols && ldt >= cols);
    hipLaunchKernelGGL(mask_copy_kernel, dim3(grid1(rows * cols)), dim3(256), 0, device->stream, source, lds, target, ldt, mask, invert, rows, cols);
    return rlt_launch_status(device);
}
int rlt_rocm_mask_zero(rlt_rocm_device* device, float* gradient, int ld, const uint8_t* mask, int invert, int rows, int cols) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(gradient && mask && rows > 0 && cols > 0 && ld >= cols);
    hipLaunchKernelGGL(mask_zero_kernel, dim3(grid1(rows * cols)), dim3(256), 0, device->stream, gradient, ld, mask, invert, rows, cols);
    return rlt_launch_status(device);
}

static int copy2d(rlt_rocm_device* device, const float* src, int lds, float* dst, int ldd, int rows, int cols) {
    hipLaunchKernelGGL(copy2d_kernel, dim3(grid1(rows * cols)), dim3(256), 0, device->stream, src, lds, dst, ldd, rows, cols);
    return rlt_launch_status(device);
}
static bool agent_ok(const rlt_sac_agent* A) {
    return A && A->batch > 0 && A->observation_dim > 0 && A->action_dim > 0 && A->actor && A->critics[0] && A->critics[1] && A->critics_target[0] &&
           A->critics_target[1] && A->observations_actions_base && A->rewards && A->terminated && A->workspace &&
           A->n_actor_layers >= 1 && A->n_critic_layers >= 1 && A->log_alpha.parameters;
}

int rlt_rocm_sac_set_per_operation(rlt_rocm_device* device, int enabled) {
    if (!device) return RLT_E_NOT_INITIALISED;
    device->sac_per_operation = enabled != 0;
    return 0;
}


// rl/algorithms/sac/operations_generic.h:243-337: the fused kernels where they fit, else one launch per reference operation
int rlt_rocm_sac_train_critic(rlt_rocm_device* device, const rlt_sac_agent* A, int ci, const float* action_noise) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A) && (ci == 0 || ci == 1) && action_noise);
    if (!device->sac_per_operation && rlt_sac_update_supported(device, A)) { const rlt_update_noise noise = {action_noise, 0, 0, nullptr}; return rlt_sac_update_critic(device, A, ci, noise); }
    if (!device->sac_per_operation && rlt_sac_wide_supported(device, A)) { const rlt_update_noise noise = {action_noise, 0, 0, nullptr}; return rlt_sac_wide_update_critics(device, A, ci, 1, noise, false); }
    RLT_REQUIRE(A->next_state_action_value_input && A->next_q[0] && A->next_q[1] && A->next_log_probabilities && A->target_action_value && A->d_output_critic[ci]);
    const int B = A->batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    const rlt_dense_layer* critic = A->critics[ci];
    RLT_REQUIRE(A->workspace_bytes >= rlt_rocm_mlp_workspace_bytes(critic, A->n_critic_layers, B) + (size_t)B * 2 * ACT * sizeof(float) + 256);
    RLT_REQUIRE(A->workspace_bytes >= rlt_rocm_mlp_workspace_bytes(A->actor, A->n_actor_layers, B) + (size_t)B * 2 * ACT * sizeof(float) + 256);
    int rc;
    float* actor_out = (float*)A->workspace;
    void* ws = (char*)A->workspace + (((size_t)B * 2 * ACT * sizeof(float) + 255) & ~(size_t)255);
    size_t ws_bytes = A->workspace_bytes - ((char*)ws - (char*)A->workspace);
    if ((rc = rlt_rocm_mlp_zero_gradient(device, critic, A->n_critic_layers))) return rc;
    const float* obs_next = A->observations_actions_base + (size_t)B * D;
    if ((rc = rlt_rocm_mlp_evaluate(device, A->actor, A->n_actor_layers, obs_next, D, actor_out, 2 * ACT, B, ws, ws_bytes))) return rc;
    float* next_actions = A->next_state_action_value_input + OBS;
    if ((rc = rlt_rocm_sas_forward(device, &A->sas, actor_out, 2 * ACT, action_noise, ACT, next_actions, D, nullptr, 0, A->next_log_probabilities, B, ACT))) return rc;
    if (A->next_final_step_mask) if ((rc = rlt_rocm_mask_copy(device, obs_next + OBS, D, next_actions, D, A->next_final_step_mask, 1, B, ACT))) return rc;
    if ((rc = copy2d(device, obs_next, D, A->next_state_action_value_input, D, B, OBS))) return rc;
    if ((rc = rlt_mlp_forward_pair(device, A->critics_target[0], A->critics_target[1], A->n_critic_layers, A->next_state_action_value_input, D, A->next_q[0], A->next_q[1], 1, B, false, ws, ws_bytes))) return rc;
    if ((rc = rlt_rocm_sac_target_action_values(device, A->next_q[0], A->next_q[1], A->rewards, A->terminated, A->next_log_probabilities, A->log_alpha.parameters,
                                               A->gamma, 0, A->target_action_value, B))) return rc;
    if ((rc = rlt_rocm_mlp_forward(device, critic, A->n_critic_layers, A->observations_actions_base, D, B))) return rc;
    const float* q = critic[A->n_critic_layers - 1].output;
    hipLaunchKernelGGL(sac_d_output_kernel, dim3(1), dim3(1024), 0, device->stream, q, (const float*)A->target_action_value, A->final_step_mask, A->d_output_critic[ci], B, 0);
    if ((rc = rlt_launch_status(device))) return rc;
    if ((rc = rlt_rocm_mlp_backward(device, critic, A->n_critic_layers, A->observations_actions_base, D, A->d_output_critic[ci], 1, nullptr, 0, B, 1, ws, ws_bytes))) return rc;
    return rlt_rocm_adam_step(device, A->critic_adam_tensors[ci], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[ci], 0.0f, nullptr);
}

// rl/algorithms/sac/operations_generic.h:488-527
int rlt_rocm_sac_update_critic_targets(rlt_rocm_device* device, const rlt_sac_agent* A) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A));
    if (!device->sac_per_operation && 4 * A->n_critic_layers <= 64) {      // all tensors in one launch (per 32)
        const float* sources[64]; float* targets[64]; uint32_t counts[64];
        int n = 0;
        for (int k = 0; k < 2; k++)
            for (int l = 0; l < A->n_critic_layers; l++) {
                const rlt_dense_layer& s = A->critics[k][l]; const rlt_dense_layer& t = A->critics_target[k][l];
                sources[n] = s.weights; targets[n] = t.weights; counts[n++] = (uint32_t)s.in_dim * s.out_dim;
                sources[n] = s.biases; targets[n] = t.biases; counts[n++] = (uint32_t)s.out_dim;
            }
        return rlt_sac_polyak_list(device, sources, targets, counts, n, A->polyak);
    }
    for (int k = 0; k < 2; k++)
        for (int l = 0; l < A->n_critic_layers; l++) {
            const rlt_dense_layer& s = A->critics[k][l]; const rlt_dense_layer& t = A->critics_target[k][l];
            int rc;
            if ((rc = rlt_rocm_polyak_update(device, s.weights, t.weights, (size_t)s.in_dim * s.out_dim, A->polyak, 0))) return rc;
            if ((rc = rlt_rocm_polyak_update(device, s.biases, t.biases, (size_t)s.out_dim, A->polyak, 0))) return rc;
        }
    return 0;
}

// rl/algorithms/sac/operations_generic.h:395-468, one launch per reference operation
int rlt_rocm_sac_train_actor(rlt_rocm_device* device, const rlt_sac_agent* A, const float* action_noise) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A) && action_noise);
    if (!device->sac_per_operation && rlt_sac_update_supported(device, A)) { const rlt_update_noise noise = {action_noise, 0, 0, nullptr}; return rlt_sac_update_actor(device, A, noise); }
    if (!device->sac_per_operation && rlt_sac_wide_supported(device, A)) { const rlt_update_noise noise = {action_noise, 0, 0, nullptr}; return rlt_sac_wide_update_actor(device, A, noise); }
    RLT_REQUIRE(A->state_action_value_input && A->d_output_actor_critics && A->d_critic_input[0] && A->d_critic_input[1] && A->d_actor_output_squashing &&
                A->d_actor_output && A->actor_pre_squashing && A->actor_log_probabilities && A->actor_actions && A->log_alpha.gradient);
    const int B = A->batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    RLT_REQUIRE(A->workspace_bytes >= rlt_rocm_mlp_workspace_bytes(A->critics[0], A->n_critic_layers, B));
    RLT_REQUIRE(A->workspace_bytes >= rlt_rocm_mlp_workspace_bytes(A->actor, A->n_actor_layers, B));
    void* ws = A->workspace; size_t ws_bytes = A->workspace_bytes;
    int rc;
    if ((rc = rlt_rocm_mlp_zero_gradient(device, A->actor, A->n_actor_layers))) return rc;
    if ((rc = rlt_rocm_fill_f32(device, A->log_alpha.gradient, 1, 1, 1, 0.0f))) return rc;
    const float* obs = A->observations_actions_base;
    if ((rc = rlt_rocm_mlp_forward(device, A->actor, A->n_actor_layers, obs, D, B))) return rc;
    const float* actor_out = A->actor[A->n_actor_layers - 1].output;
    if ((rc = rlt_rocm_sas_forward(device, &A->sas, actor_out, 2 * ACT, action_noise, ACT, A->actor_actions, ACT, A->actor_pre_squashing, ACT,
                                   A->actor_log_probabilities, B, ACT))) return rc;
    float* sav_actions = A->state_action_value_input + OBS;
    if ((rc = copy2d(device, A->actor_actions, ACT, sav_actions, D, B, ACT))) return rc;
    if (A->final_step_mask) if ((rc = rlt_rocm_mask_copy(device, obs + OBS, D, sav_actions, D, A->final_step_mask, 1, B, ACT))) return rc;
    if ((rc = copy2d(device, obs, D, A->state_action_value_input, D, B, OBS))) return rc;
    if ((rc = rlt_mlp_forward_pair(device, A->critics[0], A->critics[1], A->n_critic_layers, A->state_action_value_input, D, nullptr, nullptr, 0, B, true, ws, ws_bytes))) return rc;
    hipLaunchKernelGGL(sac_d_output_kernel, dim3(1), dim3(1024), 0, device->stream, (const float*)nullptr, (const float*)nullptr, A->final_step_mask,
                       A->d_output_actor_critics, B, 1);
    if ((rc = rlt_launch_status(device))) return rc;
    for (int k = 0; k < 2; k++)   // the critics' output activation is the identity, so d_output survives the first backward_input unchanged
        if ((rc = rlt_rocm_mlp_backward(device, A->critics[k], A->n_critic_layers, nullptr, 0, A->d_output_actor_critics, 1, A->d_critic_input[k], D, B, 0, ws, ws_bytes))) return rc;
    const float* q1 = A->critics[0][A->n_critic_layers - 1].output; const float* q2 = A->critics[1][A->n_critic_layers - 1].output;
    if ((rc = rlt_rocm_sac_min_value_d_output(device, q1, q2, A->d_critic_input[0], A->d_critic_input[1], D, D, ACT, A->d_actor_output_squashing, ACT, B))) return rc;
    if (A->final_step_mask) if ((rc = rlt_rocm_mask_zero(device, A->d_actor_output_squashing, ACT, A->final_step_mask, 1, B, ACT))) return rc;
    if ((rc = sas_backward_impl(device, &A->sas, actor_out, 2 * ACT, action_noise, ACT, A->actor_actions, ACT, A->actor_pre_squashing, ACT,
                                A->d_actor_output_squashing, ACT, A->d_actor_output, 2 * ACT, A->log_alpha.parameters, A->log_alpha.gradient, A->reset, B, ACT))) return rc;
    if ((rc = rlt_rocm_mlp_backward(device, A->actor, A->n_actor_layers, obs, D, A->d_actor_output, 2 * ACT, nullptr, 0, B, 1, ws, ws_bytes))) return rc;
    if ((rc = rlt_rocm_adam_step(device, A->actor_adam_tensors, A->n_actor_adam_tensors, &A->actor_adam, A->actor_age, 0.0f, nullptr))) return rc;
    return rlt_rocm_adam_step(device, &A->log_alpha, 1, &A->alpha_adam, A->alpha_age, 0.0f, nullptr);
}

// both train_critic calls of a loop step with a shared batch (and update_critic_targets) as one launch where the fused kernel fits
static int train_critics(rlt_rocm_device* device, const rlt_sac_agent* A, const rlt_update_noise& noise, int update_targets) {
    if (!device->sac_per_operation && rlt_sac_update_supported(device, A)) return rlt_sac_update_critics(device, A, noise, update_targets != 0);
    if (!device->sac_per_operation && rlt_sac_wide_supported(device, A)) return rlt_sac_wide_update_critics(device, A, 0, 2, noise, update_targets != 0);
    int rc;
    const float* values = noise.values;
    if (!values) {
        RLT_REQUIRE(noise.drawn);
        if ((rc = rlt_rocm_randn_f32(device, noise.drawn, (size_t)A->batch * A->action_dim, noise.seed, noise.stream))) return rc;
        values = noise.drawn;
    }
    for (int k = 0; k < 2; k++)
        if ((rc = rlt_rocm_sac_train_critic(device, A, k, values))) return rc;
    return update_targets ? rlt_rocm_sac_update_critic_targets(device, A) : 0;
}
int rlt_rocm_sac_train_critics(rlt_rocm_device* device, const rlt_sac_agent* A, const float* action_noise, int update_targets) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A) && action_noise);
    const rlt_update_noise noise = {action_noise, 0, 0, nullptr};
    return train_critics(device, A, noise, update_targets);
}
int rlt_rocm_sac_train_critics_drawn(rlt_rocm_device* device, const rlt_sac_agent* A, float* drawn_noise, uint64_t seed, uint64_t stream, int update_targets) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A));
    const rlt_update_noise noise = {nullptr, seed, stream, drawn_noise};
    return train_critics(device, A, noise, update_targets);
}
int rlt_rocm_sac_train_actor_drawn(rlt_rocm_device* device, const rlt_sac_agent* A, float* drawn_noise, uint64_t seed, uint64_t stream) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A));
    if (!device->sac_per_operation && rlt_sac_update_supported(device, A)) { const rlt_update_noise noise = {nullptr, seed, stream, drawn_noise}; return rlt_sac_update_actor(device, A, noise); }
    if (!device->sac_per_operation && rlt_sac_wide_supported(device, A)) { const rlt_update_noise noise = {nullptr, seed, stream, drawn_noise}; return rlt_sac_wide_update_actor(device, A, noise); }
    RLT_REQUIRE(drawn_noise);
    const int rc = rlt_rocm_randn_f32(device, drawn_noise, (size_t)A->batch * A->action_dim, seed, stream);
    return rc ? rc : rlt_rocm_sac_train_actor(device, A, drawn_noise);
}

// rl/algorithms/sac/loop/core/operations_generic.h:110-155 past the warm-up, as a host loop over the entry points of this library
int rlt_rocm_sac_pendulum_loop_by_calls(rlt_rocm_device* device, const rlt_sac_agent* A, const rlt_pendulum_runner* runner, const rlt_replay_buffer* rb, int n_steps,
                                        uint64_t seed, uint64_t step_offset, const rlt_sac_loop_scratch* S) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(agent_ok(A) && runner && rb && S && n_steps >= 0);
    RLT_REQUIRE(S->rollout_noise && S->noise_critic && S->noise_actor && S->env_indices && S->sample_offsets);
    RLT_REQUIRE(rb->observation_dim == A->observation_dim && rb->action_dim == A->action_dim && rb->n_envs == runner->n_envs);
    const int B = A->batch;
    int rc;
    for (int i = 0; i < n_steps; i++) {
        const uint64_t g = 8 * (step_offset + (uint64_t)i);
        // every draw is made by the kernel that consumes it (and echoed into the scratch arrays): four launches per step where the fused kernels fit
        if ((rc = rlt_rocm_pendulum_runner_step_drawn(device, runner, rb, A->actor, A->n_actor_layers, &A->sas, S->rollout_noise, seed, g + 1, g + 2))) return rc;
        if ((rc = rlt_rocm_gather_batch_drawn(device, rb, seed, g + 3, S->env_indices, S->sample_offsets, runner->episode_step_limit, B, A->observations_actions_base, A->rewards,
                                              A->terminated, nullptr, nullptr, nullptr, nullptr))) return rc;
        if ((rc = rlt_rocm_sac_train_critics_drawn(device, A, S->noise_critic, seed, g + 4, 1))) return rc;
        if ((rc = rlt_rocm_sac_train_actor_drawn(device, A, S->noise_actor, seed, g + 5))) return rc;
    }
    return 0;
}

// ---------------------------------------------------------------------------------------- sequence batches, sequential (recurrent) networks
static inline const float* seq_output(const rlt_seq_layer* layers, int n) { const rlt_seq_layer& L = layers[n - 1]; return L.kind ? L.gru.output : L.dense.output; }
static inline int seq_out_dim(const rlt_seq_layer* layers, int n) { const rlt_seq_layer& L = layers[n - 1]; return L.kind ? L.gru.hidden_dim : L.dense.out_dim; }
static bool sequence_agent_ok(const rlt_sac_sequence_agent* A) {
    if (!A || A->observation_dim <= 0 || A->action_dim <= 0 || A->n_actor_layers < 1 || A->n_critic_layers < 1) return false;
    if (!A->actor || !A->critics[0] || !A->critics[1] || !A->critics_target[0] || !A->critics_target[1] || !A->log_alpha.parameters) return false;
    const rlt_sequence_batch& K = A->batch;
    if (K.batch <= 0 || K.sequence_length <= 0 || !K.observations_actions_base || !K.rewards || !K.terminated || !K.reset || !K.next_reset_base || !K.final_step_mask ||
        !K.next_final_step_mask_base) return false;
    if (seq_out_dim(A->actor, A->n_actor_layers) != 2 * A->action_dim) return false;
    for (int k = 0; k < 2; k++) if (seq_out_dim(A->critics[k], A->n_critic_layers) != 1 || seq_out_dim(A->critics_target[k], A->n_critic_layers) != 1) return false;
    return A->workspace && A->workspace_bytes >= rlt_rocm_sac_sequence_workspace_bytes(A);
}

// what one pass of any of the agent's networks needs, rounded up so that the second half of a doubled workspace is aligned like the first
static size_t sequence_pass_workspace_bytes(const rlt_sac_sequence_agent* A, int T, int B) {
    size_t n = rlt_rocm_seq_workspace_bytes(A->actor, A->n_actor_layers, T, B);
    n = std::max(n, rlt_rocm_seq_workspace_bytes(A->critics[0], A->n_critic_layers, T, B));
    n = std::max(n, rlt_rocm_seq_workspace_bytes(A->critics_target[0], A->n_critic_layers, T, B));
    return (n + 255) & ~(size_t)255;
}
size_t rlt_rocm_sac_sequence_workspace_bytes(const rlt_sac_sequence_agent* A) {
    if (!A || !A->actor || !A->critics[0] || !A->critics_target[0]) return 0;
    const int T = A->batch.sequence_length + 1, B = A->batch.batch;
    // up to three passes run at the same time (rlt_side_begin), each in its own third; then the loss gradient of the first critic where both critics train in one call
    return 3 * sequence_pass_workspace_bytes(A, T, B) + ((sizeof(float) * (size_t)A->batch.sequence_length * B + 255) & ~(size_t)255);
}

// Agents whose networks are the reference's recurrent approximators (seq_stack.hip): a launch takes every layer of a pass, and the passes that do not depend on each other
// share one. The trained critics' loss gradients and backward passes follow, then their optimisers in one launch.
static bool sequence_agent_stacked(const rlt_sac_sequence_agent* A) {
    const int T = A->batch.sequence_length + 1, B = A->batch.batch;
    if (!rlt_seq_stack_faster(RLT_STACK_UPDATE, A->batch.sequence_length, B)) return false;
    if (!rlt_seq_stack_supported(A->actor, A->n_actor_layers, T)) return false;
    for (int k = 0; k < 2; k++)
        if (!rlt_seq_stack_supported(A->critics[k], A->n_critic_layers, T) || !rlt_seq_stack_supported(A->critics_target[k], A->n_critic_layers, T)) return false;
    // the workspace is sized by the first critic and its target: of a wider second one the passes below, which look at their share of it, refuse what does not fit
    const size_t share = sequence_pass_workspace_bytes(A, T, B);
    return rlt_rocm_seq_workspace_bytes(A->critics[1], A->n_critic_layers, T, B) <= share && rlt_rocm_seq_workspace_bytes(A->critics_target[1], A->n_critic_layers, T, B) <= share;
}
static int sequence_next_actions(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, const float* base_next, const uint8_t* next_final, int rows, const float* action_noise) {
    SequenceActions a = {};
    a.sas = A->sas; a.policy = seq_output(A->actor, A->n_actor_layers); a.noise = action_noise; a.base = base_next; a.final_step = next_final;
    a.critic_input = A->next_state_action_value_input; a.log_probabilities = A->next_log_probabilities;
    a.rows = rows; a.obs = A->observation_dim; a.act = A->action_dim;
    hipLaunchKernelGGL(sequence_actions_kernel, dim3(sequence_grid(rows)), dim3(256), 0, device->stream, a);
    return rlt_launch_status(device);
}
// target values, and the loss gradients of critics ci ... ci + count - 1 into d_output[k]; `offset`: where in the next values the first step's lies
static int sequence_targets(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, int ci, int count, int offset, float* const (&d_output)[2]) {
    const rlt_sequence_batch& K = A->batch;
    SequenceTargets a = {};
    for (int k = 0; k < 2; k++) a.next_q[k] = A->next_q[k] + offset;
    for (int k = 0; k < count; k++) { a.q[k] = seq_output(A->critics[ci + k], A->n_critic_layers); a.d_output[k] = d_output[k]; }
    a.rewards = K.rewards; a.terminated = K.terminated; a.next_log_probabilities = A->next_log_probabilities; a.log_alpha = A->log_alpha.parameters;
    a.final_step = K.final_step_mask; a.target = A->target_action_value; a.gamma = A->gamma; a.rows = K.sequence_length * K.batch; a.count = count;
    hipLaunchKernelGGL(sequence_targets_kernel, dim3(sequence_grid(a.rows)), dim3(256), 0, device->stream, a);
    return rlt_launch_status(device);
}

static int stacked_train_critics(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, int ci, int count, const float* action_noise) {
    const rlt_sequence_batch& K = A->batch;
    const int S = K.sequence_length, B = K.batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    const int first = A->include_first_step_in_targets ? 1 : 0, T = S + first, next_offset = first ? 0 : 1;
    const size_t ws_bytes = sequence_pass_workspace_bytes(A, S + 1, B);
    const float* base_next = K.observations_actions_base + (size_t)next_offset * B * D;
    const uint8_t* next_reset = K.next_reset_base + (size_t)next_offset * B;
    const uint8_t* next_final = K.next_final_step_mask_base + (size_t)next_offset * B;
    rlt_stack_forward forward[3];
    for (int k = 0; k < count; k++) forward[k] = {A->critics[ci + k], K.observations_actions_base, D, K.reset, S, B, nullptr};
    forward[count] = {A->actor, base_next, D, next_reset, T, B, nullptr};
    int rc;
    if ((rc = rlt_seq_stack_forward(device, forward, count + 1))) return rc;
    if ((rc = sequence_next_actions(device, A, base_next, next_final, T * B, action_noise))) return rc;
    const rlt_stack_forward targets[2] = {{A->critics_target[0], A->next_state_action_value_input, D, next_reset, T, B, A->next_q[0]},
                                          {A->critics_target[1], A->next_state_action_value_input, D, next_reset, T, B, A->next_q[1]}};
    if ((rc = rlt_seq_stack_forward(device, targets, 2))) return rc;
    // the last critic's loss gradient goes to the agent's buffer (where two calls leave it), the other's to the end of the workspace
    float* const d_output[2] = {count == 1 ? A->d_output : (float*)((char*)A->workspace + 3 * ws_bytes), A->d_output};
    if ((rc = sequence_targets(device, A, ci, count, first * B, d_output))) return rc;
    rlt_stack_backward backward[2];
    for (int k = 0; k < count; k++)
        backward[k] = {A->critics[ci + k], K.observations_actions_base, D, d_output[k], nullptr, K.reset, S, B, 1, 1, (char*)A->workspace + k * ws_bytes};
    if ((rc = rlt_seq_stack_backward(device, backward, count))) return rc;
    if (count == 2)
        return rlt_adam_step_pair(device, A->critic_adam_tensors[0], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[0], A->critic_adam_tensors[1], A->n_critic_adam_tensors,
                                  &A->critic_adam, A->critic_age[1]);
    return rlt_rocm_adam_step(device, A->critic_adam_tensors[ci], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[ci], 0.0f, nullptr);
}

// rl/algorithms/sac/operations_generic.h:243-337 on a sequence batch, one launch per reference operation
int rlt_rocm_sac_sequence_train_critic(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, int ci, const float* action_noise) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(sequence_agent_ok(A) && (ci == 0 || ci == 1) && action_noise);
    RLT_REQUIRE(A->next_state_action_value_input && A->next_q[0] && A->next_q[1] && A->next_log_probabilities && A->target_action_value && A->d_output);
    const rlt_sequence_batch& K = A->batch;
    const int S = K.sequence_length, B = K.batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    const int first = A->include_first_step_in_targets ? 1 : 0, T = S + first, next_offset = first ? 0 : 1;   // off_policy_runner/operations_generic.h:85-92
    const rlt_seq_layer* critic = A->critics[ci];
    if (sequence_agent_stacked(A)) return stacked_train_critics(device, A, ci, 1, action_noise);
    // two halves of the workspace: passes that do not depend on each other run at the same time, one on the handle's side stream -- the trained critic's forward
    // pass next to the actor's on the next rows, then the second target critic next to the first (each recurrence fills a twentieth of the chip)
    const size_t ws_bytes = sequence_pass_workspace_bytes(A, S + 1, B);
    void* ws = A->workspace; void* ws_side = (char*)A->workspace + ws_bytes;
    const bool overlap = S >= 48;      // short sequences: a pass is shorter than the two events that fork and join a stream cost on the host
    int rc;
    if ((rc = rlt_rocm_seq_zero_gradient(device, critic, A->n_critic_layers))) return rc;                                                  // :263
    {
        const bool side = overlap && rlt_side_begin(device);
        rc = rlt_rocm_seq_forward(device, critic, A->n_critic_layers, K.observations_actions_base, D, K.reset, S, B, side ? ws_side : ws, ws_bytes);   // :294
        rlt_side_end(device);
        if (rc) return rc;
    }
    const float* base_next = K.observations_actions_base + (size_t)next_offset * B * D;
    const uint8_t* next_reset = K.next_reset_base + (size_t)next_offset * B;
    const uint8_t* next_final = K.next_final_step_mask_base + (size_t)next_offset * B;
    if ((rc = rlt_rocm_seq_forward(device, A->actor, A->n_actor_layers, base_next, D, next_reset, T, B, ws, ws_bytes))) return rc;           // :266-273
    if ((rc = sequence_next_actions(device, A, base_next, next_final, T * B, action_noise))) return rc;
    for (int k = 1; k >= 0; k--) {                                                                                                         // :283-284 (target critic 1 on the side stream)
        const bool side = k == 1 && overlap && rlt_side_begin(device);
        rc = rlt_rocm_seq_forward(device, A->critics_target[k], A->n_critic_layers, A->next_state_action_value_input, D, next_reset, T, B, side ? ws_side : ws, ws_bytes);
        if (!rc) rc = rlt_rocm_memcpy_d2d(device, A->next_q[k], seq_output(A->critics_target[k], A->n_critic_layers), sizeof(float) * T * B);
        rlt_side_end(device);
        if (rc) return rc;
    }
    if (overlap && (rc = rlt_side_join(device))) return rc;
    // the value of the step after (offset B where the first step is included), the log-probability at the same index (:144-154); the loss gradient (:289-316)
    float* const d_output[2] = {A->d_output, nullptr};
    if ((rc = sequence_targets(device, A, ci, 1, first * B, d_output))) return rc;
    if ((rc = rlt_rocm_seq_backward(device, critic, A->n_critic_layers, K.observations_actions_base, D, A->d_output, nullptr, K.reset, S, B, 1, 0, ws, ws_bytes))) return rc;   // :329
    return rlt_rocm_adam_step(device, A->critic_adam_tensors[ci], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[ci], 0.0f, nullptr);   // :336
}

// Both critics on one batch and one set of noise (the loop's SHARED_BATCH case, rl/algorithms/sac/loop/core/operations_generic.h:127-138): what the two calls of
// train_critic would compute twice -- the actor on the next rows, its sample, both target critics, the target values -- is computed once. Agents of recurrent
// approximators (sequence_agent_stacked) take stacked_train_critics: both critics' passes and the actor's are one launch on the handle's stream, then the two target critics' one,
// the two backward passes one, and one step of both optimisers. For any other agent the two critics' passes run next to each other on the handle's three streams: first side stream critic 0 forward, then target critic 1; second side stream critic 1 forward; main
// stream actor, sample, target critic 0; after the join the target values and both loss gradients, then critic 0's backward pass on the main stream next to critic 1's
// on a side stream, then both optimisers. Every pass does what the single calls' does, on the same inputs: the results are theirs bit for bit.
int rlt_rocm_sac_sequence_train_critics(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, const float* action_noise) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(sequence_agent_ok(A) && action_noise);
    RLT_REQUIRE(A->next_state_action_value_input && A->next_q[0] && A->next_q[1] && A->next_log_probabilities && A->target_action_value && A->d_output);
    const rlt_sequence_batch& K = A->batch;
    const int S = K.sequence_length, B = K.batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    const int first = A->include_first_step_in_targets ? 1 : 0, T = S + first, next_offset = first ? 0 : 1;
    const size_t ws_bytes = sequence_pass_workspace_bytes(A, S + 1, B);
    void* ws = A->workspace; void* ws_side = (char*)A->workspace + ws_bytes; void* ws_second = (char*)A->workspace + 2 * ws_bytes;
    if (sequence_agent_stacked(A)) return stacked_train_critics(device, A, 0, 2, action_noise);
    float* d_output_first = (float*)((char*)A->workspace + 3 * ws_bytes);      // critic 0's loss gradient; critic 1's goes to the agent's buffer, where two single calls leave it
    const bool overlap = S >= 48;      // short sequences: a pass is shorter than the two events that fork and join a stream cost on the host
    int rc;
    for (int k = 0; k < 2; k++) if ((rc = rlt_rocm_seq_zero_gradient(device, A->critics[k], A->n_critic_layers))) return rc;
    {
        if (overlap) rlt_side_begin(device);      // (without a second stream everything below simply runs in order on the one stream)
        rc = rlt_rocm_seq_forward(device, A->critics[0], A->n_critic_layers, K.observations_actions_base, D, K.reset, S, B, device->side_return ? ws_side : ws, ws_bytes);
        rlt_side_end(device);
        if (rc) return rc;
        if (overlap) rlt_side_begin(device, 1);
        rc = rlt_rocm_seq_forward(device, A->critics[1], A->n_critic_layers, K.observations_actions_base, D, K.reset, S, B, device->side_return ? ws_second : ws, ws_bytes);
        rlt_side_end(device);
        if (rc) return rc;
    }
    const float* base_next = K.observations_actions_base + (size_t)next_offset * B * D;
    const uint8_t* next_reset = K.next_reset_base + (size_t)next_offset * B;
    const uint8_t* next_final = K.next_final_step_mask_base + (size_t)next_offset * B;
    if ((rc = rlt_rocm_seq_forward(device, A->actor, A->n_actor_layers, base_next, D, next_reset, T, B, ws, ws_bytes))) return rc;
    if ((rc = sequence_next_actions(device, A, base_next, next_final, T * B, action_noise))) return rc;
    for (int k = 1; k >= 0; k--) {      // target critic 1 behind critic 0's forward pass on the side stream (it waits for the copies above), target critic 0 on the main stream
        if (k == 1 && overlap) rlt_side_begin(device);
        rc = rlt_rocm_seq_forward(device, A->critics_target[k], A->n_critic_layers, A->next_state_action_value_input, D, next_reset, T, B, device->side_return ? ws_side : ws, ws_bytes);
        if (!rc) rc = rlt_rocm_memcpy_d2d(device, A->next_q[k], seq_output(A->critics_target[k], A->n_critic_layers), sizeof(float) * T * B);
        rlt_side_end(device);
        if (rc) return rc;
    }
    if (overlap && (rc = rlt_side_join(device))) return rc;
    float* const d_output[2] = {d_output_first, A->d_output};
    if ((rc = sequence_targets(device, A, 0, 2, first * B, d_output))) return rc;
    {
        if (overlap) rlt_side_begin(device);
        rc = rlt_rocm_seq_backward(device, A->critics[1], A->n_critic_layers, K.observations_actions_base, D, A->d_output, nullptr, K.reset, S, B, 1, 0, device->side_return ? ws_side : ws, ws_bytes);
        rlt_side_end(device);
        if (rc) return rc;
    }
    if ((rc = rlt_rocm_seq_backward(device, A->critics[0], A->n_critic_layers, K.observations_actions_base, D, d_output_first, nullptr, K.reset, S, B, 1, 0, ws, ws_bytes))) return rc;
    if (overlap && (rc = rlt_side_join(device))) return rc;
    for (int k = 0; k < 2; k++)
        if ((rc = rlt_rocm_adam_step(device, A->critic_adam_tensors[k], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[k], 0.0f, nullptr))) return rc;
    return 0;
}

// sac/operations_generic.h:486-527
int rlt_rocm_sac_sequence_update_critic_targets(rlt_rocm_device* device, const rlt_sac_sequence_agent* A) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(sequence_agent_ok(A) && A->n_critic_layers <= RLT_SEQ_MAX_LAYERS);
    // every tensor of both target critics in one launch per 32 tensors
    const float* sources[2 * 5 * RLT_SEQ_MAX_LAYERS]; float* targets[2 * 5 * RLT_SEQ_MAX_LAYERS]; uint32_t counts[2 * 5 * RLT_SEQ_MAX_LAYERS];
    int n = 0;
    auto pair = [&](const float* source, float* target, size_t count) { sources[n] = source; targets[n] = target; counts[n++] = (uint32_t)count; };
    for (int k = 0; k < 2; k++)
        for (int l = 0; l < A->n_critic_layers; l++) {
            const rlt_seq_layer& s = A->critics[k][l]; const rlt_seq_layer& t = A->critics_target[k][l];
            RLT_REQUIRE(s.kind == t.kind);
            if (s.kind == 0) {
                pair(s.dense.weights, t.dense.weights, (size_t)s.dense.in_dim * s.dense.out_dim); pair(s.dense.biases, t.dense.biases, (size_t)s.dense.out_dim);
            } else {
                const size_t H = s.gru.hidden_dim, I = s.gru.input_dim;
                pair(s.gru.weights_input, t.gru.weights_input, 3 * H * I); pair(s.gru.biases_input, t.gru.biases_input, 3 * H);
                pair(s.gru.weights_hidden, t.gru.weights_hidden, 3 * H * H); pair(s.gru.biases_hidden, t.gru.biases_hidden, 3 * H);
                pair(s.gru.initial_hidden_state, t.gru.initial_hidden_state, H);
            }
        }
    for (int i = 0; i < n; i++) RLT_REQUIRE(sources[i] && targets[i]);
    return rlt_sac_polyak_list(device, sources, targets, counts, n, A->polyak);
}

// sac/operations_generic.h:395-468 on a sequence batch
int rlt_rocm_sac_sequence_train_actor(rlt_rocm_device* device, const rlt_sac_sequence_agent* A, const float* action_noise) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(sequence_agent_ok(A) && action_noise);
    RLT_REQUIRE(A->state_action_value_input && A->d_output && A->d_critic_input[0] && A->d_critic_input[1] && A->d_actor_output_squashing && A->d_actor_output &&
                A->actor_pre_squashing && A->actor_log_probabilities && A->actor_actions && A->log_alpha.gradient);
    const rlt_sequence_batch& K = A->batch;
    const int S = K.sequence_length, B = K.batch, OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT, R = S * B;
    const size_t ws_bytes = sequence_pass_workspace_bytes(A, S + 1, B);
    void* ws = A->workspace; void* ws_side = (char*)A->workspace + ws_bytes;
    const bool stacked = sequence_agent_stacked(A);
    const bool overlap = S >= 48 && !stacked;      // short sequences: a pass is shorter than the two events that fork and join a stream cost on the host
    int rc;
    if (!stacked && (rc = rlt_rocm_seq_zero_gradient(device, A->actor, A->n_actor_layers))) return rc;                                      // :414
    const float* obs = K.observations_actions_base;
    if ((rc = rlt_rocm_seq_forward(device, A->actor, A->n_actor_layers, obs, D, K.reset, S, B, ws, ws_bytes))) return rc;                   // :427
    const float* actor_out = seq_output(A->actor, A->n_actor_layers);
    // sample, the critics' input rows (:428-431), and the gradient at the critics' outputs, a constant per row (:437-453): formed before the critics' passes, so that each
    // critic's forward pass and its gradient towards the input (:432-433, :458-459) can follow each other on a stream of their own -- critic 1 on the side stream, critic 0 on the main stream
    SequenceActions actions = {};
    actions.sas = A->sas; actions.policy = actor_out; actions.noise = action_noise; actions.base = obs; actions.final_step = K.final_step_mask;
    actions.critic_input = A->state_action_value_input; actions.log_probabilities = A->actor_log_probabilities; actions.actions = A->actor_actions;
    actions.pre_squashing = A->actor_pre_squashing; actions.d_output = A->d_output; actions.rows = R; actions.obs = OBS; actions.act = ACT;
    hipLaunchKernelGGL(sequence_actions_kernel, dim3(sequence_grid(R)), dim3(256), 0, device->stream, actions);
    if ((rc = rlt_launch_status(device))) return rc;
    // the inner layers of backward_input run without the reset mode (nn_models/sequential/operations_generic.h:399-407); the critics'
    // output layer has no activation function, so d_output survives the calls unchanged (both read it)
    if (stacked) {
        rlt_stack_forward forward[2]; rlt_stack_backward backward[2];
        for (int k = 0; k < 2; k++) {
            forward[k] = {A->critics[k], A->state_action_value_input, D, K.reset, S, B, nullptr};
            backward[k] = {A->critics[k], nullptr, 0, A->d_output, A->d_critic_input[k], nullptr, S, B, 0, 0, nullptr};
        }
        if ((rc = rlt_seq_stack_forward(device, forward, 2)) || (rc = rlt_seq_stack_backward(device, backward, 2))) return rc;
    }
    for (int k = 1; k >= 0 && !stacked; k--) {
        const bool side = k == 1 && overlap && rlt_side_begin(device);
        void* w = side ? ws_side : ws;
        rc = rlt_rocm_seq_forward(device, A->critics[k], A->n_critic_layers, A->state_action_value_input, D, K.reset, S, B, w, ws_bytes);
        if (!rc) rc = rlt_rocm_seq_backward(device, A->critics[k], A->n_critic_layers, nullptr, 0, A->d_output, A->d_critic_input[k], K.reset, S, B, 0, 0, w, ws_bytes);
        rlt_side_end(device);
        if (rc) return rc;
    }
    if (overlap && (rc = rlt_side_join(device))) return rc;
    void* counters = nullptr;
    if ((rc = rlt_counters(device, &counters))) return rc;
    SequenceActorGradient gradient = {};
    gradient.sas = A->sas; gradient.final_step = K.final_step_mask; gradient.reset = K.reset; gradient.policy = actor_out; gradient.noise = action_noise;
    gradient.actions = A->actor_actions; gradient.pre_squashing = A->actor_pre_squashing; gradient.log_alpha = A->log_alpha.parameters;
    for (int k = 0; k < 2; k++) { gradient.q[k] = seq_output(A->critics[k], A->n_critic_layers); gradient.d_critic_input[k] = A->d_critic_input[k]; }
    gradient.d_action = A->d_actor_output_squashing; gradient.d_policy = A->d_actor_output; gradient.d_log_alpha = A->log_alpha.gradient;
    gradient.partial = (float*)((char*)counters + 256); gradient.tickets = rlt_tickets_of(counters, 0);
    gradient.rows = R; gradient.obs = OBS; gradient.act = ACT;
    hipLaunchKernelGGL(sequence_actor_gradient_kernel, dim3(sequence_grid(R)), dim3(256), 0, device->stream, gradient);                    // :460-464
    if ((rc = rlt_launch_status(device))) return rc;
    if (stacked) {
        const rlt_stack_backward backward = {A->actor, obs, D, A->d_actor_output, nullptr, K.reset, S, B, 1, 1, ws};
        if ((rc = rlt_seq_stack_backward(device, &backward, 1))) return rc;
        return rlt_adam_step_pair(device, A->actor_adam_tensors, A->n_actor_adam_tensors, &A->actor_adam, A->actor_age, &A->log_alpha, 1, &A->alpha_adam, A->alpha_age);
    }
    if ((rc = rlt_rocm_seq_backward(device, A->actor, A->n_actor_layers, obs, D, A->d_actor_output, nullptr, K.reset, S, B, 1, 0, ws, ws_bytes))) return rc;
    if ((rc = rlt_rocm_adam_step(device, A->actor_adam_tensors, A->n_actor_adam_tensors, &A->actor_adam, A->actor_age, 0.0f, nullptr))) return rc;   // :465
    return rlt_rocm_adam_step(device, &A->log_alpha, 1, &A->alpha_adam, A->alpha_age, 0.0f, nullptr);                                      // :466
}

}  // extern "C"
