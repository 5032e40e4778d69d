// Adam step (moments, bias correction, parameter update, optional polyak target and gradient norm) for a list of
// parameter tensors in one launch, and the polyak soft update.
// reference: nn/optimizers/adam/operations_generic.h:43-66, instance/operations_generic.h:26-72,
//            utils/polyak/operations_generic.h:11-43; CUDA counterparts adam/operations_cuda.h:18-68 (scalar kernel for the
//            bias corrections), nn/layers/dense/operations_cuda.h:195-233 (one launch per layer).
#include "common.h"
#include "optim.h"

namespace {

constexpr int MAX_T = 16;
constexpr uint32_t MAX_BLOCKS = 960 - MAX_T;      // rounding up per tensor included, the workgroups' sums for the squared norm fit the counters block
struct AdamLaunch {
    rlt_adam_tensor t[MAX_T];
    // Workgroups [first_block[i], first_block[i + 1]) step tensor i, span[i] elements each: the tensor is the same for a whole workgroup and its pointers arrive with scalar loads.
    // (As a list of elements that each lane searched for its own, every launch made another trip to the argument segment before it could ask for data: 7.4 instead of 5.6 us
    // at 72 k parameters in six tensors.)
    uint32_t first_block[MAX_T + 1], span[MAX_T];
    uint32_t vec;                // bit i: tensor i is stepped four elements at a time (16-byte loads of the blocks, moments and values), but for its last one to three
    int n;
    rlt_adam_parameters p;
    float polyak;
    uint32_t* age;
    uint32_t* tickets;           // zero between launches: TICKET_LEAVES words a cache line apart, then the root (rlt_last_through)
    float* block_partials;       // [gridDim.x] sums of squared gradients
    float* out_sq_norm;          // optional
    int increment_age;
    int accumulate_norm;         // add to *out_sq_norm instead of overwriting (later chunks of one step)
    // optional: the gradients are still blocks of partial sums. Element j of tensor t is source_scale[t] times the sum over `groups`
    // blocks of `block_stride` floats of source[g * block_stride + source_offset[t] + j], added up in the order of the small-MLP
    // reduction kernel (four quarters of the blocks, each in block order, then (q0 + q1) + (q2 + q3)); it is stored in the tensor's
    // gradient before it is used
    const float* source;
    int groups, block_stride;
    uint32_t source_offset[MAX_T];
    float source_scale[MAX_T], source_add[MAX_T];
    float* extra_out; uint32_t extra_offset; float extra_scale;      // optional: one more sum of the blocks, stored scaled (not a gradient)
};

// the workgroup's tensor (the same for all of its lanes)
__device__ __forceinline__ int tensor_of(const AdamLaunch& a, uint32_t block) {
    int ti = 0;
#pragma unroll
    for (int k = 1; k < MAX_T; k++) ti += (k < a.n && block >= a.first_block[k]) ? 1 : 0;
    return __builtin_amdgcn_readfirstlane(ti);
}

// sum over the blocks of one element, every load in flight at once where there are at most 16 blocks
__device__ __forceinline__ float sum_of_blocks(const float* __restrict__ p, int groups, int stride) {
    const float* const src[1] = {p};
    float out[1];
    rlt_sum_of_blocks<1, 2>(src, groups, stride, out);
    return out[0];
}

// the step for one optimiser by workgroups [0, n_blocks) numbered `block`. With a fifth wavefront in the workgroups (TICKETS_APART) that one draws the tickets and stores the incremented age while the others
// step the elements: behind the stores the two levels of tickets were two more trips to memory at the launch's end. Such a step never adds blocks of sums up, so the kernel is built without the registers for
// them (from_blocks): with them three workgroups of five wavefronts fit a compute unit and 944 came in two rounds. Launches in a row, us, four wavefronts / five with those registers / five: 10 elements
// 4.9 / 5.0 / 4.2, 72,000 in one tensor 5.9 / 5.0 / 4.5, 700,000 7.7 / 8.8 / 6.2, 2,000,000 11.2 / 13.1 / 9.5, 500,000 in six tensors on no 16 bytes 8.3 / 9.9 / 7.0, 50,000,000 292 / 297 / 289.
constexpr uint32_t STEP_THREADS = 256;
template <bool TICKETS_APART>
__device__ __forceinline__ void adam_body(const AdamLaunch& a, uint32_t block, uint32_t n_blocks) {
    const uint32_t age = *a.age;
    // bias corrections from the un-incremented age (adam/operations_generic.h:49-58)
    float bc1, bc2;
    rlt_adam_bias_corrections(a.p, age, bc1, bc2);
    if constexpr (TICKETS_APART) {
        asm volatile("" :: "v"(bc1), "v"(bc2));      // every thread has read the age ...
        rlt_lds_barrier();                           // ... before the workgroup's ticket is drawn
        if (threadIdx.x >= STEP_THREADS) {
            if (threadIdx.x == STEP_THREADS && rlt_last_through(a.tickets, block, n_blocks) && a.increment_age) *a.age = age + 1;
            return;
        }
    }
    const int ti = tensor_of(a, block);
    const rlt_adam_tensor T = a.t[ti];
    const uint32_t begin = (block - a.first_block[ti]) * a.span[ti], end = begin + min(a.span[ti], T.count - begin);
    const float* __restrict__ const source = a.source + a.source_offset[ti];
    const float scale = a.source_scale[ti], add = a.source_add[ti];
    const bool from_blocks = !TICKETS_APART && a.source;
    float sq = 0.0f;
    if (from_blocks && a.groups > 16) {
        // many blocks: 64 elements per pass of a workgroup, four threads per element each add up a quarter of the blocks (the order of
        // rlt_sum_of_blocks) with all of a quarter's loads of up to 32 blocks in flight at once
        __shared__ float quarter[4][64];
        const uint32_t el = threadIdx.x & 63u, qtr = threadIdx.x >> 6;
        const int per = (a.groups + 3) / 4, g0 = qtr * per, g1 = min(a.groups, g0 + per);
        for (uint32_t base = begin; base < end; base += 64u) {
            const uint32_t j = min(base + el, end - 1u);
            const float* __restrict__ p = source + j;
            // the element's moments and value travel while the blocks are added up
            float m = 0.f, v2 = 0.f, param = 0.f, target = 0.f;
            if (qtr == 0) { m = T.first_moment[j]; v2 = T.second_moment[j]; param = T.parameters[j]; if (T.polyak_target) target = T.polyak_target[j]; }
            float s = 0.f;
            int gb = g0;
            for (; g1 - gb > 8; gb += 32) {
                float v[32];
#pragma unroll
                for (int u = 0; u < 32; u++) v[u] = p[(size_t)min(gb + u, g1 - 1) * a.block_stride];
#pragma unroll
                for (int u = 0; u < 32; u++) s += (gb + u < g1) ? v[u] : 0.f;
            }
            for (; gb < g1; gb += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = p[(size_t)min(gb + u, g1 - 1) * a.block_stride];
#pragma unroll
                for (int u = 0; u < 8; u++) s += (gb + u < g1) ? v[u] : 0.f;
            }
            quarter[qtr][el] = s;
            __syncthreads();
            if (qtr == 0 && base + el < end) {
                const float g = rlt_scaled_sum((quarter[0][el] + quarter[1][el]) + (quarter[2][el] + quarter[3][el]), scale, add);
                T.gradient[j] = g;
                sq += g * g;
                rlt_adam_values(a.p, T.flags, g, bc1, bc2, m, v2, param);
                T.first_moment[j] = m; T.second_moment[j] = v2; T.parameters[j] = param;
                if (T.polyak_target) T.polyak_target[j] = rlt_polyak_value(a.polyak, target, param);
            }
            __syncthreads();
        }
    } else {
    // four neighbouring elements per thread, from their gradient or from at most 16 blocks: every load is 16 bytes per lane (the same sums in the same order per element)
    typedef float f4 __attribute__((ext_vector_type(4)));
    const uint32_t vec_end = (a.vec >> ti & 1u) ? end & ~3u : begin;
    for (uint32_t j = begin + threadIdx.x * 4u; j < vec_end; j += 1024u) {
        f4 m = *reinterpret_cast<const f4*>(T.first_moment + j), v = *reinterpret_cast<const f4*>(T.second_moment + j), param = *reinterpret_cast<const f4*>(T.parameters + j);
        f4 target = {0.f, 0.f, 0.f, 0.f};
        if (T.polyak_target) target = *reinterpret_cast<const f4*>(T.polyak_target + j);
        f4 g;
        if (from_blocks) {
            const float* __restrict__ p = source + j;
            const int per = (a.groups + 3) / 4;
            f4 blk[16];
#pragma unroll
            for (int qi = 0; qi < 4; qi++)
#pragma unroll
                for (int u = 0; u < 4; u++) blk[4 * qi + u] = *reinterpret_cast<const f4*>(p + (size_t)min(qi * per + u, a.groups - 1) * a.block_stride);
            __builtin_amdgcn_sched_barrier(0);
            f4 q[4];
#pragma unroll
            for (int qi = 0; qi < 4; qi++) {
                const int g0 = qi * per, g1 = min(a.groups, g0 + per);
                f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < 4; u++) if (u < per && g0 + u < g1) sum += blk[4 * qi + u];
                q[qi] = sum;
            }
            const f4 total4 = (q[0] + q[1]) + (q[2] + q[3]);
#pragma unroll
            for (int c = 0; c < 4; c++) g[c] = rlt_scaled_sum(total4[c], scale, add);
        } else g = *reinterpret_cast<const f4*>(T.gradient + j);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            sq += g[c] * g[c];
            float mc = m[c], vc = v[c], pc = param[c];
            rlt_adam_values(a.p, T.flags, g[c], bc1, bc2, mc, vc, pc);
            m[c] = mc; v[c] = vc; param[c] = pc;
            if (T.polyak_target) target[c] = rlt_polyak_value(a.polyak, target[c], pc);
        }
        if (from_blocks) *reinterpret_cast<f4*>(T.gradient + j) = g;
        *reinterpret_cast<f4*>(T.first_moment + j) = m; *reinterpret_cast<f4*>(T.second_moment + j) = v; *reinterpret_cast<f4*>(T.parameters + j) = param;
        if (T.polyak_target) *reinterpret_cast<f4*>(T.polyak_target + j) = target;
    }
    for (uint32_t j = vec_end + threadIdx.x; j < end; j += 256u) {
        // the element's moments, value and target travel together with its gradient (or the blocks that add up to it)
        float m = T.first_moment[j], v = T.second_moment[j], param = T.parameters[j];
        const float target = T.polyak_target ? T.polyak_target[j] : 0.f;
        float g;
        if (from_blocks) {
            g = rlt_scaled_sum(sum_of_blocks(source + j, a.groups, a.block_stride), scale, add);
            T.gradient[j] = g;
        } else g = T.gradient[j];
        sq += g * g;
        rlt_adam_values(a.p, T.flags, g, bc1, bc2, m, v, param);
        T.first_moment[j] = m; T.second_moment[j] = v; T.parameters[j] = param;
        if (T.polyak_target) T.polyak_target[j] = rlt_polyak_value(a.polyak, target, param);
    }
    }
    if constexpr (TICKETS_APART) return;
    if (a.extra_out && block == n_blocks - 1 && threadIdx.x == blockDim.x - 1) *a.extra_out = sum_of_blocks(a.source + a.extra_offset, a.groups, a.block_stride) * a.extra_scale;
    if (!a.out_sq_norm) {
        asm volatile("" :: "v"(bc1), "v"(bc2));      // every thread has read the age ...
        rlt_lds_barrier();                           // ... before the workgroup's ticket is drawn; its stores may still be on their way
        if (threadIdx.x == 0 && rlt_last_through(a.tickets, block, n_blocks) && a.increment_age) *a.age = age + 1;
        return;
    }
    // the squared norm: the last workgroup adds the others' sums up, which a fence on both sides of the ticket makes visible to it
    __shared__ float partial[4];
    sq = rlt_wave_sum(sq);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float own = partial[0] + partial[1] + partial[2] + partial[3];
        if (n_blocks == 1) {      // nobody else's sum to wait for
            *a.out_sq_norm = (a.accumulate_norm ? *a.out_sq_norm : 0.0f) + own;
            if (a.increment_age) *a.age = age + 1;
            return;
        }
        a.block_partials[block] = own;
        __threadfence();
        if (rlt_last_through(a.tickets, block, n_blocks)) {
            __threadfence();
            float s = a.accumulate_norm ? *a.out_sq_norm : 0.0f;
            for (uint32_t b = 0; b < n_blocks; b++) s += ((volatile float*)a.block_partials)[b];
            *a.out_sq_norm = s;
            if (a.increment_age) *a.age = age + 1;
        }
    }
}

// not where the workgroup waits for all of its threads later on (the squared norm, sums of many blocks), nor where the gradients are blocks of sums, whose loads take longer than the tickets (a PPO iteration
// whose minibatches leave few blocks 1,452 us without the fifth wavefront, 1,468 with it)
bool tickets_apart(const AdamLaunch& a) { return !a.out_sq_norm && !a.source; }
template <bool TICKETS_APART>
__global__ __launch_bounds__(TICKETS_APART ? STEP_THREADS + 64 : STEP_THREADS) void adam_kernel(AdamLaunch a) { adam_body<TICKETS_APART>(a, blockIdx.x, gridDim.x); }
// two optimisers in one launch: workgroups [0, blocks_a) take the first
template <bool TICKETS_APART>
__global__ __launch_bounds__(TICKETS_APART ? STEP_THREADS + 64 : STEP_THREADS) void adam_pair_kernel(AdamLaunch a, AdamLaunch b, uint32_t blocks_a) {
    if (blockIdx.x < blocks_a) adam_body<TICKETS_APART>(a, blockIdx.x, blocks_a);
    else adam_body<TICKETS_APART>(b, blockIdx.x - blocks_a, gridDim.x - blocks_a);
}

__global__ __launch_bounds__(256) void adam_reset_kernel(AdamLaunch a) {
    const int ti = tensor_of(a, blockIdx.x);
    const rlt_adam_tensor T = a.t[ti];
    const uint32_t begin = (blockIdx.x - a.first_block[ti]) * a.span[ti], end = begin + min(a.span[ti], T.count - begin);
    for (uint32_t j = begin + threadIdx.x; j < end; j += blockDim.x) { T.first_moment[j] = 0.0f; T.second_moment[j] = 0.0f; }
    if (a.increment_age && blockIdx.x == 0 && threadIdx.x == 0) *a.age = 1;
}

__global__ __launch_bounds__(256) void polyak_kernel(const float* __restrict__ source, float* __restrict__ target, size_t count, float polyak, int squared) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
        float s = source[i];
        target[i] = squared ? polyak * target[i] + (1.0f - polyak) * s * s : rlt_polyak_value(polyak, target[i], s);
    }
}

}  // namespace

// Tensors that follow each other in every array (and in the blocks of partial sums) and are stepped alike are one: a network laid out as an arena of parameters, gradients and
// moments is a single tensor, with one ragged end instead of one per layer.
static void join_neighbours(AdamLaunch& a) {
    const uint32_t flags = (a.p.enable_weight_decay ? 1u : 0u) | (a.p.enable_bias_lr_factor ? 2u : 0u);      // those that make a difference
    int n = 0;
    for (int i = 1; i < a.n; i++) {
        rlt_adam_tensor& T = a.t[n];
        const rlt_adam_tensor& U = a.t[i];
        bool follows = T.parameters + T.count == U.parameters && T.gradient + T.count == U.gradient && T.first_moment + T.count == U.first_moment &&
                       T.second_moment + T.count == U.second_moment && (T.polyak_target ? T.polyak_target + T.count == U.polyak_target : !U.polyak_target) &&
                       ((T.flags ^ U.flags) & flags) == 0;
        if (a.source)
            follows = follows && a.source_offset[n] + T.count == a.source_offset[i] && a.source_scale[n] == a.source_scale[i] && a.source_add[n] == a.source_add[i];
        if (follows) { T.count += U.count; continue; }
        n++;
        a.t[n] = U;
        a.source_offset[n] = a.source_offset[i]; a.source_scale[n] = a.source_scale[i]; a.source_add[n] = a.source_add[i];
    }
    a.n = n + 1;
}
// Deals the tensors out to at most about `most` workgroups and returns their number: 64 elements per workgroup pass where many blocks are added up, four per thread
// where pointers, place in the blocks and block size are multiples of 16 bytes, one otherwise.
static uint32_t deal_out(AdamLaunch& a, uint32_t most) {
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const bool many = a.source && a.groups > 16;
    const bool source_ok = !a.source || (a.block_stride % 4 == 0 && aligned(a.source));
    uint64_t passes = 0;
    a.vec = 0;
    for (int i = 0; i < a.n; i++) {
        const rlt_adam_tensor& T = a.t[i];
        const bool vec = !many && source_ok && (!a.source || a.source_offset[i] % 4 == 0) && aligned(T.parameters) && aligned(T.gradient) && aligned(T.first_moment) &&
                         aligned(T.second_moment) && (!T.polyak_target || aligned(T.polyak_target));
        if (vec) a.vec |= 1u << i;
        a.span[i] = many ? 64u : vec ? 1024u : 256u;
        passes += (T.count + (uint64_t)a.span[i] - 1) / a.span[i];
    }
    const uint32_t rounds = (uint32_t)((passes + most - 1) / most);
    uint32_t blocks = 0;
    for (int i = 0; i < a.n; i++) {
        a.first_block[i] = blocks;
        if (rounds > 1) a.span[i] *= rounds;
        blocks += (uint32_t)((a.t[i].count + (uint64_t)a.span[i] - 1) / a.span[i]);
    }
    for (int i = a.n; i <= MAX_T; i++) a.first_block[i] = blocks;
    return blocks;
}

static void launch_adam(rlt_rocm_device* device, const AdamLaunch& a, uint32_t blocks) {
    if (tickets_apart(a)) hipLaunchKernelGGL(adam_kernel<true>, dim3(blocks), dim3(STEP_THREADS + 64), 0, device->stream, a);
    else hipLaunchKernelGGL(adam_kernel<false>, dim3(blocks), dim3(STEP_THREADS), 0, device->stream, a);
}
// [256, 4096) of the device handle's counters block hold the workgroups' sums for the squared norm
static int adam_launch(rlt_rocm_device* device, const rlt_adam_tensor* tensors, int n_tensors, const rlt_adam_parameters* p, uint32_t* age,
                       float polyak, float* out_sq_norm, bool reset) {
    void* counters = nullptr;
    int rc = rlt_counters(device, &counters);
    if (rc) return rc;
    for (int base = 0; base < n_tensors; base += MAX_T) {
        AdamLaunch a = {};
        a.n = n_tensors - base < MAX_T ? n_tensors - base : MAX_T;
        for (int i = 0; i < a.n; i++) {
            const rlt_adam_tensor& T = tensors[base + i];
            if (!T.first_moment || !T.second_moment || (!reset && (!T.parameters || !T.gradient)) || T.count == 0) return RLT_E_INVALID_ARGUMENT;
            a.t[i] = T;
        }
        if (p) a.p = *p;
        a.polyak = polyak; a.age = age;
        a.tickets = rlt_tickets_of(counters, 0); a.block_partials = (float*)((char*)counters + 256);
        a.out_sq_norm = out_sq_norm; a.accumulate_norm = base > 0;
        a.increment_age = (base + MAX_T >= n_tensors);
        if (!reset) join_neighbours(a);
        const uint32_t blocks = deal_out(a, MAX_BLOCKS);
        if (reset) hipLaunchKernelGGL(adam_reset_kernel, dim3(blocks), dim3(256), 0, device->stream, a);
        else launch_adam(device, a, blocks);
        if ((rc = rlt_launch_status(device))) return rc;
    }
    return 0;
}

static void set_source(AdamLaunch& a, const rlt_adam_source* source) {
    if (!source) return;
    a.source = source->partial; a.groups = source->groups; a.block_stride = source->block_stride;
    for (int i = 0; i < a.n; i++) { a.source_offset[i] = source->offsets[i]; a.source_scale[i] = source->scales[i]; a.source_add[i] = source->adds ? source->adds[i] : 0.0f; }
    a.extra_out = source->extra_out; a.extra_offset = source->extra_offset; a.extra_scale = source->extra_scale;
}
int rlt_adam_step_from_partials(rlt_rocm_device* device, const rlt_adam_tensor* tensors, int n, const rlt_adam_parameters* parameters, uint32_t* age, const rlt_adam_source* source, float polyak) {
    RLT_REQUIRE(tensors && n > 0 && n <= MAX_T && parameters && age && source && source->partial && source->groups > 0);
    void* counters = nullptr;
    int rc = rlt_counters(device, &counters);
    if (rc) return rc;
    AdamLaunch a = {};
    a.n = n;
    for (int i = 0; i < n; i++) {
        const rlt_adam_tensor& T = tensors[i];
        if (!T.first_moment || !T.second_moment || !T.parameters || !T.gradient || T.count == 0) return RLT_E_INVALID_ARGUMENT;
        a.t[i] = T;
    }
    a.p = *parameters; a.age = age; a.polyak = polyak;
    a.tickets = rlt_tickets_of(counters, 0); a.block_partials = (float*)((char*)counters + 256);
    a.increment_age = 1;
    set_source(a, source);
    join_neighbours(a);
    const uint32_t blocks = deal_out(a, MAX_BLOCKS);
    launch_adam(device, a, blocks);
    return rlt_launch_status(device);
}

int rlt_adam_step_pair(rlt_rocm_device* device, const rlt_adam_tensor* tensors_a, int n_a, const rlt_adam_parameters* parameters_a, uint32_t* age_a,
                       const rlt_adam_tensor* tensors_b, int n_b, const rlt_adam_parameters* parameters_b, uint32_t* age_b,
                       const rlt_adam_source* source_a, const rlt_adam_source* source_b, float polyak) {
    RLT_REQUIRE(tensors_a && tensors_b && n_a > 0 && n_b > 0 && parameters_a && parameters_b && age_a && age_b);
    if (n_a > MAX_T || n_b > MAX_T || (age_a == age_b && !source_a && !source_b)) {      // (optimisers that share an age: the second steps with the age that the first leaves)
        RLT_REQUIRE(!source_a && !source_b);
        const int rc = adam_launch(device, tensors_a, n_a, parameters_a, age_a, 0.0f, nullptr, false);
        return rc ? rc : adam_launch(device, tensors_b, n_b, parameters_b, age_b, 0.0f, nullptr, false);
    }
    void* counters = nullptr;
    int rc = rlt_counters(device, &counters);
    if (rc) return rc;
    AdamLaunch L[2] = {};
    uint32_t blocks[2];
    for (int k = 0; k < 2; k++) {
        AdamLaunch& a = L[k];
        const rlt_adam_tensor* tensors = k ? tensors_b : tensors_a;
        a.n = k ? n_b : n_a;
        for (int i = 0; i < a.n; i++) {
            const rlt_adam_tensor& T = tensors[i];
            if (!T.first_moment || !T.second_moment || !T.parameters || !T.gradient || T.count == 0) return RLT_E_INVALID_ARGUMENT;
            a.t[i] = T;
        }
        a.p = k ? *parameters_b : *parameters_a;
        a.age = k ? age_b : age_a; a.polyak = polyak;
        // the second optimiser's tickets and partial sums sit in their own part of the counters block
        a.tickets = rlt_tickets_of(counters, k); a.block_partials = (float*)((char*)counters + 256) + (k ? 480 : 0);
        a.increment_age = 1;
        const rlt_adam_source* source = k ? source_b : source_a;
        set_source(a, source);
        join_neighbours(a);
        blocks[k] = deal_out(a, MAX_BLOCKS / 2);
    }
    const dim3 grid(blocks[0] + blocks[1]);
    if (tickets_apart(L[0]) && tickets_apart(L[1])) hipLaunchKernelGGL(adam_pair_kernel<true>, grid, dim3(STEP_THREADS + 64), 0, device->stream, L[0], L[1], blocks[0]);
    else hipLaunchKernelGGL(adam_pair_kernel<false>, grid, dim3(STEP_THREADS), 0, device->stream, L[0], L[1], blocks[0]);
    return rlt_launch_status(device);
}

extern "C" {

int rlt_rocm_adam_step(rlt_rocm_device* device, const rlt_adam_tensor* tensors_host, int n_tensors, const rlt_adam_parameters* parameters_host,
                       uint32_t* age, float polyak, float* out_gradient_squared_norm) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(tensors_host && n_tensors > 0 && parameters_host && age);
    return adam_launch(device, tensors_host, n_tensors, parameters_host, age, polyak, out_gradient_squared_norm, false);
}
int rlt_rocm_adam_reset(rlt_rocm_device* device, const rlt_adam_tensor* tensors_host, int n_tensors, uint32_t* age) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(tensors_host && n_tensors > 0 && age);
    return adam_launch(device, tensors_host, n_tensors, nullptr, age, 0.0f, nullptr, true);
}
int rlt_rocm_polyak_update(rlt_rocm_device* device, const float* source, float* target, size_t count, float polyak, int squared) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(source && target);
    if (count == 0) return 0;
    size_t b = (count + 255) / 256; if (b > 960) b = 960;
    hipLaunchKernelGGL(polyak_kernel, dim3((int)b), dim3(256), 0, device->stream, source, target, count, polyak, squared);
    return rlt_launch_status(device);
}

}  // extern "C"
