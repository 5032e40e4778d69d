// GRU layer: forward with kept intermediates and backward through time.
// reference: nn/layers/gru/operations_generic.h:231-341 (evaluate / forward), :594-795 (_backward per step, from the last step to the
// first). The reference walks the sequence on the host and issues a handful of small tensor operations per step.
//
// Here the work is split by what depends on time:
//   * W_i x + b_i for ALL steps is one contraction over sequence*batch rows (gemm.hip), written straight into post_activation (at hidden width 64 and up to a thousand rows mostly
//     formed beside the recurrence, inputs_beside);
//   * the recurrence runs in ONE launch: batch rows are independent, so no grid-wide synchronisation is needed. At hidden width 64 a
//     workgroup carries four rows through the sequence on the matrix cores, at 16 and 32 a wavefront 64 / width rows on the vector units, both with W_h in registers; where there are few rows for the
//     compute units (two to five each, backward from a number of steps on: rows_forward(), rows_backward()) a workgroup carries one row on the vector units at all three widths; at other
//     widths a workgroup owns a few rows and keeps W_h and its rows' hidden state in LDS;
//   * backward does the same in reverse and stores, per step, the gradient at the gate pre-activations (one copy as the input path sees
//     it, one as the hidden path sees it, which differs in the n gate by the factor r) and the previous hidden state; the weight
//     gradients and d_input are then three contractions over sequence*batch rows (the weight gradients, too, mostly beside the recurrence where that is one workgroup per compute unit,
//     weights_beside).
#include "common.h"
#include "gemm.h"
#include <utility>

namespace {

constexpr int GRU_THREADS = 256;

struct GruArgs {
    rlt_gru_layer L;
    const float* input; const uint8_t* reset;
    float* d_output; float* buffer_input; float* buffer_hidden; float* h_previous; float* db_hn_partial; float* blocks;
    int S, B, rows_per_group;
};

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }
// the gate functions; fast = the rational approximations of math/operations_generic.h:247-255 (a wavefront-uniform switch)
__device__ __forceinline__ float gate_sigmoid(float x, int fast) { return fast ? 0.5f * rlt_fast_tanh(0.5f * x) + 0.5f : sigmoidf_(x); }
__device__ __forceinline__ float gate_tanh(float x, int fast) { return fast ? rlt_fast_tanh(x) : tanhf(x); }

// post_activation holds W_i x + b_i on entry. Thread (row, j): hidden unit j of one batch row.
__global__ __launch_bounds__(GRU_THREADS) void gru_forward_kernel(GruArgs A) {
    extern __shared__ float lds[];
    const int H = A.L.hidden_dim, H3 = 3 * H, R = A.rows_per_group;
    float* wt = lds;                 // W_h transposed: wt[k * 3H + j]
    float* hs = wt + (size_t)H3 * H; // hidden state of the workgroup's rows
    for (int i = threadIdx.x; i < H3 * H; i += blockDim.x) { const int j = i / H, k = i - j * H; wt[k * H3 + j] = A.L.weights_hidden[i]; }
    const int row = threadIdx.x / H, j = threadIdx.x - row * H, b = blockIdx.x * R + row;
    const bool active = row < R && b < A.B;
    const float bhr = active ? A.L.biases_hidden[j] : 0.f, bhz = active ? A.L.biases_hidden[H + j] : 0.f, bhn = active ? A.L.biases_hidden[2 * H + j] : 0.f;
    const float h0 = active ? A.L.initial_hidden_state[j] : 0.f;
    float h = h0;
    for (int t = 0; t < A.S; t++) {
        if (active) {
            if (t == 0 || (A.reset && A.reset[(size_t)t * A.B + b])) h = h0;
            hs[row * H + j] = h;
        }
        __syncthreads();
        if (active) {
            float ar = bhr, az = bhz, an = bhn;
            const float* hr = hs + row * H;
            for (int k = 0; k < H; k++) { const float hk = hr[k]; const float* w = wt + k * H3; ar += hk * w[j]; az += hk * w[H + j]; an += hk * w[2 * H + j]; }
            float* post = A.L.post_activation + ((size_t)t * A.B + b) * H3;
            const float r = gate_sigmoid(post[j] + ar, A.L.fast_tanh), z = gate_sigmoid(post[H + j] + az, A.L.fast_tanh);
            const float n = gate_tanh(post[2 * H + j] + an * r, A.L.fast_tanh);
            post[j] = r; post[H + j] = z; post[2 * H + j] = n;
            A.L.n_pre_pre_activation[((size_t)t * A.B + b) * H + j] = an;
            h = (1.0f - z) * n + z * h;
            A.L.output[((size_t)t * A.B + b) * H + j] = h;
        }
        __syncthreads();
    }
}

// Reverse pass. Thread (row, j). d_output is accumulated into in place as in the reference.
__global__ __launch_bounds__(GRU_THREADS) void gru_backward_kernel(GruArgs A) {
    extern __shared__ float lds[];
    const int H = A.L.hidden_dim, H3 = 3 * H, R = A.rows_per_group;
    float* w = lds;                          // W_h row-major: w[j * H + k]
    float* bs = w + (size_t)H3 * H;          // hidden-path gate gradients of the workgroup's rows: bs[row * 3H + j]
    for (int i = threadIdx.x; i < H3 * H; i += blockDim.x) w[i] = A.L.weights_hidden[i];
    const int row = threadIdx.x / H, j = threadIdx.x - row * H, b = blockIdx.x * R + row;
    const bool active = row < R && b < A.B;
    const float h0 = active ? A.L.initial_hidden_state[j] : 0.f;
    float carry = 0.f;       // gradient arriving at this step's hidden state from the step after it
    float db_hn = 0.f;
    __syncthreads();
    for (int t = A.S - 1; t >= 0; t--) {
        bool from_initial = true;
        if (active) {
            const size_t at = (size_t)t * A.B + b;
            from_initial = t == 0 || (A.reset && A.reset[at]);
            const float* post = A.L.post_activation + at * H3;
            const float r = post[j], z = post[H + j], n = post[2 * H + j];
            const float hp = from_initial ? h0 : A.L.output[((size_t)(t - 1) * A.B + b) * H + j];
            const float dh = A.d_output[at * H + j] + carry;
            A.d_output[at * H + j] = dh;
            const float gz = dh * (hp - n) * z * (1.0f - z);
            const float gn = dh * (1.0f - z) * (1.0f - n * n);
            const float gr = gn * A.L.n_pre_pre_activation[at * H + j] * r * (1.0f - r);
            float* bi = A.buffer_input + at * H3; float* bh = A.buffer_hidden + at * H3;
            bi[j] = gr; bi[H + j] = gz; bi[2 * H + j] = gn;
            bh[j] = gr; bh[H + j] = gz; bh[2 * H + j] = gn * r;
            A.h_previous[at * H + j] = hp;
            bs[row * H3 + j] = gr; bs[row * H3 + H + j] = gz; bs[row * H3 + 2 * H + j] = gn * r;
            // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
            if (!(t > 0 && from_initial)) db_hn += gn * r;
            carry = from_initial ? 0.f : dh * z;
        }
        __syncthreads();
        if (active && !from_initial) {
            float acc = 0.f;
            const float* br = bs + row * H3;
            for (int jj = 0; jj < H3; jj++) acc += br[jj] * w[jj * H + j];       // d h_prev[j] += sum over gates of buffer * W_h[., j]
            carry += acc;
        }
        __syncthreads();
    }
    if (active && A.db_hn_partial) A.db_hn_partial[(size_t)b * H + j] = db_hn;
}

// ---- hidden widths 32 and 16: W_h in registers, no workgroup barrier -----------------------------------------------------------
// A wavefront carries 64 / H batch rows; lane (row, j) owns hidden unit j of its row and keeps rows j, H + j, 2H + j of W_h (3H values) in
// registers for the whole sequence. The previous hidden state reaches the lanes of its row through a 64-float slot of LDS private to the wavefront
// (one write, H / 4 broadcast reads of four values); a step needs no workgroup barrier, and the wavefronts of a workgroup are independent (they only
// share the launch). Rows beyond the batch repeat the last row, which the same wavefront holds: they read, compute and store the same values.
// Bound: the chain of a step. What it reads is requested four steps ahead into registers that the unrolled loop names (as a queue whose entries move up it waited for
// each step's own request), a wavefront reads 64 reset flags at a time. Whole model step of 64 x 16 sequences, width 16: 111 -> 99 us, 63 x 1,000: 200 -> 188 us; width 32,
// where the 96 multiply-adds of a step hide the requests: 131.2 -> 129.7 us (64 x 64), 257 -> 254 us (64 x 1,024).
// lanes of one wavefront exchange data through LDS: the hardware executes a wavefront's LDS instructions in order, the fences keep the
// compiler from moving them across
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The steps of a sequence in groups of D whose members know their number in the group (a queue's entries are indexed by it). Whole groups are straight-line code: with an
// exit before every step the compiler waits for all requests where the paths meet. For the same reason everything requested before the loop is waited for in front of it: the
// first step of a group then waits for its own values, requested D steps before, and not for the last ones.
template <class F, int... K> __device__ __forceinline__ void gru_whole_group(int first, F& step, std::integer_sequence<int, K...>) { (step(std::integral_constant<int, K>{}, first + K), ...); }
template <class F, int... K> __device__ __forceinline__ void gru_rest(int first, int S, F& step, std::integer_sequence<int, K...>) { ((first + K < S ? step(std::integral_constant<int, K>{}, first + K) : (void)0), ...); }
template <int D, class F>
__device__ __forceinline__ void gru_steps(int S, F&& step) {
    int i = 0;
    __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
    for (; i + D <= S; i += D) gru_whole_group(i, step, std::make_integer_sequence<int, D>{});
    gru_rest(i, S, step, std::make_integer_sequence<int, D - 1>{});
}

// Reset flags of 64 consecutive steps from `first` on, as a mask in every lane of the row's group (bit i: step first + i starts an episode); steps from S on: no. A wavefront
// reads a step per lane: a byte load per step would hold the recurrence up for its widening.
template <int ROWS>
__device__ __forceinline__ uint64_t gru_reset_flags(const uint8_t* reset, int first, int S, int B, int b0, int mine) {
    if (!reset) return 0;
    const int t = first + (int)(threadIdx.x & 63);
    uint64_t mask = 0;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const uint64_t row = __ballot(t < S && reset[(size_t)min(t, S - 1) * B + min(b0 + r, B - 1)] != 0);
        mask = mine == r ? row : mask;
    }
    return mask;
}
__device__ __forceinline__ float& gru_at(float* base, unsigned bytes) { return *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + bytes); }

template <int H, bool FAST>
__global__ __launch_bounds__(GRU_THREADS) void gru_forward_reg_kernel(GruArgs A) {
    constexpr int G = 64 / H, D = 4;                        // batch rows per wavefront; steps ahead that the inputs W_i x + b_i are requested
    __shared__ __align__(16) float exchange[GRU_THREADS / 64][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), row_base = lane & ~(H - 1);
    const int b0 = (blockIdx.x * (GRU_THREADS / 64) + wave) * G;
    if (b0 >= A.B) return;                                  // whole wavefronts; no barrier follows
    const int row = min(lane / H, A.B - 1 - b0);
    float wr[H], wz[H], wn[H];
    {
        const float4* r4 = reinterpret_cast<const float4*>(A.L.weights_hidden + (size_t)u * H);
        const float4* z4 = reinterpret_cast<const float4*>(A.L.weights_hidden + (size_t)(H + u) * H);
        const float4* n4 = reinterpret_cast<const float4*>(A.L.weights_hidden + (size_t)(2 * H + u) * H);
#pragma unroll
        for (int q = 0; q < H / 4; q++) {
            const float4 a = r4[q], c = z4[q], d = n4[q];
            wr[4 * q] = a.x; wr[4 * q + 1] = a.y; wr[4 * q + 2] = a.z; wr[4 * q + 3] = a.w;
            wz[4 * q] = c.x; wz[4 * q + 1] = c.y; wz[4 * q + 2] = c.z; wz[4 * q + 3] = c.w;
            wn[4 * q] = d.x; wn[4 * q + 1] = d.y; wn[4 * q + 2] = d.z; wn[4 * q + 3] = d.w;
        }
    }
    const float bhr = A.L.biases_hidden[u], bhz = A.L.biases_hidden[H + u], bhn = A.L.biases_hidden[2 * H + u];
    const float h0 = A.L.initial_hidden_state[u];
    const size_t stride = (size_t)A.B * H;
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    float* post = A.L.post_activation + (size_t)b0 * 3 * H; float* npp = A.L.n_pre_pre_activation + (size_t)b0 * H; float* out = A.L.output + (size_t)b0 * H;
    struct In { float r, z, n; };
    float* in = post;
    auto request = [&](int t, In& v) {      // in the order of the steps; the last steps request the last one again: no branch around the loads
        v.r = gru_at(in, at3); v.z = gru_at(in + H, at3); v.n = gru_at(in + 2 * H, at3);
        in += t + 1 < A.S ? 3 * stride : 0;
    };
    In q[D];
#pragma unroll
    for (int d = 0; d < D; d++) request(d, q[d]);
    float* const xw = exchange[wave];
    float h = h0;
    for (int first = 0; first < A.S; first += 64) {
        uint64_t flags = gru_reset_flags<G>(A.reset, first + 1, A.S, A.B, b0, lane / H);      // of the steps after these
        gru_steps<D>(min(64, A.S - first), [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);      // later steps' values are not touched (and waited for) before their step
            float ar = bhr, az = bhz, an = bhn;
            xw[lane] = h;
            wave_sync();
#pragma unroll
            for (int k = 0; k < H; k += 4) {
                const float4 hv = *reinterpret_cast<const float4*>(xw + row_base + k);
                ar += hv.x * wr[k]; az += hv.x * wz[k]; an += hv.x * wn[k];
                ar += hv.y * wr[k + 1]; az += hv.y * wz[k + 1]; an += hv.y * wn[k + 1];
                ar += hv.z * wr[k + 2]; az += hv.z * wz[k + 2]; an += hv.z * wn[k + 2];
                ar += hv.w * wr[k + 3]; az += hv.w * wz[k + 3]; an += hv.w * wn[k + 3];
            }
            wave_sync();
            const float r = gate_sigmoid(q[N].r + ar, FAST), z = gate_sigmoid(q[N].z + az, FAST);
            const float n = gate_tanh(q[N].n + an * r, FAST);
            const float o = (1.0f - z) * n + z * h;
            h = flags & 1 ? h0 : o;       // the next step starts an episode
            flags >>= 1;
            gru_at(post, at3) = r; gru_at(post + H, at3) = z; gru_at(post + 2 * H, at3) = n; gru_at(npp, at) = an; gru_at(out, at) = o;
            post += 3 * stride; npp += stride; out += stride;
            request(first + i + D, q[N]);      // behind the last use of the entry
        });
    }
}

// Reverse pass at these widths: lane (row, k) keeps column k of W_h (the 3H weights that multiply the gate gradients on the way to
// d h_prev[k]); the gate gradients of the row's H units reach its lanes through three 64-float slots of LDS private to the wavefront.
template <int H>
__global__ __launch_bounds__(GRU_THREADS) void gru_backward_reg_kernel(GruArgs A) {
    // D: steps ahead that a step's saved values are requested (width 32, 64 x 64 sequences: 45.6 us with four, 45.0 with three, 47.9 with two). BLOCK: steps whose reset flags are
    // read at once, whole groups of D, so that the queue's entries keep their places from block to block
    constexpr int G = 64 / H, D = H == 32 ? 3 : 4, BLOCK = 64 / D * D;
    __shared__ __align__(16) float exchange[GRU_THREADS / 64][3][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), row_base = lane & ~(H - 1), S = A.S;
    const int b0 = (blockIdx.x * (GRU_THREADS / 64) + wave) * G;
    if (b0 >= A.B) return;
    const int row = min(lane / H, A.B - 1 - b0);
    float cr[H], cz[H], cn[H];
#pragma unroll
    for (int j = 0; j < H; j++) {
        cr[j] = A.L.weights_hidden[(size_t)j * H + u]; cz[j] = A.L.weights_hidden[(size_t)(H + j) * H + u]; cn[j] = A.L.weights_hidden[(size_t)(2 * H + j) * H + u];
    }
    const float h0 = A.L.initial_hidden_state[u];
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    const size_t stride = (size_t)A.B * H, last = (size_t)(S - 1) * stride + (size_t)b0 * H;
    struct Saved { float r, z, n, npp, dy, hp; };
    float *post = A.L.post_activation + 3 * last, *npp = A.L.n_pre_pre_activation + last, *dy = A.d_output + last, *state = A.L.output + last;
    auto request = [&](int i, Saved& v) {      // i-th step from the end; steps before the first read the first again; the state is the one before the step (the first step's is not used)
        const size_t on = i + 1 < S ? stride : 0;
        state -= on;
        v.r = gru_at(post, at3); v.z = gru_at(post + H, at3); v.n = gru_at(post + 2 * H, at3); v.npp = gru_at(npp, at); v.dy = gru_at(dy, at); v.hp = gru_at(state, at);
        post -= 3 * on; npp -= on; dy -= on;
    };
    Saved q[D];
#pragma unroll
    for (int d = 0; d < D; d++) request(d, q[d]);
    float *to_dy = A.d_output + last, *to_hp = A.h_previous + last, *bi = A.buffer_input + 3 * last, *bh = A.buffer_hidden + 3 * last;
    float* const xw = &exchange[wave][0][0];
    float carry = 0.f, db_hn = 0.f;
    for (int back = 0; back < S; back += BLOCK) {
        const int steps = min(BLOCK, S - back);
        const uint64_t flags = gru_reset_flags<G>(A.reset, S - back - steps, S, A.B, b0, lane / H);      // bit of step t = S - 1 - back - i: steps - 1 - i
        uint64_t high = flags << (64 - steps);
        gru_steps<D>(steps, [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);
            const Saved cur = q[N];
            const bool first = back + i + 1 == S, from_initial = first || (high >> 63);
            high <<= 1;
            const float hp = from_initial ? h0 : cur.hp;
            const float dh = cur.dy + carry;
            const float gz = dh * (hp - cur.n) * cur.z * (1.0f - cur.z);
            const float gn = dh * (1.0f - cur.z) * (1.0f - cur.n * cur.n);
            const float gr = gn * cur.npp * cur.r * (1.0f - cur.r);
            const float gnr = gn * cur.r;
            xw[lane] = gr; xw[64 + lane] = gz; xw[128 + lane] = gnr;
            // the rows of one wavefront restart at different steps: every lane forms the sum, a restarting row drops it
            float a0 = dh * cur.z, a1 = 0.f, a2 = 0.f;
            asm volatile("" : "+v"(a0));      // (not formed below by a multiply-add that would keep the entry's z)
            request(back + i + D, q[N]);      // behind the last use of the entry
            gru_at(to_dy, at) = dh; gru_at(to_hp, at) = hp;
            gru_at(bi, at3) = gr; gru_at(bi + H, at3) = gz; gru_at(bi + 2 * H, at3) = gn;
            gru_at(bh, at3) = gr; gru_at(bh + H, at3) = gz; gru_at(bh + 2 * H, at3) = gnr;
            to_dy -= stride; to_hp -= stride; bi -= 3 * stride; bh -= 3 * stride;
            // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
            db_hn += first || !from_initial ? gnr : 0.f;
            wave_sync();
#pragma unroll
            for (int j = 0; j < H; j += 4) {
                const float4 vr = *reinterpret_cast<const float4*>(xw + row_base + j), vz = *reinterpret_cast<const float4*>(xw + 64 + row_base + j),
                             vn = *reinterpret_cast<const float4*>(xw + 128 + row_base + j);
                a0 += vr.x * cr[j]; a1 += vz.x * cz[j]; a2 += vn.x * cn[j];
                a0 += vr.y * cr[j + 1]; a1 += vz.y * cz[j + 1]; a2 += vn.y * cn[j + 1];
                a0 += vr.z * cr[j + 2]; a1 += vz.z * cz[j + 2]; a2 += vn.z * cn[j + 2];
                a0 += vr.w * cr[j + 3]; a1 += vz.w * cz[j + 3]; a2 += vn.w * cn[j + 3];
            }
            wave_sync();
            carry = from_initial ? 0.f : a0 + (a1 + a2);
        });
    }
    if (A.db_hn_partial) gru_at(A.db_hn_partial + (size_t)b0 * H, at) = db_hn;
}

// ---- hidden width 64: the recurrence on the matrix cores -------------------------------------------------------------------------
// A workgroup of four wavefronts carries FOUR batch rows through the sequence; wavefront w owns hidden units 16 w ... 16 w + 15, W_h stays in
// registers as the B operand of v_mfma_f32_4x4x1_16b_f32 (16 blocks of a 4 x 1 by 1 x 4 product: lane 4 blk + i supplies A[i], lane 4 blk + j
// supplies B[j], register i of lane 4 blk + j receives D[i][j]; with the broadcast control set to 4 blocks every block of a group of four takes
// its A from the group's block that the instruction names). The four rows are the A side. Block 4 kg + cg takes columns 4 cg ... 4 cg + 3 of the
// wavefront's sixteen and quarter kg of the reduction, so all four columns of every block work: 48 instructions of 8 cycles for the 4 x 192 x 64
// products (with a block per unit and its gates as columns the fourth column is idle: 64). The quarters' sums meet in three lane exchanges and
// three additions that leave row kg in the lanes of group kg: lane = (row, unit) finishes its unit with no trip through LDS.
//
// Bound: the chain of a step -- barrier and one 16-byte LDS read (the state, in the order of the A operand), the matrix instructions, the lane
// exchanges, the gates -- at any batch size up to one workgroup per compute unit. What a step reads from memory is requested D steps ahead into
// registers that the unrolled loop names: as a queue whose entries move up, the compiler waits for every step's own request (and all stores
// before it) at that step's end. 64 steps at batch 64: forward 50.4 -> 35.9 us, backward 52.7 -> 35.3 us (batch 1,024: 56.4 -> 41.4 and 56.1 -> 43.8).
//
// The gates at this width on the hardware's exponential and reciprocal (v_exp_f32, v_rcp_f32: 1 ulp each; the reciprocal corrected by one
// Newton step; absolute error of a gate below 3e-7, an order below the tolerance the layer is held to): the library routines cost 500 cycles of
// a step, these 150.
__device__ __forceinline__ float corrected_rcp(float d) {      // 1 / d for d >= 1; infinite d gives 0, a NaN stays one
    const float q = __builtin_amdgcn_rcpf(d), better = fmaf(fmaf(-d, q, 1.0f), q, q);
    return d == INFINITY ? 0.0f : better;
}
__device__ __forceinline__ float hw_sigmoid(float x) { return corrected_rcp(1.0f + __expf(-x)); }
__device__ __forceinline__ float hw_tanh(float x) { return fmaf(-2.0f, corrected_rcp(__expf(2.0f * x) + 1.0f), 1.0f); }
typedef float gru_floatx4 __attribute__((ext_vector_type(4)));
typedef float gru_float4_a4 __attribute__((ext_vector_type(4), aligned(4)));      // four floats wherever they lie: rows of W_i start at any multiple of four bytes
constexpr int GM_ROWS = 4;
template <int ABID> __device__ __forceinline__ gru_floatx4 mfma4(float a, float b, gru_floatx4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 2, ABID, 0); }
// The four quarters of the reduction added up: c[row] of a lane in group kg (lanes 16 kg ...) is row `row`'s sum over quarter kg; the result is row kg's sum over all of them
__device__ __forceinline__ float sum_quarters(gru_floatx4 c) {
    auto across = [](float a, float b, auto swap) { const auto s = swap(__float_as_uint(a), __float_as_uint(b)); return __uint_as_float(s[0]) + __uint_as_float(s[1]); };
    auto swap32 = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
    auto swap16 = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
    return across(across(c[0], c[2], swap32), across(c[1], c[3], swap32), swap16);
}
// hs (two copies, by the parity of the step): the previous hidden state of the four rows in the order of the A operand: group kg's lane (cg, row) reads
// units 16 kg + 4 s + cg, s = 0 ... 3, in one 16-byte read. One workgroup barrier per step. Lane = (row kg, unit) finishes its unit; rows beyond the batch repeat the last
// row (the same wavefront's lanes hold it: they read, compute and store the same values). Memory is addressed by pointers of the workgroup that move from step to step and
// the lane's place within four rows.
template <bool FAST>
__global__ __launch_bounds__(256, 2) void gru_forward_mfma_kernel(GruArgs A) {
    constexpr int H = 64, D = 4;
    __shared__ __align__(16) float hs[2][H * GM_ROWS];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, c16 = lane & 15, u = 16 * w + c16;
    // B operand: column c16 (unit u) of gate g, reduction index 16 kg + 4 s + abid = 16 kg + k
    float wb[3][16];
#pragma unroll
    for (int g = 0; g < 3; g++) {
        const float4* src = reinterpret_cast<const float4*>(A.L.weights_hidden + (size_t)(g * H + u) * H + 16 * kg);
#pragma unroll
        for (int q = 0; q < 4; q++) { const float4 v = src[q]; wb[g][4 * q] = v.x; wb[g][4 * q + 1] = v.y; wb[g][4 * q + 2] = v.z; wb[g][4 * q + 3] = v.w; }
    }
    const int b0 = blockIdx.x * GM_ROWS, row = min(kg, A.B - 1 - b0);
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    const float bhr = A.L.biases_hidden[u], bhz = A.L.biases_hidden[H + u], bhn = A.L.biases_hidden[2 * H + u];
    const float h0 = A.L.initial_hidden_state[u];
    const size_t stride = (size_t)A.B * H;
    float* post = A.L.post_activation + (size_t)b0 * 3 * H; float* npp = A.L.n_pre_pre_activation + (size_t)b0 * H; float* out = A.L.output + (size_t)b0 * H;
    struct In { float r, z, n; };
    float* in = post;
    auto request = [&](int t, In& v) {      // in the order of the steps; the last steps request the last one again: no branch around the loads
        v.r = gru_at(in, at3); v.z = gru_at(in + H, at3); v.n = gru_at(in + 2 * H, at3);
        in += t + 1 < A.S ? 3 * stride : 0;
    };
    In q[D];
#pragma unroll
    for (int d = 0; d < D; d++) if (d < A.S) request(d, q[d]);
    const int place = ((4 * w + (c16 & 3)) * 4 + kg) * 4 + (c16 >> 2);      // this (row, unit) in hs
    float h = h0;
    hs[0][place] = h;
    for (int first = 0; first < A.S; first += 64) {
        uint64_t flags = gru_reset_flags<GM_ROWS>(A.reset, first + 1, A.S, A.B, b0, kg);      // of the steps after these
        gru_steps<D>(min(64, A.S - first), [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);      // later steps' values are not touched (and waited for) before their step
            rlt_lds_barrier();
            const float4 a = *reinterpret_cast<const float4*>(&hs[N & 1][4 * lane]);
            const float xr = q[N].r + bhr, xz = q[N].z + bhz, xn = q[N].n;
            gru_floatx4 cr = {0.f, 0.f, 0.f, 0.f}, cz = cr, cn = cr;
#define RLT_GRU_STEPS(X, s) \
            cr = mfma4<0>(X, wb[0][4 * s], cr); cn = mfma4<0>(X, wb[2][4 * s], cn); cz = mfma4<0>(X, wb[1][4 * s], cz); \
            cr = mfma4<1>(X, wb[0][4 * s + 1], cr); cn = mfma4<1>(X, wb[2][4 * s + 1], cn); cz = mfma4<1>(X, wb[1][4 * s + 1], cz); \
            cr = mfma4<2>(X, wb[0][4 * s + 2], cr); cn = mfma4<2>(X, wb[2][4 * s + 2], cn); cz = mfma4<2>(X, wb[1][4 * s + 2], cz); \
            cr = mfma4<3>(X, wb[0][4 * s + 3], cr); cn = mfma4<3>(X, wb[2][4 * s + 3], cn); cz = mfma4<3>(X, wb[1][4 * s + 3], cz);
            RLT_GRU_STEPS(a.x, 0) RLT_GRU_STEPS(a.y, 1) RLT_GRU_STEPS(a.z, 2) RLT_GRU_STEPS(a.w, 3)
            const float ar = xr + sum_quarters(cr), an = bhn + sum_quarters(cn), az = xz + sum_quarters(cz);
            const float r = FAST ? gate_sigmoid(ar, 1) : hw_sigmoid(ar), z = FAST ? gate_sigmoid(az, 1) : hw_sigmoid(az);
            const float n = FAST ? gate_tanh(xn + an * r, 1) : hw_tanh(xn + an * r);
            const float o = (1.0f - z) * n + z * h;
            h = flags & 1 ? h0 : o;       // the next step starts an episode
            flags >>= 1;
            hs[(N + 1) & 1][place] = h;
            gru_at(post, at3) = r; gru_at(post + H, at3) = z; gru_at(post + 2 * H, at3) = n; gru_at(npp, at) = an; gru_at(out, at) = o;
            post += 3 * stride; npp += stride; out += stride;
            request(first + i + D, q[N]);      // behind the last use of the entry: before it, the loop would start with copies of all entries, and with waits for them
        });
    }
}

// The same with the input gates W_i x + b_i formed beside the recurrence instead of by a launch in front of it (inputs_beside): batches of at most one workgroup per compute unit. Four
// more wavefronts, one per SIMD, form the gates of the next four steps (4 steps x 4 rows = the sixteen rows of v_mfma_f32_16x16x4) while the recurrence walks through these: wavefront p keeps
// rows 48 p ... 48 p + 47 of W_i in registers as the B operand, the steps' inputs are staged through LDS a group of four steps ahead and requested another group ahead, the gates reach the
// recurrence through LDS and never memory. Lane (n, kq) of both operands takes four consecutive inputs of every sixteen, in one 16-byte read
// (the order of the sums in rows_forward_kernel, gemm.hip: the same bits as where that is the launch in front; the tiled contraction of other shapes sums in another order).
// Bound: the recurrence's chain and, beside it, 30 instructions of 32 cycles per step at 146 inputs, in which the SIMD's vector unit stands still: a step of 64 x 1,024 sequences takes 1.0 us
// with 146 inputs, 0.69 with 3. The recurrence goes first (s_setprio); a second barrier per step that kept the others' products out of the recurrence's made it slower (64.5 -> 66.6 us).
// Launch of the input gates + recurrence / this, 64 steps, 1,024 rows: 146 inputs 77.5 / 65.5 us, 64 inputs 61.1 / 49.0, 3 inputs 57.8 / 44.0.
constexpr int GP_INPUTS = 160, GP_THREADS = 512, GP_LDX = 164, GP_LDG = 3 * 64 + 16, GP_STEP = GM_ROWS * GP_LDG + 16;      // inputs at most; row strides in LDS: eight lanes' 16-byte reads and sixteen lanes' words of four rows meet no bank twice
template <int GROUPS, bool FAST>      // GROUPS: sixteens of inputs, zeros behind the last
__global__ __launch_bounds__(GP_THREADS) void gru_forward_inputs_kernel(GruArgs A) {
    constexpr int H = 64, D = 4, E = (GM_ROWS * 16 * GROUPS + 255) / 256, TURNS = GROUPS;      // E: floats of a step that a thread stages; TURNS: reduction steps (of four inputs) between two steps of the recurrence
    __shared__ __align__(16) float hs[2][H * GM_ROWS];
    __shared__ __align__(16) float xs[2][4 * GM_ROWS * GP_LDX];      // inputs of four steps: row 4 step + batch row
    __shared__ float gates[2][D * GP_STEP];                          // their input gates
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, c16 = lane & 15;
    const int b0 = blockIdx.x * GM_ROWS, I = A.L.input_dim, S = A.S;
    for (int i = threadIdx.x; i < 2 * 4 * GM_ROWS * GP_LDX; i += GP_THREADS) (&xs[0][0])[i] = 0.f;      // columns beyond the inputs stay zero
    rlt_lds_barrier();
    if (wave >= 4) {
        const int p = wave - 4, tid = threadIdx.x - 256, live = min(GM_ROWS, A.B - b0) * I;      // live: floats of a step that exist
        float wb[3][GROUPS][4], bias[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int gate = 48 * p + 16 * j + c16;
            const float* const src = A.L.weights_input + (size_t)gate * I;
            bias[j] = A.L.biases_input[gate];
#pragma unroll
            for (int g = 0; g < GROUPS; g++) {
                const int at = 16 * g + 4 * kg;
                if (at + 4 <= I) {
                    const gru_float4_a4 v = *reinterpret_cast<const gru_float4_a4*>(src + at);
                    wb[j][g][0] = v[0]; wb[j][g][1] = v[1]; wb[j][g][2] = v[2]; wb[j][g][3] = v[3];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++) wb[j][g][r] = at + r < I ? src[at + r] : 0.f;
                }
            }
        }
        // This thread's floats of a step: where they lie in the step's inputs and in its rows in LDS. What does not exist is read as the last that does and is not used: a row beyond the batch
        // goes through as some copy, floats beyond the rows go to a column that nothing reads. No branch around a load.
        int from[E], place[E];
#pragma unroll
        for (int e = 0; e < E; e++) { const int i = tid + 256 * e, row = i / I; from[e] = min(i, live - 1); place[e] = row < GM_ROWS ? row * GP_LDX + i - row * I : GP_LDX - 1; }
        float staged[D][E];
        auto request = [&](int chunk) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                const float* const src = A.input + ((size_t)min(4 * chunk + d, S - 1) * A.B + b0) * I;
#pragma unroll
                for (int e = 0; e < E; e++) staged[d][e] = src[from[e]];
            }
        };
        auto stage = [&](int chunk) {
#pragma unroll
            for (int d = 0; d < D; d++)
#pragma unroll
                for (int e = 0; e < E; e++) xs[chunk & 1][d * GM_ROWS * GP_LDX + place[e]] = staged[d][e];
        };
        gru_floatx4 c[3];
        auto part = [&](auto number, int chunk) {      // a quarter of the products of a group of four steps
            constexpr int N = decltype(number)::value, FIRST = TURNS * N, LOW = FIRST / 4, HIGH = (FIRST + TURNS + 3) / 4;
            const float* const x = &xs[chunk & 1][c16 * GP_LDX + 4 * kg];
            if (N == 0) for (int j = 0; j < 3; j++) c[j] = gru_floatx4{0.f, 0.f, 0.f, 0.f};
            float4 a[HIGH - LOW];
#pragma unroll
            for (int g = LOW; g < HIGH; g++) a[g - LOW] = *reinterpret_cast<const float4*>(x + 16 * g);
#pragma unroll
            for (int s = FIRST; s < FIRST + TURNS; s++) {
                const float4 v = a[s / 4 - LOW];
#pragma unroll
                for (int j = 0; j < 3; j++) c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s % 4 == 0 ? v.x : s % 4 == 1 ? v.y : s % 4 == 2 ? v.z : v.w, wb[j][s / 4][s % 4], c[j], 0, 0, 0);
            }
            if (N == 3) {
#pragma unroll
                for (int j = 0; j < 3; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) gates[chunk & 1][kg * GP_STEP + r * GP_LDG + 48 * p + 16 * j + c16] = c[j][r] + bias[j];      // D: row 4 kg + r = step kg, batch row r
            }
        };
        request(0); stage(0); request(1); stage(1); request(2);
        rlt_lds_barrier();
        part(std::integral_constant<int, 0>{}, 0); part(std::integral_constant<int, 1>{}, 0); part(std::integral_constant<int, 2>{}, 0); part(std::integral_constant<int, 3>{}, 0);
        int chunk = 0;
        for (; 4 * (chunk + 1) < S; chunk++) {
            rlt_lds_barrier();
            stage(chunk + 2); request(chunk + 3);      // xs[chunk & 1] was read for the last time before this barrier
            part(std::integral_constant<int, 0>{}, chunk + 1);
            rlt_lds_barrier(); part(std::integral_constant<int, 1>{}, chunk + 1);
            rlt_lds_barrier(); part(std::integral_constant<int, 2>{}, chunk + 1);
            rlt_lds_barrier(); part(std::integral_constant<int, 3>{}, chunk + 1);
        }
        for (int t = 4 * chunk; t < S; t++) rlt_lds_barrier();
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const int w = wave, u = 16 * w + c16;
    float wb[3][16];
#pragma unroll
    for (int g = 0; g < 3; g++) {
        const float4* src = reinterpret_cast<const float4*>(A.L.weights_hidden + (size_t)(g * H + u) * H + 16 * kg);
#pragma unroll
        for (int q = 0; q < 4; q++) { const float4 v = src[q]; wb[g][4 * q] = v.x; wb[g][4 * q + 1] = v.y; wb[g][4 * q + 2] = v.z; wb[g][4 * q + 3] = v.w; }
    }
    const int row = min(kg, A.B - 1 - b0);
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    const float bhr = A.L.biases_hidden[u], bhz = A.L.biases_hidden[H + u], bhn = A.L.biases_hidden[2 * H + u];
    const float h0 = A.L.initial_hidden_state[u];
    const size_t stride = (size_t)A.B * H;
    float* post = A.L.post_activation + (size_t)b0 * 3 * H; float* npp = A.L.n_pre_pre_activation + (size_t)b0 * H; float* out = A.L.output + (size_t)b0 * H;
    const int place = ((4 * w + (c16 & 3)) * 4 + kg) * 4 + (c16 >> 2);      // this (row, unit) in hs
    float h = h0;
    hs[0][place] = h;
    rlt_lds_barrier();
    for (int first = 0; first < S; first += 64) {
        uint64_t flags = gru_reset_flags<GM_ROWS>(A.reset, first + 1, S, A.B, b0, kg);      // of the steps after these
        gru_steps<D>(min(64, S - first), [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);
            rlt_lds_barrier();
            const float4 a = *reinterpret_cast<const float4*>(&hs[N & 1][4 * lane]);
            const float* const in = &gates[((first + i) >> 2) & 1][N * GP_STEP + row * GP_LDG + u];
            const float xr = in[0] + bhr, xz = in[H] + bhz, xn = in[2 * H];
            gru_floatx4 cr = {0.f, 0.f, 0.f, 0.f}, cz = cr, cn = cr;
            RLT_GRU_STEPS(a.x, 0) RLT_GRU_STEPS(a.y, 1) RLT_GRU_STEPS(a.z, 2) RLT_GRU_STEPS(a.w, 3)
            const float ar = xr + sum_quarters(cr), an = bhn + sum_quarters(cn), az = xz + sum_quarters(cz);
            const float r = FAST ? gate_sigmoid(ar, 1) : hw_sigmoid(ar), z = FAST ? gate_sigmoid(az, 1) : hw_sigmoid(az);
            const float n = FAST ? gate_tanh(xn + an * r, 1) : hw_tanh(xn + an * r);
            const float o = (1.0f - z) * n + z * h;
            h = flags & 1 ? h0 : o;       // the next step starts an episode
            flags >>= 1;
            hs[(N + 1) & 1][place] = h;
            gru_at(post, at3) = r; gru_at(post + H, at3) = z; gru_at(post + 2 * H, at3) = n; gru_at(npp, at) = an; gru_at(out, at) = o;
            post += 3 * stride; npp += stride; out += stride;
        });
    }
}
#undef RLT_GRU_STEPS

// Reverse pass: the gate gradients of the four rows are the A side (192 reduction indices, quarter kg = the 48 of wavefront kg's units), a wavefront forms d h_prev of
// its sixteen units. gs (two copies, by the parity of the step): lane (kg, cg, row) of the A operand reads its twelve values in three 16-byte reads (neighbours lie 12
// floats apart: no two of a group share a bank). One workgroup barrier per step; lane = (row, unit) and addresses as in the forward pass.
// Four steps ahead take 145 registers, three workgroups per compute unit; where more want to run, two steps ahead and 117 registers for four (backward to the input, a row per
// wavefront as below / this: 3,100 sequences of 3 steps 23.6 / 22.2 us, 5,000 of 3 26.2 / 25.2, 6,000 of 10 52.1 / 50.4, 8,192 of 3 32.0 / 31.1).
template <int D, int WAVES>
__global__ __launch_bounds__(256, WAVES) void gru_backward_mfma_kernel(GruArgs A) {
    constexpr int H = 64;
    __shared__ __align__(16) float gs[2][3 * H * GM_ROWS];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, c16 = lane & 15, u = 16 * w + c16, S = A.S;
    // B operand: column u, reduction index (gate s >> 2, unit 16 kg + 4 (s & 3) + abid)
    float wb[48];
#pragma unroll
    for (int s = 0; s < 12; s++)
#pragma unroll
        for (int k = 0; k < 4; k++) wb[4 * s + k] = A.L.weights_hidden[(size_t)((s >> 2) * H + 16 * kg + 4 * (s & 3) + k) * H + u];
    const int b0 = blockIdx.x * GM_ROWS, row = min(kg, A.B - 1 - b0);
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    const float h0 = A.L.initial_hidden_state[u];
    const size_t stride = (size_t)A.B * H, last = (size_t)(S - 1) * stride + (size_t)b0 * H;
    struct Saved { float r, z, n, npp, dy, hp; };
    float *post = A.L.post_activation + 3 * last, *npp = A.L.n_pre_pre_activation + last, *dy = A.d_output + last, *state = A.L.output + last;
    auto request = [&](int i, Saved& v) {      // i-th step from the end; steps before the first read the first again; the state is the one before the step (the first step's is not used)
        const size_t on = i + 1 < S ? stride : 0;
        state -= on;
        v.r = gru_at(post, at3); v.z = gru_at(post + H, at3); v.n = gru_at(post + 2 * H, at3); v.npp = gru_at(npp, at); v.dy = gru_at(dy, at); v.hp = gru_at(state, at);
        post -= 3 * on; npp -= on; dy -= on;
    };
    Saved q[D];
#pragma unroll
    for (int d = 0; d < D; d++) if (d < A.S) request(d, q[d]);
    float *to_dy = A.d_output + last, *to_hp = A.h_previous + last, *bi = A.buffer_input + 3 * last, *bh = A.buffer_hidden + 3 * last;
    const int place = ((4 * w + (c16 & 3)) * 4 + kg) * 12 + (c16 >> 2);      // the r gate of this (row, unit) in gs; z and n four and eight on
    float carry = 0.f, db_hn = 0.f;
    for (int back = 0; back < S; back += 64) {
        const int steps = min(64, S - back);
        const uint64_t flags = gru_reset_flags<GM_ROWS>(A.reset, S - back - steps, S, A.B, b0, kg);      // bit of step t = S - 1 - back - i: steps - 1 - i
        uint64_t high = flags << (64 - steps);
        gru_steps<D>(steps, [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);
            const Saved cur = q[N];
            const bool first = back + i + 1 == S, from_initial = first || (high >> 63);
            high <<= 1;
            const float hp = from_initial ? h0 : cur.hp;
            const float dh = cur.dy + carry;
            const float gz = dh * (hp - cur.n) * cur.z * (1.0f - cur.z);
            const float gn = dh * (1.0f - cur.z) * (1.0f - cur.n * cur.n);
            const float gr = gn * cur.npp * cur.r * (1.0f - cur.r);
            const float gnr = gn * cur.r;
            float through = dh * cur.z;
            asm volatile("" : "+v"(through));      // (not formed below by a multiply-add that would keep the entry's z)
            request(back + i + D, q[N]);      // behind the last use of the entry: before it, the loop would start with copies of all entries, and with waits for them
            float* g = &gs[N & 1][place];
            g[0] = gr; g[4] = gz; g[8] = gnr;
            rlt_lds_barrier();
            const float4* ga = reinterpret_cast<const float4*>(&gs[N & 1][12 * lane]);
            const float4 a0 = ga[0], a1 = ga[1], a2 = ga[2];
            gru_at(to_dy, at) = dh; gru_at(to_hp, at) = hp;
            gru_at(bi, at3) = gr; gru_at(bi + H, at3) = gz; gru_at(bi + 2 * H, at3) = gn;
            gru_at(bh, at3) = gr; gru_at(bh + H, at3) = gz; gru_at(bh + 2 * H, at3) = gnr;
            to_dy -= stride; to_hp -= stride; bi -= 3 * stride; bh -= 3 * stride;
            // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
            db_hn += first || !from_initial ? gnr : 0.f;
            gru_floatx4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0, c2 = c0;
#define RLT_GRU_STEPS(X, k) \
            c0 = mfma4<0>(a0.X, wb[4 * k], c0); c1 = mfma4<0>(a1.X, wb[16 + 4 * k], c1); c2 = mfma4<0>(a2.X, wb[32 + 4 * k], c2); \
            c0 = mfma4<1>(a0.X, wb[4 * k + 1], c0); c1 = mfma4<1>(a1.X, wb[16 + 4 * k + 1], c1); c2 = mfma4<1>(a2.X, wb[32 + 4 * k + 1], c2); \
            c0 = mfma4<2>(a0.X, wb[4 * k + 2], c0); c1 = mfma4<2>(a1.X, wb[16 + 4 * k + 2], c1); c2 = mfma4<2>(a2.X, wb[32 + 4 * k + 2], c2); \
            c0 = mfma4<3>(a0.X, wb[4 * k + 3], c0); c1 = mfma4<3>(a1.X, wb[16 + 4 * k + 3], c1); c2 = mfma4<3>(a2.X, wb[32 + 4 * k + 3], c2);
            RLT_GRU_STEPS(x, 0) RLT_GRU_STEPS(y, 1) RLT_GRU_STEPS(z, 2) RLT_GRU_STEPS(w, 3)
            const float sum = sum_quarters(c0 + (c1 + c2));
            carry = from_initial ? 0.f : through + sum;
        });
    }
    if (A.db_hn_partial) gru_at(A.db_hn_partial + (size_t)b0 * H, at) = db_hn;
}

// ---- hidden widths 16, 32 and 64, a workgroup per row (rows_forward, rows_backward) -----------------------------------------------
// With few rows most compute units are idle on the kernels above, and a step of one row on the vector units is the shorter chain: at width 64 the matrix instruction forms four rows in
// 384 cycles whether they are there or not, the vector unit one row in 192; at 16 and 32 a wavefront that carries whole rows forms all their products, gates and stores one after the other. The
// first H / 16 wavefronts carry the recurrence, sixteen units each: four lanes share a hidden unit, the parts of the reduction meet in exchanges
// within four (eight) lanes. What bounds them is the number of instructions that one wavefront issues per step (about five cycles each), so four more wavefronts do the rest beside them: they request
// what the steps read (D steps ahead), hand it over through LDS a step ahead and store what the steps leave there a step later. One workgroup barrier per step.
// 64 steps at batch 64, four rows to a workgroup on the matrix cores / a row: forward recurrence 35.9 / 23 us, backward 33.2 / 23.2 (without the four wavefronts beside it 25 and 29.9);
// width 32, a step: forward 0.52 / 0.38 us (library gates), backward 0.56 / 0.25; width 16: 0.40 / 0.24 and 0.30 / 0.19.
constexpr int gru_row_threads(int H) { return 64 * (H / 16 + 4); }
enum { GATES_HARDWARE, GATES_FAST, GATES_EXACT };
__device__ __forceinline__ float quad_xor1(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true)); }
__device__ __forceinline__ float quad_xor2(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true)); }
__device__ __forceinline__ float quad_low(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x44, 0xF, 0xF, true)); }        // lanes 0, 1, 0, 1 of the four
__device__ __forceinline__ float quad_high(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xEE, 0xF, 0xF, true)); }       // lanes 2, 3, 2, 3
__device__ __forceinline__ float half_mirror(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true)); }    // lane 7 - i of the eight
__device__ __forceinline__ float row_half(float v) { return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)); }       // lane i ^ 8 of the sixteen
__device__ __forceinline__ float masked(float v, float mask) { return __int_as_float(__float_as_int(v) & __float_as_int(mask)); }
// The roles of the wavefronts beside the recurrence, each with a loop of its own: as branches within a step they held every step's barrier up (backward, 64 steps of
// 64 rows: width 16 21.7 -> 14.7 us, width 32 23.0 -> 17.8, width 64 26.3 -> 23.2).
template <class F> __device__ __forceinline__ void by_role(int role, F&& body) {
    if (role == 0) body(std::integral_constant<int, 0>{}); else if (role == 1) body(std::integral_constant<int, 1>{});
    else if (role == 2) body(std::integral_constant<int, 2>{}); else body(std::integral_constant<int, 3>{});
}
// steps 0 ... S - 1, their parity a constant
template <class F> __device__ __forceinline__ void gru_by_parity(int S, F&& step) {
    int t = 0;
    for (; t + 2 <= S; t += 2) { step(std::integral_constant<int, 0>{}); step(std::integral_constant<int, 1>{}); }
    if (t < S) step(std::integral_constant<int, 0>{});
}
// Lane (unit, kq): quarter kq of the reduction; lanes 0 and 1 of the four finish r, 2 and 3 z.
template <int H, int GATES>
__global__ __launch_bounds__(gru_row_threads(H), 4) void gru_forward_row_kernel(GruArgs A) {
    constexpr int CHAIN = H / 16, QUARTER = H / 4, D = 4;
    auto sigmoid = [](float x) { return GATES == GATES_HARDWARE ? hw_sigmoid(x) : gate_sigmoid(x, GATES == GATES_FAST); };
    auto tanh_ = [](float x) { return GATES == GATES_HARDWARE ? hw_tanh(x) : gate_tanh(x, GATES == GATES_FAST); };
    __shared__ __align__(16) float hs[2][H];                  // the previous state, by the parity of the step
    __shared__ __align__(16) float given[2][2][4 * H];        // r (z) gate's input part, n gate's, and the state that follows: (output & third) | fourth
    __shared__ float left[2][5 * H];                          // r, n, z, the n gate's hidden part, the output
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), b = blockIdx.x;
    const size_t stride = (size_t)A.B * H;
    if (w >= CHAIN) {
        by_role(w - CHAIN, [&](auto number_of_role) {
        constexpr int role = decltype(number_of_role)::value;
        const int u = lane & (H - 1), gate = role < 3 ? role : 0;      // r, z, n gate; the resets and the other two outputs
        float* in = A.L.post_activation + (size_t)b * 3 * H + gate * H;
        float* to = role < 3 ? in : A.L.n_pre_pre_activation + (size_t)b * H;
        float* out = A.L.output + (size_t)b * H;
        const size_t step = role < 3 ? 3 * stride : stride;
        const int from = (role == 0 ? 0 : role == 1 ? 2 : role == 2 ? 1 : 3) * H + u;
        const unsigned at = u * sizeof(float);
        const float bias = role < 2 ? A.L.biases_hidden[role * H + u] : 0.f, h0 = A.L.initial_hidden_state[u];
        auto request = [&](int t, float& v) { v = gru_at(in, at); in += t + 1 < A.S ? 3 * stride : 0; };      // the last steps request the last one again: no branch around the loads
        auto give = [&](int parity, float v, bool reset) {
            if (role < 2) given[parity][role][4 * u] = v + bias;
            else if (role == 2) { given[parity][0][4 * u + 1] = v; given[parity][1][4 * u + 1] = v; }
            else {
                const float keep = __int_as_float(reset ? 0 : -1), instead = reset ? h0 : 0.f;
#pragma unroll
                for (int g = 0; g < 2; g++) { given[parity][g][4 * u + 2] = keep; given[parity][g][4 * u + 3] = instead; }
            }
        };
        auto store = [&](int parity) {
            gru_at(to, at) = left[parity][from]; to += step;
            if (role == 3) { gru_at(out, at) = left[parity][4 * H + u]; out += stride; }
        };
        float q[D];
#pragma unroll
        for (int d = 0; d < D; d++) if (d < A.S) request(d, q[d]);
        uint64_t flags = gru_reset_flags<1>(A.reset, 1, A.S, A.B, b, 0);      // lowest bit: the step after the one that is handed over starts an episode
        give(0, q[0], flags & 1);
        rlt_lds_barrier();
        for (int first = 0; first < A.S; first += 64) {
            const uint64_t later = gru_reset_flags<1>(A.reset, first + 65, A.S, A.B, b, 0);      // of the steps after these
            gru_steps<D>(min(64, A.S - first), [&](auto number, int i) {
                constexpr int N = decltype(number)::value;
                __builtin_amdgcn_sched_barrier(0);
                flags = i + 1 < 64 ? flags >> 1 : later;
                give((N + 1) & 1, q[(N + 1) % D], flags & 1);
                request(first + i + D, q[N]);
                if (first + i > 0) store((N + 1) & 1);
                rlt_lds_barrier();
            });
        }
        store((A.S - 1) & 1);
        });
        return;
    }
    const int kq = lane & 3, u = 16 * w + (lane >> 2);
    const bool is_z = kq & 2, odd = kq & 1;
    float wb[3][QUARTER];
#pragma unroll
    for (int g = 0; g < 3; g++) {
        const gru_float4_a4* src = reinterpret_cast<const gru_float4_a4*>(A.L.weights_hidden + (size_t)(g * H + u) * H + QUARTER * kq);
#pragma unroll
        for (int q = 0; q < QUARTER / 4; q++) { const gru_float4_a4 v = src[q]; wb[g][4 * q] = v[0]; wb[g][4 * q + 1] = v[1]; wb[g][4 * q + 2] = v[2]; wb[g][4 * q + 3] = v[3]; }
    }
    const float bhn = A.L.biases_hidden[2 * H + u];
    float h = A.L.initial_hidden_state[u];
    hs[0][u] = h;
    __builtin_amdgcn_s_setprio(1);
    rlt_lds_barrier();
    gru_by_parity(A.S, [&](auto parity) {
        constexpr int P = decltype(parity)::value;
        gru_floatx4 a[QUARTER / 4];
#pragma unroll
        for (int k = 0; k < QUARTER / 4; k++) a[k] = reinterpret_cast<const gru_floatx4*>(&hs[P][QUARTER * kq])[k];
        const gru_floatx4 x = *reinterpret_cast<const gru_floatx4*>(&given[P][kq >> 1][4 * u]);
        __builtin_amdgcn_sched_barrier(0);      // all reads are under way before the first product
        float cr = 0.f, cz = 0.f, cn = 0.f;
#pragma unroll
        for (int k = 0; k < QUARTER / 4; k++)
#pragma unroll
            for (int j = 0; j < 4; j++) { cr = fmaf(a[k][j], wb[0][4 * k + j], cr); cz = fmaf(a[k][j], wb[1][4 * k + j], cz); cn = fmaf(a[k][j], wb[2][4 * k + j], cn); }
        float c = (is_z ? cz : cr) + quad_xor2(is_z ? cr : cz);
        cn += quad_xor2(cn);
        c += quad_xor1(c); cn += quad_xor1(cn);
        const float ac = x[0] + c, an = bhn + cn;
        const float gate = sigmoid(ac), r = quad_low(gate), z = quad_high(gate);
        const float n = tanh_(x[1] + an * r);
        const float o = (1.0f - z) * n + z * h;
        h = __int_as_float((__float_as_int(o) & __float_as_int(x[2])) | __float_as_int(x[3]));
        hs[P ^ 1][u] = h;
        left[P][kq * H + u] = odd ? is_z ? an : n : gate;
        left[P][4 * H + u] = o;
        rlt_lds_barrier();
    });
}
// Reverse pass: lane (four units, sixteenth kq of the units of each gate) forms the four units' sums over its gate gradients (width 64: 12 in three 16-byte reads; with two units to a lane and six reads LDS,
// which serves a wavefront's in eight cycles each, was the longer chain), the sixteenths meet in four exchanges, the first two of which leave a unit to each four lanes. Every gate gradient is the gradient at the state times a factor of saved values, which the wavefronts beside the recurrence form.
template <int H>
__global__ __launch_bounds__(gru_row_threads(H), 4) void gru_backward_row_kernel(GruArgs A) {
    constexpr int CHAIN = H / 16, K = H / 16, D = 4;      // K: gate gradients of a gate that a lane multiplies
    __shared__ __align__(16) float gs[2][4 * H];               // gradients at the r, z and n gate as the hidden path sees them, and at the state
    __shared__ float factor[2][4 * H];                         // of these, by the gradient at the state
    __shared__ __align__(16) float given[2][4 * H];            // gradient at the output, mask of what the step before hands on, z gate
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), b = blockIdx.x, S = A.S;
    const size_t stride = (size_t)A.B * H, last = (size_t)(S - 1) * stride + (size_t)b * H;
    if (w >= CHAIN) {
        by_role(w - CHAIN, [&](auto number_of_role) {
        constexpr int role = decltype(number_of_role)::value;
        const int u = lane & (H - 1);      // r, z, n gate, state
        const unsigned at = u * sizeof(float);
        const float h0 = A.L.initial_hidden_state[u];
        struct Saved { float z, n, first, second; };      // r gate: r, npp; z: -, state before; n: r, -; state: gradient at the output, state before (what is not named is read and not used)
        const bool from_gates = role != 3, from_state = role != 0;
        float *post = A.L.post_activation + 3 * last, *first_from = from_gates ? post : A.d_output + last;
        float* second_from = role == 0 ? A.L.n_pre_pre_activation + last : A.L.output + last - (S > 1 ? stride : 0);      // (the state before the first step is not used)
        const size_t first_step = from_gates ? 3 * stride : stride;
        auto request = [&](int i, Saved& v) {      // i-th step from the end; steps before the first read the first again
            v.z = gru_at(post + H, at); v.n = gru_at(post + 2 * H, at); v.first = gru_at(first_from, at); v.second = gru_at(second_from, at);
            const bool on = i + 1 < S;
            post -= on ? 3 * stride : 0; first_from -= on ? first_step : 0; second_from -= on && (!from_state || i + 2 < S) ? stride : 0;
        };
        Saved q[D];
#pragma unroll
        for (int d = 0; d < D; d++) if (d < S) request(d, q[d]);
        struct Kept { float n, hp; bool counts; } now, next;      // what the stores of a step need
        bool carried = false;      // the step before hands a gradient on
        auto give = [&](int parity, const Saved& v, int i, uint64_t flags) {
            const bool first = i + 1 >= S, from_initial = first || (flags >> 63);
            const float over = 1.0f - v.z, n = over * (1.0f - v.n * v.n), hp = from_initial ? h0 : v.second;
            if (role == 0) factor[parity][u] = n * v.second * v.first * (1.0f - v.first);
            else if (role == 1) factor[parity][H + u] = (hp - v.n) * v.z * over;
            else if (role == 2) factor[parity][2 * H + u] = n * v.first;
            else { const gru_floatx4 g = {v.first, __int_as_float(carried ? -1 : 0), v.z, 0.f}; *reinterpret_cast<gru_floatx4*>(&given[parity][4 * u]) = g; }
            carried = !from_initial;
            next.n = n; next.hp = hp; next.counts = first || !from_initial;      // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
        };
        float *to_input = A.buffer_input + 3 * last + (role < 2 ? role : 2) * H, *to_hidden = role < 3 ? A.buffer_hidden + 3 * last + role * H : A.h_previous + last, *to_dy = A.d_output + last;
        const size_t hidden_step = role < 3 ? 3 * stride : stride;
        float db_hn = 0.f;
        auto store = [&](int parity) {
            const float g = gs[parity][role * H + u];
            if (role < 2) gru_at(to_input, at) = g;
            else if (role == 3) { gru_at(to_input, at) = g * now.n; gru_at(to_dy, at) = g; }
            else db_hn += now.counts ? g : 0.f;
            gru_at(to_hidden, at) = role < 3 ? g : now.hp;
            to_input -= 3 * stride; to_hidden -= hidden_step; to_dy -= stride;
        };
        if (role == 3) { factor[0][3 * H + u] = 1.f; factor[1][3 * H + u] = 1.f; }
        uint64_t flags = gru_reset_flags<1>(A.reset, max(S - 64, 0), S, A.B, b, 0) << (64 - min(64, S));      // the highest bit: the step that is handed over, t = S - 1 - i
        __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
        give(0, q[0], 0, flags);
        rlt_lds_barrier();
        for (int back = 0; back < S; back += 64) {
            const int steps = min(64, S - back), rest = S - back - 64;
            const uint64_t later = rest > 0 ? gru_reset_flags<1>(A.reset, max(rest - 64, 0), rest, A.B, b, 0) << (64 - min(64, rest)) : 0;      // of the steps after these
            gru_steps<D>(steps, [&](auto number, int i) {
                constexpr int N = decltype(number)::value;
                __builtin_amdgcn_sched_barrier(0);
                if (back + i > 0) store((N + 1) & 1);      // of the step before
                now = next;
                flags = i + 1 < 64 ? flags << 1 : later;
                give((N + 1) & 1, q[(N + 1) % D], back + i + 1, flags);
                request(back + i + D, q[N]);
                rlt_lds_barrier();
            });
        }
        store((S - 1) & 1);
        if (role == 2 && A.db_hn_partial) gru_at(A.db_hn_partial + (size_t)b * H, at) = db_hn;
        });
        return;
    }
    const int kq = lane & 15, u0 = 16 * w + 4 * (lane >> 4), u = 16 * w + (lane >> 2), place = (lane & 3) * H + u;
    const bool upper8 = lane & 8, upper4 = lane & 4;
    gru_floatx4 wb[3 * K];
#pragma unroll
    for (int g = 0; g < 3; g++)
#pragma unroll
        for (int k = 0; k < K; k++) wb[K * g + k] = *reinterpret_cast<const gru_float4_a4*>(A.L.weights_hidden + (size_t)(g * H + K * kq + k) * H + u0);
    __builtin_amdgcn_s_setprio(1);
    rlt_lds_barrier();
    float f = factor[0][place], carry = 0.f;
    gru_floatx4 x = *reinterpret_cast<const gru_floatx4*>(&given[0][4 * u]);
    gru_by_parity(S, [&](auto parity) {
        constexpr int P = decltype(parity)::value;
        const float dh = x[0] + masked(carry, x[1]), z = x[2];
        gs[P][place] = dh * f;
        rlt_lds_barrier();
        typedef float Own __attribute__((ext_vector_type(K)));
        Own v[3];
#pragma unroll
        for (int g = 0; g < 3; g++) v[g] = *reinterpret_cast<const Own*>(&gs[P][g * H + K * kq]);
        f = factor[P ^ 1][place];
        x = *reinterpret_cast<const gru_floatx4*>(&given[P ^ 1][4 * u]);
        __builtin_amdgcn_sched_barrier(0);      // all reads are under way before the first product
        float c[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < 3; g++)
#pragma unroll
            for (int k = 0; k < K; k++)
#pragma unroll
                for (int a = 0; a < 4; a++) c[a] = fmaf(v[g][k], wb[K * g + k][a], c[a]);
        const float c0 = (upper8 ? c[2] : c[0]) + row_half(upper8 ? c[0] : c[2]), c1 = (upper8 ? c[3] : c[1]) + row_half(upper8 ? c[1] : c[3]);
        float sum = (upper4 ? c1 : c0) + half_mirror(upper4 ? c0 : c1);
        sum += quad_xor2(sum); sum += quad_xor1(sum);
        carry = dh * z + sum;
    });
}

// The same with the weight gradients formed beside the recurrence instead of by five launches after it that read every step's gate gradients and states back: batches of at most one
// workgroup per compute unit (weights_beside). Four more wavefronts, one per SIMD, take each step's gate gradients (gs, and the n gate's as the input path sees it), previous states and inputs from
// LDS: v_mfma_f32_16x16x4 adds a step's four rows (the reduction) to a 16 x 16 tile of the gradient; wavefront p keeps rows 48 p ... 48 p + 47 of dW_i and dW_h in accumulators (three by ten
// and three by four tiles), the recurrence's lanes add up their own gate gradients for db_i and the n gate's db_h. The inputs are staged through LDS, requested four steps ahead. A workgroup leaves one block of sums,
// gru_gradient_finish_kernel adds the blocks up in order. Bound: the recurrence's chain and, beside it, 42 instructions of 32 cycles per step at 146 inputs, in which the SIMD's vector unit stands still.
// Of a step only d_output (accumulated into, as before) and, for a gradient of the input, the input path's gate gradients go to memory.
// Recurrence + weight gradients / this + the finish, 64 steps, 1,024 rows: 146 inputs 138.5 / 85.7 us, 64 inputs 104.4 / 63.0, 3 inputs 98.9 / 54.3.
// Relative error against 64 bits (2-norm) at 3 to 146 inputs: dW_i 1.9e-7 ... 3.7e-7 (launches: 1.9e-7 ... 3.8e-7), db_i 1.1e-7 ... 2.3e-7 (1.2e-7 ... 2.2e-7).
constexpr int GW_INPUTS = 160, GW_LDX = 176, GW_LDH = 80;      // inputs at most; row strides in LDS: sixteen lanes' words of four rows meet no bank twice
__host__ __device__ constexpr size_t gru_gradient_block(int I) { return (size_t)3 * 64 * (I + 64 + 1) + 64; }      // floats: [192, I], [192, 64], 192 of db_i, 64 of the n gate's db_h
template <int TILES>      // sixteens of inputs, zeros behind the last
__global__ __launch_bounds__(GP_THREADS) void gru_backward_weights_kernel(GruArgs A) {
    constexpr int H = 64, D = 4, E = (GM_ROWS * 16 * TILES + 255) / 256;      // E: floats of a step that a thread stages
    __shared__ __align__(16) float gs[2][3 * H * GM_ROWS];
    __shared__ float gn_input[2][H * GM_ROWS];
    __shared__ float hp_rows[2][GM_ROWS * GW_LDH];
    __shared__ float xs[2][GM_ROWS * GW_LDX];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, c16 = lane & 15, S = A.S, I = A.L.input_dim;
    const int b0 = blockIdx.x * GM_ROWS, live_rows = min(GM_ROWS, A.B - b0);
    float* const block = A.blocks + (size_t)blockIdx.x * gru_gradient_block(I);
    for (int i = threadIdx.x; i < 2 * GM_ROWS * GW_LDX; i += GP_THREADS) (&xs[0][0])[i] = 0.f;
    rlt_lds_barrier();
    if (wave >= 4) {
        const int p = wave - 4, tid = threadIdx.x - 256, live = live_rows * I;
        int from[E], place[E];      // as in the forward pass; rows beyond the batch are zeros
#pragma unroll
        for (int e = 0; e < E; e++) { const int i = tid + 256 * e, r = i / I; from[e] = min(i, live - 1); place[e] = r < GM_ROWS ? r * GW_LDX + i - r * I : GW_LDX - 1; }
        const float* next = A.input + ((size_t)(S - 1) * A.B + b0) * I;      // from the last step to the first
        float staged[D][E];
        auto request = [&](int i, float (&v)[E]) {      // the steps before the first read the first again
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = next[from[e]];
            next -= i + 1 < S ? (size_t)A.B * I : 0;
        };
#pragma unroll
        for (int d = 0; d < D; d++) request(d, staged[d]);
        // A operand: lane (m, k) takes gate row 16 (3 p + a) + m of batch row k; in gs unit u of gate g lies at its place + 4 g
        const int within = (4 * (c16 & 3) + kg);
        int hidden_at[3], input_at[3];
        bool n_gate[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int tile = 3 * p + a, g = tile >> 2, pl = 16 * (tile & 3) + within;
            n_gate[a] = g == 2;
            hidden_at[a] = 12 * pl + (c16 >> 2) + 4 * g;
            input_at[a] = 4 * pl + (c16 >> 2);
        }
        gru_floatx4 ci[3][TILES], ch[3][4];
#pragma unroll
        for (int a = 0; a < 3; a++) {
#pragma unroll
            for (int j = 0; j < TILES; j++) ci[a][j] = gru_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) ch[a][j] = gru_floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const bool exists = kg < live_rows;      // rows beyond the batch count nothing
        gru_steps<D>(S, [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < E; e++) xs[N & 1][place[e]] = tid + 256 * e < live ? staged[N][e] : 0.f;      // (read for the last time before the barrier of the step between)
            request(i + D, staged[N]);
            rlt_lds_barrier();
            float ah[3], ai[3], bh[4], bx[TILES];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const float v = gs[N & 1][hidden_at[a]], n = gn_input[N & 1][input_at[a]];
                ah[a] = exists ? v : 0.f;
                ai[a] = n_gate[a] ? (exists ? n : 0.f) : ah[a];
            }
#pragma unroll
            for (int j = 0; j < 4; j++) bh[j] = hp_rows[N & 1][kg * GW_LDH + 16 * j + c16];
#pragma unroll
            for (int j = 0; j < TILES; j++) bx[j] = xs[N & 1][kg * GW_LDX + 16 * j + c16];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int a = 0; a < 3; a++) ch[a][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[a], bh[j], ch[a][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < TILES; j++)
#pragma unroll
                for (int a = 0; a < 3; a++) ci[a][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai[a], bx[j], ci[a][j], 0, 0, 0);
        });
        float* const hidden = block + (size_t)3 * H * I;
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gate = 16 * (3 * p + a) + 4 * kg + r;
#pragma unroll
                for (int j = 0; j < TILES; j++) if (16 * j + c16 < I) block[gate * I + 16 * j + c16] = ci[a][j][r];
#pragma unroll
                for (int j = 0; j < 4; j++) hidden[gate * H + 16 * j + c16] = ch[a][j][r];
            }
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const int w = wave, u = 16 * w + c16;
    float wb[48];
#pragma unroll
    for (int s = 0; s < 12; s++)
#pragma unroll
        for (int k = 0; k < 4; k++) wb[4 * s + k] = A.L.weights_hidden[(size_t)((s >> 2) * H + 16 * kg + 4 * (s & 3) + k) * H + u];
    const int row = min(kg, live_rows - 1);
    const bool exists = kg < live_rows;
    const unsigned at = (row * H + u) * sizeof(float), at3 = (row * 3 * H + u) * sizeof(float);
    const float h0 = A.L.initial_hidden_state[u];
    const size_t stride = (size_t)A.B * H, last = (size_t)(S - 1) * stride + (size_t)b0 * H;
    struct Saved { float r, z, n, npp, dy, hp; };
    float *post = A.L.post_activation + 3 * last, *npp = A.L.n_pre_pre_activation + last, *dy = A.d_output + last, *state = A.L.output + last;
    auto request = [&](int i, Saved& v) {      // as above
        const size_t on = i + 1 < S ? stride : 0;
        state -= on;
        v.r = gru_at(post, at3); v.z = gru_at(post + H, at3); v.n = gru_at(post + 2 * H, at3); v.npp = gru_at(npp, at); v.dy = gru_at(dy, at); v.hp = gru_at(state, at);
        post -= 3 * on; npp -= on; dy -= on;
    };
    Saved q[D];
#pragma unroll
    for (int d = 0; d < D; d++) if (d < S) request(d, q[d]);
    float *to_dy = A.d_output + last, *bi = A.buffer_input ? A.buffer_input + 3 * last : nullptr;
    const int place = ((4 * w + (c16 & 3)) * 4 + kg) * 12 + (c16 >> 2);
    float carry = 0.f, db_hn = 0.f, db_r = 0.f, db_z = 0.f, db_n = 0.f;
    for (int back = 0; back < S; back += 64) {
        const int steps = min(64, S - back);
        const uint64_t flags = gru_reset_flags<GM_ROWS>(A.reset, S - back - steps, S, A.B, b0, kg);
        uint64_t high = flags << (64 - steps);
        gru_steps<D>(steps, [&](auto number, int i) {
            constexpr int N = decltype(number)::value;
            __builtin_amdgcn_sched_barrier(0);
            const Saved cur = q[N];
            const bool first = back + i + 1 == S, from_initial = first || (high >> 63);
            high <<= 1;
            const float hp = from_initial ? h0 : cur.hp;
            const float dh = cur.dy + carry;
            const float gz = dh * (hp - cur.n) * cur.z * (1.0f - cur.z);
            const float gn = dh * (1.0f - cur.z) * (1.0f - cur.n * cur.n);
            const float gr = gn * cur.npp * cur.r * (1.0f - cur.r);
            const float gnr = gn * cur.r;
            float through = dh * cur.z;
            asm volatile("" : "+v"(through));      // (not formed below by a multiply-add that would keep the entry's z)
            request(back + i + D, q[N]);
            float* g = &gs[N & 1][place];
            g[0] = gr; g[4] = gz; g[8] = gnr;
            gn_input[N & 1][((4 * w + (c16 & 3)) * 4 + kg) * 4 + (c16 >> 2)] = gn;
            hp_rows[N & 1][kg * GW_LDH + u] = exists ? hp : 0.f;
            rlt_lds_barrier();
            const float4* ga = reinterpret_cast<const float4*>(&gs[N & 1][12 * lane]);
            const float4 a0 = ga[0], a1 = ga[1], a2 = ga[2];
            gru_at(to_dy, at) = dh;
            to_dy -= stride;
            if (bi) { gru_at(bi, at3) = gr; gru_at(bi + H, at3) = gz; gru_at(bi + 2 * H, at3) = gn; bi -= 3 * stride; }
            // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
            db_hn += first || !from_initial ? gnr : 0.f;
            db_r += gr; db_z += gz; db_n += gn;
            gru_floatx4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0, c2 = c0;
            RLT_GRU_STEPS(x, 0) RLT_GRU_STEPS(y, 1) RLT_GRU_STEPS(z, 2) RLT_GRU_STEPS(w, 3)
            const float sum = sum_quarters(c0 + (c1 + c2));
            carry = from_initial ? 0.f : through + sum;
        });
    }
    auto rows_sum = [&](float v) { v = exists ? v : 0.f; v += __shfl_xor(v, 16, 64); return v + __shfl_xor(v, 32, 64); };
    const float sums[4] = {rows_sum(db_r), rows_sum(db_z), rows_sum(db_n), rows_sum(db_hn)};
    if (kg == 0)
#pragma unroll
        for (int g = 0; g < 4; g++) block[gru_gradient_block(I) - 4 * H + g * H + u] = sums[g];
}
#undef RLT_GRU_STEPS

// The weight gradients after a backward pass that has left the gate gradients and the previous states of every step in memory: dW_i, dW_h and db_i of all rows in one launch (SUBSETS = H / 16
// times 48 gate rows). A workgroup takes two 16-column tiles of the inputs or of the states and a share of the rows, a wavefront 48 gate rows (three tiles; at the smaller widths also a
// share of the workgroup's rows): six tiles of v_mfma_f32_16x16x4 in accumulators, operands straight from memory (lane (m, k): row k of four, sixteen consecutive columns), requested eight
// steps of four rows ahead. Every share leaves a block of sums. Bound: latency, 2.3 us of matrix instructions per wavefront at 4,096 rows of 146 inputs among loads that memory answers in one.
// As a contraction and a sum per gradient and a launch for db_h these were five launches. Backward pass, five / this and the finish, us: 64 steps, 146 inputs, width 64: 16 rows 53.7 / 42.9,
// 64 rows 64.4 / 49.6, 256 rows 79.6 / 61.3; width 32: 64 rows 64.6 / 51.4, 1,024 rows 115.1 / 81.2; width 16: 64 rows 42.0 / 32.5. Relative error against 64 bits (2-norm) over these: dW_i
// 1.4e-7 ... 3.5e-7 (five launches 1.9e-7 ... 5.2e-7), dW_h 2.0e-7 ... 4.2e-7 (2.4e-7 ... 4.5e-7).
struct GradientArgs { const float *d_input_path, *d_hidden_path, *input, *h_previous; float* blocks; int rows, I, input_pairs; };
__host__ __device__ constexpr size_t gradient_block(int H, int I) { return (size_t)3 * H * (I + H + 1); }      // floats: [3 H, I], [3 H, H], 3 H of db_i
template <int SUBSETS>
__global__ __launch_bounds__(256) void gru_gradients_kernel(GradientArgs A) {
    constexpr int H = 16 * SUBSETS, PARTS = 4 / SUBSETS, D = 8, CHAINS = 4;      // CHAINS: accumulators per tile, a quarter of the steps each (shorter sums: a smaller error)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, k = lane >> 4, subset = wave % SUBSETS;
    const int share = blockIdx.y * PARTS + wave / SUBSETS, shares = gridDim.y * PARTS, steps = (A.rows + 3) >> 2;
    const int first = (int)((long long)steps * share / shares), end = (int)((long long)steps * (share + 1) / shares);
    const bool hidden = (int)blockIdx.x >= A.input_pairs;
    const int pair = hidden ? blockIdx.x - A.input_pairs : blockIdx.x, width = hidden ? H : A.I;
    const float* const d = (hidden ? A.d_hidden_path : A.d_input_path) + 48 * subset + m;
    const float* const x = hidden ? A.h_previous : A.input;
    const int c0 = min(32 * pair + m, width - 1), c1 = min(32 * pair + 16 + m, width - 1);      // columns beyond the width repeat the last one and are not stored
    struct Step { float a[3], b[2]; };
    auto request = [&](int s, Step& v) {      // steps and rows that do not exist read the last row
        const size_t row = (size_t)min(4 * s + k, A.rows - 1);
#pragma unroll
        for (int t = 0; t < 3; t++) v.a[t] = d[row * 3 * H + 16 * t];
        v.b[0] = x[row * width + c0]; v.b[1] = x[row * width + c1];
    };
    gru_floatx4 c[CHAINS][3][2];
    float bias[CHAINS][3] = {};
#pragma unroll
    for (int i = 0; i < CHAINS; i++)
#pragma unroll
        for (int t = 0; t < 3; t++) c[i][t][0] = c[i][t][1] = gru_floatx4{0.f, 0.f, 0.f, 0.f};
    Step v[D], ahead[D];
#pragma unroll
    for (int i = 0; i < D; i++) request(first + i, v[i]);
    for (int s = first; s < end; s += D) {
#pragma unroll
        for (int i = 0; i < D; i++) request(s + D + i, ahead[i]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < D; i++) {
            if (s + D > end || 4 * (s + i) + 3 >= A.rows) {      // the last group of a share, the last rows: what does not exist counts nothing
                const bool exists = s + i < end && 4 * (s + i) + k < A.rows;
#pragma unroll
                for (int t = 0; t < 3; t++) v[i].a[t] = exists ? v[i].a[t] : 0.f;
                v[i].b[0] = exists ? v[i].b[0] : 0.f; v[i].b[1] = exists ? v[i].b[1] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int t = 0; t < 3; t++) c[i % CHAINS][t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i].a[t], v[i].b[j], c[i % CHAINS][t][j], 0, 0, 0);
            if (blockIdx.x == 0)
#pragma unroll
                for (int t = 0; t < 3; t++) bias[i % CHAINS][t] += v[i].a[t];
        }
#pragma unroll
        for (int i = 0; i < D; i++) v[i] = ahead[i];
    }
    float* const block = A.blocks + (size_t)share * gradient_block(H, A.I);
    float* const to = block + (hidden ? (size_t)3 * H * A.I : 0);
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gate = 48 * subset + 16 * t + 4 * k + r, col = 32 * pair + 16 * j + m;
                if (col < width) to[(size_t)gate * width + col] = (c[0][t][j][r] + c[1][t][j][r]) + (c[2][t][j][r] + c[3][t][j][r]);
            }
    if (blockIdx.x == 0)
#pragma unroll
        for (int t = 0; t < 3; t++) {
            float sum = (bias[0][t] + bias[1][t]) + (bias[2][t] + bias[3][t]);
            sum += __shfl_xor(sum, 16, 64); sum += __shfl_xor(sum, 32, 64);
            if (k == 0) block[(size_t)3 * H * (A.I + H) + 48 * subset + 16 * t + m] = sum;
        }
}

// Blocks of sums added up in their order into the gradients: 64 elements per workgroup, sixteen lanes with four elements each, every sixteenth block in another group of lanes. The last
// H / 4 workgroups take four elements each of the n gate's db_h from blocks of its own (n_hidden of them, `hidden_stride` floats apart), every 256th in another thread.
__global__ __launch_bounds__(256) void gru_gradient_finish_kernel(const float* __restrict__ blocks, int n, size_t stride, const float* __restrict__ hidden, int n_hidden, size_t hidden_stride, int H, int I,
                                                                  float* dW_i, float* db_i, float* dW_h, float* db_h) {
    __shared__ float4 part[16][16];
    const int c = threadIdx.x & 15, group = threadIdx.x >> 4, count = (int)gradient_block(H, I);      // a multiple of four
    const int quad = (int)blockIdx.x - ((int)gridDim.x - H / 4);
    const bool last = quad >= 0;
    const float* const src = last ? hidden + 4 * quad : blocks + min((int)blockIdx.x * 64 + 4 * c, count - 4);
    const int many = last ? n_hidden : n, by = last ? 256 : 16;
    const size_t apart = last ? hidden_stride : stride;
    float4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int b = last ? threadIdx.x : group; b < many; b += by) { const float4 v = *reinterpret_cast<const float4*>(src + (size_t)b * apart); s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w; }
    if (last) {
        s.x = rlt_wave_sum(s.x); s.y = rlt_wave_sum(s.y); s.z = rlt_wave_sum(s.z); s.w = rlt_wave_sum(s.w);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][0] = s;
        __syncthreads();
        if (threadIdx.x < 4) {
            const float* const v = reinterpret_cast<const float*>(&part[0][0]) + threadIdx.x;
            db_h[2 * H + 4 * quad + threadIdx.x] += (v[0] + v[64]) + (v[128] + v[192]);
        }
        return;
    }
    part[group][c] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < 16; g++) sum += reinterpret_cast<const float*>(&part[g][0])[threadIdx.x];
    const int e = blockIdx.x * 64 + threadIdx.x, inputs = 3 * H * I, weights = inputs + 3 * H * H;
    if (e < inputs) dW_i[e] += sum;
    else if (e < weights) dW_h[e - inputs] += sum;
    else if (e < count) {
        const int gate = e - weights;
        const float d = db_i[gate] + sum;
        db_i[gate] = d;
        if (gate < 2 * H) db_h[gate] = d;      // (the reference copies, :679-681)
    }
}

// The same for batches whose steps are bound by memory instead of the chain: thread (w, lane) finishes (row w, unit lane), so that a wavefront's loads and stores are whole rows
// of 256 bytes (above: 64 bytes of each of four rows). Wavefront w forms the
// products of rows 48 w ... 48 w + 47 of W_h (lane = column) and the four partial sums of d h_prev meet in LDS: two workgroup barriers per step. Backward to the input, the kernel above / this
// one: 16,384 sequences of 10 steps 181 / 157 us, 3,000 of 30 90.8 / 77.3, 1,500 of 100 173 / 157; but 2,048 of 30 52.0 / 53.2, 1,024 of 100 95 / 130.
template <int ABID> __device__ __forceinline__ gru_floatx4 mfma4_all(float a, float b, gru_floatx4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, ABID, 0); }      // every block's A from block ABID
// 16 reduction steps: A register `a` holds, in block k, the four rows' values of reduction index base + k
template <int... K> __device__ __forceinline__ void sixteen_steps(float a, const float* w, gru_floatx4 (&c)[4], std::integer_sequence<int, K...>) { ((c[K & 3] = mfma4_all<K>(a, w[K], c[K & 3])), ...); }
__global__ __launch_bounds__(256) void gru_backward_rows_kernel(GruArgs A) {
    constexpr int H = 64, D = 3, GS = 3 * H + 16;      // D: steps ahead that the saved values are requested; GS: row stride of the gate gradients in LDS, rows 16 banks apart
    __shared__ float gs[GM_ROWS * GS];
    __shared__ float part[4][GM_ROWS * 64];
    const int u = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), S = A.S;
    float wb[48];
#pragma unroll
    for (int k = 0; k < 48; k++) wb[k] = A.L.weights_hidden[(size_t)(48 * w + k) * H + u];
    const bool live = blockIdx.x * GM_ROWS + w < A.B;
    const int b = live ? blockIdx.x * GM_ROWS + w : A.B - 1;      // rows beyond the batch read the last row and store nothing
    const float h0 = A.L.initial_hidden_state[u];
    float carry = 0.f, db_hn = 0.f;
    struct Saved { float r, z, n, npp, dy, hp; int restart; };
    auto request = [&](int t) {      // steps before the first read the first again; the state is the one before the step (the first step's is not used)
        const size_t at = (size_t)max(t, 0) * A.B + b;
        const float* const post = A.L.post_activation + at * 3 * H + u;
        Saved v = {post[0], post[H], post[2 * H], A.L.n_pre_pre_activation[at * H + u], A.d_output[at * H + u], A.L.output[((size_t)max(t - 1, 0) * A.B + b) * H + u], 0};
        v.restart = t <= 0 || (A.reset && A.reset[at]);
        return v;
    };
    Saved q[D];
#pragma unroll
    for (int d = 0; d < D; d++) q[d] = request(S - 1 - d);
    for (int t = S - 1; t >= 0; t--) {
        const size_t at = (size_t)t * A.B + b;
        const Saved far = request(t - D), cur = q[0];
        const float hp = cur.restart ? h0 : cur.hp;
        const float dh = cur.dy + carry;
        const float gz = dh * (hp - cur.n) * cur.z * (1.0f - cur.z);
        const float gn = dh * (1.0f - cur.z) * (1.0f - cur.n * cur.n);
        const float gr = gn * cur.npp * cur.r * (1.0f - cur.r);
        const float gnr = gn * cur.r;
        if (live) {
            float* const bi = A.buffer_input + at * 3 * H + u; float* const bh = A.buffer_hidden + at * 3 * H + u;
            A.d_output[at * H + u] = dh; A.h_previous[at * H + u] = hp;
            bi[0] = gr; bi[H] = gz; bi[2 * H] = gn;
            bh[0] = gr; bh[H] = gz; bh[2 * H] = gnr;
        }
        // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, :716-749)
        if (t == 0 || !cur.restart) db_hn += gnr;
        gs[w * GS + u] = gr; gs[w * GS + H + u] = gz; gs[w * GS + 2 * H + u] = gnr;
        rlt_lds_barrier();
        const float* const ga = gs + (u & 3) * GS + 48 * w + (u >> 2);
        const float a0 = ga[0], a1 = ga[16], a2 = ga[32];
        const gru_floatx4 zero = {0.f, 0.f, 0.f, 0.f};
        gru_floatx4 c[4] = {zero, zero, zero, zero};
        const auto steps = std::make_integer_sequence<int, 16>{};
        sixteen_steps(a0, wb, c, steps); sixteen_steps(a1, wb + 16, c, steps); sixteen_steps(a2, wb + 32, c, steps);
        const gru_floatx4 mine = (c[0] + c[1]) + (c[2] + c[3]);
#pragma unroll
        for (int row = 0; row < GM_ROWS; row++) part[w][64 * row + u] = mine[row];
        rlt_lds_barrier();
        const float sum = (part[0][64 * w + u] + part[1][64 * w + u]) + (part[2][64 * w + u] + part[3][64 * w + u]);
        carry = cur.restart ? 0.f : dh * cur.z + sum;
#pragma unroll
        for (int d = 0; d + 1 < D; d++) q[d] = q[d + 1];
        q[D - 1] = far;
    }
    if (live && A.db_hn_partial) A.db_hn_partial[(size_t)b * H + u] = db_hn;
}
// Which of the two: beyond one workgroup per compute unit, where what the steps read and write (14 rows of 64 floats each) does not fit the 256 MB of last-level cache
bool backward_by_rows(int units, int S, int B) { return rlt_div_up(B, GM_ROWS) > units && (size_t)S * B * 14 * 64 * sizeof(float) > (size_t)256 << 20; }

// db_h[n part] += sum over batch rows of the per-row sums, db_h[r, z parts] = db_i[r, z parts] (the reference copies, :679-681).
// One workgroup per hidden unit.
__global__ __launch_bounds__(256) void gru_bias_hidden_kernel(const float* __restrict__ partial, int B, int H, const float* __restrict__ db_i, float* __restrict__ db_h) {
    __shared__ float part[4];
    const int j = blockIdx.x;
    float s = 0.f;
    for (int b = threadIdx.x; b < B; b += blockDim.x) s += partial[(size_t)b * H + j];
    s = rlt_wave_sum(s);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) { db_h[2 * H + j] += (part[0] + part[1]) + (part[2] + part[3]); db_h[j] = db_i[j]; db_h[H + j] = db_i[H + j]; }
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
bool layer_ok(const rlt_gru_layer* L) {
    return L && L->weights_input && L->biases_input && L->weights_hidden && L->biases_hidden && L->initial_hidden_state && L->post_activation &&
           L->n_pre_pre_activation && L->output && L->input_dim >= 1 && L->hidden_dim >= 1 && L->hidden_dim <= GRU_THREADS;
}
int compute_units(const rlt_rocm_device* device) { return device->compute_units > 0 ? device->compute_units : 256; }
bool one_group_per_unit(const rlt_rocm_device* device, const rlt_gru_layer* L, int B) { return L->hidden_dim == 64 && rlt_div_up(B, GM_ROWS) <= compute_units(device); }
// Where the recurrence takes a workgroup per row (with input gates and weight gradients as launches of their own). us, several rows to a workgroup / a row:
// forward calls of 64 steps, width 64, 3 inputs 64 rows 41.0 / 28.3, 256 rows 50.0 / 37.4, 512 rows 53.4 / 44.5, 600 rows (three rounds of rows) 53.9 / 55.1; width 32, 64 inputs 64 rows 44.3 / 30.6, 512 rows
// 58.0 / 46.2, 1,024 rows 64.8 / 54.1; 200 inputs 1,280 rows 100 / 92, 1,536 rows 108 / 114; width 16 64 rows 33.0 / 22.7, 1,024 rows 47.7 / 38.3; 200 inputs 1,280 rows 63 / 56, 1,536 rows 68 / 75;
// 1 step at 1,280 rows 14.6 / 12.5 and 12.4 / 12.4;
// backward to the input, 64 steps, width 64 256 rows 34.1 / 24.3, 512 rows 34.3 / 28.4, 768 rows 34.9 / 37; width 32 256 rows 39.5 / 18.6, 1,024 rows 39.6 / 27.3, 1,280 rows 39.8 / 32.0, 1,536 rows 40.2 / 41.6;
// width 16 256 rows 22.6 / 15.4, 768 rows 23.1 / 21.4, 1,024 rows 23.2 / 24.4; 16 steps, width 64 256 rows 11.0 / 9.0, 512 rows 11.5 / 11.6, width 32 1,280 rows 13.3 / 12.1, width 16 768 rows 8.4 / 8.0;
// 4 steps, width 64 512 rows 5.4 / 6.8, width 32 1,280 rows 6.1 / 6.2; 1 step 3.85 / 4.0.
bool rows_forward(const rlt_rocm_device* device, int H, int B) { return B <= (H == 64 ? 2 : 5) * compute_units(device); }
bool rows_backward(const rlt_rocm_device* device, int H, int S, int B) {
    const int units = compute_units(device);
    return B <= units ? S >= 4 : B <= (H == 64 ? 2 : H == 32 ? 5 : 3) * units && S >= (H == 64 ? 20 : 8);
}
bool overlap(const float* a, size_t n, const float* b, size_t m) { return (uintptr_t)a < (uintptr_t)(b + m) && (uintptr_t)b < (uintptr_t)(a + n); }
int even_sixteens(int columns) { return 2 * rlt_div_up(columns, 32); }
// Where the input gates / the weight gradients are formed beside the recurrence. The fp32 matrix instructions and the vector unit of a SIMD take turns, so that what goes beside the
// recurrence lengthens its steps by the time it takes, on as many compute units as there are workgroups, and saves what the launches cost that share the work out over all of them.
// Forward (ns, fitted to both sides at 1 to 200 steps, 1 to 1,024 rows, 3 to 160 inputs; groups of four steps are whole): the launch in front costs a constant, by the kernel that it is and the words
// of its loads, and a share of every row; beside the recurrence a step takes 27 or 24 per sixteen inputs longer than the launch's own. us, launches / beside:
//   146 inputs 16 steps   16 rows 19.0 / 20.2, 256 rows 22.3 / 21.1; 64 steps 512 rows 62.6 / 64.8, 1,024 rows 77.5 / 65.3; 1 step 64 rows 11.5 / 8.3
//   128 inputs 13 steps   64 rows 15.8 / 17.8; 20 steps 16 rows 19.2 / 22.3; 24 steps 400 rows 31.1 / 27.0
//    64 inputs 16 steps   16 rows 15.8 / 14.9; 32 steps 16 rows 23.5 / 24.8, 256 rows 27.9 / 26.2; 64 steps 256 rows 49.0 / 46.3; 20 inputs 64 steps 16 rows 40.4 / 39.1, 1,024 rows 60.8 / 42.0
// Up to two rows per compute unit the recurrence of its own is the faster one (rows_forward; the figures above are with four rows to a workgroup): 3 inputs 16 steps 64 rows 12.8 / 13.3, 64 steps 256 rows
// 37.4 / 41.4, 512 rows 44.4 / 42.5; 146 inputs 8 steps 64 rows 13.4 / 13.0, 16 steps 256 rows 18.9 / 20.9. Over 528 shapes (1 to 128 steps, 16 to 512 rows, 3 to 160 inputs) the side that the
// rule takes is 0.4 % above the faster one on average, and nowhere more than 3 % slower than the one taken before a workgroup per row.
// Backward (54 ns a step and 46 per sixteen inputs), us, launches / beside, 64 steps:
//   146 inputs 256 rows 61.6 / 78.0, 512 rows 81.1 / 80.0, 1,024 rows 132.7 / 85.7; 64 inputs 256 rows 52.5 / 58.6, 512 rows 64.3 / 60.2; 3 inputs 64 rows 47.5 / 50.6, 1,024 rows 79.1 / 55.3;
//   146 inputs 1,024 rows 24 steps 57.7 / 44.0
bool inputs_beside(const rlt_rocm_device* device, const rlt_gru_layer* L, const float* input, int S, int B) {
    if (!one_group_per_unit(device, L, B) || L->input_dim > GP_INPUTS) return false;
    // steps are read after earlier ones are written: not where the outputs replace the inputs (the launch in front has read all of them)
    const size_t rows = (size_t)S * B, inputs = rows * L->input_dim;
    if (overlap(input, inputs, L->output, rows * 64) || overlap(input, inputs, L->n_pre_pre_activation, rows * 64) || overlap(input, inputs, L->post_activation, rows * 3 * 64)) return false;
    const int I = L->input_dim;
    const int units = compute_units(device);
    const double by_row = B <= units ? 280.0 * S - 2000.0 : rows_forward(device, 64, B) ? 70.0 * S - 500.0 : 0.0;      // what the recurrence of its own has from a workgroup per row
    const bool by_rows = I > 32 && I % 2 == 0 && rows >= 2048;      // the launch in front is rows_forward_kernel (rlt_gemm_rows_forward)
    const double launch = by_rows ? 3750.0 : I <= 32 ? 5800.0 : I % 4 == 0 ? 2400.0 : I % 2 == 0 ? 2600.0 : 3200.0;
    return (by_rows ? 27.2 : 23.8) * 4 * rlt_div_up(S, 4) * even_sixteens(I) + by_row <= launch + ((by_rows ? 0.143 : 0.185) + 0.0017 * I) * rows;
}
// The weight gradients of gru_gradients_kernel: pairs of column tiles, shares of the rows (workgroups for the whole chip, but at least eight steps of four rows to a wavefront; once, twice ... so many that no sum is longer than
// 256 steps, for its error's sake), blocks of sums
struct GradientShape { int columns, shares, blocks; };
GradientShape gradient_shape(const rlt_rocm_device* device, const rlt_gru_layer* L, int rows) {
    const int H = L->hidden_dim, parts = H == 64 ? 1 : H == 32 ? 2 : 4, columns = rlt_div_up(L->input_dim, 32) + rlt_div_up(H, 32);
    const int chip = compute_units(device) / columns > 1 ? compute_units(device) / columns : 1, most = rows / (32 * parts) > 1 ? rows / (32 * parts) : 1;
    const int shares = most < chip ? most : chip * rlt_div_up(rows, 4 * 256 * parts * chip);
    return {columns, shares, shares * parts};
}
size_t gradient_shares_bytes(const rlt_rocm_device* device, const rlt_gru_layer* L, int rows) { return gradient_shape(device, L, rows).blocks * gradient_block(L->hidden_dim, L->input_dim) * sizeof(float); }
// Where they are (widths 16, 32, 64): not where width 64 meets 65,536 rows and more of 66 to 160 inputs, an even number, which wgrad_wide_kernel (gemm.hip) reads once. us of the backward pass
// with contractions and sums per gradient / this, width 64: 146 inputs 16 steps 4,000 rows 141 / 127, 64 steps 2,048 rows 230 / 249, 16 steps 8,192 rows 247 / 303; 33 inputs 64 steps 2,048 rows 200 / 179,
// 170 inputs 64 steps 1,024 rows 167 / 143, 300 inputs 64 rows 65.9 / 52.5, 1,024 rows 212 / 189, 1,000 inputs 64 rows 78.7 / 66.5, 1,024 rows 503 / 436; width 32, 500 inputs 64 rows 84.4 / 54.0, 1,000 inputs 1,024 rows
// 256 / 250, 146 inputs 64 steps 4,096 rows 296 / 243; width 16, 146 inputs 32 steps 8,192 rows 262 / 147, 1,000 inputs 64 steps 1,024 rows 179 / 142. A stream that records a graph while the handle's
// scratch memory has room for a contraction's shares but not for these (rlt_scratch_reaches) takes the contractions too.
bool gradients_in_one(const rlt_gru_layer* L, int S, int B) {
    const int H = L->hidden_dim, I = L->input_dim;
    return (H == 16 || H == 32 || H == 64) && I <= 1024 && !(H == 64 && (size_t)S * B >= 65536 && I > 64 && I <= 160 && I % 2 == 0);
}
// (A stream that records a graph takes no launches for whose shares the handle's scratch memory has no room: a workgroup per row is then no reason for them.)
bool weights_beside(const rlt_rocm_device* device, const rlt_gru_layer* L, int S, int B, size_t room) {      // room: bytes of the caller's workspace that nothing else is kept in
    if (!one_group_per_unit(device, L, B) || L->input_dim > GW_INPUTS || rlt_div_up(B, GM_ROWS) * gru_gradient_block(L->input_dim) * sizeof(float) > room) return false;
    const bool by_launches = !device->capturing || (gradients_in_one(L, S, B) && rlt_scratch_reaches(device, gradient_shares_bytes(device, L, S * B)));
    const double by_row = !by_launches || !rows_backward(device, 64, S, B) ? 0.0 : 110.0 * S - (B <= compute_units(device) ? 1500.0 : 2000.0);      // what the recurrence of its own has from a workgroup per row
    return S * (54.0 + 46.0 * even_sixteens(L->input_dim)) + by_row <= 3400.0 + (0.35 + 0.0037 * L->input_dim) * S * B;
}
int finish_gradients(rlt_rocm_device* device, const rlt_gru_layer* L, const float* blocks, int n, size_t stride, const float* hidden, int n_hidden, size_t hidden_stride) {
    const int H = L->hidden_dim, I = L->input_dim;
    hipLaunchKernelGGL(gru_gradient_finish_kernel, dim3((unsigned)((gradient_block(H, I) + 63) / 64 + H / 4)), dim3(256), 0, device->stream, blocks, n, stride, hidden, n_hidden, hidden_stride, H, I,
                       L->d_weights_input, L->d_biases_input, L->d_weights_hidden, L->d_biases_hidden);
    return rlt_launch_status(device);
}
// the kernels' sixteens of `columns` (at most 160) columns: an even number, so that a few instances do
template <class F>
void by_sixteens(int columns, F&& launch) {
    if (columns <= 32) launch(std::integral_constant<int, 2>{});
    else if (columns <= 64) launch(std::integral_constant<int, 4>{});
    else if (columns <= 96) launch(std::integral_constant<int, 6>{});
    else if (columns <= 128) launch(std::integral_constant<int, 8>{});
    else launch(std::integral_constant<int, 10>{});
}
int rows_per_group(int H) { return GRU_THREADS / H; }
size_t lds_bytes(int H, bool backward) { return ((size_t)3 * H * H + (size_t)rows_per_group(H) * (backward ? 3 * H : H)) * sizeof(float); }

}  // namespace

extern "C" {

size_t rlt_rocm_gru_workspace_bytes(const rlt_gru_layer* L, int S, int B) {
    if (!L || S < 1 || B < 1 || L->hidden_dim < 1) return 0;
    const size_t rows = (size_t)S * B, H = (size_t)L->hidden_dim;
    return align256(rows * 3 * H * sizeof(float)) * 2 + align256(rows * H * sizeof(float)) + align256((size_t)B * H * sizeof(float)) + 256;
}

int rlt_rocm_gru_forward(rlt_rocm_device* device, const rlt_gru_layer* L, const float* input, const uint8_t* reset, int S, int B, void* workspace, size_t workspace_bytes) {
    (void)workspace; (void)workspace_bytes;
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(layer_ok(L) && input && S > 0 && B > 0);
    const int H = L->hidden_dim;
    if (lds_bytes(H, false) > (size_t)device->lds_bytes) return RLT_E_UNSUPPORTED;
    GruArgs a = {}; a.L = *L; a.input = input; a.reset = reset; a.S = S; a.B = B; a.rows_per_group = rows_per_group(H);
    if (inputs_beside(device, L, input, S, B)) {
        const dim3 grid4(rlt_div_up(B, GM_ROWS)), block(GP_THREADS);
        by_sixteens(L->input_dim, [&](auto groups) {
            constexpr int G = decltype(groups)::value;
            if (L->fast_tanh) hipLaunchKernelGGL((gru_forward_inputs_kernel<G, true>), grid4, block, 0, device->stream, a); else hipLaunchKernelGGL((gru_forward_inputs_kernel<G, false>), grid4, block, 0, device->stream, a);
        });
        return rlt_launch_status(device);
    }
    // W_i x + b_i for every step at once, into post_activation
    int rc = rlt_gemm_rows_forward(device, input, L->input_dim, L->weights_input, L->biases_input, L->post_activation, 3 * H, S * B, L->input_dim, 3 * H);
    if (rc == RLT_E_UNSUPPORTED)
        rc = rlt_gemm_forward(device, input, L->input_dim, L->weights_input, L->biases_input, RLT_ACT_IDENTITY, nullptr, nullptr, L->post_activation, 3 * H, S * B, L->input_dim, 3 * H);
    if (rc) return rc;
    if (H == 64 || H == 32 || H == 16) {
        const bool fast = L->fast_tanh != 0;      // a template parameter: as a run-time switch inside the step it cost 10% at width 64
        if (rows_forward(device, H, B)) {
            auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(B), dim3(gru_row_threads(H)), 0, device->stream, a); };
            if (H == 64) { if (fast) launch(gru_forward_row_kernel<64, GATES_FAST>); else launch(gru_forward_row_kernel<64, GATES_HARDWARE>); }
            else if (H == 32) { if (fast) launch(gru_forward_row_kernel<32, GATES_FAST>); else launch(gru_forward_row_kernel<32, GATES_EXACT>); }
            else { if (fast) launch(gru_forward_row_kernel<16, GATES_FAST>); else launch(gru_forward_row_kernel<16, GATES_EXACT>); }
            return rlt_launch_status(device);
        }
        const dim3 grid(rlt_div_up(B, GRU_THREADS / H)), block(GRU_THREADS);      // GRU_THREADS / 64 wavefronts of 64 / H rows
        if (H == 64) {
            const dim3 grid4(rlt_div_up(B, GM_ROWS));
            if (fast) hipLaunchKernelGGL(gru_forward_mfma_kernel<true>, grid4, block, 0, device->stream, a); else hipLaunchKernelGGL(gru_forward_mfma_kernel<false>, grid4, block, 0, device->stream, a);
        }
        else if (H == 32) { if (fast) hipLaunchKernelGGL((gru_forward_reg_kernel<32, true>), grid, block, 0, device->stream, a); else hipLaunchKernelGGL((gru_forward_reg_kernel<32, false>), grid, block, 0, device->stream, a); }
        else { if (fast) hipLaunchKernelGGL((gru_forward_reg_kernel<16, true>), grid, block, 0, device->stream, a); else hipLaunchKernelGGL((gru_forward_reg_kernel<16, false>), grid, block, 0, device->stream, a); }
        return rlt_launch_status(device);
    }
    const size_t lds = lds_bytes(H, false);
    RLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gru_forward_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(gru_forward_kernel, dim3(rlt_div_up(B, a.rows_per_group)), dim3(GRU_THREADS), lds, device->stream, a);
    return rlt_launch_status(device);
}

int rlt_rocm_gru_backward(rlt_rocm_device* device, const rlt_gru_layer* L, const float* input, float* d_output, float* d_input, const uint8_t* reset, int S, int B,
                          int want_weight_gradients, void* workspace, size_t workspace_bytes) {
    if (!device) return RLT_E_NOT_INITIALISED;
    RLT_REQUIRE(layer_ok(L) && d_output && S > 0 && B > 0 && (input || !want_weight_gradients));
    RLT_REQUIRE(!want_weight_gradients || (L->d_weights_input && L->d_biases_input && L->d_weights_hidden && L->d_biases_hidden));
    RLT_REQUIRE(workspace && workspace_bytes >= rlt_rocm_gru_workspace_bytes(L, S, B));
    const int H = L->hidden_dim, I = L->input_dim, rows = S * B;
    if (lds_bytes(H, true) > (size_t)device->lds_bytes) return RLT_E_UNSUPPORTED;
    char* w = reinterpret_cast<char*>(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
    float* buffer_input = (float*)w; w += align256((size_t)rows * 3 * H * sizeof(float));
    float* buffer_hidden = (float*)w; w += align256((size_t)rows * 3 * H * sizeof(float));
    float* h_previous = (float*)w; w += align256((size_t)rows * H * sizeof(float));
    float* db_hn_partial = (float*)w;
    GruArgs a = {}; a.L = *L; a.input = input; a.reset = reset; a.d_output = d_output; a.S = S; a.B = B;
    float* const blocks = d_input ? buffer_hidden : buffer_input;
    if (want_weight_gradients && weights_beside(device, L, S, B, (size_t)((char*)workspace + workspace_bytes - (char*)blocks))) {
        const int groups = rlt_div_up(B, GM_ROWS);
        a.buffer_input = d_input ? buffer_input : nullptr; a.blocks = blocks;
        by_sixteens(I, [&](auto tiles) { hipLaunchKernelGGL(gru_backward_weights_kernel<decltype(tiles)::value>, dim3(groups), dim3(GP_THREADS), 0, device->stream, a); });
        const int rc = finish_gradients(device, L, blocks, groups, gru_gradient_block(I), blocks + gradient_block(H, I), groups, gru_gradient_block(I));
        if (rc || !d_input) return rc;
        return rlt_gemm_backward_input(device, buffer_input, 3 * H, L->weights_input, d_input, I, nullptr, 0, 0, rows, I, 3 * H);      // :688
    }
    a.buffer_input = buffer_input; a.buffer_hidden = buffer_hidden;
    a.h_previous = h_previous; a.db_hn_partial = want_weight_gradients ? db_hn_partial : nullptr; a.rows_per_group = rows_per_group(H);
    if (H == 64 || H == 32 || H == 16) {
        const dim3 grid(rlt_div_up(B, GRU_THREADS / H)), block(GRU_THREADS);
        if (rows_backward(device, H, S, B)) {
            auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(B), dim3(gru_row_threads(H)), 0, device->stream, a); };
            if (H == 64) launch(gru_backward_row_kernel<64>); else if (H == 32) launch(gru_backward_row_kernel<32>); else launch(gru_backward_row_kernel<16>);
        } else if (H == 64) {
            const dim3 grid4(rlt_div_up(B, GM_ROWS));
            const int units = compute_units(device);
            if (backward_by_rows(units, S, B)) hipLaunchKernelGGL(gru_backward_rows_kernel, grid4, block, 0, device->stream, a);
            else if ((int)grid4.x > 3 * units) hipLaunchKernelGGL((gru_backward_mfma_kernel<2, 4>), grid4, block, 0, device->stream, a);
            else hipLaunchKernelGGL((gru_backward_mfma_kernel<4, 2>), grid4, block, 0, device->stream, a);
        }
        else if (H == 32) hipLaunchKernelGGL(gru_backward_reg_kernel<32>, grid, block, 0, device->stream, a);
        else hipLaunchKernelGGL(gru_backward_reg_kernel<16>, grid, block, 0, device->stream, a);
    } else {
        const size_t lds = lds_bytes(H, true);
        RLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gru_backward_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(gru_backward_kernel, dim3(rlt_div_up(B, a.rows_per_group)), dim3(GRU_THREADS), lds, device->stream, a);
    }
    int rc = rlt_launch_status(device);
    if (rc) return rc;
    const GradientShape shape = gradient_shape(device, L, rows);
    const size_t shares_bytes = gradient_shares_bytes(device, L, rows);
    if (want_weight_gradients && gradients_in_one(L, S, B) && rlt_scratch_reaches(device, shares_bytes)) {
        float* shares = nullptr;
        if ((rc = rlt_scratch(device, shares_bytes, (void**)&shares))) return rc;
        const GradientArgs g = {buffer_input, buffer_hidden, input, h_previous, shares, rows, I, rlt_div_up(I, 32)};
        const dim3 grid(shape.columns, shape.shares), block(256);
        if (H == 64) hipLaunchKernelGGL(gru_gradients_kernel<4>, grid, block, 0, device->stream, g);
        else if (H == 32) hipLaunchKernelGGL(gru_gradients_kernel<2>, grid, block, 0, device->stream, g);
        else hipLaunchKernelGGL(gru_gradients_kernel<1>, grid, block, 0, device->stream, g);
        if ((rc = finish_gradients(device, L, shares, shape.blocks, gradient_block(H, I), db_hn_partial, B, H))) return rc;
    } else if (want_weight_gradients) {
        if ((rc = rlt_gemm_wgrad(device, buffer_input, 3 * H, input, I, L->d_weights_input, L->d_biases_input, rows, I, 3 * H, false, true))) return rc;       // :677-678
        if ((rc = rlt_gemm_wgrad(device, buffer_hidden, 3 * H, h_previous, H, L->d_weights_hidden, nullptr, rows, H, 3 * H, false, true))) return rc;         // :693-742
        hipLaunchKernelGGL(gru_bias_hidden_kernel, dim3(H), dim3(256), 0, device->stream, (const float*)db_hn_partial, B, H, (const float*)L->d_biases_input, L->d_biases_hidden);
        if ((rc = rlt_launch_status(device))) return rc;
    }
    if (d_input) rc = rlt_gemm_backward_input(device, buffer_input, 3 * H, L->weights_input, d_input, I, nullptr, 0, 0, rows, I, 3 * H);           // :688
    return rc;
}

}  // extern "C"
