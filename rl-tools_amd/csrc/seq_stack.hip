// Passes of the reference's recurrent approximators (rl/algorithms/sac/loop/core/approximators_gru.h:13-74: dense, GRU, GRU, dense) over a batch of sequences, all
// layers in one launch (nn_models/sequential/operations_generic.h:277-428, nn/layers/gru/operations_generic.h:231-341, :594-795).
//
// Batch rows are independent, layers depend on each other only step by step: a workgroup carries ONE batch row, its wavefronts are the stages of a pipeline, and a
// stage works a step or two behind the previous stage (one workgroup barrier per tick orders LDS only; the slots between two stages are double-buffered). Forward: dense
// layer and first input projection | first recurrence | second input projection | second recurrence | output layer; backward, from the last step on: output layer |
// second recurrence | its input gradient | first recurrence | its input gradient and the dense layer's | the input's gradient.
// Weight gradients are contractions over all steps and rows, done afterwards for all layers by one launch on the matrix cores (and a second that adds the shares of the
// rows up).
// Bound: the instructions of a recurrence's step. A wavefront is alone on its SIMD and issues one instruction every four to five cycles whatever it is (vector, scalar,
// wait), so a step takes its instruction count: about 115 at width 32, 48 of them the products. Hence the forms below: values exchanged between lanes instead of through
// LDS, the r gate in one half of the lanes while z is in the other, stores and LDS writes by all lanes of a unit rather than under an exec mask, addresses moved on
// instead of formed, loops unrolled to the slots' parity, the stages around the recurrences without a choice of activation per step where it is relu (a tick takes as long as its longest stage: 341 -> 332 us
// for the training set of 100 sequences of 100 steps, 1,000 sequences 1,481 -> 1,456). That set (actor of width 16, critics of width 32) has four forward launches of 37.9 us on average and three backward
// launches of 35.3; a launch per layer with a row per 32 lanes took 0.59 us per step at width 32 and 0.45 at 16, one
// layer after the other, plus launches for the dense layers, projections and gradients.
#include "seq_stack.h"
#include "gemm.h"
#include "batch_tile.h"
#include <utility>

namespace {
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int MAX_IN = 16, MAX_OUT = 16, FORWARD_STAGES = 5, BACKWARD_STAGES = 6, MAX_PASSES = 3;
constexpr size_t LDS_LIMIT = 48 * 1024;      // three to four workgroups per compute unit

__device__ __forceinline__ void swap32(float& a, float& b) {      // the upper half of a's lanes against the lower half of b's
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false); a = __uint_as_float(s[0]); b = __uint_as_float(s[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {      // the odd rows of sixteen lanes of a against the even rows of b
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false); a = __uint_as_float(s[0]); b = __uint_as_float(s[1]);
}
// the sum of x over the lanes of one unit (64 / PARTS apart); every one of them receives it
template <int PARTS>
__device__ __forceinline__ float sum_parts(float x) {
    float y = x;
    if (PARTS == 4) { swap16(x, y); x += y; y = x; }
    swap32(x, y);
    return x + y;
}
// The reference's rational tanh (math/operations_generic.h:247-255) with the quotient from v_rcp_f32 and two corrections (the divisor lies in [27, 108]: no scaling is
// needed, and the result is within one rounding of the quotient)
__device__ __forceinline__ float fast_tanh(float x) {
    x = fminf(fmaxf(x, -3.0f), 3.0f);
    const float x2 = x * x, num = x * (27.0f + x2), den = 27.0f + 9.0f * x2;
    float q = __builtin_amdgcn_rcpf(den);
    q = fmaf(fmaf(-den, q, 1.0f), q, q);
    const float y = num * q;
    return fmaf(fmaf(-den, y, num), q, y);
}
template <bool FAST> __device__ __forceinline__ float gate_sigmoid(float x) { return FAST ? 0.5f * fast_tanh(0.5f * x) + 0.5f : 1.0f / (1.0f + expf(-x)); }
template <bool FAST> __device__ __forceinline__ float gate_tanh(float x) { return FAST ? fast_tanh(x) : tanhf(x); }

// Products of a vector with rows (or columns) of a recurrence's weights: every lane of a unit holds the unit's value, and a multiply-add whose first operand carries the
// row_newbcast control takes it from one lane of each row of sixteen lanes. At width 32 the rows hold units 0-15, 16-31, 0-15, 16-31: after an exchange the first two
// have units 0-15 in their lanes and the last two units 16-31, each row forms its units' three sums over that half of the reduction index, and the halves meet across the
// rows. At width 16 the rows of lanes are the three gates (and nothing): each forms its gate's sums over all sixteen units.
// (The control in the multiply-add itself: left to the compiler, each broadcast is an instruction of its own. The data of such an operand must have been written two wait
// states before it is read, which the compiler does not see to inside an asm statement: wait_for_dpp() stands between, and what it has passed is all that is multiplied.
// tests/test_dpp_wait_states.py looks the built instructions over.)
__device__ __forceinline__ void wait_for_dpp(float& x) { asm volatile("s_nop 1" : "+v"(x)); }
__device__ __forceinline__ void wait_for_dpp(float& x, float& y, float& z) { asm volatile("s_nop 1" : "+v"(x), "+v"(y), "+v"(z)); }
// Several to a statement: the compiler separates statements that hand a register on by an idle instruction, whatever they hold (sixteen of them for 48 products: the training set of 100
// sequences of 100 steps 364 -> 354 us).
#define RLT_BCAST(op, acc, x, w, k) "v_" op "_f32_dpp %" #acc ", %" #x ", %" #w " row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
#define RLT_BCAST3(op, w0, w1, w2, k) RLT_BCAST(op, 0, 3, w0, k) RLT_BCAST(op, 1, 4, w1, k) RLT_BCAST(op, 2, 5, w2, k)
#define RLT_WEIGHTS8(w, k) "v"(w[k]), "v"(w[k + 1]), "v"(w[k + 2]), "v"(w[k + 3]), "v"(w[k + 4]), "v"(w[k + 5]), "v"(w[k + 6]), "v"(w[k + 7])
// acc[i] = the products of x, y, z with sixteen weights each
__device__ __forceinline__ void broadcast_products(float (&acc)[3], float x, float y, float z, const float (&a)[16], const float (&b)[16], const float (&c)[16]) {
    asm(RLT_BCAST3("mul", 6, 14, 22, 0) RLT_BCAST3("fmac", 7, 15, 23, 1) RLT_BCAST3("fmac", 8, 16, 24, 2) RLT_BCAST3("fmac", 9, 17, 25, 3)
        RLT_BCAST3("fmac", 10, 18, 26, 4) RLT_BCAST3("fmac", 11, 19, 27, 5) RLT_BCAST3("fmac", 12, 20, 28, 6) RLT_BCAST3("fmac", 13, 21, 29, 7)
        : "=&v"(acc[0]), "=&v"(acc[1]), "=&v"(acc[2]) : "v"(x), "v"(y), "v"(z), RLT_WEIGHTS8(a, 0), RLT_WEIGHTS8(b, 0), RLT_WEIGHTS8(c, 0));
    asm(RLT_BCAST3("fmac", 6, 14, 22, 8) RLT_BCAST3("fmac", 7, 15, 23, 9) RLT_BCAST3("fmac", 8, 16, 24, 10) RLT_BCAST3("fmac", 9, 17, 25, 11)
        RLT_BCAST3("fmac", 10, 18, 26, 12) RLT_BCAST3("fmac", 11, 19, 27, 13) RLT_BCAST3("fmac", 12, 20, 28, 14) RLT_BCAST3("fmac", 13, 21, 29, 15)
        : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]) : "v"(x), "v"(y), "v"(z), RLT_WEIGHTS8(a, 8), RLT_WEIGHTS8(b, 8), RLT_WEIGHTS8(c, 8));
}
// the products of x with sixteen weights, in three sums
__device__ __forceinline__ void broadcast_products(float (&acc)[3], float x, const float (&a)[16]) {
#define RLT_BCAST1(op, i, w, k) RLT_BCAST(op, i, 3, w, k)
    asm(RLT_BCAST1("mul", 0, 4, 0) RLT_BCAST1("mul", 1, 5, 1) RLT_BCAST1("mul", 2, 6, 2) RLT_BCAST1("fmac", 0, 7, 3) RLT_BCAST1("fmac", 1, 8, 4) RLT_BCAST1("fmac", 2, 9, 5)
        RLT_BCAST1("fmac", 0, 10, 6) RLT_BCAST1("fmac", 1, 11, 7) RLT_BCAST1("fmac", 2, 12, 8) RLT_BCAST1("fmac", 0, 13, 9) RLT_BCAST1("fmac", 1, 14, 10) RLT_BCAST1("fmac", 2, 15, 11)
        RLT_BCAST1("fmac", 0, 16, 12) RLT_BCAST1("fmac", 1, 17, 13) RLT_BCAST1("fmac", 2, 18, 14) RLT_BCAST1("fmac", 0, 19, 15)
        : "=&v"(acc[0]), "=&v"(acc[1]), "=&v"(acc[2]) : "v"(x), RLT_WEIGHTS8(a, 0), RLT_WEIGHTS8(a, 8));
#undef RLT_BCAST1
}
#undef RLT_BCAST3
#undef RLT_BCAST
#undef RLT_WEIGHTS8
// a lane's weights of a [3H x H] matrix: width 32: rows (or columns) u of the three blocks, half p of the reduction index; width 16: row (column) u of block p
template <int H> struct Weights3 { float w[H == 32 ? 3 : 1][16]; };
template <int H>
__device__ __forceinline__ void load_rows3(const float* W, int u, int p, Weights3<H>& R) {
#pragma unroll
    for (int k = 0; k < (H == 32 ? 3 : 1); k++) {
        const float* from = H == 32 ? W + (size_t)(k * H + u) * H + p * 16 : W + (size_t)(min(p, 2) * H + u) * H;
#pragma unroll
        for (int q = 0; q < 16; q += 4) {
            floatx4 v;
            __builtin_memcpy(&v, from + q, sizeof v);      // 16 bytes at a time, whatever the tensor's alignment
            R.w[k][q] = v[0]; R.w[k][q + 1] = v[1]; R.w[k][q + 2] = v[2]; R.w[k][q + 3] = v[3];
        }
    }
}
template <int H>
__device__ __forceinline__ void load_columns3(const float* W, int u, int p, Weights3<H>& R) {
#pragma unroll
    for (int k = 0; k < (H == 32 ? 3 : 1); k++)
#pragma unroll
        for (int q = 0; q < 16; q++) R.w[k][q] = H == 32 ? W[(size_t)(k * H + p * 16 + q) * H + u] : (p < 3 ? W[(size_t)(p * H + q) * H + u] : 0.f);
}
__device__ __forceinline__ float half_in_rows(float v, int p) { float w = v; swap16(v, w); return p ? w : v; }
// (x, y, z have passed wait_for_dpp)
template <int H>
__device__ __forceinline__ void multiply(const Weights3<H>& R, const float& x, const float& y, const float& z, float (&acc)[3]) {
    if constexpr (H == 32) broadcast_products(acc, x, y, z, R.w[0], R.w[1], R.w[2]);
    else { broadcast_products(acc, x, R.w[0]); acc[0] += acc[1] + acc[2]; }
}
// The products of a vector (element u in the lanes of unit u) with rows u of the three blocks. rz: the first block's in the lanes with p = 0, the second's where p = 1
// (width 16: also the third's where p = 2); n: the third's in every lane.
template <int H>
__device__ __forceinline__ void products3(const Weights3<H>& R, float v, int p, float& rz, float& n) {
    float acc[3];
    float x = H == 32 ? half_in_rows(v, p) : v;
    wait_for_dpp(x);
    multiply<H>(R, x, x, x, acc);
    if (H == 32) {
        swap32(acc[0], acc[1]);
        rz = acc[0] + acc[1];
        n = sum_parts<2>(acc[2]);
    } else {
        float a = acc[0], b = acc[0];
        rz = acc[0];
        swap16(a, b); b = a; swap32(a, b);
        n = b;
    }
}
// the sum over three vectors of their products with columns u of the three blocks, in every lane of the unit
template <int H>
__device__ __forceinline__ float product_sum3(const Weights3<H>& R, float x, float y, float z, int p) {
    float acc[3];
    if (H == 32) {
        x = half_in_rows(x, p); y = half_in_rows(y, p); z = half_in_rows(z, p);
        wait_for_dpp(x, y, z);
        multiply<H>(R, x, y, z, acc);
        return sum_parts<2>(acc[0] + (acc[1] + acc[2]));
    }
    float own = p == 0 ? x : p == 1 ? y : p == 2 ? z : 0.f;      // the fourth row of lanes has zero weights, and zero times an infinity is not zero
    wait_for_dpp(own);
    multiply<H>(R, own, own, own, acc);
    return sum_parts<4>(acc[0]);
}

// A stage: `before` ticks until its first step is there, one per step, `after` ticks for the stages behind it. The steps are unrolled U at a time with their number in the
// group as a constant (slots and queues are indexed by it). Whole groups are straight-line code: with an exit before every step, or a request under a condition, the compiler waits where the paths
// meet, once in a group, for everything that is under way (100 sequences of 100 steps, with four steps ahead instead of six, whose queue fits 128 registers but for
// 16 bytes a lane in scratch memory, 354 -> 341 us a set, 1,000 sequences 1,584 -> 1,480). What was requested before the first step is waited for in front of it,
// so that a step waits for its own values and not for the last ones.
template <class F, int... D>
__device__ __forceinline__ void stage_group(int i, F& step, std::integer_sequence<int, D...>) {
    ((__builtin_amdgcn_sched_barrier(0), step(std::integral_constant<int, D>{}, i + D), rlt_lds_barrier()), ...);
}
template <class F, int... D>
__device__ __forceinline__ void stage_rest(int i, int S, F& step, std::integer_sequence<int, D...>) {
    ((i + D < S ? (step(std::integral_constant<int, D>{}, i + D), rlt_lds_barrier()) : (void)0), ...);
}
template <int U, class F>
__device__ __forceinline__ void stage(int S, int before, int after, F&& step) {
    for (int k = 0; k < before; k++) rlt_lds_barrier();
    int i = 0;
    __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
    for (; i + U <= S; i += U) stage_group(i, step, std::make_integer_sequence<int, U>{});
    stage_rest(i, S, step, std::make_integer_sequence<int, U - 1>{});
    for (int k = 0; k < after; k++) rlt_lds_barrier();
}
template <class F> __device__ __forceinline__ void by_condition(bool condition, F&& body) { if (condition) body(std::true_type{}); else body(std::false_type{}); }

// What a workgroup stages in LDS before its first step: the row's `width` values of S steps (at steps * x_step apart, rows of width4 floats) and its reset flags. request() asks for the first values of
// every thread without a condition and waits for nothing; store() writes them down, after the stages have asked for their weights: one trip to memory instead of one per value, flag and the weights.
// The training set of 100 sequences of 100 steps, five such launches: 370 -> 365 us.
template <int THREADS>
struct Staging {
    static constexpr int FIRST = 4;
    const float* x; const uint8_t* reset; size_t x_step, reset_step; int S, width, width4, reversed;
    float value[FIRST]; uint8_t flag;
    __device__ __forceinline__ size_t step(int t) const { return reversed ? S - 1 - t : t; }
    __device__ __forceinline__ void request() {
#pragma unroll
        for (int q = 0; q < FIRST; q++) { const int e = min((int)threadIdx.x + q * THREADS, S * width4 - 1), t = e / width4; value[q] = x[step(t) * x_step + min(e - t * width4, width - 1)]; }
        const uint8_t* const from = reset ? reset : reinterpret_cast<const uint8_t*>(x);      // without flags any address
        flag = from[reset ? step(min((int)threadIdx.x, S - 1)) * reset_step : 0];
    }
    // flags[t] of t < S: whether step t (as numbered here) resets; the caller sets what it knows without memory
    template <class FLAG>
    __device__ __forceinline__ void store(float* values, FLAG&& set_flag) {
#pragma unroll
        for (int q = 0; q < FIRST; q++) { const int e = threadIdx.x + q * THREADS; if (e < S * width4) values[e] = e % width4 < width ? value[q] : 0.f; }
        if ((int)threadIdx.x < S) set_flag(threadIdx.x, reset && flag);
        for (int e = threadIdx.x + FIRST * THREADS; e < S * width4; e += THREADS) { const int t = e / width4, k = e - t * width4; values[e] = k < width ? x[step(t) * x_step + k] : 0.f; }
        for (int t = threadIdx.x + THREADS; t < S; t += THREADS) set_flag(t, reset && reset[step(t) * reset_step]);
        rlt_lds_barrier();
    }
};

struct Gru { const float *W_i, *b_i, *W_h, *b_h, *h0; float *post, *npp, *out; };
struct Forward {
    const float *W0, *b0; float *pre0, *out0; Gru g[2]; const float *W3, *b3; float *pre3, *out3, *also;
    const float* x; const uint8_t* reset; int ldx, in, out, act0, S, B, H, fast, first_block;
};
struct ForwardLaunch { Forward pass[MAX_PASSES]; int n; };

// LDS of a workgroup: the slots between the stages, then the row's inputs (rows of four floats' multiples) and reset flags. A projection's slot: what the r and z gates
// and then the n gate receive (width 16: a fourth row that nobody reads).
template <int H> struct ForwardSlots { float p1[2][4 * H], h1[2][H], p2[2][4 * H], h2[2][H]; };

// the input projection of one step into a slot; the biases of the hidden path's r and z gates ride along
template <int H> struct Projection { Weights3<H> R; float brz, bn; };
template <int H>
__device__ __forceinline__ void load_projection(const Gru& G, int u, int p, Projection<H>& J) {
    load_rows3<H>(G.W_i, u, p, J.R);
    J.brz = p < 2 ? G.b_i[p * H + u] + G.b_h[p * H + u] : 0.f; J.bn = G.b_i[2 * H + u];
}
template <int H>
__device__ __forceinline__ void project(const Projection<H>& J, float v, int u, int p, float* slot) {
    float rz, n;
    products3<H>(J.R, v, p, rz, n);
    slot[p * H + u] = rz + J.brz;      // width 16: the third row is overwritten by the next line, the fourth is nobody's
    slot[2 * H + u] = n + J.bn;
}
template <int H, bool FAST, class READY>
__device__ __forceinline__ void recurrence(const Forward& P, int layer, int lag, const float (*in)[4 * H], float (*out)[H], const uint8_t* flags, int b, int lane, READY& ready) {
    constexpr int PARTS = 64 / H;
    const Gru& G = P.g[layer];
    const int u = lane & (H - 1), p = lane / H;
    Weights3<H> R;
    load_rows3<H>(G.W_h, u, p, R);
    const float bn = G.b_h[2 * H + u], h0 = G.h0[u];
    // where a lane stores what it keeps of a step, moved on from step to step. Width 32: r / z, then n / the n gate's hidden part in the two halves; width 16: one of the
    // four in each row of lanes. The output by all lanes of a unit.
    const size_t stride = (size_t)P.B * H;
    float* const post = G.post + (size_t)b * 3 * H + u; float* const npp = G.npp + (size_t)b * H + u;
    float* keep1 = PARTS == 2 ? post + p * H : p < 3 ? post + p * H : npp; float* keep2 = p ? npp : post + 2 * H; float* keep3 = G.out + (size_t)b * H + u;
    const size_t stride1 = PARTS == 2 || p < 3 ? 3 * stride : stride, stride2 = p ? stride : 3 * stride;
    float h = h0;
    ready();
    stage<2>(P.S, lag, FORWARD_STAGES - 1 - lag, [&](auto d, int t) {
        constexpr int PAR = decltype(d)::value & 1;
        const float x = in[PAR][PARTS == 2 ? p * H + u : min(p, 1) * H + u], xn = in[PAR][2 * H + u];
        const uint8_t flag = flags[t + 1];      // the next step starts from the initial state (the flags end with one more entry)
        float rz, n_hidden;
        __builtin_amdgcn_sched_barrier(0);
        products3<H>(R, h, p, rz, n_hidden);
        __builtin_amdgcn_sched_barrier(0);      // the three words travel while the products are formed
        const bool restart = flag;
        const float an = n_hidden + bn, s = gate_sigmoid<FAST>(x + rz);
        float r = s, z = s;
        if (PARTS == 2) swap32(r, z);
        else { swap16(r, z); float r2 = r, z2 = z; swap32(r, r2); swap32(z, z2); }
        const float n = gate_tanh<FAST>(xn + an * r);
        const float o = n + z * (h - n);
        h = restart ? h0 : o;
        out[PAR][u] = o;
        if (PARTS == 2) { *keep1 = s; *keep2 = p ? an : n; keep2 += stride2; }
        else *keep1 = p < 2 ? s : p == 2 ? n : an;
        *keep3 = o;
        keep1 += stride1; keep3 += stride;
    });
}
template <int H, bool FAST>
__device__ __forceinline__ void forward_row(const Forward& P, int b, char* lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), p = lane / H, S = P.S, in4 = (P.in + 3) & ~3;
    ForwardSlots<H>& L = *reinterpret_cast<ForwardSlots<H>*>(lds);
    float* const xs = reinterpret_cast<float*>(lds + ((sizeof(ForwardSlots<H>) + 15) & ~(size_t)15));
    uint8_t* const flags = reinterpret_cast<uint8_t*>(xs + (size_t)S * in4);
    Staging<64 * FORWARD_STAGES> staging = {P.x + (size_t)b * P.ldx, P.reset ? P.reset + b : nullptr, (size_t)P.B * P.ldx, (size_t)P.B, S, P.in, in4, 0, {}, 0};
    staging.request();
    auto ready = [&]() {
        if (threadIdx.x == 0) flags[S] = 0;
        staging.store(xs, [&](int t, bool resets) { flags[t] = t == 0 || resets; });
    };
    if (wave == 0) {
        // the dense layer and the first recurrence's input projection
        float w0[MAX_IN];
#pragma unroll
        for (int k = 0; k < MAX_IN; k++) w0[k] = k < P.in ? P.W0[(size_t)u * P.in + k] : 0.f;
        const float b0 = P.b0[u];
        Projection<H> J;
        load_projection<H>(P.g[0], u, p, J);
        float* keep = ((p & 1) ? P.out0 : P.pre0) + (size_t)b * H + u;
        const size_t stride = (size_t)P.B * H;
        const int in = P.in, act0 = P.act0;
        const float* row = xs;
        ready();
        by_condition(act0 == RLT_ACT_RELU, [&](auto relu) { stage<2>(S, 0, FORWARD_STAGES - 1, [&](auto d, int) {      // the approximators' activation without the others' branches in every step
            float acc = b0;
            const floatx4* x = reinterpret_cast<const floatx4*>(row);
#pragma unroll
            for (int q = 0; q < MAX_IN / 4; q++)
                if (q == 0 || 4 * q < in) { const floatx4 v = x[q]; acc += v[0] * w0[4 * q]; acc += v[1] * w0[4 * q + 1]; acc += v[2] * w0[4 * q + 2]; acc += v[3] * w0[4 * q + 3]; }
            row += in4;
            const float o = rlt_act(acc, decltype(relu)::value ? (int)RLT_ACT_RELU : act0);
            *keep = (p & 1) ? o : acc;
            keep += stride;
            project<H>(J, o, u, p, L.p1[decltype(d)::value & 1]);
        }); });
    }
    else if (wave == 1) recurrence<H, FAST>(P, 0, 1, L.p1, L.h1, flags, b, lane, ready);
    else if (wave == 2) {
        Projection<H> J;
        load_projection<H>(P.g[1], u, p, J);
        ready();
        stage<2>(S, 2, 2, [&](auto d, int) { project<H>(J, L.h1[decltype(d)::value & 1][u], u, p, L.p2[decltype(d)::value & 1]); });
    }
    else if (wave == 3) recurrence<H, FAST>(P, 1, 3, L.p2, L.h2, flags, b, lane, ready);
    else {
        // the output layer: lane = output, all of the reduction
        float w3[H];
        const int o = min(lane, P.out - 1);
#pragma unroll
        for (int k = 0; k < H; k++) w3[k] = P.W3[(size_t)o * H + k];
        const float b3 = P.b3[o];
        // (without a third place the second is written twice)
        float* pre3 = P.pre3 + (size_t)b * P.out + o; float* out3 = P.out3 + (size_t)b * P.out + o; float* also = P.also ? P.also + (size_t)b * P.out + o : out3;
        const size_t stride = (size_t)P.B * P.out;
        ready();
        stage<2>(S, 4, 0, [&](auto d, int) {
            const floatx4* h = reinterpret_cast<const floatx4*>(L.h2[decltype(d)::value & 1]);
            float a0 = b3, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
            for (int q = 0; q < H / 4; q++) { const floatx4 v = h[q]; a0 += v[0] * w3[4 * q]; a1 += v[1] * w3[4 * q + 1]; a2 += v[2] * w3[4 * q + 2]; a3 += v[3] * w3[4 * q + 3]; }
            const float y = (a0 + a1) + (a2 + a3);
            *pre3 = y; *out3 = y; *also = y;
            pre3 += stride; out3 += stride; also += stride;
        });
    }
}
__global__ __launch_bounds__(64 * FORWARD_STAGES, 5) void seq_stack_forward_kernel(ForwardLaunch K) {
    extern __shared__ __attribute__((aligned(16))) char lds_stack[];
    int k = 0;
    if (K.n > 1 && (int)blockIdx.x >= K.pass[1].first_block) k = 1;
    if (K.n > 2 && (int)blockIdx.x >= K.pass[2].first_block) k = 2;
    const Forward& P = K.pass[k];
    const int b = blockIdx.x - P.first_block;
    if (P.H == 32) { if (P.fast) forward_row<32, true>(P, b, lds_stack); else forward_row<32, false>(P, b, lds_stack); }
    else { if (P.fast) forward_row<16, true>(P, b, lds_stack); else forward_row<16, false>(P, b, lds_stack); }
}

// ---- backward
struct GruBack { const float *W_i, *W_h, *h0, *post, *npp, *out; float *g, *gnr, *hp, *db_hn; };      // g [rows][3H]: gradients at the r, z, n pre-activations of the input path; gnr [rows][H]: of the hidden path's n (r, z are the same)
struct Backward {
    GruBack g[2]; const float *W0, *pre0, *W3, *d_output; float *d_pre0, *d_input; const uint8_t* reset; int in, out, act0, S, B, H, want_w, first_block;
};
struct BackwardLaunch { Backward pass[MAX_PASSES]; int n; };
template <int H> struct BackwardSlots { float dy2[2][H], g2[2][3 * H], dy1[2][H], g1[2][3 * H], dp0[2][H]; };
constexpr int AHEAD = 4;      // steps ahead of its use that a saved value is requested (a load takes several steps)

// A recurrence's way back, step i of S (from the last on). dy: the gradient at its output from the stage above, held in a register from the tick before.
template <int H, class READY>
__device__ __forceinline__ void recurrence_back(const Backward& P, int layer, int lag, const float (*dy)[H], float (*g)[3 * H], const uint8_t* flags, int b, int lane, READY& ready) {
    const GruBack& G = P.g[layer];
    const int u = lane & (H - 1), p = lane / H, S = P.S;
    Weights3<H> R;
    load_columns3<H>(G.W_h, u, p, R);
    const float h0 = G.h0[u];
    const size_t stride = (size_t)P.B * H, last = (size_t)(S - 1) * stride + (size_t)b * H;      // the row's last step in an array of H columns
    const float* post = G.post + 3 * last + u; const float* npp = G.npp + last + u; const float* state = G.out + last + u;
    struct Saved { float r, z, n, npp, hp; };
    Saved queue[AHEAD];
    auto request = [&](int i, Saved& v) {      // step i's values, beyond the last step the last one's again; the state is the one before the step (the first step takes the initial one)
        const size_t on = i + 1 < S ? stride : 0;
        state -= on;
        v.r = post[0]; v.z = post[H]; v.n = post[2 * H]; v.npp = *npp; v.hp = *state;
        post -= 3 * on; npp -= on;
    };
#pragma unroll
    for (int d = 0; d < AHEAD; d++) request(d, queue[d]);
    const bool want_w = P.want_w;
    float* to_g = want_w ? G.g + 3 * last + u : nullptr; float* to_gnr = want_w ? G.gnr + last + u : nullptr; float* to_hp = want_w ? G.hp + last + u : nullptr;
    float carry = 0.f, db_hn = 0.f, above = 0.f;
    ready();
    for (int k = 0; k < lag - 1; k++) rlt_lds_barrier();
    above = dy[0][u];
    uint8_t flag = flags[0];
    rlt_lds_barrier();
    by_condition(want_w, [&](auto want) { stage<AHEAD>(S, 0, BACKWARD_STAGES + 1 - lag, [&](auto d, int i) {
        constexpr int N = decltype(d)::value;
        const Saved v = queue[N];
        const float dh = above + carry;
        above = dy[(N + 1) & 1][u];      // the next step's
        const bool from_initial = flag;
        flag = flags[min(i + 1, S - 1)];
        const float hp = from_initial ? h0 : v.hp, t = dh * (1.0f - v.z);
        const float gz = t * (hp - v.n) * v.z;
        const float gn = t * (1.0f - v.n * v.n);
        const float gr = gn * v.npp * v.r * (1.0f - v.r);
        const float gnr = gn * v.r;
        float through = dh * v.z;
        asm volatile("" : "+v"(through));      // (not formed below by a multiply-add that would keep the entry's z)
        request(i + AHEAD, queue[N]);      // behind the last use of the entry: before it, the group would start with copies of all entries, and with waits for them
        g[N & 1][u] = gr; g[N & 1][H + u] = gz; g[N & 1][2 * H + u] = gn;
        const float sum = product_sum3<H>(R, gr, gz, gnr, p);
        carry = from_initial ? 0.f : through + sum;
        if constexpr (decltype(want)::value) {
            to_g[0] = gr; to_g[H] = gz; to_g[2 * H] = gn; *to_gnr = gnr; *to_hp = hp;
            to_g -= 3 * stride; to_gnr -= stride; to_hp -= stride;
            // the reference drops reset samples from the b_hn gradient, but for the sequence's first step (their buffer rows are zeroed before that sum, gru/operations_generic.h:716-749)
            db_hn += from_initial && i + 1 < S ? 0.f : gnr;
        }
    }); });
    if (want_w && p == 0) G.db_hn[(size_t)b * H + u] = db_hn;
}
template <int H>
__device__ __forceinline__ void backward_row(const Backward& P, int b, char* lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), p = lane / H, S = P.S, out4 = (P.out + 3) & ~3;
    BackwardSlots<H>& L = *reinterpret_cast<BackwardSlots<H>*>(lds);
    // the loss gradient and the reset flags, from the last step on
    float* const ds = reinterpret_cast<float*>(lds + ((sizeof(BackwardSlots<H>) + 15) & ~(size_t)15));
    uint8_t* const flags = reinterpret_cast<uint8_t*>(ds + (size_t)S * out4);
    Staging<64 * BACKWARD_STAGES> staging = {P.d_output + (size_t)b * P.out, P.reset ? P.reset + b : nullptr, (size_t)P.B * P.out, (size_t)P.B, S, P.out, out4, 1, {}, 0};
    staging.request();
    auto ready = [&]() { staging.store(ds, [&](int i, bool resets) { flags[i] = i == S - 1 || resets; }); };
    // ticks behind the first stage: 2 (second recurrence), 3, 5 (first recurrence), 6, 7
    if (wave == 0) {
        float w3[MAX_OUT];
#pragma unroll
        for (int o = 0; o < MAX_OUT; o++) w3[o] = o < P.out ? P.W3[(size_t)o * H + u] : 0.f;
        const int out = P.out;
        const float* row = ds;
        ready();
        stage<2>(S, 0, BACKWARD_STAGES + 1, [&](auto d, int) {
            const floatx4* x = reinterpret_cast<const floatx4*>(row);
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < MAX_OUT / 4; q++)
                if (q == 0 || 4 * q < out) { const floatx4 v = x[q]; s += v[0] * w3[4 * q]; s += v[1] * w3[4 * q + 1]; s += v[2] * w3[4 * q + 2]; s += v[3] * w3[4 * q + 3]; }
            row += out4;
            L.dy2[decltype(d)::value & 1][u] = s;
        });
    }
    else if (wave == 1) recurrence_back<H>(P, 1, 2, L.dy2, L.g2, flags, b, lane, ready);
    else if (wave == 2) {
        Weights3<H> R;
        load_columns3<H>(P.g[1].W_i, u, p, R);
        ready();
        stage<2>(S, 3, 4, [&](auto d, int) {
            constexpr int PAR = decltype(d)::value & 1;
            L.dy1[PAR][u] = product_sum3<H>(R, L.g2[PAR][u], L.g2[PAR][H + u], L.g2[PAR][2 * H + u], p);
        });
    }
    else if (wave == 3) recurrence_back<H>(P, 0, 5, L.dy1, L.g1, flags, b, lane, ready);
    else if (wave == 4) {
        Weights3<H> R;
        load_columns3<H>(P.g[0].W_i, u, p, R);
        float queue[AHEAD];
        const size_t stride = (size_t)P.B * H, last = (size_t)(S - 1) * stride + (size_t)b * H + u;
        const float* from = P.pre0 + last;
        float* to = P.want_w ? P.d_pre0 + last : nullptr;
        const int act0 = P.act0;
        auto request = [&](int i, float& v) { v = *from; from -= i + 1 < S ? stride : 0; };
#pragma unroll
        for (int d = 0; d < AHEAD; d++) request(d, queue[d]);
        ready();
        by_condition(to != nullptr, [&](auto want) { by_condition(act0 == RLT_ACT_RELU, [&](auto relu) { stage<AHEAD>(S, 6, 1, [&](auto d, int i) {
            constexpr int N = decltype(d)::value, PAR = N & 1;
            float slope = rlt_dact(queue[N], decltype(relu)::value ? (int)RLT_ACT_RELU : act0);
            asm volatile("" : "+v"(slope));
            request(i + AHEAD, queue[N]);
            const float v = product_sum3<H>(R, L.g1[PAR][u], L.g1[PAR][H + u], L.g1[PAR][2 * H + u], p) * slope;
            L.dp0[PAR][u] = v;
            if constexpr (decltype(want)::value) { *to = v; to -= stride; }
        }); }); });
    } else {
        float w0[H];
        const int k = min(lane, P.in - 1);
        if (P.d_input) {
#pragma unroll
            for (int j = 0; j < H; j++) w0[j] = P.W0[(size_t)j * P.in + k];
        }
        const size_t stride = (size_t)P.B * P.in;
        float* to = P.d_input ? P.d_input + (size_t)(S - 1) * stride + (size_t)b * P.in + k : nullptr;
        ready();
        stage<2>(S, 7, 0, [&](auto dd, int) {
            if (!to) return;
            const floatx4* d = reinterpret_cast<const floatx4*>(L.dp0[decltype(dd)::value & 1]);
            float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
            for (int q = 0; q < H / 4; q++) { const floatx4 v = d[q]; a0 += v[0] * w0[4 * q]; a1 += v[1] * w0[4 * q + 1]; a2 += v[2] * w0[4 * q + 2]; a3 += v[3] * w0[4 * q + 3]; }
            *to = (a0 + a1) + (a2 + a3);
            to -= stride;
        });
    }
}
__global__ __launch_bounds__(64 * BACKWARD_STAGES, 4) void seq_stack_backward_kernel(BackwardLaunch K) {
    extern __shared__ __attribute__((aligned(16))) char lds_stack[];
    int k = 0;
    if (K.n > 1 && (int)blockIdx.x >= K.pass[1].first_block) k = 1;
    if (K.n > 2 && (int)blockIdx.x >= K.pass[2].first_block) k = 2;
    const Backward& P = K.pass[k];
    if (P.H == 32) backward_row<32>(P, blockIdx.x - P.first_block, lds_stack);
    else backward_row<16>(P, blockIdx.x - P.first_block, lds_stack);
}

// ---- weight gradients: a list of contractions d^T x over the rows (steps times batch), each job's rows shared out to SPLITS groups of workgroups (a multiple of the
// eight XCDs, so that an XCD reads an eighth of the rows); the second launch adds the shares up in order and onto the gradients
constexpr int MAX_JOBS = 20, WAVES = 4, MT = 2, TM = 16 * MT, SPLITS = 32;
struct Job {
    const float* a; const float* b; float* gradient; float* bias; float* bias_copy;      // bias (optional): column sums of a; bias_copy: receives the first copy_n of the result as well
    int lda, m, ldb, n, rows, overwrite, copy_n, first_block, first_element;             // n = 0: only the column sums
};
struct JobLaunch { Job job[MAX_JOBS]; int n, elements; float* partial; };      // partial [SPLITS][elements], a job's m n products then its m column sums
__device__ __forceinline__ int find_job(const JobLaunch& K, int at, bool element) {
    int k = 0;
    for (int q = 1; q < K.n; q++) if (at >= (element ? K.job[q].first_element : K.job[q].first_block)) k = q;
    return k;
}
__global__ __launch_bounds__(64 * WAVES) void seq_gradient_kernel(JobLaunch K) {
    using namespace rlt_batch;
    __shared__ Parts<WAVES, MT> P;
    const int split = blockIdx.x % SPLITS, block = blockIdx.x / SPLITS;
    const Job& J = K.job[find_job(K, block, false)];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = J.n ? (J.n + TN - 1) / TN : 1, tile = block - J.first_block, mt = tile / tiles, nt = tile - mt * tiles;
    const int per = ((J.rows + WAVES * SPLITS - 1) / (WAVES * SPLITS) + 3) & ~3, k0 = (WAVES * split + wave) * per, k1 = min(J.rows, k0 + per);
    rlt_batch::floatx4 c[MT][2];
    float bias[MT];
    tile_product<MT>(J.a, J.lda, J.m, TM * mt, J.n ? J.b : J.a, J.n ? J.ldb : J.lda, J.n, TN * nt, J.rows, k0, k1, r, g, c, bias);
    place_parts(P, wave, r, g, c, bias);
    rlt_lds_barrier();
    float* const out = K.partial + (size_t)split * K.elements + J.first_element;
    for (int e = threadIdx.x; e < TM * TN; e += 64 * WAVES) {
        const int em = e / TN, en = e % TN;
        if (TM * mt + em < J.m && TN * nt + en < J.n) out[(size_t)(TM * mt + em) * J.n + TN * nt + en] = (P.tile[0][em][en] + P.tile[1][em][en]) + (P.tile[2][em][en] + P.tile[3][em][en]);
    }
    if (nt == 0 && threadIdx.x < TM && TM * mt + (int)threadIdx.x < J.m)
        out[(size_t)J.m * J.n + TM * mt + threadIdx.x] = (P.bias[0][threadIdx.x] + P.bias[1][threadIdx.x]) + (P.bias[2][threadIdx.x] + P.bias[3][threadIdx.x]);
}
__global__ __launch_bounds__(256) void seq_gradient_finish_kernel(JobLaunch K) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= K.elements) return;
    const Job& J = K.job[find_job(K, e, true)];
    float v[SPLITS];
#pragma unroll
    for (int k = 0; k < SPLITS; k++) v[k] = K.partial[(size_t)k * K.elements + e];
#pragma unroll
    for (int s = 1; s < SPLITS; s *= 2)
#pragma unroll
        for (int k = 0; k + s < SPLITS; k += 2 * s) v[k] += v[k + s];
    const int at = e - J.first_element, products = J.m * J.n;
    float* const dst = at < products ? (J.gradient ? J.gradient + at : nullptr) : (J.bias ? J.bias + (at - products) : nullptr);
    if (!dst) return;
    const float value = J.overwrite ? v[0] : *dst + v[0];
    *dst = value;
    if (at >= products && at - products < J.copy_n) J.bias_copy[at - products] = value;
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t forward_lds(int H, int in, int S) { return (H == 32 ? sizeof(ForwardSlots<32>) : sizeof(ForwardSlots<16>)) + 16 + (size_t)S * ((in + 3) & ~3) * sizeof(float) + S + 1; }
size_t backward_lds(int H, int out, int S) { return (H == 32 ? sizeof(BackwardSlots<32>) : sizeof(BackwardSlots<16>)) + 16 + (size_t)S * ((out + 3) & ~3) * sizeof(float) + S; }
}  // namespace

bool rlt_seq_stack_shape(const rlt_seq_layer* L, int n) {
    if (!L || n != 4 || L[0].kind != 0 || L[1].kind != 1 || L[2].kind != 1 || L[3].kind != 0) return false;
    const int H = L[0].dense.out_dim, in = L[0].dense.in_dim, out = L[3].dense.out_dim;
    if ((H != 16 && H != 32) || in < 1 || in > MAX_IN || out < 1 || out > MAX_OUT || L[3].dense.in_dim != H) return false;
    for (int l = 1; l < 3; l++) if (L[l].gru.input_dim != H || L[l].gru.hidden_dim != H) return false;
    return true;
}

bool rlt_seq_stack_supported(const rlt_seq_layer* L, int n, int steps) {
    if (!rlt_seq_stack_shape(L, n) || steps < 1 || L[3].dense.activation != RLT_ACT_IDENTITY) return false;
    const int H = L[0].dense.out_dim, in = L[0].dense.in_dim, out = L[3].dense.out_dim;
    if (L[0].dense.activation < 0 || L[0].dense.activation > RLT_ACT_SIGMOID) return false;
    for (int l = 1; l < 3; l++) {
        const rlt_gru_layer& G = L[l].gru;
        if ((G.fast_tanh != 0) != (L[1].gru.fast_tanh != 0)) return false;
        if (!G.weights_input || !G.biases_input || !G.weights_hidden || !G.biases_hidden || !G.initial_hidden_state || !G.post_activation || !G.n_pre_pre_activation || !G.output) return false;
    }
    for (int l = 0; l < 4; l += 3) { const rlt_dense_layer& D = L[l].dense; if (!D.weights || !D.biases || !D.pre_activations || !D.output) return false; }
    return forward_lds(H, in, steps) <= LDS_LIMIT && backward_lds(H, out, steps) <= LDS_LIMIT;
}

int rlt_seq_stack_forward(rlt_rocm_device* device, const rlt_stack_forward* passes, int n) {
    RLT_REQUIRE(n >= 1 && n <= MAX_PASSES);
    ForwardLaunch K = {};
    K.n = n;
    int blocks = 0; size_t lds = 0;
    for (int k = 0; k < n; k++) {
        const rlt_stack_forward& a = passes[k];
        const rlt_seq_layer* L = a.layers;
        RLT_REQUIRE(a.x && a.steps > 0 && a.batch > 0 && a.ldx >= L[0].dense.in_dim);
        Forward& P = K.pass[k];
        P = {L[0].dense.weights, L[0].dense.biases, L[0].dense.pre_activations, L[0].dense.output, {}, L[3].dense.weights, L[3].dense.biases, L[3].dense.pre_activations, L[3].dense.output, a.also,
             a.x, a.reset, a.ldx, L[0].dense.in_dim, L[3].dense.out_dim, L[0].dense.activation, a.steps, a.batch, L[0].dense.out_dim, L[1].gru.fast_tanh != 0, blocks};
        for (int l = 0; l < 2; l++) {
            const rlt_gru_layer& G = L[1 + l].gru;
            P.g[l] = {G.weights_input, G.biases_input, G.weights_hidden, G.biases_hidden, G.initial_hidden_state, G.post_activation, G.n_pre_pre_activation, G.output};
        }
        blocks += a.batch;
        const size_t need = forward_lds(P.H, P.in, P.S);
        lds = need > lds ? need : lds;
    }
    hipLaunchKernelGGL(seq_stack_forward_kernel, dim3(blocks), dim3(64 * FORWARD_STAGES), lds, device->stream, K);
    return rlt_launch_status(device);
}

size_t rlt_seq_stack_workspace_bytes(const rlt_seq_layer* L, int steps, int batch) {
    const size_t H = L[0].dense.out_dim, rows = (size_t)steps * batch;
    return align256((11 * H * rows + 2 * H * batch) * sizeof(float));      // per recurrence 3H + H + H, the dense layer's gradient H; the b_hn sums
}

int rlt_seq_stack_backward(rlt_rocm_device* device, const rlt_stack_backward* passes, int n) {
    RLT_REQUIRE(n >= 1 && n <= 2);
    BackwardLaunch K = {};
    K.n = n;
    JobLaunch J = {};
    int blocks = 0, job_blocks = 0; size_t lds = 0;
    auto job = [&](const float* a, int lda, int m, const float* b, int ldb, int cols, int rows, float* gradient, float* bias, float* bias_copy, int copy_n, int overwrite) {
        J.job[J.n++] = {a, b, gradient, bias, bias_copy, lda, m, ldb, cols, rows, overwrite, copy_n, job_blocks, J.elements};
        job_blocks += rlt_div_up(m, TM) * (cols ? rlt_div_up(cols, rlt_batch::TN) : 1);
        J.elements += m * cols + m;
    };
    for (int k = 0; k < n; k++) {
        const rlt_stack_backward& a = passes[k];
        const rlt_seq_layer* L = a.layers;
        RLT_REQUIRE(a.d_output && a.steps > 0 && a.batch > 0 && (!a.want_w || (a.x && a.workspace)) && (a.want_w || a.d_input));
        const int H = L[0].dense.out_dim, in = L[0].dense.in_dim, out = L[3].dense.out_dim, rows = a.steps * a.batch;
        Backward& P = K.pass[k];
        float* w = (float*)a.workspace;
        P.W0 = L[0].dense.weights; P.pre0 = L[0].dense.pre_activations; P.W3 = L[3].dense.weights; P.d_output = a.d_output; P.d_input = a.d_input; P.reset = a.reset;
        P.in = in; P.out = out; P.act0 = L[0].dense.activation; P.S = a.steps; P.B = a.batch; P.H = H; P.want_w = a.want_w; P.first_block = blocks;
        for (int l = 0; l < 2; l++) {
            const rlt_gru_layer& G = L[1 + l].gru;
            GruBack& B = P.g[l];
            B = {G.weights_input, G.weights_hidden, G.initial_hidden_state, G.post_activation, G.n_pre_pre_activation, G.output, nullptr, nullptr, nullptr, nullptr};
            if (a.want_w) {
                RLT_REQUIRE(G.d_weights_input && G.d_biases_input && G.d_weights_hidden && G.d_biases_hidden);
                B.g = w; B.gnr = B.g + (size_t)3 * H * rows; B.hp = B.gnr + (size_t)H * rows; w = B.hp + (size_t)H * rows;
                B.db_hn = w; w += (size_t)H * a.batch;
                job(B.g, 3 * H, 3 * H, l ? L[1].gru.output : L[0].dense.output, H, H, rows, G.d_weights_input, G.d_biases_input, G.d_biases_hidden, 2 * H, a.overwrite);
                job(B.g, 3 * H, 2 * H, B.hp, H, H, rows, G.d_weights_hidden, nullptr, nullptr, 0, a.overwrite);
                job(B.gnr, H, H, B.hp, H, H, rows, G.d_weights_hidden + (size_t)2 * H * H, nullptr, nullptr, 0, a.overwrite);
                job(B.db_hn, H, H, nullptr, 0, 0, a.batch, nullptr, G.d_biases_hidden + 2 * H, nullptr, 0, a.overwrite);
            }
        }
        if (a.want_w) {
            RLT_REQUIRE(L[0].dense.d_weights && L[0].dense.d_biases && L[3].dense.d_weights && L[3].dense.d_biases);
            P.d_pre0 = w;
            job(P.d_pre0, H, H, a.x, a.ldx, in, rows, L[0].dense.d_weights, L[0].dense.d_biases, nullptr, 0, a.overwrite);
            job(a.d_output, out, out, L[2].gru.output, H, H, rows, L[3].dense.d_weights, L[3].dense.d_biases, nullptr, 0, a.overwrite);
        }
        blocks += a.batch;
        const size_t need = backward_lds(H, out, a.steps);
        lds = need > lds ? need : lds;
    }
    void* scratch = nullptr;
    int rc;
    if (J.n) {
        if ((rc = rlt_scratch(device, (size_t)SPLITS * J.elements * sizeof(float), &scratch))) return rc;
        J.partial = (float*)scratch;
    }
    hipLaunchKernelGGL(seq_stack_backward_kernel, dim3(blocks), dim3(64 * BACKWARD_STAGES), lds, device->stream, K);
    if ((rc = rlt_launch_status(device)) || !J.n) return rc;
    hipLaunchKernelGGL(seq_gradient_kernel, dim3(job_blocks * SPLITS), dim3(64 * WAVES), 0, device->stream, J);
    if ((rc = rlt_launch_status(device))) return rc;
    hipLaunchKernelGGL(seq_gradient_finish_kernel, dim3(rlt_div_up(J.elements, 256)), dim3(256), 0, device->stream, J);
    return rlt_launch_status(device);
}
