// Passes of the reference's recurrent approximators (rl/algorithms/sac/loop/core/approximators_gru.h:13-74: dense, GRU, GRU, dense) over a batch of sequences, all
// layers in one launch (nn_models/sequential/operations_generic.h:277-428, nn/layers/gru/operations_generic.h:231-341, :594-795).
//
// Batch rows are independent, layers depend on each other only step by step: a workgroup carries ONE batch row, its five wavefronts are the stages of a pipeline, and a
// stage works on the step behind the previous stage's (one workgroup barrier per tick orders LDS only; the slots between two stages are double-buffered by the step's
// parity). Forward: dense layer and first input projection | first recurrence | second input projection | second recurrence | output layer; backward, from the last
// step on: output layer and second recurrence | its input gradient | first recurrence | its input gradient and the dense layer's | the input's gradient.
// Within a stage lane (u, p) owns hidden unit u and a share p of the reduction index (half of it at width 32, a quarter at 16), with its 3 H / (64 / H) weights in
// registers; the vector of the step arrives through LDS (16-byte broadcast reads) and the shares are added with v_permlane32_swap / v_permlane16_swap.
// Weight gradients are contractions over all steps and rows, done afterwards for all layers by one launch on the matrix cores (and a second that adds the shares of the
// rows up).
// Bound: the chain of dependent steps, TODO us per step at width 32 (a launch per layer and direction with a row per 32 lanes took 0.58 us per step, one layer
// after the other, plus a launch per dense layer, projection and gradient: TODO). Workgroups of up to three models share a launch.
#include "seq_stack.h"
#include "gemm.h"
#include "batch_tile.h"

namespace {
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
constexpr int MAX_IN = 16, MAX_OUT = 16, STAGES = 5, THREADS = 64 * STAGES, MAX_PASSES = 3;
constexpr size_t LDS_LIMIT = 48 * 1024;      // three to four workgroups per compute unit

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// the sum of x over the lanes of one unit (lanes 64 / PARTS apart); every one of them receives it
template <int PARTS>
__device__ __forceinline__ float sum_parts(float x) {
    if (PARTS == 4) { const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false); x = __uint_as_float(s[0]) + __uint_as_float(s[1]); }
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
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

// rows u, H + u, 2H + u of a [3H x H] matrix (or, transposed, its columns u of the three blocks), this lane's share of the reduction index
template <int H>
struct Weights3 { float w[3][H * H / 64]; };
template <int H>
__device__ __forceinline__ void load_rows3(const float* W, int u, int p, Weights3<H>& R) {
    constexpr int KP = H * H / 64;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int q = 0; q < KP; q += 4) {
            floatx4 v;
            __builtin_memcpy(&v, W + (size_t)(k * H + u) * H + p * KP + q, sizeof v);      // 16 bytes at a time, whatever the tensor's alignment
            R.w[k][q] = v[0]; R.w[k][q + 1] = v[1]; R.w[k][q + 2] = v[2]; R.w[k][q + 3] = v[3];
        }
}
template <int H>
__device__ __forceinline__ void load_columns3(const float* W, int u, int p, Weights3<H>& R) {
    constexpr int KP = H * H / 64;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int q = 0; q < KP; q++) R.w[k][q] = W[(size_t)(k * H + p * KP + q) * H + u];
}
// the three products of a vector v (LDS, H values) with rows u of the three blocks
template <int H>
__device__ __forceinline__ void products3(const Weights3<H>& R, const float* v, int p, float (&out)[3]) {
    constexpr int KP = H * H / 64, PARTS = 64 / H;
    float acc[3] = {0.f, 0.f, 0.f};
    floatx4 x[KP / 4];
#pragma unroll
    for (int q = 0; q < KP / 4; q++) x[q] = reinterpret_cast<const floatx4*>(v + p * KP)[q];
#pragma unroll
    for (int q = 0; q < KP; q++)
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k] += x[q / 4][q % 4] * R.w[k][q];
#pragma unroll
    for (int k = 0; k < 3; k++) out[k] = sum_parts<PARTS>(acc[k]);
}
// the sum over three vectors (LDS, 3 x H values) of their products with columns u of the three blocks
template <int H>
__device__ __forceinline__ float product_sum3(const Weights3<H>& R, const float* v, int p) {
    constexpr int KP = H * H / 64, PARTS = 64 / H;
    float acc[3] = {0.f, 0.f, 0.f};
    floatx4 x[3][KP / 4];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int q = 0; q < KP / 4; q++) x[k][q] = reinterpret_cast<const floatx4*>(v + k * H + p * KP)[q];
#pragma unroll
    for (int q = 0; q < KP; q++)
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k] += x[k][q / 4][q % 4] * R.w[k][q];
    return sum_parts<PARTS>(acc[0] + (acc[1] + acc[2]));
}

struct Gru { const float *W_i, *b_i, *W_h, *b_h, *h0; float *post, *npp, *out; };
struct Forward {
    const float *W0, *b0; float *pre0, *out0; Gru g[2]; const float *W3, *b3; float *pre3, *out3, *also;
    const float* x; const uint8_t* reset; int ldx, in, out, act0, S, B, H, fast, first_block;
};
struct ForwardLaunch { Forward pass[MAX_PASSES]; int n; };

// LDS of a workgroup: the row's inputs (rows of four floats' multiples) and reset flags, then the slots between the stages
template <int H> struct ForwardSlots { float dense[H], own[2][H], p1[2][3 * H], h1[2][H], p2[2][3 * H], h2[2][H]; };

template <int H, bool FAST>
__device__ __forceinline__ void recurrence(const Forward& P, int layer, int lag, const float (*in)[3 * H], float* own, float (*out)[H], const uint8_t* flags, int b, int lane) {
    constexpr int PARTS = 64 / H;
    const Gru& G = P.g[layer];
    const int u = lane & (H - 1), p = lane / H, S = P.S;
    Weights3<H> R;
    load_rows3<H>(G.W_h, u, p, R);
    const float br = G.b_h[u], bz = G.b_h[H + u], bn = G.b_h[2 * H + u], h0 = G.h0[u];
    float h = h0;
    if (p == 0) own[u] = h0;
    for (int tick = 0; tick < S + STAGES - 1; tick++) {
        const int t = tick - lag;
        if (t >= 0 && t < S) {
            const float* x = in[t & 1];
            const float xr = x[u], xz = x[H + u], xn = x[2 * H + u];
            float a[3];
            products3<H>(R, own, p, a);
            const float an = bn + a[2];
            const float r = gate_sigmoid<FAST>(xr + (br + a[0])), z = gate_sigmoid<FAST>(xz + (bz + a[1]));
            const float n = gate_tanh<FAST>(xn + an * r);
            h = (1.0f - z) * n + z * h;
            const size_t at = (size_t)t * P.B + b;
            // what a restart at the next step takes in place of this step's state
            const bool restart = t + 1 < S && flags[t + 1];
            const float out_h = h;
            if (restart) h = h0;
            wave_sync();
            if (p == 0) { out[t & 1][u] = out_h; own[u] = h; }
            wave_sync();
            float* const post = G.post + at * 3 * H;
            if (p < 2) { post[p * H + u] = p ? z : r; (p ? G.npp + at * H : post + 2 * H)[u] = p ? an : n; }
            if (p == PARTS - 1) G.out[at * H + u] = out_h;
        }
        rlt_lds_barrier();
    }
}
template <int H>
__device__ __forceinline__ void projection(const Gru& G, int S, int lag, const float (*in)[H], float (*out)[3 * H], int lane) {
    const int u = lane & (H - 1), p = lane / H;
    Weights3<H> R;
    load_rows3<H>(G.W_i, u, p, R);
    const float br = G.b_i[u], bz = G.b_i[H + u], bn = G.b_i[2 * H + u];
    for (int tick = 0; tick < S + STAGES - 1; tick++) {
        const int t = tick - lag;
        if (t >= 0 && t < S) {
            float a[3];
            products3<H>(R, in[t & 1], p, a);
            if (p == 0) { float* o = out[t & 1]; o[u] = br + a[0]; o[H + u] = bz + a[1]; o[2 * H + u] = bn + a[2]; }
        }
        rlt_lds_barrier();
    }
}
template <int H, bool FAST>
__device__ __forceinline__ void forward_row(const Forward& P, int b, char* lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), p = lane / H, S = P.S, in4 = (P.in + 3) & ~3;
    ForwardSlots<H>& L = *reinterpret_cast<ForwardSlots<H>*>(lds);
    float* const xs = reinterpret_cast<float*>(lds + ((sizeof(ForwardSlots<H>) + 15) & ~(size_t)15));
    uint8_t* const flags = reinterpret_cast<uint8_t*>(xs + (size_t)S * in4);
    for (int i = threadIdx.x; i < S * in4; i += THREADS) { const int t = i / in4, k = i - t * in4; xs[i] = k < P.in ? P.x[((size_t)t * P.B + b) * P.ldx + k] : 0.f; }
    for (int t = threadIdx.x; t < S; t += THREADS) flags[t] = t == 0 || (P.reset && P.reset[(size_t)t * P.B + b]);
    rlt_lds_barrier();
    if (wave == 0) {
        // the dense layer and the first recurrence's input projection
        float w0[MAX_IN];
#pragma unroll
        for (int k = 0; k < MAX_IN; k++) w0[k] = k < P.in ? P.W0[(size_t)u * P.in + k] : 0.f;
        const float b0 = P.b0[u];
        Weights3<H> R;
        load_rows3<H>(P.g[0].W_i, u, p, R);
        const float br = P.g[0].b_i[u], bz = P.g[0].b_i[H + u], bn = P.g[0].b_i[2 * H + u];
        for (int t = 0; t < S + STAGES - 1; t++) {
            if (t < S) {
                float acc = b0;
                const floatx4* x = reinterpret_cast<const floatx4*>(xs + (size_t)t * in4);
#pragma unroll
                for (int q = 0; q < MAX_IN / 4; q++)
                    if (4 * q < P.in) { const floatx4 v = x[q]; acc += v[0] * w0[4 * q]; acc += v[1] * w0[4 * q + 1]; acc += v[2] * w0[4 * q + 2]; acc += v[3] * w0[4 * q + 3]; }
                const float o = rlt_act(acc, P.act0);
                if (p < 2) (p ? P.out0 : P.pre0)[((size_t)t * P.B + b) * H + u] = p ? o : acc;
                if (p == 0) L.dense[u] = o;
                wave_sync();
                float a[3];
                products3<H>(R, L.dense, p, a);
                wave_sync();
                if (p == 0) { float* d = L.p1[t & 1]; d[u] = br + a[0]; d[H + u] = bz + a[1]; d[2 * H + u] = bn + a[2]; }
            }
            rlt_lds_barrier();
        }
    }
    else if (wave == 1) recurrence<H, FAST>(P, 0, 1, L.p1, L.own[0], L.h1, flags, b, lane);
    else if (wave == 2) projection<H>(P.g[1], S, 2, L.h1, L.p2, lane);
    else if (wave == 3) recurrence<H, FAST>(P, 1, 3, L.p2, L.own[1], L.h2, flags, b, lane);
    else {
        // the output layer: lane = output, all of the reduction
        float w3[H];
        const int o = min(lane, P.out - 1);
#pragma unroll
        for (int k = 0; k < H; k++) w3[k] = P.W3[(size_t)o * H + k];
        const float b3 = P.b3[o];
        for (int tick = 0; tick < S + STAGES - 1; tick++) {
            const int t = tick - 4;
            if (t >= 0) {
                const floatx4* h = reinterpret_cast<const floatx4*>(L.h2[t & 1]);
                float a0 = b3, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
                for (int q = 0; q < H / 4; q++) { const floatx4 v = h[q]; a0 += v[0] * w3[4 * q]; a1 += v[1] * w3[4 * q + 1]; a2 += v[2] * w3[4 * q + 2]; a3 += v[3] * w3[4 * q + 3]; }
                const float y = (a0 + a1) + (a2 + a3);
                const size_t at = ((size_t)t * P.B + b) * P.out + lane;
                if (lane < P.out) { P.pre3[at] = y; P.out3[at] = y; if (P.also) P.also[at] = y; }
            }
            rlt_lds_barrier();
        }
    }
}
__global__ __launch_bounds__(THREADS) void seq_stack_forward_kernel(ForwardLaunch K) {
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
template <int H> struct BackwardSlots { float own[2][3 * H], g2[2][3 * H], dy1[2][H], g1[2][3 * H], dp0[2][H]; };

template <int H, bool TOP>
__device__ __forceinline__ void recurrence_back(const Backward& P, int layer, int lag, const float* d_out, const float (*dy)[H], float* own, float (*g)[3 * H], const uint8_t* flags, int b, int lane) {
    constexpr int PARTS = 64 / H, DEPTH = 4;
    const GruBack& G = P.g[layer];
    const int u = lane & (H - 1), p = lane / H, S = P.S;
    Weights3<H> R;
    load_columns3<H>(G.W_h, u, p, R);
    const float h0 = G.h0[u];
    float w3[TOP ? MAX_OUT : 1];
    if (TOP) {
#pragma unroll
        for (int o = 0; o < MAX_OUT; o++) w3[o] = o < P.out ? P.W3[(size_t)o * H + u] : 0.f;
    }
    // a step's saved values, requested DEPTH steps ahead (a load takes longer than a step); the lanes of a unit load different ones and exchange them
    struct Saved { float rz, nn, hp; };
    auto request = [&](int t) {
        const size_t at = (size_t)(t > 0 ? t : 0) * P.B + b, before = (size_t)(t > 1 ? t - 1 : 0) * P.B + b;
        Saved v;
        v.rz = G.post[at * 3 * H + (p & 1) * H + u]; v.nn = ((p & 1) ? G.npp + at * H : G.post + at * 3 * H + 2 * H)[u]; v.hp = G.out[before * H + u];
        return v;
    };
    Saved queue[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; d++) queue[d] = request(S - 1 - d);
    float carry = 0.f, db_hn = 0.f;
    for (int tick = 0; tick < S + STAGES - 1; tick++) {
        const int t = S - 1 - (tick - lag);
        if (t >= 0 && t < S) {
            const Saved cur = queue[0];
#pragma unroll
            for (int d = 0; d + 1 < DEPTH; d++) queue[d] = queue[d + 1];
            queue[DEPTH - 1] = request(t - DEPTH);
            float r, z, n, npp;
            if (PARTS == 2) {
                const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(cur.rz), __float_as_uint(cur.rz), false, false), c = __builtin_amdgcn_permlane32_swap(__float_as_uint(cur.nn), __float_as_uint(cur.nn), false, false);
                r = __uint_as_float(a[0]); z = __uint_as_float(a[1]); n = __uint_as_float(c[0]); npp = __uint_as_float(c[1]);
            } else {
                const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(cur.rz), __float_as_uint(cur.rz), false, false), c = __builtin_amdgcn_permlane16_swap(__float_as_uint(cur.nn), __float_as_uint(cur.nn), false, false);
                r = __uint_as_float(a[0]); z = __uint_as_float(a[1]); n = __uint_as_float(c[0]); npp = __uint_as_float(c[1]);
            }
            float dh = carry;
            if (TOP) {
                const float* d = d_out + (size_t)t * P.out;
                float s = 0.f;
#pragma unroll
                for (int o = 0; o < MAX_OUT; o++) if (o < P.out) s += d[o] * w3[o];
                dh += s;
            } else dh += dy[t & 1][u];
            const bool from_initial = flags[t];
            const float hp = from_initial ? h0 : cur.hp;
            const float gz = dh * (hp - n) * z * (1.0f - z);
            const float gn = dh * (1.0f - z) * (1.0f - n * n);
            const float gr = gn * npp * r * (1.0f - r);
            const float gnr = gn * r;
            if (p == 0) { own[u] = gr; own[H + u] = gz; own[2 * H + u] = gnr; float* s = g[t & 1]; s[u] = gr; s[H + u] = gz; s[2 * H + u] = gn; }
            wave_sync();
            const float sum = product_sum3<H>(R, own, p);
            wave_sync();
            carry = from_initial ? 0.f : dh * z + sum;
            if (P.want_w) {
                const size_t at = (size_t)t * P.B + b;
                if (p < 2) { G.g[at * 3 * H + p * H + u] = p ? gz : gr; (p ? G.gnr + at * H : G.g + at * 3 * H + 2 * H)[u] = p ? gnr : gn; }
                if (p == PARTS - 1) G.hp[at * H + u] = hp;
                // the reference drops reset samples (t > 0) from the b_hn gradient (their buffer rows are zeroed before that sum, gru/operations_generic.h:716-749)
                if (!(t > 0 && from_initial)) db_hn += gnr;
            }
        }
        rlt_lds_barrier();
    }
    if (P.want_w && p == 0) G.db_hn[(size_t)b * H + u] = db_hn;
}
template <int H>
__device__ __forceinline__ void backward_row(const Backward& P, int b, char* lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = lane & (H - 1), p = lane / H, S = P.S;
    BackwardSlots<H>& L = *reinterpret_cast<BackwardSlots<H>*>(lds);
    float* const ds = reinterpret_cast<float*>(lds + ((sizeof(BackwardSlots<H>) + 15) & ~(size_t)15));
    uint8_t* const flags = reinterpret_cast<uint8_t*>(ds + (size_t)S * P.out);
    for (int i = threadIdx.x; i < S * P.out; i += THREADS) { const int t = i / P.out; ds[i] = P.d_output[((size_t)t * P.B + b) * P.out + (i - t * P.out)]; }
    for (int t = threadIdx.x; t < S; t += THREADS) flags[t] = t == 0 || (P.reset && P.reset[(size_t)t * P.B + b]);
    rlt_lds_barrier();
    if (wave == 0) recurrence_back<H, true>(P, 1, 0, ds, nullptr, L.own[1], L.g2, flags, b, lane);
    else if (wave == 1) {
        Weights3<H> R;
        load_columns3<H>(P.g[1].W_i, u, p, R);
        for (int tick = 0; tick < S + STAGES - 1; tick++) {
            const int t = S - 1 - (tick - 1);
            if (t >= 0 && t < S) { const float d = product_sum3<H>(R, L.g2[t & 1], p); if (p == 0) L.dy1[t & 1][u] = d; }
            rlt_lds_barrier();
        }
    }
    else if (wave == 2) recurrence_back<H, false>(P, 0, 2, nullptr, L.dy1, L.own[0], L.g1, flags, b, lane);
    else if (wave == 3) {
        Weights3<H> R;
        load_columns3<H>(P.g[0].W_i, u, p, R);
        constexpr int DEPTH = 4;
        float queue[DEPTH];
        auto request = [&](int t) { return P.pre0[((size_t)(t > 0 ? t : 0) * P.B + b) * H + u]; };
#pragma unroll
        for (int d = 0; d < DEPTH; d++) queue[d] = request(S - 1 - d);
        for (int tick = 0; tick < S + STAGES - 1; tick++) {
            const int t = S - 1 - (tick - 3);
            if (t >= 0 && t < S) {
                const float pre = queue[0];
#pragma unroll
                for (int d = 0; d + 1 < DEPTH; d++) queue[d] = queue[d + 1];
                queue[DEPTH - 1] = request(t - DEPTH);
                const float d = product_sum3<H>(R, L.g1[t & 1], p) * rlt_dact(pre, P.act0);
                if (p == 0) L.dp0[t & 1][u] = d;
                if (p == 0 && P.want_w) P.d_pre0[((size_t)t * P.B + b) * H + u] = d;
            }
            rlt_lds_barrier();
        }
    } else {
        float w0[H];
        const int k = min(lane, P.in - 1);
        if (P.d_input) {
#pragma unroll
            for (int j = 0; j < H; j++) w0[j] = P.W0[(size_t)j * P.in + k];
        }
        for (int tick = 0; tick < S + STAGES - 1; tick++) {
            const int t = S - 1 - (tick - 4);
            if (P.d_input && t >= 0 && t < S) {
                const floatx4* d = reinterpret_cast<const floatx4*>(L.dp0[t & 1]);
                float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
                for (int q = 0; q < H / 4; q++) { const floatx4 v = d[q]; a0 += v[0] * w0[4 * q]; a1 += v[1] * w0[4 * q + 1]; a2 += v[2] * w0[4 * q + 2]; a3 += v[3] * w0[4 * q + 3]; }
                if (lane < P.in) P.d_input[((size_t)t * P.B + b) * P.in + lane] = (a0 + a1) + (a2 + a3);
            }
            rlt_lds_barrier();
        }
    }
}
__global__ __launch_bounds__(THREADS) void seq_stack_backward_kernel(BackwardLaunch K) {
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
size_t forward_lds(int H, int in, int S) { return (H == 32 ? sizeof(ForwardSlots<32>) : sizeof(ForwardSlots<16>)) + 16 + (size_t)S * ((in + 3) & ~3) * sizeof(float) + S; }
size_t backward_lds(int H, int out, int S) { return (H == 32 ? sizeof(BackwardSlots<32>) : sizeof(BackwardSlots<16>)) + 16 + (size_t)S * out * sizeof(float) + S; }
}  // namespace

bool rlt_seq_stack_supported(const rlt_seq_layer* L, int n, int steps) {
    if (!L || n != 4 || steps < 1 || L[0].kind != 0 || L[1].kind != 1 || L[2].kind != 1 || L[3].kind != 0) return false;
    const int H = L[0].dense.out_dim, in = L[0].dense.in_dim, out = L[3].dense.out_dim;
    if ((H != 16 && H != 32) || in < 1 || in > MAX_IN || out < 1 || out > MAX_OUT || L[3].dense.in_dim != H || L[3].dense.activation != RLT_ACT_IDENTITY) return false;
    if (L[0].dense.activation < 0 || L[0].dense.activation > RLT_ACT_SIGMOID) return false;
    for (int l = 1; l < 3; l++) {
        const rlt_gru_layer& G = L[l].gru;
        if (G.input_dim != H || G.hidden_dim != H || (G.fast_tanh != 0) != (L[1].gru.fast_tanh != 0)) return false;
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
    hipLaunchKernelGGL(seq_stack_forward_kernel, dim3(blocks), dim3(THREADS), lds, device->stream, K);
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
    hipLaunchKernelGGL(seq_stack_backward_kernel, dim3(blocks), dim3(THREADS), lds, device->stream, K);
    if ((rc = rlt_launch_status(device)) || !J.n) return rc;
    hipLaunchKernelGGL(seq_gradient_kernel, dim3(job_blocks * SPLITS), dim3(64 * WAVES), 0, device->stream, J);
    if ((rc = rlt_launch_status(device))) return rc;
    hipLaunchKernelGGL(seq_gradient_finish_kernel, dim3(rlt_div_up(J.elements, 256)), dim3(256), 0, device->stream, J);
    return rlt_launch_status(device);
}
