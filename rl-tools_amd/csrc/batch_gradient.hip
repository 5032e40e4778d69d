// Weight gradients d_pre^T x of three-layer networks over a whole batch, each element complete in one workgroup, with Adam's step in the same launch
// (nn/layers/dense/operations_generic.h:227-260, nn/optimizers/adam/instance/operations_generic.h:26-72).
//
// The kernels that run a batch's passes on sixteen-row tiles (sac_wide.hip) leave activations and pre-activation gradients in memory (4 KB per row at width 256);
// here a workgroup takes a tile of 16 x 32 elements of a weight gradient and its four wavefronts a quarter of the rows each, on v_mfma_f32_16x16x4_f32, operands
// straight from L2. The alternative, a block of partial sums per sixteen rows (281 KB at 17-256-256-6) that a later launch adds up, moves sixteen times the bytes of the
// gradients themselves at batch 256 and 250 times at batch 4,000.
// Up to 512 rows a workgroup sees the whole batch and finishes its elements. Beyond that the batch is shared out to two, four or eight groups of workgroups that lie on
// different XCDs: the rows of a large batch (16 MB at 4,001 rows) do not fit an XCD's 4 MB of L2, and with every XCD reading all of them the launch took 32.6 us at
// 4,001 rows; with an eighth of the rows per XCD 15.5 us, and a second launch adds the eight sums up (4 us).
// Bound: latency up to a few hundred rows (the trip to memory for the first operands, 16 steps of the matrix pipe, the exchange between the wavefronts, the stores),
// then the loads of the operands from L2: each row of a network is read by its 8 to 16 column tiles.
#include "batch_gradient.h"
#include "optim.h"
#include "batch_tile.h"

namespace {
using namespace rlt_batch;
constexpr int WAVES = 4, THREADS = 64 * WAVES, SPLIT_ROWS = 512, MAX_SPLITS = 8;
struct GradientLaunch {
    rlt_gradient_net net[2]; int blocks0, batch, splits, total0, total; float polyak;      // total0, total: gradient elements of the first network, of both
    rlt_gradient_scalar scalar; int has_scalar;
    rlt_gradient_guard guard;      // of networks that step
    float* partial;      // splits > 1: [splits][total] sums, the networks' elements one after the other, segments in order
};

__host__ __device__ inline int segment_size(const rlt_gradient_net& N, int k) { return k == 0 ? N.hid * N.in : k == 2 ? N.hid * N.hid : k == 4 ? N.out * N.hid : k == 5 ? N.out : N.hid; }

// an element whose gradient is complete: added onto the caller's gradient, or stored and stepped from the optimiser's values
struct Held { float first, second, value, target; };
__device__ __forceinline__ Held hold(const rlt_gradient_net& N, int segment, size_t at) {
    Held h = {0.f, 0.f, 0.f, 0.f};
    if (N.step) {
        h.first = N.first_moment[segment][at]; h.second = N.second_moment[segment][at]; h.value = N.parameter[segment][at];
        if (N.target[segment]) h.target = N.target[segment][at];
    }
    return h;
}
__device__ __forceinline__ void finish(const rlt_gradient_net& N, int segment, size_t at, float sum, Held h, float bc1, float bc2, float polyak, bool is_void) {
    float* const gradient = N.gradient[segment] + at;
    if (!N.step) { *gradient += sum; return; }
    *gradient = sum;
    if (is_void) return;
    rlt_adam_values(N.adam, N.flags[segment], sum, bc1, bc2, h.first, h.second, h.value);
    N.first_moment[segment][at] = h.first; N.second_moment[segment][at] = h.second; N.parameter[segment][at] = h.value;
    if (N.target[segment]) N.target[segment][at] = rlt_polyak_value(polyak, h.target, h.value);
}
// log_alpha's step, by one wavefront
__device__ __forceinline__ void finish_scalar(const rlt_gradient_scalar& Z, int lane, bool is_void) {
    float s = (lane < Z.n ? Z.values[lane] : 0.f) + (64 + lane < Z.n ? Z.values[64 + lane] : 0.f);
    s = rlt_wave_sum(s);
    if (lane == 0) {
        *Z.tensor.gradient = s * Z.scale;
        if (is_void) return;
        float bc1, bc2;
        rlt_adam_bias_corrections(Z.adam, *Z.age, bc1, bc2);
        rlt_adam_apply(Z.adam, Z.tensor, 0, s * Z.scale, bc1, bc2, 0.0f);
    }
}

// What a step's launch waits for before anything else: the age's bias corrections and the word of a launch that gave up, on their way together (one after the other they cost SAC's update set
// 0.1 to 0.3 us of 86)
__device__ __forceinline__ void step_scalars(const rlt_gradient_net& N, const rlt_gradient_guard& G, float& bc1, float& bc2, bool& is_void) {
    const unsigned fault = *G.fault, age = *N.age;
    rlt_adam_bias_corrections(N.adam, age, bc1, bc2);
    is_void = fault != 0;
}
__device__ __forceinline__ void give_ages_back(const rlt_gradient_guard& G) {      // by one thread of the launch (which reads the ages from `before`)
#pragma unroll
    for (int k = 0; k < 3; k++) if (G.age[k]) *G.age[k] = G.before[k];
}

// TM: rows of the tile. 16 where a workgroup sees the whole batch (few rows: as many workgroups as the gradients give); 32 where the batch is shared out, which gives
// eight times the workgroups (four loads for four matrix instructions instead of three for two)
template <bool SPLIT>
__global__ __launch_bounds__(THREADS) void batch_gradient_kernel(GradientLaunch K) {
    constexpr int TM = SPLIT ? 32 : 16, PER_THREAD = TM * TN / THREADS;
    __shared__ Parts<WAVES, TM / 16> P;
    const int split = SPLIT ? blockIdx.x % K.splits : 0, block = SPLIT ? blockIdx.x / K.splits : blockIdx.x;      // splits divide 8: a split's workgroups lie on 8 / splits XCDs
    const int y = block >= K.blocks0 ? 1 : 0;
    const rlt_gradient_net& N = y ? K.net[1] : K.net[0];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), B = K.batch;
    // which tile of which layer's gradient: layer 2 first (the most tiles), then 1, then 3
    const int MT = (N.hid + TM - 1) / TM, N2 = (N.hid + TN - 1) / TN, N1 = (N.in + TN - 1) / TN;
    int t = block - (y ? K.blocks0 : 0), segment, tiles, rows, cols, lda, ldb, before = 0;      // before: elements of the segments in front of this one
    const float *a, *b;
    if (t < MT * N2) { segment = 2; before = N.hid * N.in + N.hid; tiles = N2; a = N.d2; lda = N.hid; rows = N.hid; b = N.h1; ldb = N.hid; cols = N.hid; }
    else if ((t -= MT * N2) < MT * N1) { segment = 0; tiles = N1; a = N.d1; lda = N.hid; rows = N.hid; b = N.x; ldb = N.ldx; cols = N.in; }
    else { t -= MT * N1; segment = 4; before = N.hid * N.in + N.hid + N.hid * N.hid + N.hid; tiles = N2; a = N.d3; lda = N.ld3; rows = N.out; b = N.h2; ldb = N.hid; cols = N.hid; }
    const int mt = t / tiles, nt = t - mt * tiles;
    // this wavefront's rows of the batch
    const int shares = SPLIT ? WAVES * K.splits : WAVES, per = ((B + shares - 1) / shares + 3) & ~3, k0 = (WAVES * split + wave) * per, k1 = min(B, k0 + per);
    // what the step needs of this thread's elements travels before the operands
    Held held[PER_THREAD];
    float bc1 = 0.f, bc2 = 0.f;
    bool is_void = false;
    if (!SPLIT) {
#pragma unroll
        for (int u = 0; u < PER_THREAD; u++) {
            const int e = threadIdx.x + u * THREADS, em = TM * mt + e / TN, en = TN * nt + e % TN;
            held[u] = hold(N, segment, em < rows && en < cols ? (size_t)em * cols + en : 0);
        }
        if (N.step) step_scalars(N, K.guard, bc1, bc2, is_void);
    }
    floatx4 c[TM / 16][2];
    float bias[TM / 16];
    tile_product<TM / 16>(a, lda, rows, TM * mt, b, ldb, cols, TN * nt, B, k0, k1, r, g, c, bias);
    place_parts(P, wave, r, g, c, bias);
    rlt_lds_barrier();
    const size_t first = SPLIT ? (size_t)split * K.total + (y ? K.total0 : 0) + before : 0;      // where this segment's sums of this split lie
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
        const int e = threadIdx.x + u * THREADS, em = e / TN, en = e % TN;
        if (TM * mt + em < rows && TN * nt + en < cols) {
            const float sum = (P.tile[0][em][en] + P.tile[1][em][en]) + (P.tile[2][em][en] + P.tile[3][em][en]);
            const size_t at = (size_t)(TM * mt + em) * cols + TN * nt + en;
            if (SPLIT) K.partial[first + at] = sum;
            else finish(N, segment, at, sum, held[u], bc1, bc2, K.polyak, is_void);
        }
    }
    // the layer's bias gradient: column sums of the left operand, by the workgroups of the first column tile
    if (nt == 0 && threadIdx.x < TM && TM * mt + (int)threadIdx.x < rows) {
        const int at = TM * mt + threadIdx.x;
        const float sum = (P.bias[0][threadIdx.x] + P.bias[1][threadIdx.x]) + (P.bias[2][threadIdx.x] + P.bias[3][threadIdx.x]);
        if (SPLIT) K.partial[first + (size_t)rows * cols + at] = sum;
        else finish(N, segment + 1, at, sum, hold(N, segment + 1, at), bc1, bc2, K.polyak, is_void);
    }
    if (!SPLIT && K.has_scalar && blockIdx.x == gridDim.x - 1 && wave == 0) finish_scalar(K.scalar, lane, is_void);
    if (!SPLIT && is_void && blockIdx.x == 0 && threadIdx.x == 0) give_ages_back(K.guard);
}

// the splits' sums added up, in order, and the elements finished
__global__ __launch_bounds__(256) void finish_kernel(GradientLaunch K) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    unsigned fault = 0;
    if (K.net[0].step) fault = *K.guard.fault;      // (both networks step or neither does)
    if (e < K.total) {
        const int y = e >= K.total0 ? 1 : 0;
        const rlt_gradient_net& N = y ? K.net[1] : K.net[0];
        int at = e - (y ? K.total0 : 0), segment = 0;
#pragma unroll
        for (int k = 0; k < 5; k++) if (segment == k && at >= segment_size(N, k)) { at -= segment_size(N, k); segment = k + 1; }
        float v[MAX_SPLITS];
#pragma unroll
        for (int k = 0; k < MAX_SPLITS; k++) v[k] = k < K.splits ? K.partial[(size_t)k * K.total + e] : 0.f;
        const Held h = hold(N, segment, at);
        float bc1 = 0.f, bc2 = 0.f;
        if (N.step) rlt_adam_bias_corrections(N.adam, *N.age, bc1, bc2);
        const float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        finish(N, segment, at, sum, h, bc1, bc2, K.polyak, fault != 0);
    }
    if (K.has_scalar && blockIdx.x == gridDim.x - 1 && threadIdx.x < 64) finish_scalar(K.scalar, threadIdx.x, fault != 0);
    if (fault != 0 && blockIdx.x == 0 && threadIdx.x == 0) give_ages_back(K.guard);
}

int blocks_of(const rlt_gradient_net& N, int TM) {
    const int MT = rlt_div_up(N.hid, TM), N2 = rlt_div_up(N.hid, TN);
    return MT * N2 + MT * rlt_div_up(N.in, TN) + rlt_div_up(N.out, TM) * N2;
}
int elements_of(const rlt_gradient_net& N) { int n = 0; for (int k = 0; k < 6; k++) n += segment_size(N, k); return n; }
// Groups of workgroups that the batch is shared out to: one per SPLIT_ROWS rows; and where there are several, and a launch behind this one adds their sums up anyway, as many
// as give every compute unit a workgroup (a narrow network's gradients are few tiles: 15 at width 65)
int splits_for(const rlt_gradient_net* nets, int n_nets, int batch) {
    int s = 1, tiles = 0;
    for (int k = 0; k < n_nets; k++) tiles += blocks_of(nets[k], 32);
    while (s < MAX_SPLITS && batch > s * SPLIT_ROWS) s *= 2;
    while (s > 1 && s < MAX_SPLITS && tiles * s < 256) s *= 2;
    return s;
}
}  // namespace

size_t rlt_batch_gradients_partial_floats(const rlt_gradient_net* nets, int n_nets, int batch) {
    const int splits = splits_for(nets, n_nets, batch);
    if (splits == 1) return 0;
    size_t n = 0;
    for (int k = 0; k < n_nets; k++) n += elements_of(nets[k]);
    return n * splits;
}

int rlt_batch_gradients(rlt_rocm_device* device, const rlt_gradient_net* nets, int n_nets, int batch, float polyak, const rlt_gradient_scalar* scalar, float* partial,
                        const rlt_gradient_guard* guard) {
    RLT_REQUIRE(nets && n_nets >= 1 && n_nets <= 2 && batch > 0 && (!scalar || scalar->n <= 128) && (n_nets == 1 || nets[0].step == nets[1].step) && (!nets[0].step || (guard && guard->fault)));
    GradientLaunch K = {};
    K.splits = splits_for(nets, n_nets, batch);
    int blocks = 0;
    for (int k = 0; k < n_nets; k++) {
        K.net[k] = nets[k]; blocks += blocks_of(nets[k], K.splits > 1 ? 32 : 16); K.total += elements_of(nets[k]);
        if (k == 0) { K.blocks0 = blocks; K.total0 = K.total; }
    }
    K.batch = batch; K.polyak = polyak; K.partial = partial;
    if (scalar) { K.scalar = *scalar; K.has_scalar = 1; }
    if (guard) K.guard = *guard;
    if (K.splits == 1) {
        hipLaunchKernelGGL((batch_gradient_kernel<false>), dim3(blocks), dim3(THREADS), 0, device->stream, K);
        return rlt_launch_status(device);
    }
    RLT_REQUIRE(partial);
    hipLaunchKernelGGL((batch_gradient_kernel<true>), dim3(blocks * K.splits), dim3(THREADS), 0, device->stream, K);
    const int rc = rlt_launch_status(device);
    if (rc) return rc;
    hipLaunchKernelGGL(finish_kernel, dim3(rlt_div_up(K.total, 256)), dim3(256), 0, device->stream, K);
    return rlt_launch_status(device);
}
