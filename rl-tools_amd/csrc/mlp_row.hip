// The forward pass of a three-layer network over a batch of up to a few thousand rows, a row or a few per workgroup
// (reference: nn_models/mlp/operations_generic.h:77-130 evaluate / forward; acting calls it with one row).
//
// What bounds it: a chain of three dependent layers behind one trip to memory for 72 k weights (256 wide). Sixteen-row tiles on the matrix cores (mlp_wide_kernel)
// spend 8,192 cycles of a compute unit's matrix pipeline per 256 x 256 layer, whatever the rows that are there, and want the weights copied into consumption order
// by a launch of their own. Here a workgroup of sixteen wavefronts takes R rows on the vector units: 16,384 of the 65,536 products of a layer and row per SIMD, 1,024 cycles, from
// W as it lies, and as many workgroups run as there are R-row groups. Wavefront w owns units 16 w ... 16 w + 15; lane (g, c) = (lane / 16, lane % 16) holds
// positions 4 c + 64 j ... + 3 of the rows of units 16 w + 4 q + g, so a load instruction reads four runs of 256 bytes; all of a wavefront's weights of all
// layers are requested before the first layer starts, the sixteen lanes' sums meet in row operations, and only the activations go through LDS.
// One row of 17-256-256-6: 13.0 -> 5.2 us per call (10.6 us of sixteen-row tile and 3.1 of copies before; 4 us is what a call that launches anything costs);
// 256 rows: 14.9 -> 5.7 us; 1,024: 14.8 -> 7.7 us. What is left is the launch and the one trip to memory.
#include "mlp_row.h"
#include "sac_heads.h"
#include "sac_update.h"

typedef float row_floatx4 __attribute__((ext_vector_type(4)));

namespace {
constexpr int MAX_H = 256, MAX_IN = 128, MAX_OUT = 16, WAVES = 16, THREADS = WAVES * 64;
struct RowNet { const float* W[3]; const float* b[3]; float* pre[3]; float* out[3]; int act[3]; int in, hid, n_out; };
struct RowLaunch { RowNet net; const float* x; int ldx; float* y; int ldy; int batch; };

// R: rows per workgroup. N1: sixteens of inputs. FULL: 256 wide, no position to mask
template <int R, int N1, bool FULL>
__global__ __launch_bounds__(THREADS) void mlp_row_kernel(RowLaunch A) {
    __shared__ __attribute__((aligned(16))) float xs[R][MAX_IN], h1[R][MAX_H], h2[R][MAX_H];
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const RowNet& N = A.net;
    const int IN = N.in, HID = FULL ? MAX_H : N.hid, OUT = N.n_out, row0 = blockIdx.x * R;
    // inputs, zero beyond the width; rows beyond the batch repeat the last one and are not stored
    for (int e = threadIdx.x; e < R * 16 * N1; e += THREADS) {
        const int r = e / (16 * N1), k = e % (16 * N1);
        const float v = A.x[(size_t)min(row0 + r, A.batch - 1) * A.ldx + min(k, IN - 1)];
        xs[r][k] = k < IN ? v : 0.f;
    }
    const bool on = FULL || 16 * wave < HID;
    const int mine = 16 * wave + 4 * (c & 3) + g;      // the unit whose sum this lane keeps (c < 4)
    float w1[4][N1];
    row_floatx4 w2[4][4], w3;
    const float b1 = N.b[0][min(mine, HID - 1)], b2 = N.b[1][min(mine, HID - 1)], b3 = N.b[2][min(wave, OUT - 1)];
    const row_floatx4 none = {0.f, 0.f, 0.f, 0.f};
    if (on) {
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int j = 0; j < N1; j++) {
                const float v = N.W[0][(size_t)min(16 * wave + 4 * q + g, HID - 1) * IN + min(c + 16 * j, IN - 1)];
                w1[q][j] = c + 16 * j < IN ? v : 0.f;
            }
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) {      // the width is a multiple of four
                const row_floatx4 v = *reinterpret_cast<const row_floatx4*>(N.W[1] + (size_t)min(16 * wave + 4 * q + g, HID - 1) * HID + min(4 * c + 64 * j, HID - 4));
                w2[q][j] = FULL || 4 * c + 64 * j < HID ? v : none;
            }
    }
    {   // layer 3: a wavefront per output, four positions per lane
        const row_floatx4 v = *reinterpret_cast<const row_floatx4*>(N.W[2] + (size_t)min(wave, OUT - 1) * HID + min(4 * lane, HID - 4));
        w3 = FULL || 4 * lane < HID ? v : none;
    }
    // A row's sums meet in all of their sixteen lanes: PACK rows of a unit lie in lanes c = 4 (row of the PACK) + q, which apply the activation function to all of them at once (a row at a time it
    // is a chain for each, 16 of 64 lanes at work: 1,024 rows of 17-256-256-6 9.0 -> 7.7 us, 2,048 13.6 -> 11.2; with tanh 10.3 -> 7.9 and 15.9 -> 11.9)
    constexpr int PACK = R < 4 ? R : 4;
    auto keep = [&](float& kept, float (&s)[4], int u) {
#pragma unroll
        for (int q = 0; q < 4; q++) { const float sum = rlt_sac::row16_sum(s[q]); kept = (PACK == 1 ? c & 3 : c) == 4 * u + q ? sum : kept; }
    };
    auto finish = [&](int l, float kept, float bias, float (*next)[MAX_H], int first) {
        const int r = PACK == 1 ? first : first + (c >> 2);
        if (c < 4 * PACK) {
            const float pre = kept + bias, o = rlt_act(pre, N.act[l]);
            const bool ok = FULL || mine < HID;
            next[r][mine] = ok ? o : 0.f;
            if (ok && row0 + r < A.batch) {
                if (N.pre[l]) N.pre[l][(size_t)(row0 + r) * HID + mine] = pre;
                if (N.out[l]) N.out[l][(size_t)(row0 + r) * HID + mine] = o;
            }
        }
    };
    rlt_lds_barrier();
    if (on) {
#pragma unroll
        for (int first = 0; first < R; first += PACK) {
            float kept = 0.f;
#pragma unroll
            for (int u = 0; u < PACK; u++) {
                float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < N1; j++) {
                    const float a = xs[first + u][c + 16 * j];
#pragma unroll
                    for (int q = 0; q < 4; q++) s[q] += w1[q][j] * a;
                }
                keep(kept, s, u);
            }
            finish(0, kept, b1, h1, first);
        }
    } else if (c < 4) {
#pragma unroll
        for (int r = 0; r < R; r++) { h1[r][mine] = 0.f; h2[r][mine] = 0.f; }
    }
    rlt_lds_barrier();
    if (on) {
#pragma unroll
        for (int first = 0; first < R; first += PACK) {
            float kept = 0.f;
#pragma unroll
            for (int u = 0; u < PACK; u++) {
                float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const row_floatx4 a = *reinterpret_cast<const row_floatx4*>(&h1[first + u][4 * c + 64 * j]);
#pragma unroll
                    for (int q = 0; q < 4; q++)
#pragma unroll
                        for (int e = 0; e < 4; e++) s[q] += w2[q][j][e] * a[e];
                }
                keep(kept, s, u);
            }
            finish(1, kept, b2, h2, first);
        }
    }
    rlt_lds_barrier();
    if (wave < OUT) {
        float kept = 0.f;      // row r's output in lane r
#pragma unroll
        for (int r = 0; r < R; r++) {
            const row_floatx4 a = *reinterpret_cast<const row_floatx4*>(&h2[r][4 * lane]);
            const float s = rlt_sac::groups_sum(rlt_sac::row16_sum((w3[0] * a[0] + w3[1] * a[1]) + (w3[2] * a[2] + w3[3] * a[3])));
            kept = lane == r ? s : kept;
        }
        if (lane < R && row0 + lane < A.batch) {
            const size_t row = row0 + lane;
            const float pre = kept + b3, o = rlt_act(pre, N.act[2]);
            if (N.pre[2]) N.pre[2][row * OUT + wave] = pre;
            if (N.out[2]) N.out[2][row * OUT + wave] = o;
            if (A.y) A.y[row * A.ldy + wave] = o;
        }
    }
}

template <int R>
void launch(rlt_rocm_device* device, const RowLaunch& a) {
    const dim3 grid(rlt_div_up(a.batch, R));
#define RLT_LAUNCH_ROW(N1) \
    do { if (a.net.hid == MAX_H) hipLaunchKernelGGL((mlp_row_kernel<R, N1, true>), grid, dim3(THREADS), 0, device->stream, a); \
         else hipLaunchKernelGGL((mlp_row_kernel<R, N1, false>), grid, dim3(THREADS), 0, device->stream, a); } while (0)
    if (a.net.in <= 32) RLT_LAUNCH_ROW(2); else RLT_LAUNCH_ROW(MAX_IN / 16);
#undef RLT_LAUNCH_ROW
}
}  // namespace

int rlt_mlp_row_forward(rlt_rocm_device* device, const rlt_dense_layer* L, int n_layers, const float* x, int ldx, float* y, int ldy, int batch, bool keep) {
    if (n_layers != 3 || batch < 1 || batch > RLT_MLP_ROW_MAX_BATCH || L[0].in_dim > MAX_IN || L[2].out_dim > MAX_OUT) return RLT_E_UNSUPPORTED;
    const int hid = L[0].out_dim;
    if (hid < 4 || hid > MAX_H || hid % 4 != 0 || L[1].out_dim != hid) return RLT_E_UNSUPPORTED;
    for (int l = 1; l < 3; l++) if ((reinterpret_cast<uintptr_t>(L[l].weights) & 15u) != 0) return RLT_E_UNSUPPORTED;
    // nothing here needs the weight copies' buffer, but a program that makes its first pass through this call may record the passes behind it into a graph
    if (!device->capturing) { const int rc = rlt_mlp_wide_reserve(device); if (rc) return rc; }
    RowLaunch a = {};
    for (int l = 0; l < 3; l++) {
        a.net.W[l] = L[l].weights; a.net.b[l] = L[l].biases; a.net.act[l] = L[l].activation;
        if (keep) { a.net.pre[l] = L[l].pre_activations; a.net.out[l] = L[l].output; }
    }
    a.net.in = L[0].in_dim; a.net.hid = hid; a.net.n_out = L[2].out_dim;
    a.x = x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.batch = batch;
    // Workgroups are one to a compute unit. Rows per workgroup 1, 2, 4, 8 (256 ... 2,048 rows), calls in a row: 5.8, 6.2, 7.7, 11.2 us per call of 17-256-256-6, 5.2, 5.1, 6.0, 7.9 us at width 128 (11.3 to
    // 12.6 and 8.7 to 8.9 on the tiles of mlp_wide_kernel with the weight copies before them; where the line lies: rlt_mlp_row_first).
    const int units = device->compute_units > 0 ? device->compute_units : 256;
    if (batch <= units) launch<1>(device, a); else if (batch <= 2 * units) launch<2>(device, a); else if (batch <= 4 * units) launch<4>(device, a); else launch<8>(device, a);
    return rlt_launch_status(device);
}
