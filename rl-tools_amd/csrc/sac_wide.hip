// One launch for the network passes of a SAC critic update, one for those of an actor update, for three-layer networks of any hidden width
// up to 256 (the zoo's agents are 256 wide: src/rl/zoo/acrobot-swingup-v0/sac.h, ant-v4): actors obs -> h -> h -> 2 act, critics
// obs + act -> h -> h -> 1, at most 128 critic inputs and 8 actions.
// reference: rl/algorithms/sac/operations_generic.h:243-337 (train_critic), :395-468 (train_actor),
//            nn/layers/sample_and_squash/operations_generic.h:148-398, nn_models/mlp/operations_generic.h:128-260.
//
// A workgroup of sixteen wavefronts takes 16, 8 or 4 rows of the batch (tile_rows()) through the passes that depend on each other; passes that do not depend on each other have workgroups
// of their own (a role each), which hand over a few values per row through memory:
//   critic update   target roles: actor on the next observations -> squashed sample and its log-probability -> one target critic on [next observation | sample];
//                   critic roles: trained critic forward on the current rows -> (wait for the targets' values) -> TD target -> MSE gradient -> backward
//   actor update    a role per critic: actor forward -> squashed sample -> critic forward and the gradient of -value / batch with respect to the action; critic 0's goes on
//                   (with critic 1's values): gradient of the smaller value per row -> sample_and_squash backward (entropy term, log_alpha gradient) -> actor backward
// The same kernel runs TD3's two updates (rl/algorithms/td3/operations_generic.h:170-281; actors obs -> h -> h -> act with a tanh output followed by the
// td3_sampling layer): the critic update with the target actor, the smoothing noise on the next action and no entropy term (each critic's targets are formed with
// sampling noise of its own, so each has its own pair of target roles), the actor update through critic 0 only.
// Wavefront w owns hidden units 16 w .. 16 w + 15 of every layer: it computes that tile of the 16 x h activations from the whole previous
// layer (LDS, behind a workgroup barrier; the products of the first two layers and of the way back between them, `chunks`, run over the tile's rows only, the narrow ones
// over sixteen whatever the tile, the rows beyond it being nobody's), contributes the units' share of the output layer's reduction (the partial tiles are added in
// wavefront order), and in the backward pass owns the same units' pre-activation gradients.
// Weights are read from memory (L2) straight into the B operands of v_mfma_f32_16x16x4_f32, the next pass's while this one runs; hidden widths that are no multiple
// of 16 are completed with zero operands. The reduction index of a 16-deep chunk is dealt to the four lane groups as k = 16 j + 4 g + i for the i-th of four
// instructions, so that activations (LDS) and weights (memory) are both read 16 bytes at a time.
// The trained network's activations and pre-activation gradients go to memory (4 KB per row at width 256); the weight gradients and the optimisers' steps are the next
// launch (batch_gradient.hip). Before, a workgroup ended with its sixteen rows' weight gradients (6.5 us on the matrix pipe at width 256) and a block of partial sums
// that the optimisers' launch added up, and took all passes one after the other. At width 256, batch 256 (kernel and optimisers' launch; before / now): SAC critics
// 55.7 + 10.6 / 26.0 + 8.2 us, SAC actor 65.6 + 10.6 / 33.9 + 8.2 us; TD3 critics (27 + 8 inputs) 61.1 + 11.9 / 28.1 + 8.0 us, TD3 actor 50.5 + 8.4 / 35.9 + 8.0 us.
// With four rows per workgroup instead of sixteen: SAC critics / actor 26.5 / 33.8 -> 20.1 / 23.5 us, TD3 critics (eight) / actor 28.9 / 34.5 -> 24.9 / 25.2 us (23.9 / 23.0 with the noise drawn by several wavefronts).
// Bound: a workgroup's layer of R x 256 x 256 is R * 512 cycles of one compute unit's matrix pipeline (0.9 us with four rows, 3.4 with sixteen) and 256 KB of weights from L2 (1.7 us at
// 64 B per cycle, while something else runs), and the longest chain has three of them (critic update) or four (actor update); the trips to memory at the start (3 us) and for the
// values handed over (2 us) and the narrow layers between them come on top.
#include "sac_update.h"
#include "optim.h"
#include "rng.h"
#include "sac_heads.h"
#include "batch_gradient.h"

namespace {
using namespace rlt_sac;
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) floatx4* lptr4;
constexpr int FEW = 4;      // first-layer chunks that leave registers for a whole pass's operands at once
constexpr int ROWS = 16, MAX_H = 256, WAVES = MAX_H / 16, THREADS = 64 * WAVES, S = MAX_H + 4, MAX_D = 128, SXS = MAX_D + 4, MAX_ACT = 8, MAX_OUT = 16, D3S = MAX_OUT + 1,
              MISC = 64, YP = ROWS * D3S;
enum { MODE_CRITIC = 0, MODE_ACTOR = 1, MODE_TD3_CRITIC = 2, MODE_TD3_ACTOR = 3 };      // SAC's two updates, TD3's two updates

// W1f, W2f, W2b: copies of the weights in the order the wavefronts consume them (wide_prepare_kernel)
struct WNet { const float *W1, *b1, *W2, *b2, *W3, *b3; int in, hid, out, act_h, vec3; const float *W1f, *W2f, *W2b; };      // vec3: the rows of W3 can be read 16 bytes at a time
struct Trained { float *h1, *h2, *d1, *d2, *d3; };      // [batch][hid] each, d3 [batch][MAX_OUT]
constexpr int EXCHANGE = ROWS * (1 + MAX_ACT), LOG_PROB_SLOT = 4;      // words per tile: critic update [slot][row] (slot = 2 set + target, then the log-probabilities), actor update [row] values, then [row][action]
struct WideArgs {
    WNet actor, critic[2], target[2];
    const float* batch_base;               // [2][batch][obs + act]: current rows, then next rows
    const float* rewards; const uint8_t* terminated;
    const float* noise;                    // [batch][act], or NULL: drawn from (noise_seed, noise_stream + *stream_offset)
    uint64_t noise_seed, noise_stream; float* out_noise; const uint64_t* stream_offset;
    // TD3's critic update with its draws made here (noise, noise_second and target_noise NULL): the second critic's sampling noise and the smoothing noise
    // clamp(N(0, 1) * target_noise_std, -clip, clip) on streams of their own, the latter stored to out_target_noise
    uint64_t noise_stream_second, target_noise_stream; float target_noise_std, target_noise_clip; float* out_target_noise;
    const float* log_alpha;
    rlt_sas_parameters sas;
    float gamma;
    int batch, obs, act;
    int groups, roles, n_critics, by_xcd;   // row tiles, workgroups per tile, critics trained by the launch; by_xcd: workgroups of a role lie on as few XCDs as possible (each has its own L2)
    Trained trained[2];                    // where the trained networks' activations and gradients go
    float* extra;                          // actor update: [groups] the tiles' shares of the log_alpha gradient
    uint64_t* exchange; unsigned max_poll; unsigned* fault;      // [groups][EXCHANGE] values handed from role to role: the value in the low word, a tag in the high one, zero before the launch
    float* out_log_probabilities; float* out_target_action_value; float* out_actions; float* out_pre_squashing;
    // TD3 (rl/algorithms/td3/operations_generic.h:170-281): `actor` is the target actor in the critic update and has `act` outputs; they pass tanh and the
    // td3_sampling layer (sac_heads.h); the critic update adds target_noise [batch][act] (already clamped) to the next action; the actor update goes through critic[0] only
    float sampling_std; int ignore_termination; const float* target_noise; float* out_pre_clip;
    const float* noise_second;             // TD3 critic update of both critics in one launch: the sampling noise of the second, each critic's targets being formed with its own
};

__device__ __forceinline__ floatx4 mfma16(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
template <int ACT_H> __device__ __forceinline__ float act_hidden(float x, int f) { return rlt_act(x, ACT_H >= 0 ? ACT_H : f); }
template <int ACT_H> __device__ __forceinline__ float dact_hidden(float o, int f) { return rlt_dact_from_output(o, ACT_H >= 0 ? ACT_H : f); }

// The loads of operands are unconditional, from addresses clamped into the arrays: a load that some wavefronts skip makes the compiler wait for every load in flight before
// the first value requested ahead of it is used (4 us at the start of a launch: the input rows, requested first, were waited for together with all weights). What lies
// beyond a layer's shape is masked where it is used.
// Weights are read from copies laid out in consumption order: [wavefront's 16 units][16-deep chunk j][lane][4] -- lane (c, g) finds W[16 w + c][16 j + 4 g ... + 3]
// (forward copies of the first and second layers) or W[16 j + 4 g ... + 3][16 w + c] (backward copy of the second), zero beyond the layer's shape, and a wavefront's
// load is 1 KB of consecutive addresses. Straight from W a lane's 16 bytes lie a row apart from its neighbour's: 64 lines per load, which the compute unit's address
// pipeline takes 64 cycles for; first layers whose rows are no multiple of 16 bytes (17 or 35 inputs) take four such loads per chunk, 5 us at the start of a launch.
// A wavefront without units asks for nothing, the others for chunks in groups of STEP up to the width; within a group, chunks beyond it are asked for at one address by all lanes. A load
// that nobody uses still takes sixteen cycles of a compute unit's return path: at width 65, with all sixteen wavefronts asking for all chunks, 224 of 288 were such (SAC's
// actor update at width 65 over 600 rows 32.5 -> 29.0 us, update set at width 32 over 100 rows 47.3 -> 41.2, forward + backward of 17-48-48-6 at 256 rows 12.5 -> 10.9). The first layer's few chunks one by one.
// EVERY: where every wavefront has units and all sixteen chunks of the second layer are there, there is nothing to leave out, and the selects cost more than they save (forward +
// backward of 256 units 36.2 us with them, 35.4 without; SAC's update set 86.2 and 86.0).
template <int NT1C> constexpr int FIRST_STEP = NT1C <= FEW ? 1 : 4;      // (five chunks and more: the branches cost more)
// How the weights come: FORM_ANY and FORM_EVERY (see EVERY above) from the copies; FORM_DIRECT, MLP passes of exactly 256 units whose second layer lies on 16 bytes, from the layers themselves, without
// the launch that makes the copies (3.2 to 3.7 us). What a lane needs of the second layer on the way forward is four values that lie a row apart from its neighbours'; it is asked for as it lies, four
// neighbouring lanes 64 bytes of one row (a 256 x 256 layer in 1.85 us, as from the copies; 6.96 where every lane has a row of its own), and dealt out in registers by selects that fetch from the
// neighbouring lane, 128 per wavefront and layer beside 64 matrix instructions. On the way back only tiles of sixteen rows need such a dealing, by moves that the compiler sees (deal_values). Rows of the first layer are any number of floats; its few
// chunks go through the wavefront's own part of the LDS. 17-256-256-6, copies / direct: step with the gradients' clearing, forward + backward in one call and Adam 28.5 / 28.1 us at 256 rows, 34.8 / 34.5 at
// 1,000, 42.9 / 42.6 at 2,048, 48.4 / 48.1 at 3,000, 52.7 / 52.5 at 4,096; forward pass alone 15.0 / 13.8 at 2,049 rows, 16.5 / 15.1 at 4,096; backward pass alone 16.0 / 12.7 at 256, 21.3 / 19.2 at 1,000,
// 27.3 / 25.7 at 2,048, 30.7 / 29.3 at 3,000, 34.0 / 33.0 at 4,096. The updates of SAC and TD3, whose
// chains have two or three layers to deal out one after the other, keep the copies (sets at 256 rows 66.3 / 67.6 and 78.0 / 78.7).
enum { FORM_ANY = 0, FORM_EVERY = 1, FORM_DIRECT = 2 };
constexpr int W1S = 36, W1_STAGE = 16 * W1S;      // a wavefront's sixteen rows of two chunks, the rows four banks apart
// a's values of the upper lanes of pairs against b's of the lower ones, as selects whose first operand comes through the lane control (left to the compiler, the exchange is an instruction of its own).
// The compiler does not look into an asm statement, so the statement brings its wait states itself (tests/test_dpp_wait_states.py looks the built instructions over): two between what writes an operand and
// the lane control that reads it; two behind a deal's last ones before a matrix instruction reads what they leave; and it must not write a register that a matrix instruction is still writing. On tiles of
// four and eight rows those are the 4 x 4 x 1 ones, which take four: the three states in front of the first select and one more. On tiles of sixteen rows they take ten, too many to wait for; there no
// output is of the compiler's choice: b is exchanged in place, a goes to spare's registers and leaves its own as the next exchange's, so that each holds a value that the compiler itself wrote there.
#define RLT_SELECT(to, from, own, CONTROL) "v_cndmask_b32_dpp %" #to ", %" #from ", %" #own ", vcc " CONTROL " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
#define RLT_EXCHANGE(CONTROL, END)                                                                                                                                 \
    if constexpr (R == ROWS)                                                                                                                                       \
        asm("s_nop 1\n\ts_mov_b64 vcc, %6\n\t" RLT_SELECT(0, 2, 4, CONTROL) RLT_SELECT(1, 3, 5, CONTROL) "s_mov_b64 vcc, %7\n\t" RLT_SELECT(2, 4, 2, CONTROL)      \
            RLT_SELECT(3, 5, 3, CONTROL) END : "+&v"(x0), "+&v"(x1), "+&v"(b0), "+&v"(b1), "+&v"(a0), "+&v"(a1) : "s"(~upper), "s"(upper) : "vcc");                 \
    else                                                                                                                                                           \
        asm("s_nop 2\n\ts_mov_b64 vcc, %8\n\t" RLT_SELECT(0, 6, 4, CONTROL) RLT_SELECT(1, 7, 5, CONTROL) "s_mov_b64 vcc, %9\n\t" RLT_SELECT(2, 4, 6, CONTROL)      \
            RLT_SELECT(3, 5, 7, CONTROL) END : "=&v"(x0), "=&v"(x1), "=&v"(y0), "=&v"(y1) : "v"(a0), "v"(a1), "v"(b0), "v"(b1), "s"(~upper), "s"(upper) : "vcc")
constexpr uint64_t LANES_1 = 0xAAAAAAAAAAAAAAAAull, LANES_2 = 0xCCCCCCCCCCCCCCCCull;      // lanes with that bit
template <int R, uint64_t upper> __device__ __forceinline__ void exchange(floatx4& a, floatx4& b, floatx4& spare) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        float a0 = a[i], a1 = a[i + 1], b0 = b[i], b1 = b[i + 1], x0 = spare[i], x1 = spare[i + 1], y0 = 0.f, y1 = 0.f;
        if constexpr (upper == LANES_1) { RLT_EXCHANGE("quad_perm:[1,0,3,2]", ""); }
        else { RLT_EXCHANGE("quad_perm:[2,3,0,1]", "s_nop 1"); }
        a[i] = x0; a[i + 1] = x1;
        if constexpr (R == ROWS) { b[i] = b0; b[i + 1] = b1; spare[i] = a0; spare[i + 1] = a1; } else { b[i] = y0; b[i + 1] = y1; }
    }
}
#undef RLT_EXCHANGE
#undef RLT_SELECT
// 16 bytes of load t in lane u of a group of four lanes <-> load u in lane t
template <int R>
__device__ __forceinline__ void deal_loads(floatx4& b0, floatx4& b1, floatx4& b2, floatx4& b3, floatx4& spare) {
    exchange<R, LANES_1>(b0, b1, spare); exchange<R, LANES_1>(b2, b3, spare);
    exchange<R, LANES_2>(b0, b2, spare); exchange<R, LANES_2>(b1, b3, spare);
}
// The same between groups of four lanes: moves that leave a group its own
template <int CONTROL, int GROUPS> __device__ __forceinline__ float into_groups(float own, float from) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(own), __float_as_int(from), CONTROL, 0xF, GROUPS, false));
}
template <int FROM_LOWER, int FROM_UPPER, int UPPER> __device__ __forceinline__ void exchange_groups(floatx4& a, floatx4& b) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x = into_groups<FROM_LOWER, UPPER>(a[i], b[i]), y = into_groups<FROM_UPPER, 0xF & ~UPPER>(b[i], a[i]);
        a[i] = x; b[i] = y;
    }
}
// value i of four loads in group of four lanes q of sixteen <-> value q in group i
__device__ __forceinline__ void deal_values(floatx4& b0, floatx4& b1, floatx4& b2, floatx4& b3) {
    floatx4 x0 = {b0[0], b1[0], b2[0], b3[0]}, x1 = {b0[1], b1[1], b2[1], b3[1]}, x2 = {b0[2], b1[2], b2[2], b3[2]}, x3 = {b0[3], b1[3], b2[3], b3[3]};
    exchange_groups<0x114, 0x104, 0xA>(x0, x1); exchange_groups<0x114, 0x104, 0xA>(x2, x3);      // row_shr:4, row_shl:4
    exchange_groups<0x128, 0x128, 0xC>(x0, x2); exchange_groups<0x128, 0x128, 0xC>(x1, x3);      // row_ror:8
    b0 = floatx4{x0[0], x1[0], x2[0], x3[0]}; b1 = floatx4{x0[1], x1[1], x2[1], x3[1]}; b2 = floatx4{x0[2], x1[2], x2[2], x3[2]}; b3 = floatx4{x0[3], x1[3], x2[3], x3[3]};
}
// forward: rows 16 w + c of W2, half h of the reduction; after deal_second() element 4 p + t of lane (c, g) holds k = 64 p + 16 g + 4 t ...
__device__ __forceinline__ void request_second(const float* W2, int wave, int c, int g, int half, floatx4 (&b)[8]) {
    const float* const mine = W2 + (size_t)(16 * wave + (c & 12)) * MAX_H + 128 * half + 16 * g + 4 * (c & 3);
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int t = 0; t < 4; t++) b[4 * p + t] = *reinterpret_cast<const floatx4*>(mine + t * MAX_H + 64 * p);
}
template <int R>
__device__ __forceinline__ void deal_second(floatx4 (&b)[8]) {
    floatx4 spare = {0.f, 0.f, 0.f, 0.f};
    deal_loads<R>(b[0], b[1], b[2], b[3], spare); deal_loads<R>(b[4], b[5], b[6], b[7], spare);
}
// backward: columns 16 w ... of W2. Tiles of sixteen rows: after deal_values() element j of lane (c, g) holds rows 16 j + 4 g ... + 3 of column own_column(w, c). Tiles of four and eight need no
// dealing: element j of lane l holds row 16 (l / 4) + j, columns 16 w + 4 (l % 4) ... + 3 (column_products), and the sums end in the same column.
template <int R>
__device__ __forceinline__ void request_second_columns(const float* W2, int wave, int c, int g, floatx4 (&b)[MAX_H / 16]) {
    const float* const mine = W2 + (size_t)(R == ROWS ? 4 * g + (c >> 2) : 16 * (4 * g + (c >> 2))) * MAX_H + 16 * wave + 4 * (c & 3);
#pragma unroll
    for (int j = 0; j < MAX_H / 16; j++) b[j] = *reinterpret_cast<const floatx4*>(mine + (size_t)(R == ROWS ? 16 : 1) * j * MAX_H);
}
template <int FORM> __device__ __forceinline__ int own_column(int wave, int c) { return 16 * wave + (FORM == FORM_DIRECT ? 4 * (c & 3) + (c >> 2) : c); }
// first layer: rows 16 w + 4 q + g, column 16 j + c into element q of chunk j; place_first() turns them into the operands that the copies hold
template <int NT1C>
__device__ __forceinline__ void request_first(const float* W1, int in, int wave, int c, int g, floatx4 (&b)[NT1C]) {
#pragma unroll
    for (int j = 0; j < NT1C; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) b[j][q] = W1[(size_t)(16 * wave + 4 * q + g) * in + min(16 * j + c, in - 1)];
}
template <int NT1C>
__device__ __forceinline__ void place_first(int in, lptr stage, int c, int g, floatx4 (&b)[NT1C]) {
#pragma unroll
    for (int j0 = 0; j0 < NT1C; j0 += 2) {
#pragma unroll
        for (int j = j0; j < j0 + 2; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) stage[(4 * q + g) * W1S + 16 * (j & 1) + c] = 16 * j + c < in ? b[j][q] : 0.f;
        wave_sync();
#pragma unroll
        for (int j = j0; j < j0 + 2; j++) b[j] = *(lptr4)(stage + c * W1S + 16 * (j & 1) + 4 * g);
        wave_sync();
    }
}
template <int JN, bool EVERY = false, int STEP = 4>
__device__ __forceinline__ void load_swizzled(const float* __restrict__ copy, int tiles, bool on, int wave, int lane, int j0, floatx4 (&b)[JN]) {      // tiles: chunks of the copy; on: this wavefront has units
    if (EVERY) {
        const float* const mine = copy + ((size_t)wave * tiles * 64 + lane) * 4;
#pragma unroll
        for (int j = 0; j < JN; j++) b[j] = *reinterpret_cast<const floatx4*>(mine + (size_t)min(j0 + j, tiles - 1) * 256);
        return;
    }
    if (!on) return;
    const uint32_t mine = ((uint32_t)wave * tiles * 64 + lane) * 16;
#pragma unroll
    for (int q = 0; q < JN; q += STEP) {
        if (j0 + q >= tiles) return;
#pragma unroll
        for (int j = q; j < q + STEP && j < JN; j++)
            b[j] = *reinterpret_cast<const floatx4*>(reinterpret_cast<const char*>(copy) + (j0 + j < tiles ? mine + (uint32_t)(j0 + j) * 1024 : 0));
    }
}
// A workgroup's rows R against this lane's column: sixteen on v_mfma_f32_16x16x4_f32, or eight or four on v_mfma_f32_4x4x1_16b_f32 (sixteen blocks of 4 x 1 by 1 x 4: block 4 g + q takes
// columns 4 q .. 4 q + 3 of the wavefront's sixteen and lane group g's share of the reduction, so the weights lie in the lanes as the other instruction has them, and half the rows
// are half the cycles). The activations of four chunks are one read per four rows: block q of a group of four holds those of chunk 4 J + q and hands them to the other three.
template <int R> struct Sums { floatx4 s[R == 16 ? 1 : R / 4][2]; };
template <int R> __device__ __forceinline__ void clear(Sums<R>& A) {
#pragma unroll
    for (int h = 0; h < (R == 16 ? 1 : R / 4); h++) A.s[h][0] = A.s[h][1] = floatx4{0.f, 0.f, 0.f, 0.f};
}
template <int Q> __device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 2, Q, 0); }
template <int R, int Q>
__device__ __forceinline__ void chunk4(Sums<R>& A, const floatx4 (&a)[R / 4], floatx4 b) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int h = 0; h < R / 4; h++) A.s[h][i & 1] = mfma4<Q>(a[h][i], b[i], A.s[h][i & 1]);
}
// A += in[rows][16 (j0 + j) + ...] * b[j], j0 a multiple of four; ROWS_AS_THEY_LIE: b[4 p + t] holds k = 64 p + 16 g + 4 t ... (deal_second) instead of 16 (4 p + t) + 4 g ...
template <int R, bool ROWS_AS_THEY_LIE = false, int JN>
__device__ __forceinline__ void chunks(Sums<R>& A, lptr in, int stride, int c, int g, int j0, int steps, const floatx4 (&b)[JN]) {
    if constexpr (R == 16) {
#pragma unroll
        for (int j = 0; j < JN; j++) {
            if (j0 + j < steps) {
                const floatx4 a = *(lptr4)(in + c * stride + (ROWS_AS_THEY_LIE ? 64 * ((j0 + j) >> 2) + 16 * g + 4 * (j & 3) : 16 * (j0 + j) + 4 * g));
                A.s[0][0] = mfma16(a[0], b[j][0], A.s[0][0]); A.s[0][1] = mfma16(a[1], b[j][1], A.s[0][1]);
                A.s[0][0] = mfma16(a[2], b[j][2], A.s[0][0]); A.s[0][1] = mfma16(a[3], b[j][3], A.s[0][1]);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < JN; j += 4) {
            if (j0 + j < steps) {
                floatx4 a[R / 4];      // (columns of chunks beyond the width hold anything: nobody multiplies them)
#pragma unroll
                for (int h = 0; h < R / 4; h++) a[h] = *(lptr4)(in + ((c & 3) + 4 * h) * stride + 16 * (j0 + j) + (ROWS_AS_THEY_LIE ? 16 * g + (c & 12) : 4 * (c & 12) + 4 * g));
                chunk4<R, 0>(A, a, b[j]);
                if (j + 1 < JN && j0 + j + 1 < steps) chunk4<R, 1>(A, a, b[j + 1 < JN ? j + 1 : 0]);
                if (j + 2 < JN && j0 + j + 2 < steps) chunk4<R, 2>(A, a, b[j + 2 < JN ? j + 2 : 0]);
                if (j + 3 < JN && j0 + j + 3 < steps) chunk4<R, 3>(A, a, b[j + 3 < JN ? j + 3 : 0]);
            }
        }
    }
}
// the finished sums: element v of lane (c, g) belongs to row R / 4 * g + v, column c (the shares of the lane groups are added up in exchanges that leave each half of the rows)
template <int R>
__device__ __forceinline__ void finished(const Sums<R>& A, float (&out)[R / 4]) {
    floatx4 s[R == 16 ? 1 : R / 4];
#pragma unroll
    for (int h = 0; h < (R == 16 ? 1 : R / 4); h++) s[h] = A.s[h][0] + A.s[h][1];
    if constexpr (R == 16) {
#pragma unroll
        for (int v = 0; v < 4; v++) out[v] = s[0][v];
    } else {
        constexpr int E = R / 4;
        float t[2 * E];
#pragma unroll
        for (int v = 0; v < 2 * E; v++) {      // row v and row 2 E + v
            const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[v / 4][v & 3]), __float_as_uint(s[(2 * E + v) / 4][(2 * E + v) & 3]), false, false);
            t[v] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        }
#pragma unroll
        for (int v = 0; v < E; v++) {
            const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(t[v]), __float_as_uint(t[E + v]), false, false);
            out[v] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        }
    }
}

// Tiles of four and eight rows times 256 rows of W as request_second_columns() has asked for them: block l / 4 of the matrix instruction takes its sixteen rows of the reduction, instruction i column
// i of each lane's four. out: as finished() leaves it, for column own_column(): the blocks' shares are added up in exchanges that leave each half of the rows, then each half of the columns.
template <int CTRL> __device__ __forceinline__ float lane_move(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true)); }
template <int R>
__device__ __forceinline__ void column_products(lptr in, int stride, int lane, const floatx4 (&b)[MAX_H / 16], float (&out)[R / 4]) {
    constexpr int N = R / 4, E = R / 4;
    floatx4 sum[N][4];
#pragma unroll
    for (int h = 0; h < N; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) sum[h][i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j0 = 0; j0 < MAX_H / 16; j0 += 4) {
        floatx4 a[N];
#pragma unroll
        for (int h = 0; h < N; h++) a[h] = *(lptr4)(in + ((lane & 3) + 4 * h) * stride + 16 * (lane >> 2) + j0);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int h = 0; h < N; h++)
#pragma unroll
                for (int i = 0; i < 4; i++) sum[h][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[h][j], b[j0 + j][i], sum[h][i], 0, 0, 0);
    }
    float t[E][4];      // rows E g + v, column i of the lane's four, summed over the lane groups
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float s[2 * E];
#pragma unroll
        for (int v = 0; v < 2 * E; v++) {
            const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[v / 4][i][v & 3]), __float_as_uint(sum[(2 * E + v) / 4][i][(2 * E + v) & 3]), false, false);
            s[v] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        }
#pragma unroll
        for (int v = 0; v < E; v++) {
            const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[v]), __float_as_uint(s[E + v]), false, false);
            t[v][i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        }
    }
    const bool third = lane & 8, second = lane & 4;      // which column of the four this lane ends with: (lane / 4) % 4
#pragma unroll
    for (int v = 0; v < E; v++) {
        const float p = (third ? t[v][2] : t[v][0]) + lane_move<0x128>(third ? t[v][0] : t[v][2]);
        const float q = (third ? t[v][3] : t[v][1]) + lane_move<0x128>(third ? t[v][1] : t[v][3]);
        const float lower = lane_move<0x104>(p), upper = lane_move<0x114>(q);      // the first column's share of the group above, the second's of the group below
        out[v] = second ? q + upper : p + lower;
    }
}

// profiling builds (-DRLT_WIDE_PROFILE): thread 0 of workgroup 0 notes the constant-rate clock at the stage boundaries, rlt_sac_wide_ticks copies the notes out
#ifdef RLT_WIDE_PROFILE
__device__ unsigned long long rlt_wide_ticks[2][32];
#define RLT_TICK(i) do { if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) rlt_wide_ticks[MODE & 1][i] = wall_clock64(); } while (0)
#else
#define RLT_TICK(i) do {} while (0)
#endif

// A wavefront's weight operands of one network: its 16 units' rows of W1 and W2 (the B operands of layers 1 and 2), row c of W3 for its 16 units, its lane's biases
template <int NT1C>
struct Operands { floatx4 w1[NT1C], w2a[8], w2b[8], w3; float b1, b2; };
__device__ __forceinline__ floatx4 load_w3(const WNet& N, int wave, int c, int g) {      // row c of W3 (c < out), this wavefront's 16 units
    floatx4 w3;
    const int k = 16 * wave + 4 * g;
    const float* row = N.W3 + (size_t)min(c, N.out - 1) * N.hid;
    if (N.vec3) w3 = *reinterpret_cast<const floatx4*>(row + min(k, N.hid - 4));      // hid is a multiple of 4 here
    else {
#pragma unroll
        for (int i = 0; i < 4; i++) w3[i] = row[min(k + i, N.hid - 1)];
    }
    return w3;
}
__device__ __forceinline__ void mask_w3(const WNet& N, int wave, int c, int g, floatx4& w3) {
#pragma unroll
    for (int i = 0; i < 4; i++) if (c >= N.out || 16 * wave + 4 * g + i >= N.hid) w3[i] = 0.f;
}
// everything of network N that forward3 reads from memory, requested at once (few first-layer operands leave room for the whole second layer; otherwise its second
// half is requested after the first layer has run)
template <int NT1C, int FORM>
__device__ __forceinline__ void load_first(const WNet& N, bool on, int wave, int c, int g, floatx4 (&b)[NT1C]) {
    if (FORM == FORM_DIRECT) request_first(N.W1, N.in, wave, c, g, b);
    else load_swizzled<NT1C, false, FIRST_STEP<NT1C>>(N.W1f, (N.in + 15) >> 4, on, wave, c + 16 * g, 0, b);
}
template <int FORM>
__device__ __forceinline__ void load_second(const WNet& N, int tiles, bool on, int wave, int c, int g, int half, floatx4 (&b)[8]) {
    if (FORM == FORM_DIRECT) request_second(N.W2, wave, c, g, half, b);
    else load_swizzled<8, FORM == FORM_EVERY>(N.W2f, tiles, on, wave, c + 16 * g, 8 * half, b);
}
template <int NT1C, int FORM = FORM_ANY>
__device__ __forceinline__ void load_operands(const WNet& N, int wave, int c, int g, Operands<NT1C>& W) {
    const int n = 16 * wave + c, tiles = (N.hid + 15) >> 4;
    const bool on = wave < tiles;
    if (FORM == FORM_ANY && !on) return;
    load_first<NT1C, FORM>(N, on, wave, c, g, W.w1);
    W.b1 = N.b1[min(n, N.hid - 1)]; W.b2 = N.b2[min(n, N.hid - 1)];
    load_second<FORM>(N, tiles, on, wave, c, g, 0, W.w2a);
    if (NT1C <= FEW) load_second<FORM>(N, tiles, on, wave, c, g, 1, W.w2b);
    W.w3 = load_w3(N, wave, c, g);
}

// The three layers of network N on the workgroup's rows x [16][xstride]: this wavefront's tile of h1 and h2 (after the activation) into
// LDS, then its units' share of the output layer's reduction into yp[wave]. Three workgroup barriers, which every wavefront meets; after
// the last one output_tile() returns the output layer's sums (without the bias).
// The operands W are in registers (or on their way) when the call starts. With PREFETCH each group of them is requested again for network `next` as soon as this
// network has used it, so that the next forward3 finds its operands loaded: a wavefront's weights are 16 KB per layer from L2, a compute unit's 256 KB, which
// took as long as the layers' arithmetic when they were requested at the start of each pass.
// First layers of more than two chunks fill too many registers for that: then only the second layer's first half (and the small operands) are requested ahead, the
// first layer's own operands at the start of the pass (W1_READY = false) and the second half after the first layer, as before.
// LIVE: the activations of rows from `live` on (beyond the batch) are zero -- zero inputs alone leave NaNs there where a weight or a bias is infinite
// KEEP: the hidden layers' pre-activations and outputs are also stored to memory, rows [row0, row0 + 16) of [batch x hid] arrays (forward() of a network keeps them)
struct KeepArgs { float* pre[2]; float* out[2]; int row0, batch; };
template <int R, int ACT_H, bool KEEP, bool LIVE>
__device__ __forceinline__ void place_hidden(const WNet& N, const Sums<R>& sums, float bias, lptr h, int n, int g, const KeepArgs* keep, int layer, int live) {
    const bool n_ok = n < N.hid;
    float acc[R / 4];
    finished<R>(sums, acc);
#pragma unroll
    for (int v = 0; v < R / 4; v++) {
        const int row = R / 4 * g + v;
        const float pre = acc[v] + bias, o = act_hidden<ACT_H>(pre, N.act_h);
        h[row * S + n] = n_ok && (!LIVE || row < live) ? o : 0.f;
        if (KEEP && n_ok && keep->row0 + row < keep->batch) {
            const size_t at = (size_t)(keep->row0 + row) * N.hid + n;
            if (keep->pre[layer]) keep->pre[layer][at] = pre;
            if (keep->out[layer]) keep->out[layer][at] = o;
        }
    }
}
template <int R, int ACT_H, int NT1C, bool PREFETCH, bool W1_READY, bool KEEP = false, int FORM = FORM_ANY, bool LIVE = false>
__device__ __forceinline__ void forward3(const WNet& N, Operands<NT1C>& W, const WNet& next, lptr x, int xstride, lptr h1, lptr h2, lptr yp, lptr stage, int wave, int c, int g, const KeepArgs* keep = nullptr,
                                         int live = ROWS) {
    constexpr bool DIRECT = FORM == FORM_DIRECT;
    const int n = 16 * wave + c, tiles = DIRECT ? MAX_H / 16 : (N.hid + 15) >> 4, lane = c + 16 * g, next_tiles = DIRECT ? MAX_H / 16 : (next.hid + 15) >> 4;
    const bool on = DIRECT || wave < tiles, next_on = DIRECT || wave < next_tiles;
    const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
    if (!W1_READY) load_first<NT1C, FORM>(N, on, wave, c, g, W.w1);
    if (DIRECT) place_first(N.in, stage, c, g, W.w1);
    if (on) {
        Sums<R> sums;
        clear(sums);
        chunks<R>(sums, x, xstride, c, g, 0, (N.in + 15) >> 4, W.w1);
        place_hidden<R, ACT_H, KEEP, LIVE>(N, sums, W.b1, h1, n, g, keep, 0, live);
    }
    if (NT1C > FEW) load_second<FORM>(N, tiles, on, wave, c, g, 1, W.w2b);
    if (PREFETCH) {
        if (NT1C <= FEW) load_first<NT1C, FORM>(next, next_on, wave, c, g, W.w1);
        W.b1 = next.b1[min(n, next.hid - 1)];
    }
    if (DIRECT) deal_second<R>(W.w2a);      // (while the others finish their tiles of the first layer)
    rlt_lds_barrier();
    {
        Sums<R> sums;
        clear(sums);
        if (on) chunks<R, DIRECT>(sums, h1, S, c, g, 0, tiles, W.w2a);
        if (PREFETCH) load_second<FORM>(next, next_tiles, next_on, wave, c, g, 0, W.w2a);
        if (DIRECT) deal_second<R>(W.w2b);
        if (on) chunks<R, DIRECT>(sums, h1, S, c, g, 8, tiles, W.w2b);
        if (PREFETCH && NT1C <= FEW) load_second<FORM>(next, next_tiles, next_on, wave, c, g, 1, W.w2b);
        if (on) place_hidden<R, ACT_H, KEEP, LIVE>(N, sums, W.b2, h2, n, g, keep, 1, live);
        if (PREFETCH) W.b2 = next.b2[min(n, next.hid - 1)];
    }
    rlt_lds_barrier();
    if (on) {
        mask_w3(N, wave, c, g, W.w3);
        const floatx4 a = *(lptr4)(h2 + c * S + 16 * wave + 4 * g);
        floatx4 y = zero4;
        y = mfma16(a[0], W.w3[0], y); y = mfma16(a[1], W.w3[1], y); y = mfma16(a[2], W.w3[2], y); y = mfma16(a[3], W.w3[3], y);
#pragma unroll
        for (int v = 0; v < 4; v++) yp[(wave * ROWS + 4 * g + v) * D3S + c] = y[v];
    }
    if (PREFETCH) W.w3 = load_w3(next, wave, c, g);
    rlt_lds_barrier();
}
// the sums of the partial tiles, in wavefront order: element v of lane (c, g) belongs to row 4 g + v, column c
__device__ __forceinline__ floatx4 output_tile(lptr yp, int tiles, int c, int g) {
    floatx4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w0 = 0; w0 < WAVES; w0 += 4) {      // four tiles' reads in flight together; tiles beyond the width's are never written
        float p[4][4];
#pragma unroll
        for (int w = 0; w < 4; w++)
#pragma unroll
            for (int v = 0; v < 4; v++) p[w][v] = yp[((w0 + w) * ROWS + 4 * g + v) * D3S + c];
#pragma unroll
        for (int w = 0; w < 4; w++)
            if (w0 + w < tiles)
#pragma unroll
                for (int v = 0; v < 4; v++) y[v] += p[w][v];
    }
    return y;
}

// column n of W3 for this lane's share of the reduction over the outputs, and the second layer's backward copy: the operands of a backward pass, requested ahead of it
struct BackOperands { float w3[MAX_OUT / 4]; floatx4 w2[MAX_H / 16]; };
template <int R, int FORM = FORM_ANY>
__device__ __forceinline__ void load_back_operands(const WNet& N, int wave, int c, int g, BackOperands& W) {
    const int n = 16 * wave + c, tiles = (N.hid + 15) >> 4;
#pragma unroll
    for (int ks = 0; ks < MAX_OUT / 4; ks++) W.w3[ks] = N.W3[(size_t)min(4 * ks + g, N.out - 1) * N.hid + min(n, N.hid - 1)];
    if (FORM == FORM_DIRECT) request_second_columns<R>(N.W2, wave, c, g, W.w2);
    else load_swizzled<MAX_H / 16, FORM == FORM_EVERY>(N.W2b, tiles, wave < tiles, wave, c + 16 * g, 0, W.w2);
}
// this wavefront's tile of d_pre2 = (d_pre3 W3) f'(h2) into g2 (may be h2 itself); returns the lane's share of its unit's column sum
template <int ACT_H, bool LIVE = false>
__device__ __forceinline__ float backward_layer3(const WNet& N, const BackOperands& W, lptr d3, lptr h2, lptr g2, int wave, int c, int g, int live = ROWS) {
    const int n = 16 * wave + c;
    const bool n_ok = n < N.hid;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
#pragma unroll
    for (int ks = 0; ks < MAX_OUT / 4; ks++) acc = mfma16(d3[c * D3S + 4 * ks + g], 4 * ks + g < N.out ? W.w3[ks] : 0.f, acc);      // columns of d_pre3 beyond the output width are zero
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int idx = (4 * g + v) * S + n;
        const float d = n_ok && (!LIVE || 4 * g + v < live) ? acc[v] * dact_hidden<ACT_H>(h2[idx], N.act_h) : 0.f;
        g2[idx] = d; sum += d;
    }
    return sum;
}
// this wavefront's tile of d_pre1 = (d_pre2 W2) f'(h1) into p1 (may be h1 itself); returns the lane's share of its unit's column sum
template <int R, int ACT_H, int FORM = FORM_ANY, bool LIVE = false>
__device__ __forceinline__ float backward_layer2(const WNet& N, BackOperands& W, lptr g2, lptr h1, lptr p1, int wave, int c, int g, int live = ROWS) {
    const int n = own_column<FORM>(wave, c), tiles = FORM == FORM_DIRECT ? MAX_H / 16 : (N.hid + 15) >> 4;
    const bool n_ok = n < N.hid;
    float acc[R / 4], sum = 0.f;
    if constexpr (FORM == FORM_DIRECT && R != ROWS) column_products<R>(g2, S, c + 16 * g, W.w2, acc);
    else {
        Sums<R> sums;
        clear(sums);
        if (FORM == FORM_DIRECT) {
#pragma unroll
            for (int j = 0; j < MAX_H / 16; j += 4) deal_values(W.w2[j], W.w2[j + 1], W.w2[j + 2], W.w2[j + 3]);
        }
        chunks<R>(sums, g2, S, c, g, 0, tiles, W.w2);
        finished<R>(sums, acc);
    }
#pragma unroll
    for (int v = 0; v < R / 4; v++) {
        const int row = R / 4 * g + v, idx = row * S + n;
        const float d = n_ok && (!LIVE || row < live) ? acc[v] * dact_hidden<ACT_H>(h1[idx], N.act_h) : 0.f;
        p1[idx] = d; sum += d;
    }
    return sum;
}
// A tile of a weight gradient over the workgroup's sixteen rows, d^T x: d [16][S], its columns 16 mt ...; x [16][stride], its columns 16 nt ...; into dst [rows][cols]
__device__ __forceinline__ void gradient_tile(lptr d, int mt, lptr x, int stride, int nt, int rows, int cols, float* dst, int c, int g) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < ROWS / 4; ks++) acc = mfma16(d[(4 * ks + g) * S + 16 * mt + c], x[(4 * ks + g) * stride + 16 * nt + c], acc);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int m = 16 * mt + 4 * g + v, n = 16 * nt + c;
        if (m < rows && n < cols) dst[(size_t)m * cols + n] = acc[v];
    }
}
// The workgroup's 16 rows of an array between memory and LDS: wavefront w takes row w, all of a lane's loads are on their way before the first is written (a loop that
// writes each element before the next load cost 3.8 us at the start of a launch, three trips to memory one after the other; and the operands' wait with it). Columns from `cols` on are zero.
template <int N>
__device__ __forceinline__ void request_row(const float* row, int cols, int lane, float (&v)[N]) {
#pragma unroll
    for (int u = 0; u < N; u++) { v[u] = 0.f; if (64 * u < cols) v[u] = row[min(64 * u + lane, cols - 1)]; }
}
template <int N>
__device__ __forceinline__ void place_row(lptr to, bool ok, int cols, int end, int lane, const float (&v)[N]) {
#pragma unroll
    for (int u = 0; u < N; u++) if (64 * u + lane < end) to[64 * u + lane] = ok && 64 * u + lane < cols ? v[u] : 0.f;
}
template <int R>
__device__ __forceinline__ void store_rows(lptr from, float* to, int hid, int row0, int batch, int wave, int lane) {      // a row to each wavefront, or to two or four of them, 64 columns in turn
    const int mine = R == WAVES ? wave : wave % R, part = R == WAVES ? 0 : wave / R;
    if (row0 + mine >= batch) return;
    float* const row = to + (size_t)(row0 + mine) * hid;
    for (int n = lane + 64 * part; n < hid; n += 64 * WAVES / R) row[n] = from[mine * S + n];
}
// A value handed from one workgroup to another of the same launch: one 8-byte store that carries its own tag, so that nothing has to be ordered around it. The wait is
// bounded (rlt_rocm_set_wait_limit: at most max_poll - 1 looks, with a bound of one none); a workgroup that gives up sets the fault word and goes on with zero, and the next
// launch, which has the gradients of nothing then, leaves parameters, moments, targets and ages as they were (rlt_gradient_guard).
__device__ __forceinline__ void hand_over(uint64_t* word, float value) {
    __hip_atomic_store(word, (1ull << 32) | (uint64_t)__float_as_uint(value), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int N>
__device__ __forceinline__ void take_over(uint64_t* const (&word)[N], float (&value)[N], unsigned max_poll, unsigned* fault) {
    for (unsigned tries = 0;;) {
        if (++tries >= max_poll) {
#pragma unroll
            for (int i = 0; i < N; i++) value[i] = 0.f;
            __hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        bool all = true;
        uint64_t w[N];
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = __hip_atomic_load(word[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // one trip for all of them
#pragma unroll
        for (int i = 0; i < N; i++) { all = all && (w[i] >> 32) != 0; value[i] = __uint_as_float((uint32_t)w[i]); }
        if (all) return;
        __builtin_amdgcn_s_sleep(1);
    }
}
// The copies of the weights that load_swizzled reads, made anew before every update (the optimisers change the weights between them): thread t of block (x, job) writes
// the 16 bytes of lane t % 64 of one (wavefront, chunk) pair, for the wavefronts that have units. Forward copies read 16
// consecutive bytes of a row, backward copies four values a row apart (the 16 lanes of a group read 64 consecutive bytes each time).
constexpr int PREP_JOBS = 12;
struct PrepArgs {
    const float* W[PREP_JOBS]; float* dst[PREP_JOBS]; int units[PREP_JOBS], depth[PREP_JOBS], backward[PREP_JOBS];      // W [units][depth], or for a backward copy [depth][units]
    uint64_t* clear; int n_clear;                      // words that the next launch wants zero
    uint32_t* age[3]; uint32_t* age_before;            // optimiser ages that are advanced, their values before that left in age_before (read by the optimisers' launch)
};
size_t copy_floats(int depth) { return (size_t)WAVES * ((depth + 15) >> 4) * 256; }
__global__ __launch_bounds__(256) void wide_prepare_kernel(PrepArgs P) {
    const int job = blockIdx.y, units = P.units[job], depth = P.depth[job], chunks = (depth + 15) >> 4;
    const int t = blockIdx.x * 256 + threadIdx.x;
    for (int i = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x; i < P.n_clear; i += gridDim.x * gridDim.y * 256) P.clear[i] = 0;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 3 && P.age_before) {
        uint32_t* const age = threadIdx.x == 0 ? P.age[0] : threadIdx.x == 1 ? P.age[1] : P.age[2];
        if (age) { const uint32_t before = *age; P.age_before[threadIdx.x] = before; *age = before + 1; }
    }
    if (t >= ((units + 15) >> 4) * chunks * 64) return;
    const int lane = t & 63, pair = t >> 6, w = pair / chunks, j = pair - w * chunks, c = lane & 15, g = lane >> 4;
    const int n = 16 * w + c, k = 16 * j + 4 * g;
    const float* W = P.W[job];
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    if (n < units) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (k + i < depth) v[i] = P.backward[job] ? W[(size_t)(k + i) * units + n] : W[(size_t)n * depth + k + i];
    }
    *reinterpret_cast<floatx4*>(P.dst[job] + (size_t)t * 4) = v;
}
// The copies of a launch: asked for one by one (a copy that is asked for again is shared), then made by one launch.
struct Copies {
    PrepArgs args = {}; int jobs = 0, blocks = 1; float* next;
    explicit Copies(float* memory) : next(memory) {}
    const float* copy(const float* W, int units, int depth, bool backward) {
        for (int q = 0; q < jobs; q++) if (args.W[q] == W && args.backward[q] == (int)backward) return args.dst[q];
        args.W[jobs] = W; args.dst[jobs] = next; args.units[jobs] = units; args.depth[jobs] = depth; args.backward[jobs] = backward;
        next += copy_floats(depth);
        const int b = rlt_div_up(((units + 15) >> 4) * ((depth + 15) >> 4) * 64, 256);
        if (b > blocks) blocks = b;
        return args.dst[jobs++];
    }
    void forward(WNet& N) { N.W1f = copy(N.W1, N.hid, N.in, false); N.W2f = copy(N.W2, N.hid, N.hid, false); }
    void backward(WNet& N) { N.W2b = copy(N.W2, N.hid, N.hid, true); }
    int launch(rlt_rocm_device* device) {
        hipLaunchKernelGGL(wide_prepare_kernel, dim3(blocks, jobs), dim3(256), 0, device->stream, args);
        return rlt_launch_status(device);
    }
};
constexpr size_t MAX_COPY_FLOATS = (size_t)WAVES * (MAX_H / 16) * 256, MAX_W1_COPY_FLOATS = (size_t)WAVES * (MAX_D / 16) * 256;

// EVERY: all networks have more than 240 units
template <int MODE, int ACT_H, int NT1C, bool EVERY, int R>
__global__ __launch_bounds__(THREADS) void sac_wide_kernel(WideArgs A) {
    constexpr int FORM = EVERY ? FORM_EVERY : FORM_ANY;
    constexpr bool CRITIC = MODE == MODE_CRITIC || MODE == MODE_TD3_CRITIC, TD3 = MODE == MODE_TD3_CRITIC || MODE == MODE_TD3_ACTOR;
    extern __shared__ __attribute__((aligned(16))) float lds_wide[];
    const int G = A.groups;
    const int place = A.by_xcd ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
    if (place >= A.roles * G) return;
    const int role = place / G, gi = place - role * G;
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool scalar_wave = wave == 0;
    const int OBS = A.obs, ACT = A.act, D = OBS + ACT, B = A.batch;
    const lptr xa = (lptr)lds_wide, h1 = xa + ROWS * SXS, h2 = h1 + ROWS * S, ta = h2 + ROWS * S, tb = ta + ROWS * S,
               d3 = tb + ROWS * S, d3c = d3 + ROWS * D3S, da = d3c + ROWS * D3S, yp = da + 2 * ROWS * D3S, misc = yp + WAVES * YP;
    const int row0 = gi * R, row_end = min(B, row0 + R);      // the tile's rows (with eight, the other eight of the sixteen that the narrow products run over belong to nobody)
    const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
    uint64_t* const exchange = A.exchange + (size_t)gi * EXCHANGE;
    const bool row_ok = row0 + c < row_end;
    // critic update: target roles [set][target critic] first, then a role per trained critic; actor update: critic 1's role (SAC), then the role that goes on with the actor
    const int n_target_roles = CRITIC ? 2 * (TD3 ? A.n_critics : 1) : 0;
    const bool target_role = CRITIC && role < n_target_roles;
    const int set = target_role ? role >> 1 : 0;

    RLT_TICK(0);
    // the input rows: next rows for the target roles, else the current ones. The actor reads the observation columns, zero beyond them until the sample is in place: what the
    // batch holds there meets zero weights in the actor's last chunk, and must not be a NaN or an infinity
    float in_row[3];
    const bool trained_role = CRITIC && !target_role;
    request_row(A.batch_base + (target_role ? (size_t)B * D : 0) + (size_t)min(row0 + wave, row_end - 1) * D, trained_role ? D : OBS, lane, in_row);
    if (trained_role) {
        // ---- a trained critic
        const int y = role - n_target_roles;
        const WNet trained = y ? A.critic[1] : A.critic[0];      // by value: an index into the kernel's argument would keep all of it in private memory
        const Trained T = y ? A.trained[1] : A.trained[0];
        const int HID = trained.hid, tiles = (HID + 15) >> 4;
        Operands<NT1C> W;
        load_operands<NT1C, FORM>(trained, wave, c, g, W);
        place_row(xa + wave * SXS, row0 + wave < row_end, D, SXS, lane, in_row);
        float reward[4] = {0.f, 0.f, 0.f, 0.f}, alpha = 0.f, b3 = 0.f;
        bool terminated[4] = {false, false, false, false};
        if (scalar_wave) {
            b3 = trained.b3[0];
            if (!TD3) alpha = expf(*A.log_alpha);
#pragma unroll
            for (int v = 0; v < 4; v++) { const int row = min(row0 + 4 * g + v, B - 1); reward[v] = A.rewards[row]; terminated[v] = A.terminated[row] != 0; }
        }
        rlt_lds_barrier();      // the input rows are in place
        RLT_TICK(1);
        forward3<R, ACT_H, NT1C, false, true, false, FORM>(trained, W, trained, xa, SXS, h1, h2, yp, nullptr, wave, c, g);
        RLT_TICK(2);
        BackOperands K;
        load_back_operands<R, FORM>(trained, wave, c, g, K);      // on their way while the targets' values are waited for
        store_rows<R>(h1, T.h1, HID, row0, row_end, wave, lane);
        store_rows<R>(h2, T.h2, HID, row0, row_end, wave, lane);
        if (scalar_wave) {
            // TD target of rows 4 g + v (meaningful in the lanes c == 0, which hold output 0), MSE gradient at the critic's pre-activation:
            // loss weight batch * 0.5 / n with n = batch rows (no masks), times the MSE gradient's 2 / batch (rl/algorithms/sac/operations_generic.h:298-316)
            const floatx4 yc = output_tile(yp, tiles, c, g);
            // (TD3: loss weight batch / n, rl/algorithms/td3/operations_generic.h:200-212)
            const float loss_weight = TD3 ? (float)B / (float)B : (1.0f / (float)B) * ((float)B * 0.5f);
            const float constant = 2.0f / (float)B * loss_weight;
            uint64_t* const slot = exchange + (TD3 ? 2 * y : 0) * ROWS;
            uint64_t* word[TD3 ? 8 : 12];
            float value[TD3 ? 8 : 12];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                word[v] = slot + 4 * g + v; word[4 + v] = slot + ROWS + 4 * g + v;
                if (!TD3) word[(TD3 ? 0 : 8) + v] = exchange + LOG_PROB_SLOT * ROWS + 4 * g + v;
            }
            take_over(word, value, A.max_poll, A.fault);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = 4 * g + v;
                const float q_min = fminf(value[v], value[4 + v]);
                const float min_q = TD3 ? q_min : q_min - alpha * value[(TD3 ? 0 : 8) + v];
                const float future = (terminated[v] && !(TD3 && A.ignore_termination)) ? 0.0f : A.gamma * min_q;
                const float y_target = reward[v] + future;
                const bool ok = c == 0 && row0 + row < row_end;
                // (SAC's critics share their targets; TD3's are formed with each critic's own sampling noise: the last critic's stay, as after two calls)
                if (A.out_target_action_value && ok && y == (TD3 ? A.n_critics - 1 : 0)) A.out_target_action_value[row0 + row] = y_target;
                const float diff = (yc[v] + b3) - y_target;
                const float dp = ok ? diff * constant : 0.f;
                d3[row * D3S + c] = dp;
                if (row0 + row < row_end) T.d3[(size_t)(row0 + row) * MAX_OUT + c] = dp;
            }
        }
        rlt_lds_barrier();      // d_pre3 is in place
        RLT_TICK(3);
        if (wave < tiles) backward_layer3<ACT_H>(trained, K, d3, h2, ta, wave, c, g);
        rlt_lds_barrier();      // every wavefront's tile of d_pre2 is in place
        store_rows<R>(ta, T.d2, HID, row0, row_end, wave, lane);
        if (wave < tiles) backward_layer2<R, ACT_H>(trained, K, ta, h1, tb, wave, c, g);
        rlt_lds_barrier();
        store_rows<R>(tb, T.d1, HID, row0, row_end, wave, lane);
        RLT_TICK(4);
        return;
    }

    // ---- target roles and the actor update: the actor (critic update: on the next observations; actor update: on the observations)
    const int critic_index = target_role ? (role & 1) : (role == A.roles - 1 ? 0 : 1);
    const bool owner = !CRITIC && critic_index == 0;
    const bool writes = target_role ? role == 0 : owner;      // of the roles that compute the same sample, the one that stores what is asked for
    const WNet Q = CRITIC ? (critic_index ? A.target[1] : A.target[0]) : (critic_index ? A.critic[1] : A.critic[0]);
    Operands<NT1C> W;
    load_operands<NT1C, FORM>(A.actor, wave, c, g, W);      // on their way while the input rows are written
    place_row(xa + wave * SXS, row0 + wave < row_end, OBS, SXS, lane, in_row);
    float alpha = 0.f, actor_b3 = 0.f, q_b3 = 0.f;
    if (scalar_wave) {
        actor_b3 = c < A.actor.out ? A.actor.b3[c] : 0.f; q_b3 = Q.b3[0];
        if (!TD3) alpha = expf(*A.log_alpha);
    }
    // The noise of the sample's values a = g and g + 4 by wavefronts 1 and 2, the smoothing noise by 3 and 4, into LDS for the first wavefront: a draw is a few hundred instructions, and one wavefront that
    // made up to four of them kept all others waiting at the first barrier, 5.2 us after the start of TD3's critics with 8 actions, 3.9 of its actor (critics 26.2 -> 23.9 us, actor 25.8 -> 23.0, the set at
    // 256 rows 78.2 -> 72.8; SAC with one action makes a single draw: 66.3 -> 66.0)
    if (wave >= 1 && wave <= (MODE == MODE_TD3_CRITIC ? 4 : 2)) {
        const int a = g + 4 * ((wave - 1) & 1);
        float value = 0.f;
        if (a < ACT && row_ok) {
            const size_t i = (size_t)(row0 + c) * ACT + a;
            if (MODE == MODE_TD3_CRITIC && wave > 2) {
                if (A.target_noise) value = A.target_noise[i];
                else {
                    const float scaled = rlt_randn_element(A.noise_seed, A.target_noise_stream + *A.stream_offset, i) * A.target_noise_std + 0.0f;
                    value = clampf(scaled, -A.target_noise_clip, A.target_noise_clip);
                    if (writes) A.out_target_noise[i] = value;
                }
            } else {
                const float* const given = (MODE == MODE_TD3_CRITIC && set) ? A.noise_second : A.noise;
                value = given ? given[i] : rlt_randn_element(A.noise_seed, ((MODE == MODE_TD3_CRITIC && set) ? A.noise_stream_second : A.noise_stream) + *A.stream_offset, i);
                if (A.out_noise && writes) A.out_noise[i] = value;
            }
        }
        d3c[64 * (wave - 1) + lane] = value;      // (d3c is next written by the first wavefront, after it has read these)
    }
    HeadItem item[2];
    RLT_TICK(13);
    rlt_lds_barrier();      // the input rows are in place
    RLT_TICK(5);
    forward3<R, ACT_H, NT1C, true, true, false, FORM>(A.actor, W, Q, xa, SXS, h1, h2, yp, nullptr, wave, c, g);
    RLT_TICK(6);
    if (scalar_wave) {
        const floatx4 out = output_tile(yp, (A.actor.hid + 15) >> 4, c, g);
#pragma unroll
        for (int v = 0; v < 4; v++) d3[(4 * g + v) * D3S + c] = c < A.actor.out ? out[v] + actor_b3 : 0.f;
        const float noise[2] = {d3c[lane], d3c[64 + lane]}, target_noise[2] = {MODE == MODE_TD3_CRITIC ? d3c[128 + lane] : 0.f, MODE == MODE_TD3_CRITIC ? d3c[192 + lane] : 0.f};
        wave_sync();
        float log_prob = 0.f;
        if (TD3) td3_head_forward(OBS, ACT, A.sampling_std, d3, D3S, xa, SXS, noise, target_noise, CRITIC, c, g, item);
        else log_prob = head_forward(A.sas, OBS, ACT, d3, D3S, xa, SXS, noise, c, g, item);
        if (TD3) {
            if (owner && row_ok && A.out_pre_clip) {
#pragma unroll
                for (int j = 0; j < 2; j++)
                    if (g + 4 * j < ACT) A.out_pre_clip[(size_t)(row0 + c) * ACT + g + 4 * j] = item[j].sample;
            }
        } else if (g == 0 && writes) {
            if (CRITIC) hand_over(exchange + LOG_PROB_SLOT * ROWS + c, log_prob);
            if (A.out_log_probabilities && row_ok) A.out_log_probabilities[row0 + c] = log_prob;
        }
        if (!TD3 && owner && row_ok) {
#pragma unroll
            for (int j = 0; j < 2; j++)
                if (g + 4 * j < ACT) {
                    if (A.out_actions) A.out_actions[(size_t)(row0 + c) * ACT + g + 4 * j] = item[j].action;
                    if (A.out_pre_squashing) A.out_pre_squashing[(size_t)(row0 + c) * ACT + g + 4 * j] = item[j].sample;
                }
        }
    }
    rlt_lds_barrier();      // the action columns of xa are in place
    RLT_TICK(7);
    forward3<R, ACT_H, NT1C, false, NT1C <= FEW, false, FORM>(Q, W, Q, xa, SXS, ta, tb, yp, nullptr, wave, c, g);
    RLT_TICK(8);
    const int qtiles = (Q.hid + 15) >> 4;
    if (CRITIC) {
        if (scalar_wave && c == 0) {
            const floatx4 q = output_tile(yp, qtiles, c, g);
#pragma unroll
            for (int v = 0; v < 4; v++) hand_over(exchange + (2 * set + critic_index) * ROWS + 4 * g + v, q[v] + q_b3);
        }
        return;
    }

    // ---- actor update: the gradient of -value / batch with respect to the action (TD3: critic 0 only, rl/algorithms/td3/operations_generic.h:260)
    const float loss_weight = (1.0f / (float)B) * -1.0f;       // rl/algorithms/sac/operations_generic.h:437-453 with n = batch rows
    BackOperands K;
    load_back_operands<R, FORM>(Q, wave, c, g, K);
    float w1[4];
#pragma unroll
    for (int i = 0; i < 4; i++) { const int unit = 16 * wave + 4 * g + i; w1[i] = (c < ACT && unit < Q.hid) ? Q.W1[(size_t)unit * D + OBS + c] : 0.f; }
    if (scalar_wave) {
        const floatx4 out = output_tile(yp, qtiles, c, g);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (c == 0) misc[4 * g + v] = out[v] + q_b3;
            d3c[(4 * g + v) * D3S + c] = (c == 0 && row0 + 4 * g + v < row_end) ? loss_weight : 0.f;
        }
    }
    rlt_lds_barrier();
    if (wave < qtiles) backward_layer3<ACT_H>(Q, K, d3c, tb, tb, wave, c, g);
    rlt_lds_barrier();
    RLT_TICK(9);
    if (wave < qtiles) {
        backward_layer2<R, ACT_H>(Q, K, tb, ta, ta, wave, c, g);
        wave_sync();
        // d value / d action = the action columns of d_pre1 W1: this wavefront's units' share of the reduction
        floatx4 acc = zero4;
        const floatx4 a = *(lptr4)(ta + c * S + 16 * wave + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) acc = mfma16(a[i], w1[i], acc);
#pragma unroll
        for (int v = 0; v < 4; v++) yp[(wave * ROWS + 4 * g + v) * D3S + c] = acc[v];
    }
    rlt_lds_barrier();
    RLT_TICK(10);
    if (!owner) {
        if (scalar_wave) {
            const floatx4 out = output_tile(yp, qtiles, c, g);
#pragma unroll
            for (int v = 0; v < 4; v++) if (c < ACT) hand_over(exchange + ROWS + (4 * g + v) * MAX_ACT + c, out[v]);
            if (g == 0) hand_over(exchange + c, misc[c]);
        }
        return;
    }
    const WNet trained = A.actor;
    const Trained T = A.trained[0];
    const int HID = trained.hid, tiles = (HID + 15) >> 4;
    load_back_operands<R, FORM>(trained, wave, c, g, K);
    store_rows<R>(h1, T.h1, HID, row0, row_end, wave, lane);
    store_rows<R>(h2, T.h2, HID, row0, row_end, wave, lane);
    if (scalar_wave) {
        // sample_and_squash backward on the gradient of the smaller value; TD3: the td3_sampling layer's backward (zero where the sample was clamped,
        // nn/layers/td3_sampling/operations_generic.h:139-163) and the derivative of the actor's tanh output
        const floatx4 out = output_tile(yp, qtiles, c, g);
#pragma unroll
        for (int v = 0; v < 4; v++) { da[(4 * g + v) * D3S + c] = out[v]; d3[(4 * g + v) * D3S + c] = 0.f; }
        bool first = true;
        if (!TD3) {
            uint64_t* const mine = exchange + ROWS + c * MAX_ACT;
            uint64_t* const word[3] = {exchange + c, mine + min(g, ACT - 1), mine + min(g + 4, ACT - 1)};
            float value[3];
            take_over(word, value, A.max_poll, A.fault);
            first = misc[c] < value[0];
#pragma unroll
            for (int j = 0; j < 2; j++) if (g + 4 * j < ACT) da[(ROWS + c) * D3S + g + 4 * j] = value[1 + j];
        }
        wave_sync();
        const lptr dak = da + (first ? 0 : 1) * ROWS * D3S + c * D3S;
        const float alpha_over_b = alpha / (float)B;
        float entropy = 0.f;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int a = g + 4 * j;
            if (a < ACT) {
                if (TD3) {
                    const float d_mean = (item[j].sample < -1.0f || item[j].sample > 1.0f) ? 0.0f : dak[a];
                    if (row_ok) d3[c * D3S + a] = d_mean * (1.0f - item[j].mean * item[j].mean);
                    continue;
                }
                float d_mu, d_ls;
                head_backward(A.sas, item[j], dak[a], alpha_over_b, d_mu, d_ls, entropy);
                if (row_ok) { d3[c * D3S + a] = d_mu; d3[c * D3S + ACT + a] = d_ls; }
            }
        }
        entropy = groups_sum(entropy);
        // d log_alpha: sum over the rows of alpha (entropy - target entropy), divided by the batch size by the optimiser
        const float per_row = (g == 0 && row_ok) ? alpha * (entropy - A.sas.target_entropy) : 0.f;
        const float tile_sum = row16_sum(per_row);
        wave_sync();
#pragma unroll
        for (int v = 0; v < 4; v++) if (row0 + 4 * g + v < row_end) T.d3[(size_t)(row0 + 4 * g + v) * MAX_OUT + c] = d3[(4 * g + v) * D3S + c];
        if (lane == 0 && A.extra) A.extra[gi] = tile_sum;
    }
    rlt_lds_barrier();      // d_pre3 is in place
    RLT_TICK(11);
    if (wave < tiles) backward_layer3<ACT_H>(trained, K, d3, h2, ta, wave, c, g);
    rlt_lds_barrier();      // every wavefront's tile of d_pre2 is in place
    store_rows<R>(ta, T.d2, HID, row0, row_end, wave, lane);
    if (wave < tiles) backward_layer2<R, ACT_H>(trained, K, ta, h1, tb, wave, c, g);
    rlt_lds_barrier();
    store_rows<R>(tb, T.d1, HID, row0, row_end, wave, lane);
    RLT_TICK(12);
}

constexpr size_t LDS_FLOATS = (size_t)ROWS * SXS + 4 * ROWS * S + 4 * ROWS * D3S + WAVES * YP + MISC, DIRECT_LDS_FLOATS = LDS_FLOATS + WAVES * W1_STAGE;

// ---- Forward and backward pass of one three-layer network over a few thousand rows at most, on the same machinery (nn_models/mlp/operations_generic.h:103-204: forward, the
// loss gradient given or formed from a target as the MSE's, backward with weight gradients): a workgroup takes 16, 8 or 4 rows through the three layers and back and leaves
// activations and pre-activation gradients in memory; the weight gradients over the whole batch are the next launch (batch_gradient.hip). Narrow networks, whose gradients are few
// tiles there and few bytes here, go the other way (BLOCKS): a workgroup forms its sixteen rows' weight gradients out of LDS and leaves them as a block, and the next launch adds the
// blocks up (which way is taken: sum_blocks()). Where a batch is too small to fill the chip with the 64-row tiles of the one-pass kernel for large batches (mlp_fused.hip: 4,096 rows are 64 tiles for 256
// compute units, and a tile takes its 74 us whatever the batch), sixteen-row tiles are a launch of 256 workgroups.
struct MlpWideArgs {
    WNet net;
    const float* x; int ldx; float* y; int ldy;
    float* copy_x;                             // [batch x in], or NULL: the input rows once more, where y lies in their memory and the weight gradients are formed by the next launch
    const float* d_output; int ldd; const float* target; int ldt; float mse_scale;
    int batch;
    float* partial; int count;                 // BLOCKS: [workgroups][count] blocks dW1 | db1 | dW2 | db2 | dW3 | db3
    Trained kept;                              // MLP_FORWARD_BACKWARD: hidden activations; both: the gradients at the hidden pre-activations (and, unless the caller's array serves, the last)
    const float* out1; const float* out2;      // MLP_BACKWARD: the outputs of layers 1 and 2 that a forward() left in memory, [batch x hid] each; d_output is then the gradient at the last pre-activations
    float* keep_pre[3]; float* keep_out[3]; int act3;      // MLP_FORWARD: every layer's pre-activations and outputs as forward() keeps them (each may be NULL); the last layer's activation
};
enum { MLP_FORWARD_BACKWARD = 0, MLP_BACKWARD = 1, MLP_FORWARD = 2 };
enum { MLP_ANY = 0, MLP_BLOCKS = 1, MLP_EVERY = 2, MLP_DIRECT = 3 };      // MLP_BLOCKS: weight gradients as blocks; MLP_EVERY: more than 240 units, every wavefront has some; MLP_DIRECT: FORM_DIRECT
template <int ACT_H, int NT1C, int PASS, int KIND, int R>
__global__ __launch_bounds__(THREADS) void mlp_wide_kernel(MlpWideArgs A) {
    constexpr bool BACKWARD_ONLY = PASS == MLP_BACKWARD, BLOCKS = KIND == MLP_BLOCKS;
    constexpr int FORM = KIND == MLP_DIRECT ? FORM_DIRECT : KIND == MLP_EVERY ? FORM_EVERY : FORM_ANY;
    constexpr bool EVERY = FORM != FORM_ANY;
    extern __shared__ __attribute__((aligned(16))) float lds_wide[];
    static_assert(R == 16 || !BLOCKS, "blocks are formed over sixteen rows");
    const int gi = blockIdx.x;
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const lptr xa = (lptr)lds_wide, h1 = xa + ROWS * SXS, h2 = h1 + ROWS * S, ta = h2 + ROWS * S, tb = ta + ROWS * S, d3 = tb + ROWS * S, yp = d3 + 4 * ROWS * D3S, stage = yp + WAVES * YP + MISC + wave * W1_STAGE;
    const WNet N = A.net;
    const int B = A.batch, IN = N.in, HID = N.hid, OUT = N.out, tiles = (HID + 15) >> 4, row0 = gi * R, row_end = min(B, row0 + R);
    const bool on = wave < tiles;
    const bool my_row = row0 + wave < row_end;
    const size_t row_at = min(row0 + wave, row_end - 1);
    Operands<NT1C> W;
    BackOperands K;
    float b3 = 0.f, s3 = 0.f, given[4] = {0.f, 0.f, 0.f, 0.f};      // given: this lane's elements of the gradient at the output, or of the target it is formed from
    auto request_given = [&] {
        const float* const from = A.target ? A.target : A.d_output;
        const int ld = A.target ? A.ldt : A.ldd;
#pragma unroll
        for (int v = 0; v < 4; v++) given[v] = from[(size_t)min(row0 + 4 * g + v, B - 1) * ld + min(c, OUT - 1)];
    };
    if (BACKWARD_ONLY || (PASS == MLP_FORWARD_BACKWARD && !EVERY)) request_given();
    if (BACKWARD_ONLY) {
        // the hidden activations come back from memory (zero beyond the batch and beyond the width, up to the multiple of 16 that the tiles run to)
        float v1[4], v2[4], vx[3];
        if (BLOCKS) request_row(A.x + row_at * A.ldx, IN, lane, vx);
        request_row(A.out1 + row_at * HID, HID, lane, v1);
        request_row(A.out2 + row_at * HID, HID, lane, v2);
        if (on) load_back_operands<R, FORM>(N, wave, c, g, K);
        place_row(h1 + wave * S, my_row, HID, 16 * tiles, lane, v1);
        place_row(h2 + wave * S, my_row, HID, 16 * tiles, lane, v2);
        if (BLOCKS) place_row(xa + wave * SXS, my_row, IN, SXS, lane, vx);
        if (wave == 0) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float d = c < OUT && row0 + 4 * g + v < row_end ? given[v] : 0.f;
                d3[(4 * g + v) * D3S + c] = d;
                s3 += d;
            }
        }
    } else {
        float v[3];
        request_row(A.x + row_at * A.ldx, IN, lane, v);
        load_operands<NT1C, FORM>(N, wave, c, g, W);
        b3 = N.b3[min(c, OUT - 1)];
        place_row(xa + wave * SXS, my_row, IN, SXS, lane, v);
        if (PASS == MLP_FORWARD_BACKWARD && !BLOCKS && A.copy_x && my_row) {
#pragma unroll
            for (int u = 0; u < 3; u++) if (64 * u + lane < IN) A.copy_x[row_at * IN + 64 * u + lane] = v[u];
        }
    }
    rlt_lds_barrier();
    if (PASS == MLP_FORWARD) {
        const KeepArgs keep = {{A.keep_pre[0], A.keep_pre[1]}, {A.keep_out[0], A.keep_out[1]}, row0, row_end};
        forward3<R, ACT_H, NT1C, false, true, true, FORM>(N, W, N, xa, SXS, h1, h2, yp, stage, wave, c, g, &keep);
        if (wave == 0) {
            const floatx4 out = output_tile(yp, tiles, c, g);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + 4 * g + v;
                if (c < OUT && row < row_end) {
                    const float pre = out[v] + b3;
                    if (A.keep_pre[2]) A.keep_pre[2][(size_t)row * OUT + c] = pre;
                    const float o = rlt_act(pre, A.act3);
                    if (A.keep_out[2]) A.keep_out[2][(size_t)row * OUT + c] = o;
                    if (A.y) A.y[(size_t)row * A.ldy + c] = o;
                }
            }
        }
        return;
    }
    if (PASS == MLP_FORWARD_BACKWARD) {
        forward3<R, ACT_H, NT1C, false, true, false, FORM, BLOCKS>(N, W, N, xa, SXS, h1, h2, yp, stage, wave, c, g, nullptr, B - row0);
        if (EVERY) request_given();      // (all of W fills the registers until here)
        load_back_operands<R, FORM>(N, wave, c, g, K);
        if (!BLOCKS) {
            store_rows<R>(h1, A.kept.h1, HID, row0, row_end, wave, lane);
            store_rows<R>(h2, A.kept.h2, HID, row0, row_end, wave, lane);
        }
    }
    if (!BACKWARD_ONLY && wave == 0) {
        // lane (c, g): output column c of rows 4 g + v; the gradient at the output (the last layer has no activation): given, or the MSE's against the target
        const floatx4 out = output_tile(yp, tiles, c, g);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = row0 + 4 * g + v;
            const bool ok = c < OUT && row < row_end;
            const float yv = out[v] + b3;
            if (ok && A.y) A.y[(size_t)row * A.ldy + c] = yv;
            float d = 0.f;
            if (ok) d = A.target ? (yv - given[v]) * A.mse_scale : given[v];
            d3[(4 * g + v) * D3S + c] = d;
            s3 += d;
            if (!BLOCKS && row < row_end) A.kept.d3[(size_t)row * MAX_OUT + c] = d;
        }
    }
    if (!BACKWARD_ONLY) rlt_lds_barrier();      // d_pre3 is in place (the backward pass alone: with the activations)
    const float s2 = on ? backward_layer3<ACT_H, BLOCKS>(N, K, d3, h2, ta, wave, c, g, B - row0) : 0.f;
    if (BLOCKS) {
        float* const block = A.partial + (size_t)gi * A.count;
        float* const to_b1 = block + HID * IN; float* const to_w2 = to_b1 + HID; float* const to_b2 = to_w2 + HID * HID; float* const to_w3 = to_b2 + HID; float* const to_b3 = to_w3 + OUT * HID;
        const int n = 16 * wave + c, spare = WAVES - tiles;
        // Wavefronts without units (half of them and more up to width 128) form dW3 and dW2 while the others go on with the backward pass and dW1; without enough of them each does its units' rows
        const bool spread = spare >= tiles;
        auto last_layer = [&](int u) {      // dW3: columns 16 u ...
            floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < ROWS / 4; ks++) acc = mfma16(d3[(4 * ks + g) * D3S + c], h2[(4 * ks + g) * S + 16 * u + c], acc);
#pragma unroll
            for (int v = 0; v < 4; v++) if (4 * g + v < OUT && 16 * u + c < HID) to_w3[(4 * g + v) * HID + 16 * u + c] = acc[v];
        };
        if (spread ? !on && wave - tiles < tiles : on) last_layer(spread ? wave - tiles : wave);
        rlt_lds_barrier();      // every wavefront's tile of d_pre2 is in place
        if (on) {
            const float s1 = backward_layer2<R, ACT_H, FORM, BLOCKS>(N, K, ta, h1, tb, wave, c, g, B - row0);
            wave_sync();            // dW1's rows are this wavefront's own tile of d_pre1
#pragma unroll 2
            for (int nt = 0; nt < (IN + 15) >> 4; nt++) gradient_tile(tb, wave, xa, SXS, nt, HID, IN, block, c, g);
            const float b1 = groups_sum(s1), b2 = groups_sum(s2);
            if (g == 0 && n < HID) { to_b1[n] = b1; to_b2[n] = b2; }
        }
        if (!spread && on) {
#pragma unroll 4
            for (int nt = 0; nt < tiles; nt++) gradient_tile(ta, wave, h1, S, nt, HID, HID, to_w2, c, g);
        } else if (spread && !on) {
#pragma unroll 2
            for (int p = wave - tiles; p < tiles * tiles; p += spare) gradient_tile(ta, p / tiles, h1, S, p % tiles, HID, HID, to_w2, c, g);
        }
        if (wave == 0) {
            s3 = groups_sum(s3);
            if (g == 0 && c < OUT) to_b3[c] = s3;
        }
        return;
    }
    rlt_lds_barrier();      // every wavefront's tile of d_pre2 is in place
    store_rows<R>(ta, A.kept.d2, HID, row0, row_end, wave, lane);
    if (on) backward_layer2<R, ACT_H, FORM>(N, K, ta, h1, tb, wave, c, g);
    rlt_lds_barrier();
    store_rows<R>(tb, A.kept.d1, HID, row0, row_end, wave, lane);
}
// gradient[e] += the sum over the workgroups' blocks of element e: a workgroup takes 64 elements, its wavefronts a quarter of the blocks each, sixteen blocks' loads in flight
struct BlockSum { const float* partial; int blocks, count, total; float* gradient[6]; int end[6]; };
__global__ __launch_bounds__(256) void block_sum_kernel(BlockSum R) {
    __shared__ float quarter[4][64];
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6, e = blockIdx.x * 64 + lane, per = (R.blocks + 3) / 4, end = min(R.blocks, (q + 1) * per);
    const float* from = R.partial + min(e, R.total - 1);
    float sum = 0.f;
    for (int b0 = q * per; b0 < end; b0 += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = from[(size_t)min(b0 + u, end - 1) * R.count];
#pragma unroll
        for (int u = 0; u < 16; u++) sum += b0 + u < end ? v[u] : 0.f;
    }
    quarter[q][lane] = sum;
    __syncthreads();
    if (q != 0 || e >= R.total) return;
    int k = 0, begin = 0;
#pragma unroll
    for (int i = 0; i < 5; i++) if (e >= R.end[i]) { k = i + 1; begin = R.end[i]; }
    float* const to = k == 0 ? R.gradient[0] : k == 1 ? R.gradient[1] : k == 2 ? R.gradient[2] : k == 3 ? R.gradient[3] : k == 4 ? R.gradient[4] : R.gradient[5];
    to[e - begin] += (quarter[0][lane] + quarter[1][lane]) + (quarter[2][lane] + quarter[3][lane]);
}
// Whether the workgroups' blocks are added up (else the weight gradients are a contraction over the whole batch of their own): where the network is narrow, and the batch not so long that
// the blocks are many bytes; the backward pass alone, which has the activations in memory already, sooner goes the other way. Blocks / contraction, us, outputs 6. Forward + backward: 17-65 at
// 256 rows 12.5 / 14.9, 4,096 16.5 / 21.2; 65-80 at 2,048 17.3 / 18.7; 17-100 at 64 14.2 / 14.5, 4,096 21.9 / 22.8; 17-112 at 4,096 23.2 / 23.3; 40-112 at 256 15.2 / 15.9, 2,048 19.7 / 19.3;
// 17-128 at 128 15.9 / 15.0, 256 16.0 / 16.0, 512 16.6 / 18.1, 1,000 17.9 / 17.9; 60-128 at 512 17.9 / 18.4, 768 18.8 / 18.0; 20-144 at 512 20.5 / 21.0, 768 21.3 / 20.5; 17-160 at 512
// 21.7 / 21.5. Backward alone: 17-65 at 4,096 14.0 / 17.1; 65-80 at 2,048 13.9 / 14.3; 17-100 at 64 11.6 / 11.2, 256 11.8 / 12.3, 2,048 15.1 / 14.8, 4,096 19.3 / 18.0; 17-112 at 1,000
// 13.3 / 13.3, 2,048 15.7 / 15.0; 40-112 at 1,000 13.9 / 13.3; 17-128 at 300 13.2 / 13.1; 128-64 at 1,000 11.6 / 11.9, 4,096 17.6 / 15.9.
bool sum_blocks(int hid, int in, int batch, bool backward_only) {
    const int products = hid * (hid + in);
    const int64_t work = (int64_t)products * batch;
    if (backward_only) return products <= 15000 && work <= 24000000 && (batch > 128 || products <= 8192);
    return products <= 15000 ? work <= 62914560 : products <= 24576 && batch > 256 && work <= 13000000;
}

bool hidden_ok(int a) { return a == RLT_ACT_RELU || a == RLT_ACT_TANH || a == RLT_ACT_FAST_TANH || a == RLT_ACT_SIGMOID; }
bool net_ok(const rlt_dense_layer* L, int n, int in, int out, int& hid, int last_activation = RLT_ACT_IDENTITY) {
    if (!L || n != 3) return false;
    for (int l = 0; l < 3; l++) if (!L[l].weights || !L[l].biases) return false;
    if (hid == 0) hid = L[0].out_dim;
    return hid >= 1 && hid <= MAX_H && L[0].in_dim == in && L[0].out_dim == hid && L[1].in_dim == hid && L[1].out_dim == hid && L[2].in_dim == hid && L[2].out_dim == out &&
           L[0].activation == L[1].activation && hidden_ok(L[0].activation) && L[2].activation == last_activation;
}
bool aligned16(const float* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
WNet net_of(const rlt_dense_layer* L) {
    const int in = L[0].in_dim, hid = L[0].out_dim;
    return {L[0].weights, L[0].biases, L[1].weights, L[1].biases, L[2].weights, L[2].biases, in, hid, L[2].out_dim, L[0].activation,
            hid % 4 == 0 && aligned16(L[2].weights)};
}
// the network's six gradient buffers as segments [dW1, db1, dW2, db2, dW3, db3], and the parameters that they belong to
struct Segments { float* gradient[6]; float* parameter[6]; uint32_t size[6]; };
Segments segments_of(const rlt_dense_layer* L) {
    const uint32_t hid = L[0].out_dim;
    return {{L[0].d_weights, L[0].d_biases, L[1].d_weights, L[1].d_biases, L[2].d_weights, L[2].d_biases},
            {L[0].weights, L[0].biases, L[1].weights, L[1].biases, L[2].weights, L[2].biases},
            {hid * L[0].in_dim, hid, hid * hid, hid, L[2].out_dim * hid, (uint32_t)L[2].out_dim}};
}

struct Optimiser {
    const rlt_dense_layer* trained; const rlt_adam_tensor* tensors; int n_tensors; const rlt_adam_parameters* parameters; uint32_t* age;
    const rlt_adam_tensor* second; const rlt_adam_parameters* second_parameters; uint32_t* second_age; float second_scale;
    const rlt_dense_layer* soft_target;
};

// What the gradients' launch needs of a trained network and its optimiser. A tensor of the optimiser may span several segments where those follow each other in memory;
// false unless the tensors cover the six segments exactly. The soft update of the target rides along where the tensors' parameters are the network's own.
bool describe(const Optimiser& O, rlt_gradient_net& N, bool* targets_fused) {
    const Segments s = segments_of(O.trained);
    if (!O.tensors || O.n_tensors < 1 || O.n_tensors > RLT_TAIL_TENSORS) return false;
    const Segments soft = O.soft_target ? segments_of(O.soft_target) : Segments{};
    uint32_t covered = 0;
    *targets_fused = O.soft_target != nullptr;
    for (int i = 0; i < O.n_tensors; i++) {
        const rlt_adam_tensor& T = O.tensors[i];
        if (T.polyak_target || !T.parameters || !T.gradient || !T.first_moment || !T.second_moment) return false;
        int k = 0;
        while (k < 6 && s.gradient[k] != T.gradient) k++;
        uint32_t at = 0;
        for (; k < 6 && at < T.count && s.gradient[k] == T.gradient + at; k++) {
            if (covered & (1u << k)) return false;
            covered |= 1u << k;
            N.gradient[k] = s.gradient[k]; N.parameter[k] = T.parameters + at; N.first_moment[k] = T.first_moment + at; N.second_moment[k] = T.second_moment + at; N.flags[k] = T.flags;
            N.target[k] = soft.parameter[k];
            if (N.parameter[k] != s.parameter[k]) *targets_fused = false;
            at += s.size[k];
        }
        if (at != T.count) return false;
    }
    N.in = O.trained[0].in_dim; N.hid = O.trained[0].out_dim; N.out = O.trained[2].out_dim;
    N.step = 1; N.adam = *O.parameters;
    return covered == 63u;
}
// room for a batch's activations and gradients of a trained network; floats
size_t trained_floats(int hid, int batch) { return (((size_t)hid * batch * 4 + (size_t)MAX_OUT * batch) + 63) & ~(size_t)63; }
Trained place_trained(float* base, int hid, int batch) {
    const size_t n = (size_t)hid * batch;
    return {base, base + n, base + 2 * n, base + 3 * n, base + 4 * n};
}
void set_rows(rlt_gradient_net& N, const Trained& T, const float* x, int ldx) { N.x = x; N.ldx = ldx; N.h1 = T.h1; N.h2 = T.h2; N.d1 = T.d1; N.d2 = T.d2; N.d3 = T.d3; N.ld3 = MAX_OUT; }

// Rows of a workgroup's tile: four or eight while every tile and role then has a compute unit of its own, sixteen beyond; four only where every network has more than 240 units (MLP passes with any
// activation function, SAC and TD3 updates with relu; the other instances were not built). Fewer rows are fewer
// cycles of the matrix pipeline per layer (sixteen 8,192 at width 256, eight 4,096, four 2,048) on more compute units; the same weights travel to each. In us, sixteen / eight / four
// rows, 256 rows of the batch, width 256: forward + backward, Adam and the gradients' clearing 35.1 / 32.2 / 29.0, SAC's update set 85.7 / 74.0 / 66.4, TD3's 90.7 / 80.9 / 77.9
// (its critics' six roles take eight rows). Sixteen rows everywhere / this rule: forward + backward of 17 inputs, width 256, 512 rows 29.0 / 23.2, 1,024 32.5 / 27.2, 2,048 (eight) 38.3 / 34.9; width 240
// (eight) at 64, 256, 2,048 rows 25.0 / 21.9, 26.3 / 22.7, 39.1 / 36.0; 192 21.1 / 19.3 at 256, 27.9 / 26.2 at 2,048; 128 16.9 / 16.4 and 21.4 / 21.3. SAC's set, width 256, 512 rows 92.0 / 76.2, 1,024 (critics
// sixteen, actor eight) 104.2 / 97.8; fast_tanh (eight) at 256 88.6 / 79.3; width 192 67.8 / 62.5, 128 54.9 / 52.3, 80 50.9 / 49.8 at 256. TD3's, 256 wide, 512 rows 94.3 / 85.3; 80 wide, 256 rows 51.8 / 51.0. Four and eight rows leave the same bits, sixteen others: a critic trained by a call of its own takes sixteen where both in one call do
// (roles_of_both), as the two ways leave the same bits.
int tile_rows(const rlt_rocm_device* device, int batch, int roles, int roles_of_both, bool four) {
    const int most = device->compute_units < 256 ? device->compute_units : 256;
    return rlt_div_up(batch, 8) * roles_of_both > most ? ROWS : four && rlt_div_up(batch, 4) * roles <= most ? 4 : 8;
}
template <int MODE>
int launch_wide(rlt_rocm_device* device, WideArgs& a, const Optimiser* opts, int n_opts, float polyak, bool* targets_done) {
    rlt_gradient_net net[2] = {};
    bool fused[2] = {false, false};
    for (int k = 0; k < n_opts; k++) {      // the agent's Adam tensors are not its networks' gradient buffers: the caller takes the per-operation path
        if (!describe(opts[k], net[k], &fused[k])) return RLT_E_UNSUPPORTED;
        if (opts[k].second && (opts[k].second->polyak_target || !opts[k].second->parameters || !opts[k].second->gradient || !opts[k].second->first_moment || !opts[k].second->second_moment)) return RLT_E_UNSUPPORTED;
    }
    const bool fuse_targets = targets_done && n_opts == 2 && fused[0] && fused[1];
    if (targets_done) *targets_done = fuse_targets;
    if (!fuse_targets) for (int k = 0; k < n_opts; k++) for (int q = 0; q < 6; q++) net[k].target[q] = nullptr;
    constexpr bool CRITIC_UPDATE = MODE == MODE_CRITIC || MODE == MODE_TD3_CRITIC;
    a.n_critics = n_opts;
    a.roles = MODE == MODE_CRITIC ? 2 + n_opts : MODE == MODE_TD3_CRITIC ? 3 * n_opts : MODE == MODE_ACTOR ? 2 : 1;
    int act = a.actor.act_h;
    bool every = a.actor.hid > MAX_H - 16;
    for (int k = 0; k < 2; k++) {
        if (a.critic[k].act_h != act || a.target[k].act_h != act) act = -1;
        every = every && a.critic[k].hid > MAX_H - 16 && a.target[k].hid > MAX_H - 16;
    }
    const bool every_relu = every && act == RLT_ACT_RELU;      // the instances of EVERY, and with them those of four rows
    const int rows = tile_rows(device, a.batch, a.roles, MODE == MODE_CRITIC ? 4 : MODE == MODE_TD3_CRITIC ? 6 : a.roles, every_relu);
    const int groups = rlt_div_up(a.batch, rows);
    const size_t copies_floats = 5 * (MAX_COPY_FLOATS + MAX_W1_COPY_FLOATS) + 3 * MAX_COPY_FLOATS;
    const size_t trained_each = trained_floats(net[0].hid, a.batch), exchange_words = (size_t)groups * EXCHANGE, extra_floats = (size_t)(groups + 63) & ~(size_t)63,
                 partial_floats = (rlt_batch_gradients_partial_floats(net, n_opts, a.batch) + 63) & ~(size_t)63;
    void* scratch = nullptr;
    int rc = rlt_scratch(device, (copies_floats + n_opts * trained_each + extra_floats + partial_floats) * sizeof(float) + exchange_words * sizeof(uint64_t) + 256, &scratch);
    if (rc) return rc;
    float* const kept = (float*)scratch + copies_floats; float* const extra = kept + n_opts * trained_each;
    for (int k = 0; k < n_opts; k++) {
        a.trained[k] = place_trained(kept + k * trained_each, net[k].hid, a.batch);
        set_rows(net[k], a.trained[k], a.batch_base, a.obs + a.act);
    }
    a.extra = opts[0].second ? extra : nullptr;
    float* const partial = extra + extra_floats;
    a.exchange = (uint64_t*)(partial + partial_floats);
    uint32_t* const age_before = (uint32_t*)(a.exchange + exchange_words);
    for (int k = 0; k < n_opts; k++) net[k].age = age_before + k;
    a.max_poll = device->wait_limit; a.fault = device->fault;
    device->fault_armed = 1;
    {   // every network runs forward; the critics (their targets' own weights are another matter) and in the actor update the actor are also walked backwards
        Copies copies((float*)scratch);
        copies.forward(a.actor);
        for (int k = 0; k < 2; k++) { copies.forward(a.critic[k]); copies.backward(a.critic[k]); if (CRITIC_UPDATE) copies.forward(a.target[k]); }
        if (!CRITIC_UPDATE) copies.backward(a.actor);
        copies.args.clear = a.exchange; copies.args.n_clear = (int)exchange_words;
        for (int k = 0; k < n_opts; k++) copies.args.age[k] = opts[k].age;
        copies.args.age[2] = opts[0].second ? opts[0].second_age : nullptr; copies.args.age_before = age_before;
        if ((rc = copies.launch(device))) return rc;
    }
    a.stream_offset = device->stream_offset;
    a.groups = groups;
    // A workgroup waits for others of its tile only, and all are resident where there is a compute unit for each: then a role's workgroups are kept on neighbouring
    // positions of the XCDs' round (workgroup b runs on XCD b % 8), so that few XCDs read a network's weights. Larger grids are numbered role by role, so that whoever
    // is waited for was dispatched before whoever waits.
    a.by_xcd = device->update_one_xcd && device->xcd_stride == 8 && a.roles * groups <= device->compute_units;
    const size_t lds_bytes = LDS_FLOATS * sizeof(float);
    const dim3 grid(a.by_xcd ? 8 * rlt_div_up(a.roles * groups, 8) : a.roles * groups);
#define RLT_LAUNCH_WIDE_ROWS(ACT, NT, EVERY, R)                                                                                                           \
    do {                                                                                                                                                  \
        RLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(sac_wide_kernel<MODE, ACT, NT, EVERY, R>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes)); \
        hipLaunchKernelGGL((sac_wide_kernel<MODE, ACT, NT, EVERY, R>), grid, dim3(THREADS), lds_bytes, device->stream, a);                                \
    } while (0)
#define RLT_LAUNCH_WIDE(ACT, NT) do { if (rows == 8) RLT_LAUNCH_WIDE_ROWS(ACT, NT, false, 8); else RLT_LAUNCH_WIDE_ROWS(ACT, NT, false, ROWS); } while (0)
#define RLT_LAUNCH_WIDE_EVERY(ACT, NT) do { if (rows == 4) RLT_LAUNCH_WIDE_ROWS(ACT, NT, true, 4); else if (rows == 8) RLT_LAUNCH_WIDE_ROWS(ACT, NT, true, 8); else RLT_LAUNCH_WIDE_ROWS(ACT, NT, true, ROWS); } while (0)
#define RLT_LAUNCH_WIDE_ACT(NT)                                                                                                                           \
    do {                                                                                                                                                  \
        if (every_relu) RLT_LAUNCH_WIDE_EVERY(RLT_ACT_RELU, NT);                                                                                          \
        else if (act == RLT_ACT_RELU) RLT_LAUNCH_WIDE(RLT_ACT_RELU, NT);                                                                                  \
        else if (act == RLT_ACT_FAST_TANH) RLT_LAUNCH_WIDE(RLT_ACT_FAST_TANH, NT); else RLT_LAUNCH_WIDE(-1, NT);                                          \
    } while (0)
    // the first layer's chunks that the code is unrolled for: up to 64 inputs they leave registers for all of a pass's weights at once
    if (a.obs + a.act <= 32) RLT_LAUNCH_WIDE_ACT(2); else if (a.obs + a.act <= 64) RLT_LAUNCH_WIDE_ACT(4); else RLT_LAUNCH_WIDE_ACT(MAX_D / 16);
#undef RLT_LAUNCH_WIDE_ACT
#undef RLT_LAUNCH_WIDE
#undef RLT_LAUNCH_WIDE_EVERY
#undef RLT_LAUNCH_WIDE_ROWS
    if ((rc = rlt_launch_status(device))) return rc;
    const rlt_gradient_guard guard = {device->fault, {opts[0].age, n_opts > 1 ? opts[1].age : nullptr, opts[0].second ? opts[0].second_age : nullptr}, age_before};
    if (opts[0].second) {
        const rlt_gradient_scalar scalar = {a.extra, groups, opts[0].second_scale, *opts[0].second, *opts[0].second_parameters, age_before + 2};
        return rlt_batch_gradients(device, net, n_opts, a.batch, polyak, &scalar, partial, &guard);
    }
    return rlt_batch_gradients(device, net, n_opts, a.batch, polyak, nullptr, partial, &guard);
}

void set_noise(WideArgs& a, const rlt_update_noise& N) { a.noise = N.values; a.noise_seed = N.seed; a.noise_stream = N.stream; a.out_noise = N.values ? nullptr : N.drawn; }
void common_args(WideArgs& a, const rlt_sac_agent* A) {
    a.actor = net_of(A->actor);
    for (int k = 0; k < 2; k++) { a.critic[k] = net_of(A->critics[k]); a.target[k] = net_of(A->critics_target[k]); }
    a.batch_base = A->observations_actions_base; a.rewards = A->rewards; a.terminated = A->terminated; a.log_alpha = A->log_alpha.parameters;
    a.sas = A->sas; a.gamma = A->gamma; a.batch = A->batch; a.obs = A->observation_dim; a.act = A->action_dim;
}
}  // namespace

bool rlt_sac_wide_supported(const rlt_rocm_device* device, const rlt_sac_agent* A) {
    const int OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    if (OBS < 1 || ACT < 1 || ACT > MAX_ACT || D > MAX_D || A->batch < 1) return false;
    if (A->final_step_mask || A->next_final_step_mask || A->reset) return false;
    if (A->batch > 2048) return false;      // larger batches are the per-layer kernels' ground
    int hid_a = 0, hid_c = 0;
    if (!net_ok(A->actor, A->n_actor_layers, OBS, 2 * ACT, hid_a)) return false;
    for (int k = 0; k < 2; k++)
        if (!net_ok(A->critics[k], A->n_critic_layers, D, 1, hid_c) || !net_ok(A->critics_target[k], A->n_critic_layers, D, 1, hid_c)) return false;
    return LDS_FLOATS * sizeof(float) <= (size_t)device->lds_bytes;
}

int rlt_sac_wide_update_critics(rlt_rocm_device* device, const rlt_sac_agent* A, int first, int count, const rlt_update_noise& noise, bool update_targets) {
    if (!rlt_sac_wide_supported(device, A)) return RLT_E_UNSUPPORTED;
    RLT_REQUIRE(first >= 0 && count >= 1 && first + count <= 2 && (!update_targets || count == 2));
    for (int k = first; k < first + count; k++) for (int l = 0; l < 3; l++) RLT_REQUIRE(A->critics[k][l].d_weights && A->critics[k][l].d_biases);
    WideArgs a = {};
    common_args(a, A);
    if (count == 1) { a.critic[0] = net_of(A->critics[first]); a.critic[1] = a.critic[0]; }
    set_noise(a, noise);
    a.out_log_probabilities = A->next_log_probabilities; a.out_target_action_value = A->target_action_value;
    Optimiser O[2];
    for (int k = 0; k < count; k++)
        O[k] = {A->critics[first + k], A->critic_adam_tensors[first + k], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[first + k], nullptr, nullptr, nullptr, 0.0f,
                update_targets ? A->critics_target[first + k] : nullptr};
    bool targets_done = false;
    const int rc = launch_wide<MODE_CRITIC>(device, a, O, count, A->polyak, &targets_done);
    if (rc || !update_targets || targets_done) return rc;
    return rlt_rocm_sac_update_critic_targets(device, A);
}

int rlt_sac_wide_update_actor(rlt_rocm_device* device, const rlt_sac_agent* A, const rlt_update_noise& noise) {
    if (!rlt_sac_wide_supported(device, A)) return RLT_E_UNSUPPORTED;
    for (int l = 0; l < 3; l++) RLT_REQUIRE(A->actor[l].d_weights && A->actor[l].d_biases);
    RLT_REQUIRE(A->log_alpha.gradient);
    WideArgs a = {};
    common_args(a, A);
    set_noise(a, noise);
    a.out_log_probabilities = A->actor_log_probabilities; a.out_actions = A->actor_actions; a.out_pre_squashing = A->actor_pre_squashing;
    const Optimiser O = {A->actor, A->actor_adam_tensors, A->n_actor_adam_tensors, &A->actor_adam, A->actor_age, &A->log_alpha, &A->alpha_adam, A->alpha_age, 1.0f / (float)A->batch, nullptr};
    return launch_wide<MODE_ACTOR>(device, a, &O, 1, 0.0f, nullptr);
}

// ---- TD3: the same kernel with the td3_sampling head (rl/algorithms/td3/operations_generic.h:170-281)

bool rlt_td3_wide_supported(const rlt_rocm_device* device, const rlt_td3_agent* A) {
    const int OBS = A->observation_dim, ACT = A->action_dim, D = OBS + ACT;
    if (OBS < 1 || ACT < 1 || ACT > MAX_ACT || D > MAX_D || A->batch < 1 || A->batch > 2048) return false;
    if (A->final_step_mask || A->next_final_step_mask) return false;
    int hid_a = 0, hid_c = 0;
    if (!net_ok(A->actor, A->n_actor_layers, OBS, ACT, hid_a, RLT_ACT_TANH) || !net_ok(A->actor_target, A->n_actor_layers, OBS, ACT, hid_a, RLT_ACT_TANH)) return false;
    for (int k = 0; k < 2; k++)
        if (!net_ok(A->critics[k], A->n_critic_layers, D, 1, hid_c) || !net_ok(A->critics_target[k], A->n_critic_layers, D, 1, hid_c)) return false;
    return LDS_FLOATS * sizeof(float) <= (size_t)device->lds_bytes;
}

int rlt_td3_wide_update_critic(rlt_rocm_device* device, const rlt_td3_agent* A, int ci, const float* sampling_noise) {
    if (!rlt_td3_wide_supported(device, A)) return RLT_E_UNSUPPORTED;
    for (int l = 0; l < 3; l++) RLT_REQUIRE(A->critics[ci][l].d_weights && A->critics[ci][l].d_biases);
    RLT_REQUIRE(A->target_next_action_noise && sampling_noise);
    WideArgs a = {};
    a.actor = net_of(A->actor_target); a.critic[0] = net_of(A->critics[ci]); a.critic[1] = a.critic[0];
    for (int k = 0; k < 2; k++) a.target[k] = net_of(A->critics_target[k]);
    a.batch_base = A->observations_actions_base; a.rewards = A->rewards; a.terminated = A->terminated; a.noise = sampling_noise; a.target_noise = A->target_next_action_noise;
    a.sampling_std = A->sampling_std; a.ignore_termination = A->ignore_termination;
    a.gamma = A->gamma; a.batch = A->batch; a.obs = A->observation_dim; a.act = A->action_dim;
    a.out_target_action_value = A->target_action_value;
    const Optimiser O = {A->critics[ci], A->critic_adam_tensors[ci], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[ci], nullptr, nullptr, nullptr, 0.0f, nullptr};
    return launch_wide<MODE_TD3_CRITIC>(device, a, &O, 1, 0.0f, nullptr);
}

// both critics on the agent's batch in one launch (three roles per critic: two target chains and the trained critic), each with its own sampling noise for the target actor's td3_sampling layer:
// what rlt_td3_wide_update_critic for critic 0 and then for critic 1 leave, bit for bit
int rlt_td3_wide_update_critics(rlt_rocm_device* device, const rlt_td3_agent* A, const float* sampling_noise_first, const float* sampling_noise_second, const rlt_td3_critic_draws* draws, bool update_targets) {
    if (!rlt_td3_wide_supported(device, A)) return RLT_E_UNSUPPORTED;
    for (int k = 0; k < 2; k++) for (int l = 0; l < 3; l++) RLT_REQUIRE(A->critics[k][l].d_weights && A->critics[k][l].d_biases);
    RLT_REQUIRE(A->target_next_action_noise && (draws || (sampling_noise_first && sampling_noise_second)));
    WideArgs a = {};
    a.actor = net_of(A->actor_target);
    for (int k = 0; k < 2; k++) { a.critic[k] = net_of(A->critics[k]); a.target[k] = net_of(A->critics_target[k]); }
    a.batch_base = A->observations_actions_base; a.rewards = A->rewards; a.terminated = A->terminated;
    if (draws) {        // the three noise tensors are drawn by the kernel; the smoothing noise is left in the agent's buffer as target_action_noise leaves it
        a.noise_seed = draws->seed; a.noise_stream = draws->sampling_stream[0]; a.noise_stream_second = draws->sampling_stream[1]; a.target_noise_stream = draws->target_noise_stream;
        a.target_noise_std = draws->target_noise_std; a.target_noise_clip = draws->target_noise_clip; a.out_target_noise = A->target_next_action_noise;
    } else { a.noise = sampling_noise_first; a.noise_second = sampling_noise_second; a.target_noise = A->target_next_action_noise; }
    a.sampling_std = A->sampling_std; a.ignore_termination = A->ignore_termination;
    a.gamma = A->gamma; a.batch = A->batch; a.obs = A->observation_dim; a.act = A->action_dim;
    a.out_target_action_value = A->target_action_value;
    Optimiser O[2];
    for (int k = 0; k < 2; k++)
        O[k] = {A->critics[k], A->critic_adam_tensors[k], A->n_critic_adam_tensors, &A->critic_adam, A->critic_age[k], nullptr, nullptr, nullptr, 0.0f, update_targets ? A->critics_target[k] : nullptr};
    bool targets_done = false;      // the targets' soft update rides along in the optimisers' launch where the tensors correspond
    const int rc = launch_wide<MODE_TD3_CRITIC>(device, a, O, 2, A->critic_polyak, &targets_done);
    if (rc || !update_targets || targets_done) return rc;
    return rlt_rocm_td3_update_critic_targets(device, A);
}

int rlt_td3_wide_update_actor(rlt_rocm_device* device, const rlt_td3_agent* A, const float* sampling_noise, uint64_t seed, uint64_t stream) {
    if (!rlt_td3_wide_supported(device, A)) return RLT_E_UNSUPPORTED;
    for (int l = 0; l < 3; l++) RLT_REQUIRE(A->actor[l].d_weights && A->actor[l].d_biases);
    WideArgs a = {};
    a.actor = net_of(A->actor);
    for (int k = 0; k < 2; k++) { a.critic[k] = net_of(A->critics[0]); a.target[k] = a.critic[k]; }       // the policy gradient goes through critic 0 (:260)
    a.batch_base = A->observations_actions_base; a.noise = sampling_noise; a.noise_seed = seed; a.noise_stream = stream;      // sampling_noise NULL: drawn from (seed, stream)
    a.sampling_std = A->sampling_std;
    a.gamma = A->gamma; a.batch = A->batch; a.obs = A->observation_dim; a.act = A->action_dim;
    a.out_pre_clip = A->actor_pre_clip;
    const Optimiser O = {A->actor, A->actor_adam_tensors, A->n_actor_adam_tensors, &A->actor_adam, A->actor_age, nullptr, nullptr, nullptr, 0.0f, nullptr};
    return launch_wide<MODE_TD3_ACTOR>(device, a, &O, 1, 0.0f, nullptr);
}


// The weight copies of the calls below have a buffer of their own: forward() and evaluate() have never touched the handle's scratch buffer at these batch sizes, and callers hold
// data there across them. RLT_E_CAPTURING: not there yet, and the stream records a graph.
int rlt_mlp_wide_reserve(rlt_rocm_device* device) {
    constexpr size_t COPY_BYTES = (2 * MAX_COPY_FLOATS + MAX_W1_COPY_FLOATS) * sizeof(float);
    if (device->copy_scratch_bytes >= COPY_BYTES) return 0;
    if (device->capturing) return RLT_E_CAPTURING;
    if (device->copy_scratch) RLT_HIP(hipFree(device->copy_scratch));
    device->copy_scratch = nullptr; device->copy_scratch_bytes = 0;
    RLT_HIP(hipMalloc(&device->copy_scratch, COPY_BYTES));
    device->copy_scratch_bytes = COPY_BYTES;
    return 0;
}

// Whether rows of y lie in the memory of other rows of `in`: a tile's outputs may then be written before the tile of those rows has read them.
static bool rows_cross(const float* y, int ldy, int cols, const float* in, int ld, int in_cols, int batch) {
    if (!y || !in) return false;
    const intptr_t W = sizeof(float), apart = (intptr_t)y - (intptr_t)in, row = ld * W;
    if (apart >= (batch - 1) * row + in_cols * W || -apart >= ((intptr_t)(batch - 1) * ldy + cols) * W) return false;
    return ldy != ld || apart + cols * W > row || apart + row < in_cols * W;
}
// ---- forward + backward of a three-layer network on tiles of a few rows (see mlp_wide_kernel), or the backward pass alone from the outputs that a forward() left in
// the layers; RLT_E_UNSUPPORTED: the caller takes another path
static int mlp_wide_launch(rlt_rocm_device* device, const rlt_dense_layer* L, int n_layers, const float* x, int ldx, float* y, int ldy,
                           const float* d_output, int ldd, const float* target, int ldt, float mse_scale, int batch, int pass) {
    const bool backward_only = pass == MLP_BACKWARD, forward_only = pass == MLP_FORWARD;
    if (n_layers != 3 || batch < 1 || batch > RLT_MLP_WIDE_MAX_BATCH || L[0].in_dim < 1 || L[0].in_dim > MAX_D || L[2].out_dim < 1 || L[2].out_dim > MAX_OUT) return RLT_E_UNSUPPORTED;
    int hid = 0;
    // the backward pass alone is handed the gradient at the last pre-activations: the last layer's activation plays no part in it
    // (forward() applies the last layer's activation per element when it stores the outputs)
    if (!net_ok(L, 3, L[0].in_dim, L[2].out_dim, hid, pass == MLP_FORWARD_BACKWARD ? RLT_ACT_IDENTITY : L[2].activation)) return RLT_E_UNSUPPORTED;
    for (int l = 0; l < 3; l++) if (!forward_only && (!L[l].d_weights || !L[l].d_biases)) return RLT_E_UNSUPPORTED;
    if (backward_only && (!L[0].output || !L[1].output)) return RLT_E_UNSUPPORTED;
    if (LDS_FLOATS * sizeof(float) > (size_t)device->lds_bytes) return RLT_E_UNSUPPORTED;
    MlpWideArgs a = {};
    a.net = net_of(L);
    a.x = x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.d_output = d_output; a.ldd = ldd; a.target = target; a.ldt = ldt; a.mse_scale = mse_scale; a.batch = batch;
    a.out1 = L[0].output; a.out2 = L[1].output;
    if (forward_only) for (int l = 0; l < 3; l++) { a.keep_pre[l] = L[l].pre_activations; a.keep_out[l] = L[l].output; }
    a.act3 = L[2].activation;
    const int IN = L[0].in_dim, OUT = L[2].out_dim;
    int rc = 0;
    rlt_gradient_net net = {};
    net.in = IN; net.hid = hid; net.out = OUT;
    float* partial = nullptr;
    // (an output in the memory of the input would leave the contraction over the whole batch without its operand: the rows are kept once more)
    const bool in_place = y && (uintptr_t)y < (uintptr_t)(x + (size_t)(batch - 1) * ldx + IN) && (uintptr_t)x < (uintptr_t)(y + (size_t)(batch - 1) * ldy + OUT);
    const bool blocks = !forward_only && sum_blocks(hid, IN, batch, backward_only);
    const bool every = hid > MAX_H - 16;
    int rows = blocks ? ROWS : tile_rows(device, batch, 1, 1, every);      // (the instances of MLP_EVERY are those of four rows, MLP_BLOCKS has sixteen only)
    // one tile reads all of its rows before it writes any: a batch of at most sixteen stays one where its outputs lie in the memory of other rows' inputs
    auto crosses = [&](const float* out, int ld, int cols) {
        return rows_cross(out, ld, cols, x, ldx, IN, batch) || rows_cross(out, ld, cols, target, ldt, OUT, batch) || rows_cross(out, ld, cols, d_output, ldd, OUT, batch);
    };
    if (rows < batch && batch <= ROWS && !backward_only) {
        bool apart = !crosses(y, ldy, OUT);
        for (int l = 0; l < 3; l++) apart = apart && !crosses(a.keep_pre[l], L[l].out_dim, L[l].out_dim) && !crosses(a.keep_out[l], L[l].out_dim, L[l].out_dim);
        if (!apart) rows = ROWS;
    }
    const int groups = rlt_div_up(batch, rows);
    const int exact = hid * IN + hid + hid * hid + hid + OUT * hid + OUT;
    if (blocks) {
        void* scratch = nullptr;
        a.count = (exact + 63) & ~63;
        if ((rc = rlt_scratch(device, (size_t)groups * a.count * sizeof(float), &scratch))) return rc;
        a.partial = (float*)scratch;
    } else if (!forward_only) {
        void* scratch = nullptr;
        const size_t copy_floats = in_place ? ((size_t)batch * IN + 63) & ~(size_t)63 : 0;
        if ((rc = rlt_scratch(device, (trained_floats(hid, batch) + copy_floats + rlt_batch_gradients_partial_floats(&net, 1, batch)) * sizeof(float), &scratch))) return rc;
        a.kept = place_trained((float*)scratch, hid, batch);
        a.copy_x = in_place ? (float*)scratch + trained_floats(hid, batch) : nullptr;
        partial = (float*)scratch + trained_floats(hid, batch) + copy_floats;
        set_rows(net, a.kept, in_place ? a.copy_x : x, in_place ? IN : ldx);
    }
    // (forward + backward of 33 to 64 inputs on tiles of eight rows, whose four chunks of the first layer lie in registers beside the second's values, from the copies: 32.9 / 34.4 us at 1,500 rows of 33
    // inputs, copies / direct, 36.3 / 38.1 at 2,048 of 64)
    const bool crowded = pass == MLP_FORWARD_BACKWARD && rows == 8 && IN > 32 && IN <= 64;
    const bool direct = !blocks && !crowded && hid == MAX_H && aligned16(a.net.W2) && DIRECT_LDS_FLOATS * sizeof(float) <= (size_t)device->lds_bytes;
    // (a pass that needs no copies asks for their buffer too, unless the stream records a graph: the program may record one that does)
    if ((!direct || !device->capturing) && (rc = rlt_mlp_wide_reserve(device))) return rc;
    if (!direct) {
        Copies copies((float*)device->copy_scratch);
        if (!backward_only) copies.forward(a.net);
        if (!forward_only) copies.backward(a.net);
        if ((rc = copies.launch(device))) return rc;
    }
    const size_t lds_bytes = (direct ? DIRECT_LDS_FLOATS : LDS_FLOATS) * sizeof(float);
#define RLT_LAUNCH_MLP_WIDE_ROWS(ACT, NT, P, FORM, R)                                                                                                           \
    do {                                                                                                                                                       \
        RLT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(mlp_wide_kernel<ACT, NT, P, FORM, R>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes)); \
        hipLaunchKernelGGL((mlp_wide_kernel<ACT, NT, P, FORM, R>), dim3(groups), dim3(THREADS), lds_bytes, device->stream, a);                                 \
    } while (0)
#define RLT_LAUNCH_MLP_WIDE(ACT, NT, P, FORM)                                                                                                                   \
    do {                                                                                                                                                       \
        constexpr int FEWEST = FORM == MLP_BLOCKS ? ROWS : FORM >= MLP_EVERY ? 4 : 8;                                                                          \
        if (rows < FEWEST) return RLT_E_UNSUPPORTED;                                                                                                           \
        if (rows == 4) RLT_LAUNCH_MLP_WIDE_ROWS(ACT, NT, P, FORM, FEWEST);                                                                                     \
        else if (rows == 8) RLT_LAUNCH_MLP_WIDE_ROWS(ACT, NT, P, FORM, (FEWEST > 8 ? FEWEST : 8));                                                             \
        else RLT_LAUNCH_MLP_WIDE_ROWS(ACT, NT, P, FORM, ROWS);                                                                                                 \
    } while (0)
    const bool relu = a.net.act_h == RLT_ACT_RELU;
#define RLT_LAUNCH_MLP_WIDE_PASS(P, FORM)                                                                                                                       \
    do {                                                                                                                                                       \
        if (IN <= 32) { if (relu) RLT_LAUNCH_MLP_WIDE(RLT_ACT_RELU, 2, P, FORM); else RLT_LAUNCH_MLP_WIDE(-1, 2, P, FORM); }                                     \
        else if (IN <= 64) { if (relu) RLT_LAUNCH_MLP_WIDE(RLT_ACT_RELU, 4, P, FORM); else RLT_LAUNCH_MLP_WIDE(-1, 4, P, FORM); }                                \
        else { if (relu) RLT_LAUNCH_MLP_WIDE(RLT_ACT_RELU, MAX_D / 16, P, FORM); else RLT_LAUNCH_MLP_WIDE(-1, MAX_D / 16, P, FORM); }                            \
    } while (0)
    if (forward_only) { if (direct) RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD, MLP_DIRECT); else if (every) RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD, MLP_EVERY); else RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD, MLP_ANY); }
    else if (backward_only) { if (blocks) RLT_LAUNCH_MLP_WIDE_PASS(MLP_BACKWARD, MLP_BLOCKS); else if (direct) RLT_LAUNCH_MLP_WIDE_PASS(MLP_BACKWARD, MLP_DIRECT); else if (every) RLT_LAUNCH_MLP_WIDE_PASS(MLP_BACKWARD, MLP_EVERY); else RLT_LAUNCH_MLP_WIDE_PASS(MLP_BACKWARD, MLP_ANY); }
    else { if (blocks) RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD_BACKWARD, MLP_BLOCKS); else if (direct) RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD_BACKWARD, MLP_DIRECT); else if (every) RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD_BACKWARD, MLP_EVERY); else RLT_LAUNCH_MLP_WIDE_PASS(MLP_FORWARD_BACKWARD, MLP_ANY); }
#undef RLT_LAUNCH_MLP_WIDE_PASS
#undef RLT_LAUNCH_MLP_WIDE
#undef RLT_LAUNCH_MLP_WIDE_ROWS
    if ((rc = rlt_launch_status(device))) return rc;
    if (forward_only) return 0;
    const Segments seg = segments_of(L);
    if (blocks) {
        BlockSum R = {a.partial, groups, a.count, exact, {}, {}};
        for (int k = 0, end = 0; k < 6; k++) { R.gradient[k] = seg.gradient[k]; R.end[k] = end += (int)seg.size[k]; }
        hipLaunchKernelGGL(block_sum_kernel, dim3(rlt_div_up(exact, 64)), dim3(256), 0, device->stream, R);
        return rlt_launch_status(device);
    }
    for (int k = 0; k < 6; k++) net.gradient[k] = seg.gradient[k];
    if (backward_only) { net.h1 = L[0].output; net.h2 = L[1].output; net.d3 = d_output; net.ld3 = ldd; }
    return rlt_batch_gradients(device, &net, 1, batch, 0.0f, nullptr, partial);
}
int rlt_mlp_wide_forward_backward(rlt_rocm_device* device, const rlt_dense_layer* L, int n_layers, const float* x, int ldx, float* y, int ldy,
                                  const float* d_output, int ldd, const float* target, int ldt, float mse_scale, int batch) {
    return mlp_wide_launch(device, L, n_layers, x, ldx, y, ldy, d_output, ldd, target, ldt, mse_scale, batch, MLP_FORWARD_BACKWARD);
}
int rlt_mlp_wide_backward(rlt_rocm_device* device, const rlt_dense_layer* L, int n_layers, const float* x, int ldx, const float* d_pre_last, int ldd, int batch) {
    return mlp_wide_launch(device, L, n_layers, x, ldx, nullptr, 0, d_pre_last, ldd, nullptr, 0, 0.0f, batch, MLP_BACKWARD);
}
int rlt_mlp_wide_forward(rlt_rocm_device* device, const rlt_dense_layer* L, int n_layers, const float* x, int ldx, float* y, int ldy, int batch, bool keep) {
    if (keep) return mlp_wide_launch(device, L, n_layers, x, ldx, y, ldy, nullptr, 0, nullptr, 0, 0.0f, batch, MLP_FORWARD);
    rlt_dense_layer plain[3];      // evaluate(): nothing is kept
    if (n_layers != 3) return RLT_E_UNSUPPORTED;
    for (int l = 0; l < 3; l++) { plain[l] = L[l]; plain[l].pre_activations = nullptr; plain[l].output = nullptr; }
    return mlp_wide_launch(device, plain, n_layers, x, ldx, y, ldy, nullptr, 0, nullptr, 0, 0.0f, batch, MLP_FORWARD);
}

#ifdef RLT_WIDE_PROFILE
extern "C" int rlt_sac_wide_ticks(unsigned long long* out) { return (int)hipMemcpyFromSymbol(out, HIP_SYMBOL(rlt_wide_ticks), sizeof(unsigned long long) * 64); }
#endif
