// The product that weight gradients over a batch are made of: a tile of d^T x, rows of the batch being the reduction (used by batch_gradient.hip and seq_stack.hip).
#pragma once
#include "common.h"

namespace rlt_batch {
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int TN = 32, CHUNK = 8;      // columns of a tile; steps of four rows whose operands are requested together

__device__ __forceinline__ float groups_sum(float v) { asm volatile("" : "+v"(v)); v += __shfl_xor(v, 16, 64); v += __shfl_xor(v, 32, 64); return v; }

// One wavefront's share of a tile of 16 MT x 32: rows [k0, k1) of the `rows` rows, on v_mfma_f32_16x16x4_f32, operands straight from memory (a chunk ahead). c[q][h][v] of
// lane (r, g) = element (16 q + 4 g + v, 16 h + r); bias[q]: the column sums of the left operand (all lanes of a column hold the same sum).
template <int MT>
__device__ __forceinline__ void tile_product(const float* a, int lda, int m_count, int m0, const float* b, int ldb, int n_count, int n0, int rows, int k0, int k1, int r, int g,
                                             floatx4 (&c)[MT][2], float (&bias)[MT]) {
    const float* pa[MT]; bool m_ok[MT];
#pragma unroll
    for (int q = 0; q < MT; q++) { const int m = m0 + 16 * q + r; m_ok[q] = m < m_count; pa[q] = a + (m_ok[q] ? m : 0); c[q][0] = c[q][1] = floatx4{0.f, 0.f, 0.f, 0.f}; bias[q] = 0.f; }
    const int na = n0 + r, nb = na + 16;
    const bool a_ok = na < n_count, b_ok = nb < n_count;
    const float* pb0 = b + (a_ok ? na : 0); const float* pb1 = b + (b_ok ? nb : 0);
    float va[MT][CHUNK], v0[CHUNK], v1[CHUNK];
    auto request = [&](int kb) {
#pragma unroll
        for (int s = 0; s < CHUNK; s++) {
            const int k = kb + 4 * s + g, kc = min(k, rows - 1);
#pragma unroll
            for (int q = 0; q < MT; q++) { va[q][s] = pa[q][(size_t)kc * lda]; if (k >= k1 || !m_ok[q]) va[q][s] = 0.f; }
            v0[s] = pb0[(size_t)kc * ldb]; v1[s] = pb1[(size_t)kc * ldb];
            if (k >= k1 || !a_ok) v0[s] = 0.f;      // both operands: zero times another share's infinity is not zero
            if (k >= k1 || !b_ok) v1[s] = 0.f;
        }
    };
    if (k0 < k1) request(k0);
    for (int kb = k0; kb < k1; kb += 4 * CHUNK) {
        float xa[MT][CHUNK], x0[CHUNK], x1[CHUNK];
#pragma unroll
        for (int s = 0; s < CHUNK; s++) {
            x0[s] = v0[s]; x1[s] = v1[s];
#pragma unroll
            for (int q = 0; q < MT; q++) xa[q][s] = va[q][s];
        }
        if (kb + 4 * CHUNK < k1) request(kb + 4 * CHUNK);
#pragma unroll
        for (int s = 0; s < CHUNK; s++)
#pragma unroll
            for (int q = 0; q < MT; q++) {
                c[q][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[q][s], x0[s], c[q][0], 0, 0, 0);
                c[q][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[q][s], x1[s], c[q][1], 0, 0, 0);
                bias[q] += xa[q][s];
            }
    }
#pragma unroll
    for (int q = 0; q < MT; q++) bias[q] = groups_sum(bias[q]);
}
// the tiles of a workgroup's wavefronts side by side in LDS, where their sum is formed
template <int WAVES, int MT>
struct Parts { float tile[WAVES][16 * MT][TN + 1]; float bias[WAVES][16 * MT]; };
template <int WAVES, int MT>
__device__ __forceinline__ void place_parts(Parts<WAVES, MT>& P, int wave, int r, int g, const floatx4 (&c)[MT][2], const float (&bias)[MT]) {
#pragma unroll
    for (int q = 0; q < MT; q++) {
#pragma unroll
        for (int v = 0; v < 4; v++) { P.tile[wave][16 * q + 4 * g + v][r] = c[q][0][v]; P.tile[wave][16 * q + 4 * g + v][16 + r] = c[q][1][v]; }
        if (g == 0) P.bias[wave][16 * q + r] = bias[q];
    }
}
}  // namespace rlt_batch
