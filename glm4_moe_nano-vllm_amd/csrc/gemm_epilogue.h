// gemm_epilogue.h — what the kernels for few rows (gemm_smallm.hip, gemm_midm.hip) do with a finished tile.
#pragma once
#include "gemm_internal.h"

// Lane (c,g4) holds, per (rt, mt), columns n..n+3 of token
// row 16*mt + c
template <int MODE, int RT, int MT>
__device__ __forceinline__ void gemm_row_epilogue(const GemmParams& p, f32x4_t (&acc)[RT][MT], int grp, int m0,
                                                  int mcnt, int ncol0, int c, int g4) {
    if (MODE == GEMM_PLAIN && p.ypart != nullptr) {
        // K-split: this workgroup's fp32 partial sums; bias and the bf16 rounding belong to the consumer
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = 16 * mt + c;
            if (row >= mcnt) continue;
            float* prow = p.ypart + (int64_t)(m0 + row) * p.N;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int n = ncol0 + 16 * rt + 4 * g4;
                if (n < p.N) *reinterpret_cast<f32x4_t*>(prow + n) = acc[rt][mt];
            }
        }
        return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int row = 16 * mt + c;
        if (row >= mcnt) continue;
        bf16_t* yrow = p.y + (int64_t)(m0 + row) * p.ldy;
        if (gemm_paired(MODE)) {
            // row tiles [0, RT/2) are gate columns, [RT/2, RT) the matching up columns
#pragma unroll
            for (int j = 0; j < RT / 2; ++j) {
                const int n = ncol0 + 16 * j + 4 * g4;
                if (n < p.N) {  // N % 4 == 0 is checked on the host
                    float o[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        o[r] = MODE == GEMM_GLU ? glm_glu_fast(p.act, acc[j][mt][r], acc[RT / 2 + j][mt][r])
                                                : rbf(glm_silu(rbf(acc[j][mt][r]))) * rbf(acc[RT / 2 + j][mt][r]);
                    u32x2_t v = {pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
                    *reinterpret_cast<u32x2_t*>(yrow + n) = v;
                }
            }
        } else {
            float sc = 1.0f;
            bool scaled = false;
            if (MODE == GEMM_DOWN && grp < p.n_scaled) {
                sc = bf2f(p.scale[m0 + row]);
                scaled = true;
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int n = ncol0 + 16 * rt + 4 * g4;
                if (n >= p.N) continue;
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float a = acc[rt][mt][r];
                    if (MODE == GEMM_PLAIN && p.bias) a += bf2f(p.bias[n + r]);
                    if (scaled) a = rbf(a) * sc;
                    o[r] = a;
                }
                if (MODE == GEMM_PLAIN) {
                    if (p.yf != nullptr) {
                        f32x4_t v;
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] = glm_act_precise(p.act, o[r], n + r);
                        *reinterpret_cast<f32x4_t*>(p.yf + (int64_t)(m0 + row) * p.ldy + n) = v;
                        continue;
                    }
                    if (p.act.kind != GLM_ACT_NONE) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[r] = glm_act_fast(p.act, o[r], n + r);
                    }
                }
                u32x2_t v = {pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
                *reinterpret_cast<u32x2_t*>(yrow + n) = v;
            }
        }
    }
}
