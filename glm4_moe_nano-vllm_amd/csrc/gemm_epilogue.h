// gemm_epilogue.h — what the kernels for few rows (gemm_smallm.hip, gemm_midm.hip) do with a finished tile.
#pragma once
#include "gemm_internal.h"

// p.act on every element of a finished tile.  What is inlined is chosen for the tile, not per element: a kernel that runs once in a step fetches its
// instructions from far away, and with every kind of activation behind every element 128 x 128 tiles had 60 KB of code, of which even
// rows without any jumped over all (32768 fp32 columns x 2048 at 128 rows inside a step of Dafolorn 49.6 us, by itself time after time 37.6).  own: 16 bytes
// of LDS per lane and 16-byte piece (the next RT * MT - 1 pieces 1024 bytes apart), in which the long forms are a loop (LOOP).
template <bool LOOP, int RT, int MT>
__device__ __forceinline__ void gemm_activate(const GemmParams& p, f32x4_t (&acc)[RT][MT], int ncol0, int g4, f32x4_t* own) {
    auto each = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[rt][mt][r] = f(acc[rt][mt][r], ncol0 + 16 * rt + 4 * g4 + r);
    };
    const bool f32 = p.yf != nullptr;
    if (!f32 && p.act.kind == GLM_ACT_XIELU) each([&](float a, int) { return glm_xielu_fast(p.act.a, p.act.b, a); });
    else if (!f32 && p.act.kind >= GLM_ACT_GATE) each([&](float a, int n) { return glm_act_cols(p.act, a, n); });
    else if constexpr (!LOOP) each([&](float a, int n) { return f32 ? glm_act_precise(p.act, a, n) : glm_act_fast(p.act, a, n); });
    else {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) own[(rt * MT + mt) * 64] = acc[rt][mt];
#pragma unroll 1
        for (int i = 0; i < RT * MT; ++i) {
            f32x4_t v = own[i * 64];
            const int n = ncol0 + 16 * (i / MT) + 4 * g4;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = f32 ? glm_act_precise(p.act, v[r], n + r) : glm_act_fast(p.act, v[r], n + r);
            own[i * 64] = v;
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = own[(rt * MT + mt) * 64];
    }
}

// Lane (c,g4) holds, per (rt, mt), columns n..n+3 of token
// row 16*mt + c
template <int MODE, int RT, int MT, bool LOOP = false>
__device__ __forceinline__ void gemm_row_epilogue(const GemmParams& p, f32x4_t (&acc)[RT][MT], int grp, int m0,
                                                  int mcnt, int ncol0, int c, int g4, f32x4_t* own = nullptr) {
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
    if constexpr (MODE == GEMM_PLAIN) {
        if (p.bias != nullptr) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int n = ncol0 + 16 * rt + 4 * g4;
                if (n >= p.N) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float b = bf2f(p.bias[n + r]);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[rt][mt][r] += b;
                }
            }
        }
        if (p.act.kind != GLM_ACT_NONE) gemm_activate<LOOP>(p, acc, ncol0, g4, own);
        if (p.yf != nullptr) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int row = 16 * mt + c;
                if (row >= mcnt) continue;
                float* yrow = p.yf + (int64_t)(m0 + row) * p.ldy;
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const int n = ncol0 + 16 * rt + 4 * g4;
                    if (n < p.N) *reinterpret_cast<f32x4_t*>(yrow + n) = acc[rt][mt];
                }
            }
            return;
        }
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
                    if (scaled) a = rbf(a) * sc;
                    o[r] = a;
                }
                u32x2_t v = {pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
                *reinterpret_cast<u32x2_t*>(yrow + n) = v;
            }
        }
    }
}
