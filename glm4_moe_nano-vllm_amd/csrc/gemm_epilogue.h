// gemm_epilogue.h — what the kernels for few rows (gemm_smallm.hip, gemm_midm.hip) do with a finished tile.
#pragma once
#include "gemm_internal.h"
#include <type_traits>

// p.act on every element of a finished tile.  What is inlined is chosen for the tile, not per element: a kernel that runs once in a step fetches its instructions
// from far away, and with every kind of activation behind every element 128 x 128 tiles had 60 KB of code, of which even rows without any jumped over all.
// A kind known at compile time also leaves no branch inside: the tests of glm_act_cols were one per element.  The long forms leave 16-row pieces without a row
// out, and where LDS is free (LOOP) they are a loop over the pieces there; own: 16 bytes per lane and piece (the next RT * MT - 1 pieces 1024 bytes apart).
// Every kind behind every element / chosen for the tile with the kinds' tests inside and all pieces / this, us: fp32 rows 300 x 2048 x 2048 with a soft cap
// 14.5 / 15.4 / 13.0, with gates 14.1 / 15.3 / 12.7, 128 x 32768 x 2048 capped 38.4 / 37.6 / 34.1, the same behind 64 MiB of other traffic 35.0 / 27.9 / 26.1; bf16
// rows with gates 13.2 / 13.3 / 11.3, 1000 x 2048 x 2048 20.4 / 19.2 / 16.6; streaming kernel, 40 x 2048 x 2056 capped 22.1 / 24.7 / 20.1, gates 20.5 / 19.5 / 18.0,
// 7 x 9728 x 2048 capped 17.3 / 17.6 / 16.4.
template <bool LOOP, int RT, int MT>
__device__ __forceinline__ void gemm_activate(const GemmParams& p, f32x4_t (&acc)[RT][MT], int mcnt, int ncol0, int g4, f32x4_t* own) {
    auto each = [&](auto&& f, int rows) __attribute__((always_inline)) {   // (16 x 16 pieces of `rows` rows)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (16 * mt >= rows) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[rt][mt][r] = f(acc[rt][mt][r], ncol0 + 16 * rt + 4 * g4 + r);
            }
    };
    auto looped = [&](auto&& f) __attribute__((always_inline)) {
        if constexpr (!LOOP) each(f, mcnt);
        else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) own[(mt * RT + rt) * 64] = acc[rt][mt];
            const int last = min((mcnt + 15) >> 4, MT) * RT - 1;
            f32x4_t v = own[0];
#pragma unroll 1
            for (int i = 0; i <= last; ++i) {
                const f32x4_t next = own[min(i + 1, last) * 64];   // (its round trip runs under this piece)
                const int n = ncol0 + 16 * (i % RT) + 4 * g4;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = f(v[r], n + r);
                own[i * 64] = v;
                v = next;
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt][mt] = own[(mt * RT + rt) * 64];
        }
    };
    const GlmAct t = p.act;
    const bool f32 = p.yf != nullptr;
    auto precise = [&](auto kind) __attribute__((always_inline)) { looped([&](float a, int n) { return glm_act_precise(GlmAct{decltype(kind)::value, t.a, t.b}, a, n); }); };
    auto cols = [&](auto kind) __attribute__((always_inline)) { each([&](float a, int n) { return glm_act_cols(GlmAct{decltype(kind)::value, t.a, t.b}, a, n); }, 16 * MT); };
    using std::integral_constant;
    if (!f32 && t.kind == GLM_ACT_XIELU) each([&](float a, int) { return glm_xielu_fast(t.a, t.b, a); }, 16 * MT);
    else if (!f32 && t.kind == GLM_ACT_SILU_GATE) cols(integral_constant<int, GLM_ACT_SILU_GATE>{});
    else if (!f32 && t.kind == GLM_ACT_RELU2_GATE) cols(integral_constant<int, GLM_ACT_RELU2_GATE>{});
    else if (!f32 && t.kind == GLM_ACT_GATE) cols(integral_constant<int, GLM_ACT_GATE>{});
    else if (t.kind == GLM_ACT_SOFTCAP) precise(integral_constant<int, GLM_ACT_SOFTCAP>{});
    else if (t.kind == GLM_ACT_XIELU) precise(integral_constant<int, GLM_ACT_XIELU>{});
    else if (t.kind == GLM_ACT_SILU_GATE) precise(integral_constant<int, GLM_ACT_SILU_GATE>{});
    else if (t.kind == GLM_ACT_RELU2_GATE) precise(integral_constant<int, GLM_ACT_RELU2_GATE>{});
    else if (t.kind == GLM_ACT_GATE) precise(integral_constant<int, GLM_ACT_GATE>{});
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
        if (p.act.kind != GLM_ACT_NONE) gemm_activate<LOOP>(p, acc, mcnt, ncol0, g4, own);
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
