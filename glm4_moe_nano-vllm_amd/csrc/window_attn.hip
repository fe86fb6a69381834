// window_attn.hip — varlen causal attention with a sliding window and a learned sink per head for prompts and long portions of
// prompts: q rows of the step against expanded k / v rows (the portion's own tokens and the part of the sequence's history that
// the window still reaches).  Head sizes of keys and values are independent, multiples of 8.  gfx950 only.
//
// Roofline: MFMA.  A workgroup owns 128 query rows of one (sequence, head); each of its 4 waves two 16-row query tiles, so
// that every K / V fragment read from LDS feeds two tiles.  64-key tiles are staged by LDS-DMA, double-buffered, one barrier per
// tile, only over the keys the rows can see: [first row - window + 1, last row], and walked as in attn_units.h.  The sink joins the
// denominator once, at the end.
#include "common.h"
#include "attn_lds.h"
#include "attn_units.h"

namespace {

__device__ const u32x4_t wa_zero_page[4] = {};

struct WinArgs {
    const bf16_t* q;   // [rows, ldq], head h at h*dk
    int64_t ldq;
    const bf16_t *k, *v;  // [Tk, ldkv], head h at h*dkn / h*dv
    int64_t ldkv;
    const bf16_t* kr;  // [Tk, ldr] the last dk - dkn key columns, shared by all heads
    int64_t ldr;
    const float* cs;   // [rows, (dk - dkn) / 2, 2] rotation of those query columns, pairs (2i, 2i+1)
    const bf16_t* gate;  // [rows, ldg] factors of the output, laid out like out, or nullptr
    int64_t ldg;
    bf16_t* out;       // [rows, ldo], head h at h*dv
    int64_t ldo;
    const int32_t *q_start;  // [S+1] first q / out row of every sequence's portion
    const int32_t *k_start;  // [S+1] first k / v row
    const int32_t *tile_seq, *tile_off;  // [n_tiles]
    const float* sink;
    int S, n_tiles, H, dk, dkn, dv, window;
    int64_t Tq, Tk;
    float scale;
};

enum : int { WA_PLAIN = 0, WA_PADDED = 1, WA_ROTATED = 2 };   // heads as wide as the tiles, narrower ones, or (of any width) with key columns in rows of their own

// DK, DV: multiples of 64
template <int DK, int DV, int FORM>
__global__ __launch_bounds__(256, (DK + DV) <= 320 ? 2 : 1) void window_attn_kernel(const WinArgs a) {
    using SL = Slab<DK, DV, 2, GA_SOFTMAX>;
    constexpr int KS = SL::KS, VT = SL::VT, KTILE = 64 * SL::KB, STAGE = KTILE + 64 * SL::VB;
    constexpr int KCPR = DK / 8, VCPR = DV / 8, KDMA = DK / 32, VDMA = DV / 32;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    // XCD-aware order: workgroups with equal id % 8 share an XCD and take one contiguous run of (head, tile) items
    const int total = a.n_tiles * a.H, per = (total + 7) >> 3;
    const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || item >= total) return;
    const int h = item / a.n_tiles, tile = item % a.n_tiles;
    const int seq = a.tile_seq[tile], qo = a.tile_off[tile];
    const int qs = a.q_start[seq], nq = a.q_start[seq + 1] - qs;
    const int ks0 = a.k_start[seq], nk = a.k_start[seq + 1] - ks0;
    const int hist = nk - nq;  // keys in front of the portion's first token
    if (qo >= nq || hist < 0) return;
    const int qlast = min(qo + 127, nq - 1);
    const int jlo = max(0, hist + qo - a.window + 1), jhi = hist + qlast;
    const int n = (jhi - jlo + 64) >> 6;
    const unsigned base = lds_addr(smem);
    const bf16_t* kbase = a.k + (int64_t)(ks0 + jlo) * a.ldkv + (int64_t)h * a.dkn;
    const bf16_t* rbase = a.kr ? a.kr + (int64_t)(ks0 + jlo) * a.ldr : kbase;
    const bf16_t* vbase = a.v + (int64_t)(ks0 + jlo) * a.ldkv + (int64_t)h * a.dv;
    const int nkeys = jhi - jlo + 1;
    // Sources of the DMA pieces: as in group_attn.hip (chunks that do not divide a piece evenly: offsets of all pieces, one base).  With the last dk - dkn key
    // columns in rows of their own a piece has two sources and takes addresses, per lane a row of either or zeros.
    constexpr int KRP = 64 / KCPR, VRP = 64 / VCPR, KEVEN = 64 % KCPR == 0, KPER = KEVEN ? 8 / KRP : KDMA, VEVEN = 64 % VCPR == 0, VPER = VEVEN ? 8 / VRP : VDMA;
    auto k_piece = [&](int lane, int i, int& row, int& ch) {
        const int q = (w * KDMA + i) * 64 + lane;
        row = q / KCPR;
        ch = (q % KCPR) ^ attn_swz(row);
    };
    unsigned koff[KPER], voff[VPER];   // bytes
    unsigned krot = 0;                 // bit i: piece i of a period is of the other rows
#pragma unroll
    for (int i = 0; i < KPER; ++i) {
        int row, ch;
        k_piece(lane, i, row, ch);
        const bool rot = ch * 8 >= a.dkn;
        krot |= rot ? 1u << i : 0u;
        koff[i] = ch * 8 < a.dk ? (unsigned)(rot ? row * (int)a.ldr + ch * 8 - a.dkn : row * (int)a.ldkv + ch * 8) * 2u : ATTN_BEYOND;
    }
#pragma unroll
    for (int i = 0; i < VPER; ++i) {
        const int q = (w * VDMA + i) * 64 + lane, row = q / VCPR, ch = (q % VCPR) ^ attn_swz(row);
        voff[i] = ch * 8 < a.dv ? (unsigned)(row * (int)a.ldkv + ch * 8) * 2u : ATTN_BEYOND;
    }
    const int kvb = (int)a.ldkv * 2;   // bytes of a row
    const bool padded = FORM == WA_PADDED || (FORM == WA_ROTATED && (a.dk != DK || a.dv != DV));
    auto issue = [&](int it, auto) __attribute__((always_inline)) {
        const int first = (n - 1 - it) * 64, left = nkeys - first;
        const char* kb = reinterpret_cast<const char*>(kbase + (int64_t)first * a.ldkv);
        const char* vb = reinterpret_cast<const char*>(vbase + (int64_t)first * a.ldkv);
        char* st = smem + (it & 1) * STAGE;
        const bool whole = !padded && left >= 64;
        if constexpr (FORM == WA_ROTATED) {
            const char* rb = reinterpret_cast<const char*>(rbase + (int64_t)first * a.ldr);
            if (whole) {
#pragma unroll
                for (int i = 0; i < KDMA; ++i) {
                    const int64_t step = (int64_t)(i / KPER) * 8;
                    lds_dma16(krot >> (i % KPER) & 1 ? rb + step * a.ldr * 2 + koff[i % KPER] : kb + step * kvb + koff[i % KPER], st + (w * KDMA + i) * 1024);
                }
            } else {
                int ln = lane;
                asm volatile("" : "+v"(ln));   // (rows worked out here and now: kept over the tiles they cost the loop its registers)
#pragma unroll
                for (int i = 0; i < KDMA; ++i) {
                    int row, ch;
                    k_piece(ln, i, row, ch);
                    const int64_t step = (int64_t)(i / KPER) * 8;
                    const char* s = krot >> (i % KPER) & 1 ? rb + step * a.ldr * 2 + koff[i % KPER] : kb + step * kvb + koff[i % KPER];
                    lds_dma16(koff[i % KPER] == ATTN_BEYOND || row >= left ? (const void*)wa_zero_page : (const void*)s, st + (w * KDMA + i) * 1024);
                }
            }
        } else if (whole) {
#pragma unroll
            for (int i = 0; i < KDMA; ++i) lds_dma16(kb + (int64_t)(i / KPER) * 8 * kvb + koff[i % KPER], st + (w * KDMA + i) * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < KDMA; ++i)
                lds_dma16(attn_rows(kb + (int64_t)(i / KPER) * 8 * kvb, left - 8 * (i / KPER), kvb), koff[i % KPER], st + (w * KDMA + i) * 1024);
        }
        if (whole) {
#pragma unroll
            for (int i = 0; i < VDMA; ++i) lds_dma16(vb + (int64_t)(i / VPER) * 8 * kvb + voff[i % VPER], st + KTILE + (w * VDMA + i) * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < VDMA; ++i)
                lds_dma16(attn_rows(vb + (int64_t)(i / VPER) * 8 * kvb, left - 8 * (i / VPER), kvb), voff[i % VPER], st + KTILE + (w * VDMA + i) * 1024);
        }
    };
    issue(0, std::integral_constant<int, 0>{});   // in front of everything that waits for the queries
    // The walk hides keys and takes maxima in front of the scale, which has to be positive there: the queries take its sign, and are zeros where it is zero.
    const unsigned sign = a.scale < 0.f ? 0x80008000u : 0u, keep = a.scale == 0.f ? 0u : ~0u;
    const float scale = a.scale == 0.f ? 1.f : fabsf(a.scale);
    // this wave's rows: tile t holds rows qo + 64 t + 16 w + c (the two half-dead tiles of the causal edge cost all waves the same)
    SL S;
    S.init(lane);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int r0 = qo + 64 * t + 16 * w, r = r0 + c;
        const bool some = r0 < nq;
        const int a0 = hist + r0, a1 = hist + min(r0 + 15, nq - 1);
        S.rp[t] = r < nq ? hist + r : -1;      // key index of the row itself
        S.rlo[t] = S.rp[t] - a.window + 1;
        S.any_lo[t] = some ? a0 - a.window + 1 : 1 << 30;
        S.any_hi[t] = some ? a1 : -1;
        S.full_lo[t] = some ? a1 - a.window + 1 : 1 << 30;
        S.full_hi[t] = some ? a0 : -1;
        const bf16_t* qp = a.q + (int64_t)(qs + min(r, nq - 1)) * a.ldq + (int64_t)h * a.dk;
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int k = 32 * i + 8 * g;
            S.qf[t][i] = u32x4_t{0, 0, 0, 0};
            if (k < a.dk) S.qf[t][i] = *reinterpret_cast<const u32x4_t*>(qp + k);
            if (k >= a.dkn && k < a.dk) {  // rotated here: a lane holds whole pairs
                const float* cs = a.cs + (int64_t)(qs + min(r, nq - 1)) * (a.dk - a.dkn) + (k - a.dkn);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float u = bflo(S.qf[t][i][j]), v = bfhi(S.qf[t][i][j]), co = cs[2 * j], si = cs[2 * j + 1];
                    S.qf[t][i][j] = pack2bf(u * co - v * si, v * co + u * si);
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < KS; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) S.qf[t][i][j] = (S.qf[t][i][j] & keep) ^ sign;
            asm volatile("" : "+v"(S.qf[t][i]));
        }
    attn_tiles<DK, DV, GA_SOFTMAX, KDMA + VDMA>(S, base, n, jlo, g, scale * GA_LOG2E, false, issue);
    const float sk = a.sink[h] * GA_LOG2E;
    u32x2_t gt[2][VT];   // all of them at once: behind a store each would wait for it (128 + 128, window of 1024, 15074 rows of 16 heads: 177.0 / 168.4 us)
    if (a.gate) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bf16_t* gp = a.gate + (int64_t)(qs + min(qo + 64 * t + 16 * w + c, nq - 1)) * a.ldg + (int64_t)h * a.dv;
#pragma unroll
            for (int d = 0; d < VT; ++d) gt[t][d] = *reinterpret_cast<const u32x2_t*>(gp + (16 * d + 4 * g < a.dv ? 16 * d + 4 * g : 0));
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float l = S.mass(t);
        const int r = qo + 64 * t + 16 * w + c;
        if (r >= nq) continue;
        const float M = fmaxf(S.m_run[t], sk), f = __builtin_amdgcn_exp2f(S.m_run[t] - M);
        const float inv = f / (l * f + __builtin_amdgcn_exp2f(sk - M));
        bf16_t* o = a.out + (int64_t)(qs + r) * a.ldo + (int64_t)h * a.dv;
#pragma unroll
        for (int d = 0; d < VT; ++d) {
            const int dim = 16 * d + 4 * g;
            if (a.gate) S.acc[t][d] *= f32x4_t{bflo(gt[t][d][0]), bfhi(gt[t][d][0]), bflo(gt[t][d][1]), bfhi(gt[t][d][1])};
            if (dim < a.dv) *reinterpret_cast<u32x2_t*>(o + dim) = u32x2_t{pack2bf(S.acc[t][d][0] * inv, S.acc[t][d][1] * inv), pack2bf(S.acc[t][d][2] * inv, S.acc[t][d][3] * inv)};
        }
    }
}

template <int DK, int DV>
int launch_window(const WinArgs& a, hipStream_t st) {
    constexpr int LDS = 2 * 64 * (DK + DV) * 2;
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    auto kern = a.dkn != a.dk ? window_attn_kernel<DK, DV, WA_ROTATED> : a.dk != DK || a.dv != DV ? window_attn_kernel<DK, DV, WA_PADDED> : window_attn_kernel<DK, DV, WA_PLAIN>;
    GLM_SET_MAX_LDS(kern, LDS, "glm_window_attn_prefill");
    const int64_t per = ((int64_t)a.n_tiles * a.H + 7) / 8;
    GLM_CHECK_ARG(per * 8 < (1ll << 31), GLM_ERR_UNSUPPORTED, "glm_window_attn_prefill: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)(per * 8)), dim3(256), LDS, st, a);
    GLM_CHECK_LAUNCH("glm_window_attn_prefill");
    return GLM_OK;
}

template <int DK>
int launch_window_dv(const WinArgs& a, hipStream_t st) {
    if (a.dv <= 64) return launch_window<DK, 64>(a, st);
    if (a.dv <= 128) return launch_window<DK, 128>(a, st);
    if (a.dv <= 192) return launch_window<DK, 192>(a, st);
    return launch_window<DK, 256>(a, st);
}

}  // namespace

extern "C" int glm_window_attn_prefill(const void* q, int64_t ldq, const void* k, const void* v, int64_t ldkv, const void* kr, int64_t ldr, int rotp, const float* cs,
                                       const void* gate, int64_t ldg, void* out, int64_t ldo,
                                       const int32_t* q_start, const int32_t* k_start, const int32_t* tile_seq, const int32_t* tile_off, int n_tiles, int S,
                                       int64_t Tq, int64_t Tk, int H, int dk, int dv, int window, float scale, const float* sink, glm_stream_t stream) {
    GLM_CHECK_ARG(q && k && v && out && q_start && k_start && tile_seq && tile_off && sink, GLM_ERR_INVALID, "glm_window_attn_prefill: null pointer");
    GLM_CHECK_ARG(H > 0 && dk > 0 && dv > 0 && dk % 8 == 0 && dv % 8 == 0 && ldq >= (int64_t)H * dk && ldkv >= (int64_t)H * (dk - rotp > dv ? dk - rotp : dv) && ldo >= (int64_t)H * dv &&
                      ldq % 8 == 0 && ldkv % 8 == 0 && ldo % 4 == 0 && window > 0 && S > 0 && n_tiles >= 0 && Tq >= 0 && Tk >= Tq && ldkv < (1 << 24) &&
                      glm_aligned16(q) && glm_aligned16(k) && glm_aligned16(v), GLM_ERR_INVALID,
                  "glm_window_attn_prefill: bad shape H=%d dk=%d dv=%d ldq=%ld ldkv=%ld window=%d", H, dk, dv, (long)ldq, (long)ldkv, window);
    GLM_CHECK_ARG(dk <= 256 && dv <= 256, GLM_ERR_UNSUPPORTED, "glm_window_attn_prefill: head sizes up to 256 (dk=%d dv=%d)", dk, dv);
    GLM_CHECK_ARG(rotp >= 0 && rotp < dk && rotp % 8 == 0 && (rotp == 0 || (kr && cs && ldr >= rotp && ldr % 8 == 0 && ldr < (1 << 24) && glm_aligned16(kr))) &&
                      (!gate || (ldg >= (int64_t)H * dv && ldg % 4 == 0)), GLM_ERR_INVALID, "glm_window_attn_prefill: bad rotated part of %d columns or gate", rotp);
    if (n_tiles == 0) return GLM_OK;
    WinArgs a = {(const bf16_t*)q, ldq, (const bf16_t*)k, (const bf16_t*)v, ldkv, rotp ? (const bf16_t*)kr : nullptr, ldr, cs, (const bf16_t*)gate, ldg, (bf16_t*)out, ldo,
                 q_start, k_start, tile_seq, tile_off, sink, S, n_tiles, H, dk, dk - rotp, dv, window, Tq, Tk, scale};
    hipStream_t st = glm_s(stream);
    if (dk <= 64) return launch_window_dv<64>(a, st);
    if (dk <= 128) return launch_window_dv<128>(a, st);
    if (dk <= 192) return launch_window_dv<192>(a, st);
    return launch_window_dv<256>(a, st);
}
