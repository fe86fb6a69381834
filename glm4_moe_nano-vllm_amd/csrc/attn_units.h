// attn_units.h — the walk of a wave over the 64-key tiles of a prompt's attention, shared by group_attn.hip and window_attn.hip: two 16-row tiles of
// queries (or the two maps of one) per wave, keys and values in LDS, double-buffered.  What the callers add: which keys a row sees, where the
// tiles come from, what becomes of the sums.
#pragma once
#include "attn_lds.h"

namespace {

constexpr float GA_LOG2E = 1.4426950408889634f;
// forms of the tiled kernels
// (GA_TWO_MAPS: the scores have a soft cap that 2^score fits under as it is; GA_TWO_MAPS_ANY: any cap, or none)
enum : int { GA_SOFTMAX = 0, GA_TWO_MAPS = 1, GA_SIGMOID_KV = 2, GA_TWO_MAPS_ANY = 3 };
constexpr float GA_CAP_FITS = 55.f;  // cap log2(e) <= 80: the sums of 2^score stay far inside fp32 whatever their number
__host__ __device__ constexpr bool ga_two(int form) { return form == GA_TWO_MAPS || form == GA_TWO_MAPS_ANY; }

// the two products of a 32-key slab and the softmax between them, for NT tiles of 16 query rows (lane c holds row c of each)
// (two maps: of two tiles, tile t holds map t's rows of the queries and meets the keys' half t; in one tile a row's queries are
// zeros in the other map's half)
template <int DK, int DV, int NT, int F>
struct Slab {
    static constexpr bool SPLIT = ga_two(F) && NT == 2;
    static constexpr int KS = DK / 32, KQ = SPLIT ? KS / 2 : KS, VT = DV / 16, KB = DK * 2, VB = DV * 2;
    static constexpr bool VEARLY = DK + DV <= 256 && DV <= 128;  // all fragments of a slab in registers beside the next one's
    u32x4_t qf[NT][KQ];
    f32x4_t acc[NT][VT];
    float m_run[NT], l_run[NT], slope[NT];                // slope: per key, in units of the unscaled score; sigmoid: the bias in log2 units
    float cap_in, cap_out;                                // soft cap: exponent per unit of score, cap in log2 units (0: none)
    float cap_lim, ca0, ca1, ca2, ca3;                    // scores up to cap_lim: odd polynomial
    int rp[NT], rlo[NT];                                  // position of the lane's row and the first one it sees; rp < 0: no row
    int any_lo[NT], any_hi[NT], full_lo[NT], full_hi[NT]; // keys that some row / every row of the tile sees
    unsigned k_rel[2], v_rel[4];

    __device__ __forceinline__ void init(int lane) {
        const int c = lane & 15, g = lane >> 4;
        // K row c, chunk 4 i + g (its low three bits depend on the parity of i only); V row 4 g + qq
#pragma unroll
        for (int e = 0; e < 2; ++e) k_rel[e] = c * KB + (((4 * e + g) ^ attn_swz(c)) << 4);
        const int qq = (lane >> 2) & 3, pp = lane & 3, vr = 4 * g + qq;
#pragma unroll
        for (int e = 0; e < 4; ++e) v_rel[e] = vr * VB + (((2 * e + (pp >> 1)) ^ attn_swz(vr)) << 4) + ((pp & 1) << 3);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            m_run[t] = -INFINITY;
            l_run[t] = 0.f;
#pragma unroll
            for (int d = 0; d < VT; ++d) acc[t][d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    // cap tanh(s / cap) in log2 units, by tanh y = 1 - 2 / (1 + e^(2 y))
    __device__ __forceinline__ void cap_exact(f32x4_t (&s)[2]) const {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[kt][r] = fmaf(-2.f * cap_out, __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[kt][r] * cap_in)), cap_out);
    }
    // Largest magnitude of the eight scores, as glm_largest8.  (Inline asm right behind the products: the choice between tanh's two forms changed from run to run.)
    __device__ __forceinline__ static float size(const f32x4_t (&s)[2]) {
        f32x4_t m[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) m[i >> 2][i & 3] = fabsf(s[i >> 2][i & 3]);
        return glm_largest8(m);
    }
    // up to a fifth of the cap tanh is its odd polynomial of degree 7 (the next term is below 2e-8 of the cap)
    __device__ __forceinline__ void cap_small(f32x4_t (&s)[2]) const {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float u = s[kt][r] * s[kt][r];
                s[kt][r] *= fmaf(fmaf(fmaf(ca3, u, ca2), u, ca1), u, ca0);
            }
    }
    // One 32-key slab, its parts one after the other: decoding, a tile or two, and head sizes whose fragments of two slabs do not fit the registers.  kst,
    // vst, fst: LDS addresses of its first key row, value row and (sigmoid form) the keys' factors; j0: position of its first key.  K fragments in groups of four, the
    // first V fragments beside the last of them, the others a group ahead of their products.  4096 and 3707 tokens, 16 heads, all K fragments at once / this, us: heads
    // of 256 over 4 key heads, softmax 552 / 516, two maps 793 / 767, sigmoid weights 401 / 382; 256 + 128 442 / 409, two maps under a
    // cap 686 / 640 (one after the other under it: 657); every head by itself with a sink 544 / 488, 192 + 128 249 / 232; 64 + 256 and 128 + 256, which have no more than four,
    // 418 / 418 and 449 / 455.
    __device__ __forceinline__ void run(unsigned kst, unsigned vst, int j0, int g, float sc, unsigned fst, bool biased) {
        bool live[NT], some = false;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            live[t] = j0 <= any_hi[t] && j0 + 31 >= any_lo[t];
            some = some || live[t];
        }
        if (!some) return;
        constexpr int VG = VEARLY ? VT : 4, VN = VT / VG;   // V fragments per request group
        constexpr int KG = KS <= 4 ? KS : 4, KN = (KS + KG - 1) / KG;   // K fragments per request group
        u32x4_t kf[2][KS], ks[2];
        constexpr int VB2 = VN > 1 ? 2 : 1;                             // V groups in registers
        u32x2_t vf[VB2][VG][2];
        auto read_v = [&](auto GI) {
            static_for<VG>([&](auto I) {
                constexpr int gi = decltype(GI)::value, i = decltype(I)::value, d = gi * VG + i;
                lds_read_tr16_b64<(d >> 2) * 128>(vf[gi % VB2][i][0], vst + v_rel[d & 3]);
                lds_read_tr16_b64<(d >> 2) * 128 + 16 * VB>(vf[gi % VB2][i][1], vst + v_rel[d & 3]);
            });
        };
        if constexpr (F == GA_SIGMOID_KV) {  // (in front of the K fragments: in when they are)
            lds_read_b128<0>(ks[0], fst + 16 * g);
            lds_read_b128<64>(ks[1], fst + 16 * g);
        }
        f32x4_t s[NT][2];
        static_for<KN>([&](auto GI) {
            constexpr int k0 = decltype(GI)::value * KG, kn = KS - k0 < KG ? KS - k0 : KG;
            static_for<kn>([&](auto I) {
                constexpr int i = k0 + decltype(I)::value;
                lds_read_b128<(i >> 1) * 128>(kf[0][i], kst + k_rel[i & 1]);
                lds_read_b128<(i >> 1) * 128 + 16 * KB>(kf[1][i], kst + k_rel[i & 1]);
            });
            if constexpr (k0 + KG >= KS) {
                read_v(std::integral_constant<int, 0>{});
                // the K fragments are in; the V fragments (issued last) may still be on their way
                asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(2 * VG <= 15 ? 2 * VG : 15) : "memory");
                if constexpr (F == GA_SIGMOID_KV) asm volatile("" : "+v"(ks[0]), "+v"(ks[1]));
            } else {
                wait_lds();
            }
#pragma unroll
            for (int i = k0; i < k0 + kn; ++i) asm volatile("" : "+v"(kf[0][i]), "+v"(kf[1][i]));
            static_for<kn>([&](auto I) {   // (the tiles' chains side by side: little else covers their latency where a CU holds one workgroup)
                constexpr int i = k0 + decltype(I)::value;
                static_for<NT>([&](auto T) {
                    constexpr int t = decltype(T)::value;
                    if constexpr (!SPLIT || i / KQ == t) {
                        if constexpr (i % KQ == 0) {
                            first_scores<t>(s[t], kf, j0, g, biased);
                        } else {
#pragma unroll
                            for (int kt = 0; kt < 2; ++kt) add_score<t>(s[t], kf, kt, i % KQ, s[t][kt]);
                        }
                    }
                });
            });
        });
        constexpr bool JOINT = F == GA_TWO_MAPS && NT > 1 && DK > 64;   // both maps under the cap at once
        if constexpr (JOINT) {
            if (__any(!(fmaxf(size(s[0]), size(s[1])) <= cap_lim))) {
                cap_exact(s[0]);
                cap_exact(s[1]);
            } else {
                cap_small(s[0]);
                cap_small(s[1]);
            }
        }
        bf16x8_t pf[NT];
        static_for<NT>([&](auto T) {
            constexpr int t = decltype(T)::value;
            if (live[t]) {
                pf[t] = weights<t, true, JOINT>(s[t], j0, g, sc, ks);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) pf[t][i] = (__bf16)0.f;
            }
        });
        static_for<VN>([&](auto GI) {
            constexpr int gi = decltype(GI)::value;
            wait_lds();
            vpin(vf[gi % VB2]);
            if constexpr (gi + 1 < VN) {
                read_v(std::integral_constant<int, gi + 1>{});
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < VG; ++i) {
                const u32x4_t vv = {vf[gi % VB2][i][0][0], vf[gi % VB2][i][0][1], vf[gi % VB2][i][1][0], vf[gi % VB2][i][1][1]};
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t][gi * VG + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf[t], acc[t][gi * VG + i], 0, 0, 0);
            }
        });
    }
    template <int N>
    __device__ __forceinline__ static void vpin(u32x2_t (&v)[N][2]) {
#pragma unroll
        for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i][0]), "+v"(v[i][1]));
    }
    // scores of tile T: start from the distance bias where there is one
    template <int T>
    __device__ __forceinline__ void add_score(f32x4_t (&s)[2], const u32x4_t (&kf)[2][KS], int kt, int i, const f32x4_t& to) const {
        s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[kt][SPLIT ? T * KQ + i : i]), __builtin_bit_cast(bf16x8_t, qf[T][i]), to, 0, 0, 0);
    }
    template <int T>
    __device__ __forceinline__ void first_scores(f32x4_t (&s)[2], const u32x4_t (&kf)[2][KS], int j0, int g, bool biased) const {
        if (F == GA_SOFTMAX && biased) {
            const float b0 = slope[T] * (float)(j0 + 4 * g - rp[T]);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                f32x4_t bias4;
#pragma unroll
                for (int r = 0; r < 4; ++r) bias4[r] = fmaf(slope[T], (float)(16 * kt + r), b0);
                add_score<T>(s, kf, kt, 0, bias4);
            }
        } else {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) add_score<T>(s, kf, kt, 0, f32x4_t{0.f, 0.f, 0.f, 0.f});
        }
    }
    template <int T>
    __device__ __forceinline__ void scores(f32x4_t (&s)[2], const u32x4_t (&kf)[2][KS], int j0, int g, bool biased) const {
        first_scores<T>(s, kf, j0, g, biased);
#pragma unroll
        for (int i = 1; i < KQ; ++i)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) add_score<T>(s, kf, kt, i, s[kt]);
    }
    // weights of tile T; fac: sigmoid form, factors of the lane's keys times scale and log2 e, negative; EDGE: some keys may be hidden; CAPPED: the scores
    template <int T, bool EDGE, bool CAPPED = false>
    __device__ __forceinline__ bf16x8_t weights(f32x4_t (&s)[2], int j0, int g, float sc, const u32x4_t (&fac)[2]) {
        bf16x8_t pf;
        if constexpr (F == GA_SIGMOID_KV) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const f32x4_t f = __builtin_bit_cast(f32x4_t, fac[kt]) * -sc;
#pragma unroll
                for (int r = 0; r < 4; ++r) s[kt][r] = fmaf(s[kt][r], f[r], -slope[T]);
            }
        }
        if constexpr (F == GA_TWO_MAPS && !CAPPED) {
            if (__any(!(size(s) <= cap_lim))) cap_exact(s);
            else cap_small(s);
        }
        if (F == GA_TWO_MAPS_ANY && cap_out > 0.f) cap_exact(s);
        if (EDGE && (j0 < full_lo[T] || j0 + 31 > full_hi[T])) {
            const int jl = j0 + 4 * g;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = jl + 16 * kt + r;
                    if (j > rp[T] || j < rlo[T]) s[kt][r] = F == GA_SIGMOID_KV ? INFINITY : -INFINITY;
                }
        }
        float m_use = 0.f;
        if constexpr (F == GA_SOFTMAX || F == GA_TWO_MAPS_ANY) {
            float mx = glm_largest8(s) * sc;
            if (__any(mx > m_run[T] + 8.0f || (m_run[T] == -INFINITY && mx > -INFINITY))) {
                mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                const float m_new = fmaxf(m_run[T], mx);
                const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run[T] - m_new);
                l_run[T] *= alpha;
#pragma unroll
                for (int d = 0; d < VT; ++d) acc[T][d] *= alpha;
                m_run[T] = m_new;
            }
            m_use = m_run[T] == -INFINITY ? 0.f : m_run[T];
        }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float p;
                if constexpr (F == GA_SIGMOID_KV) p = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[kt][r]));
                else if constexpr (F == GA_TWO_MAPS) p = __builtin_amdgcn_exp2f(s[kt][r]);
                else p = __builtin_amdgcn_exp2f(fmaf(s[kt][r], sc, -m_use));
                if constexpr (F != GA_SIGMOID_KV) l_run[T] += p;
                pf[4 * kt + r] = (__bf16)p;
            }
        return pf;
    }
    template <int T>
    __device__ __forceinline__ void values(const bf16x8_t pf, const u32x2_t (&vf)[VT][2]) {
#pragma unroll
        for (int d = 0; d < VT; ++d) {
            const u32x4_t vv = {vf[d][0][0], vf[d][0][1], vf[d][1][0], vf[d][1][1]};
            acc[T][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf, acc[T][d], 0, 0, 0);
        }
    }
    __device__ __forceinline__ void set_cap(float cap, float scale) {
        if constexpr (!ga_two(F)) return;
        cap_in = cap > 0.f ? 2.f * GA_LOG2E * scale / cap : 0.f;
        cap_out = cap * GA_LOG2E;
        const float k = cap > 0.f ? scale / cap : 0.f, kk = k * k;
        cap_lim = k > 0.f ? 0.2f / k : 0.f;
        ca0 = cap_out * k;
        ca1 = ca0 * kk * (-1.f / 3.f);
        ca2 = ca0 * kk * kk * (2.f / 15.f);
        ca3 = ca0 * kk * kk * kk * (-17.f / 315.f);
        if constexpr (F == GA_TWO_MAPS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) m_run[t] = 0.f;
        }
    }
    __device__ __forceinline__ float mass(int t) const {
        float l = l_run[t];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        return l;
    }
};

// All n tiles of 64 keys, the first of them position jlo, from the last to the first.  issue(it, k) brings tile n - 1 - it to LDS buffer it & 1 (k: it, 2 from there on; keys,
// behind them the values or, sigmoid form, the keys' factors), at least PIECES DMA instructions of every wave, in the order of it; the caller has done so for it = 0,
// in front of its wait for the queries (a workgroup's start is two trips to memory instead of three; asked for here / there, us: 15074 tokens of 4 prompts, 16 heads, windows of 1024
// 173.9 / 171.9, two maps under a cap 573 / 568, 192 + 128 406 / 404; 5 prompts of 2500 in chunks 89.4 / 87.7, of 900 with two maps 63.5 / 61.3).  S holds the queries, the ranges of
// visible keys and, in the end, the sums.
template <int DK, int DV, int F, int PIECES, class Issue>
__device__ __forceinline__ void attn_tiles(Slab<DK, DV, 2, F>& S, unsigned base, int n, int jlo, int g, float sc, bool biased, Issue&& issue) {
    using SL = Slab<DK, DV, 2, F>;
    constexpr bool KV = F == GA_SIGMOID_KV;
    constexpr int VT = SL::VT, KB = SL::KB, VB = SL::VB, KTILE = 64 * KB, STAGE = KTILE + (KV ? 256 : 64 * VB);
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    auto slabs = [&]() __attribute__((always_inline)) {
        for (int it = 0; it < n; ++it) {
            wait_vm<0>();
            __builtin_amdgcn_s_barrier();
            if (it == 0 && n > 1) issue(1, I1{});
            else if (it + 1 < n) issue(it + 1, I2{});
            const unsigned st = base + (it & 1) * STAGE;
#pragma unroll
            for (int s = 1; s >= 0; --s)
                S.run(st + s * 32 * KB, st + (KV ? 0 : KTILE) + s * 32 * VB, jlo + (n - 1 - it) * 64 + s * 32, g, sc, st + KTILE + s * 128, biased);
        }
    };
    if constexpr (SL::VEARLY) {
        // ---- units (slab, tile): the scores of the next unit are started in front of the weights of this one, and the fragments they need are
        // requested a unit ahead, so that neither LDS nor the matrix pipe's latency stands between a unit's parts.  Per tile of 64 keys (slabs 1, 0):
        //   (1, t0)  scores (1, t1); V of slab 1, K of slab 0 requested; weights, values
        //   (1, t1)  scores (0, t0); weights, values
        //   (0, t0)  scores (0, t1); V of slab 0 requested; weights; the next tile has arrived, the one after it is requested into this
        //            tile's buffer, whose last fragments are in (barrier), K of the next tile's slab 1 requested; values
        //   (0, t1)  scores of the next tile's (1, t0); weights, values
        // One tile or two go by slabs, which pass by what no row sees: 40 tokens, 15 heads over 3 of 128 7.6 (before units), 8.0 (units), 7.9.
        // 15074 tokens of 4 prompts, 16 heads of 128 + 128, slabs one after the other / units, us: softmax 348 / 316, two maps of 64 under a cap
        // 617 / 584, sigmoid weights 323 / 314, windows of 1024 193 / 181.  What is left: LDS reads (every wave reads all keys and values for 32
        // rows, 2300 of some 5000 clocks a tile with the staging), exponentials and products beside one another, some 8 us of start and end per
        // workgroup.
        constexpr int KS = SL::KS, FR = KV ? 2 : 0;
        u32x4_t kf[2][KS], fac[2][2];   // K fragments; factors of the keys of slab 1 and 0 (sigmoid)
        u32x2_t vf[VT][2];
        f32x4_t sa[2], sb[2];
        auto read_k = [&](unsigned st, auto slabc) {
            constexpr int sl = decltype(slabc)::value;
            const unsigned kst = st + sl * 32 * KB;
            static_for<KS>([&](auto I) {
                constexpr int i = decltype(I)::value;
                lds_read_b128<(i >> 1) * 128>(kf[0][i], kst + S.k_rel[i & 1]);
                lds_read_b128<(i >> 1) * 128 + 16 * KB>(kf[1][i], kst + S.k_rel[i & 1]);
            });
            if constexpr (KV) {
                const unsigned fst = st + KTILE + sl * 128 + 16 * g;
                lds_read_b128<0>(fac[1 - sl][0], fst);
                lds_read_b128<64>(fac[1 - sl][1], fst);
            }
        };
        auto read_v = [&](unsigned st, auto slabc) {
            const unsigned vst = st + (KV ? 0 : KTILE) + decltype(slabc)::value * 32 * VB;
            static_for<VT>([&](auto I) {
                constexpr int d = decltype(I)::value;
                lds_read_tr16_b64<(d >> 2) * 128>(vf[d][0], vst + S.v_rel[d & 3]);
                lds_read_tr16_b64<(d >> 2) * 128 + 16 * VB>(vf[d][1], vst + S.v_rel[d & 3]);
            });
        };
        // the registers pass through: no use moves above the wait
        auto k_here = [&]() {
            wait_lds();
#pragma unroll
            for (int i = 0; i < KS; ++i) asm volatile("" : "+v"(kf[0][i]), "+v"(kf[1][i]));
            if constexpr (KV) asm volatile("" : "+v"(fac[0][0]), "+v"(fac[0][1]), "+v"(fac[1][0]), "+v"(fac[1][1]));
        };
        auto v_here = [&]() {
#pragma unroll
            for (int d = 0; d < VT; ++d) asm volatile("" : "+v"(vf[d][0]), "+v"(vf[d][1]));
        };
        auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
        auto seen = [&](int j, int t) { return j <= S.any_hi[t] && j + 31 >= S.any_lo[t]; };   // by some row of the tile
        if (n <= 2) return slabs();
        if (n > 1) {
            issue(1, I1{});
            wait_vm<PIECES>();   // (a wave that brings more waits for some of them too)
        } else {
            wait_vm<0>();
        }
        __builtin_amdgcn_s_barrier();
        read_k(base, I1{});
        if constexpr (KV) asm volatile("" : "=v"(fac[1][0]), "=v"(fac[1][1]));
        k_here();
        S.template scores<0>(sa, kf, jlo + (n - 1) * 64 + 32, g, biased);
        auto tile = [&](auto edgec, int it) {
            constexpr bool EDGE = decltype(edgec)::value;
            const unsigned st = base + (it & 1) * STAGE;
            const int j0 = jlo + (n - 1 - it) * 64, j1 = j0 + 32;
            const bool more = it + 1 < n;
            // (1, t0)
            S.template scores<1>(sb, kf, j1, g, biased);
            fence();
            read_v(st, I1{});
            read_k(st, I0{});
            const bool s10 = !EDGE || seen(j1, 0), s11 = !EDGE || seen(j1, 1), s00 = !EDGE || seen(j0, 0), s01 = !EDGE || seen(j0, 1);
            bf16x8_t pf;
            if (s10) pf = S.template weights<0, EDGE>(sa, j1, g, sc, fac[0]);
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(2 * KS + FR) : "memory");  // (the K fragments may still be on their way)
            v_here();
            if (s10) S.template values<0>(pf, vf);
            fence();
            // (1, t1)
            k_here();
            S.template scores<0>(sa, kf, j0, g, biased);
            fence();
            if (s11) {
                pf = S.template weights<1, EDGE>(sb, j1, g, sc, fac[0]);
                S.template values<1>(pf, vf);
            }
            fence();
            // (0, t0)
            S.template scores<1>(sb, kf, j0, g, biased);
            fence();
            read_v(st, I0{});
            if (s00) pf = S.template weights<0, EDGE>(sa, j0, g, sc, fac[1]);
            wait_lds();
            v_here();
            if (more) {
                wait_vm<0>();
                __builtin_amdgcn_s_barrier();
                if (it + 2 < n) issue(it + 2, I2{});
            }
            // (behind the last tile: whatever the other buffer holds, for scores that nobody uses; a branch would part the reads from their wait)
            read_k(base + ((it + 1) & 1) * STAGE, I1{});
            if (s00) S.template values<0>(pf, vf);
            fence();
            // (0, t1)
            k_here();
            S.template scores<0>(sa, kf, j0 - 32, g, biased);
            fence();
            if (s01) {
                pf = S.template weights<1, EDGE>(sb, j0, g, sc, fac[1]);
                S.template values<1>(pf, vf);
            }
            fence();
        };
        // tiles of which every row sees every key, and the others
        const int in_lo = max(S.full_lo[0], S.full_lo[1]), in_hi = min(S.full_hi[0], S.full_hi[1]);
        auto inside = [&](int it) { const int j0 = jlo + (n - 1 - it) * 64; return j0 >= in_lo && j0 + 63 <= in_hi; };
        int it = 0;
        while (it < n) {
            while (it < n && inside(it)) tile(std::false_type{}, it++);
            while (it < n && !inside(it)) tile(std::true_type{}, it++);
        }
    } else {
        slabs();
    }
}

}  // namespace
