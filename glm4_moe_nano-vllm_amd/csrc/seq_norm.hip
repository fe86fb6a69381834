// seq_norm.hip — what happens between two sublayers of a decoder with a 32-bit residual stream, norms in front of and behind
// every sublayer and a short causal convolution over time on what a sublayer reads:
//
//     x_out = x_in + rms(y) * g_post          (y: the finished sublayer's output, optional)
//     h     = rms(x_out) * g_pre              (optional)
//     h     = h + conv(h)                     (optional; depthwise, causal, TAPS taps)
//
// in ONE launch.  gfx950 only.  Roofline: HBM — x_in and y are read once, x_out and h written once (seq_norm_stream_kernel; the
// two-pass seq_norm_kernel, which reads a row again, is for very wide rows and very long convolutions).
//
// The convolution needs the h of the TAPS-1 tokens before.  Inside a step's rows they are RECOMPUTED from x_in and y (a halo
// of TAPS-1 rows per workgroup: no hand-off between workgroups, x_out goes to another buffer than x_in); for tokens of
// earlier steps they come from the sequence's state rows.  The state is double-buffered per sequence (a step reads row set
// state_in and writes row set state_out), because the workgroup that writes a portion's last inputs is not the one that reads
// the previous portion's.  Everything is fp32 up to the store of h, and a token's h is the same arithmetic whether it was
// computed in this step or kept from an earlier one: cutting a sequence differently gives the same bits here.
#include "common.h"
#include <type_traits>

namespace {

struct SeqNormArgs {
    const float* x_in;        // [T, ldx], row r or row_index[r]
    const int32_t* row_index; // optional gather of x_in / y rows (no convolution then)
    int64_t ldx;
    float* x_out;             // [T, ldx] or nullptr
    void* x_cast;             // [T, ldc] x_out in the activation dtype, or nullptr
    int64_t ldc;
    const void* y;            // [T, ldy] or nullptr
    int64_t ldy;
    int y_f32, n_slabs;       // fp32 y: sum of n_slabs slabs (K-slice partial sums)
    int64_t slab_stride;
    const float* g_post;      // [wp]
    const float* g_pre;       // [wp] or nullptr
    const bf16_t* conv_w;     // [TAPS][wp] or nullptr (bf16 in either activation dtype: the checkpoint's values)
    float* state;             // [state rows][TAPS-1][wp]
    const int32_t* pos;       // [T] position of the row in its sequence (< 0: unused row)
    const int32_t* seq_of;    // [T]
    const int32_t* q_start;   // [S+1] first row of every sequence's portion
    const int32_t* state_in;  // [S]
    const int32_t* state_out; // [S] (< 0: keep nothing)
    int64_t n_state;          // state rows
    void* h;                  // [T, ldh]
    int64_t ldh;
    int act_f32;              // activation dtype: 0 bf16, 1 fp32
    int64_t T;
    int width, wp;            // true width (the mean's divisor), padded width (multiple of 8, zero padding)
    float eps;
};

constexpr int SN_NT = 256;

// y, or the first slab of it
__device__ __forceinline__ f32x4_t sn_load_y1(const SeqNormArgs& a, int64_t row, int col) {
    if (!a.y_f32) {
        const u32x2_t u = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const bf16_t*>(a.y) + row * a.ldy + col);
        return f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])};
    }
    return *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(a.y) + row * a.ldy + col);
}
__device__ __forceinline__ f32x4_t sn_load_y(const SeqNormArgs& a, int64_t row, int col) {
    f32x4_t v = sn_load_y1(a, row, col);
    const float* p = reinterpret_cast<const float*>(a.y) + row * a.ldy + col;
    for (int s = 1; s < a.n_slabs; ++s) v += *reinterpret_cast<const f32x4_t*>(p + s * a.slab_stride);
    return v;
}

__device__ __forceinline__ float sn_sumsq(const f32x4_t& v) { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]; }

// x_out of one row at four columns
__device__ __forceinline__ f32x4_t sn_x(const SeqNormArgs& a, int64_t row, int col, float ry) {
    f32x4_t x = *reinterpret_cast<const f32x4_t*>(a.x_in + row * a.ldx + col);
    if (a.y) {
        const f32x4_t y = sn_load_y(a, row, col), g = *reinterpret_cast<const f32x4_t*>(a.g_post + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = x[i] + y[i] * ry * g[i];
    }
    return x;
}

__device__ __forceinline__ void sn_store(void* base, int64_t off, int f32, const f32x4_t& v) {
    if (f32) *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(base) + off) = v;
    else *reinterpret_cast<u32x2_t*>(reinterpret_cast<bf16_t*>(base) + off) = u32x2_t{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
}

// TR rows per workgroup; TAPS = 1: no convolution
template <int TAPS, int TR>
__global__ __launch_bounds__(SN_NT) void seq_norm_kernel(const SeqNormArgs a) {
    constexpr int HALO = TAPS - 1, NR = TR + HALO;
    __shared__ float s_ry[NR], s_rx[NR], s_red[2][SN_NT / 64];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * TR;
    const int64_t r1 = min(r0 + TR, a.T);  // rows [r0, r1) belong to this workgroup
    const float inv_w = 1.0f / (float)a.width;
    int64_t lo = r0;  // first halo row that is needed: rows of the same sequence only
    if constexpr (TAPS > 1) lo = max(r0 - HALO, (int64_t)a.q_start[a.seq_of[r0]]);
    auto src = [&](int64_t r) -> int64_t { return a.row_index ? a.row_index[r] : r; };

    // ---- pass 1: the two reciprocal root mean squares of every row ----
    if constexpr (TR == 1) {  // the whole workgroup on one row at a time
        for (int64_t r = lo; r < r1; ++r) {
            const int64_t row = src(r);
            float ry = 0.f, s = 0.f;
            if (a.y) {
                for (int c = tid * 4; c < a.wp; c += SN_NT * 4) s += sn_sumsq(sn_load_y(a, row, c));
                s = wave_sum(s);
                if (lane == 0) s_red[0][wid] = s;
                __syncthreads();
                s = 0.f;
#pragma unroll
                for (int w = 0; w < SN_NT / 64; ++w) s += s_red[0][w];
                ry = 1.0f / sqrtf(s * inv_w + a.eps);
            }
            if (a.g_pre) {
                s = 0.f;
                for (int c = tid * 4; c < a.wp; c += SN_NT * 4) s += sn_sumsq(sn_x(a, row, c, ry));
                s = wave_sum(s);
                if (lane == 0) s_red[1][wid] = s;
                __syncthreads();
                s = 0.f;
#pragma unroll
                for (int w = 0; w < SN_NT / 64; ++w) s += s_red[1][w];
            }
            if (tid == 0) {
                s_ry[r - r0 + HALO] = ry;
                s_rx[r - r0 + HALO] = 1.0f / sqrtf(s * inv_w + a.eps);
            }
            __syncthreads();
        }
    } else {
        for (int64_t r = lo + wid; r < r1; r += SN_NT / 64) {
            const int64_t row = src(r);
            float ry = 0.f, s = 0.f;
            if (a.y) {
                for (int c = lane * 4; c < a.wp; c += 256) s += sn_sumsq(sn_load_y(a, row, c));
                ry = 1.0f / sqrtf(wave_sum(s) * inv_w + a.eps);
            }
            if (a.g_pre) {
                s = 0.f;
                for (int c = lane * 4; c < a.wp; c += 256) s += sn_sumsq(sn_x(a, row, c, ry));
                s = wave_sum(s);
            }
            if (lane == 0) {
                s_ry[r - r0 + HALO] = ry;
                s_rx[r - r0 + HALO] = 1.0f / sqrtf(s * inv_w + a.eps);
            }
        }
        __syncthreads();
    }

    // ---- pass 2: four columns per thread, down the rows; the last HALO inputs of the convolution ride in registers ----
    for (int c = tid * 4; c < a.wp; c += SN_NT * 4) {
        f32x4_t gp = {0.f, 0.f, 0.f, 0.f};
        if (a.g_pre) gp = *reinterpret_cast<const f32x4_t*>(a.g_pre + c);
        f32x4_t w[TAPS], hist[TAPS];  // hist[k-1]: h of k tokens ago
        if constexpr (TAPS > 1) {
#pragma unroll
            for (int j = 0; j < TAPS; ++j) {
                const u32x2_t u = *reinterpret_cast<const u32x2_t*>(a.conv_w + (int64_t)j * a.wp + c);
                w[j] = f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])};
            }
        }
        auto pre = [&](int64_t r, const f32x4_t& x) {
            const float rx = s_rx[r - r0 + HALO];
            f32x4_t h;
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = x[i] * rx * gp[i];
            return h;
        };
        int cur = -1;  // sequence whose history `hist` holds
        for (int64_t r = r0; r < r1; ++r) {
            const f32x4_t x = sn_x(a, src(r), c, s_ry[r - r0 + HALO]);
            if (a.x_out) *reinterpret_cast<f32x4_t*>(a.x_out + r * a.ldx + c) = x;
            if (a.x_cast) sn_store(a.x_cast, r * a.ldc + c, a.act_f32, x);
            if (!a.g_pre) continue;
            const f32x4_t h = pre(r, x);
            f32x4_t o = h;
            if constexpr (TAPS > 1) {
                const int s = a.seq_of[r], p = a.pos[r], qs = a.q_start[s];
                if (s != cur) {
                    cur = s;
                    const int64_t sin = min(max((int64_t)a.state_in[s], (int64_t)0), a.n_state - 1);
#pragma unroll
                    for (int k = 1; k < TAPS; ++k) {
                        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
                        if (p - k >= 0) {
                            if (r - k >= qs) v = pre(r - k, sn_x(a, r - k, c, s_ry[r - k - r0 + HALO]));
                            else v = *reinterpret_cast<const f32x4_t*>(a.state + (sin * HALO + (HALO - (qs - (r - k)))) * a.wp + c);
                        }
                        hist[k - 1] = v;
                    }
                }
                f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = HALO; k >= 1; --k)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = acc[i] + w[TAPS - 1 - k][i] * hist[k - 1][i];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = h[i] + (acc[i] + w[TAPS - 1][i] * h[i]);
#pragma unroll
                for (int k = HALO; k >= 2; --k) hist[k - 1] = hist[k - 2];
                hist[0] = h;
                const int qe = a.q_start[s + 1];
                const int64_t so = a.state_out[s];
                if (so >= 0 && so < a.n_state && p >= 0) {
                    const int e = qe - 1 - (int)r;  // tokens of the portion behind this one
                    if (e < HALO) *reinterpret_cast<f32x4_t*>(a.state + (so * HALO + (HALO - 1 - e)) * a.wp + c) = h;
                    if (e == 0 && qe - qs < HALO) {  // a portion shorter than the history: the older inputs move up
                        const int64_t sin = min(max((int64_t)a.state_in[s], (int64_t)0), a.n_state - 1);
                        for (int i = 0; i < HALO - (qe - qs); ++i)
                            *reinterpret_cast<f32x4_t*>(a.state + (so * HALO + i) * a.wp + c) =
                                *reinterpret_cast<const f32x4_t*>(a.state + (sin * HALO + i + (qe - qs)) * a.wp + c);
                    }
                }
            }
            sn_store(a.h, r * a.ldh + c, a.act_f32, o);
        }
    }
}

// ---- one pass: every thread owns eight columns and keeps its gains, taps and the convolution's history in registers; the rows of
// the workgroup's run go by one after the other, the next row's loads in flight.  The reduction over a row's x_out^2 and the one
// over the next row's y^2 share a barrier. ----
template <int CTRL, int ROWS>
__device__ __forceinline__ float sn_dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float sn_wave_sum(float v) {  // the sum over the wave, in lane 63
    v = sn_dpp_add<0x111, 0xf>(v);  // row_shr:1
    v = sn_dpp_add<0x112, 0xf>(v);
    v = sn_dpp_add<0x114, 0xf>(v);
    v = sn_dpp_add<0x118, 0xf>(v);
    v = sn_dpp_add<0x142, 0xa>(v);  // row_bcast:15
    v = sn_dpp_add<0x143, 0xc>(v);  // row_bcast:31
    return v;
}

struct Row8 {
    f32x4_t a, b;
};
__device__ __forceinline__ Row8 sn_ld8f(const float* p) { return {*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 4)}; }
__device__ __forceinline__ void sn_st8f(float* p, const Row8& v) {
    *reinterpret_cast<f32x4_t*>(p) = v.a;
    *reinterpret_cast<f32x4_t*>(p + 4) = v.b;
}
__device__ __forceinline__ void sn_st8(void* base, int64_t off, int f32, const Row8& v) {
    if (f32) sn_st8f(reinterpret_cast<float*>(base) + off, v);
    else
        *reinterpret_cast<u32x4_t*>(reinterpret_cast<bf16_t*>(base) + off) =
            u32x4_t{pack2bf(v.a[0], v.a[1]), pack2bf(v.a[2], v.a[3]), pack2bf(v.b[0], v.b[1]), pack2bf(v.b[2], v.b[3])};
}
__device__ __forceinline__ float sn_sumsq8(const Row8& v) { return sn_sumsq(v.a) + sn_sumsq(v.b); }

// Tables that no launch changes while it reads them: through the scalar cache, so that a row's bookkeeping waits for no vector load or store
__device__ __forceinline__ int sn_table(const int32_t* p, int64_t i) { return reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(p))[i]; }
// `bytes` of a row; nothing if there is no such buffer
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sn_row(const void* base, int64_t off, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(base) + off), 0, base ? bytes : 0, 0x00020000);
}
// (The second half is 16 bytes of the vector offset and not a scalar one: that is taken off the length before the offset is compared with it, and a buffer of no length has none to take off.
// Opaque: kept over the loop, the sum would take a register of its own.)
__device__ __forceinline__ void sn_put8f(__amdgpu_buffer_rsrc_t rs, int at, const Row8& v) {
    asm volatile("" : "+v"(at));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v.a), rs, at, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v.b), rs, at + 16, 0, 0);
}
__device__ __forceinline__ u32x4_t sn_pack8(const Row8& v) {
    return u32x4_t{pack2bf(v.a[0], v.a[1]), pack2bf(v.a[2], v.a[3]), pack2bf(v.b[0], v.b[1]), pack2bf(v.b[2], v.b[3])};
}
__device__ __forceinline__ Row8 sn_unpack8(const u32x4_t& u) {
    return {f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])}, f32x4_t{bflo(u[2]), bfhi(u[2]), bflo(u[3]), bfhi(u[3])}};
}

// sn_load_y with four slabs in flight; one or two that are left by themselves (as a group of four that reads the last slab again for those that there are not / this, us,
// runs of four rows, four taps: two slabs, 1200 rows of 2048 21.8 / 20.2, of 4096 34.2 / 30.9; six, 1200 of 4096 57.0 / 53.3)
__device__ __forceinline__ f32x4_t sn_load_slabs(const SeqNormArgs& a, int64_t row, int col) {
    f32x4_t v = sn_load_y1(a, row, col);
    const float* p = reinterpret_cast<const float*>(a.y) + row * a.ldy + col;
    int s = 1;
    for (; s + 2 < a.n_slabs; s += 4) {
        f32x4_t t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = *reinterpret_cast<const f32x4_t*>(p + min(s + j, a.n_slabs - 1) * a.slab_stride);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (s + j < a.n_slabs) v += t[j];
    }
    for (; s < a.n_slabs; ++s) v += *reinterpret_cast<const f32x4_t*>(p + s * a.slab_stride);
    return v;
}

// ANY: y or the activations may be fp32 (y in slabs: then it is summed up where it is requested).
// FORM: SN_RUNS, as described at the loop.  SN_ONE: one row per workgroup, behind the TAPS-1 in front of it: nothing waits behind its stores, so those are under tests, and the rows in front
// have neither stores nor a convolution.  SN_TESTS: the same for runs shorter than 16 rows with six and eight taps, of which a third and more are rows in front.  Stores issued
// whatever there is / this, us, prompts: four taps 64 rows of 4096 9.6 / 7.5, 300 14.7 / 11.6, 1024 of 2048 16.4 / 14.1, without y 11.9 / 8.9, 2000 of 1024
// 16.8 / 14.0; eight taps 300 of 2048 18.8 / 13.5, 2000 of them in runs of four 26.4 / 21.5; six taps 1024 of 4096 21.8 / 18.7.  Runs of 16 rows, eight taps 116 / 124.
constexpr int SN_ONE = 0, SN_TESTS = 1, SN_RUNS = 2;
template <int TAPS, int NT, bool ANY, int FORM>
__global__ __launch_bounds__(NT, (TAPS <= 4 && NT <= 512 ? 4 : 1)) void seq_norm_stream_kernel(const SeqNormArgs a, int tr) {
    constexpr int HALO = TAPS - 1, NW = NT / 64;
    constexpr bool RUN = FORM != SN_ONE, ALL = FORM == SN_RUNS;
    __shared__ float s_red[2][2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int c = tid * 8, cl = min(c, a.wp - 8);   // cl: what a thread behind the row's end reads instead
    const bool on = c < a.wp;
    const int64_t r0 = (int64_t)blockIdx.x * tr, r1 = RUN ? min(r0 + tr, a.T) : r0 + 1;
    const float inv_w = 1.0f / (float)a.width;
    int s = 0, qs = 0, qe = 0, sin = 0, so = 0;
    auto sequence = [&](int64_t r) {
        s = sn_table(a.seq_of, r);
        qs = sn_table(a.q_start, s);
        qe = sn_table(a.q_start, s + 1);
        sin = (int)min(max((int64_t)sn_table(a.state_in, s), (int64_t)0), a.n_state - 1);
        so = sn_table(a.state_out, s);
    };
    int64_t lo = r0;
    if constexpr (TAPS > 1) {
        sequence(r0);
        lo = max(r0 - HALO, (int64_t)qs);
    }
    const Row8 zero = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    Row8 gq = zero, gp = zero, hist[TAPS];
    u32x4_t w[TAPS];  // eight taps packed
    if (a.y) gq = sn_ld8f(a.g_post + cl);
    if (a.g_pre) gp = sn_ld8f(a.g_pre + cl);
    if constexpr (TAPS > 1) {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) w[j] = *reinterpret_cast<const u32x4_t*>(a.conv_w + (int64_t)j * a.wp + cl);
    }
#pragma unroll
    for (int j = 0; j < TAPS; ++j) hist[j] = zero;
    auto tap = [](const u32x4_t& p, int i) { return (i & 1) ? bfhi(p[i >> 1]) : bflo(p[i >> 1]); };
    auto source = [&](int64_t r) -> int64_t { return a.row_index ? sn_table(a.row_index, r) : r; };
    using Y = typename std::conditional<ANY, Row8, u32x4_t>::type;
    auto load_x = [&](int64_t r) { return sn_ld8f(a.x_in + source(r) * a.ldx + cl); };
    auto load_y = [&](int64_t r) -> Y {
        const int64_t row = source(r);
        if constexpr (ANY) return {sn_load_slabs(a, row, cl), sn_load_slabs(a, row, cl + 4)};
        else return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const bf16_t*>(a.y) + row * a.ldy + cl);
    };
    auto value = [](const Y& y) -> Row8 {
        if constexpr (ANY) return y;
        else return sn_unpack8(y);
    };
    auto sumsq = [&](const Row8& v) { return on ? sn_sumsq8(v) : 0.f; };
    // sums over the workgroup of two values per thread
    auto reduce2 = [&](float u, float v, int par, float& su, float& sv) {
        u = sn_wave_sum(u);
        v = sn_wave_sum(v);
        if (lane == 63) {
            s_red[par][0][wid] = u;
            s_red[par][1][wid] = v;
        }
        __syncthreads();
        su = sv = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            su += s_red[par][0][i];
            sv += s_red[par][1][i];
        }
    };
    // A row's x and the next row's y are there when its turn comes; the next x and the y behind it are requested first thing.  Every store of a turn is
    // issued whatever the launch has (buffers that there are not: of no length), and y stays as it was read until it is used, so that a turn waits for the loads of the
    // one before and not for its stores.  (It read sequence tables and state rows' numbers for every
    // row, unpacked y where it read it and stored under tests, and so waited for everything it had just asked for.)  In a step, us, that / this: four taps, y and x out, 15074
    // rows of 2048 86 / 70, 7180 40 / 35, 5000 of 4096 56 / 51; eight slabs, 700 of 2048 56 / 48; without y 57 / 44; without taps 50 / 46.  Non-temporal stores of x 74,
    // written through 106 (a lane's two halves go in two stores).
    Row8 x = load_x(lo);
    Y y{}, y1{};
    float ry = 0.f, su, sv;
    int par = 0;
    if (a.y) {
        y = load_y(lo);
        if (!ANY && lo + 1 < r1) y1 = load_y(lo + 1);
        reduce2(sumsq(value(y)), 0.f, par, su, sv);
        ry = 1.0f / sqrtf(su * inv_w + a.eps);
        par ^= 1;
    }
    // (what was requested so far is waited for here: a wait in the loop counts what is behind a load on every way to it)
    asm volatile("" : "+v"(x.a), "+v"(x.b), "+v"(gq.a), "+v"(gq.b), "+v"(gp.a), "+v"(gp.b));
    if constexpr (!ANY) asm volatile("" : "+v"(y), "+v"(y1));
    const bool f32 = ANY && a.act_f32;
    const int rowb = a.wp * 4, actb = a.wp * (f32 ? 4 : 2);
    auto put = [&](void* base, int64_t ld, int64_t r, bool mine, const Row8& v) __attribute__((always_inline)) {   // activations
        if (!ALL && !(mine && base)) return;
        const __amdgpu_buffer_rsrc_t rs = sn_row(base, r * ld * (f32 ? 4 : 2), mine ? actb : 0);
        if (f32) sn_put8f(rs, c * 4, v);
        else __builtin_amdgcn_raw_buffer_store_b128(sn_pack8(v), rs, c * 2, 0, 0);
    };
    // of a portion's first row r, out of the state (waited for here, not in every turn)
    auto history = [&](int64_t r) __attribute__((always_inline)) {
        const int p = sn_table(a.pos, r);
#pragma unroll
        for (int k = 1; k < TAPS; ++k) {
            hist[k - 1] = zero;
            if (on && p - k >= 0) hist[k - 1] = sn_ld8f(a.state + ((int64_t)sin * HALO + (HALO - k)) * a.wp + c);
        }
#pragma unroll
        for (int k = 1; k < TAPS; ++k) asm volatile("" : "+v"(hist[k - 1].a), "+v"(hist[k - 1].b));
    };
    if constexpr (TAPS > 1 && !RUN) {
        if (a.g_pre && lo == qs) history(lo);
    }
    for (int64_t r = lo; r < r1; ++r) {
        if constexpr (TAPS > 1) {  // opaque: unpacked outside the loop the taps would take twice the registers
#pragma unroll
            for (int j = 0; j < TAPS; ++j) asm volatile("" : "+v"(w[j]));
        }
        Row8 xn = zero;
        Y y2{};
        if (r + 1 < r1) xn = load_x(r + 1);
        if constexpr (ANY) {
            if (a.y && r + 1 < r1) y1 = load_y(r + 1);
        } else if (a.y && r + 2 < r1) y2 = load_y(r + 2);
        if (a.y) {
            const Row8 v = value(y);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x.a[i] = x.a[i] + v.a[i] * ry * gq.a[i];
                x.b[i] = x.b[i] + v.b[i] * ry * gq.b[i];
            }
        }
        const bool mine = TAPS == 1 || r >= r0;
        if (ALL || (mine && a.x_out)) sn_put8f(sn_row(a.x_out, r * a.ldx * 4, mine ? rowb : 0), c * 4, x);
        put(a.x_cast, a.ldc, r, mine, x);
        reduce2(sumsq(x), a.y && r + 1 < r1 ? sumsq(value(y1)) : 0.f, par, su, sv);
        par ^= 1;
        Row8 o = zero;
        if (a.g_pre) {
            const float rx = 1.0f / sqrtf(su * inv_w + a.eps);
            Row8 h;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h.a[i] = x.a[i] * rx * gp.a[i];
                h.b[i] = x.b[i] * rx * gp.b[i];
            }
            o = h;
            if constexpr (TAPS > 1) {
                if constexpr (RUN) {
                    if (r == qe) sequence(r);  // the next sequence's portion begins
                    if (r == qs) history(r);
                }
                if (ALL || mine) {
                    Row8 acc = zero;
#pragma unroll
                    for (int k = HALO; k >= 1; --k)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            acc.a[i] = acc.a[i] + tap(w[TAPS - 1 - k], i) * hist[k - 1].a[i];
                            acc.b[i] = acc.b[i] + tap(w[TAPS - 1 - k], 4 + i) * hist[k - 1].b[i];
                        }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        o.a[i] = h.a[i] + (acc.a[i] + tap(w[TAPS - 1], i) * h.a[i]);
                        o.b[i] = h.b[i] + (acc.b[i] + tap(w[TAPS - 1], 4 + i) * h.b[i]);
                    }
                    const int e = qe - 1 - (int)r;  // tokens of the portion behind this one
                    if (mine && e < HALO && so >= 0 && so < a.n_state && sn_table(a.pos, r) >= 0 && on) {
                        sn_st8f(a.state + ((int64_t)so * HALO + (HALO - 1 - e)) * a.wp + c, h);
                        if (e == 0)  // a portion shorter than the history: the older inputs move up
                            for (int i = 0; i < HALO - (qe - qs); ++i)
                                sn_st8f(a.state + ((int64_t)so * HALO + i) * a.wp + c, sn_ld8f(a.state + ((int64_t)sin * HALO + i + (qe - qs)) * a.wp + c));
                    }
                }
#pragma unroll
                for (int k = HALO; k >= 2; --k) hist[k - 1] = hist[k - 2];
                hist[0] = h;
            }
        }
        put(a.h, a.ldh, r, mine, o);
        if (a.y) ry = 1.0f / sqrtf(sv * inv_w + a.eps);
        x = xn;
        y = y1;
        if constexpr (!ANY) y1 = y2;
    }
}

// ---- some hundred rows and fewer, a row per workgroup: nothing but latency, so whatever does not depend on something else is requested first
// (the row with its slabs, four of them at a time, gains and taps; then seq_of -> q_start -> state), and only then come the sums.  Rows with
// others of their portion in front of them form those as well, as the stream kernel does: the next row is requested in front of this one's sums, and the sum over
// this x_out^2 and the one over the next y^2 share a barrier.  The arithmetic is the stream kernel's. ----
template <int TAPS, int NT>
__global__ __launch_bounds__(NT) void seq_norm_row_kernel(const SeqNormArgs a) {
    constexpr int HALO = TAPS - 1, NW = NT / 64;
    __shared__ float s_red[2][2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int c = tid * 8;
    const bool on = c < a.wp;
    const int64_t r0 = blockIdx.x;
    const float inv_w = 1.0f / (float)a.width;
    const Row8 zero = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    auto load_row = [&](int64_t r, Row8& x, Row8& y, auto in_flight) {
        constexpr int SF = decltype(in_flight)::value;  // slabs requested at a time
        x = y = zero;
        if (!on) return;
        const int64_t row = a.row_index ? a.row_index[r] : r;
        x = sn_ld8f(a.x_in + row * a.ldx + c);
        if (!a.y) return;
        if (!a.y_f32) {
            const u32x4_t u = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const bf16_t*>(a.y) + row * a.ldy + c);
            y.a = f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])};
            y.b = f32x4_t{bflo(u[2]), bfhi(u[2]), bflo(u[3]), bfhi(u[3])};
            return;
        }
        const float* p = reinterpret_cast<const float*>(a.y) + row * a.ldy + c;
        y = sn_ld8f(p);
        for (int s0 = 1; s0 < a.n_slabs; s0 += SF) {  // (added up in their order)
            Row8 v[SF];
#pragma unroll
            for (int i = 0; i < SF; ++i) v[i] = sn_ld8f(p + (int64_t)min(s0 + i, a.n_slabs - 1) * a.slab_stride);
#pragma unroll
            for (int i = 0; i < SF; ++i)
                if (s0 + i < a.n_slabs) {
                    y.a += v[i].a;
                    y.b += v[i].b;
                }
        }
    };
    int par = 0;
    auto reduce = [&](float u) {
        u = sn_wave_sum(u);
        if (lane == 63) s_red[par][0][wid] = u;
        __syncthreads();
        float su = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) su += s_red[par][0][i];
        par ^= 1;
        return su;
    };
    auto reduce2 = [&](float u, float v, float& sv) {
        v = sn_wave_sum(v);
        if (lane == 63) s_red[par][1][wid] = v;
        const int at = par;
        const float su = reduce(u);
        sv = 0.f;
#pragma unroll
        for (int i = 0; i < NW; ++i) sv += s_red[at][1][i];
        return su;
    };
    Row8 x, y, gq = zero, gp = zero;
    load_row(r0, x, y, std::integral_constant<int, 4>{});
    u32x4_t w[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) w[j] = u32x4_t{0, 0, 0, 0};
    if (on) {
        if (a.y) gq = sn_ld8f(a.g_post + c);
        if (a.g_pre) gp = sn_ld8f(a.g_pre + c);
        if constexpr (TAPS > 1) {
#pragma unroll
            for (int j = 0; j < TAPS; ++j) w[j] = *reinterpret_cast<const u32x4_t*>(a.conv_w + (int64_t)j * a.wp + c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    auto residual = [&](Row8& x, const Row8& y, float ry) {  // x_out
        if (!a.y) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x.a[i] = x.a[i] + y.a[i] * ry * gq.a[i];
            x.b[i] = x.b[i] + y.b[i] * ry * gq.b[i];
        }
    };
    auto rms = [&](float su) { return 1.0f / sqrtf(su * inv_w + a.eps); };
    auto normed = [&](const Row8& x, float rx) {
        Row8 h;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h.a[i] = x.a[i] * rx * gp.a[i];
            h.b[i] = x.b[i] * rx * gp.b[i];
        }
        return h;
    };
    Row8 hist[TAPS];       // hist[k - 1]: h of k tokens ago, in front of the portion as the state has it
    int n = 0, e = 0, d = 0, p = 0;  // tokens of the portion, of them behind this row and (as far as the taps reach) in front of it; the row's position
    int64_t so = -1;
    bool keep = false;
    // the row itself: y with its scale, the h of the tokens in front of it
    auto finish = [&](Row8& x, const Row8& y, float ry, const Row8 (&hist)[TAPS]) __attribute__((always_inline)) {
        residual(x, y, ry);
        if (on) {
            if (a.x_out) sn_st8f(a.x_out + r0 * a.ldx + c, x);
            if (a.x_cast) sn_st8(a.x_cast, r0 * a.ldc + c, a.act_f32, x);
        }
        if (!a.g_pre) return;
        const Row8 h = normed(x, rms(reduce(sn_sumsq8(x))));
        Row8 o = h;
        if constexpr (TAPS > 1) {
            auto tap = [](const u32x4_t& p, int i) { return (i & 1) ? bfhi(p[i >> 1]) : bflo(p[i >> 1]); };
            Row8 acc = zero;
#pragma unroll
            for (int k = HALO; k >= 1; --k) {
                const bool there = k <= d || p - k >= 0;  // (in front of the sequence the state holds nothing)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc.a[i] = acc.a[i] + tap(w[TAPS - 1 - k], i) * (there ? hist[k - 1].a[i] : 0.f);
                    acc.b[i] = acc.b[i] + tap(w[TAPS - 1 - k], 4 + i) * (there ? hist[k - 1].b[i] : 0.f);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o.a[i] = h.a[i] + (acc.a[i] + tap(w[TAPS - 1], i) * h.a[i]);
                o.b[i] = h.b[i] + (acc.b[i] + tap(w[TAPS - 1], 4 + i) * h.b[i]);
            }
            if (keep) {
                float* to = a.state + so * HALO * a.wp + c;
                sn_st8f(to + (int64_t)(HALO - 1 - e) * a.wp, h);
                // a portion shorter than the history, whose rows are n = d + 1 with the last one: the older inputs move up
#pragma unroll
                for (int k = 1; k < HALO; ++k)
                    if (e == 0 && k + n <= HALO) sn_st8f(to + (int64_t)(k - 1) * a.wp, hist[HALO - k - 1]);
            }
        }
        if (on) sn_st8(a.h, r0 * a.ldh + c, a.act_f32, o);
    };
    if constexpr (TAPS > 1) {
        const int s = a.seq_of[r0], qs = a.q_start[s], qe = a.q_start[s + 1];
        p = a.pos[r0];
        d = (int)min(r0 - qs, (int64_t)HALO);
        const int64_t sin = min(max((int64_t)a.state_in[s], (int64_t)0), a.n_state - 1);
        so = a.state_out[s];
        n = qe - qs;
        e = qe - 1 - (int)r0;
        keep = e < HALO && on && so >= 0 && so < a.n_state && p >= 0;
        const float* st = a.state + sin * HALO * a.wp + c;
#pragma unroll
        for (int k = 1; k < TAPS; ++k) {
            hist[k - 1] = zero;
            if (on && r0 - d == qs) hist[k - 1] = sn_ld8f(st + (int64_t)(HALO - k) * a.wp);
        }
        // (uniform; this row comes again, out of the cache.  It ends here by itself: joining the others would make them wait for what is on its way)
        if (d > 0) {
            Row8 xn, yn;
            float sv, ry = 0.f;
            load_row(r0 - d, x, y, std::integral_constant<int, 2>{});
            if (a.y) ry = rms(reduce(sn_sumsq8(y)));
            for (int64_t q = r0 - d; q < r0; ++q) {
                load_row(q + 1, xn, yn, std::integral_constant<int, 2>{});
                residual(x, y, ry);
                const float rx = rms(reduce2(sn_sumsq8(x), sn_sumsq8(yn), sv));
#pragma unroll
                for (int k = HALO; k >= 2; --k) hist[k - 1] = hist[k - 2];
                hist[0] = normed(x, rx);
                ry = rms(sv);
                x = xn;
                y = yn;
            }
            finish(x, y, ry, hist);
            return;
        }
    }
    finish(x, y, a.y ? rms(reduce(sn_sumsq8(y))) : 0.f, hist);
}

// Rows of a run: `rows`, but four at least, or eight at least
//   - where runs of four are more workgroups than there is room for at once, and take more turns than runs of eight.  Runs of four / eight, us: 2000 rows of 4096, six taps 40.3 / 30.8, 1200 of
//     8192, four taps 44.8 / 35.4; beside that the shorter ones: 2000 of 2048, four taps, 17.3 / 18.2, 1024 of 4096, six taps 22.3 / 28.3;
//   - where y (or h) is fp32 and there are enough workgroups to be bound by memory: the rows in front are read again.  Four taps, 2048 columns: eight slabs, 2100 rows 60.9 / 48.0, 3000 96.7 / 62.9,
//     four 2100 36.0 / 34.3, 4000 53.0 / 47.4, two 3000 30.1 / 29.8, 4000 37.7 / 34.4, one 4000 28.4 / 26.8; fewer rows are a chain: six slabs, 1200 29.7 / 35.4, 1600 34.6 / 37.6.  Of
//     512 threads a CU has one workgroup or two, and their turns decide as well: six slabs, 1200 rows of 4096 53.3 / 47.8, 2100 84.4 / 97.5.
template <int TAPS, int NT>
int seq_norm_run(int64_t T, int rows, bool any, int slabs) {
    constexpr int HALO = TAPS - 1, WAVES = TAPS <= 4 ? 16 : 12, WGW = NT / 64;   // waves of a CU that the registers are there for
    const int four = rows < 4 ? 4 : rows > 32 ? 32 : rows;
    if (four >= 8) return four;
    auto wgs = [&](int n) { return (T + n - 1) / n; };
    auto turns = [&](int n, int64_t at_once) { return (wgs(n) + at_once - 1) / at_once * (n + HALO); };
    const int64_t fit = 256 * ((TAPS == 8 && any ? 8 : WAVES) / WGW);
    if (turns(8, fit) < turns(four, fit)) return 8;
    if (any && wgs(8) * WGW >= (slabs >= 4 ? 1000 : 1900) && (NT < 512 || turns(8, 256) < turns(four, 256))) return 8;
    return four;
}

template <int TAPS, int NT>
int launch_seq_norm_stream(const SeqNormArgs& a, int64_t n_seq, hipStream_t st) {
    // decode: seq_norm_row_kernel; else runs of rows long enough to spread the halo and the register setup, short enough
    // to fill the chip: a row is a chain of one load, two reductions and a store, with one row's loads in flight per workgroup, so some hundred rows
    // stay one to a workgroup, re-reading the halo, as long as those are no more than four waves a SIMD (2048 workgroups of 64 threads: two), and
    // longer runs are cut for as many.  Four taps, us, runs of eight rows and more for 512 workgroups / this: 1024 columns at 800 rows 19.4 / 10.4, at 2048 20.6 / 15.9, at 8000
    // 46 / 33; 2048 at 600 rows 21.5 / 12.5, at 1024 21.9 / 16.0 (1025: 21.8, runs of eight), at 6000 45 / 40, at 15074 108 / 98 (without taps
    // 95 / 83; 2048 workgroups 78 where 1024 took 75; with loads a turn ahead
    // 512, 768, 1024 and 2048 workgroups 72.1, 70.5, 70.5 and 76.3).  Wider rows, of 512 and 1024 threads, have four and eight waves a SIMD with 512 workgroups.
    // Runs of eight rows at least / of four (two: equal but for slabs), us: 40 single rows and 5400 of prompts 35 / 31, without y 26.9 / 22.0, 3000 rows 22.7 / 20.4, 1200 19 / 16.
    constexpr int WGS = NT >= 512 ? 512 : 4096 / (NT / 64) > 2048 ? 2048 : 4096 / (NT / 64);
    if constexpr (NT < 1024 || TAPS == 1) {  // (1024 threads do not have the registers for rows, taps and history at once)
        // With taps: portions of one row, up to three quarters of the CUs.  Longer ones take the stream kernel, which knows where a portion begins before it
        // asks for a row; with a row per CU and more there is less to hide.  Stream / row kernel, four taps, us: two slabs of 2048 columns, 1 row 4.96 /
        // 4.70, 32 5.24 / 5.01, 128 6.20 / 6.02 (6.27 with one end for both branches), 200 7.10 / 7.08, 256 7.52 / 7.62, four slabs 1 5.40 / 4.84, 128 7.22 / 6.82; two of
        // 4096, 1 5.96 / 5.16, 128 8.67 / 8.04, 256 10.63 / 10.40; prompts of 64, 211 and 512 tokens, two slabs of 2048, 8.8 / 9.3, 9.9 / 10.3, 14.6 / 15.5, without the pipeline of the rows in
        // front 10.3, 11.0, 15.2.  No taps: 2048 columns, 1 row 3.74 / 3.54, 512 6.79 / 6.32.
        if (TAPS == 1 ? a.T <= 512 : a.T <= 192 && (n_seq <= 0 || n_seq >= a.T)) {
            hipLaunchKernelGGL((seq_norm_row_kernel<TAPS, NT>), dim3((unsigned)a.T), dim3(NT), 0, st, a);
            GLM_CHECK_LAUNCH("glm_seq_norm");
            return GLM_OK;
        }
    }
    const bool any = a.act_f32 || (a.y && a.y_f32);
    int tr = a.T <= 512 ? 1 : (int)((a.T + WGS - 1) / WGS);
    if (tr > 1) tr = seq_norm_run<TAPS, NT>(a.T, tr, any, a.y && a.y_f32 ? a.n_slabs : 1);
    const dim3 grid((unsigned)((a.T + tr - 1) / tr));
    auto launch = [&](auto formc) {
        constexpr int FORM = decltype(formc)::value;
        if (any) hipLaunchKernelGGL((seq_norm_stream_kernel<TAPS, NT, true, FORM>), grid, dim3(NT), 0, st, a, tr);
        else hipLaunchKernelGGL((seq_norm_stream_kernel<TAPS, NT, false, FORM>), grid, dim3(NT), 0, st, a, tr);
    };
    if (tr == 1) launch(std::integral_constant<int, SN_ONE>{});
    else if (TAPS > 4 && tr < 16) launch(std::integral_constant<int, (TAPS > 4 ? SN_TESTS : SN_RUNS)>{});
    else launch(std::integral_constant<int, SN_RUNS>{});
    GLM_CHECK_LAUNCH("glm_seq_norm");
    return GLM_OK;
}

template <int TAPS>
int launch_seq_norm(const SeqNormArgs& a, int64_t n_seq, hipStream_t st) {
    if constexpr (TAPS <= 8) {
        if (a.wp <= 512) return launch_seq_norm_stream<TAPS, 64>(a, n_seq, st);
        if (a.wp <= 1024) return launch_seq_norm_stream<TAPS, 128>(a, n_seq, st);
        if (a.wp <= 2048) return launch_seq_norm_stream<TAPS, 256>(a, n_seq, st);
        if (a.wp <= 4096) return launch_seq_norm_stream<TAPS, 512>(a, n_seq, st);
        if (TAPS <= 4 && a.wp <= 8192) return launch_seq_norm_stream<TAPS, (TAPS <= 4 ? 1024 : 512)>(a, n_seq, st);
    }
    // few rows (decode): one row per workgroup; many: 16 rows share a halo
    if (a.T <= 512) hipLaunchKernelGGL((seq_norm_kernel<TAPS, 1>), dim3((unsigned)a.T), dim3(SN_NT), 0, st, a);
    else hipLaunchKernelGGL((seq_norm_kernel<TAPS, 16>), dim3((unsigned)((a.T + 15) / 16)), dim3(SN_NT), 0, st, a);
    GLM_CHECK_LAUNCH("glm_seq_norm");
    return GLM_OK;
}

// one workgroup per token row: fp32 residual row (the table's row times `scale`) and (optionally) the row in the activation dtype.  freq: a sinusoidal position
// vector is added, sin(p f_i) at the even columns 2i and cos(p f_i) at the odd ones; the angle is taken in double and brought into
// one turn before it is rounded, so far positions are as exact as near ones.
__global__ __launch_bounds__(SN_NT) void embed_rows_kernel(const int64_t* ids, const void* table, int64_t ldw, int64_t vocab, const int32_t* pos,
                                                           const double* freq, float* x, int64_t ldx, void* cast, int64_t ldc, int act_f32, int width, int wp, int vec, float scale) {
    const int64_t t = blockIdx.x;
    const int64_t id = ids[t];
    const bool ok = id >= 0 && id < vocab;  // (an id outside the table gives a row of zeros)
    for (int c = threadIdx.x * 4; c < wp; c += SN_NT * 4) {
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
        if (ok) {
            if (vec) {  // whole rows of the table, padding included
                if (act_f32) v = *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(table) + id * ldw + c);
                else {
                    const u32x2_t u = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const bf16_t*>(table) + id * ldw + c);
                    v = f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])};
                }
            } else {
                for (int i = 0; i < 4; ++i)
                    if (c + i < width) v[i] = act_f32 ? reinterpret_cast<const float*>(table)[id * ldw + c + i] : bf2f(reinterpret_cast<const bf16_t*>(table)[id * ldw + c + i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= scale;
        if (freq) {
            const double p = (double)max(pos[t], 0);
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                if (c + i >= width) break;
                const double turns = p * freq[(c + i) >> 1] * 0.15915494309189533577;
                const float ang = (float)((turns - rint(turns)) * 6.28318530717958647693);
                v[i] += sinf(ang);
                if (c + i + 1 < width) v[i + 1] += cosf(ang);
            }
        }
        *reinterpret_cast<f32x4_t*>(x + t * ldx + c) = v;
        if (cast) sn_store(cast, t * ldc + c, act_f32, v);
    }
}

}  // namespace

extern "C" int glm_seq_norm_taps(int taps) {
    for (int t : {1, 2, 3, 4, 6, 8, 16, 32})
        if (taps >= 1 && taps <= t) return t;
    return -1;
}

extern "C" int glm_seq_norm_step(const float* x_in, const int32_t* row_index, int64_t ldx, float* x_out, void* x_cast, int64_t ldc,
                            const void* y, int64_t ldy, int y_f32, int n_slabs, int64_t slab_stride, const float* g_post,
                            const float* g_pre, const void* conv_w, int taps, float* state, int64_t n_state, const int32_t* pos,
                            const int32_t* seq_of, const int32_t* q_start, const int32_t* state_in, const int32_t* state_out,
                            void* h, int64_t ldh, int act_f32, int64_t T, int64_t n_seq, int width, int wp, float eps,
                                 glm_stream_t stream) {
    GLM_CHECK_ARG(x_in && T >= 0 && width > 0 && wp >= width && wp % 8 == 0 && ldx >= wp && ldx % 4 == 0, GLM_ERR_INVALID,
                  "glm_seq_norm: bad shape T=%ld width=%d wp=%d ldx=%ld", (long)T, width, wp, (long)ldx);
    GLM_CHECK_ARG(!y || (g_post && ldy >= wp && ldy % 4 == 0 && n_slabs >= 1 && (y_f32 || n_slabs == 1)), GLM_ERR_INVALID,
                  "glm_seq_norm: bad sublayer output (ldy=%ld slabs=%d)", (long)ldy, n_slabs);
    GLM_CHECK_ARG((!g_pre) == (!h) && (!h || (ldh >= wp && ldh % 4 == 0)) && (!x_cast || (ldc >= wp && ldc % 4 == 0)), GLM_ERR_INVALID,
                  "glm_seq_norm: bad output (ldh=%ld ldc=%ld)", (long)ldh, (long)ldc);
    GLM_CHECK_ARG(taps == 1 || (conv_w && g_pre && state && n_state > 0 && pos && seq_of && q_start && state_in && state_out && !row_index && x_out != x_in),
                  GLM_ERR_INVALID, "glm_seq_norm: the convolution needs weights, state, positions and x_out apart from x_in");
    GLM_CHECK_ARG(taps >= 1 && glm_seq_norm_taps(taps) == taps, GLM_ERR_UNSUPPORTED, "glm_seq_norm: %d taps (see glm_seq_norm_taps)", taps);
    GLM_CHECK_ARG(T < (1ll << 31), GLM_ERR_UNSUPPORTED, "glm_seq_norm: too many rows");
    if (T == 0) return GLM_OK;
    SeqNormArgs a = {x_in, row_index, ldx, x_out, x_cast, ldc, y, ldy, y_f32, n_slabs, slab_stride, g_post, g_pre, (const bf16_t*)conv_w, state,
                     pos, seq_of, q_start, state_in, state_out, n_state, h, ldh, act_f32, T, width, wp, eps};
    hipStream_t st = glm_s(stream);
    switch (taps) {
        case 1: return launch_seq_norm<1>(a, n_seq, st);
        case 2: return launch_seq_norm<2>(a, n_seq, st);
        case 3: return launch_seq_norm<3>(a, n_seq, st);
        case 4: return launch_seq_norm<4>(a, n_seq, st);
        case 6: return launch_seq_norm<6>(a, n_seq, st);
        case 8: return launch_seq_norm<8>(a, n_seq, st);
        case 16: return launch_seq_norm<16>(a, n_seq, st);
        default: return launch_seq_norm<32>(a, n_seq, st);
    }
}

extern "C" int glm_seq_norm(const float* x_in, const int32_t* row_index, int64_t ldx, float* x_out, void* x_cast, int64_t ldc,
                            const void* y, int64_t ldy, int y_f32, int n_slabs, int64_t slab_stride, const float* g_post,
                            const float* g_pre, const void* conv_w, int taps, float* state, int64_t n_state, const int32_t* pos,
                            const int32_t* seq_of, const int32_t* q_start, const int32_t* state_in, const int32_t* state_out,
                            void* h, int64_t ldh, int act_f32, int64_t T, int width, int wp, float eps, glm_stream_t stream) {
    return glm_seq_norm_step(x_in, row_index, ldx, x_out, x_cast, ldc, y, ldy, y_f32, n_slabs, slab_stride, g_post, g_pre, conv_w, taps, state, n_state, pos, seq_of, q_start, state_in,
                             state_out, h, ldh, act_f32, T, 0, width, wp, eps, stream);
}

extern "C" int glm_embed_rows(const int64_t* ids, const void* table, int64_t ldw, int64_t vocab, const int32_t* pos, const double* freq,
                              float* x, int64_t ldx, void* cast, int64_t ldc, int act_f32, int64_t T, int width, int wp, float scale,
                              glm_stream_t stream) {
    GLM_CHECK_ARG(ids && table && x && T >= 0 && width > 0 && wp >= width && wp % 8 == 0 && ldw >= width && ldx >= wp && ldx % 4 == 0 &&
                      (!cast || (ldc >= wp && ldc % 4 == 0)) && (!freq || pos), GLM_ERR_INVALID, "glm_embed_rows: bad shape T=%ld width=%d wp=%d", (long)T, width, wp);
    if (T == 0) return GLM_OK;
    const int vec = width == wp && ldw % 8 == 0 && glm_aligned16(table);
    hipLaunchKernelGGL(embed_rows_kernel, dim3((unsigned)T), dim3(SN_NT), 0, glm_s(stream), ids, table, ldw, vocab, pos, freq, x, ldx, cast, ldc, act_f32, width, wp, vec, scale);
    GLM_CHECK_LAUNCH("glm_embed_rows");
    return GLM_OK;
}
