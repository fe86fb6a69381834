// depth_norm.hip — what happens between two sublayers of a decoder whose sublayers read the 32-bit residual as it is, are closed by an
// RMS norm in groups, and whose layers hand on a learned average over all depths:
//
//     x_out  = x_in + norm(y) * g_post               norm: every one of `groups` equal parts divided by its own root mean square
//     x_next = sum_j coef[j] depth_j + coef[n] x_out  (optional; depth_j: n earlier rows of the same token, one plane each)
//     h      = x_next + conv(x_next)                 (optional; depthwise, causal, TAPS taps)      or
//     h      = norm(x_next) * g_pre                  (optional)
//
// in one launch (many rows: two).  y is the finished sublayer's output, or — pair_pos — the rows of a token's k experts, summed with their fp32 weights.
// gfx950 only.  Roofline: HBM — every row is read and written once.
//
// A part of the vector belongs to lanes of one wave (up to 512 columns) or to whole waves, eight columns per lane: with parts of at most
// 512 columns no sum leaves its wave, and the kernel has no barrier.  A workgroup takes one row.
// The convolution's inputs of the TAPS-1 tokens in front of it are recomputed (rows of the same step) or come from the sequence's
// state rows, which are double-buffered: a step reads row set state_in and writes row set state_out.  Everything is fp32 up to the store
// of h, the same arithmetic for a token of this step as for one whose row was kept.
//
// Steps of many rows, and prompts of some hundred, take two launches, norm and average (every row for itself) and depth_conv: re-reading x_next costs four bytes a
// column; with runs of sixteen rows, recomputing the TAPS-1 in front cost a fifth of rows that are k experts and several depths
// wide.
#include "common.h"

namespace {

struct DepthArgs {
    const float* x_in;         // [T, ld], row r or row_index[r]
    const int32_t* row_index;  // optional gather of x_in / y / depth rows (no convolution then)
    int64_t ld;                // pitch of x_in, x_out, x_next and the depth rows
    const void* y;             // [T, ldy], or with pair_pos [n_rows, ldy], or nullptr
    int64_t ldy;
    const int32_t* pair_pos;   // [T, k] row of y of the token's j-th expert (outside [0, n_rows): none)
    const float* pair_w;       // [T, k]
    int k;
    int64_t n_rows;
    const float* g_post;       // [wp]
    float* x_out;              // or nullptr
    void* x_cast;              // x_out in the activation dtype, or nullptr
    int64_t ldc;
    const float* depth;        // plane j at depth + j * depth_stride, or nullptr
    int64_t depth_stride;
    int n_depth;
    const float* coef;         // [n_depth + 1]
    float* x_next;             // or nullptr
    const float* g_pre;        // [wp] or nullptr
    const bf16_t* conv_w;      // [TAPS][wp]
    float* state;              // [state rows][TAPS-1][wp]
    const int32_t *pos, *seq_of, *q_start, *state_in, *state_out;
    int64_t n_state;
    void* h;                   // [T, ldh] or nullptr
    int64_t ldh;
    int act_f32;
    int64_t T;
    int width, wp, groups, gs;
    int lpg, gpw, wpg, cpw;    // lanes per part inside a wave, parts per wave; waves per part, columns per wave
    float eps;
};

struct Col8 {
    float v[8];
};
__device__ __forceinline__ Col8 dn_zero() { return {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}}; }

// n of the eight columns at p are there; VEC: all of them or none, 16-byte aligned
template <bool VEC>
__device__ __forceinline__ Col8 dn_ldf(const float* p, int n) {
    Col8 o = dn_zero();
    if constexpr (VEC) {
        if (n) {
            const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o.v[i] = a[i];
                o.v[4 + i] = b[i];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < n) o.v[i] = p[i];
    }
    return o;
}
template <bool VEC>
__device__ __forceinline__ void dn_stf(float* p, const Col8& o, int n) {
    if constexpr (VEC) {
        if (n) {
            *reinterpret_cast<f32x4_t*>(p) = f32x4_t{o.v[0], o.v[1], o.v[2], o.v[3]};
            *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{o.v[4], o.v[5], o.v[6], o.v[7]};
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < n) p[i] = o.v[i];
    }
}
template <bool VEC>
__device__ __forceinline__ Col8 dn_ldh(const bf16_t* p, int n) {
    Col8 o = dn_zero();
    if constexpr (VEC) {
        if (n) {
            const u32x4_t u = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o.v[2 * i] = bflo(u[i]);
                o.v[2 * i + 1] = bfhi(u[i]);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < n) o.v[i] = bf2f(p[i]);
    }
    return o;
}
template <bool VEC>
__device__ __forceinline__ Col8 dn_ld(const void* p, int64_t off, int f32, int n) {
    return f32 ? dn_ldf<VEC>(reinterpret_cast<const float*>(p) + off, n) : dn_ldh<VEC>(reinterpret_cast<const bf16_t*>(p) + off, n);
}
template <bool VEC>
__device__ __forceinline__ void dn_st(void* p, int64_t off, int f32, const Col8& o, int n) {
    if (f32) {
        dn_stf<VEC>(reinterpret_cast<float*>(p) + off, o, n);
        return;
    }
    bf16_t* q = reinterpret_cast<bf16_t*>(p) + off;
    if constexpr (VEC) {
        if (n) *reinterpret_cast<u32x4_t*>(q) = u32x4_t{pack2bf(o.v[0], o.v[1]), pack2bf(o.v[2], o.v[3]), pack2bf(o.v[4], o.v[5]), pack2bf(o.v[6], o.v[7])};
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < n) q[i] = f2bf(o.v[i]);
    }
}
__device__ __forceinline__ float dn_sumsq(const Col8& a) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += a.v[i] * a.v[i];
    return s;
}

// this lane's columns: nc of eight from column c
__device__ __forceinline__ void dn_columns(const DepthArgs& a, int lane, int wid, int& c, int& nc) {
    int gi, o;
    if (a.wpg == 1) {
        gi = wid * a.gpw + lane / a.lpg;
        o = (lane % a.lpg) * 8;
        if (lane / a.lpg >= a.gpw) gi = a.groups;
    } else {
        gi = wid / a.wpg;
        o = (wid % a.wpg) * a.cpw + lane * 8;
        if (lane * 8 >= a.cpw) o = a.gs;
    }
    nc = gi < a.groups ? min(8, max(0, a.gs - o)) : 0;
    c = nc ? gi * a.gs + o : 0;
}
// 1 / root mean square of this lane's part
__device__ __forceinline__ float dn_part_rms(const DepthArgs& a, const Col8& v, int lane, int wid, float (*s_red)[16], int& par) {
    float q = dn_sumsq(v);
    for (int s = 1; s < a.lpg; s <<= 1) q += __shfl_xor(q, s, 64);
    if (a.wpg > 1) {
        if (lane == 0) s_red[par][wid] = q;
        __syncthreads();
        q = 0.f;
        const int w0 = wid / a.wpg * a.wpg;
        for (int i = 0; i < a.wpg; ++i) q += s_red[par][w0 + i];
        par ^= 1;
    }
    return 1.0f / sqrtf(q / (float)a.gs + a.eps);
}
struct DepthRow {   // of one row: x_in, the first four depths
    Col8 x, e0[4];
};
template <bool VEC>
__device__ __forceinline__ void dn_fetch(const DepthArgs& a, int64_t row, int c, int nc, DepthRow& f) {
    f.x = dn_ldf<VEC>(a.x_in + row * a.ld + c, nc);
    const float* d = a.depth ? a.depth + row * a.ld + c : nullptr;
#pragma unroll
    for (int u = 0; u < 4; ++u) f.e0[u] = a.depth && u < a.n_depth ? dn_ldf<VEC>(d + u * a.depth_stride, nc) : dn_zero();
}
// x_out and x_next of one row (f of x_in, y and the depths), the loads together
template <bool VEC>
__device__ __forceinline__ void dn_row(const DepthArgs& a, int64_t row, int c, int nc, int lane, int wid, float (*s_red)[16], int& par, const DepthRow& f, Col8& x, Col8& xn) {
    x = f.x;
    const float* d = a.depth ? a.depth + row * a.ld + c : nullptr;
    if (a.y) {
        Col8 y = dn_zero();
        if (!a.pair_pos) {
            y = dn_ld<VEC>(a.y, row * a.ldy + c, a.act_f32, nc);
        } else if (VEC && !a.act_f32) {
            for (int j0 = 0; j0 < a.k; j0 += 8) {  // eight experts' rows in flight
                u32x4_t e[8];
                float we[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int p = j0 + j < a.k ? a.pair_pos[row * a.k + j0 + j] : -1;
                    const bool ok = p >= 0 && p < a.n_rows;
                    we[j] = ok ? a.pair_w[row * a.k + j0 + j] : 0.f;
                    e[j] = u32x4_t{0, 0, 0, 0};
                    if (ok && nc) e[j] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const bf16_t*>(a.y) + (int64_t)p * a.ldy + c);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        y.v[2 * i] = fmaf(we[j], bflo(e[j][i]), y.v[2 * i]);
                        y.v[2 * i + 1] = fmaf(we[j], bfhi(e[j][i]), y.v[2 * i + 1]);
                    }
            }
        } else {
            for (int j = 0; j < a.k; ++j) {
                const int p = a.pair_pos[row * a.k + j];
                if (p < 0 || p >= a.n_rows) continue;
                const Col8 e = dn_ld<VEC>(a.y, (int64_t)p * a.ldy + c, a.act_f32, nc);
#pragma unroll
                for (int i = 0; i < 8; ++i) y.v[i] = fmaf(a.pair_w[row * a.k + j], e.v[i], y.v[i]);
            }
        }
        const Col8 gq = dn_ldf<VEC>(a.g_post + c, nc);
        const float ry = dn_part_rms(a, y, lane, wid, s_red, par);
#pragma unroll
        for (int i = 0; i < 8; ++i) x.v[i] = x.v[i] + y.v[i] * ry * gq.v[i];
    }
    xn = x;
    if (!a.depth) return;
    Col8 avg = dn_zero();
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (u < a.n_depth) {
#pragma unroll
            for (int i = 0; i < 8; ++i) avg.v[i] = fmaf(a.coef[u], f.e0[u].v[i], avg.v[i]);
        }
    for (int j = 4; j < a.n_depth; j += 4) {
        Col8 e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = j + u < a.n_depth ? dn_ldf<VEC>(d + (j + u) * a.depth_stride, nc) : dn_zero();
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (j + u < a.n_depth) {
#pragma unroll
                for (int i = 0; i < 8; ++i) avg.v[i] = fmaf(a.coef[j + u], e[u].v[i], avg.v[i]);
            }
    }
    const float cx = a.coef[a.n_depth];
#pragma unroll
    for (int i = 0; i < 8; ++i) xn.v[i] = fmaf(cx, x.v[i], avg.v[i]);
}

// One row per workgroup.  TAPS > 1: with the convolution, for which the TAPS-1 rows in front are computed as well, as far as they are of
// this step.  What bounds it with few rows is a chain of trips to memory.  Up to 512 threads, four taps and one round of the chip (NT, with registers for it) the row, the depths and the taps are requested
// in front of the sequence's tables, not behind them and not behind the stores: behind k = 6 experts and one to three depths, four taps, in a step, us: 100 rows of 2048 10.8 / 9.2, 9 rows
// 10.2 / 8.8, 60 rows of 4096 13.3 / 10.5, without experts 7.8 / 6.3.
template <int TAPS, bool VEC, int NT>
__global__ __launch_bounds__(NT) void depth_norm_kernel(const DepthArgs a) {
    constexpr int HALO = TAPS - 1;
    constexpr bool EARLY = NT <= 512;
    __shared__ float s_red[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int c, nc, par = 0;
    dn_columns(a, lane, wid, c, nc);
    const int64_t r = blockIdx.x;
    Col8 x, xn, hist[TAPS];
    DepthRow f;
    u32x4_t wk[TAPS];
    if constexpr (EARLY) {
        dn_fetch<VEC>(a, r, c, nc, f);   // (the convolution's rows are not gathered)
#pragma unroll
        for (int k = 0; k < TAPS; ++k) wk[k] = *reinterpret_cast<const u32x4_t*>(a.conv_w + (int64_t)k * a.wp + c);
    }
    int s = 0, qs = 0, qe = 0;
    int64_t sin = 0, lo = r;
    if constexpr (TAPS > 1) {
        s = a.seq_of[r];
        qs = a.q_start[s];
        qe = a.q_start[s + 1];
        sin = min(max((int64_t)a.state_in[s], (int64_t)0), a.n_state - 1);
        lo = max(r - HALO, (int64_t)qs);
        const int p = a.pos[r];
#pragma unroll
        for (int k = 1; k < TAPS; ++k)  // what lies in front of the portion
            hist[k - 1] = dn_ldf<VEC>(a.state + (sin * HALO + (r - k < qs ? HALO - (qs - (r - k)) : 0)) * a.wp + c, p - k >= 0 && r - k < qs ? nc : 0);
        for (int64_t q = lo; q < r; ++q) {
            DepthRow e;
            dn_fetch<VEC>(a, q, c, nc, e);
            dn_row<VEC>(a, q, c, nc, lane, wid, s_red, par, e, x, xn);
#pragma unroll
            for (int k = 1; k < TAPS; ++k)
                if (r - q == k) hist[k - 1] = xn;
        }
    }
    const int64_t row = TAPS == 1 && a.row_index ? (int64_t)a.row_index[r] : r;
    if constexpr (!EARLY) dn_fetch<VEC>(a, row, c, nc, f);
    dn_row<VEC>(a, row, c, nc, lane, wid, s_red, par, f, x, xn);
    if (a.x_out) dn_stf<VEC>(a.x_out + r * a.ld + c, x, nc);
    if (a.x_cast) dn_st<VEC>(a.x_cast, r * a.ldc + c, a.act_f32, x, nc);
    if (a.depth && a.x_next) dn_stf<VEC>(a.x_next + r * a.ld + c, xn, nc);
    if (tid < a.wp - a.width) {  // padding columns are zeros
        const int pc = a.width + tid;
        if (a.x_cast) {
            if (a.act_f32) reinterpret_cast<float*>(a.x_cast)[r * a.ldc + pc] = 0.f;
            else reinterpret_cast<bf16_t*>(a.x_cast)[r * a.ldc + pc] = 0;
        }
        if (a.h) {
            if (a.act_f32) reinterpret_cast<float*>(a.h)[r * a.ldh + pc] = 0.f;
            else reinterpret_cast<bf16_t*>(a.h)[r * a.ldh + pc] = 0;
        }
    }
    if (!a.h) return;
    Col8 h = xn;
    if (a.g_pre) {
        const Col8 gp = dn_ldf<VEC>(a.g_pre + c, nc);
        const float rx = dn_part_rms(a, xn, lane, wid, s_red, par);
#pragma unroll
        for (int i = 0; i < 8; ++i) h.v[i] = xn.v[i] * rx * gp.v[i];
    }
    if constexpr (TAPS > 1) {
        Col8 acc = dn_zero();
#pragma unroll
        for (int k = HALO; k >= 0; --k) {
            Col8 w;
            if constexpr (EARLY) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    w.v[2 * i] = bflo(wk[TAPS - 1 - k][i]);
                    w.v[2 * i + 1] = bfhi(wk[TAPS - 1 - k][i]);
                }
            } else {
                w = dn_ldh<VEC>(a.conv_w + (int64_t)(TAPS - 1 - k) * a.wp + c, nc);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) acc.v[i] = acc.v[i] + w.v[i] * (k ? hist[k ? k - 1 : 0].v[i] : xn.v[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) h.v[i] = xn.v[i] + acc.v[i];
        const int64_t so = a.state_out[s];
        const int e = qe - 1 - (int)r;  // tokens of the portion behind this one
        if (e < HALO && so >= 0 && so < a.n_state && a.pos[r] >= 0) {
            dn_stf<VEC>(a.state + (so * HALO + (HALO - 1 - e)) * a.wp + c, xn, nc);
            if (e == 0)  // a portion shorter than the history: the older inputs move up
                for (int i = 0; i < HALO - (qe - qs); ++i)
                    dn_stf<VEC>(a.state + (so * HALO + i) * a.wp + c, dn_ldf<VEC>(a.state + (sin * HALO + i + (qe - qs)) * a.wp + c, nc), nc);
        }
    }
    dn_st<VEC>(a.h, r * a.ldh + c, a.act_f32, h, nc);
}

// Tables that no launch changes while it reads them: through the scalar cache, so that a row's bookkeeping waits for no vector load or store
__device__ __forceinline__ int dn_table(const int32_t* p, int64_t i) { return reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(p))[i]; }
__device__ __forceinline__ void dn_put(void* base, int64_t off, int bytes, int at, const u32x4_t& v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(base) + off, 0, bytes, 0x00020000), at, 0, 0);
}

// h = x + conv(x) and the state, eight columns per thread down a run of rows, UN rows at a time, the next ones' loads in flight: what a turn needs of memory was requested
// a turn ago, rows stay as they were read until they are used, and every store is issued (of no length behind the run's end), so that no turn waits for what it has just
// asked for or stored.  (Padding columns masked
// where they were read and the state row's number read for every row, as it was / this, us in a step, four taps, runs of 16 rows: 15074 rows of 2048 41.3 / 38.3, 5000 of 4096
// 35 / 25.6, 700 of 2048 16.8 / 10.3, 40 single rows and 5400 of prompts 74 / 42.)
template <int TAPS, bool F32>
__global__ __launch_bounds__(256) void depth_conv_kernel(const DepthArgs a, const float* __restrict__ xs, int tr) {
    constexpr int HALO = TAPS - 1, UN = TAPS <= 4 ? 2 : 1;
    const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
    if (c >= a.wp) return;
    const int nc = min(8, a.width - c);   // (the padding columns of x are not written by anyone)
    const int64_t r0 = (int64_t)blockIdx.x * tr, r1 = min(r0 + tr, a.T);
    struct Raw {
        f32x4_t a, b;
    };
    auto raw = [&](const float* p) -> Raw { return {*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 4)}; };
    auto masked = [&](const Raw& v) {
        Col8 o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o.v[i] = i < nc ? (i < 4 ? v.a[i & 3] : v.b[i & 3]) : 0.f;
        return o;
    };
    u32x4_t w[TAPS];   // eight taps packed
    Col8 hist[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        w[j] = *reinterpret_cast<const u32x4_t*>(a.conv_w + (int64_t)j * a.wp + c);
        hist[j] = dn_zero();
    }
    auto tap = [](const u32x4_t& p, int i) { return (i & 1) ? bfhi(p[i >> 1]) : bflo(p[i >> 1]); };
    int s = 0, qs = 0, qe = 0, so = 0;
    int64_t sin = 0;
    auto sequence = [&](int64_t r) {   // and the inputs of the tokens in front of row r
        s = dn_table(a.seq_of, r);
        qs = dn_table(a.q_start, s);
        qe = dn_table(a.q_start, s + 1);
        sin = min(max((int64_t)dn_table(a.state_in, s), (int64_t)0), a.n_state - 1);
        so = dn_table(a.state_out, s);
        const int p = dn_table(a.pos, r);
        Raw t[TAPS];
#pragma unroll
        for (int k = 1; k < TAPS; ++k) {
            t[k - 1] = Raw{};
            if (p - k < 0) continue;
            if (r - k >= qs) t[k - 1] = raw(xs + (r - k) * a.ld + c);
            else t[k - 1] = raw(a.state + (sin * HALO + (HALO - (qs - (r - k)))) * a.wp + c);
        }
#pragma unroll
        for (int k = 1; k < TAPS; ++k) {
            asm volatile("" : "+v"(t[k - 1].a), "+v"(t[k - 1].b));   // (waited for here, not in every turn)
            hist[k - 1] = masked(t[k - 1]);
        }
    };
    Raw x[UN], xn[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
        x[u] = xn[u] = Raw{};
        if (r0 + u < r1) x[u] = raw(xs + (r0 + u) * a.ld + c);
    }
    sequence(r0);
#pragma unroll
    for (int u = 0; u < UN; ++u) asm volatile("" : "+v"(x[u].a), "+v"(x[u].b));
#pragma unroll
    for (int j = 0; j < TAPS; ++j) asm volatile("" : "+v"(w[j]));
    const int rowb = a.wp * (F32 ? 4 : 2);
    for (int64_t r = r0; r < r1; r += UN) {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) asm volatile("" : "+v"(w[j]));  // opaque: unpacked outside the loop the taps would take twice the registers
#pragma unroll
        for (int u = 0; u < UN; ++u)
            if (r + UN + u < r1) xn[u] = raw(xs + (r + UN + u) * a.ld + c);
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int64_t row = r + u;
            const bool there = row < r1;
            if (there && row == qe) sequence(row);  // the next sequence's portion begins
            const Col8 xv = masked(x[u]);
            Col8 acc = dn_zero(), h;
#pragma unroll
            for (int k = HALO; k >= 1; --k)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc.v[i] = acc.v[i] + tap(w[TAPS - 1 - k], i) * hist[k - 1].v[i];
#pragma unroll
            for (int i = 0; i < 8; ++i) h.v[i] = xv.v[i] + (acc.v[i] + tap(w[TAPS - 1], i) * xv.v[i]);
            if constexpr (F32) {
                dn_put(a.h, row * a.ldh * 4, there ? rowb : 0, c * 4, __builtin_bit_cast(u32x4_t, f32x4_t{h.v[0], h.v[1], h.v[2], h.v[3]}));
                dn_put(a.h, row * a.ldh * 4, there ? rowb : 0, c * 4 + 16, __builtin_bit_cast(u32x4_t, f32x4_t{h.v[4], h.v[5], h.v[6], h.v[7]}));
            } else {
                dn_put(a.h, row * a.ldh * 2, there ? rowb : 0, c * 2, u32x4_t{pack2bf(h.v[0], h.v[1]), pack2bf(h.v[2], h.v[3]), pack2bf(h.v[4], h.v[5]), pack2bf(h.v[6], h.v[7])});
            }
            const int e = qe - 1 - (int)row;  // tokens of the portion behind this one
            if (there && e < HALO && so >= 0 && so < a.n_state && dn_table(a.pos, row) >= 0) {
                dn_stf<true>(a.state + ((int64_t)so * HALO + (HALO - 1 - e)) * a.wp + c, xv, 8);
                if (e == 0)  // a portion shorter than the history: the older inputs move up
                    for (int i = 0; i < HALO - (qe - qs); ++i)
                        dn_stf<true>(a.state + ((int64_t)so * HALO + i) * a.wp + c, dn_ldf<true>(a.state + (sin * HALO + i + (qe - qs)) * a.wp + c, 8), 8);
            }
#pragma unroll
            for (int k = HALO; k >= 2; --k) hist[k - 1] = hist[k - 2];
            hist[0] = xv;
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) x[u] = xn[u];
    }
}

constexpr int64_t DN_SPLIT_ROWS = 512;   // rows from which norm and convolution are launches of their own
// and rows beyond one per sequence: a row in the middle of a portion computes the TAPS-1 in front of it as well, one after the other.  One launch / two, whole steps of four layers, us: two
// prompts of 150 and 131 1004 / 982, one of 500 1239 / 1209, 90 rows and 300 of prompts (4096 columns) 2850 / 2808; below, the host's launches take longer than the kernels: one prompt of
// 20 881 / 896, of 40 869 / 878, of 135 912 / 921, 60 rows and 40 of a prompt 944 / 950.
// The rows in front (their number times what one costs: one that is only read 1, a norm 2, with one depth 3, with more of them or with experts' rows 5) have to be worth the other launch, in
// which portions of one row wait for their states one after the other: 8, and 5 for rows of more than 256 threads.  One / two launches, us, 400 rows of four prompts, then of forty single rows
// and prompts: 2048 columns, four taps, a norm 9.9 / 9.9, 10.1 / 12.3, nothing in front 5.8 / 7.1, 6.0 / 9.9, one depth 14.5 / 10.7, 14.1 / 13.2, six experts 17.7 / 10.9, 17.5 / 13.5; two
// taps, a norm 7.1 / 8.8, 7.2 / 9.5, experts 10.0 / 9.6, 9.6 / 10.5; six taps, nothing 9.3 / 8.3, 10.1 / 13.2, a norm 19.7 / 11.2, 20.0 / 15.9; 4096 columns, four taps, a norm 16.9 / 13.0,
// 16.5 / 16.4, nothing 8.7 / 7.7, 9.0 / 10.8; two taps, experts, 512 rows 18.6 / 15.5, 18.3 / 16.6.
constexpr int64_t DN_SPLIT_EXTRA = 256;

// Rows of a run.  Four and more for 1024 workgroups, 16 at most: portions that begin inside a run wait for their state one after the other, and shorter runs read more
// rows twice.  16 rows / 512 workgroups / this / 2048, us: 15074 rows of 2048 38.3 / 38.3 / 38.3 / 41.3, 5000 of 4096 25.6 / 25.8 / 25.3 / 26.4, 700 of 2048 10.3 / 6.2 / 6.2 /
// 6.3, 40 single rows and 5400 of prompts 41.8 / 31.6 / 24.4 / 20.0, 60 and 5800 44.7 / 36.9 / 25.4 / 22.0.
// Longer ones with more than four taps, where a run of four begins with five to 31 rows of its own, for some long portions (single rows would wait in them):
//   - six and eight taps, for as many threads with columns as 512 workgroups of 2048 columns have.  The rule above / this, us: six taps, 3000 rows of 2048 13.0 / 11.6, of 4096
//     19.3 / 16.8, 5000 of 2048 17.6 / 14.7; eight, 3000 of 4096 23.3 / 19.5, 4000 of 2048 19.0 / 15.6, 7000 24.9 / 20.8; of 1024 columns both are the same to 4 %
//   - 16 and 32, for one workgroup per CU (its registers), whose rounds take as long as the run and two or three rows more: 16 taps, 1200 rows of 1024 18.2 / 13.4, 3000 of 2048
//     37.5 / 28.0 (runs of 16 32.0), 32 taps, 1500 of 2048 51.0 / 38.4, 4000 of 4096 167 / 144
template <int TAPS>
int depth_conv_run(int64_t T, int wp, int64_t seqs) {
    const int64_t cols = (wp + 2047) / 2048;
    auto even = [](int64_t per) { return (int)(per < 4 ? 4 : per > 16 ? 16 : (per + 1) / 2 * 2); };
    if (TAPS <= 4 || seqs > 8 || T < 128 * seqs) return even((T * cols + 1023) / 1024);
    if (TAPS <= 8) return even((T * wp + (1 << 20) - 1) >> 20);
    int best = 4;
    auto time = [&](int n) { return ((T + n - 1) / n * cols + 255) / 256 * (2 * n + 5); };
    for (int n = 6; n <= 16; n += 2)
        if (time(n) < time(best)) best = n;
    return best;
}

template <int TAPS>
int launch_depth_conv(const DepthArgs& a, int64_t seqs, const float* xs, hipStream_t st) {
    const int tr = depth_conv_run<TAPS>(a.T, a.wp, seqs);
    const dim3 grid((unsigned)((a.T + tr - 1) / tr), (unsigned)((a.wp + 2047) / 2048));
    if (a.act_f32) hipLaunchKernelGGL((depth_conv_kernel<TAPS, true>), grid, dim3(256), 0, st, a, xs, tr);
    else hipLaunchKernelGGL((depth_conv_kernel<TAPS, false>), grid, dim3(256), 0, st, a, xs, tr);
    GLM_CHECK_LAUNCH("glm_depth_norm(convolution)");
    return GLM_OK;
}

template <int TAPS>
int launch_depth_norm(const DepthArgs& a, int64_t seqs, int nt, bool vec, hipStream_t st) {
    if constexpr (TAPS > 1) {
        const float* xs = a.depth ? a.x_next : a.y ? a.x_out : a.x_in;
        const bool whole = glm_aligned16(xs) && glm_aligned16(a.h) && glm_aligned16(a.conv_w) && glm_aligned16(a.state);
        const int again = (TAPS - 1) * (!a.y ? 1 : a.pair_pos || (a.depth && a.n_depth > 1) ? 5 : a.depth && a.n_depth ? 3 : 2);
        if (xs && (a.T > DN_SPLIT_ROWS || (a.T >= seqs + DN_SPLIT_EXTRA && whole && again >= (nt > 256 ? 5 : 8)))) {
            if (a.y || a.depth || a.x_cast || a.x_out) {
                DepthArgs b = a;
                b.h = nullptr;
                const int rc = launch_depth_norm<1>(b, seqs, nt, vec, st);
                if (rc != GLM_OK) return rc;
            }
            return launch_depth_conv<TAPS>(a, seqs, xs, st);
        }
    }
    if constexpr (TAPS > 1 && TAPS <= 4) {
        // (a CU has room for eight waves of it: as long as the rows are one round.  Beyond / the form for 1024 threads, us, single rows: 257 of 3072 columns 11.5 / 9.5, 300 of 4096 14.8 / 12.9, behind
        // experts 17.6 / 15.9; 512 of 2048, still one round, 9.2 / 10.3)
        if (vec && nt <= 512 && a.T * (nt / 64) <= 8 * 256) {
            hipLaunchKernelGGL((depth_norm_kernel<TAPS, true, 512>), dim3((unsigned)a.T), dim3(nt), 0, st, a);
            GLM_CHECK_LAUNCH("glm_depth_norm");
            return GLM_OK;
        }
    }
    if (vec) hipLaunchKernelGGL((depth_norm_kernel<TAPS, true, 1024>), dim3((unsigned)a.T), dim3(nt), 0, st, a);
    else hipLaunchKernelGGL((depth_norm_kernel<TAPS, false, 1024>), dim3((unsigned)a.T), dim3(nt), 0, st, a);
    GLM_CHECK_LAUNCH("glm_depth_norm");
    return GLM_OK;
}

}  // namespace

extern "C" int glm_depth_norm_taps(int taps) {
    for (int t : {1, 2, 3, 4, 6, 8, 16, 32})
        if (taps >= 1 && taps <= t) return t;
    return -1;
}

extern "C" int glm_depth_norm(const float* x_in, const int32_t* row_index, int64_t ld, const void* y, int64_t ldy, const int32_t* pair_pos, const float* pair_w, int k, int64_t n_rows,
                              const float* g_post, float* x_out, void* x_cast, int64_t ldc, const float* depth, int64_t depth_stride, int n_depth, const float* coef, float* x_next,
                              const float* g_pre, const void* conv_w, int taps, float* state, int64_t n_state, const int32_t* pos, const int32_t* seq_of, const int32_t* q_start,
                              const int32_t* state_in, const int32_t* state_out, void* h, int64_t ldh, int act_f32, int64_t T, int width, int wp, int groups, float eps,
                              glm_stream_t stream) {
    return glm_depth_norm_portions(x_in, row_index, ld, y, ldy, pair_pos, pair_w, k, n_rows, g_post, x_out, x_cast, ldc, depth, depth_stride, n_depth, coef, x_next, g_pre, conv_w, taps, state,
                                   n_state, pos, seq_of, q_start, state_in, state_out, h, ldh, act_f32, T, T, width, wp, groups, eps, stream);
}

extern "C" int glm_depth_norm_portions(const float* x_in, const int32_t* row_index, int64_t ld, const void* y, int64_t ldy, const int32_t* pair_pos, const float* pair_w, int k, int64_t n_rows,
                              const float* g_post, float* x_out, void* x_cast, int64_t ldc, const float* depth, int64_t depth_stride, int n_depth, const float* coef, float* x_next,
                              const float* g_pre, const void* conv_w, int taps, float* state, int64_t n_state, const int32_t* pos, const int32_t* seq_of, const int32_t* q_start,
                              const int32_t* state_in, const int32_t* state_out, void* h, int64_t ldh, int act_f32, int64_t T, int64_t seqs, int width, int wp, int groups, float eps,
                              glm_stream_t stream) {
    GLM_CHECK_ARG(x_in && T >= 0 && width > 0 && wp >= width && wp % 8 == 0 && wp - width < 8 && ld >= wp && ld % 4 == 0 && groups > 0 && width % groups == 0, GLM_ERR_INVALID,
                  "glm_depth_norm: bad shape T=%ld width=%d wp=%d groups=%d ld=%ld", (long)T, width, wp, groups, (long)ld);
    GLM_CHECK_ARG(!y || (g_post && ldy >= wp && ldy % 8 == 0), GLM_ERR_INVALID, "glm_depth_norm: bad sublayer output (ldy=%ld)", (long)ldy);
    GLM_CHECK_ARG(!pair_pos || (y && pair_w && k > 0 && n_rows > 0), GLM_ERR_INVALID, "glm_depth_norm: bad expert rows (k=%d rows=%ld)", k, (long)n_rows);
    GLM_CHECK_ARG((!h || (ldh >= wp && ldh % 8 == 0)) && (!x_cast || (ldc >= wp && ldc % 8 == 0)), GLM_ERR_INVALID, "glm_depth_norm: bad output (ldh=%ld ldc=%ld)", (long)ldh, (long)ldc);
    GLM_CHECK_ARG(!depth || (coef && n_depth >= 0 && depth_stride >= 0 && depth_stride % 4 == 0), GLM_ERR_INVALID, "glm_depth_norm: bad depth rows (n=%d)", n_depth);
    GLM_CHECK_ARG(taps == 1 || (conv_w && h && !g_pre && state && n_state > 0 && pos && seq_of && q_start && state_in && state_out && !row_index && x_out != x_in && x_next != x_in),
                  GLM_ERR_INVALID, "glm_depth_norm: the convolution needs weights, state, positions and outputs apart from x_in");
    GLM_CHECK_ARG(taps >= 1 && glm_depth_norm_taps(taps) == taps, GLM_ERR_UNSUPPORTED, "glm_depth_norm: %d taps (see glm_depth_norm_taps)", taps);
    GLM_CHECK_ARG(T < (1ll << 31), GLM_ERR_UNSUPPORTED, "glm_depth_norm: too many rows");
    DepthArgs a = {x_in, row_index, ld, y, ldy, pair_pos, pair_w, k, n_rows, g_post, x_out, x_cast, ldc, depth, depth_stride, n_depth, coef, x_next, g_pre, (const bf16_t*)conv_w, state,
                   pos, seq_of, q_start, state_in, state_out, n_state, h, ldh, act_f32, T, width, wp, groups, width / groups, 64, 1, 1, 0, eps};
    int waves;
    if (a.gs > 512) {  // whole waves per part
        a.wpg = (a.gs + 511) / 512;
        a.cpw = ((a.gs + a.wpg - 1) / a.wpg + 7) / 8 * 8;
        waves = groups * a.wpg;
    } else {           // a power of two of lanes per part
        a.lpg = 1;
        while (a.lpg * 8 < a.gs) a.lpg *= 2;
        a.gpw = 64 / a.lpg;
        waves = (groups + a.gpw - 1) / a.gpw;
    }
    GLM_CHECK_ARG(waves <= 16, GLM_ERR_UNSUPPORTED, "glm_depth_norm: %d parts of %d columns need %d waves (16 at most)", groups, a.gs, waves);
    if (T == 0) return GLM_OK;
    const bool vec = a.gs % 8 == 0 && glm_aligned16(x_in) && glm_aligned16(y) && glm_aligned16(h) && glm_aligned16(x_cast) && glm_aligned16(depth);
    const int nt = waves * 64;
    hipStream_t st = glm_s(stream);
    switch (taps) {
        case 1: return launch_depth_norm<1>(a, seqs, nt, vec, st);
        case 2: return launch_depth_norm<2>(a, seqs, nt, vec, st);
        case 3: return launch_depth_norm<3>(a, seqs, nt, vec, st);
        case 4: return launch_depth_norm<4>(a, seqs, nt, vec, st);
        case 6: return launch_depth_norm<6>(a, seqs, nt, vec, st);
        case 8: return launch_depth_norm<8>(a, seqs, nt, vec, st);
        case 16: return launch_depth_norm<16>(a, seqs, nt, vec, st);
        default: return launch_depth_norm<32>(a, seqs, nt, vec, st);
    }
}
