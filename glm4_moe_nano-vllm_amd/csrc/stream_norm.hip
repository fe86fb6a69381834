// stream_norm.hip — what happens between two sublayers of a decoder whose residual is several parallel streams ("hyper-
// connections", fp32 throughout).  With the finished sublayer's output y and its matrices
//
//     x'_t = sum_s mix[s, t] x_s + out[t] * (scale . y)      all streams at once from the old ones     (optional: y)
//     u    = sum_s in[s] x'_s                                 what the next sublayer's norm reads
//     h    = u / rms(u) * gain                                RMS norm with ONE gain                     (optional: h)
//     h    = h + (h_prev - h) . shift                         token shift; h_prev: the previous token's h, zero for the first
//
// in ONE launch.  gfx950 only.  Roofline: HBM — the streams are read once and written once, y read once, h written once.
//
// A workgroup takes a run of rows one after the other; a thread owns VC columns of every stream, the next row's loads are in
// flight while a row is worked on, and one barrier per row carries the reduction.  The token shift needs the h of the row in
// front of the run: it is RECOMPUTED from x_in and y (no hand-off between workgroups, so x_out is another buffer than x_in), or
// read from the sequence's state row where the portion begins.  A step reads state row state_in and writes row state_out,
// because the workgroup that writes a portion's last h is not the one that reads the previous portion's.  A token's h is the
// same arithmetic whether it was computed in this step or kept from an earlier one.
#include "common.h"
#include <type_traits>

namespace {

struct StreamNormArgs {
    const float* x_in;        // element (row r, stream s, column c) at r*ldx + s*sx + c; sx = 0: all streams are the same row
    int64_t ldx, sx;
    const int32_t* row_index; // optional gather of x_in / y rows (no token shift, no x_out then)
    float* x_out;             // [T][S][wp] or nullptr
    const void* y;            // [T, ldy] or nullptr
    int64_t ldy;
    int y_f32;
    const float* y_scale;     // [wp]
    const float* mix_out;     // [S*S] mix[from*S + to], then [S] out
    const float* w_in;        // [S]
    float gain;
    const float* shift;       // [wp] or nullptr
    float* state;             // [n_state][wp]
    int64_t n_state;
    const int32_t* pos;       // [T] position of the row in its sequence (< 0: unused row)
    const int32_t* seq_of;    // [T]
    const int32_t* q_start;   // [n_seq+1]
    const int32_t *state_in, *state_out;  // [n_seq] (state_out < 0: keep nothing)
    void* h;                  // [T, ldh] or nullptr
    int64_t ldh;
    int h_f32;
    int64_t T;
    int S, width, wp;         // streams, true width (the mean's divisor), padded width (multiple of 8, zero padding)
    float eps;
};

__device__ __forceinline__ f32x4_t st_load4(const void* base, int64_t off, int f32) {
    if (f32) return *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(base) + off);
    const u32x2_t u = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const bf16_t*>(base) + off);
    return f32x4_t{bflo(u[0]), bfhi(u[0]), bflo(u[1]), bfhi(u[1])};
}
__device__ __forceinline__ float st_sumsq(const f32x4_t& v) { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]; }

// Tables that no launch changes while it reads them: through the scalar cache, so that a row's bookkeeping waits for no vector load or store
__device__ __forceinline__ int st_table(const int32_t* p, int64_t i) { return reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(p))[i]; }
// `bytes` of a row; nothing if there is no such buffer
__device__ __forceinline__ __amdgpu_buffer_rsrc_t st_row(const void* base, int64_t off, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(base) + off), 0, base ? bytes : 0, 0x00020000);
}

// S streams, NV vectors of four columns per thread, NT threads: wp <= 4 NV NT.  ANY: y or h may be fp32
template <int S, int NV, int NT, bool ANY>
__global__ __launch_bounds__(NT) void stream_norm_kernel(const StreamNormArgs a, int tr) {
    constexpr int NW = NT / 64, NTEMP = 2;   // NTEMP: cache policy bit of a store, not to be kept
    __shared__ float s_red[2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const int64_t r0 = (int64_t)blockIdx.x * tr, r1 = min(r0 + tr, a.T);
    const float inv_w = 1.0f / (float)a.width;
    const bool shifted = a.shift != nullptr, y_f32 = ANY && a.y_f32, h_f32 = ANY && a.h_f32;
    int s = 0, qs = 0, qe = 0, sin = 0, so = 0;
    auto sequence = [&](int64_t r) {
        s = st_table(a.seq_of, r);
        qs = st_table(a.q_start, s);
        qe = st_table(a.q_start, s + 1);
        sin = (int)min(max((int64_t)st_table(a.state_in, s), (int64_t)0), a.n_state - 1);
        so = st_table(a.state_out, s);
    };
    int64_t lo = r0;
    if (shifted) {
        sequence(r0);
        if (r0 > qs) lo = r0 - 1;
    }
    // vector j of this thread: columns 4 (tid + j NT) .. + 3; at: what a thread behind the row's end reads instead
    int col[NV], at[NV];
    bool on[NV];
    f32x4_t ys[NV], sh[NV], hist[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        col[j] = 4 * (tid + j * NT);
        on[j] = col[j] < a.wp;
        at[j] = min(col[j], a.wp - 4);
        ys[j] = a.y ? *reinterpret_cast<const f32x4_t*>(a.y_scale + at[j]) : zero;
        sh[j] = shifted ? *reinterpret_cast<const f32x4_t*>(a.shift + at[j]) : zero;
        hist[j] = zero;
    }
    float mix[S][S], wo[S], wi[S];
#pragma unroll
    for (int f = 0; f < S; ++f) {
        wi[f] = a.w_in ? a.w_in[f] : 0.f;
        wo[f] = a.y ? a.mix_out[S * S + f] : 0.f;
#pragma unroll
        for (int t = 0; t < S; ++t) mix[f][t] = a.y ? a.mix_out[f * S + t] : 0.f;
    }
    using Y = typename std::conditional<ANY, f32x4_t, u32x2_t>::type;   // y as it was read
    auto load_row = [&](int64_t r, f32x4_t (&x)[S][NV], Y (&y)[NV]) __attribute__((always_inline)) {
        const int64_t row = a.row_index ? st_table(a.row_index, r) : r;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
#pragma unroll
            for (int t = 0; t < S; ++t) x[t][j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(a.x_in + row * a.ldx + t * a.sx + at[j]));
        }
        if (a.y) {
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                if constexpr (ANY) y[j] = st_load4(a.y, row * a.ldy + at[j], y_f32);
                else y[j] = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const bf16_t*>(a.y) + row * a.ldy + at[j]);
            }
        }
    };
    auto value = [](const Y& y, int i) -> float {
        if constexpr (ANY) return y[i];
        else return i & 1 ? bfhi(y[i >> 1]) : bflo(y[i >> 1]);
    };
    f32x4_t x[S][NV], xn[S][NV];
    Y y[NV], yn[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        y[j] = yn[j] = Y{};
#pragma unroll
        for (int t = 0; t < S; ++t) x[t][j] = xn[t][j] = zero;
    }
    load_row(lo, x, y);
    // Every store of a turn is issued whatever the launch has (buffers that there are not: of no length), and y stays as it was read until it is used, so that a turn waits
    // for the loads of the one before it and not for its stores.  (It unpacked y where it read it, read the sequence tables for every row and stored under tests, and so waited
    // for everything it had just asked for.)  In a step, two streams, us, that / this: 11137 rows of 2048 102 / 80 with a token shift, 84 / 75 without, without y 53 / 37;
    // 5500 61 / 41, 44 / 36; 4600 of 4096 77 / 68, 70 / 64; 700 of 2048 11.9 / 10.3.
    // (What was requested so far is waited for here: a wait in the loop counts what is behind a load on every way to it.)
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        asm volatile("" : "+v"(y[j]), "+v"(ys[j]), "+v"(sh[j]));
#pragma unroll
        for (int t = 0; t < S; ++t) asm volatile("" : "+v"(x[t][j]));
    }
    int par = 0;
    for (int64_t r = lo; r < r1; ++r) {
        if (r + 1 < r1) load_row(r + 1, xn, yn);
        const bool mine = r >= r0;
        float sq = 0.f;
        f32x4_t u[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            if (a.y) {
                f32x4_t v[S];
#pragma unroll
                for (int t = 0; t < S; ++t) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float acc = wo[t] * (ys[j][i] * value(y[j], i));
#pragma unroll
                        for (int f = 0; f < S; ++f) acc = fmaf(mix[f][t], x[f][j][i], acc);
                        v[t][i] = acc;
                    }
                }
#pragma unroll
                for (int t = 0; t < S; ++t) x[t][j] = v[t];
            }
            u[j] = zero;
#pragma unroll
            for (int t = 0; t < S; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) u[j][i] = fmaf(wi[t], x[t][j][i], u[j][i]);
            sq += on[j] ? st_sumsq(u[j]) : 0.f;
        }
#pragma unroll
        for (int t = 0; t < S; ++t) {
            const __amdgpu_buffer_rsrc_t rs = st_row(a.x_out, (r * S + t) * a.wp * 4, mine ? a.wp * 4 : 0);
#pragma unroll
            for (int j = 0; j < NV; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, x[t][j]), rs, col[j] * 4, 0, NTEMP);
        }
        f32x4_t o[NV];
        if (a.h) {
            sq = wave_sum(sq);
            if constexpr (NW > 1) {
                if (lane == 0) s_red[par][wid] = sq;
                __syncthreads();
                sq = 0.f;
#pragma unroll
                for (int w = 0; w < NW; ++w) sq += s_red[par][w];
                par ^= 1;
            }
            const float rms = sqrtf(sq * inv_w + a.eps), f = a.gain / rms;
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[j][i] = u[j][i] * f;
            if (shifted) {
                if (r == qe) sequence(r);  // the next sequence's portion begins
                if (r == qs) {
                    // first token of its sequence: whatever the state row holds is not its
                    const bool fresh = st_table(a.pos, r) <= 0;
#pragma unroll
                    for (int j = 0; j < NV; ++j) hist[j] = fresh ? zero : *reinterpret_cast<const f32x4_t*>(a.state + (int64_t)sin * a.wp + at[j]);
#pragma unroll
                    for (int j = 0; j < NV; ++j) asm volatile("" : "+v"(hist[j]));   // (waited for here, not in every turn)
                }
                const bool keep = mine && r == qe - 1 && so >= 0 && so < a.n_state && st_table(a.pos, r) >= 0;
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    const f32x4_t hv = o[j];
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[j][i] = fmaf(hist[j][i] - hv[i], sh[j][i], hv[i]);
                    hist[j] = hv;
                    if (keep && on[j]) *reinterpret_cast<f32x4_t*>(a.state + (int64_t)so * a.wp + col[j]) = hv;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < NV; ++j) o[j] = zero;
        }
        const __amdgpu_buffer_rsrc_t rs = st_row(a.h, r * a.ldh * (h_f32 ? 4 : 2), mine ? a.wp * (h_f32 ? 4 : 2) : 0);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            if (h_f32) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o[j]), rs, col[j] * 4, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{pack2bf(o[j][0], o[j][1]), pack2bf(o[j][2], o[j][3])}, rs, col[j] * 2, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            y[j] = yn[j];
#pragma unroll
            for (int t = 0; t < S; ++t) x[t][j] = xn[t][j];
        }
    }
}

// any number of streams and any width: one row per workgroup, rows read again for every use
constexpr int SW_NT = 256;
__global__ __launch_bounds__(SW_NT) void stream_norm_any_kernel(const StreamNormArgs a) {
    __shared__ float s_red[SW_NT / 64];
    const int tid = threadIdx.x, S = a.S;
    const int64_t r = blockIdx.x;
    const float inv_w = 1.0f / (float)a.width;
    auto stream = [&](int64_t row, int t, int c) {  // x'_t at column c
        float v = 0.f;
        if (!a.y) return a.x_in[row * a.ldx + t * a.sx + c];
        const float yv = a.y_f32 ? reinterpret_cast<const float*>(a.y)[row * a.ldy + c] : bf2f(reinterpret_cast<const bf16_t*>(a.y)[row * a.ldy + c]);
        v = a.mix_out[S * S + t] * (a.y_scale[c] * yv);
        for (int f = 0; f < S; ++f) v = fmaf(a.mix_out[f * S + t], a.x_in[row * a.ldx + f * a.sx + c], v);
        return v;
    };
    auto collapsed = [&](int64_t row, int c) {
        float u = 0.f;
        for (int t = 0; t < S; ++t) u = fmaf(a.w_in[t], stream(row, t, c), u);
        return u;
    };
    auto factor = [&](int64_t row) {
        float sq = 0.f;
        for (int c = tid; c < a.wp; c += SW_NT) {
            const float u = collapsed(row, c);
            sq += u * u;
        }
        sq = wave_sum(sq);
        __syncthreads();
        if ((tid & 63) == 0) s_red[tid >> 6] = sq;
        __syncthreads();
        sq = 0.f;
        for (int w = 0; w < SW_NT / 64; ++w) sq += s_red[w];
        return a.gain / sqrtf(sq * inv_w + a.eps);
    };
    const int64_t row = a.row_index ? a.row_index[r] : r;
    if (a.x_out)
        for (int c = tid; c < a.wp; c += SW_NT)
            for (int t = 0; t < S; ++t) a.x_out[(r * S + t) * a.wp + c] = stream(row, t, c);
    if (!a.h) return;
    int s = 0;
    bool from_row = false, from_state = false;
    int64_t so = -1, sin = 0;
    if (a.shift) {
        s = a.seq_of[r];
        from_row = r > a.q_start[s];
        from_state = !from_row && a.pos[r] > 0;
        sin = min(max((int64_t)a.state_in[s], (int64_t)0), a.n_state - 1);
        if (r == a.q_start[s + 1] - 1 && a.pos[r] >= 0) so = a.state_out[s];
    }
    const float f = factor(row), fp = from_row ? factor(row - 1) : 0.f;
    for (int c = tid; c < a.wp; c += SW_NT) {
        const float hv = collapsed(row, c) * f;
        float o = hv;
        if (a.shift) {
            const float prev = from_row ? collapsed(row - 1, c) * fp : from_state ? a.state[sin * a.wp + c] : 0.f;
            o = fmaf(prev - hv, a.shift[c], hv);
            if (so >= 0 && so < a.n_state) a.state[so * a.wp + c] = hv;
        }
        if (a.h_f32) reinterpret_cast<float*>(a.h)[r * a.ldh + c] = o;
        else reinterpret_cast<bf16_t*>(a.h)[r * a.ldh + c] = f2bf(o);
    }
}

template <int S, int NV, int NT>
int launch_stream(const StreamNormArgs& a, hipStream_t st) {
    // decode: one row per workgroup; else runs of rows long enough to spread the halo, short enough to fill the chip
    constexpr int WGS = NT >= 512 ? 512 : 4096 / (NT / 64) > 2048 ? 2048 : 4096 / (NT / 64);   // four waves on every SIMD
    // (of eight rows at least / of four, two streams of 2048, us: 40 single rows and 5400 of prompts 40.7 / 37.2, 36.6 / 33.3 without a shift, 3000 rows 25.9 / 23.6, 24.1 / 20.9)
    int tr = a.T <= 512 ? 1 : (int)((a.T + WGS - 1) / WGS);
    const bool any = (a.y && a.y_f32) || (a.h && a.h_f32);
    if (tr > 1) {
        tr = tr < 4 ? 4 : tr > 32 ? 32 : tr;
        // Runs of eight rows at least where those of four are more workgroups than there is room for at once (registers: four waves on a SIMD, three with eight streams) and take as many turns,
        // us, four / eight: eight streams of 4096, 1200 rows 96.8 / 82.1 with a shift, 83.9 / 73.4, 3000 166 / 155, 145 / 142.
        const int64_t fit = 256 * ((S == 8 && (NT <= 256 || (NT == 512 && any)) ? 12 : 16) / (NT / 64));
        auto turns = [&](int n) { return ((a.T + n - 1) / n + fit - 1) / fit * (n + (a.shift ? 1 : 0)); };
        if (tr < 8 && turns(8) <= turns(tr)) tr = 8;
    }
    const dim3 grid((unsigned)((a.T + tr - 1) / tr));
    if (any) hipLaunchKernelGGL((stream_norm_kernel<S, NV, NT, true>), grid, dim3(NT), 0, st, a, tr);
    else hipLaunchKernelGGL((stream_norm_kernel<S, NV, NT, false>), grid, dim3(NT), 0, st, a, tr);
    GLM_CHECK_LAUNCH("glm_stream_norm");
    return GLM_OK;
}

template <int S>
int launch_stream_width(const StreamNormArgs& a, hipStream_t st) {
    constexpr int NV = S <= 3 ? 2 : 1;
    constexpr int PER = 4 * NV;
    if (a.wp <= 64 * PER) return launch_stream<S, NV, 64>(a, st);
    if (a.wp <= 128 * PER) return launch_stream<S, NV, 128>(a, st);
    if (a.wp <= 256 * PER) return launch_stream<S, NV, 256>(a, st);
    if (a.wp <= 512 * PER) return launch_stream<S, NV, 512>(a, st);
    if (a.wp <= 1024 * PER) return launch_stream<S, NV, 1024>(a, st);
    hipLaunchKernelGGL(stream_norm_any_kernel, dim3((unsigned)a.T), dim3(SW_NT), 0, st, a);
    GLM_CHECK_LAUNCH("glm_stream_norm");
    return GLM_OK;
}

}  // namespace

extern "C" int glm_stream_norm(const float* x_in, int64_t ldx, int64_t sx, const int32_t* row_index, float* x_out, const void* y, int64_t ldy, int y_f32,
                               const float* y_scale, const float* mix_out, const float* w_in, float gain, const float* shift, float* state, int64_t n_state,
                               const int32_t* pos, const int32_t* seq_of, const int32_t* q_start, const int32_t* state_in, const int32_t* state_out, void* h,
                               int64_t ldh, int h_f32, int64_t T, int S, int width, int wp, float eps, glm_stream_t stream) {
    GLM_CHECK_ARG(x_in && T >= 0 && T < (1ll << 31) && S >= 1 && width > 0 && wp >= width && wp % 8 == 0 && ldx >= wp && ldx % 4 == 0 && sx >= 0 && sx % 4 == 0 &&
                      (sx == 0 || (sx >= wp && ldx >= S * sx)), GLM_ERR_INVALID,
                  "glm_stream_norm: bad shape T=%ld S=%d width=%d wp=%d ldx=%ld sx=%ld", (long)T, S, width, wp, (long)ldx, (long)sx);
    GLM_CHECK_ARG(!y || (y_scale && mix_out && ldy >= wp && ldy % 4 == 0), GLM_ERR_INVALID, "glm_stream_norm: bad sublayer output (ldy=%ld)", (long)ldy);
    GLM_CHECK_ARG((x_out || h) && (!h || (w_in && ldh >= wp && ldh % 4 == 0)), GLM_ERR_INVALID, "glm_stream_norm: bad output (ldh=%ld)", (long)ldh);
    GLM_CHECK_ARG(x_out != x_in && !(row_index && x_out), GLM_ERR_INVALID, "glm_stream_norm: x_out must be apart from x_in, and gathered rows have none");
    GLM_CHECK_ARG(!shift || (h && state && n_state > 0 && pos && seq_of && q_start && state_in && state_out && !row_index), GLM_ERR_INVALID,
                  "glm_stream_norm: the token shift needs h, state and positions");
    if (T == 0) return GLM_OK;
    StreamNormArgs a = {x_in, ldx, sx, row_index, x_out, y, ldy, y_f32, y_scale, mix_out, w_in, gain, shift, state, n_state, pos, seq_of, q_start, state_in, state_out,
                        h, ldh, h_f32, T, S, width, wp, eps};
    hipStream_t st = glm_s(stream);
    switch (S) {
        case 1: return launch_stream_width<1>(a, st);
        case 2: return launch_stream_width<2>(a, st);
        case 3: return launch_stream_width<3>(a, st);
        case 4: return launch_stream_width<4>(a, st);
        case 5: return launch_stream_width<5>(a, st);
        case 6: return launch_stream_width<6>(a, st);
        case 8: return launch_stream_width<8>(a, st);
        default: break;
    }
    hipLaunchKernelGGL(stream_norm_any_kernel, dim3((unsigned)T), dim3(SW_NT), 0, st, a);
    GLM_CHECK_LAUNCH("glm_stream_norm");
    return GLM_OK;
}
