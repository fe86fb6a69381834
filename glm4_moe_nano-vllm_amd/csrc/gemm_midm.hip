// gemm_midm.hip — bf16 projections of some dozen to some hundred rows per weight matrix: batched decode of many sequences, short
// prompts, the experts of a short prompt.  gfx950 only.
//
// What bounds it: the weights are still read once and dominate the HBM bytes, but an output tile must be small for the grid to cover
// the chip, and every workgroup pulls its own activation and weight rows through L2 -> LDS, some 32 bytes per clock and CU: the tile is
// chosen for that traffic and for the number of workgroups (midm_tile_of), from 32 rows x 16 weight rows up to 128 x 128.
//   * a stage = one 64-wide K chunk of the tile's activation and weight rows, a whole 128-byte line per row (with 32-wide chunks, half
//     lines: 14336 x 4096 at 128 rows 53 instead of 45 us, 4096 x 12288 at 64 rows 60 instead of 45);
//   * 16-byte pieces are swizzled at the source, piece ^ ((row >> 1) & 7): the 16 rows of a fragment read cover all banks;
//   * the fragments of a k-step are read under the MFMAs of the one before;
//   * workgroups that share weight rows sit on one XCD, next to one another, and every XCD has as many.
// Two bodies.  Split (few tiles, a long K, experts): the waves split K, not the tile.  A wave computes the whole output tile over its own
// chunks, every staged byte is read from LDS exactly once, and there is no workgroup barrier in the loop: a wave waits for its own DMA only
// (counted vmcnt) and refills a stage once it is in registers; the partial tiles are summed through LDS in wave order, each wave finishes its
// share of the rows.  Shared (more tiles): the waves split the tile over one ring of three or four stages with a barrier per stage; no ring per
// wave, so the tile can be larger and a stage's bytes serve more MFMAs.  14336 x 4096 at 64 rows 37 -> 28 us, at 128 56 -> 38, at 211 61 -> 43,
// 4096 x 4096 at 1000 rows 58 -> 43 (tiled), 10944 gated columns x 4096 at 64 rows 53 -> 43.
#include "gemm_internal.h"
#include "gemm_epilogue.h"
#include <type_traits>

namespace {

typedef __attribute__((address_space(3))) void mm_lds_void;
typedef __attribute__((address_space(1))) const void mm_glb_void;

constexpr int MM_KC = 64;     // K columns of a stage
constexpr int MM_ROWB = 128;  // bytes of a staged row

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mm_rsrc(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}
template <int OFF>
__device__ __forceinline__ void mm_lds_read(u32x4_t& dst, unsigned addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}

template <int MT, int RT>
struct MmFrags {                       // one k-step of 32 columns
    u32x4_t w[RT], x[MT];
    template <int I>
    __device__ __forceinline__ void read_w(unsigned a) {
        mm_lds_read<I * 2048>(w[I], a);
        if constexpr (I + 1 < RT) read_w<I + 1>(a);
    }
    template <int I>
    __device__ __forceinline__ void read_x(unsigned a) {
        mm_lds_read<(RT + I) * 2048>(x[I], a);
        if constexpr (I + 1 < MT) read_x<I + 1>(a);
    }
    __device__ __forceinline__ void read(unsigned a) {
        read_w<0>(a);
        read_x<0>(a);
    }
    // every read has arrived; the registers pass through, so that no use moves above the wait
    __device__ __forceinline__ void settle() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < RT; ++i) asm volatile("" : "+v"(w[i]));
#pragma unroll
        for (int i = 0; i < MT; ++i) asm volatile("" : "+v"(x[i]));
    }
};

template <int MT, int RT>
struct MmShared : MmFrags<MT, RT> {    // the same out of a shared stage: the wave's weight rows and activation rows apart
    template <int I>
    __device__ __forceinline__ void read_rows(unsigned a) {
        mm_lds_read<I * 2048>(this->x[I], a);
        if constexpr (I + 1 < MT) read_rows<I + 1>(a);
    }
    __device__ __forceinline__ void read(unsigned aw, unsigned ax) {
        this->template read_w<0>(aw);
        read_rows<0>(ax);
    }
};

// The QKV projection's epilogue (glm_gemm_qkv_rope_store) on T row tiles out of one half of a head, tile t's columns from ncol0 + sub +
// 64 t / T: bias, rounding of the packed value, rotation of the first half's columns i and i + 32 (row tiles t and t + T / 2 in the same
// lane), rows of q / k / v and of the caches.  The tiled kernel's arithmetic and rounding points, so the fused launch stays bit-identical to
// the projection and the split kernel.
template <int T, int MPW>
__device__ __forceinline__ void midm_qkv_rows(const GemmParams& p, const f32x4_t (&acc)[T][MPW], int m0, int mcnt, int ncol0, int sub, int c, int g4) {
    constexpr int TC = 64 / T;   // columns from tile to tile
    const int nh = p.qkv_nh, nkv = p.qkv_nkv, head = ncol0 >> 7, half = (ncol0 >> 6) & 1;
    const bool is_q = head < nh, is_k = !is_q && head < nh + nkv;
    const int kh = is_q ? head : is_k ? head - nh : head - nh - nkv;
    bf16_t* dense = is_q ? p.qkv_q : is_k ? p.qkv_k : p.qkv_v;
    bf16_t* cache = is_q ? nullptr : is_k ? p.qkv_kc : p.qkv_vc;
    const int64_t ldd = (int64_t)(is_q ? nh : nkv) * 128;
#pragma unroll
    for (int j = 0; j < MPW; ++j) {
        const int row = 16 * j + c;
        if (row >= mcnt) continue;
        const int64_t m = m0 + row;
        float o[T][4];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int n = ncol0 + sub + TC * t + 4 * g4;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[t][r] = rbf(acc[t][j][r] + (p.bias ? bf2f(p.bias[n + r]) : 0.0f));
        }
        if (half == 0 && (is_q || is_k)) {
            const float* cs = p.qkv_cs + p.qkv_pos[m] * 64 + sub;
#pragma unroll
            for (int t = 0; t < T / 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float cv = cs[TC * t + 4 * g4 + r], sv = cs[32 + TC * t + 4 * g4 + r], x1 = o[t][r], x2 = o[t + T / 2][r];
                    o[t][r] = x1 * cv - x2 * sv;
                    o[t + T / 2][r] = x2 * cv + x1 * sv;
                }
        }
        int64_t slot = -1;
        if (cache != nullptr && p.qkv_slots != nullptr) slot = p.qkv_slots[m];
        const bool to_cache = slot >= 0 && slot < p.qkv_nslots;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const u32x2_t v = {pack2bf(o[t][0], o[t][1]), pack2bf(o[t][2], o[t][3])};
            const int col = kh * 128 + 64 * half + sub + TC * t + 4 * g4;
            if (dense != nullptr) *reinterpret_cast<u32x2_t*>(dense + m * ldd + col) = v;
            if (to_cache) *reinterpret_cast<u32x2_t*>(cache + slot * nkv * 128 + col) = v;
        }
    }
}

// rows m0 .. m0 + mcnt - 1, columns from ncol0; MT 16-row activation tiles, RT 16-row weight tiles
// (BYROW: only so that the two kernels have a body each, which the compiler wants)
template <int MODE, int MT, int RT, int NW, int NST, bool BYROW>
__device__ __forceinline__ void midm_body(const GemmParams& p, char* smem, int m0, int mcnt, int ncol0) {
    constexpr int D = 2 * (MT + RT);           // DMA instructions of a stage
    constexpr int STAGE = D * 1024;
    constexpr int HALF = 8 * RT;               // paired modes: gate rows of the tile, then as many up rows
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g4 = lane >> 4;
    const unsigned ring = (unsigned)(uintptr_t)(const mm_lds_void*)smem + wid * NST * STAGE;
    char* ringp = smem + wid * NST * STAGE;

    // ---- sources: instruction i brings rows 8 i + (lane >> 3), piece lane & 7 of the LDS row
    const int r8 = lane >> 3, pc = lane & 7;
    const __amdgpu_buffer_rsrc_t wrs = mm_rsrc(p.w), xrs = mm_rsrc(p.x);
    unsigned wvo[2 * RT], xvo[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int row = 8 * i + r8;
        const int wr = gemm_paired(MODE) ? (row < HALF ? 0 : p.N) + min(ncol0 + (row < HALF ? row : row - HALF), p.N - 1) : min(ncol0 + row, p.N - 1);
        wvo[i] = ((unsigned)wr * (unsigned)p.ldw + (pc ^ ((row >> 1) & 7)) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = m0 + min(8 * i + r8, mcnt - 1);   // rows past the end repeat the last one; they are never stored
        xvo[i] = ((unsigned)row * (unsigned)p.ldx + (pc ^ (((8 * i + r8) >> 1) & 7)) * 8) * 2u;
    }
    // ---- this wave's chunks: wid, wid + NW, ... of the K columns
    const int n = max(0, (p.K / MM_KC - wid + NW - 1) / NW);
    auto issue = [&](int j, int slot) {
        char* st = ringp + slot * STAGE;
        const int soff = (j * NW + wid) * MM_ROWB;
#pragma unroll
        for (int i = 0; i < 2 * RT; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (mm_lds_void*)(st + i * 1024), 16, wvo[i], soff, 0, 0);
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (mm_lds_void*)(st + (2 * RT + i) * 1024), 16, xvo[i], soff, 0, 0);
    };
    // stage j has arrived, the younger ones stay in flight
    auto arrived = [&](int j) {
        if (j + NST <= n) asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NST - 1) * D) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    f32x4_t acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    unsigned rel[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) rel[ks] = c * MM_ROWB + (((4 * ks + g4) ^ ((c >> 1) & 7)) << 4);
    auto mm = [&](const MmFrags<MT, RT>& f) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f.w[rt]), __builtin_bit_cast(bf16x8_t, f.x[mt]), acc[rt][mt], 0, 0, 0);
    };
    if (n > 0) {
#pragma unroll
        for (int j = 0; j < NST; ++j)
            if (j < n) issue(j, j);
        MmFrags<MT, RT> f0, f1;        // the two k-steps of a stage
        int slot = 0;
        arrived(0);
        f0.read(ring + rel[0]);
        f0.settle();
        for (int j = 0; j < n; ++j) {
            f1.read(ring + slot * STAGE + rel[1]);
            __builtin_amdgcn_sched_barrier(0);
            mm(f0);
            f1.settle();               // the stage is in registers: its slot takes chunk j + NST
            if (j + NST < n) issue(j + NST, slot);
            slot = slot + 1 == NST ? 0 : slot + 1;
            if (j + 1 < n) {
                arrived(j + 1);
                f0.read(ring + slot * STAGE + rel[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            mm(f1);
            if (j + 1 < n) f0.settle();
        }
    }

    // ---- sum of the waves' tiles, in wave order; wave w finishes row tiles w MT / NW .. (more waves than tiles: the first MT waves one each)
    constexpr int MPW = MT < NW ? 1 : MT / NW;
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            *reinterpret_cast<f32x4_t*>(red + (((wid * MT + mt) * RT + rt) * 64 + lane) * 4) = acc[rt][mt];
    __syncthreads();
    if (MT < NW && wid >= MT) return;
    f32x4_t sum[RT][MPW];
#pragma unroll
    for (int j = 0; j < MPW; ++j)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            f32x4_t s = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; ++w)
                s += *reinterpret_cast<const f32x4_t*>(red + (((w * MT + wid * MPW + j) * RT + rt) * 64 + lane) * 4);
            sum[rt][j] = s;
        }
    const int first = 16 * MPW * wid;
    if (first >= mcnt) return;
    if constexpr (MODE == GEMM_PLAIN && RT == 4) {
        if (p.qkv_q != nullptr) {
            midm_qkv_rows<4, MPW>(p, sum, m0 + first, mcnt - first, ncol0, 0, c, g4);
            return;
        }
    }
    // (behind the waves' tiles: nobody else's)
    f32x4_t* own = reinterpret_cast<f32x4_t*>(smem) + (NW * MT + wid * MPW) * RT * 64 + lane;
    gemm_row_epilogue<MODE, RT, MPW, true>(p, sum, 0, m0 + first, mcnt - first, ncol0, c, g4, own);
}

// row block and column tile of this workgroup
__device__ __forceinline__ void midm_tile(int mblocks, int interleaved, int& m, int& ntile) {
    if (interleaved) {   // column tiles dealt to the XCDs (workgroups b, b + 8, ...) one by one, their row blocks behind one another
        const int q = blockIdx.x >> 3;
        m = q % mblocks;
        ntile = q / mblocks * 8 + (blockIdx.x & 7);
    } else {             // few column tiles: an XCD takes a run of all tiles
        const int lin = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
        ntile = lin / mblocks;
        m = lin % mblocks;
    }
}

template <int MODE, int MT, int RT, int NW, int NST>
constexpr int midm_lds() {
    constexpr int MPW = MT < NW ? 1 : MT / NW, ring = NW * NST * (MT + RT) * 2048, red = (NW * MT + (MT < NW ? MT : NW) * MPW) * RT * 1024;
    return ring > red ? ring : red;
}

// BYROW: an XCD takes a run of all tiles row block by row block; interleaved is the number of column tiles
template <int MODE, int MT, int RT, int NW, int NST, bool BYROW>
__global__ __launch_bounds__(NW * 64) void gemm_midm_kernel(const GemmParams p, int mblocks, int interleaved) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int COLS = gemm_paired(MODE) ? 8 * RT : 16 * RT;
    int m, ntile;
    if constexpr (BYROW) {
        midm_tile(interleaved, 0, ntile, m);
        if (m >= mblocks) return;
    } else midm_tile(mblocks, interleaved, m, ntile);
    const int m0 = m * (16 * MT);
    if (ntile * COLS >= p.N) return;
    midm_body<MODE, MT, RT, NW, NST, BYROW>(p, smem, m0, min(16 * MT, (int)p.R - m0), ntile * COLS);
}

#if GLM_EXPERTS
// The split body for experts: rows m0 .. m0 + mcnt - 1 of group grp, 64 weight rows, two waves and two workgroups per CU, so that one is at work
// while the other starts or sums up.  MT: 16-row activation tiles, two where the rows are no more (the chip then moves half as many activation
// bytes as weight bytes, not as many).  once: no other row block reads these weights, which then leave the caches to the activations (nt; with
// several blocks it costs a tenth).  A wave sends the other one the half of its partial tile that it does not finish, and everything that the
// end needs is loaded before the stream.  65 experts of 1408 x 4096, gate|up / down, us: 211 tokens 270 / 155 (without all this) -> 247 / 142, 350
// 294 / 165 -> 277 / 161, 600 477 / 236 -> 465 / 220; 64 of 1024 x 2048 at 300 tokens 109 / 63 -> 106 / 60.  Not taken: 32 weight rows (278 / 154 at
// 211 tokens) or 128 (248 / 147), a third stage (equal), one wave (264 / 151), two or four column tiles as one stream (253 / 149, 300 / 168).
// Registers are held to what lets two waves share a SIMD: with all that one wave may have the compiler took 260, accumulators moved in and out of the
// far half of them in the loop.  Without / with that bound, gate|up, rows alike: 40 per expert of 64 of 1024 x 2048 122 / 110, of 9 of 2048 x 4096
// 85 / 72, 28 of 257 of 512 x 2048 220 / 193, of 65 of 1408 x 4096 280 / 261; down 40 of 64 of 1024 x 2048 61.2 / 59.8.
template <int MODE, int MT>
__device__ __forceinline__ void midm_expert_body(const GemmParams& p, char* smem, int grp, int m0, int mcnt, int ncol0, bool once, int reach) {
    constexpr int RT = 4, NW = 2, NST = 2, D = 2 * (MT + RT), STAGE = D * 1024, MPW = MT / NW;
    constexpr int HALF = 8 * RT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g4 = lane >> 4;
    const unsigned ring = (unsigned)(uintptr_t)(const mm_lds_void*)smem + wid * NST * STAGE;
    char* ringp = smem + wid * NST * STAGE;
    const int r8 = lane >> 3, pc = lane & 7;
    const __amdgpu_buffer_rsrc_t wrs = mm_rsrc(p.w + (int64_t)grp * p.w_gstride), xrs = mm_rsrc(p.x);
    unsigned wvo[2 * RT], xvo[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int row = 8 * i + r8;
        const int wr = gemm_paired(MODE) ? (row < HALF ? 0 : p.N) + min(ncol0 + (row < HALF ? row : row - HALF), p.N - 1) : min(ncol0 + row, p.N - 1);
        wvo[i] = ((unsigned)wr * (unsigned)p.ldw + (pc ^ ((row >> 1) & 7)) * 8) * 2u;
    }
    const int n = max(0, (p.K / MM_KC - wid + NW - 1) / NW);   // this wave's chunks: wid, wid + NW, ...
    auto issue_w = [&](auto ntc, int j, int slot) {
        const int soff = (j * NW + wid) * MM_ROWB;
#pragma unroll
        for (int i = 0; i < 2 * RT; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (mm_lds_void*)(ringp + slot * STAGE + i * 1024), 16, wvo[i], soff, 0, decltype(ntc)::value ? 2 : 0);
    };
    int last = 0;
    auto source = [&](int i) {
        const int m = m0 + min(8 * i + r8, mcnt - 1);   // rows past the end repeat the last one; they are never stored
        return MODE == GEMM_GATEUP && p.src ? p.src[m] : m;
    };
    auto issue_x = [&](auto far_rows, int j, int slot) {
        const int soff = (j * NW + wid) * MM_ROWB;
        char* st = ringp + slot * STAGE + 2 * RT * 1024;
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) {
            if constexpr (decltype(far_rows)::value)
                __builtin_amdgcn_global_load_lds((mm_glb_void*)(p.x + (int64_t)source(i) * p.ldx + (pc ^ (((8 * i + r8) >> 1) & 7)) * 8 + soff / 2),
                                                 (mm_lds_void*)(st + i * 1024), 16, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (mm_lds_void*)(st + i * 1024), 16, xvo[i], soff, 0, 0);
        }
    };
    if (n > 0) {   // (ahead of the wait for the row numbers)
        if (once) issue_w(std::true_type{}, 0, 0);
        else issue_w(std::false_type{}, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int src = source(i);
        xvo[i] = ((unsigned)src * (unsigned)p.ldx + (pc ^ (((8 * i + r8) >> 1) & 7)) * 8) * 2u;
        last = max(last, src);
    }
    float sc[MPW];   // of this wave's rows; a load inside the stream would wait behind every DMA in flight
    const bool scaled = MODE == GEMM_DOWN && grp < p.n_scaled;
#pragma unroll
    for (int j = 0; j < MPW; ++j) {
        const int row = 16 * (MPW * wid + j) + c;
        sc[j] = scaled && row < mcnt ? bf2f(p.scale[m0 + row]) : 1.0f;
        asm volatile("" : "+v"(sc[j]));
    }
    unsigned rel[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) rel[ks] = c * MM_ROWB + (((4 * ks + g4) ^ ((c >> 1) & 7)) << 4);
    f32x4_t acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto mm = [&](const MmFrags<MT, RT>& f) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f.w[rt]), __builtin_bit_cast(bf16x8_t, f.x[mt]), acc[rt][mt], 0, 0, 0);
    };
    auto stream = [&](auto far_rows, auto ntc) {
        auto arrived = [&](int j) {    // stage j has, the younger ones stay in flight
            if (j + NST <= n) asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NST - 1) * D) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        };
#pragma unroll
        for (int j = 0; j < NST; ++j)
            if (j < n) {
                if (j > 0) issue_w(ntc, j, j);
                issue_x(far_rows, j, j);
            }
        MmFrags<MT, RT> f0, f1;        // the two k-steps of a stage
        int slot = 0;
        arrived(0);
        f0.read(ring + rel[0]);
        f0.settle();
        for (int j = 0; j < n; ++j) {
            f1.read(ring + slot * STAGE + rel[1]);
            __builtin_amdgcn_sched_barrier(0);
            mm(f0);
            f1.settle();               // the stage is in registers: its slot takes chunk j + NST
            if (j + NST < n) {
                issue_w(ntc, j + NST, slot);
                issue_x(far_rows, j + NST, slot);
            }
            slot = slot + 1 == NST ? 0 : slot + 1;
            if (j + 1 < n) {
                arrived(j + 1);
                f0.read(ring + slot * STAGE + rel[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            mm(f1);
            if (j + 1 < n) f0.settle();
        }
    };
    if (n > 0) {
        // gathered rows (of an x whose length nobody here knows) beyond what 32-bit offsets reach: the wave looks its rows up again at every stage
        if (MODE == GEMM_GATEUP && __any(last >= reach)) {
            if constexpr (MODE == GEMM_GATEUP) stream(std::true_type{}, std::false_type{});
        } else if (once) stream(std::false_type{}, std::true_type{});
        else stream(std::false_type{}, std::false_type{});
    }

    // ---- sum of the waves' tiles, in wave order: wave w finishes row tiles w MPW ..
    __syncthreads();               // the rings are read
    f32x4_t* red = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
    for (int j = 0; j < MPW; ++j)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const f32x4_t a = wid == 0 ? acc[rt][MPW + j] : acc[rt][j];
            red[((wid * MPW + j) * RT + rt) * 64 + lane] = a;
        }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MPW; ++j) {
        f32x4_t sum[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const f32x4_t other = red[(((1 - wid) * MPW + j) * RT + rt) * 64 + lane];
            sum[rt] = wid == 0 ? acc[rt][j] + other : other + acc[rt][MPW + j];
        }
        const int row = 16 * (MPW * wid + j) + c;
        if (row >= mcnt) continue;
        bf16_t* yrow = p.y + (int64_t)(m0 + row) * p.ldy + ncol0 + 4 * g4;
        const int left = p.N - ncol0 - 4 * g4;   // N % 4 == 0 is checked on the host
        if constexpr (gemm_paired(MODE)) {
#pragma unroll
            for (int h = 0; h < RT / 2; ++h) {
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = rbf(glm_silu(rbf(sum[h][r]))) * rbf(sum[RT / 2 + h][r]);
                if (16 * h < left) *reinterpret_cast<u32x2_t*>(yrow + 16 * h) = u32x2_t{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
            }
        } else {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = scaled ? rbf(sum[rt][r]) * sc[j] : sum[rt][r];
                if (16 * rt < left) *reinterpret_cast<u32x2_t*>(yrow + 16 * rt) = u32x2_t{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
            }
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(128, 2) void gemm_midm_experts_kernel(const GemmParams p, int reach) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int* sh = reinterpret_cast<int*>(smem);
    glm_locate_block(p.offs, p.G, p.R, 64, blockIdx.y, sh);
    __syncthreads();
    const int grp = __builtin_amdgcn_readfirstlane(sh[0]);
    const int m0 = __builtin_amdgcn_readfirstlane(sh[1]);
    const int mcnt = __builtin_amdgcn_readfirstlane(sh[2]);
    __syncthreads();   // everyone has read sh before the first DMA lands on it
    if (grp < 0) return;
    const int ncol0 = blockIdx.x * (gemm_paired(MODE) ? 32 : 64);
    const bool once = p.offs[grp + 1] - p.offs[grp] <= 64;
    if (mcnt <= 32) midm_expert_body<MODE, 2>(p, smem, grp, m0, mcnt, ncol0, once, reach);
    else midm_expert_body<MODE, 4>(p, smem, grp, m0, mcnt, ncol0, once, reach);
}

template <int MODE>
int launch_midm_experts(const GemmParams& p, hipStream_t st) {
    constexpr int LDS = 2 * 2 * (4 + 4) * 2048;   // two waves, two stages
    const int cols = gemm_paired(MODE) ? 32 : 64;
    const int64_t gy = p.R / 64 + p.G;
    GLM_CHECK_ARG(gy <= 65535, GLM_ERR_UNSUPPORTED, "gemm_midm: grid too large");
    auto kern = gemm_midm_experts_kernel<MODE>;
    const int64_t reach = (1ll << 30) / p.ldx;
    hipLaunchKernelGGL(kern, dim3((unsigned)((p.N + cols - 1) / cols), (unsigned)gy), dim3(128), LDS, st, p, (int)reach);
    GLM_CHECK_LAUNCH("gemm_midm");
    return GLM_OK;
}

#endif  // GLM_EXPERTS

// rows m0 .. m0 + mcnt - 1, columns from ncol0, tile shared by the workgroup: WM x WN waves of MT x RT 16-row tiles each.  Every wave brings
// its share of a stage (one 64-wide K chunk of all rows); the counted wait is for its own share, the barrier behind it for the others', and
// it also says that every wave has the stage before in registers: its slot takes the chunk NST - 1 ahead.
template <int MODE, int WM, int WN, int MT, int RT, int NST, bool NT>
__device__ __forceinline__ void midm_shared_body(const GemmParams& p, char* smem, int m0, int mcnt, int ncol0, int slice) {
    static_assert(RT == 2, "the QKV epilogue takes the two columns that turn together from one lane");
    constexpr int NW = WM * WN, WR = 16 * RT * WN, XR = 16 * MT * WM;   // weight rows and activation rows of a stage
    constexpr int STAGE = (WR + XR) * MM_ROWB, D = (WR + XR) / 8 / NW, DW = WR / 8 / NW;
    constexpr int HALF = 8 * RT;               // paired modes: gate rows of a wave's columns, then as many up rows
    static_assert(NST * STAGE >= NW * RT * MT * 1024, "gemm_activate's pieces");
    static_assert(WR % (8 * NW) == 0 && XR % (8 * NW) == 0 && NST >= 2, "whole DMA instructions per wave");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wid % WN, wm = wid / WN;
    const int c = lane & 15, g4 = lane >> 4;
    const unsigned ring = (unsigned)(uintptr_t)(const mm_lds_void*)smem;
    const int r8 = lane >> 3, pc = lane & 7;
    const int K = p.ksplit > 1 ? p.K / p.ksplit : p.K;   // (equal slices of whole chunks)
    const __amdgpu_buffer_rsrc_t wrs = mm_rsrc(p.w + (int64_t)slice * K), xrs = mm_rsrc(p.x + (int64_t)slice * K);
    const bool qkv = MODE == GEMM_PLAIN && p.qkv_q != nullptr;   // a wave's two row tiles are 32 columns apart
    unsigned vo[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const bool isw = i < DW;
        const int row = 8 * ((isw ? i : i - DW) * NW + wid) + r8;
        int src;
        if (!isw) src = m0 + min(row, mcnt - 1);    // rows past the end repeat the last one; they are never stored
        else if (gemm_paired(MODE)) {
            const int rr = row % (16 * RT), col = ncol0 + row / (16 * RT) * HALF + rr % HALF;
            src = (rr < HALF ? 0 : p.N) + min(col, p.N - 1);
        } else src = min(ncol0 + (qkv ? (row & ~63) + (row >> 5 & 1) * 16 + (row >> 4 & 1) * 32 + (row & 15) : row), p.N - 1);
        vo[i] = ((unsigned)src * (unsigned)(isw ? p.ldw : p.ldx) + (pc ^ ((row >> 1) & 7)) * 8) * 2u;
    }
    const int n = K / MM_KC;
    auto issue = [&](int j, int slot) {
        const int soff = j * MM_ROWB;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const bool isw = i < DW;
            char* dst = smem + slot * STAGE + (isw ? 0 : WR * MM_ROWB) + ((isw ? i : i - DW) * NW + wid) * 1024;
            if (isw && NT) __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (mm_lds_void*)dst, 16, vo[i], soff, 0, 2);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(isw ? wrs : xrs, (mm_lds_void*)dst, 16, vo[i], soff, 0, 0);
        }
    };
    f32x4_t acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    unsigned rel_w[2], rel_x[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const unsigned r = c * MM_ROWB + (((4 * ks + g4) ^ ((c >> 1) & 7)) << 4);
        rel_w[ks] = r + wn * RT * 2048;
        rel_x[ks] = r + WR * MM_ROWB + wm * MT * 2048;
    }
#pragma unroll
    for (int j = 0; j < NST - 1; ++j)
        if (j < n) issue(j, j);
    int slot = 0;
    for (int j = 0; j < n; ++j) {
        if (j + NST - 1 <= n) asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NST - 2) * D) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        MmShared<MT, RT> f0, f1;
        const unsigned st = ring + slot * STAGE;
        f0.read(st + rel_w[0], st + rel_x[0]);
        if (j + NST - 1 < n) issue(j + NST - 1, slot == 0 ? NST - 1 : slot - 1);
        f0.settle();
        f1.read(st + rel_w[1], st + rel_x[1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f0.w[rt]), __builtin_bit_cast(bf16x8_t, f0.x[mt]), acc[rt][mt], 0, 0, 0);
        f1.settle();
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f1.w[rt]), __builtin_bit_cast(bf16x8_t, f1.x[mt]), acc[rt][mt], 0, 0, 0);
        slot = slot + 1 == NST ? 0 : slot + 1;
    }
    if (MODE == GEMM_PLAIN && p.act.kind != GLM_ACT_NONE) __syncthreads();   // the ring is read: gemm_activate's pieces lie in it
    const int first = 16 * MT * wm;
    if (first >= mcnt) return;
    if constexpr (MODE == GEMM_PLAIN) {
        if (qkv) {
            midm_qkv_rows<2, MT>(p, acc, m0 + first, mcnt - first, ncol0 + wn / 2 * 64, wn % 2 * 16, c, g4);
            return;
        }
    }
    // (slab s of the partial sums: rows s R ..)
    gemm_row_epilogue<MODE, RT, MT, true>(p, acc, 0, slice * (int)p.R + m0 + first, mcnt - first, ncol0 + wn * (gemm_paired(MODE) ? HALF : 16 * RT), c, g4,
                                     reinterpret_cast<f32x4_t*>(smem) + wid * RT * MT * 64 + lane);
}

template <int WM, int WN, int MT, int RT, int NST>
constexpr int midm_shared_lds() { return NST * (16 * RT * WN + 16 * MT * WM) * MM_ROWB; }

template <int MODE, int WM, int WN, int MT, int RT, int NST, bool NT>
__global__ __launch_bounds__(WM * WN * 64) void gemm_midm_shared_kernel(const GemmParams p, int mblocks, int interleaved) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int COLS = (gemm_paired(MODE) ? 8 : 16) * RT * WN, ROWS = 16 * MT * WM;
    int m, ntile;
    midm_tile(mblocks, interleaved, m, ntile);
    if (ntile * COLS >= p.N) return;
    midm_shared_body<MODE, WM, WN, MT, RT, NST, NT>(p, smem, m * ROWS, min(ROWS, (int)p.R - m * ROWS), ntile * COLS, blockIdx.z);
}

// Column tiles are dealt to the XCDs one by one where there are many, unless a last turn that not every XCD has is a second round for those that have it: 85
// column tiles of three row blocks are 33 workgroups on five XCDs of 32 CUs and 30 on the others.  Those go in runs.  Dealt / in runs, us, cold weights: 96 rows of
// 2720 x 512 6.2 / 4.4, 70 of 2720 x 4032 15.0 / 11.0, 65 of 2720 x 8192 25.3 / 18.2, 190 of 2688 x 1024 9.4 / 6.2, 330 of 5300 x 2048 20.4 / 18.7, gate|up 36.5 / 22.4.
inline bool midm_dealt(int nt, int64_t mblocks) {
    return nt >= 64 && ((nt + 7) / 8 * 8 * mblocks <= 256 || nt * mblocks > 256);
}

template <int MODE, int MT, int RT, int NW, int NST>
int launch_midm_cfg(const GemmParams& p, hipStream_t st) {
    static_assert(MT % NW == 0 || NW % MT == 0, "row tiles split over the waves");
    constexpr int LDS = midm_lds<MODE, MT, RT, NW, NST>();
    static_assert(LDS <= 160 * 1024, "the rings of all waves must fit the CU's LDS");
    const int cols = gemm_paired(MODE) ? 8 * RT : 16 * RT, nt = (p.N + cols - 1) / cols;
    const int64_t mblocks = (p.R + 16 * MT - 1) / (16 * MT);
    const bool dealt = midm_dealt(nt, mblocks);
    const int64_t gx = dealt ? (int64_t)(nt + 7) / 8 * 8 * mblocks : (nt * mblocks + 7) / 8 * 8;
    GLM_CHECK_ARG(gx < (1 << 30), GLM_ERR_UNSUPPORTED, "gemm_midm: grid too large");
    // Few columns under many rows: column tile by column tile every XCD would pull all the activations, which outweigh the weights.  That order / row
    // block by row block, us: 2000 rows of 64 x 8192 23.1 / 13.4, x 16384 40.6 / 21.3, x 4096 13.7 / 8.9, x 2048 7.2 / 6.4, 1000 of 128 x 8192
    // 23.0 / 13.0, 512 of 128 x 8192 14.9 / 12.6, of 40 x 8192 11.2 / 10.1; but 300 of 64 x 8192 10.0 / 11.8, of 128 x 4096 7.2 / 8.9.  (A kernel
    // of its own: one that takes both orders is 0.2 us slower in the other.)
    const bool byrow = RT == 1 && !dealt && nt > 1 && p.R >= 512 && p.R * 3 > p.N * 7;
    auto kern = byrow ? gemm_midm_kernel<MODE, MT, RT, NW, NST, RT == 1> : gemm_midm_kernel<MODE, MT, RT, NW, NST, false>;
    if (LDS > 64 * 1024) GLM_SET_MAX_LDS(kern, LDS, "gemm_midm");
    hipLaunchKernelGGL(kern, dim3((unsigned)gx), dim3(NW * 64), LDS, st, p, (int)mblocks, byrow ? nt : (int)dealt);
    GLM_CHECK_LAUNCH("gemm_midm");
    return GLM_OK;
}

template <int MODE, int WM, int WN, int MT, int RT, int NST, bool NT>
int launch_midm_shared(const GemmParams& p, hipStream_t st) {
    constexpr int LDS = midm_shared_lds<WM, WN, MT, RT, NST>();
    static_assert(LDS <= 160 * 1024, "the ring must fit the CU's LDS");
    const int cols = (gemm_paired(MODE) ? 8 : 16) * RT * WN, nt = (p.N + cols - 1) / cols;
    const int64_t mblocks = (p.R + 16 * MT * WM - 1) / (16 * MT * WM);
    const bool dealt = midm_dealt(nt, mblocks);
    const int64_t gx = dealt ? (int64_t)(nt + 7) / 8 * 8 * mblocks : (nt * mblocks + 7) / 8 * 8;
    GLM_CHECK_ARG(gx < (1 << 30), GLM_ERR_UNSUPPORTED, "gemm_midm: grid too large");
    auto kern = gemm_midm_shared_kernel<MODE, WM, WN, MT, RT, NST, NT>;
    if (LDS > 64 * 1024) GLM_SET_MAX_LDS(kern, LDS, "gemm_midm");
    hipLaunchKernelGGL(kern, dim3((unsigned)gx, 1, (unsigned)(p.ksplit > 1 ? p.ksplit : 1)), dim3(WM * WN * 64), LDS, st, p, (int)mblocks, (int)dealt);
    GLM_CHECK_LAUNCH("gemm_midm");
    return GLM_OK;
}

// The tile of a dense projection: the first of these with a workgroup per CU at most.  More and smaller workgroups put more of the chip to
// work and have more bytes on their way; a larger tile pulls fewer, and two rounds of one cost more than one round of the next.  Split, 64 x 64,
// 128 x 64, 128 x 128 (64 rows: 64 x 128), us, cold operands, * the one taken: 4096 x 4096 at 64 rows 16.5 / 21.2 / - / 30 (32 x 32, a round of which comes first, 13.5*), at 211 24.5 / 20.5* /
// 30.0 / 36.2, at 512 47 / - / 31.8* / 40.2; 14336 x 4096 at 64 36.7 / 27.6* / - / 37.5, at 128 56 / 42.6 / 37.7* / 46.3, at 211 77 / 61.5 / 52 /
// 43.0*; 2048 x 2048 at 1000 rows - / 16.9 / 17.2* / 19.8 (512 tiles of 64 x 64), at 2000 - / 35.2 / 25.9 / 23.7*; 32768 x 2048 at 64 42 / 30.1 / - / 27.6*.
// A long K favours split waves at 64 x 64 too, which read each staged byte once: 4096 x 12288 at 211 rows 50 (shared 58), K = 8192 36 (40).
enum MidmTile { MM_NONE, MM_SPLIT16, MM_SPLIT32x32, MM_SPLIT32, MM_SPLIT64, MM_64, MM_128x64, MM_64x128, MM_128 };

MidmTile midm_tile_of(int mode, const GemmParams& p) {
    const int64_t n = gemm_paired(mode) ? 2 * (int64_t)p.N : (int64_t)p.N;
    auto fits = [&](int rows, int cols) { return (n + cols - 1) / cols * ((p.R + rows - 1) / rows) <= 256; };
    // A short reduction is mostly the two ends, a ring filled once and the sum of the waves: the shared tile's are shorter with gate and up rows in
    // it, and with a hundred row blocks and more.  Shared 64 x 64 / split 64 x 32, us: 1024 x 256 at 300 rows 4.3 / 3.8, 264 x 512 at 700 5.7 / 4.7,
    // 512 x 384 at 1000 4.7 / 4.1, fp32 rows 6.2 / 4.8, 64 x 512 at 3000 5.2 / 4.6, at 8000 6.1 / 6.4; gated columns 512 x 128 at 96 rows 3.0 / 3.4,
    // 1024 x 320 at 128 4.1 / 4.2, 256 x 512 at 300 4.4 / 3.9, 132 x 512 at 700 4.6 / 4.4, at 1500 4.9 / 5.5.
    // A workgroup takes in some 50 GB/s of weights that no cache holds, whatever it does, so tiles of 32 rows whose K is split over eight waves come
    // first, as few columns as one round of the chip allows.  Others / these, us, cold weights.  16 columns, formerly 64 x 32 over four waves:
    // 100 rows of 64 x 2048 6.6 / 4.1, x 256 3.5 / 2.9, 211 of 64 x 4096 11.1 / 6.8, 2000 of 64 x 2048 7.4 / 5.6, 33 of 376 x 8192 16.3 / 9.5, 128 of
    // 1024 x 2048 8.9 / 6.2, 64 of 2048 x 2048 10.2 / 7.1, 33 of 2048 x 4096 14.4 / 8.9, 64 of 1024 x 6144 22.7 / 13.0, 100 of 640 x 512 4.6 / 3.8.  32
    // columns: 128 of 2048 x 2048 9.9 / 8.2, x 4096 15.9 / 12.4, 48 of 3072 x 768 6.1 / 5.3, 96 of 2048 x 512 4.7 / 4.4, 70 of 2048 x 8192 22.6 / 18.2, gated
    // 100 of 1024 x 2048 9.3 / 7.4.  (48 columns: 128 of 2304 x 2048 9.95 / 9.5 in a row of its own, but 9.8 / 9.9 inside a step, 100 of 3072 x 768
    // 6.4 / 7.6: not taken.)
    // (The same chunks by wave and the same order of the eight sums in all of them and in the QKV epilogue's tile.)
    if (!gemm_paired(mode) && p.K >= (p.N < 384 ? 256 : 512) && fits(32, 16)) return MM_SPLIT16;
    if (p.K >= 512 && fits(32, 32)) return MM_SPLIT32x32;
    if (fits(64, 32) && (gemm_paired(mode) ? p.K >= (p.R <= 1000 ? 384 : 576) : p.K > 512 || p.R <= 4096)) return MM_SPLIT32;
    if (fits(64, 64)) return p.K >= 8192 ? MM_SPLIT64 : MM_64;
    if (p.R <= 64) return fits(64, 128) ? MM_64x128 : MM_NONE;
    if (fits(128, 64)) return MM_128x64;
    return fits(128, 128) ? MM_128 : MM_NONE;
}

// Weights that only one row block reads go past the caches, which they leave to the activations (nt), from 64 MiB on.  Kept / past them, us, weights not in
// the caches: 128 rows of 32768 x 2048 33.1 / 31.5, 64 of 14336 x 4096 32.0 / 29.4, gated 49.9 / 47.2; steps: 64 GLM sequences over fp8 experts 2149 / 2131, 128
// Dafolorn ones 469.7 / 462.0, 100 Gulozen ones 1146 / 1142.  Weights that are still in the 256 MiB behind the L2 from the last time are read from HBM
// all the same (64 of 14336 x 4096 21.8 / 29.1, 128 of 12288 x 2048, gated, 14.7 / 17.2), so a layer whose matrices may all lie there is spared: what
// matrices below the line gain by themselves (41 of 8928 x 576 6.5 / 6.0) steps do not show (Dafolorn with it on those too 465.7, Gulozen 1147).  With two row blocks and more, and in the split tiles,
// single projections gained as much and steps lost it again (a prompt of 211 1.886 / 1.904 ms).  A kernel of its own: chosen inside the loop, for every DMA
// instruction, it cost all others 1 to 5 % (gate|up 965 of 456 x 6912 32.9 / 31.3, 300 of 1024 x 2048 12.1 / 11.7, plain 300 of 2048 x 2048 12.6 / 12.4).
constexpr int64_t MM_NT_BYTES = 64 << 20;

template <int MODE>
int launch_midm_tile(MidmTile tile, const GemmParams& p, hipStream_t st) {
    if constexpr (MODE == GEMM_PLAIN) {   // half a head in the QKV epilogue of 32 rows; the sums are the same in all three
        if (p.qkv_q != nullptr && (tile == MM_SPLIT16 || tile == MM_SPLIT32x32)) return launch_midm_cfg<MODE, 2, 4, 8, 1>(p, st);
    }
    const bool nt = (gemm_paired(MODE) ? 2 : 1) * (int64_t)p.N * p.ldw * 2 >= MM_NT_BYTES;
    switch (tile) {
        case MM_SPLIT16:
            if constexpr (!gemm_paired(MODE)) return launch_midm_cfg<MODE, 2, 1, 8, 2>(p, st);
            break;
        case MM_SPLIT32x32: return launch_midm_cfg<MODE, 2, 2, 8, 2>(p, st);
        case MM_SPLIT32:   // (half a head in the QKV epilogue; the sums are the same in both tiles)
            if (MODE != GEMM_PLAIN || p.qkv_q == nullptr) return launch_midm_cfg<MODE, 4, 2, 4, 2>(p, st);
            [[fallthrough]];
        case MM_SPLIT64: return launch_midm_cfg<MODE, 4, 4, 4, 2>(p, st);
        case MM_64: return nt && p.R <= 64 ? launch_midm_shared<MODE, 2, 2, 2, 2, 4, true>(p, st) : launch_midm_shared<MODE, 2, 2, 2, 2, 4, false>(p, st);
        case MM_128x64: return nt && p.R <= 128 ? launch_midm_shared<MODE, 2, 2, 4, 2, 3, true>(p, st) : launch_midm_shared<MODE, 2, 2, 4, 2, 3, false>(p, st);
        case MM_64x128: return nt && p.R <= 64 ? launch_midm_shared<MODE, 2, 4, 2, 2, 3, true>(p, st) : launch_midm_shared<MODE, 2, 4, 2, 2, 3, false>(p, st);
        case MM_128: return nt && p.R <= 128 ? launch_midm_shared<MODE, 2, 4, 4, 2, 4, true>(p, st) : launch_midm_shared<MODE, 2, 4, 4, 2, 4, false>(p, st);
        default: break;
    }
    GLM_CHECK_ARG(false, GLM_ERR_UNSUPPORTED, "gemm_midm: no tile for %ld rows, N=%d", (long)p.R, p.N);
}

template <int MODE>
int launch_midm(const GemmParams& p, hipStream_t st) {
#if GLM_EXPERTS
    if constexpr (MODE == GEMM_GATEUP || MODE == GEMM_DOWN) {
        if (p.offs != nullptr) return launch_midm_experts<MODE>(p, st);
    }
#endif
    return launch_midm_tile<MODE>(midm_tile_of(MODE, p), p, st);
}

// K slices of a projection whose tiles are a quarter of the chip at most, and the tile for them: as many as bring a workgroup to every CU.  A
// smaller tile with at least four slices goes before a larger one with more (fewer partial sums for the same workgroups).  With the norm that
// adds them up, one pass / slices, us, cold weights: 4096 x 12288 at 64 rows 36.9 / 27.5 (4 of 64 x 64), at 128 46.1 / 35.3 (4 of 128 x 64), at 211 54.5 / 43.5 (4 of
// 128 x 128); 2048 x 8192 at 33 17.5 / 13.6, at 64 19.1 / 14.7, at 128 22.3 / 17.5, at 400 33.8 / 29.5; 2048 x 4096 at 33 11.5 / 11.0, at 64 12.6 / 11.8, at 211 16.7 /
// 16.2; 4096 x 4096 at 64 17.8 / 16.1; 1024 x 4096 at 64 12.0 / 10.4; least of all K = 4096 at 128 rows: 2048 columns 14.7 / 15.2, 1024 12.1 / 12.7.  K = 2048: 7.1 /
// 6.7 without the norm, whose wider reads take that back.
int midm_slices(int64_t M, int N, int K, MidmTile* tile) {
    if (M <= 32 || K % 64 != 0 || K < 4096 || N % 4 != 0) return 1;
    if (M < 96 && (int64_t)N * K >= 1ll << 29) return 1;   // up to 95 rows slices have no other kernel, and this one's offsets (of padded rows) are 32-bit
    static const struct { MidmTile t; int rows, cols; } tiles[] = {{MM_64, 64, 64}, {MM_128x64, 128, 64}, {MM_128, 128, 128}};
    for (const auto& c : tiles) {
        if ((c.rows == 64) != (M <= 64)) continue;
        const int64_t n = (M + c.rows - 1) / c.rows * ((N + c.cols - 1) / c.cols);
        int best = 1;
        for (int s = 2; s <= 8 && s * n <= 256 && K / s >= 512; ++s)
            if (K % (64 * s) == 0) best = s;
        if (best < 4) continue;
        *tile = c.t;
        return best;
    }
    return 1;
}

}  // namespace

bool glm_midm_takes(int mode, const GemmParams& p) {
    if (p.ksplit > 1 || p.wscale != nullptr || p.K % 64 != 0) return false;
    if (p.offs != nullptr) {
        // Experts with 24 to 95 rows on average: the weight-streaming kernel's blocks of 32 rows read an expert's weights once per block.  gate|up,
        // down, us, rows dealt at random: 65 of 1408 x 4096 at 28 rows 330 / 184 there, 247 / 142 here, at 55 557 / 279 and 277 / 161.
        // With fewer rows, where there are column tiles for several rounds of the chip: there every 32 weight rows move as many activation
        // bytes.  There / here: gate|up 65 of 1408 x 4096 at 9 rows 232 / 236, at 13 240 / 236, at 18 251 / 239, at 22 264 / 241, 64 of 1024 x 2048
        // at 11 95.9 / 97.7, at 15 99.6 / 99.0, at 20 107 / 101, 129 of 512 x 1024 at 18 63 / 57, of 768 x 2048 at 7 133 / 137; one round: 17 of
        // 1408 x 4096 at 18 74 / 79, 65 of 352 x 4096 at 14 68 / 75.  Down 65 of 1408 x 4096 at 7 129 / 120, at 9 133 / 122, at 18 145 / 131, 129 of
        // 768 x 2048 at 7 80 / 77, at 4 68 / 73, 17 of 1408 x 4096 at 18 44 / 40, 64 of 1024 x 2048 at 11 54.7 / 54.6; 33 of 1024 x 1024 at 15 19.6 / 21.0,
        // 9 of 2048 x 4096 at 13 31 / 40.  Down with K of 256, 512 or 1024 is ahead later than with lengths
        // between: 129 of 512 x 1024 at 7 33.0 / 34.3, at 12 34.6 / 35.0, at 20 38.1 / 35.6, 64 of
        // 1024 x 2048 at 7 47.3 / 48.7, at 12 50.4 / 49.8, 160 of 256 x 2048 at 7 50.2 / 51.7, at 14 56 / 54, but 64 of 768 x 2048 at 9 39.9 / 38.9, 65 of
        // 704 x 4096 at 7 77 / 72.
        const int64_t rows = p.R_hint > 0 ? p.R_hint : p.R;
        if (mode != GEMM_GATEUP && mode != GEMM_DOWN) return false;
        const int64_t G = p.G, tiles = (p.N + (mode == GEMM_GATEUP ? 31 : 63)) / (mode == GEMM_GATEUP ? 32 : 64) * G;
        const int few = p.K <= 1024 && (p.K & (p.K - 1)) == 0 ? 12 : 6;
        const bool enough = rows >= 24 * G || (mode == GEMM_GATEUP ? rows >= 13 * G && tiles >= 2048 : rows > few * G && tiles >= 1024);
        return enough && rows < 96 * G && p.R * p.ldx * 2 < (1ll << 31) && (mode == GEMM_GATEUP ? 2 : 1) * (int64_t)p.N * p.ldw * 2 < (1ll << 31);
    }
    if (p.src != nullptr || p.G > 1 || p.R <= 32) return false;
    // (a loop of the tiled kernel that is asked for keeps its shapes)
    if (p.R >= 96 && (glm_option(GLM_OPT_LARGEM_VARIANT) >= 0 || glm_option(GLM_OPT_LARGEM_CFG) != 0)) return false;
    // Feed-forwards below 96 rows: the streaming kernel has configurations for them with a workgroup per 16 act columns or 32 columns and block of
    // 32 rows.  It is ahead where K is a few chunks, half of these tiles' time being the ends then, and in long down projections of four 16-row
    // pieces, whose activations it brings in once for all columns of a workgroup.  Streaming / here, us, weights not in the caches: gate|up 1024 x 384 at 48 4.3 / 4.7,
    // 1536 x 512 4.66 / 4.74, 2048 x 512 4.5 / 4.8, 1536 x 768 5.1 / 5.2, but 1024 x 896 5.8 / 5.2, 1024 x 1024 at 33 5.8 / 5.3, 1024 x 4096 at 48 13.0 /
    // 11.2, at 64 13.1 / 12.3, 2048 x 2048 at 48 8.2 / 8.0, at 64 8.4 / 8.5, 768 x 12288 at 64 32.8 / 29.3, 2048 x 16384 at 41 74 / 48.  Down 2048 x 256 at 64
    // 3.5 / 3.8, 4096 x 384 at 33 4.6 / 4.8, 2048 x 448 at 48 4.6 / 4.8, but 2048 x 512 at 64 5.3 / 4.7; 1024 x 4096 at 40 8.7 / 7.9, at 48 8.4 / 8.4, at 52
    // 8.3 / 8.7, at 64 8.9 / 9.4; 2048 x 6144 at 48 12.7 / 12.3, at 52 12.3 / 12.2, at 56 12.2 / 12.6, at 64 12.6 / 13.3; 2048 x 12288 at 48 24.4 / 21.3, at
    // 52 22.7 / 21.4, at 56 22.3 / 22.2, at 64 22.1 / 23.5, but 2304 x 5120 at 56 18.6 / 14.6, 64 x 4096 at 64 8.9 / 8.6, 2048 x 3072 at 64 17.2 / 9.7.
    if (p.R < 96 && mode != GEMM_PLAIN) {
        const int64_t n = (p.R + 31) / 32 * p.N;
        if (mode == GEMM_DOWN) {
            if (p.K < 512 ? n <= 8192 : p.K >= 4096 && p.R > 48 && p.R <= 64 && p.N >= 128 && p.N <= 2048) return false;
        } else if (p.K > 320 && p.K <= 768 && p.N >= 1024 && n <= 4096) return false;
    }
    const int64_t wrows = gemm_paired(mode) ? 2 * (int64_t)p.N : (int64_t)p.N;
    if (p.R * p.ldx * 2 >= (1ll << 31) || wrows * p.ldw * 2 >= (1ll << 31)) return false;   // 32-bit offsets
    // Beyond one round of the largest tile the tiled kernel's 128 x 256 and 256 x 256 ones pull less (14336 x 4096 at 400 rows, 448 tiles: 60 us
    // there, 76 here; 9728 x 2048 at 400, 304: 31 / 39; 6144 x 2048 at 1000, 384: 33 / 42), and 64 rows of more than 32768 columns stay with
    // the weight-streaming kernel.
    return midm_tile_of(mode, p) != MM_NONE;
}

int glm_midm_slices(int64_t M, int N, int K) {
    MidmTile tile;
    return midm_slices(M, N, K, &tile);
}

bool glm_midm_takes_slices(const GemmParams& p) {
    MidmTile tile;
    if (p.R <= 32 || p.K % (64ll * p.ksplit) != 0 || p.R * p.ldx * 2 >= (1ll << 31) || (int64_t)p.N * p.ldw * 2 >= (1ll << 31)) return false;
    // (up to 95 rows there is no other kernel for slices of another number)
    return p.R < 96 || midm_slices(p.R, p.N, p.K, &tile) == p.ksplit;
}

int glm_launch_gemm_midm_slices(const GemmParams& p, hipStream_t st) {
    GLM_CHECK_ARG(p.N % 4 == 0 && p.ldx % 8 == 0 && p.ldw % 8 == 0 && glm_aligned16(p.x) && glm_aligned16(p.w) && glm_aligned16(p.ypart), GLM_ERR_UNSUPPORTED,
                  "gemm_midm(slices): needs N%%4==0, ldx/ldw%%8==0, 16B-aligned x/W/partial sums (N=%d)", p.N);
    MidmTile tile = p.R <= 64 ? MM_64 : MM_128x64;
    midm_slices(p.R, p.N, p.K, &tile);
    return launch_midm_tile<GEMM_PLAIN>(tile, p, st);
}

int glm_launch_gemm_midm(int mode, const GemmParams& p, hipStream_t st) {
    GLM_CHECK_ARG(p.K % 64 == 0 && p.N % 4 == 0 && p.ldx % 8 == 0 && p.ldy % 4 == 0 && p.ldw % 8 == 0 && glm_aligned16(p.x) && glm_aligned16(p.w) &&
                      (((uintptr_t)p.y) & 7) == 0,
                  GLM_ERR_UNSUPPORTED, "gemm_midm: needs K%%64==0, N%%4==0, ldx/ldw%%8==0, ldy%%4==0, 16B-aligned x/W (K=%d N=%d)", p.K, p.N);
#if GLM_EXPERTS
    if (mode == GEMM_GATEUP) return launch_midm<GEMM_GATEUP>(p, st);
    if (mode == GEMM_DOWN) return launch_midm<GEMM_DOWN>(p, st);
#endif
    if (mode == GEMM_GLU) return launch_midm<GEMM_GLU>(p, st);
    return launch_midm<GEMM_PLAIN>(p, st);
}
