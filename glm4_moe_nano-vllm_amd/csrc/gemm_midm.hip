// gemm_midm.hip — bf16 projections of some dozen to some hundred rows per weight matrix: batched decode of many sequences, short
// prompts, the experts of a short prompt.  gfx950 only.
//
// What bounds it: the weights are still read once and dominate the HBM bytes, but an output tile must be small for the grid to cover
// the chip, and every workgroup pulls its own activation rows through L2 -> LDS (about 11 TB/s over the chip, which binds from some 200 tiles
// on): the tile (64 rows x 64 or 32 weight rows) is chosen for that traffic, and the LDS reads behind it are not allowed to exceed it.  So the waves of a workgroup split
// K, not the tile: a wave computes the whole output tile over its own K chunks, every staged byte is read from LDS exactly once, and
// there is no workgroup barrier in the loop — a wave waits for its own DMA only (counted vmcnt), as in the weight-streaming kernels.
//   * a stage = one 64-wide K chunk of the tile's activation and weight rows, a whole 128-byte line per row (with 32-wide chunks, half
//     lines: 14336 x 4096 at 128 rows 53 instead of 45 us, 4096 x 12288 at 64 rows 60 instead of 45);
//   * 16-byte pieces are swizzled at the source, piece ^ ((row >> 1) & 7): the 16 rows of a fragment read cover all banks;
//   * the fragments of a k-step are read under the MFMAs of the one before, a freed stage is refilled right after;
//   * the partial tiles of the waves are summed through LDS in wave order, each wave finishes its share of the rows;
//   * workgroups that share weight rows sit on one XCD, next to one another, and every XCD has as many.
#include "gemm_internal.h"
#include "gemm_epilogue.h"

namespace {

typedef __attribute__((address_space(3))) void mm_lds_void;

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

// The QKV projection's epilogue (glm_gemm_qkv_rope_store) on a tile of 64 columns, one half of a head: bias, rounding of the packed value,
// rotation of the first half's columns i and i + 32 (row tiles t and t + 2 in the same lane), rows of q / k / v and of the caches.  The
// tiled kernel's arithmetic and rounding points, so the fused launch stays bit-identical to the projection and the split kernel.
template <int MPW>
__device__ __forceinline__ void midm_qkv_rows(const GemmParams& p, const f32x4_t (&acc)[4][MPW], int m0, int mcnt, int ncol0, int c, int g4) {
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
        float o[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int n = ncol0 + 16 * t + 4 * g4;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[t][r] = rbf(acc[t][j][r] + (p.bias ? bf2f(p.bias[n + r]) : 0.0f));
        }
        if (half == 0 && (is_q || is_k)) {
            const float* cs = p.qkv_cs + p.qkv_pos[m] * 64;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float cv = cs[16 * t + 4 * g4 + r], sv = cs[32 + 16 * t + 4 * g4 + r], x1 = o[t][r], x2 = o[t + 2][r];
                    o[t][r] = x1 * cv - x2 * sv;
                    o[t + 2][r] = x2 * cv + x1 * sv;
                }
        }
        int64_t slot = -1;
        if (cache != nullptr && p.qkv_slots != nullptr) slot = p.qkv_slots[m];
        const bool to_cache = slot >= 0 && slot < p.qkv_nslots;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const u32x2_t v = {pack2bf(o[t][0], o[t][1]), pack2bf(o[t][2], o[t][3])};
            const int col = kh * 128 + 64 * half + 16 * t + 4 * g4;
            if (dense != nullptr) *reinterpret_cast<u32x2_t*>(dense + m * ldd + col) = v;
            if (to_cache) *reinterpret_cast<u32x2_t*>(cache + slot * nkv * 128 + col) = v;
        }
    }
}

// rows m0 .. m0 + mcnt - 1 of group grp, columns from ncol0; MT 16-row activation tiles, RT 16-row weight tiles
template <int MODE, int MT, int RT, int NW, int NST>
__device__ __forceinline__ void midm_body(const GemmParams& p, char* smem, int grp, int m0, int mcnt, int ncol0) {
    constexpr int D = 2 * (MT + RT);           // DMA instructions of a stage
    constexpr int STAGE = D * 1024;
    constexpr int HALF = 8 * RT;               // paired modes: gate rows of the tile, then as many up rows
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g4 = lane >> 4;
    const unsigned ring = (unsigned)(uintptr_t)(const mm_lds_void*)smem + wid * NST * STAGE;
    char* ringp = smem + wid * NST * STAGE;

    // ---- sources: instruction i brings rows 16 i + (lane >> 2), piece lane & 3 of the LDS row
    const int r8 = lane >> 3, pc = lane & 7;
    const __amdgpu_buffer_rsrc_t wrs = mm_rsrc(p.w + (int64_t)grp * p.w_gstride), xrs = mm_rsrc(p.x);
    unsigned wvo[2 * RT], xvo[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int row = 8 * i + r8;
        const int wr = gemm_paired(MODE) ? (row < HALF ? 0 : p.N) + min(ncol0 + (row < HALF ? row : row - HALF), p.N - 1) : min(ncol0 + row, p.N - 1);
        wvo[i] = ((unsigned)wr * (unsigned)p.ldw + (pc ^ ((row >> 1) & 7)) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = 8 * i + r8, m = m0 + min(row, mcnt - 1);   // rows past the end repeat the last one; they are never stored
        const int src = p.src ? p.src[m] : m;
        xvo[i] = ((unsigned)src * (unsigned)p.ldx + (pc ^ ((row >> 1) & 7)) * 8) * 2u;
    }
    // ---- this wave's chunks: wid, wid + 4, ... of the K columns
    const int n = max(0, (p.K / MM_KC - wid + NW - 1) / NW);
    auto issue = [&](int j, int slot) {
        const int soff = (j * NW + wid) * MM_ROWB;
        char* st = ringp + slot * STAGE;
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

    // ---- sum of the waves' tiles, in wave order; wave w finishes row tiles w MT / 4 ..
    constexpr int MPW = MT / NW;
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
            *reinterpret_cast<f32x4_t*>(red + (((wid * MT + mt) * RT + rt) * 64 + lane) * 4) = acc[rt][mt];
    __syncthreads();
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
            midm_qkv_rows<MPW>(p, sum, m0 + first, mcnt - first, ncol0, c, g4);
            return;
        }
    }
    gemm_row_epilogue<MODE, RT, MPW>(p, sum, grp, m0 + first, mcnt - first, ncol0, c, g4);
}

template <int MODE, int MT, int RT, int NW, int NST>
constexpr int midm_lds() {
    constexpr int ring = NW * NST * (MT + RT) * 2048, red = NW * MT * RT * 1024;
    return (ring > red ? ring : red) + 16;
}

template <int MODE, int MT, int RT, int NW, int NST>
__global__ __launch_bounds__(NW * 64) void gemm_midm_kernel(const GemmParams p_in, int mblocks, int interleaved) {
    GemmParams p = p_in;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int COLS = gemm_paired(MODE) ? 8 * RT : 16 * RT;
    if (MODE == GEMM_PLAIN && p_in.ksplit > 1) {   // K slice of this workgroup (whole pairs of chunks)
        const int per = (p_in.K / 64 + p_in.ksplit - 1) / p_in.ksplit * 64, kb = blockIdx.z * per;
        p.x = p_in.x + kb;
        p.w = p_in.w + kb;
        p.K = max(0, min(per, p_in.K - kb));
        p.ypart = p_in.ypart + (int64_t)blockIdx.z * p_in.R * p_in.N;
    }
    int grp = 0, m0, mcnt, ntile;
    if (p.offs) {
        int* sh = reinterpret_cast<int*>(smem + midm_lds<MODE, MT, RT, NW, NST>() - 16);
        glm_locate_block(p.offs, p.G, p.R, 16 * MT, blockIdx.y, sh);
        __syncthreads();
        grp = __builtin_amdgcn_readfirstlane(sh[0]);
        m0 = __builtin_amdgcn_readfirstlane(sh[1]);
        mcnt = __builtin_amdgcn_readfirstlane(sh[2]);
        ntile = blockIdx.x;
        if (grp < 0) return;
    } else {
        int m;
        if (interleaved) {   // column tiles dealt to the XCDs (workgroups b, b + 8, ...) one by one, their row blocks behind one another
            const int q = blockIdx.x >> 3;
            m = q % mblocks;
            ntile = q / mblocks * 8 + (blockIdx.x & 7);
        } else {             // few column tiles: an XCD takes a run of all tiles
            const int lin = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
            ntile = lin / mblocks;
            m = lin % mblocks;
        }
        m0 = m * (16 * MT);
        mcnt = min(16 * MT, (int)p.R - m0);
    }
    if (ntile * COLS >= p.N) return;
    midm_body<MODE, MT, RT, NW, NST>(p, smem, grp, m0, mcnt, ntile * COLS);
}

template <int MODE, int MT, int RT, int NW, int NST>
int launch_midm_cfg(const GemmParams& p, hipStream_t st) {
    static_assert(MT % NW == 0, "row tiles split over the waves");
    constexpr int LDS = midm_lds<MODE, MT, RT, NW, NST>();
    static_assert(LDS <= 160 * 1024, "the rings of all waves must fit the CU's LDS");
    const int cols = gemm_paired(MODE) ? 8 * RT : 16 * RT, nt = (p.N + cols - 1) / cols;
    const int64_t mblocks = (p.R + 16 * MT - 1) / (16 * MT);
    const bool dealt = nt >= 64;
    const int64_t gx = p.offs ? nt : dealt ? (int64_t)(nt + 7) / 8 * 8 * mblocks : (nt * mblocks + 7) / 8 * 8, gy = p.offs ? p.R / (16 * MT) + p.G : 1;
    GLM_CHECK_ARG(gx < (1 << 30) && gy <= 65535, GLM_ERR_UNSUPPORTED, "gemm_midm: grid too large");
    auto kern = gemm_midm_kernel<MODE, MT, RT, NW, NST>;
    if (LDS > 64 * 1024) GLM_SET_MAX_LDS(kern, LDS, "gemm_midm");
    hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)gy, (unsigned)(p.ksplit > 1 ? p.ksplit : 1)), dim3(NW * 64), LDS, st, p, (int)mblocks, (int)dealt);
    GLM_CHECK_LAUNCH("gemm_midm");
    return GLM_OK;
}

// tiles of 64 rows and 32 columns
int64_t small_tiles(int mode, const GemmParams& p) {
    const int cols = gemm_paired(mode) ? 16 : 32;
    return (int64_t)((p.N + cols - 1) / cols) * ((p.R + 63) / 64);
}

// Up to a workgroup per CU: 64 x 32 with four waves.  Beyond: workgroups of two waves, three to a CU, so that one's start and end lie under
// the others' loops.  A long K pays those once per tile and the activation traffic always: 64 x 64.  Four waves 64 x 32, two waves 64 x 32,
// four waves 64 x 64, us, cold operands: 2048 x 2048 at 128 rows (128 tiles) 8.2 / 10.7 / 15.8; 6144 x 2048 at 256 (768) 20.6 / 17.0 / 34.0;
// 14336 x 4096 at 128 (896) 58.9 / 55.4 / 59.3; 4096 x 12288 at 128 (256) 42.7 / 53.4 / 66.2, at 256 (512) 74.2 / 79.5 / 66.1.
template <int MODE>
int launch_midm(const GemmParams& p, hipStream_t st) {
    // experts: two waves, two workgroups per CU, so that one is at work while the other starts or sums up (short K, many tiles; four waves: 211
    // tokens on 65 experts of 1408 x 4096 291 / 186 us instead of 274 / 154)
    if (p.offs != nullptr) return launch_midm_cfg<MODE, 4, 4, 2, 2>(p, st);
    if (MODE == GEMM_PLAIN && p.qkv_q != nullptr) return launch_midm_cfg<MODE, 4, 4, 4, 2>(p, st);   // (half a head; the sums are the same in both tiles)
    if (small_tiles(MODE, p) <= 256) return launch_midm_cfg<MODE, 4, 2, 4, 2>(p, st);
    return p.K >= 8192 ? launch_midm_cfg<MODE, 4, 4, 4, 2>(p, st) : launch_midm_cfg<MODE, 4, 2, 2, 2>(p, st);
}

}  // namespace

bool glm_midm_takes(int mode, const GemmParams& p) {
    if (p.ksplit > 1 || p.wscale != nullptr || p.K % 64 != 0) return false;
    if (p.offs != nullptr) {
        // Experts with 24 to 95 rows on average: the weight-streaming kernel's blocks of 32 rows read an expert's weights once per block.
        // gate|up, down of 1408 x 4096, us: 26 rows 298 / 160 there, 261 / 147 here; 55 rows 557 / 279 and 307 / 174; 18 rows 263 / 149 and
        // 265 / 145; of 1024 x 2048: 20 rows 108 / 57 and 106 / 60, 38 rows 168 / 82 and 109 / 62.
        const int64_t rows = p.R_hint > 0 ? p.R_hint : p.R;
        if (mode != GEMM_GATEUP && mode != GEMM_DOWN) return false;
        return rows >= 24 * (int64_t)p.G && rows < 96 * (int64_t)p.G && p.R * p.ldx * 2 < (1ll << 31) &&
               (mode == GEMM_GATEUP ? 2 : 1) * (int64_t)p.N * p.ldw * 2 < (1ll << 31);
    }
    if (p.src != nullptr || p.G > 1 || p.R <= 32) return false;
    // (a loop of the tiled kernel that is asked for keeps its shapes)
    if (p.R >= 96 && (glm_option(GLM_OPT_LARGEM_VARIANT) >= 0 || glm_option(GLM_OPT_LARGEM_CFG) != 0)) return false;
    const bool paired = gemm_paired(mode);
    const int64_t wrows = paired ? 2 * (int64_t)p.N : (int64_t)p.N;
    if (p.R * p.ldx * 2 >= (1ll << 31) || wrows * p.ldw * 2 >= (1ll << 31)) return false;   // 32-bit offsets
    const int64_t tiles = small_tiles(mode, p);
    // Fewer rows than the tiled kernel takes: the weight-streaming kernel gets ahead where it has a wave of workgroups to spare (32768 x 2048
    // at 64 rows, 1024 tiles, 31 us, here 35; 18944 x 4096, 592, 50 / 49; 14336 x 4096 45 / 37; 2048 x 6144 62 / 16).
    // A gated projection runs there in blocks of 32 rows: 10944 gated columns x 4096 (684 tiles) 75 us, here 52.
    if (p.R < 96) return tiles <= (paired ? 1100 : 600);
    // (A short reduction is a handful of steps of the tiled kernel's loop: K = 512, 128 rows: 2048 columns 11.5 / 4.8, 14336 (896 tiles)
    // 13.6 / 12.0; 256 rows: 2048 16.9 / 4.9, 14336 (1792) 18.7 / 20.8.  Beyond 256 rows nothing here has such a projection and few columns.)
    if (p.K <= 512) return p.R <= 256 && tiles <= 900;
    // The tiled kernel's time is its K loop's as long as its tiles are one round of the chip; here it grows with the tiles (L2 -> LDS
    // traffic, about 11 TB/s).  Tiled / here, us: 2048 x 6144 at 128 rows (128 tiles) 68 / 16, 6144 x 2048 at 256 (768) 28 / 17, 14336 x 4096
    // at 128 (896) 66 / 55, 9728 x 2048 at 200 (1216) 33 / 33, 6144 x 2048 at 400 (1344) 28 / 29, 14336 x 4096 at 200 (1792) 60 / 77.
    const int64_t big = (p.R + 127) / 128 * ((p.N + (paired ? 127 : 255)) / (paired ? 128 : 256));
    return tiles <= 1100 * ((big + 255) / 256);
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
