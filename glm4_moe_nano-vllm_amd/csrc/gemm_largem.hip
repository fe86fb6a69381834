// gemm_largem.hip — LDS-tiled bf16 MFMA GEMM for the prefill regime (many rows per weight
// matrix): dense QKV/O/MLP projections and the grouped expert projections at T >> E.  gfx950.
//
//   * out^T = W · x^T: weight rows on the MFMA row axis (A), tokens on the column axis (B), so a
//     lane's 4 accumulator registers are 4 consecutive output columns of one token and gate/up sit in the same lanes for the
//     fused epilogue.  8 waves as 4(n) x 2(m), wave tile 64(n) x 128(m) (128-row tiles: 64 x 64).
//   * both operand tiles are staged by LDS-DMA (buffer_load ... lds, 1 KiB per instruction); the LDS image is lane-linear, bank
//     conflicts of the 16-row ds_read_b128 fragment reads are removed by permuting the SOURCE chunk: chunk' = chunk ^
//     ((row >> 1) & 7) for 128-B rows, chunk ^ ((row >> 1) & 2) for 64-B rows (found by enumerating the b128 lane groups).
//   * token rows of the B operand are gathered through sorted_token (per-lane source offset of the DMA), so the grouped GEMM
//     needs no pre-gathered activation copy.
//   * raw s_barriers and COUNTED s_waitcnt vmcnt: the DMA of later tiles stays in flight across the barriers.  Fragment reads are
//     inline asm (hipcc would drain the DMA before them).  Waves 4-7 run one barrier behind waves 0-3, so that the two waves of a
//     SIMD alternate between a load interval and an MFMA interval.
//   * persistent: one workgroup per CU walks a list of tiles; the grid is remapped so that one XCD gets a contiguous run of tiles,
//     ordered in bands of 4 row blocks x all n-tiles (n-tile major): the workgroups co-resident on an XCD form a supertile whose
//     operand panels are shared through that XCD's L2.
//
// What bounds it: power, in the products for the most part, and the traffic that feeds them.  On normal values the products alone, from registers, reach 2070
// TFLOP/s, this kernel without its DMA 1813, with operands in L2 1629, as it is 1526 (16384 x 8192 x 8192); on zeros it runs 1.25 to 1.35 times as
// fast, so what counts is both cycles and switching.  Cycles: the ring of the 256-row tiles (CfgR) holds FIVE 32-KiB operand
// tiles (W and X of two K tiles and the next W) in all 160 KiB of LDS, in the order they are needed; an operand's slot is refilled as
// soon as its own last fragment read has retired, so a piece has one to one and a half K tiles to arrive (two 64-KiB buffers: half to
// one, which a loaded memory side does not make), and a phase is 32 MFMAs between two barriers instead of 16 (fp8 x fp8: 16 of four
// times the work).  Switching: consecutive MFMAs share one operand (rows of tiles in alternating direction).  Both together, TFLOP/s
// on normal values, all bit-identical, four steps in one process and the last again with the next in one on another card:
//                               16384 x 8192 x 8192   15074 x 14336 x 4096   15074 x 4096 x 12288   15074 x 6144 x 2048   x 2048 x 6144
//   two buffers, 16 per phase          1363                  1264                   1247                   1204                 1311
//   ... 32 per phase                   1371                  1326                   1282                   1253                 1340
//   ring of five, 32 per phase         1407                  1329                   1315                   1245                 1344
//   ... alternating direction          1439                  1333                   1350                   1257                 1362
//   the same, the other card           1537                  1425                   1440                   1310                 1449
//   ... decisions and stores by wave   1546                  1496                   1447                   1322                 1462
// (Also measured: one barrier per K tile and fragments read a quarter of a tile ahead into 96 registers, 1187 to 1266; wave
// priority in the MFMA interval, equal; K slices of the fragments outermost or tiles of the other operand outermost, equal; 2, 3, 6
// or 8 row blocks per band, up to 7 % slower.)  A tile's stores cost 2 % (K = 8192) to 6 % (K = 2048): all CUs reach them together.
#include "gemm_internal.h"
#include <type_traits>


namespace {

constexpr int LM_BN = 256;    // weight rows per tile (MFMA row axis); 4 waves x 64 rows
constexpr int LM_BAND_ROWS = 4;  // row blocks per L2 supertile band
constexpr int LM_CUT_K = 512;    // shortest reduction whose last tiles are cut
constexpr int LM_SLOT = 32768;   // CfgR: bytes of a ring slot, one operand tile
constexpr int LM_THROUGH_K = 2048;   // longest reduction whose output is written through the L2
constexpr int64_t LM_THROUGH_BF16 = 400 << 20, LM_THROUGH_F32 = 240 << 20;   // bytes of it, at most
constexpr int LM_SC1 = 16;           // cache policy bit of a store: device scope
constexpr int64_t LM_WIDE = 1 << 25;   // output pitch from which 16 fp32 rows do not fit into a buffer

// Tile configurations (the kernel is written once over these):
//   CfgR 256(n) x 256(m) x 64(k), five 32-KiB slots of one operand tile each, two phases of 32 MFMAs per K tile
//   CfgR192 the same with 192(m): phases of 24 MFMAs
//   CfgA 256(n) x 128(m) x 64(k), 3-stage ring, wave tile 64x64  (16 LDS reads + 6 DMA per 32 MFMA)
//   CfgB 256(n) x 256(m) x 32(k), 4-stage ring, wave tile 64x128 (12 LDS reads + 4 DMA per 32 MFMA): only where K is no whole
//        number of 64 or an operand spans 2 GiB (the plain form)
template <int BM_, int BK_, int NSTAGE_, bool RING_ = false, bool W8_ = false, bool A8_ = false, bool WIDE_ = false>
struct LmCfg {
    static constexpr int BM = BM_, BK = BK_, NSTAGE = NSTAGE_;
    static constexpr bool RING = RING_;
    // A8: BOTH operands are OCP fp8 e4m3 in memory and in LDS, BK = 128 elements = 128-byte tile rows — the LDS image,
    // the DMA pieces, the swizzle and the two ds_read_b128 per 16-row tile are byte for byte those of the bf16 CfgR (chunk g4
    // and chunk 4 + g4 of a row are exactly the two register halves of a v_mfma_scale_f32_16x16x128_f8f6f4 operand); a
    // phase is 16 block-scaled MFMAs of K = 128 instead of 32 of K = 32.
    static constexpr bool A8 = A8_;
    static_assert(!A8 || (BK_ == 128 && !W8_), "fp8 x fp8: 128-byte rows of 128 elements");
    // W8: the weight operand is OCP fp8 e4m3 in memory AND in LDS (half the DMA instructions, half the LDS bytes and
    // fragment-read bytes of the weight tile); a fragment is converted to bf16 (exactly: every e4m3 value is a bf16
    // value) between its ds_read and the MFMA, and the per-row dequantisation scale multiplies the fp32 accumulator in the
    // epilogue (WSCALE) — the arithmetic of the expansion pass + bf16 kernel it replaces, bit for bit.
    static constexpr bool W8 = W8_;
    static constexpr bool WIDE = WIDE_;            // output rows too far apart for buffers of 16 (fp8 weights: they have no plain form)
    static constexpr int RB = A8 ? BK : BK * 2;    // bytes per ACTIVATION tile row (and per weight tile row unless W8)
    static constexpr int CPR = RB / 16;            // 16-B chunks per row
    static constexpr int RPI = 1024 / RB;          // rows per DMA instruction
    static constexpr int WRB = W8 ? BK : RB;       // bytes per WEIGHT tile row
    static constexpr int WCPR = WRB / 16;
    static constexpr int WRPI = 1024 / WRB;
    static_assert(!W8 || WRB == 64, "fp8 weight tiles: 64-byte rows (BK = 64)");
    static constexpr int W_DMA = LM_BN / WRPI / 8; // weight DMA instructions per wave per tile
    static constexpr int X_DMA = BM / RPI / 8;     // activation DMA instructions per wave per tile
    static constexpr int DPW = W_DMA + X_DMA;
    static constexpr int KS = A8 ? 2 : BK / 32;    // MFMA k-steps per tile (A8: the two 16-byte halves of ONE K = 128 operand)
    static constexpr int MT = BM / 2 / 16;         // 16-token MFMA tiles per wave (2 waves along m)
    static constexpr int XH = MT / 2;              // of these in each of a K tile's two phases (ring)
    static constexpr int WT = LM_BN * WRB;         // weight tile bytes
    static constexpr int XT = BM * RB;
    static constexpr int STAGE = WT + XT;
    static_assert(!RING || (WT <= LM_SLOT && XT <= LM_SLOT), "an operand tile is one slot");
    static constexpr int LDS = RING ? 5 * LM_SLOT : NSTAGE * STAGE;
    static constexpr int DIST = NSTAGE - 1;        // prefetch distance in tiles
    static constexpr int NF = KS * (4 + MT);       // fragment registers (u32x4) per tile
    // source-chunk permutation that makes the 16-row ds_read_b128 fragment reads conflict free
    __device__ static constexpr int swz(int row) { return RB == 128 ? ((row >> 1) & 7) : ((row >> 1) & 2); }
    // fp8 weight rows are 64 B and a fragment read is a ds_read_b64 at row*64 + 16*slot + 8*(g4 & 1): the 32 lanes of a
    // half wave are rows c = 0..15 x two 8-byte halves; rows c, c+4, c+8, c+12 share their banks unless their slots
    // differ, so slot = chunk ^ ((row >> 2) & 3) — each half wave then covers all 64 banks exactly once
    __device__ static constexpr int wswz(int row) { return W8 ? ((row >> 2) & 3) : swz(row); }
};
using LmCfgA = LmCfg<128, 64, 3>;
using LmCfgB = LmCfg<256, 32, 4>;
using LmCfgR = LmCfg<256, 64, 2, true>;
using LmCfgR192 = LmCfg<192, 64, 2, true>;
using LmCfgR8 = LmCfg<256, 64, 2, true, true>;  // fp8 weight operand (its tiles fill half a slot)
using LmCfgA8 = LmCfg<128, 64, 3, false, true>;
using LmCfgC88 = LmCfg<256, 128, 2, false, false, true>;  // fp8 x fp8 on the block-scaled MFMA: two 64-KiB buffers, the rest of the LDS holds scales
using LmCfgA8Wide = LmCfg<128, 64, 3, false, true, false, true>;
using LmCfgC88Wide = LmCfg<256, 128, 2, false, false, true, true>;

// configurations whose last tiles may be cut (the 128-row one's ring fits into theirs)
template <int MODE, class C>
__host__ __device__ constexpr bool lm_cuts() { return C::RING && C::BM == 256 && !C::W8 && MODE != GEMM_SLICES; }

// single projections of one matrix, with a bias or not
template <int MODE>
__host__ __device__ constexpr bool lm_single() { return MODE != GEMM_GATEUP && MODE != GEMM_DOWN && MODE != GEMM_GLU && MODE != GEMM_SLICES; }

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void glb_void_t;

__device__ const u32x4_t g_zero_page_lm[4] = {};

__device__ __forceinline__ void glds16(const void* gsrc, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((glb_void_t*)gsrc, (lds_void_t*)lds_wave_base, 16, 0, 0);
}
// buffer_load_dwordx4 ... offen lds: per-lane byte offset in a VGPR, K position in the scalar offset
__device__ __forceinline__ void blds16(__amdgpu_buffer_rsrc_t rsrc, void* lds_wave_base, unsigned voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t*)lds_wave_base, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ void lds_read_b128(u32x4_t& dst, unsigned addr) {
    asm volatile("ds_read_b128 %0, %1" : "=v"(dst) : "v"(addr));
}
__device__ __forceinline__ unsigned lds_addr(const void* p) {
    return (unsigned)(uintptr_t)(const lds_void_t*)p;
}
template <int OFF>
__device__ __forceinline__ void lds_read_b128_o(u32x4_t& dst, unsigned addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read_b64_o(u32x2_t& dst, unsigned addr) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}
// 8 fp8 e4m3 (k ascending from byte 0) -> the bf16x8 MFMA fragment, exact
__device__ __forceinline__ u32x4_t lm_fp8x8_to_bf16x8(const u32x2_t d) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf2_t;
    const bf2_t a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d[0], 1.0f, false);
    const bf2_t b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d[0], 1.0f, true);
    const bf2_t c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d[1], 1.0f, false);
    const bf2_t e = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d[1], 1.0f, true);
    return u32x4_t{__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, c),
                   __builtin_bit_cast(unsigned, e)};
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}
// wait for all LDS reads; every fragment register is named so that no consumer moves above it
__device__ __forceinline__ void lds_wait(u32x4_t (&f)[12]) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]),
                   "+v"(f[8]), "+v"(f[9]), "+v"(f[10]), "+v"(f[11])
                 :
                 : "memory");
}
__device__ __forceinline__ void lds_wait(u32x4_t (&f)[16]) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]),
                   "+v"(f[8]), "+v"(f[9]), "+v"(f[10]), "+v"(f[11]), "+v"(f[12]), "+v"(f[13]), "+v"(f[14]), "+v"(f[15])
                 :
                 : "memory");
}
// counted wait: leave the newest `tiles` tiles' DMA (DPW instructions each) in flight
template <int DPW>
__device__ __forceinline__ void dma_wait_leave(int tiles) {
    if (tiles <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (tiles == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(DPW) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * DPW) : "memory");
}

// Row blocks of MB rows that the groups have (uniform)
__device__ __forceinline__ int lm_row_blocks(const int32_t* __restrict__ offs, int G, int MB, int lane) {
    int n = 0;
    for (int g = lane; g < G; g += 64) n += (offs[g + 1] - offs[g] + MB - 1) / MB;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    return __builtin_amdgcn_readfirstlane(n);
}

// The (group, first row, rows) of row-block number `target` of a lane, targets of the lanes in any order; g = -1 if there is none.
__device__ __forceinline__ void lm_locate_lanes(const int32_t* __restrict__ offs, int G, int64_t R, int MB, int target, int lane, int& g, int& m0, int& cnt) {
    g = -1;
    m0 = 0;
    cnt = 0;
    if (offs == nullptr) {  // all groups have the R rows (one group, or the K slices of GEMM_SLICES)
        const int nb = (int)((R + MB - 1) / MB);
        if (target < nb * G) {
            g = target / nb;
            m0 = (target % nb) * MB;
            cnt = (int)((R - m0) < MB ? (R - m0) : MB);
        }
        return;
    }
    int base = 0;
    for (int b = 0; b < G; b += 64) {  // row blocks of 64 groups at a time, summed over the lanes; every lane searches in the sums
        const int gi = b + lane;
        int lo = 0, c = 0;
        if (gi < G) {
            lo = offs[gi];
            c = offs[gi + 1] - lo;
        }
        int incl = (c + MB - 1) / MB;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        int at = 0;  // groups of these 64 that end at or before the target
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) at += (__shfl(incl, at + o - 1, 64) + base <= target) ? o : 0;
        const int before = __shfl(incl, at > 0 ? at - 1 : 0, 64);
        const int glo = __shfl(lo, at, 64), gc = __shfl(c, at, 64), end = __shfl(incl, at, 64);
        if (g < 0 && target >= base && target < base + end && b + at < G) {
            const int off = (target - base - (at > 0 ? before : 0)) * MB;
            g = b + at;
            m0 = glo + off;
            cnt = gc - off < MB ? gc - off : MB;
        }
        base += __shfl(incl, 63, 64);
    }
}

// Between two tiles the next tile's first operand tiles are put in flight BEFORE the finished tile's epilogue, so that their
// latency hides behind the epilogue's stores.
// LEAN: operand tiles come in by buffer_load ... lds with a per-lane byte offset that is fixed for the whole tile and the K position in
// the SCALAR offset, fragment reads use one base register per k-step plus immediate offsets, 16-byte stores (the packed results of two
// neighbouring 16-column tiles are exchanged between the lane rows).  Needs K % BK == 0, x and W spans < 2 GiB, N % 8 == 0.  The other
// form covers everything else.
// blocks: row blocks there are, or more than the list has (CUT: of 256 rows).  CUT: tiles of 256 rows from `first` on, each in two of 128.
template <int MODE, class C, bool LEAN, bool WSCALE, bool CUT>
__device__ __forceinline__ void largem_tiles(const GemmParams& p, char* smem, int n_tiles, int total_tiles, int LM_BAND, int blocks, int first) {
    constexpr bool F32 = MODE == GEMM_SLICES || MODE == GEMM_F32 || MODE == GEMM_CAP || MODE == GEMM_XIELU32 || MODE == GEMM_COLS32;  // stores fp32 rows (p.yf)
    constexpr bool BIAS = lm_single<MODE>() && MODE != GEMM_QKV;   // (in the common epilogue)
    constexpr bool GROUPED = MODE == GEMM_GATEUP || MODE == GEMM_DOWN;
    static_assert(LEAN || (!C::RING && !C::W8 && !C::A8), "the plain form has the plain ring");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wid & 3, wm = wid >> 2;
    const int c = lane & 15, g4 = lane >> 4;
    const int K = p.K;
    const int nk = (K + C::BK - 1) / C::BK;

    // XCD-aware tile list (bijective for any tile count): workgroups with equal id%8 share an XCD and get one
    // contiguous run of the band-ordered tile list
    int chunk_base, chunk_len;
    {
        const int q = total_tiles >> 3, r = total_tiles & 7, x = blockIdx.x & 7;
        chunk_base = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q;
        chunk_len = q + (x < r ? 1 : 0);
    }
    const int pstep = gridDim.x >> 3;  // host launches a multiple of 8 workgroups
    const int pos0 = blockIdx.x >> 3;

    // tile state: *_c = tile being computed / stored, plain = tile whose operands are being staged
    int grp = -1, m0 = 0, mcnt = 0, ntile = 0;
    // Tile table: lane i of every wave holds tile position ti0 + i of this workgroup's list, found for 64 positions at a time by the
    // wave itself (no LDS, no barrier: the ring takes all of the LDS).
    int tab_g = -1, tab_m0 = 0, tab_cn = 0;
    int ti = 0;  // next position of the list
    // next valid tile of the list (uniform)
    auto find_tile = [&]() -> bool {
        while (pos0 + ti * pstep < chunk_len) {
            if ((ti & 63) == 0) {
                const int bid = chunk_base + pos0 + (ti + lane) * pstep;
                if constexpr (MODE != GEMM_SLICES) {
                    const int half = CUT ? bid & 1 : 0;
                    int t = CUT ? first + (bid >> 1) : bid;
                    const int band = t / (LM_BAND * n_tiles), b0 = band * LM_BAND;
                    const int high = max(1, min(LM_BAND, blocks - b0));   // row blocks of the band
                    t -= b0 * n_tiles;
                    const int blk = b0 + t % high, ntile_ = t / high;
                    constexpr int BLK = CUT ? 256 : C::BM;
                    if (GROUPED && p.offs != nullptr) {
                        lm_locate_lanes(p.offs, p.G, p.R, BLK, blk, lane, tab_g, tab_m0, tab_cn);
                    } else {
                        const int64_t left = p.R - (int64_t)blk * BLK;
                        tab_g = 0;
                        tab_m0 = blk * BLK;
                        tab_cn = (int)(left < BLK ? left : (int64_t)BLK);
                    }
                    if constexpr (CUT) {
                        tab_m0 += half * 128;
                        tab_cn = min(tab_cn - half * 128, 128);
                    }
                    if (bid >= total_tiles || tab_cn <= 0 || ntile_ >= n_tiles) tab_g = -1;
                    tab_cn |= ntile_ << 9;  // up to 256 rows, up to 2^22 column tiles (checked by the host)
                } else {
                    const int band = bid / (LM_BAND * n_tiles), rem = bid % (LM_BAND * n_tiles);
                    lm_locate_lanes(nullptr, p.G, p.R, C::BM, band * LM_BAND + rem % LM_BAND, lane, tab_g, tab_m0, tab_cn);
                    tab_cn |= (rem / LM_BAND) << 9;
                }
            }
            const int at = ti & 63;
            ++ti;
            grp = __builtin_amdgcn_readlane(tab_g, at);
            if (grp >= 0) {
                m0 = __builtin_amdgcn_readlane(tab_m0, at);
                const int cn = __builtin_amdgcn_readlane(tab_cn, at);
                mcnt = cn & 511;
                ntile = cn >> 9;
                return true;
            }
        }
        return false;
    };

    // ---- DMA sources.  One instruction = RPI tile rows x CPR chunks (1 KiB); lane → row
    // +(lane / CPR), LDS position lane % CPR holds global chunk (lane % CPR) ^ swz(row). ----
    const bf16_t* wsrc[C::W_DMA];
    const bf16_t* xsrc[C::X_DMA];
    int wch[C::W_DMA], xch[C::X_DMA];
    unsigned wvo[C::W_DMA], xvo[C::X_DMA];  // LEAN: byte offsets of this lane's chunk at k = 0
    __amdgpu_buffer_rsrc_t wrs, xrs;
    if (LEAN) xrs = make_rsrc(p.x);
    auto setup_sources = [&]() {
        if constexpr (LEAN) {
            // descriptor of the group's weights (wave-uniform)
            const int64_t goff = (int64_t)grp * p.w_gstride;
            if constexpr (C::W8 || C::A8) wrs = make_rsrc(reinterpret_cast<const char*>(p.w) + goff);  // fp8: strides in bytes
            else wrs = make_rsrc(p.w + goff);
#pragma unroll
            for (int i = 0; i < C::W_DMA; ++i) {
                const int row = (wid * C::W_DMA + i) * C::WRPI + lane / C::WCPR;
                const int ch = (lane % C::WCPR) ^ C::wswz(row);
                int wr;
                if (gemm_paired(MODE)) wr = (row >> 7) * p.N + min(ntile * 128 + (row & 127), p.N - 1);
                else wr = min(ntile * LM_BN + row, p.N - 1);
                if constexpr (C::W8 || C::A8) wvo[i] = (unsigned)(wr * (int)p.ldw + ch * 16);
                else wvo[i] = (unsigned)(wr * (int)p.ldw + ch * 8) * 2u;
            }
#pragma unroll
            for (int i = 0; i < C::X_DMA; ++i) {
                const int row = (wid * C::X_DMA + i) * C::RPI + lane / C::CPR;
                const int ch = (lane % C::CPR) ^ C::swz(row);
                const int mr = row < mcnt ? row : 0;
                const int srow = p.src ? p.src[m0 + mr] : m0 + mr;
                if constexpr (C::A8) xvo[i] = (unsigned)(srow * (int)p.ldx + ch * 16);  // fp8 activations: ldx in bytes
                else xvo[i] = (unsigned)(srow * (int)p.ldx + (MODE == GEMM_SLICES ? grp * K : 0) + ch * 8) * 2u;
            }
        } else {
            const bf16_t* wg = p.w + (int64_t)grp * p.w_gstride;
#pragma unroll
            for (int i = 0; i < C::W_DMA; ++i) {
                const int row = (wid * C::W_DMA + i) * C::RPI + lane / C::CPR;  // 0..255
                const int ch = (lane % C::CPR) ^ C::swz(row);
                wch[i] = ch;
                int wr;
                if (gemm_paired(MODE)) {
                    const int half = row >> 7;  // 0: gate rows, 1: up rows
                    wr = half * p.N + min(ntile * 128 + (row & 127), p.N - 1);
                } else {
                    wr = min(ntile * LM_BN + row, p.N - 1);
                }
                wsrc[i] = wg + (int64_t)wr * p.ldw + ch * 8;
            }
#pragma unroll
            for (int i = 0; i < C::X_DMA; ++i) {
                const int row = (wid * C::X_DMA + i) * C::RPI + lane / C::CPR;  // 0..BM-1
                const int ch = (lane % C::CPR) ^ C::swz(row);
                xch[i] = ch;
                const int mr = row < mcnt ? row : 0;
                const int64_t srow = p.src ? (int64_t)p.src[m0 + mr] : (int64_t)(m0 + mr);
                xsrc[i] = p.x + srow * p.ldx + (MODE == GEMM_SLICES ? (int64_t)grp * K : 0) + ch * 8;
            }
        }
    };
    const bf16_t* zero = reinterpret_cast<const bf16_t*>(g_zero_page_lm);
    // this wave's DMA of an operand tile of K tile kt to LDS offset off
    auto stage_w = [&](int off, int kt) {
        char* dst = smem + off + wid * C::W_DMA * 1024;
        const int k0 = kt * C::BK;
#pragma unroll
        for (int i = 0; i < C::W_DMA; ++i) {
            if constexpr (LEAN) blds16(wrs, dst + i * 1024, wvo[i], k0 * ((C::W8 || C::A8) ? 1 : 2));
            else glds16(k0 + wch[i] * 8 < K ? wsrc[i] + k0 : zero, dst + i * 1024);
        }
    };
    auto stage_x = [&](int off, int kt) {
        char* dst = smem + off + wid * C::X_DMA * 1024;
        const int k0 = kt * C::BK;
#pragma unroll
        for (int i = 0; i < C::X_DMA; ++i) {
            if constexpr (LEAN) blds16(xrs, dst + i * 1024, xvo[i], k0 * (C::A8 ? 1 : 2));
            else glds16(k0 + xch[i] * 8 < K ? xsrc[i] + k0 : zero, dst + i * 1024);
        }
    };
    auto stage = [&](int slot, int kt) {
        stage_w(slot * C::STAGE, kt);
        stage_x(slot * C::STAGE + C::WT, kt);
    };
    // A8 DOWN: the E8M0 block scales of the tile's activation rows behind the two buffers (16 KiB), two 1-KiB LDS-DMA pieces
    // per wave.  LDS image: 16-byte slot (g * 256 + row) = the scales of (row, natural block 4 kt + g) for kt = 0 .. 15 — a
    // lane (row c of X tile mt, lane row g4) reads ONE dword of its slot every four K tiles (bytes kt & ~3 .. + 3) and shifts
    // the byte of the K tile into place (one ds_read_u8 per X tile and K tile out of [row][64 B] records: 8-way bank conflicts,
    // the down projection gained nothing over bf16).
    constexpr bool XBS = C::A8 && MODE == GEMM_DOWN;
    constexpr int XBS_OFF = C::NSTAGE * C::STAGE;
    auto stage_scales = [&]() {
        if constexpr (XBS) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int slot = (wid * 2 + i) * 64 + lane;       // lane-linear destination: slot = g * 256 + row
                const int row = slot & 255, g = slot >> 8;
                const int mr = row < mcnt ? row : 0;
                glds16(p.xbscale + (int64_t)(m0 + mr) * 64 + g * 16, smem + XBS_OFF + (wid * 2 + i) * 1024);
            }
        }
    };
    auto fill_ring = [&]() {
        if constexpr (C::RING) {
            // operand tile j (W of K tile k: 2k, X: 2k + 1) lives in slot j % 5
            stage_w(0, 0);
            stage_x(LM_SLOT, 0);
            if (nk > 1) {
                stage_w(2 * LM_SLOT, 1);
                stage_x(3 * LM_SLOT, 1);
            }
        } else if constexpr (C::A8) {
            // both operands of K tile 0 and the weights of K tile 1 (their slot is the first one the loop refills)
            stage_scales();
            stage(0, 0);
            if (nk > 1) stage_w(C::STAGE, 1);
        } else {
#pragma unroll
            for (int d = 0; d < C::DIST; ++d)
                if (d < nk) stage(d, d);
        }
    };

    // ---- fragment read offsets relative to the stage base: lane (c,g4) reads row +c, chunk 4ks+g4
    unsigned rel[C::NF];  // per k-step: 4 weight fragments then MT activation fragments
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int wrow;
            if (gemm_paired(MODE)) wrow = (t < 2 ? wn * 32 + 16 * t : 128 + wn * 32 + 16 * (t - 2)) + c;
            else wrow = wn * 64 + 16 * t + c;
            if constexpr (C::W8)  // 8 bytes: k = 32 ks + 8 g4 .. +8 = chunk 2 ks + (g4 >> 1), half g4 & 1
                rel[ks * (4 + C::MT) + t] = wrow * C::WRB + (((2 * ks + (g4 >> 1)) ^ C::wswz(wrow)) << 4) + ((g4 & 1) << 3);
            else
                rel[ks * (4 + C::MT) + t] = wrow * C::RB + (((4 * ks + g4) ^ C::swz(wrow)) << 4);
        }
#pragma unroll
        for (int t = 0; t < C::MT; ++t) {
            const int xrow = wm * (C::BM / 2) + 16 * t + c;
            rel[ks * (4 + C::MT) + 4 + t] = (C::RING ? 0 : C::WT) + xrow * C::RB + (((4 * ks + g4) ^ C::swz(xrow)) << 4);
        }
    }
    const unsigned base = lds_addr(smem);
    // LEAN: one base per k-step and operand; the tile index inside the operand is an immediate offset
    // (the swizzle depends on the low bits of the row only, i.e. on c)
    unsigned fbw[C::KS], fbx[C::KS];
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) {
        fbw[ks] = base + rel[ks * (4 + C::MT)];
        fbx[ks] = base + rel[ks * (4 + C::MT) + 4];
    }
    // all fragment reads of a K tile (slot byte offset so, wave-uniform)
    // W8: behind the read wait, the weight fragments fp8 -> bf16 (the asm reads are invisible to the compiler: nothing may
    // touch fr[] between a read and the lgkmcnt wait, which is why they have registers of their own)
    auto frags_cvt = [&](u32x4_t (&f)[C::NF], u32x2_t (&fr)[C::W8 ? C::KS * 4 : 1]) {
        if constexpr (C::W8) {
#pragma unroll
            for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    asm volatile("" : "+v"(fr[ks * 4 + t]));
                    f[ks * (4 + C::MT) + t] = lm_fp8x8_to_bf16x8(fr[ks * 4 + t]);
                }
        }
    };
    auto read_frags = [&](u32x4_t (&f)[C::NF], u32x2_t (&fr)[C::W8 ? C::KS * 4 : 1], unsigned so) {
        static_for<C::KS>([&](auto ksc) {
            constexpr int ks = decltype(ksc)::value;
            const unsigned aw = fbw[ks] + so, ax = fbx[ks] + so;
            static_for<4>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                constexpr int off = gemm_paired(MODE) ? (t < 2 ? 16 * t : 128 + 16 * (t - 2)) * C::WRB : 16 * t * C::WRB;
                if constexpr (C::W8) lds_read_b64_o<off>(fr[ks * 4 + t], aw);  // fp8 as read; frags_cvt() fills f[]
                else lds_read_b128_o<off>(f[ks * (4 + C::MT) + t], aw);
            });
            static_for<C::MT>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                lds_read_b128_o<16 * t * C::RB>(f[ks * (4 + C::MT) + 4 + t], ax);
            });
        });
    };

    // Store instructions a wave issues behind the ring fill of the next tile, where their number is known: the waits that open a tile
    // leave that many in flight (vmcnt counts in issue order).  -1: not known, wait for everything.
    constexpr int LM_NOUT = gemm_paired(MODE) ? 2 : 4;
    constexpr int STORES = C::MT * (F32 ? 4 : LM_NOUT / 2);
    int pending_stores = 0;
    // leave `pending_stores` stores and L later DMA instructions in flight
    auto wait_behind_stores = [&](auto lc) {
        constexpr int L = decltype(lc)::value;
        if (LEAN && pending_stores == STORES) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(STORES + L) : "memory");
        else if (pending_stores == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    if (!find_tile()) return;
    setup_sources();
    fill_ring();
    for (;;) {
        // the tile whose ring is filling is now the tile being computed
        const int grp_c = grp, m0_c = m0, mcnt_c = mcnt, ntile_c = ntile;
        f32x4_t acc[4][C::MT];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < C::MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        using I0 = std::integral_constant<int, 0>;
        using IH = std::integral_constant<int, C::XH>;

        if constexpr (C::RING) {
            if (nk > 1) wait_behind_stores(std::integral_constant<int, C::DPW>{});  // K tile 1 stays in flight
            else wait_behind_stores(I0{});
        } else {
            wait_behind_stores(I0{});
        }
        __builtin_amdgcn_s_barrier();                 // every share of the first K tile(s) landed
        if constexpr (C::RING || C::A8) {
        // ---- two phases per K tile, each = load interval | barrier | 32 MFMAs (fp8 x fp8: 16 of K = 128) | barrier; waves 4-7 run
        // one barrier behind waves 0-3, so the two waves of a SIMD alternate between the two kinds of interval.
        //   phase   fragment reads of K tile kt        DMA issued: ring                    DMA issued: two buffers (A8)           MFMAs
        //     A     W tiles 0-3 (8), X tiles 0-3 (8)   W(kt+2) -> slot of X(kt-1)          X(kt+1) -> buffer of kt-1             W0-3 x X0-3
        //     B     X tiles 4-7 (8)                    X(kt+2) -> slot of W(kt)            W(kt+2) -> buffer of kt               W0-3 x X4-7
        //           then the counted wait for this wave's share of K tile kt+1 (what is younger stays in flight)
        // Every load interval ends with lgkmcnt(0) BEFORE its barrier, so a fragment read has retired when its wave passes that
        // barrier.  Barrier epochs: waves 0-3 run load interval P (= 2 kt + phase) in epoch 2P, waves 4-7 in epoch 2P+1.
        //   WAR  W(kt) is last read in load interval 2kt (retired by the end of epoch 4kt+1) and its slot refilled from load
        //        interval 2kt+1 (epoch >= 4kt+2).  X(kt-1) is last read in load interval 2kt-1 (epoch <= 4kt-1) and its slot
        //        refilled from load interval 2kt (epoch >= 4kt).
        //   RAW  K tile kt+1 is first read in load interval 2kt+2 (epoch >= 4kt+4); every wave waited for its own pieces of
        //        it at the end of load interval 2kt+1 (epoch <= 4kt+3), i.e. before barrier 4kt+4.
        // Between tiles: the last fragment read retires before the last barrier but one, and every wave passes the barrier after the
        // loop before it refills the ring.
        if (wid >= 4) __builtin_amdgcn_s_barrier();   // the stagger
        constexpr int XH = C::XH;
        u32x4_t fw[8], fx[2 * XH];  // [k-step][W tile 0-3], [k-step][X tile of the current half]
        int sxw[8] = {127, 127, 127, 127, 127, 127, 127, 127};  // A8: per X tile, the E8M0 scale bytes of four K tiles (127 = 2^0:
                                                                 // gate|up, whose activation scale is per token)
        int ksh = 0;                                             // 8 * (K tile & 3): the byte of the current K tile
        const unsigned sx_base = lds_addr(smem) + XBS_OFF + (g4 * 256 + wm * (C::BM / 2) + c) * 16;
        auto rd_s = [&](int kt_) {  // every fourth K tile, in its phase A (behind the same lgkmcnt wait)
            if constexpr (XBS) {
                if ((kt_ & 3) == 0) {
                    const unsigned a_ = sx_base + kt_;
#define GLM_RD_S(J) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(sxw[J]) : "v"(a_), "i"((J) * 256))
                    GLM_RD_S(0); GLM_RD_S(1); GLM_RD_S(2); GLM_RD_S(3); GLM_RD_S(4); GLM_RD_S(5); GLM_RD_S(6); GLM_RD_S(7);
#undef GLM_RD_S
                }
            }
        };
        u32x2_t fwr[C::W8 ? 8 : 1];  // W8: the fragments as read (fp8), converted into fw behind the read wait
        auto pin = [&](u32x4_t& r) { asm volatile("" : "+v"(r)); };
        // W tiles 0-3, both k-steps
        auto rd_w = [&](unsigned so) {
            static_for<C::KS>([&](auto ksc) {
                constexpr int ks = decltype(ksc)::value;
                const unsigned aw = fbw[ks] + so;
                static_for<4>([&](auto tc) {
                    constexpr int t = decltype(tc)::value;
                    constexpr int off = gemm_paired(MODE) ? (t < 2 ? 16 * t : 128 + 16 * (t - 2)) * C::WRB : 16 * t * C::WRB;
                    if constexpr (C::W8) lds_read_b64_o<off>(fwr[ks * 4 + t], aw);
                    else lds_read_b128_o<off>(fw[ks * 4 + t], aw);
                });
            });
        };
        // X tiles m0 .. m0+3 into fx[ks * 4 + j], both k-steps
        auto rd_x = [&](unsigned so, auto m0c) {
            constexpr int mt0 = decltype(m0c)::value;
            static_for<C::KS>([&](auto ksc) {
                constexpr int ks = decltype(ksc)::value;
                const unsigned ax = fbx[ks] + so;
                static_for<XH>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    lds_read_b128_o<16 * (mt0 + j) * C::RB>(fx[ks * XH + j], ax);
                });
            });
        };
        auto reads_done = [&](bool with_w) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (with_w) {
                if constexpr (C::W8) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        asm volatile("" : "+v"(fwr[i]));
                        fw[i] = lm_fp8x8_to_bf16x8(fwr[i]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) pin(fw[i]);
                if constexpr (XBS) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(sxw[j]));
                }
            }
#pragma unroll
            for (int i = 0; i < 2 * XH; ++i) pin(fx[i]);
        };
        // W tiles 0-3 x X tiles m0 .. m0+3, every MFMA sharing an operand with the one before it
        auto mfmas = [&](auto m0c) {
            constexpr int mt0 = decltype(m0c)::value;
            if constexpr (C::A8) {
                // ONE K = 128 MFMA per (W tile, X tile): registers 0-3 = chunk g4, registers 4-7 = chunk 4 + g4 of the row
                typedef int v8i_t __attribute__((ext_vector_type(8)));
                typedef unsigned u32x8_t __attribute__((ext_vector_type(8)));
                static_for<16>([&](auto ic) {
                    constexpr int i = decltype(ic)::value, t = i / 4, j = t & 1 ? 3 - i % 4 : i % 4;
                    const u32x8_t a8 = __builtin_shufflevector(fw[t], fw[4 + t], 0, 1, 2, 3, 4, 5, 6, 7);
                    const u32x8_t b8 = __builtin_shufflevector(fx[j], fx[4 + j], 0, 1, 2, 3, 4, 5, 6, 7);
                    acc[t][mt0 + j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        __builtin_bit_cast(v8i_t, a8), __builtin_bit_cast(v8i_t, b8), acc[t][mt0 + j], 0, 0, 0, 127, 0,
                        XBS ? (int)((unsigned)sxw[mt0 + j] >> ksh) : 127);
                });
            } else {
                static_for<C::KS * 4 * XH>([&](auto ic) {
                    constexpr int i = decltype(ic)::value, ks = i / (4 * XH);
                    constexpr int t = ks & 1 ? 3 - i / XH % 4 : i / XH % 4, j = i / XH & 1 ? XH - 1 - i % XH : i % XH;
                    acc[t][mt0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fw[ks * 4 + t]),
                                                                              __builtin_bit_cast(bf16x8_t, fx[ks * XH + j]), acc[t][mt0 + j], 0, 0, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto close_load = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
        };
        unsigned ow = 0, ox = C::RING ? LM_SLOT : 0, of = 4 * LM_SLOT;  // ring: slots of W(kt) and X(kt), and the free one
        auto next2 = [](unsigned o) { return o >= 3 * LM_SLOT ? o - 3 * LM_SLOT : o + 2 * LM_SLOT; };
        // rows_a, rows_b: this wave has rows in the phase; where it has none its MFMA interval is a barrier
        auto k_tiles = [&](auto rows_a, auto rows_b) __attribute__((always_inline)) {
#pragma unroll 1
            for (int kt = 0; kt < nk; ++kt) {
                const bool has1 = kt + 1 < nk, has2 = kt + 2 < nk;
                if constexpr (C::A8) {
                    ow = ox = (kt & 1) * C::STAGE;
                    ksh = (kt & 3) * 8;
                }
                // ---- phase A
                rd_w(ow);
                rd_x(ox, I0{});
                rd_s(kt);
                __builtin_amdgcn_sched_barrier(0);  // the reads are issued before the DMA, which then runs under their round trip
                if constexpr (C::RING) {
                    if (has2) stage_w(of, kt + 2);
                } else {
                    if (has1) stage_x((ow ^ C::STAGE) + C::WT, kt + 1);
                }
                reads_done(true);
                close_load();
                if (rows_a) mfmas(I0{});
                __builtin_amdgcn_s_barrier();
                // ---- phase B
                rd_x(ox, IH{});
                __builtin_amdgcn_sched_barrier(0);
                if (has2) {
                    if constexpr (C::RING) stage_x(ow, kt + 2);
                    else stage_w(ow, kt + 2);
                }
                reads_done(false);
                constexpr int YOUNGER = C::RING ? C::DPW : C::W_DMA;
                if (!has2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                else if (C::RING && kt == 0) wait_behind_stores(std::integral_constant<int, YOUNGER>{});  // (K tile 1 was issued in front of them)
                else asm volatile("s_waitcnt vmcnt(%0)" ::"i"(YOUNGER) : "memory");
                close_load();
                if (rows_b) mfmas(IH{});
                __builtin_amdgcn_s_barrier();
                if constexpr (C::RING) {
                    of = ox;
                    ow = next2(ow);
                    ox = next2(ox);
                }
            }
        };
        // A group's last rows go through a loop of their own: with the tests in the one loop whole tiles were 1 to 2 % slower.  Without / with, us:
        // gate|up, down of 64 experts, 6 of 1024 x 2048 at 6000 tokens 337 / 308, 200 / 186, 8 of 1408 x 4096 at 4096 800 / 774, 445 / 431, at 15074
        // 2181 / 2184, 1258 / 1222.  (The rows dealt anew to both waves along m: 10 to 40 registers spilled, whole tiles 2 to 5 % slower.)
        // A projection without groups has one such block per column tile: there the second loop costs more than it gives (0.3 to 1 %).
        if (!GROUPED || C::BM != 256 || mcnt_c > 192) k_tiles(std::true_type{}, std::true_type{});
        else if constexpr (GROUPED) k_tiles(mcnt_c > wm * 128, mcnt_c > wm * 128 + 64);
        if (wid < 4) __builtin_amdgcn_s_barrier();  // match the other group's extra barrier
        } else {
        // ---- main loop: two phases per K tile, waves 4-7 run ONE BARRIER BEHIND waves 0-3 ----
        //   phase 1: DMA issue of tile kt+DIST + LDS fragment reads of tile kt + counted wait for
        //            this wave's share of tile kt+1, then barrier
        //   phase 2: the tile's MFMAs, then barrier
        // The two waves that share a SIMD (w, w+4) are therefore always in opposite phases: one feeds
        // the matrix pipe while the other issues loads (in lockstep the pipe idles ~60 % of the time).
        // Ordering under the stagger (the other group sits one barrier earlier/later):
        //   RAW  tile kt+1 is read in phase 1 of kt+1, i.e. after this group's B2(kt) = other group's
        //        B1(kt) (or later); every wave waited for its share of kt+1 BEFORE its own B1(kt).
        //   WAR  tile kt+DIST overwrites the slot of kt-1 in phase 1 of kt, i.e. after this group's
        //        B2(kt-1) >= other group's B1(kt-1); every wave finished reading kt-1 before its own
        //        B1(kt-1).
        if (wid >= 4) __builtin_amdgcn_s_barrier();   // the stagger
        int so = 0;  // ring slot of tile kt, its offset
        for (int kt = 0; kt < nk; ++kt) {
            // ---------------- phase 1 ----------------
            u32x4_t f[C::NF];
            u32x2_t fr[C::W8 ? C::KS * 4 : 1];
            if (kt + C::DIST < nk) {  // into the slot of tile kt-1
                const int no = so == 0 ? (C::NSTAGE - 1) * C::STAGE : so - C::STAGE;
                stage_w(no, kt + C::DIST);
                stage_x(no + C::WT, kt + C::DIST);
            }
            if constexpr (LEAN) {
                read_frags(f, fr, so);
            } else {
                const unsigned sb = base + so;
#pragma unroll
                for (int i = 0; i < C::NF; ++i) lds_read_b128(f[i], sb + rel[i]);
            }
            // this wave's share of tile kt+1: leave only the tiles newer than kt+1 in flight
            if constexpr (C::DIST == 2) {
                if (kt + C::DIST < nk) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(C::DPW) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else dma_wait_leave<C::DPW>(min(kt + C::DIST, nk - 1) - (kt + 1));
            lds_wait(f);
            frags_cvt(f, fr);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();  // B1
            // ---------------- phase 2 ----------------
            if constexpr (!LEAN) __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
                for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                    for (int mt = 0; mt < C::MT; ++mt)
                        acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, f[ks * (4 + C::MT) + nt]),
                            __builtin_bit_cast(bf16x8_t, f[ks * (4 + C::MT) + 4 + mt]), acc[nt][mt], 0, 0, 0);
            if constexpr (!LEAN) __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();  // B2
            so = so == (C::NSTAGE - 1) * C::STAGE ? 0 : so + C::STAGE;
        }
        if (wid < 4) __builtin_amdgcn_s_barrier();  // match the other group's extra barrier
        }

        // The epilogue of the fp8 x fp8 gate|up kernel LOADS (weight-row scales, token scales) and vector-memory results return in issue
        // order — behind the ring fill they cost a whole fill latency per tile (epilogue 23.5k cycles against 6.0k for bf16).
        // There the next tile's fill is issued once the first 16-row block of the epilogue has its loads back, i.e. behind them and
        // in front of the bulk of the stores, which lie on both sides of it: the next tile waits for everything.
        // (The scale vectors as LDS-DMA pieces of the ring fill: no gain.)
        constexpr bool LATE_FILL = C::A8 && gemm_paired(MODE);
        // What the epilogue reads of the finished tile's rows and columns: requested in front of the ring fill (waiting for a load issued behind the
        // fill would drain the fill first).
        float e_row[C::MT], e_col[4][4];
        unsigned e_bias[4][2];
        // column of the wave's first output column, or gate column, of tile t
        auto col = [&](int t, int r) { return gemm_paired(MODE) ? ntile_c * 128 + wn * 32 + 16 * (t & 1) + 4 * g4 + r : ntile_c * LM_BN + wn * 64 + 16 * t + 4 * g4 + r; };
        if constexpr (LEAN) {
            if constexpr (MODE == GEMM_DOWN) {
                const bool sc_on = grp_c < p.n_scaled;
#pragma unroll
                for (int mt = 0; mt < C::MT; ++mt) {
                    const int row = wm * (C::BM / 2) + 16 * mt + c;
                    e_row[mt] = (sc_on && row < mcnt_c) ? bf2f(p.scale[m0_c + row]) : 1.0f;
                }
            }
            if constexpr (WSCALE && !LATE_FILL) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        e_col[t][r] = p.wscale[(int64_t)grp_c * p.wscale_gstride + (gemm_paired(MODE) && t > 1 ? p.N : 0) + min(col(t, r), p.N - 1)];
            }
        }
        // The plain form's bias too: read element by element between its stores, which it then waited for, us, behind a tile's four stores of a row block / behind
        // each of them / this: 664 x 1168 x 1640 28.4 / 30.5 / 24.5, 1554 x 24 x 168 10.4 / 10.9 / 6.7, 4100 x 2044 x 2056 68.9 / 72.5 / 61.3, 12000 x 6148 x
        // 2056 343 / 360 / 309 (306 without a bias).
        if constexpr (BIAS) {
            if (p.bias != nullptr) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; r += 2) e_bias[t][r >> 1] = p.bias[min(col(t, r), p.N - 1)] | (unsigned)p.bias[min(col(t, r + 1), p.N - 1)] << 16;
            }
        }
        // ---- next tile: every wave is past its last LDS read, so the ring can be refilled right away ----
        const bool more = find_tile();
        if (more) setup_sources();   // (its own loads — the gathered source rows — go out here, behind the epilogue's)
        if constexpr (LEAN && MODE == GEMM_DOWN) {
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt) asm volatile("" : "+v"(e_row[mt]));  // the loads stay above the fill
        }
        if constexpr (LEAN && WSCALE && !LATE_FILL) {
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(e_col[i >> 2][i & 3]));
        }
        if constexpr (BIAS) {
            if (p.bias != nullptr) {
#pragma unroll
                for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(e_bias[i >> 1][i & 1]));
            }
        }
        auto start_next = [&]() {
            if (more) fill_ring();
        };
        if constexpr (!LATE_FILL) start_next();
        __builtin_amdgcn_sched_barrier(0);   // (pending_stores counts on the order)

        // ---- epilogue of the finished tile ----
        int stored = -1;  // (pending_stores)
        constexpr int NOUT = gemm_paired(MODE) ? 2 : 4;  // 16-column output tiles per wave
        const int ncol_w = gemm_paired(MODE) ? ntile_c * 128 + wn * 32 : ntile_c * LM_BN + wn * 64;
        const bool scaled = MODE == GEMM_DOWN && grp_c < p.n_scaled;
        // the mode's activation on an element of column tile t; kind: p.act.kind where it is one of several with long code (GEMM_COLS32, with_kind)
        auto act = [&](float a, int t, int r, auto kind) __attribute__((always_inline)) {
            const int n = ncol_w + 16 * t + 4 * g4 + r;
            if constexpr (MODE == GEMM_XIELU) return glm_xielu_fast(p.act.a, p.act.b, a);
            else if constexpr (MODE == GEMM_XIELU32) return glm_act_precise(GlmAct{GLM_ACT_XIELU, p.act.a, p.act.b}, a, n);
            else if constexpr (MODE == GEMM_CAP || MODE == GEMM_CAP16) return p.act.a * tanhf(a / p.act.a);
            else if constexpr (MODE == GEMM_COLS) return glm_act_cols(p.act, a, n);
            else if constexpr (MODE == GEMM_COLS32) return glm_act_precise(GlmAct{decltype(kind)::value, p.act.a, p.act.b}, a, n);
            else return a;
        };
        auto with_kind = [&](auto&& f) __attribute__((always_inline)) {
            if constexpr (MODE != GEMM_COLS32) f(std::integral_constant<int, GLM_ACT_NONE>{});
            else if (p.act.kind == GLM_ACT_SILU_GATE) f(std::integral_constant<int, GLM_ACT_SILU_GATE>{});
            else if (p.act.kind == GLM_ACT_RELU2_GATE) f(std::integral_constant<int, GLM_ACT_RELU2_GATE>{});
            else f(std::integral_constant<int, GLM_ACT_GATE>{});
        };
        if constexpr (MODE == GEMM_QKV) {
            // ---- QKV epilogue: bias, bf16 rounding (the packed qkv value of the reference, linear.py:75), rotary on the
            // first 64 dims of every q / k head, split, cache scatter.  A wave's 64 columns are one half of one head (ncol_w
            // is a multiple of 64): the rotary half pairs column i with i + 32 = accumulator tiles t and t + 2 in the SAME
            // lane and register, so the rotation is lane-local.  Arithmetic and rounding points are qkv_post_kernel's
            // (rope8: products and the difference / sum rounded separately, -ffp-contract=off): bit-identical outputs.
            const int head = ncol_w >> 7, half = (ncol_w >> 6) & 1;
            const int nh = p.qkv_nh, nkv = p.qkv_nkv;
            const bool is_q = head < nh, is_k = !is_q && head < nh + nkv;
            const bool rot = half == 0 && (is_q || is_k);
            const int kh = is_q ? head : (is_k ? head - nh : head - nh - nkv);
            bf16_t* dense = is_q ? p.qkv_q : (is_k ? p.qkv_k : p.qkv_v);
            bf16_t* cache = is_q ? nullptr : (is_k ? p.qkv_kc : p.qkv_vc);
            const int64_t ldd = (int64_t)(is_q ? nh : nkv) * 128;
            if (is_q && mcnt_c == C::BM) stored = STORES;  // (k and v: cache rows by slot)
            const bool col_ok = ncol_w < p.N;
            u32x2_t bias_p[4];  // four consecutive bias values per tile, packed (N is a whole number of 64-column blocks)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                bias_p[t] = (p.bias && col_ok) ? *reinterpret_cast<const u32x2_t*>(p.bias + ncol_w + 16 * t + 4 * g4) : u32x2_t{0u, 0u};
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt) {
                const int row = wm * (C::BM / 2) + 16 * mt + c;
                const bool row_ok = row < mcnt_c && col_ok;
                const int64_t m = m0_c + (row_ok ? row : 0);
                float o[4][4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    o[t][0] = rbf(acc[t][mt][0] + bflo(bias_p[t][0]));
                    o[t][1] = rbf(acc[t][mt][1] + bfhi(bias_p[t][0]));
                    o[t][2] = rbf(acc[t][mt][2] + bflo(bias_p[t][1]));
                    o[t][3] = rbf(acc[t][mt][3] + bfhi(bias_p[t][1]));
                }
                if (rot) {  // wave-uniform
                    const float* cs = p.qkv_cs + p.qkv_pos[m] * 64;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const f32x4_t cv = *reinterpret_cast<const f32x4_t*>(cs + 16 * t + 4 * g4);
                        const f32x4_t sv = *reinterpret_cast<const f32x4_t*>(cs + 32 + 16 * t + 4 * g4);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float x1 = o[t][r], x2 = o[t + 2][r];
                            o[t][r] = x1 * cv[r] - x2 * sv[r];
                            o[t + 2][r] = x2 * cv[r] + x1 * sv[r];
                        }
                    }
                }
                u32x2_t v[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = u32x2_t{pack2bf(o[t][0], o[t][1]), pack2bf(o[t][2], o[t][3])};
                int64_t slot = -1;
                if (cache != nullptr && p.qkv_slots != nullptr && row_ok) slot = p.qkv_slots[m];
                const bool to_cache = slot >= 0 && slot < p.qkv_nslots;
#pragma unroll
                for (int t = 0; t < 4; t += 2) {
                    const u32x2_t a = __builtin_amdgcn_permlane16_swap(v[t][0], v[t + 1][0], false, false);
                    const u32x2_t b = __builtin_amdgcn_permlane16_swap(v[t][1], v[t + 1][1], false, false);
                    const int cw = 64 * half + 16 * (t + (g4 & 1)) + 8 * (g4 >> 1);  // column inside the head
                    const u32x4_t o4 = u32x4_t{a[0], b[0], a[1], b[1]};
                    if (row_ok) {
                        if (dense != nullptr) *reinterpret_cast<u32x4_t*>(dense + m * ldd + kh * 128 + cw) = o4;
                        if (to_cache) *reinterpret_cast<u32x4_t*>(cache + (slot * nkv + kh) * 128 + cw) = o4;
                    }
                }
            }
        } else if constexpr (LATE_FILL) {
            // ---- fp8 x fp8 gate|up: the accumulator x weight-row scale x token scale is the bf16 GEMM's value up to the
            // fp8 roundings of its inputs; same rounding points behind it (mlp.py:49-53: bf16 gate_up, bf16 silu, bf16
            // product).  The product is then quantised for the down projection's fp8 operand in MX form, decided locally:
            // a wave's 32 act columns of a token ARE one 32-element block (ncol_w is a multiple of 32) — amax over the lane's 8
            // values and the 3 other lane rows of the token, E8M0 scale 2^(floor(log2 amax) - 8) (OCP MX: e4m3 emax = 8) or,
            // where that would push amax past 448, the next power of two (nothing saturates), e4m3 = RNE(v / scale).  act8 [R, I] bytes + one scale byte per (row, block) at
            // (block & 3) * 16 + (block >> 2) of the row's 64-byte record — the order the down kernel's lanes read it in.
            const float* ws = p.wscale + (int64_t)grp_c * p.wscale_gstride;
            float wsg[2][4], wsu[2][4];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n1 = min(ncol_w + 16 * t + 4 * g4 + r, p.N - 1);
                    wsg[t][r] = ws[n1];
                    wsu[t][r] = ws[p.N + n1];
                }
            unsigned char* y8 = reinterpret_cast<unsigned char*>(p.y);
            const bool col_ok = ncol_w < p.N;
            float xs_all[C::MT];   // token scales of the wave's 8 row blocks: all requested in front of the ring fill
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt) {
                const int row = wm * (C::BM / 2) + 16 * mt + c;
                const int64_t m = m0_c + ((row < mcnt_c && col_ok) ? row : 0);
                xs_all[mt] = p.xscale[p.src ? p.src[m] : m];
            }
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt) {
                const int row = wm * (C::BM / 2) + 16 * mt + c;
                const bool row_ok = row < mcnt_c && col_ok;
                const int64_t m = m0_c + (row_ok ? row : 0);
                const float xs = xs_all[mt];
                float v[2][4];
                float amax = 0.f;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float ga = acc[t][mt][r] * wsg[t][r] * xs, ua = acc[t + 2][mt][r] * wsu[t][r] * xs;
                        v[t][r] = rbf(rbf(glm_silu(rbf(ga))) * rbf(ua));
                        amax = fmaxf(amax, fabsf(v[t][r]));
                    }
                amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
                amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                const unsigned ab = __float_as_uint(amax);
                const int eb = (int)((ab >> 23) & 0xffu);   // biased exponent (0: zero or subnormal block)
                // 2^(floor(log2 amax) - 8) maps amax into [256, 512); above 448 = 1.75 x 2^8 it would saturate: one step up then
                const int sb = eb == 0 ? 127 : min(max(eb - 8 + ((ab & 0x7fffffu) > 0x600000u ? 1 : 0), 1), 253);
                const float inv = __uint_as_float((unsigned)(254 - sb) << 23);    // 2^(127 - sb), exact
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float q[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) q[r] = fminf(fmaxf(v[t][r] * inv, -448.0f), 448.0f);
                    int d = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
                    d = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], d, true);
                    const int n = ncol_w + 16 * t + 4 * g4;
                    if (row_ok && n < p.N) *reinterpret_cast<int*>(y8 + m * p.ldy + n) = d;
                }
                if (row_ok && g4 == 0) p.ybscale[m * 64 + wn * 16 + ntile_c] = (unsigned char)sb;
                if (mt == 0) start_next();
            }
        } else if constexpr (LEAN) {
            // Decisions (bias, scale, kind of column) once per wave and not per element, and stores through buffers of 16 of the tile's own rows and its columns: what lies
            // behind them is dropped by the bounds check, so every store is issued, with one offset for all of a tile's rows.  Between a tile's loops the matrix pipe
            // stands still: the instructions here are what counts.  15074 rows, us, with a test and a 64-bit address per element or row / this: 6144 x
            // 2048 with a bias 329 / 285, xIELU 314 / 298, 4096 x 2048 half of them gates 207 / 188, 8192 x 2048 of SiLU and gates 411 / 377, 10240 x
            // 2048 of three kinds 507 / 467, plain 6144 x 2048 283 / 281; down of 8 of 64 experts, 4096 x 1408, 1258 / 1238.
            constexpr unsigned BEYOND = 0x80000000u;
            constexpr unsigned es = F32 ? 4u : 2u;
            const unsigned pitch = (unsigned)p.ldy * es;   // (16 rows are below 2 GiB: launch_largem)
            const int64_t first = ((MODE == GEMM_SLICES ? (int64_t)grp_c * p.R : 0) + m0_c + wm * (C::BM / 2)) * p.ldy + ncol_w;
            char* ybase = F32 ? reinterpret_cast<char*>(p.yf + first) : reinterpret_cast<char*>(p.y + first);
            const int left = ncol_w < p.N ? mcnt_c - wm * (C::BM / 2) : 0;
            auto rows16 = [&](int mt) __attribute__((always_inline)) {
                const int rows = min(left - 16 * mt, 16);
                return __builtin_amdgcn_make_buffer_rsrc(ybase + (int64_t)mt * 16 * pitch, 0, rows > 0 ? (unsigned)(rows - 1) * pitch + (unsigned)(p.N - ncol_w) * es : 0u,
                                                         0x00020000);
            };
            const unsigned lrow = (unsigned)c * pitch;
            // Of short reductions (much output for its time) whole cache lines are written through the L2: what stays dirty there is written out when a tile of operands needs
            // the place and, 32 MiB of it, at the launch's end.  Kept dirty / through, us, in a step: 15074 x 4096 x 256 52.2 / 47.4, x 2048 x 2048 98.0 / 95.4,
            // x 6144 x 2048 (xIELU) 320 / 315, 11137 x 4096 x 2048 gated 279 / 274, and attention behind such a launch 582 / 570, 173 / 170.  Experts lose 2 to 3 %, rows that start inside
            // a line 12 % (15074 x 9232 x 2048 419 / 470).  By itself, times of kept dirty, up to a round of tiles: K of 256 to 1024 0.83 to 0.95 (3756 x 2048 x 512 13.4 / 11.4), of several
            // rounds 0.90 to 0.98, of 2048 0.98 to 1.0; rows of 16 KiB (8192 columns) 0.94 to 1.07, 1.00 in the mean (3756 x 8192 x 512 34.4 / 36.1; such a launch inside a step of width 4096,
            // 36 rows and four prompts of 930, 48 / 50, the step 4430 / 4460).  With weights that come from memory, as in a step, and more than some 40 G multiply-adds 1.00 to 1.08, but steps with
            // such launches written through take 0.990 to 0.997 of the time (Dafolorn, Napadra, Gulozen, Loselix 2k, prompts of 15074 rows).
            // Not the largest outputs, which no cache holds.  bf16 of 256 to 400 MiB 1.00 to 1.03 by themselves, but a step with six launches of 324 MiB (15074 x 11264 x 2048) 0.987 to 0.995; beyond
            // 1.02 to 1.3 (16198 x 18688 x 1536 707 / 782, 10212 x 31872 x 128 188 / 246), fp32 beyond 240 MiB 1.04 to 1.22 (13055 x 15872 x 384 248 / 303, 11943 x 23040 x 2048 929 / 1067).
            // The line: whole steps of 2048 columns gain 1 to 2.5 % by it on three cards of four, 0 to -1 % on the fourth, nearly all of it from K = 2048.  Beyond it K of 2560 and 3072 take 0.95 to
            // 1.0 of the time by themselves (4200 x 2048 x 3072 51.4 / 49.2, 15074 x 6144 x 3072 403 / 402), 4096 and 6144 0.97 to 1.02, but steps with those get nothing: eleven of 15 kinds 0.1 to
            // 0.7 % slower, one 1 % faster.
            const bool through = !GROUPED && K <= LM_THROUGH_K && p.R * p.ldy * (F32 ? 4 : 2) <= (F32 ? LM_THROUGH_F32 : LM_THROUGH_BF16) && ((pitch | (unsigned)(F32 ? (uintptr_t)p.yf : (uintptr_t)p.y)) & 127u) == 0;
            auto put = [&](const u32x4_t v, const __amdgpu_buffer_rsrc_t yrs, unsigned at) __attribute__((always_inline)) {
                if (through) __builtin_amdgcn_raw_buffer_store_b128(v, yrs, at, 0, LM_SC1);
                else __builtin_amdgcn_raw_buffer_store_b128(v, yrs, at, 0, 0);
            };
            // stores f of every element
            auto finish = [&](auto&& f) __attribute__((always_inline)) {
                if constexpr (F32) {   // four columns per store
#pragma unroll
                    for (int mt = 0; mt < C::MT; ++mt) {
                        const __amdgpu_buffer_rsrc_t yrs = rows16(mt);
#pragma unroll
                        for (int t = 0; t < NOUT; ++t) {
                            const int n = 16 * t + 4 * g4;
                            f32x4_t o;
#pragma unroll
                            for (int r = 0; r < 4; ++r) o[r] = f(t, mt, r);
                            put(__builtin_bit_cast(u32x4_t, o), yrs, ncol_w + n < p.N ? lrow + n * 4 : BEYOND);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    return;
                }
                // tiles (t, t+1): after the swaps lane row g4 holds 8 consecutive columns of tile t + (g4 & 1),
                // starting at column 8 * (g4 >> 1)
#pragma unroll
                for (int mt = 0; mt < C::MT; ++mt) {
                    const __amdgpu_buffer_rsrc_t yrs = rows16(mt);
#pragma unroll
                    for (int t = 0; t < NOUT; t += 2) {
                        const int n = 16 * (t + (g4 & 1)) + 8 * (g4 >> 1);
                        const u32x2_t a = __builtin_amdgcn_permlane16_swap(pack2bf(f(t, mt, 0), f(t, mt, 1)), pack2bf(f(t + 1, mt, 0), f(t + 1, mt, 1)), false, false);
                        const u32x2_t b = __builtin_amdgcn_permlane16_swap(pack2bf(f(t, mt, 2), f(t, mt, 3)), pack2bf(f(t + 1, mt, 2), f(t + 1, mt, 3)), false, false);
                        const u32x4_t o = {a[0], b[0], a[1], b[1]};
                        if constexpr (C::WIDE) {
                            if (16 * mt + c < left && ncol_w + n < p.N) *reinterpret_cast<u32x4_t*>(p.y + first + (16 * mt + c) * p.ldy + n) = o;
                        } else put(o, yrs, ncol_w + n < p.N ? lrow + n * 2 : BEYOND);
                    }
                    __builtin_amdgcn_sched_barrier(0);   // (the other rows' values would take registers that are not there)
                }
            };
            auto sum = [&](int t, int mt, int r) { return WSCALE ? acc[t][mt][r] * e_col[t][r] : acc[t][mt][r]; };
            if constexpr (gemm_paired(MODE)) {
                finish([&](int t, int mt, int r) {
                    const float g = sum(t, mt, r), u = sum(t + 2, mt, r);
                    return MODE == GEMM_GLU ? glm_glu_fast(p.act, g, u) : rbf(glm_silu(rbf(g))) * rbf(u);
                });
            } else if constexpr (MODE == GEMM_DOWN) {
                if (scaled) finish([&](int t, int mt, int r) { return rbf(sum(t, mt, r)) * e_row[mt]; });
                else finish(sum);
            } else {
                bool plain = !BIAS || p.bias == nullptr;
                if (plain) {
                    if constexpr (MODE == GEMM_COLS) {   // (a wave's 64 columns are of one kind nearly always)
                        const int n1 = ncol_w + 64, ca = (int)p.act.a, cb = (int)p.act.b;
                        const bool relu2 = p.act.kind == GLM_ACT_RELU2_GATE, silu = p.act.kind == GLM_ACT_SILU_GATE;
                        auto sigmoid = [&](float a) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * a)); };
                        if (relu2 && n1 <= ca && n1 <= cb) finish([&](int t, int mt, int r) { return fmaxf(acc[t][mt][r], 0.f) * fmaxf(acc[t][mt][r], 0.f); });
                        else if (relu2 ? ncol_w >= ca && n1 <= cb : !silu && n1 <= ca) finish(sum);
                        else if (ncol_w >= (relu2 ? cb : ca)) finish([&](int t, int mt, int r) { return sigmoid(acc[t][mt][r]); });
                        else if (silu && n1 <= ca) finish([&](int t, int mt, int r) { return acc[t][mt][r] * sigmoid(acc[t][mt][r]); });
                        else finish([&](int t, int mt, int r) { return glm_act_cols(p.act, acc[t][mt][r], ncol_w + 16 * t + 4 * g4 + r); });
                    } else {
                        with_kind([&](auto kind) __attribute__((always_inline)) { finish([&](int t, int mt, int r) { return act(acc[t][mt][r], t, r, kind); }); });
                    }
                } else if constexpr (BIAS) {
                    with_kind([&](auto kind) __attribute__((always_inline)) {
                        finish([&](int t, int mt, int r) { return act(acc[t][mt][r] + (r & 1 ? bfhi(e_bias[t][r >> 1]) : bflo(e_bias[t][r >> 1])), t, r, kind); });
                    });
                }
            }
            if constexpr (!C::WIDE) stored = STORES;
        } else {
        with_kind([&](auto kind) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < C::MT; ++mt) {
            const int row = wm * (C::BM / 2) + 16 * mt + c;
            const bool row_ok = row < mcnt_c;
            bf16_t* yrow = p.y + (int64_t)(m0_c + (row_ok ? row : 0)) * p.ldy;
            const float sc = (scaled && row_ok) ? bf2f(p.scale[m0_c + row]) : 1.0f;
#pragma unroll
            for (int t = 0; t < NOUT; ++t) {
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (gemm_paired(MODE)) {
                        float ga = acc[t][mt][r], ua = acc[t + 2][mt][r];
                        if constexpr (WSCALE) {  // weights expanded from fp8: per-row scale on the fp32 accumulators
                            const float* ws = p.wscale + (int64_t)grp_c * p.wscale_gstride;
                            const int n1 = min(ncol_w + 16 * t + 4 * g4 + r, p.N - 1);
                            ga *= ws[n1];
                            ua *= ws[p.N + n1];
                        }
                        o[r] = MODE == GEMM_GLU ? glm_glu_fast(p.act, ga, ua) : rbf(glm_silu(rbf(ga))) * rbf(ua);
                    } else {
                        float a = acc[t][mt][r];
                        if constexpr (WSCALE) a *= p.wscale[(int64_t)grp_c * p.wscale_gstride + min(ncol_w + 16 * t + 4 * g4 + r, p.N - 1)];
                        if (BIAS && p.bias) a += r & 1 ? bfhi(e_bias[t][r >> 1]) : bflo(e_bias[t][r >> 1]);
                        if (scaled) a = rbf(a) * sc;
                        o[r] = act(a, t, r, kind);
                    }
                }
                const int n = ncol_w + 16 * t + 4 * g4;
                if constexpr (F32) {  // fp32 rows: four columns per store
                    const int64_t slab = MODE == GEMM_SLICES ? (int64_t)grp_c * p.R : 0;
                    if (row_ok && n < p.N) *reinterpret_cast<f32x4_t*>(p.yf + (slab + m0_c + row) * p.ldy + n) = f32x4_t{o[0], o[1], o[2], o[3]};
                } else if (row_ok && n < p.N) *reinterpret_cast<u32x2_t*>(yrow + n) = u32x2_t{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
            }
        }
        });
        }
        pending_stores = stored;
        if (!more) break;
    }
}

// Tiles are equal and every CU takes its share of them, so what does not fill a round costs one: the tiles behind whole rounds, if they are half a round at
// most, are cut in two, half a tile for every CU, on the 128-row configuration and its ring (0.7 of a tile's time).  One kind of tile / this, us: 11137 rows of
// 2048 x 2048 (1.4 rounds) 83.7 / 74.9, of 3072 x 2048 (2.1) 129 / 117, of 6144 x 2048 (4.1) 220 / 209, gated 4096 x 2048 (5.5) 266 / 262, 15074 of 2304 x 2048 (2.1)
// 128 / 118, x 512 46.6 / 42.4, 4500 of 4096 x 4096 154 / 132; a forward pass of 9000 rows 5.07 / 4.84 ms, one of 15074 rows with few such launches the same.
template <int MODE, class C, bool LEAN, bool WSCALE>
__global__ __launch_bounds__(512) void gemm_largem_kernel(const GemmParams p, int n_tiles, int total_tiles, int LM_BAND, int tail) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int blocks = (int)((p.R + C::BM - 1) / C::BM);
    // Groups: the list has the row blocks that the groups have, counted here, and not the most that as many rows could make (the host knows no more): the positions
    // without a tile were all in the last XCD's share, so that the others took up to two rounds more.  List of the most / of what there is, us: gate|up, down of 64
    // experts, 6 of 1024 x 2048 at 2400 tokens 192 / 153, 117 / 96, at 6000 314 / 293, 188 / 176, at 15074 646 / 604, 404 / 377; 8 of 1408 x 4096 at 2400 600 /
    // 564, 341 / 318, at 4096 842 / 756, 489 / 438, at 15074 2387 / 2379, 1355 / 1328.  (Without halves behind whole rounds: 0 to 3 % slower.)
    // A list of the most that is one round stays: a workgroup has one position at most, and counting would put a trip to memory in front of it.
    if constexpr (MODE == GEMM_GATEUP || MODE == GEMM_DOWN) {
        if (p.offs != nullptr && total_tiles <= (int)gridDim.x) {
            blocks = 1 << 30;
        } else if (p.offs != nullptr) {
            blocks = lm_row_blocks(p.offs, p.G, C::BM, threadIdx.x & 63);
            total_tiles = blocks * n_tiles;
            const int wgs = gridDim.x, rest = total_tiles % wgs;
            tail = lm_cuts<MODE, C>() && p.K >= LM_CUT_K && total_tiles > wgs && 2 * rest <= wgs ? rest : 0;
            total_tiles -= tail;
        }
    }
    largem_tiles<MODE, C, LEAN, WSCALE, false>(p, smem, n_tiles, total_tiles, LM_BAND, blocks, 0);
    if constexpr (lm_cuts<MODE, C>()) {
        if (tail > 0) largem_tiles<MODE, LmCfgA, true, WSCALE, true>(p, smem, n_tiles, 2 * tail, LM_BAND, blocks, total_tiles);
    }
}

// option largem_variant: -1 by shape, LM_VAR_LEAN the same, any other number the plain form
constexpr int LM_VAR_LEAN = 86787;

template <int MODE, class C, bool LEAN>
int launch_largem_cfg(const GemmParams& p, hipStream_t st) {
    const int cols_per_wg = gemm_paired(MODE) ? 128 : LM_BN;
    const int n_tiles = (p.N + cols_per_wg - 1) / cols_per_wg;
    const int64_t combos = p.offs ? (p.R / C::BM + p.G) : (p.R + C::BM - 1) / C::BM * (MODE == GEMM_SLICES ? p.G : 1);
    // (a band higher than the rows' blocks would be mostly positions without a tile: 74 tiles of one block took two passes of 256
    // workgroups)
    const int LM_BAND = p.offs ? LM_BAND_ROWS : (int)(combos < LM_BAND_ROWS ? combos : (int64_t)LM_BAND_ROWS);
    const bool dense = p.offs == nullptr && MODE != GEMM_SLICES;
    int64_t total = (combos + LM_BAND - 1) / LM_BAND * LM_BAND * n_tiles;
    if (total <= 0) return GLM_OK;
    GLM_CHECK_ARG(total < (1ll << 30) && n_tiles < (1 << 22), GLM_ERR_UNSUPPORTED, "gemm_largem: grid too large");
    // the per-row scale of fp8-expanded weights is its own instantiation: as a run-time test it sat inside the epilogue's
    // element loop (a branch per accumulator register)
    // (dense projections have no weight scales)
    constexpr bool SCALES = MODE == GEMM_GATEUP || MODE == GEMM_DOWN;
    auto kern = (C::W8 || C::A8 || (SCALES && p.wscale)) ? gemm_largem_kernel<MODE, C, LEAN, SCALES || C::W8 || C::A8>
                                                         : gemm_largem_kernel<MODE, C, LEAN, !(C::W8 || C::A8) ? false : true>;
    constexpr int LDS_BYTES = C::LDS + ((C::A8 && MODE == GEMM_DOWN) ? 16 * 1024 : 0);
    GLM_SET_MAX_LDS(kern, LDS_BYTES, "gemm_largem");
    // one workgroup per CU (the ring takes most of the LDS), a multiple of 8 so that every XCD gets the same count
    static int n_cu = 0;
    if (n_cu == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
            glm_set_error("gemm_largem: hipGetDeviceProperties failed");
            return GLM_ERR_LAUNCH;
        }
        n_cu = prop.multiProcessorCount;
    }
    int64_t nwg = (n_cu / 8) * 8;
    if (nwg < 8) nwg = 8;
    const int64_t need = (total + 7) / 8 * 8;
    if (nwg > need) nwg = need;
    int64_t tail = 0;
    if (lm_cuts<MODE, C>() && dense && combos * n_tiles > nwg && p.K >= LM_CUT_K) {
        tail = combos * n_tiles % nwg;
        if (2 * tail > nwg) tail = 0;
        if (tail > 0) total = combos * n_tiles - tail;
    }
    // Positions without a tile keep every XCD's share of the list at whole bands (4 row blocks by 8 column tiles at a time, one copy in its L2), so they stay
    // where leaving them out saves no round.  With / without them inside a forward pass of 15074 rows, us: 2048 x 2048 (1.8 rounds of tiles, 2 of positions)
    // 95.4 / 100, fp32 logits 184 / 194; where they are a round, 15074 of 14336 x 4096 (12.9 and 13.1): a pass of such layers 31.2 / 30.9 ms.
    if (dense && tail == 0 && (combos * n_tiles + nwg - 1) / nwg < (total + nwg - 1) / nwg) total = combos * n_tiles;
    hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(512), LDS_BYTES, st, p, n_tiles, (int)total, LM_BAND, (int)tail);
    GLM_CHECK_LAUNCH("gemm_largem");
    return GLM_OK;
}

// option largem_cfg (GLM_LARGEM_CFG=A|B at start-up) overrides the tile configuration (A/B measurements)
int cfg_choice() { return glm_option(GLM_OPT_LARGEM_CFG); }

template <int MODE>
int launch_largem(const GemmParams& p, hipStream_t st) {
    // 256-row blocks pay off once a group fills most of one; smaller groups keep the 128-row tile
    const int ch = cfg_choice();
    const int64_t avg_rows = (p.R_hint > 0 ? p.R_hint : p.R) / (p.G > 0 && MODE != GEMM_SLICES ? p.G : 1);
    // ... and a projection onto <= 128 columns (the router logits at prefill: N = E = 64) is one column tile however the rows
    // are cut, so its parallelism is its row-block count: 128-row blocks (75.8 -> 55.1 us at T = 16384)
    // ... and so is every single projection whose 128-row tiles are at most one round of the chip (the tiles themselves: launch_largem_cfg leaves out
    // positions without one where they would be a second round): a K step costs two thirds.  256-row / 128-row tiles, us: 14336 x 4096 at 400 rows 86 /
    // 59, 4096 x 12288 at 1200 234 / 153, 6144 x 2048 at 1100 (216 tiles, 288 positions) 43.3 / 32.8, 12288 x 4096 at 600 74.4 / 65.1, 10240 x 4096 at 700
    // 75.2 / 61.0, 3072 x 2048 at 2600 41.0 / 32.6; beyond a round 6144 x 2048 at 1281 43.7 / 53.0, 9728 x 2048 at 800 48 / 60.  (What is a round of 128 x
    // 128 tiles does not come here, gemm_midm.hip.)
    const bool one_round = p.offs == nullptr && MODE != GEMM_SLICES && p.wscale == nullptr && !p.w_fp8 &&
                           (p.R + 127) / 128 * ((p.N + (gemm_paired(MODE) ? 127 : 255)) / (gemm_paired(MODE) ? 128 : 256)) <= 256;
    const bool use_b = ch == 2 || (ch == 0 && avg_rows >= 192 && !one_round && !(lm_single<MODE>() && p.offs == nullptr && p.N <= 128));
    // the lean form addresses x, the group's weights and a tile's rows of y through 32-bit buffer offsets and has no K tail path
    const int var = glm_option(GLM_OPT_LARGEM_VARIANT);
    const int64_t wrows = gemm_paired(MODE) ? 2 * (int64_t)p.N : (int64_t)p.N;
    const bool lean_ok = p.K % 64 == 0 && p.R * p.ldx * 2 < (1ll << 31) && wrows * p.ldw * 2 < (1ll << 31) &&
                         p.N % 8 == 0 && p.ldy % 8 == 0 && glm_aligned16(p.y);
    const bool wide = p.ldy >= LM_WIDE;
    if (p.w_fp8) {
        // fp8 weight operand: the lean form only;
        // what they do not cover (a K tail, offsets past 2^31) goes back to the caller, which expands the stack instead
        if (!lean_ok || (wide && MODE != GEMM_DOWN) || p.wscale == nullptr || p.ldw % 16 != 0 || p.w_gstride % 16 != 0) {
            glm_set_error("gemm_largem(fp8 weights): shape not covered (K=%d N=%d ldw=%ld)", p.K, p.N, (long)p.ldw);
            return GLM_ERR_UNSUPPORTED;
        }
        if constexpr (MODE != GEMM_GATEUP && MODE != GEMM_DOWN) {
            glm_set_error("gemm_largem(fp8 weights): only the grouped expert projections are quantised");
            return GLM_ERR_UNSUPPORTED;
        } else {
            if (wide) {
                if constexpr (MODE == GEMM_DOWN) return launch_largem_cfg<MODE, LmCfgA8Wide, true>(p, st);
            }
            if (use_b) return launch_largem_cfg<MODE, LmCfgR8, true>(p, st);
            return launch_largem_cfg<MODE, LmCfgA8, true>(p, st);
        }
    }
    const bool lean = lean_ok && !wide && (var < 0 || var == LM_VAR_LEAN);
    // One round of 192-row tiles where 256-row ones would leave CUs without work and 128-row ones would be two rounds.  256 / 192, us: 4200 rows of 2048 x 2048 38.4 /
    // 34.0, x 8192 134 / 120, 4780 38.6 / 36.5, 141 / 132, 6100 42.0 / 39.5, 153 / 145, 3000 of 3072 x 2048 39.1 / 34.6, of 4096 x 4096 81.8 / 76.6, 1300 of 6144 x 2048
    // 42.3 / 36.0, gated 4096 x 2048 50.4 / 40.7.  Where they are two rounds for one or two with a cut tail, a tile's K step costing seven eighths, 0.95 to 1.1 of the time.
    if constexpr (lm_single<MODE>() || MODE == GEMM_GLU) {
        const int64_t cols = (p.N + (gemm_paired(MODE) ? 127 : 255)) / (gemm_paired(MODE) ? 128 : 256);
        if (lean && use_b && ch == 0 && p.offs == nullptr && (p.R + 191) / 192 * cols <= 256) return launch_largem_cfg<MODE, LmCfgR192, true>(p, st);
    }
    if (lean) return use_b ? launch_largem_cfg<MODE, LmCfgR, true>(p, st) : launch_largem_cfg<MODE, LmCfgA, true>(p, st);
    if constexpr (MODE == GEMM_QKV) {  // 16-byte-store form only
        glm_set_error("gemm_largem(qkv epilogue): the plain form has no such epilogue");
        return GLM_ERR_UNSUPPORTED;
    } else return use_b ? launch_largem_cfg<MODE, LmCfgB, false>(p, st) : launch_largem_cfg<MODE, LmCfgA, false>(p, st);
}

}  // namespace

#if !GLM_DENSE_ONLY
// fp8 x fp8 grouped expert projections on the block-scaled MFMA, on
// 256-row blocks.  Strides of x / w in BYTES.
int glm_launch_gemm_largem_a8(int mode, const GemmParams& p, hipStream_t st) {
    const int64_t avg_rows = (p.R_hint > 0 ? p.R_hint : p.R) / (p.G > 0 ? p.G : 1);
    const int64_t wrows = mode == GEMM_GATEUP ? 2 * (int64_t)p.N : (int64_t)p.N;
    const bool ok = (mode == GEMM_GATEUP || mode == GEMM_DOWN) && p.a8 && p.wscale != nullptr && p.offs != nullptr && avg_rows >= 192 &&
                    p.K % 128 == 0 && p.N % 8 == 0 && p.ldx % 16 == 0 && p.ldw % 16 == 0 && p.w_gstride % 16 == 0 &&
                    p.R * p.ldx < (1ll << 31) && wrows * p.ldw < (1ll << 31) && glm_aligned16(p.x) && glm_aligned16(p.w) &&
                    (mode == GEMM_GATEUP ? (p.xscale != nullptr && p.ybscale != nullptr && p.ldy % 4 == 0 && (((uintptr_t)p.y) & 3) == 0 &&
                                            p.N % 32 == 0 && p.N <= 2048)
                                         : (p.xbscale != nullptr && glm_aligned16(p.xbscale) && p.K <= 2048 && p.ldy % 8 == 0 && glm_aligned16(p.y)));
    if (!ok) {
        glm_set_error("gemm_largem(fp8 x fp8): shape not covered (mode %d R=%ld G=%d N=%d K=%d)", mode, (long)p.R, p.G, p.N, p.K);
        return GLM_ERR_UNSUPPORTED;
    }
    if (mode == GEMM_GATEUP) return launch_largem_cfg<GEMM_GATEUP, LmCfgC88, true>(p, st);
    if (p.ldy >= LM_WIDE) return launch_largem_cfg<GEMM_DOWN, LmCfgC88Wide, true>(p, st);
    return launch_largem_cfg<GEMM_DOWN, LmCfgC88, true>(p, st);
}

// QKV projection with the split / rotary / cache-store epilogue: the product loop on the tiled configurations only
int glm_launch_gemm_largem_qkv(const GemmParams& p, hipStream_t st) {
    const int Nexp = (p.qkv_nh + 2 * p.qkv_nkv) * 128;
    if (p.qkv_q == nullptr || p.N != Nexp || p.offs != nullptr || p.K % 64 != 0 || p.R < 1 || p.ldx % 8 != 0 || p.ldw % 8 != 0 ||
        !glm_aligned16(p.x) || !glm_aligned16(p.w) || !glm_aligned16(p.qkv_q) || !glm_aligned16(p.qkv_cs) ||
        (p.qkv_k && !glm_aligned16(p.qkv_k)) || (p.qkv_v && !glm_aligned16(p.qkv_v)) || (p.qkv_kc && !glm_aligned16(p.qkv_kc)) ||
        (p.qkv_vc && !glm_aligned16(p.qkv_vc)) || (p.bias && (((uintptr_t)p.bias) & 7) != 0) || p.R * p.ldx * 2 >= (1ll << 31) || (int64_t)p.N * p.ldw * 2 >= (1ll << 31)) {
        glm_set_error("gemm_largem(qkv epilogue): shape not covered (R=%ld N=%d K=%d)", (long)p.R, p.N, p.K);
        return GLM_ERR_UNSUPPORTED;
    }
    GemmParams q = p;
    q.y = p.qkv_q;  // never stored through; keeps the generic alignment checks meaningful
    q.ldy = p.N;
    if (glm_midm_takes(GEMM_PLAIN, q)) return glm_launch_gemm_midm(GEMM_PLAIN, q, st);  // where glm_gemm_bf16 goes there, bit-identical to it
    return launch_largem<GEMM_QKV>(q, st);
}
#endif  // !GLM_DENSE_ONLY

int glm_launch_gemm_largem(int mode, const GemmParams& p, hipStream_t st) {
    GLM_CHECK_ARG(p.K % 8 == 0 && p.N % 4 == 0 && p.ldx % 8 == 0 && p.ldy % 4 == 0 && p.ldw % 8 == 0 &&
                      glm_aligned16(p.x) && glm_aligned16(p.w) && (((uintptr_t)p.y) & 7) == 0,
                  GLM_ERR_UNSUPPORTED,
                  "gemm_largem: needs K%%8==0, N%%4==0, ldx%%8==0, ldy%%4==0, 16B-aligned x/W (K=%d N=%d)",
                  p.K, p.N);
#if GLM_EXPERTS
    if (mode == GEMM_GATEUP) return launch_largem<GEMM_GATEUP>(p, st);
    if (mode == GEMM_DOWN) return launch_largem<GEMM_DOWN>(p, st);
#endif  // GLM_EXPERTS
    if (mode == GEMM_ACT && p.yf != nullptr) switch (p.act.kind) {
        case GLM_ACT_NONE: return launch_largem<GEMM_F32>(p, st);
        case GLM_ACT_SOFTCAP: return launch_largem<GEMM_CAP>(p, st);
        case GLM_ACT_XIELU: return launch_largem<GEMM_XIELU32>(p, st);
        default: return launch_largem<GEMM_COLS32>(p, st);
    }
    if (mode == GEMM_ACT) switch (p.act.kind) {
        case GLM_ACT_NONE: return launch_largem<GEMM_PLAIN>(p, st);
        case GLM_ACT_SOFTCAP: return launch_largem<GEMM_CAP16>(p, st);
        case GLM_ACT_XIELU: return launch_largem<GEMM_XIELU>(p, st);
        default: return launch_largem<GEMM_COLS>(p, st);
    }
    if (mode == GEMM_SLICES) return launch_largem<GEMM_SLICES>(p, st);
    if (mode == GEMM_GLU) return launch_largem<GEMM_GLU>(p, st);
    return launch_largem<GEMM_PLAIN>(p, st);
}
