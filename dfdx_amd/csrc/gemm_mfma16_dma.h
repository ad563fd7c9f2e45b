// The LDS-DMA kernel of gemm_mfma16_dma.hip (its description is there) and the macro that launches an instance of it; the
// instances are compiled in two files: the plain ones beside the planner, the EXTRA ones in gemm_mfma16_dma_extra.hip.
#pragma once
#include "gemm_internal.h"
#include <algorithm>
#include <type_traits>

namespace dfdx_rocm {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#define DFDX_LDS __attribute__((address_space(3)))
#define DFDX_GLB __attribute__((address_space(1)))

constexpr int BK = 64;
constexpr int STAGES = 2;

}  // namespace

struct DmaParams {
    const uint16_t *a;
    const uint16_t *b;
    uint16_t *c;
    const uint16_t *bias;
    int m, n, k;
    int lda, ldb;
    int64_t ldc;
    int64_t a_b1, a_b2, b_b1, b_b2, c_b1, c_b2, bias_b1, bias_b2;
    int nb2, kbatches;
    int tiles_m, tiles_n, tiles_per_batch, total_blocks;
    int accumulate, bias_mode;
    int group_m;
    // split-k: `splits` workgroups per C tile, each covering `chunk` k-loop steps, f32 partials in `ws`
    int splits, chunk;
    int grid;  // workgroups launched (<= total_blocks: each walks blockIdx.x, blockIdx.x + grid, ...)
    float *ws;
    int64_t ws_ld, ws_split_stride;
    // sums of A's rows over the contraction as a second result (KSUM instances, split-k only): f32 partial sums in
    // ws_ksum[(split * (BM / 64) + tile column) * 8 + wave][tiles_m * BM], combined by the reduce kernel
    float *ws_ksum;
    int ws_ksum_stride;
    const uint16_t *with;  // second operand of the EXTRA instances, laid out like c
    int steps;  // (batch of the contraction, k tile) pairs: the last batch may end early
};

namespace {
typedef DmaParams Params;

// A 16-byte store of C in the non-temporal form (`global_store_dwordx4 ... nt`): the lines are not kept in the caches on
// their way to memory.  For C of whole lines that is written once and not read back by this launch.  Measured on MI355X against the
// cached form, over buffer sets that defeat the 256 MB last-level cache: 128 x (1024 x 64 x 1024), 268 MB of C, 71 -> 57 us
// (the output stops evicting the operand tiles); 8192 x 1024 x 1024 24.7 -> 18.8 us; 4096^3 109 -> 105 us; one encoder
// block, forward + backward, 1288 -> 1268 us.  Launch after launch on ONE buffer set whose output fits that cache the
// cached form is up to 6 % faster (256 x (512 x 64 x 512): 29.1 vs 30.9 us) -- a state no training step is in.
__device__ __forceinline__ void stream16(void *p, u32x4 v) { __builtin_nontemporal_store(v, (u32x4 *)p); }

// 16 bytes of C at any element (ANY) or on the 16-byte grid.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef u32x2 u32x2_any __attribute__((aligned(2)));
template <bool ANY> __device__ __forceinline__ u32x4 load16(const void *p) {
    if constexpr (ANY) return *(const u32x4_any *)p;
    else return *(const u32x4 *)p;
}
// Eight columns of a row of C that starts anywhere.  Stores that lie on words run at nearly the rate of aligned ones, those that lie on the
// upper half of a word at a third of it (4096 x 1024 x 4096 f16 33.5 us, 4094 columns 35.5, 4095 45.4): where the row starts on such a
// half (`odd`) the lane gives its first column away and stores the seven behind it and the first of its right neighbour, `next`; the ends of a
// run of neighbours, `first` and `last`, store what is left of them in smaller pieces.  4096 x 1024 x 4095 so: 38.1 us, 4096 x 256 x 4095 26.5 ->
// 20.0, 2048 x 1024 x 50257 231 -> 212.
typedef u32x4 u32x4_word __attribute__((aligned(4)));
typedef u32x2 u32x2_word __attribute__((aligned(4)));
__device__ __forceinline__ void store_words(void *p, u32x4 v) { *(u32x4_word *)p = v; }
__device__ __forceinline__ void store_columns(uint16_t *p, bool odd, u32x4 v, uint32_t next, bool first, bool last) {
    const uint32_t by = odd ? 16u : 0u;
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = __builtin_amdgcn_alignbit(e < 3 ? v[e < 3 ? e + 1 : 3] : next, v[e], by);
    uint16_t *const at = p + (odd ? 1 : 0);
    if (!(odd && last)) {
        store_words(at, w);
    } else {
        *(u32x2_word *)at = u32x2{w[0], w[1]};
        *(uint32_t *)(at + 4) = w[2];
        at[6] = (uint16_t)w[3];
    }
    if (odd && first) p[0] = (uint16_t)v[0];
}

template <typename T> struct Mma;
template <> struct Mma<_Float16> {
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint16_t v) { return (float)__builtin_bit_cast(_Float16, v); }
    static __device__ __forceinline__ uint16_t from_f32(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {  // v_cvt_pk_f16_f32: RNE, lo in bits 15:0
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, h2));
    }
};
template <> struct Mma<__bf16> {
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
    static __device__ __forceinline__ uint16_t from_f32(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }  // RNE, quiet NaNs
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {  // v_cvt_pk_bf16_f32: RNE, quiet NaNs
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, b2));
    }
};

// DPP row rotation by 8 lanes: the lanes of the 4-lane banks selected by BANK_MASK (bit b = lanes 4b..4b+3 of every
// 16-lane row) receive `src` of the lane 8 places away in their row, the other lanes keep `keep`.
template <int BANK_MASK> __device__ __forceinline__ uint32_t lane8_trade(uint32_t keep, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)keep, (int)src, 0x128 /* row_ror:8 */, 0xF, BANK_MASK, false);
}

// Swizzle of an m/n-contiguous tile ([k][ROWS] in LDS, ROWS*2 bytes per k-row): XOR applied to the 16 B
// chunk index of k-row k.  A 16-lane group of a transposing read touches 4 consecutive k-rows x 2 chunks,
// a second group the same chunks 8 k-rows further: the XOR spreads those over distinct banks.
template <int ROWS> __device__ __forceinline__ int mc_swizzle(int k) {
    if constexpr (ROWS % 128 == 0) return (4 * (k & 3)) ^ (2 * ((k >> 3) & 1));
    else return (4 * ((k >> 1) & 1)) ^ (2 * ((k >> 3) & 1));  // ROWS == 64, 192: bit 3 of the bank slot comes from k & 1
}

// One operand tile in LDS, filled by LDS-DMA loads (16 B per lane, 1 KB contiguous per wave instruction).
// PERM (k-contiguous B tiles of wave tiles that are at least 32 columns wide): the fragments of such a tile do not take
// 16 consecutive rows but the rows 8q + 4 * (fragment parity) + 0..3, q = 0..3, of a 32-row group (see the epilogue: a
// lane then owns 8 consecutive columns of C without any exchange between lanes).  The swizzle follows the lane that
// reads the row, (2 * (r / 8 % 4) + r % 4 / 2), so that the banks a fragment read touches are those of the plain order.
template <int ROWS, int NWAVES, bool KC, bool PERM = false> struct DmaTile {
    static constexpr int BYTES = ROWS * BK * 2;
    static constexpr int INSTRS = BYTES / 1024;
    static constexpr int IPW = INSTRS / NWAVES;
    static_assert(INSTRS % NWAVES == 0 && IPW >= 1, "tile does not divide over the waves");
    static constexpr int CPR = KC ? BK / 8 : ROWS / 8;  // 16 B chunks per LDS row
    // Byte offset from the tile origin in global memory, plus 1024 * (IPW - 1 - i): the wave's IPW instructions share
    // ONE LDS base, that of the last 1 KB piece (one M0 write instead of IPW), and reach their own piece through the
    // instruction offset -1024 * (IPW - 1 - i), which the hardware adds to the global address as well.
    static_assert((IPW - 1) * 1024 <= 4096, "instruction offsets are 13-bit signed");
    uint32_t goff[IPW];

    __device__ __forceinline__ void init(int ld, int rows_left, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < IPW; i++) {
            const int slot = (wave * IPW + i) * 64 + lane;  // 16 B slot index inside the tile
            const int r = slot / CPR, cp = slot % CPR;
            if constexpr (KC) {
                const int c = PERM ? cp ^ ((((r >> 3) & 3) << 1) | ((r >> 1) & 1)) : cp ^ ((r >> 1) & 7);
                goff[i] = (uint32_t)(min(r, rows_left - 1) * ld + c * 8) * 2u + (uint32_t)(1024 * (IPW - 1 - i));
            } else {
                const int c = cp ^ mc_swizzle<ROWS>(r);
                goff[i] = (uint32_t)(r * ld + min(c * 8, rows_left - 8)) * 2u + (uint32_t)(1024 * (IPW - 1 - i));
            }
        }
    }
    template <int I> __device__ __forceinline__ void issue_one(const char *origin, DFDX_LDS void *lds) const {
        if constexpr (I < IPW) {
            __builtin_amdgcn_global_load_lds((const DFDX_GLB void *)(origin + goff[I]), lds, 16, -1024 * (IPW - 1 - I), 0);
            issue_one<I + 1>(origin, lds);
        }
    }
    // LDS byte address of the wave's last 1 KB piece inside a tile that starts at byte `tile` of the LDS allocation
    static __device__ __forceinline__ uint32_t wave_base(uint32_t tile, int wave) { return tile + (uint32_t)(wave * IPW + IPW - 1) * 1024u; }
    // `lds_last`: wave_base of the destination tile, wave-uniform (a scalar register: it goes to M0 as it is)
    __device__ __forceinline__ void issue(const uint16_t *g, uint32_t lds_last) const {
        issue_one<0>((const char *)g, (DFDX_LDS void *)(uintptr_t)lds_last);
    }
};

// Waves per SIMD that the two LDS stages of a BM x BN x 64 tile let a CU hold (160 KB of LDS, 8-wave workgroups on 4
// SIMDs): the register budget the kernel is compiled for, so that a scalar-register spill into vector lanes cannot
// push the 128 x 128 tile past 128 VGPRs and halve its occupancy.
constexpr int dma_waves_per_simd(int bm, int bn, int waves) {
    const int wgs = 163840 / (2 * (bm + bn) * 64 * 2);
    const int w = (wgs < 1 ? 1 : wgs) * waves / 4;
    return w < 2 ? 2 : (w > 6 ? 6 : w);
}

// EDGE = false is the instance for problems made of whole tiles (no per-row bias, no bias together with beta = 1): its
// epilogue has only the two interior forms.  With the general form compiled in as well, the compiler guards the
// fragment registers against a load of that form it cannot prove complete, with a wait for ALL memory traffic in the
// middle of the k loop -- where every wave then stalls on the tile prefetched for the step after.
//
// EDGE = 2 is the edge form for a C off the 16-byte grid (odd extents or leading dimensions, any address): the same pieces of
// eight columns as element-aligned accesses, which global memory allows at the cost of the lines they straddle, and the
// last columns of a row one by one.  These stores take the cached form, so that the two writers of a straddled line meet in L2.
//
// EXTRA: what is done with a finished value besides bias and beta (EXTRA_* in gemm_internal.h): what the op behind a Linear layer, or in front of its backward, would otherwise read and write C once more for.
//
// KSUM = true (A stored [k][m] only, split-k only) adds a second result: the sums of A's rows over the contraction --
// the bias gradient of a Linear layer when A is grad_out^T and the product is the weight gradient.  The A tile sits in
// LDS as 64 k-rows of BM values; its column sums need no MFMA and no fragment: every thread reads ONE 16-byte piece
// (8 values of one k-row) per k tile and adds it to 8 f32 sums of its own.  The 512 threads cover 512 of the tile's
// 64 * BM / 8 pieces; the workgroups of a tile row all hold the same A tiles, so tile column q < BM / 64 takes the q-th
// 512 pieces and the others none.  At the end of a work item lanes that hold the same 8 columns are added up and each
// wave leaves its sums in a workspace slot of its own; the split-k reduce kernel adds the slots.
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, bool A_KC, bool B_KC, int EDGE, bool KSUM = false, int EXTRA = EXTRA_NONE>
__global__ __launch_bounds__(WAVES_M *WAVES_N * 64, dma_waves_per_simd(BM, BN, WAVES_M *WAVES_N)) void gemm_mfma16_dma_kernel(const Params p) {
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
    constexpr int TM = WTM / 16, TN = WTN / 16;
    static_assert(WTM % 64 == 0 && WTN % 16 == 0, "wave tile must be a multiple of 64 x 16");
    constexpr int Q = TM / 4;  // tile rows per quarter of a k step
    // B stored along k and a wave tile of whole fragment pairs: the rows (n) of B are dealt to the fragments so that the
    // two accumulators acc[i][2jp], acc[i][2jp + 1] of a lane hold 8 CONSECUTIVE columns of C, n = 32 jp + 8 lq + 0..7
    // (fragment 2jp + par, MFMA row 4 lq + v  <->  n = 32 jp + 8 lq + 4 par + v), instead of two runs of 4 that the lane
    // rows would have to trade.  Same products, same k order, same bits; the epilogue loses its cross-lane exchange.
    constexpr bool PERM = B_KC && TN % 2 == 0;
    using TA = DmaTile<BM, NW, A_KC>;
    using TB = DmaTile<BN, NW, B_KC, PERM>;
    constexpr int STAGE_BYTES = TA::BYTES + TB::BYTES;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid % 64, wave = tid / 64;
    const int wm0 = (wave / WAVES_N) * WTM, wn0 = (wave % WAVES_N) * WTN;
    const int l16 = lane % 16, lq = lane / 16;

    // ---- work items ---------------------------------------------------------
    // A work item is one C tile (of one batch, or of one k split).  The workgroup is persistent: it walks the
    // work items blockIdx.x, blockIdx.x + gridDim.x, ... and keeps ONE load pipeline running across them, so
    // the stores of a finished tile overlap with the loads (already in flight) and MFMAs of the next one.
    // The arguments that only a work item's start and end need are read from memory there, not held in scalar registers
    // through the k loop (4096^3 f16, registers spilled to vector lanes: 17 - 32 with all arguments held, none now).  Small tiles gain:
    // 1024^3 f16 12.2 -> 11.6 us, 8192 x 1024 x 64 12.4 -> 11.9; with the plain instances holding them 12.0 and 12.3, and the large
    // products, which lost 0.5 - 1.7 % when batches that lie anywhere came in, level (4096^3 103.2 and 103.2, the 256-row ones 0.5 % slower).
    typedef const __attribute__((address_space(4))) Params ArgParams;
    auto late_args = [&]() -> ArgParams * {
        ArgParams *args = (ArgParams *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(args));
        return args;
    };
    struct Work {
        int batch, split, bm0, bn0, it0, iters;
    };
    const int ktiles = p.k / BK;
    auto decode = [&](auto &p, int index) -> Work {
        Work w;
        const int work = xcd_remap(index, p.total_blocks);
        const int bidx = work / p.tiles_per_batch;  // k pieces of a batch, batch after batch
        const int tile = work % p.tiles_per_batch;
        const int gsize = p.group_m * p.tiles_n;
        const int group = tile / gsize;
        const int first_m = group * p.group_m;
        const int gm = min(p.tiles_m - first_m, p.group_m);
        w.bm0 = (first_m + (tile % gsize) % gm) * BM;
        w.bn0 = ((tile % gsize) / gm) * BN;
        w.batch = p.splits > 1 ? bidx / p.splits : bidx;
        w.split = p.splits > 1 ? bidx - w.batch * p.splits : 0;
        // k-loop steps run over (batch, k-tile) pairs; with split-k this item owns steps [it0, it0 + iters)
        w.it0 = w.split * p.chunk;
        w.iters = min(p.steps - w.it0, p.chunk);
        return w;
    };

    // ---- global side: the load pipeline ("fetch" state runs ahead of the compute state) ------------------
    const int64_t a_step = A_KC ? BK : (int64_t)BK * p.lda;
    const int64_t b_step = B_KC ? BK : (int64_t)BK * p.ldb;
    int f_index = blockIdx.x;   // work item whose tiles are being requested
    Work fw = decode(p, f_index);
    int f_left = 0, f_kb = 0, f_kt = 0, f_stage = 0;
    const uint16_t *a_next = nullptr, *b_next = nullptr;
    TA ta;
    TB tb;
    auto a_origin = [&](const Work &w, int kb) -> const uint16_t * {
        const uint16_t *base = p.a + (int64_t)(kb / p.nb2) * p.a_b1 + (int64_t)(kb % p.nb2) * p.a_b2;
        return A_KC ? base + (int64_t)w.bm0 * p.lda : base + w.bm0;
    };
    auto b_origin = [&](const Work &w, int kb) -> const uint16_t * {
        const uint16_t *base = p.b + (int64_t)(kb / p.nb2) * p.b_b1 + (int64_t)(kb % p.nb2) * p.b_b2;
        return B_KC ? base + (int64_t)w.bn0 * p.ldb : base + w.bn0;
    };
    auto begin_fetch = [&]() {  // position the pipeline on the first tile of work item fw
        f_left = fw.iters;
        f_kb = p.kbatches > 1 ? fw.it0 / ktiles : fw.batch;
        f_kt = p.kbatches > 1 ? fw.it0 % ktiles : fw.it0;
        a_next = a_origin(fw, f_kb) + f_kt * a_step;
        b_next = b_origin(fw, f_kb) + f_kt * b_step;
        // wave and lane as new values: the tile coordinates derived from them are needed once per work item only and
        // are recomputed here instead of being carried through the k loop
        int f_wave = wave, f_lane = lane;
        asm volatile("" : "+v"(f_wave), "+v"(f_lane));
        // (rows that lie along memory are read in whole pieces: the stored rows go on to the next multiple of eight)
        ta.init(p.lda, (A_KC ? p.m : (p.m + 7) & ~7) - fw.bm0, f_wave, f_lane);
        tb.init(p.ldb, (B_KC ? p.n : (p.n + 7) & ~7) - fw.bn0, f_wave, f_lane);
    };
    begin_fetch();
    bool fetching = true;
    const uint32_t smem_addr = (uint32_t)(uintptr_t)(DFDX_LDS const uint8_t *)smem;
    const uint32_t lds_last_a = __builtin_amdgcn_readfirstlane(TA::wave_base(smem_addr, wave));
    const uint32_t lds_last_b = __builtin_amdgcn_readfirstlane(TB::wave_base(smem_addr + TA::BYTES, wave));
    auto issue = [&]() {
        const uint32_t st = (uint32_t)f_stage * STAGE_BYTES;
        f_stage ^= 1;
        ta.issue(a_next, lds_last_a + st);
        tb.issue(b_next, lds_last_b + st);
        if (--f_left == 0) {  // next request belongs to the next work item (if any)
            f_index += gridDim.x;
            fetching = f_index < p.total_blocks;
            if (fetching) {
                fw = decode(*late_args(), f_index);
                begin_fetch();
            }
            return;
        }
        a_next += a_step;
        b_next += b_step;
        if (++f_kt == ktiles) {
            f_kt = 0;
            ++f_kb;
            a_next = a_origin(fw, f_kb);
            b_next = b_origin(fw, f_kb);
        }
    };

    // ---- LDS side: per-lane fragment addresses ------------------------------
    // k-contiguous: lane reads row w0 + 16*t + l16, logical chunk 4*ks + lq
    int a_off[2], b_off[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const int c = ks * 4 + lq;
        a_off[ks] = (wm0 + l16) * BK * 2 + ((c ^ ((l16 >> 1) & 7)) * 16);
        b_off[ks] = (wn0 + (PERM ? 8 * (l16 / 4) + l16 % 4 : l16)) * BK * 2 + ((c ^ ((l16 >> 1) & 7)) * 16);
    }
    // m/n-contiguous: lane 16*g + L supplies the address of X[k = 8*g + L/4 (+32*ks, +4)][col = w0 + 16*t + 4*(L%4)];
    // the transposing read hands lane L the 4 k-values of column w0 + 16*t + L.  k + 4 and k + 32 leave the
    // swizzle bits of k alone, so the four reads of one 16-column tile (two k steps x two halves) differ only by
    // immediate offsets from one per-lane address.
    //
    // These reads are issued from inline asm: the compiler puts a vmcnt(0) in front of every transposing-read
    // builtin while an LDS-DMA load is outstanding (it cannot see that the load targets the other stage), which
    // would make the prefetched tile arrive half a tile early.  The price is that the compiler does not track
    // their completion either: every consumer sits behind an explicit `fence` (see below).
    const int tr_k = lq * 8 + l16 / 4;
    const int tr_col = 4 * (l16 % 4);
    auto tr_base = [&](auto rows_tag, int col0) -> uint32_t {  // byte offset inside the operand tile, k step 0, low half
        constexpr int ROWS = decltype(rows_tag)::value;
        const int col = col0 + tr_col;
        const int c = col / 8, half = (col / 4) % 2;
        return (uint32_t)(tr_k * ROWS * 2 + ((c ^ mc_swizzle<ROWS>(tr_k)) * 16) + half * 8);
    };
    uint32_t a_tr[A_KC ? 1 : TM], b_tr[B_KC ? 1 : TN];
    if constexpr (!A_KC) {
#pragma unroll
        for (int i = 0; i < TM; i++) a_tr[i] = tr_base(std::integral_constant<int, BM>{}, wm0 + i * 16);
    }
    if constexpr (!B_KC) {
#pragma unroll
        for (int j = 0; j < TN; j++) b_tr[j] = TA::BYTES + tr_base(std::integral_constant<int, BN>{}, wn0 + j * 16);
    }
    auto lds_addr = [](const uint8_t *p) -> uint32_t { return (uint32_t)(uintptr_t)(DFDX_LDS const uint8_t *)p; };
    auto tr_frag = [&](uint32_t addr, auto rows_tag, auto ks_tag) -> u32x4 {
        constexpr int OFF = decltype(ks_tag)::value * 32 * decltype(rows_tag)::value * 2;
        constexpr int HI = 4 * decltype(rows_tag)::value * 2;
        u32x2 l, h;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(l) : "v"(addr), "i"(OFF));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(h) : "v"(addr), "i"(OFF + HI));
        return u32x4{l[0], l[1], h[0], h[1]};
    };
    // `fence<N>(x...)`: at most N LDS operations issued by this wave may still be outstanding (they complete in
    // order); the fragments passed in are re-defined by the asm so that nothing that uses them can move above it.
    auto tie = [](u32x4 &x) { asm volatile("" : "+v"(x)); };
    constexpr int OPS_A = A_KC ? 1 : 2, OPS_B = B_KC ? 1 : 2;  // LDS instructions per fragment

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[i][j][v] = 0.0f;

    u32x4 fa[TM], fb[2][TN];
    // KSUM: the thread's piece of every A tile is chunk ks_chunk = tid % CH (8 columns) of one k-row, at byte ks_off of
    // the tile (the swizzle depends on the k-row only, so the same place in every tile).
    constexpr int CH = BM / 8, KS_SHARE = BM / 64;  // pieces per k-row; tile columns that share a tile's pieces
    static_assert(!KSUM || (!A_KC && NW == 8 && (CH == 32 || CH == 16)), "row sums: [k][m] tiles of 8-wave workgroups");
    [[maybe_unused]] float ks_sum[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    [[maybe_unused]] u32x4 ks_piece;
    [[maybe_unused]] uint32_t ks_off = 0;
    [[maybe_unused]] int ks_chunk = 0;
    [[maybe_unused]] bool ks_on = false;
    [[maybe_unused]] auto ks_begin = [&](int bn0) {
        const int tn = bn0 / BN;
        ks_on = tn < KS_SHARE;
        const int cell = (ks_on ? tn : 0) * 512 + tid;
        const int krow = cell / CH;
        ks_chunk = cell % CH;  // lanes CH apart hold the same chunk of neighbouring k-rows
        ks_off = (uint32_t)(krow * BM * 2 + (ks_chunk ^ mc_swizzle<BM>(krow)) * 16);
    };
    [[maybe_unused]] auto ks_read = [&](const uint8_t *sa) {  // asm: see the note on the transposing reads above
        if constexpr (KSUM) asm volatile("ds_read_b128 %0, %1" : "=v"(ks_piece) : "v"(lds_addr(sa) + ks_off));
    };
    [[maybe_unused]] auto ks_add = [&]() {  // after a wait for every LDS read of the wave
        if constexpr (KSUM) {
            tie(ks_piece);
            if (ks_on) {
#pragma unroll
                for (int e = 0; e < 8; e++) ks_sum[e] += Mma<T>::to_f32((uint16_t)(ks_piece[e / 2] >> ((e & 1) * 16)));
            }
        }
    };
    auto read_a = [&](const uint8_t *sa, auto ks_tag, int i0, int i1) {
        constexpr int ks = decltype(ks_tag)::value;
        [[maybe_unused]] const uint32_t base = lds_addr(sa);
#pragma unroll
        for (int i = 0; i < TM; i++)
            if (i >= i0 && i < i1) {
                if constexpr (A_KC) fa[i] = *(const u32x4 *)(sa + a_off[ks] + i * 16 * BK * 2);
                else fa[i] = tr_frag(base + a_tr[i], std::integral_constant<int, BM>{}, ks_tag);
            }
    };
    auto read_b = [&](const uint8_t *sa, auto ks_tag, u32x4(&bf)[TN]) {
        constexpr int ks = decltype(ks_tag)::value;
        const uint8_t *sb = sa + TA::BYTES;
        [[maybe_unused]] const uint32_t base = lds_addr(sa);
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (B_KC) bf[j] = *(const u32x4 *)(sb + b_off[ks] + (PERM ? (j / 2) * 32 + (j % 2) * 4 : j * 16) * BK * 2);
            else bf[j] = tr_frag(base + b_tr[j], std::integral_constant<int, BN>{}, ks_tag);
        }
    };
    // Completion of the asm-issued (transposing) reads.  `left` = LDS instructions issued after the youngest one
    // that must be complete; the hardware counter saturates the wait at 15.
    auto fence_a = [&](auto left_tag, int i0, int i1) {
        if constexpr (!A_KC) {
            constexpr int LEFT = decltype(left_tag)::value > 15 ? 15 : decltype(left_tag)::value;
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(LEFT));
#pragma unroll
            for (int i = 0; i < TM; i++)
                if (i >= i0 && i < i1) tie(fa[i]);
        }
    };
    auto fence_b = [&](auto left_tag, u32x4(&bf)[TN]) {
        if constexpr (!B_KC) {
            constexpr int LEFT = decltype(left_tag)::value > 15 ? 15 : decltype(left_tag)::value;
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(LEFT));
#pragma unroll
            for (int j = 0; j < TN; j++) tie(bf[j]);
        }
    };
    // swapped operands: the lane ends up with m = l16 and 4 consecutive n = 4*lq + 0..3 per 16x16 tile
    auto mma = [&](const u32x4(&bf)[TN], int i0, int i1) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int i = 0; i < TM; i++)
                if (i >= i0 && i < i1) acc[i][j] = Mma<T>::mfma(bf[j], fa[i], acc[i][j]);
        }
    };
    // Make the oldest requested tile visible to every wave, then request the next one into the stage that the
    // previously computed tile occupied.  Callers guarantee that this wave has issued all its LDS reads of
    // that previous tile; lgkmcnt(0) makes sure they are done.  (vmcnt(0) also covers the stores of a finished
    // C tile: they had a whole k step to drain.)
    // `behind`: how many memory instructions this wave issued AFTER its last tile request -- the stores of the C tile
    // finished before this one (one of the compile-time counts below, else 0).  The counter retires in issue order, so
    // waiting until that many are left means: the requested tile has landed, the stores may still be draining.  With
    // one k tile per work item (attention scores) a wait for everything would stop every workgroup until its previous
    // C tile is in memory, and the chip would alternate between storing and computing.
    constexpr int ST_PLAIN = TM * TN / 2, ST_ACC = (TM * (TN / 2) > 8 ? TM / 2 : TM) * TN / 2, ST_SPLIT = TM * TN;
    static_assert(ST_SPLIT < 64, "vmcnt is a 6-bit count");
    constexpr auto wait_vm_lgkm0 = [](int vm) { return (vm & 15) | ((vm >> 4) << 14) | 0x0070; };  // vmcnt(vm) & lgkmcnt(0)
    auto sync_tile = [&](int behind = 0) {
        if (behind == ST_PLAIN) __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(ST_PLAIN));
        else if (behind == ST_ACC) __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(ST_ACC));
        else if (behind == ST_SPLIT) __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(ST_SPLIT));
        else __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) & lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (fetching) issue();
    };

    // one 64-wide k tile from stage `cs`; HAS_NEXT: the next tile belongs to the same work item (hand the stage
    // over and prefetch its first fragments while the last MFMAs of this tile run)
    // LDS instructions per group of reads, as issued below: half of the A fragments, all B fragments of a k step
    constexpr int RA = 2 * Q * OPS_A, RB = TN * OPS_B, KS_READS = KSUM ? 1 : 0;
    constexpr std::integral_constant<int, 0> K0{};
    constexpr std::integral_constant<int, 1> K1{};
#define DFDX_LEFT(n) std::integral_constant<int, (n)> {}
    // First fragments of a tile, in the order the fences of tile_body assume: A rows [0, 2Q), B, A rows [2Q, TM).
    auto read_first = [&](const uint8_t *st) {
        read_a(st, K0, 0, 2 * Q);
        read_b(st, K0, fb[0]);
        read_a(st, K0, 2 * Q, TM);
    };
    auto tile_body = [&](int cs, auto has_next_tag) {
        constexpr bool HAS_NEXT = decltype(has_next_tag)::value;
        const uint8_t *sa = smem + cs * STAGE_BYTES;
        const uint8_t *sn = smem + (cs ^ 1) * STAGE_BYTES;
        // ---- k step 0 (B buffer 0); prefetch k step 1 of this tile.  Outstanding on entry, oldest first:
        //      A[0,2Q), B, A[2Q,TM) of this k step.
        fence_b(DFDX_LEFT(RA), fb[0]);
        fence_a(DFDX_LEFT(RA / 2 + RB + RA), 0, Q);
        mma(fb[0], 0, Q);
        __builtin_amdgcn_sched_barrier(0);
        fence_a(DFDX_LEFT(RB + RA), Q, 2 * Q);
        mma(fb[0], Q, 2 * Q);
        __builtin_amdgcn_sched_barrier(0);
        fence_a(DFDX_LEFT(RA / 2), 2 * Q, 3 * Q);
        mma(fb[0], 2 * Q, 3 * Q);
        __builtin_amdgcn_sched_barrier(0);
        read_a(sa, K1, 0, 2 * Q);
        read_b(sa, K1, fb[1]);
        __builtin_amdgcn_sched_barrier(0);
        fence_a(DFDX_LEFT(RA + RB), 3 * Q, TM);
        mma(fb[0], 3 * Q, TM);
        __builtin_amdgcn_sched_barrier(0);
        // ---- k step 1 (B buffer 1); prefetch k step 0 of the next tile
        fence_b(DFDX_LEFT(0), fb[1]);
        fence_a(DFDX_LEFT(RA / 2 + RB), 0, Q);
        mma(fb[1], 0, Q);
        __builtin_amdgcn_sched_barrier(0);
        read_a(sa, K1, 2 * Q, TM);
        ks_read(sa);  // KSUM: the last (youngest) LDS read of this tile, consumed behind a wait for all of them
        __builtin_amdgcn_sched_barrier(0);
        fence_a(DFDX_LEFT(RB + RA + KS_READS), Q, 2 * Q);
        mma(fb[1], Q, 2 * Q);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (HAS_NEXT) {
            // Every LDS read of this tile has been issued: wait for them and hand the stage over TWO MFMA groups before
            // the end of the tile, so that the requests for the tile after next and the first fragment reads of the
            // next one are issued under MFMAs instead of in front of an idle matrix core.  The two waves that share a
            // SIMD (w and w + NW/2) take opposite orders: one issues its MFMA group while the other issues requests.
            __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) & lgkmcnt(0)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            fence_a(DFDX_LEFT(0), 2 * Q, TM);
            ks_add();
            const bool mfma_first = __builtin_amdgcn_readfirstlane(wave) >= NW / 2;
            if (mfma_first) {
                mma(fb[1], 2 * Q, 3 * Q);
                mma(fb[1], 3 * Q, TM);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (fetching) issue();
            __builtin_amdgcn_sched_barrier(0);
            read_a(sn, K0, 0, 2 * Q);
            read_b(sn, K0, fb[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (!mfma_first) {
                mma(fb[1], 2 * Q, 3 * Q);
                mma(fb[1], 3 * Q, TM);
            }
            __builtin_amdgcn_sched_barrier(0);
            read_a(sn, K0, 2 * Q, TM);
        } else {
            fence_a(DFDX_LEFT(RA / 2 + KS_READS), 2 * Q, 3 * Q);
            mma(fb[1], 2 * Q, 3 * Q);
            __builtin_amdgcn_sched_barrier(0);
            fence_a(DFDX_LEFT(0), 3 * Q, TM);
            mma(fb[1], 3 * Q, TM);
            ks_add();
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- epilogue of one work item: lane holds m = l16 (per tile), n = 4*lq + 0..3 -------------
    // Returns the number of stores it issued after its last load (see sync_tile), 0 when that is not a fixed count.
    auto store_tile = [&](const Work &w) -> int {
        ArgParams &p = *late_args();
        const int bm0 = w.bm0, bn0 = w.bn0, split = w.split, batch = w.batch;
        if constexpr (KSUM) {
            // Lanes that hold the same 8 columns (they differ in the k-row) are added up; the first CH lanes of each wave
            // store.  These stores come before the C tile's: the count returned below stays a lower bound of what was
            // issued after the last load.
            if (ks_on) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
#pragma unroll
                    for (int d = CH; d < 64; d *= 2) ks_sum[e] += __shfl_xor(ks_sum[e], d, 64);
                }
                if (lane < CH) {
                    float *slot = p.ws_ksum + (int64_t)(((batch * p.splits + split) * KS_SHARE + bn0 / BN) * 8 + wave) * p.ws_ksum_stride + bm0 + ks_chunk * 8;
                    *(f32x4 *)slot = f32x4{ks_sum[0], ks_sum[1], ks_sum[2], ks_sum[3]};  // rows padded to whole tiles
                    *(f32x4 *)(slot + 4) = f32x4{ks_sum[4], ks_sum[5], ks_sum[6], ks_sum[7]};
                }
#pragma unroll
                for (int e = 0; e < 8; e++) ks_sum[e] = 0.0f;
            }
        }
    // f32 partial tile into the workspace (padded to whole tiles: no bounds checks).  KSUM instances run for split plans
    // only: without the other forms of the epilogue the bf16 256 x 256 instance spills far fewer registers in its k loop.
    if (KSUM || p.splits > 1) {
        float *wbase = p.ws + (int64_t)(batch * p.splits + split) * p.ws_split_stride;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            float *wrow = wbase + (int64_t)(bm0 + wm0 + i * 16 + l16) * p.ws_ld + bn0 + wn0 + lq * (PERM ? 8 : 4);
#pragma unroll
            for (int j = 0; j < TN; j++) *(f32x4 *)(wrow + (PERM ? (j / 2) * 32 + (j % 2) * 4 : j * 16)) = acc[i][j];
        }
        return ST_SPLIT;
    }
    if constexpr (!KSUM) {
    constexpr bool ANY = EDGE == 2;
    static_assert(!ANY || (EXTRA == EXTRA_NONE && TN % 2 == 0), "see launch_mfma16dma_ragged");
    [[maybe_unused]] auto columns_left = [](const uint16_t *q, int left) -> u32x4 {  // up to seven values, zeros behind them
        u32x4 r = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 7; e++)
            if (e < left) r[e / 2] |= (uint32_t)q[e] << (e % 2 * 16);
        return r;
    };
    const int cb = p.kbatches > 1 ? 0 : batch;
    uint16_t *cbase = p.c + (int64_t)(cb / p.nb2) * p.c_b1 + (int64_t)(cb % p.nb2) * p.c_b2;
    const uint16_t *const bias = p.bias + (int64_t)(cb / p.nb2) * p.bias_b1 + (int64_t)(cb % p.nb2) * p.bias_b2;
    // two finished values (rounded, packed) and their partners; see EXTRA_*
    [[maybe_unused]] auto extra = [](uint32_t o, uint32_t w) -> uint32_t {
        const float lo = Mma<T>::to_f32((uint16_t)(o & 0xffffu)), hi = Mma<T>::to_f32((uint16_t)(o >> 16));
        const float wl = Mma<T>::to_f32((uint16_t)(w & 0xffffu)), wh = Mma<T>::to_f32((uint16_t)(w >> 16));
        if constexpr (EXTRA == EXTRA_RELU) return Mma<T>::pack2(fmaxf(lo, 0.0f), fmaxf(hi, 0.0f));
        if constexpr (EXTRA == EXTRA_RESIDUAL) return Mma<T>::pack2(lo + wl, hi + wh);
        if constexpr (EXTRA == EXTRA_MASK) return (wl > 0.0f ? o & 0xffffu : 0u) | (wh > 0.0f ? o & 0xffff0000u : 0u);
        return o;
    };
    if constexpr (TN % 2 == 0) {
        // 16 B per lane: two neighbouring 16x16 tiles exchange halves between the lane rows (16-lane groups) so
        // that a lane ends up with 8 consecutive columns of one of them.  v_permlane16_swap(x, y) trades lane
        // rows 1 and 3 of x against lane rows 0 and 2 of y: afterwards lane row lq holds, in (x, y), columns
        // 8*(lq/2) .. +3 and +4 .. +7 of tile j + (lq & 1).  A wave instruction then writes 64 contiguous
        // bytes per matrix row instead of 32, which is what the memory system needs to reach its write rate.
        {
            // The lane's piece among those of a row that one instruction stores (eight of them where it covers whole lines, else four), and a value of
            // the lane that holds the next one.
            [[maybe_unused]] const int quarter = PERM ? lq : (lq & 1) * 2 + (lq >> 1);
            [[maybe_unused]] const int piece = TN == 4 ? (l16 >> 3) * 4 + quarter : quarter;
            [[maybe_unused]] const int quarter_after = (quarter + 1) % 4, lq_after = PERM ? quarter_after : (quarter_after & 1) * 2 + (quarter_after >> 1);
            [[maybe_unused]] const int after = (lq_after * 16 + (quarter == 3 ? l16 ^ 8 : l16)) * 4;
            // (rows of a lane lie 8 or 16 apart: all of them start on the same half of a word)
            [[maybe_unused]] const bool odd = (((uintptr_t)cbase >> 1) + (uint32_t)l16 * (uint32_t)p.ldc & 1) != 0;
            // (all rows of the problem, then; tiles of 96 columns a wave take no others, see takes_on)
            [[maybe_unused]] const bool words = TN == 6 || (((uintptr_t)cbase >> 1 | (uint32_t)p.ldc) & 1) == 0;
            [[maybe_unused]] auto right = [&](uint32_t x) -> uint32_t { return (uint32_t)__builtin_amdgcn_ds_bpermute(after, (int)x); };
            // The general form: bounds checks, either bias, beta = 1 with the old value loaded where it is used (edge
            // tiles, per-row bias, very large ldc).
            auto rows = [&]() {
                u32x4 cbias[TN / 2];
                float rbias_all[TM];
                if (p.bias_mode == BIAS_PER_COL) {
#pragma unroll
                    for (int jp = 0; jp < TN / 2; jp++) {
                        const int gn = bn0 + wn0 + (PERM ? jp * 32 + lq * 8 : (2 * jp + (lq & 1)) * 16 + (lq >> 1) * 8);
                        if constexpr (ANY) {
                            if (gn + 8 <= p.n) cbias[jp] = load16<true>(bias + gn);
                            else cbias[jp] = columns_left(bias + gn, p.n - gn);
                        } else {
                            cbias[jp] = *(const u32x4 *)(bias + min(gn, p.n - 8));
                        }
                    }
                }
                if (p.bias_mode == BIAS_PER_ROW) {
#pragma unroll
                    for (int i = 0; i < TM; i++) rbias_all[i] = Mma<T>::to_f32(bias[min(bm0 + wm0 + i * 16 + l16, p.m - 1)]);
                }
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const int gm_row = bm0 + wm0 + i * 16 + l16;
                    const bool row_ok = gm_row < p.m;
                    uint16_t *crow = cbase + (int64_t)gm_row * p.ldc;
#pragma unroll
                    for (int jp = 0; jp < TN / 2; jp++) {
                        float v[8];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if constexpr (PERM) {
                                v[e] = acc[i][2 * jp][e];
                                v[4 + e] = acc[i][2 * jp + 1][e];
                            } else {
                                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][2 * jp][e]),
                                                                                __float_as_uint(acc[i][2 * jp + 1][e]), false, false);
                                v[e] = __uint_as_float(r[0]);
                                v[4 + e] = __uint_as_float(r[1]);
                            }
                        }
                        const int gn = bn0 + wn0 + (PERM ? jp * 32 + lq * 8 : (2 * jp + (lq & 1)) * 16 + (lq >> 1) * 8);
                        if (!row_ok || gn >= p.n) continue;  // (n % 8 == 0 unless ANY: all 8 columns are in range)
                        const bool whole = !ANY || gn + 8 <= p.n;
                        if (p.bias_mode == BIAS_PER_ROW) {
#pragma unroll
                            for (int e = 0; e < 8; e++) v[e] += rbias_all[i];
                        }
                        if (p.bias_mode == BIAS_PER_COL) {
                            const u32x4 bv = cbias[jp];
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                v[2 * e] += Mma<T>::to_f32((uint16_t)(bv[e] & 0xffffu));
                                v[2 * e + 1] += Mma<T>::to_f32((uint16_t)(bv[e] >> 16));
                            }
                        }
                        if (p.accumulate) {
                            u32x4 old;
                            if (whole) old = load16<ANY>(EXTRA == EXTRA_FROM ? p.with + (crow + gn - p.c) : crow + gn);
                            else old = columns_left(crow + gn, p.n - gn);
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                v[2 * e] += Mma<T>::to_f32((uint16_t)(old[e] & 0xffffu));
                                v[2 * e + 1] += Mma<T>::to_f32((uint16_t)(old[e] >> 16));
                            }
                        }
                        u32x4 o;
#pragma unroll
                        for (int e = 0; e < 4; e++) o[e] = Mma<T>::pack2(v[2 * e], v[2 * e + 1]);
                        if constexpr (EXTRA != EXTRA_NONE && EXTRA != EXTRA_FROM) {  // (never together with ANY)
                            u32x4 w = {0u, 0u, 0u, 0u};
                            if constexpr (EXTRA != EXTRA_RELU) w = *(const u32x4 *)(p.with + (crow + gn - p.c));
#pragma unroll
                            for (int e = 0; e < 4; e++) o[e] = extra(o[e], w[e]);
                        }
                        if (whole) {
                            if constexpr (!ANY) *(u32x4 *)(crow + gn) = o;
                            else if (words) store_words(crow + gn, o);
                            else store_columns(crow + gn, odd, o, right(o[0]), quarter == 0, quarter == 3 || gn + 16 > p.n);
                        } else {
#pragma unroll
                            for (int e = 0; e < 7; e++)
                                if (gn + e < p.n) crow[gn + e] = (uint16_t)(o[e / 2] >> (e % 2 * 16));
                        }
                    }
                }
            };
            // Interior tiles address C as wave-uniform base (scalar registers) + one 32-bit per-lane byte offset
            // + immediate: no address arithmetic in vector registers per access.
            const int wave_u = __builtin_amdgcn_readfirstlane(wave);
            char *const tile_base = (char *)(cbase + (int64_t)(bm0 + (wave_u / WAVES_N) * WTM) * p.ldc + bn0 + (wave_u % WAVES_N) * WTN);
            const uint32_t lane_off = (uint32_t)(l16 * (int)p.ldc + (PERM ? lq * 8 : (lq & 1) * 16 + (lq >> 1) * 8)) * 2u;
            const int64_t row_step = p.ldc * 32;  // 16 rows, bytes
            // A wave tile that is 64 columns wide (TN == 4) writes whole 128 B lines: after the 16-lane swaps a lane
            // row holds the left 64 B of matrix row l16 in one register set and the right 64 B in another; lanes
            // l16 < 8 and l16 >= 8 then trade one set each (DPP row rotation by 8), so that one store instruction
            // covers rows 0..7 x 128 B and a second one rows 8..15.  Measured on the device with plain store kernels,
            // a CU retires 134 GB/s of whole-line stores but only 38 GB/s when every line arrives as two 64 B
            // halves from different instructions (and 19 GB/s in 32 B pieces); with half lines the stores of a
            // K = 64 work item take longer to leave the CU than its MFMAs take to compute.
            [[maybe_unused]] const uint32_t line_off =
                (uint32_t)((l16 & 7) * (int)p.ldc * 2 + (l16 >> 3) * 64 + (PERM ? lq : (lq & 1) * 2 + (lq >> 1)) * 16);
            [[maybe_unused]] const int64_t half_step = p.ldc * 16;  // 8 rows, bytes
            // Pure overwrite of an interior tile, optionally with a per-column bias (every forward product of whole
            // tiles, Linear's fused bias included): no bounds checks, no read of C; the bias values are fetched and
            // widened once, before the first store.
            auto rows_plain = [&](auto bias_tag, auto words_tag) {
                constexpr bool BIAS = decltype(bias_tag)::value;
                // Rounded to the 16-bit type first, the lane rows then trade PACKED pairs: half as many cross-lane
                // instructions as trading the f32 values (the conversions and trades of a K = 64 work item cost
                // the vector ALU more cycles than its MFMAs cost the matrix core).
                [[maybe_unused]] float cb[TN][4];  // bias of the columns the lane holds before the trade
                if constexpr (BIAS) {
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        u32x2 bv;
                        const uint16_t *const bias_at = bias + bn0 + wn0 + (PERM ? (j / 2) * 32 + lq * 8 + (j % 2) * 4 : j * 16 + lq * 4);
                        if constexpr (ANY) bv = *(const u32x2_any *)bias_at;
                        else bv = *(const u32x2 *)bias_at;
                        cb[j][0] = Mma<T>::to_f32((uint16_t)(bv[0] & 0xffffu));
                        cb[j][1] = Mma<T>::to_f32((uint16_t)(bv[0] >> 16));
                        cb[j][2] = Mma<T>::to_f32((uint16_t)(bv[1] & 0xffffu));
                        cb[j][3] = Mma<T>::to_f32((uint16_t)(bv[1] >> 16));
                    }
                }
                constexpr bool WITH = EXTRA == EXTRA_RESIDUAL || EXTRA == EXTRA_MASK;
                constexpr int IG = !WITH ? TM : TM * (TN / 2) > 8 ? TM / 2 : TM;  // tile rows per batch of `with`, as in rows_accumulate
                [[maybe_unused]] const int64_t to_with = WITH ? (const char *)p.with - (const char *)p.c : 0;
                [[maybe_unused]] u32x4 with[WITH ? IG : 1][TN / 2];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    if constexpr (WITH) {
                        if (i % IG == 0) {
#pragma unroll
                            for (int u = 0; u < IG; u++)
#pragma unroll
                                for (int jp = 0; jp < TN / 2; jp++)
                                    with[u][jp] = *(const u32x4 *)(tile_base + to_with + (i + u) * row_step + (TN == 4 ? jp * half_step + line_off : jp * 64 + lane_off));
                        }
                    }
                    u32x4 o[TN / 2];
#pragma unroll
                    for (int jp = 0; jp < TN / 2; jp++) {
                        uint32_t pk[2][2];  // [tile 2jp / 2jp + 1][columns 4*lq + 0,1 / 2,3]
#pragma unroll
                        for (int t = 0; t < 2; t++)
#pragma unroll
                            for (int h = 0; h < 2; h++) {
                                float x = acc[i][2 * jp + t][2 * h], y = acc[i][2 * jp + t][2 * h + 1];
                                if constexpr (BIAS) {
                                    x += cb[2 * jp + t][2 * h];
                                    y += cb[2 * jp + t][2 * h + 1];
                                }
                                pk[t][h] = Mma<T>::pack2(x, y);
                            }
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            if constexpr (PERM) {  // the lane's own 8 consecutive columns, 32 jp + 8 lq + 0..7
                                o[jp][h] = pk[0][h];
                                o[jp][2 + h] = pk[1][h];
                            } else {
                                const auto r = __builtin_amdgcn_permlane16_swap(pk[0][h], pk[1][h], false, false);
                                o[jp][h] = r[0];      // columns 8*(lq/2) + 2h, + 1 of tile 2jp + (lq & 1)
                                o[jp][2 + h] = r[1];  // columns 8*(lq/2) + 4 + 2h, + 1
                            }
                        }
                    }
                    if constexpr (TN == 4) {
                        u32x4 lo, hi;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            hi[e] = lane8_trade<0x3>(o[1][e], o[0][e]);  // rows 8..15: left halves come from lanes + 8
                            lo[e] = lane8_trade<0xC>(o[0][e], o[1][e]);  // rows 0..7: right halves come from lanes - 8
                        }
                        if constexpr (EXTRA != EXTRA_NONE) {
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                lo[e] = extra(lo[e], with[WITH ? i % IG : 0][0][e]);
                                hi[e] = extra(hi[e], with[WITH ? i % IG : 0][1][e]);
                            }
                        }
                        if constexpr (ANY && decltype(words_tag)::value) {
                            store_words(tile_base + i * row_step + line_off, lo);
                            store_words(tile_base + i * row_step + half_step + line_off, hi);
                        } else if constexpr (ANY) {
                            store_columns((uint16_t *)(tile_base + i * row_step + line_off), odd, lo, right(lo[0]), piece == 0, piece == 7);
                            store_columns((uint16_t *)(tile_base + i * row_step + half_step + line_off), odd, hi, right(hi[0]), piece == 0, piece == 7);
                        } else {
                            stream16(tile_base + i * row_step + line_off, lo);
                            stream16(tile_base + i * row_step + half_step + line_off, hi);
                        }
                    } else {
#pragma unroll
                        for (int jp = 0; jp < TN / 2; jp++) {
                            if constexpr (EXTRA != EXTRA_NONE) {
#pragma unroll
                                for (int e = 0; e < 4; e++) o[jp][e] = extra(o[jp][e], with[WITH ? i % IG : 0][jp][e]);
                            }
                            if constexpr (ANY && decltype(words_tag)::value) store_words(tile_base + i * row_step + jp * 64 + lane_off, o[jp]);
                            else if constexpr (ANY) store_columns((uint16_t *)(tile_base + i * row_step + jp * 64 + lane_off), odd, o[jp], right(o[jp][0]), piece == 0, piece == 3);
                            else stream16(tile_base + i * row_step + jp * 64 + lane_off, o[jp]);
                        }
                    }
                }
            };
            // beta = 1 on an interior tile without bias (every gradient product of whole tiles): all old values are
            // requested before the first store goes out.  The memory counter retires in issue order, so waiting for a
            // load also waits for every store issued before it: the interleaved form of `rows` drains the stores of
            // the tile sixteen times; here the loads overlap each other and are waited for in issue order.
            auto rows_accumulate = [&]() {
                constexpr int IG = TM * (TN / 2) > 8 ? TM / 2 : TM;  // tile rows per batch: at most 8 vectors in flight
                char *const base = tile_base;
                const char *const old_base = EXTRA == EXTRA_FROM ? tile_base + ((const char *)p.with - (const char *)p.c) : tile_base;
#pragma unroll
                for (int i0 = 0; i0 < TM; i0 += IG) {
                    u32x4 old[IG][TN / 2];
#pragma unroll
                    for (int i = 0; i < IG; i++)
#pragma unroll
                        for (int jp = 0; jp < TN / 2; jp++) {
                            if constexpr (TN == 4) old[i][jp] = load16<ANY>(old_base + (i0 + i) * row_step + jp * half_step + line_off);
                            else old[i][jp] = load16<ANY>(old_base + (i0 + i) * row_step + jp * 64 + lane_off);
                        }
#pragma unroll
                    for (int i = 0; i < IG; i++) {
                        float v[TN / 2][8];
#pragma unroll
                        for (int jp = 0; jp < TN / 2; jp++)
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                if constexpr (PERM) {
                                    v[jp][e] = acc[i0 + i][2 * jp][e];
                                    v[jp][4 + e] = acc[i0 + i][2 * jp + 1][e];
                                } else {
                                    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i0 + i][2 * jp][e]),
                                                                                    __float_as_uint(acc[i0 + i][2 * jp + 1][e]), false, false);
                                    v[jp][e] = __uint_as_float(r[0]);
                                    v[jp][4 + e] = __uint_as_float(r[1]);
                                }
                            }
                        if constexpr (TN == 4) {  // whole lines: v[0] becomes rows 0..7, v[1] rows 8..15 (see line_off)
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                const uint32_t left = __float_as_uint(v[0][e]), right = __float_as_uint(v[1][e]);
                                v[1][e] = __uint_as_float(lane8_trade<0x3>(right, left));
                                v[0][e] = __uint_as_float(lane8_trade<0xC>(left, right));
                            }
                        }
#pragma unroll
                        for (int jp = 0; jp < TN / 2; jp++) {
                            u32x4 o;
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                o[e] = Mma<T>::pack2(v[jp][2 * e] + Mma<T>::to_f32((uint16_t)(old[i][jp][e] & 0xffffu)),
                                                     v[jp][2 * e + 1] + Mma<T>::to_f32((uint16_t)(old[i][jp][e] >> 16)));
                            char *const at = base + (i0 + i) * row_step + (TN == 4 ? jp * half_step + line_off : jp * 64 + lane_off);
                            if constexpr (!ANY) *(u32x4 *)at = o;
                            else if (words) store_words(at, o);
                            else store_columns((uint16_t *)at, odd, o, right(o[0]), piece == 0, piece == (TN == 4 ? 7 : 3));
                        }
                    }
                }
            };
            // Every form ends by telling the compiler, with a wait that costs nothing, that the loads it issued are
            // complete: "at most as many memory instructions outstanding as the stores issued after the last load" (the
            // counter retires in issue order, and every loaded value has been consumed by then).  The general form
            // cannot count its stores and waits for them (edge tiles).
            constexpr auto vmcnt_only = [](int vm) { return (vm & 15) | ((vm >> 4) << 14) | 0x0F70; };
            const bool interior = !EDGE || (bm0 + BM <= p.m && bn0 + BN <= p.n && p.bias_mode != BIAS_PER_ROW && p.ldc < (1 << 26));
            if (interior && !p.accumulate) {
                auto by_bias = [&](auto words_tag) {
                    if (p.bias_mode == BIAS_PER_COL) rows_plain(std::true_type{}, words_tag);
                    else rows_plain(std::false_type{}, words_tag);
                };
                if (!ANY || words) by_bias(std::true_type{});
                else if constexpr (ANY) by_bias(std::false_type{});
                // stores behind the last load: the loads of `with` come in batches like those of rows_accumulate
                constexpr int ST_BEHIND = EXTRA == EXTRA_RESIDUAL || EXTRA == EXTRA_MASK ? ST_ACC : ST_PLAIN;
                __builtin_amdgcn_s_waitcnt(vmcnt_only(ST_BEHIND));
                return ST_BEHIND;
            } else if (!EDGE || (interior && p.bias_mode == BIAS_NONE)) {
                rows_accumulate();
                __builtin_amdgcn_s_waitcnt(vmcnt_only(ST_ACC));
                return ST_ACC;
            } else if constexpr (EDGE) {
                rows();
                __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
            }
            return 0;
        }
    }
    if constexpr (TN % 2 != 0) {  // a single 16-column tile per wave: 8 B per lane (the host guarantees n % 4 == 0 etc.)
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int gm_row = bm0 + wm0 + i * 16 + l16;
            if (gm_row >= p.m) continue;
            uint16_t *crow = cbase + (int64_t)gm_row * p.ldc;
            const float rbias = (p.bias_mode == BIAS_PER_ROW) ? Mma<T>::to_f32(bias[gm_row]) : 0.0f;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int gn = bn0 + wn0 + j * 16 + lq * 4;
                if (gn >= p.n) continue;  // n % 4 == 0: the 4 columns are all in range
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = acc[i][j][e] + rbias;
                if (p.bias_mode == BIAS_PER_COL) {
                    const u32x2 bv = *(const u32x2 *)(bias + gn);
                    v[0] += Mma<T>::to_f32((uint16_t)(bv[0] & 0xffffu));
                    v[1] += Mma<T>::to_f32((uint16_t)(bv[0] >> 16));
                    v[2] += Mma<T>::to_f32((uint16_t)(bv[1] & 0xffffu));
                    v[3] += Mma<T>::to_f32((uint16_t)(bv[1] >> 16));
                }
                if (p.accumulate) {
                    const u32x2 old = *(const u32x2 *)(EXTRA == EXTRA_FROM ? p.with + (crow + gn - p.c) : crow + gn);
                    v[0] += Mma<T>::to_f32((uint16_t)(old[0] & 0xffffu));
                    v[1] += Mma<T>::to_f32((uint16_t)(old[0] >> 16));
                    v[2] += Mma<T>::to_f32((uint16_t)(old[1] & 0xffffu));
                    v[3] += Mma<T>::to_f32((uint16_t)(old[1] >> 16));
                }
                u32x2 o = {Mma<T>::pack2(v[0], v[1]), Mma<T>::pack2(v[2], v[3])};
                if constexpr (EXTRA != EXTRA_NONE && EXTRA != EXTRA_FROM) {
                    u32x2 w = {0u, 0u};
                    if constexpr (EXTRA != EXTRA_RELU) w = *(const u32x2 *)(p.with + (crow + gn - p.c));
                    o = u32x2{extra(o[0], w[0]), extra(o[1], w[1])};
                }
                *(u32x2 *)(crow + gn) = o;
            }
        }
    }
    }
    return 0;
    };

    // ---- compute state ---------------------------------------------------------------------------------------
    int c_index = blockIdx.x;
    Work cw = fw;
    int c_left = cw.iters, c_stage = 0;
    int behind = 0;  // stores of the previous work item that may still be in flight
    if constexpr (KSUM) ks_begin(cw.bn0);
    issue();
    sync_tile();
    read_first(smem);
    for (;;) {
        for (; c_left > 1; --c_left) {
            tile_body(c_stage, std::true_type{});  // waits for everything outstanding and requests a tile
            behind = 0;
            c_stage ^= 1;
        }
        tile_body(c_stage, std::false_type{});
        c_stage ^= 1;
        // Work item finished.  Hand the stage over BEFORE the stores are issued: the wait inside sync_tile then
        // covers the next tile's loads and the stores of the PREVIOUS item only, and this item's stores drain while
        // the next tile is computed.  (Converting the accumulators before that wait was tried: it costs registers
        // inside the k loop and lost.)
        const bool more = c_index + (int)gridDim.x < p.total_blocks;
        if (more) sync_tile(behind);
        behind = __builtin_amdgcn_readfirstlane(store_tile(cw));
        if (!more) break;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][v] = 0.0f;
        c_index += gridDim.x;
        cw = decode(*late_args(), c_index);
        c_left = cw.iters;
        if constexpr (KSUM) ks_begin(cw.bn0);
        read_first(smem + c_stage * STAGE_BYTES);
    }
}


#undef DFDX_LEFT

// X(id, BM, BN, WAVES_M, WAVES_N); ids are 1-based inside this family and shared with the ring tiles (gemm_mfma16_ring.h).
#define DFDX_MFMA16_DMA_VARIANTS(X) \
    X(1, 256, 256, 2, 4)            \
    X(2, 256, 128, 4, 2)            \
    X(3, 128, 128, 2, 4)            \
    X(4, 256, 64, 4, 2)             \
    X(5, 128, 64, 2, 4)             \
    X(10, 256, 192, 4, 2)

// Persistent launch: as many workgroups as the chip holds at once (what LDS and registers allow per compute
// unit, rounded to a multiple of the 8 XCDs so that work item i and i + grid land on the same XCD), or one per
// work item when there are fewer.
// Used inside a function template with T, BM, BN, WM, WN; `p`, `compute_units` and `stream` in scope.
#define DFDX_LAUNCH(AKC, BKC, EDGE, ...)                                                                       \
    do {                                                                                                       \
        auto kern = gemm_mfma16_dma_kernel<T, BM, BN, WM, WN, AKC, BKC, EDGE, ##__VA_ARGS__>;                  \
        static PerDevice occupancy_on;                                                                         \
        std::atomic<int> &known = occupancy_on.here();                                                         \
        int per_cu = known.load(std::memory_order_acquire);                                                    \
        if (per_cu == 0) {                                                                                     \
            hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                               (int)lds);                                                      \
            if (e != hipSuccess) return e;                                                                     \
            int occ = 0;                                                                                       \
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void *)kern, NT, lds);               \
            if (e != hipSuccess) return e;                                                                     \
            per_cu = occ < 1 ? 1 : occ;                                                                        \
            known.store(per_cu, std::memory_order_release);                                                    \
        }                                                                                                      \
        const int resident = (compute_units < 8 ? 8 : compute_units) * per_cu / 8 * 8;                         \
        p.grid = p.total_blocks <= resident ? p.total_blocks : resident;                                       \
        kern<<<dim3((unsigned)p.grid), dim3(NT), lds, stream>>>(p);                                            \
    } while (0)

// whole tiles only, and nothing but the two interior epilogue forms: the instance without the general form
template <int BM, int BN> inline bool needs_edge_form(const Params &p) {
    return p.m % BM != 0 || p.n % BN != 0 || p.bias_mode == BIAS_PER_ROW || p.ldc >= (1 << 26) || (p.accumulate && p.bias_mode != BIAS_NONE);
}

}  // namespace
}  // namespace dfdx_rocm
