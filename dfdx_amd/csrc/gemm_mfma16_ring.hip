// MFMA GEMM for 16-bit inputs (f16 / bf16), f32 accumulate, gfx950 (CDNA4): small tiles behind a deep ring of LDS stages, for
// products whose tiles do not fill the chip for long, and for any length of the contraction.
//
// What bounds those products is the time that a k tile takes from memory into LDS: with one tile requested ahead
// (gemm_mfma16_dma.hip) a workgroup waits 0.8 - 1.1 us per 64 of k, whatever the tile.  Here DEPTH tiles are on their way, the
// tile in hand is in registers, and every workgroup makes one tile of C (no persistent walk: all places are taken at once).  A k tile of
// 64 x 64 then takes 0.19 us, one of 128 x 128 0.43: what LDS can take in and give out, (BM + BN) * 128 bytes written once and read by
// the waves of a row or column each, at 128 bytes a clock.  f16, on buffers that the last-level cache holds, persistent tiles -> here:
// 1344 x 3072 x 768 28.9 -> 13.2 us, 529 x 768 x 768 10.1 -> 5.8, 1536 x 1344 x 768 (A, B across k) 16.6 -> 9.5, and with
// k off the tile, against the register-staged tiles, 768 x 529 x 3072 17.2 -> 10.1, 1536 x 1528 x 400 24.0 -> 10.4.
//   - more stages than four gain nothing (64 x 64, six and eight stages: level), three let a third workgroup on the compute unit;
//   - the steady part of the k loop is straight code of two steps (per step: one wait, one barrier, the fragment reads of the next
//     tile, two groups of MFMAs with the requests between them): with the requests' bookkeeping in it the loop took 10 - 20 % longer;
//   - a last k tile that is not whole is requested piece by piece: pieces beyond the contraction come from a line of zeros, so that
//     the order of the sum, and its bits, are those of every other 16-bit tile;
//   - C goes through LDS: one epilogue of whole rows for any layout, alignment and number of columns; what it reads besides (bias, old
//     values, the other operand of a residual or mask) is requested before the k loop (3152 x 768 x 768 + residual 15.6 -> 14.0 us);
//   - the sums of A's rows (a Linear layer's bias gradient) are one more product, with ones, in the waves that hold the first columns
//     of C: no reduction of its own is launched (two launches of 4 us each for every Linear layer's backward).
#include "gemm_mfma16_dma.h"
#include "gemm_mfma16_ring.h"

namespace dfdx_rocm {
namespace {

__device__ __align__(16) uint32_t ring_zeros[4];  // what a lane beyond the contraction loads

// A DmaTile whose last k tile may be partial: pieces beyond `k_left` come from ring_zeros.
template <int ROWS, int NWAVES, bool KC, bool PERM> struct RingTile : DmaTile<ROWS, NWAVES, KC, PERM> {
    using Base = DmaTile<ROWS, NWAVES, KC, PERM>;
    template <int I> __device__ __forceinline__ void issue_part(const char *origin, int k_left, int wave, int lane, DFDX_LDS void *lds) const {
        if constexpr (I < Base::IPW) {
            constexpr int BACK = 1024 * (Base::IPW - 1 - I);
            const int slot = (wave * Base::IPW + I) * 64 + lane, r = slot / Base::CPR, cp = slot % Base::CPR;
            const int k = !KC ? r : 8 * (PERM ? cp ^ ((((r >> 3) & 3) << 1) | ((r >> 1) & 1)) : cp ^ ((r >> 1) & 7));
            const char *from = k < k_left ? origin + this->goff[I] : (const char *)ring_zeros + BACK;
            __builtin_amdgcn_global_load_lds((const DFDX_GLB void *)from, lds, 16, -BACK, 0);
            issue_part<I + 1>(origin, k_left, wave, lane, lds);
        }
    }
};

template <int N> __device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70); }
// at most `ahead` tiles of L requests each still on their way
template <int L, int MOST> __device__ __forceinline__ void wait_tiles(int ahead) {
    if (ahead >= MOST) wait_vm<L * MOST>();
    else if constexpr (MOST > 0) wait_tiles<L, MOST - 1>(ahead);
}

// An LDS fragment in two halves: LDS reads are issued from inline asm (the compiler would wait for every LDS-DMA load in front of a
// transposing read) and become a matrix operand only behind the wait that `landed` stands for.
struct Frag {
    u32x2 lo, hi;
};
struct FragK {
    u32x4 v;
};
__device__ __forceinline__ void landed(Frag &f) { asm volatile("" : "+v"(f.lo), "+v"(f.hi)); }
__device__ __forceinline__ void landed(FragK &f) { asm volatile("" : "+v"(f.v)); }
__device__ __forceinline__ u32x4 operand(const Frag &f) { return u32x4{f.lo[0], f.lo[1], f.hi[0], f.hi[1]}; }
__device__ __forceinline__ u32x4 operand(const FragK &f) { return f.v; }

template <typename T> __device__ __forceinline__ u32x4 ones();
template <> __device__ __forceinline__ u32x4 ones<_Float16>() { return u32x4{0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u}; }
template <> __device__ __forceinline__ u32x4 ones<__bf16>() { return u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u}; }

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int DEPTH, bool A_KC, bool B_KC>
__device__ __forceinline__ void ring_tile(const RingParams &p, const int index, uint8_t *smem) {
    constexpr int NW = WAVES_M * WAVES_N, NT = NW * 64;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, TM = WTM / 16, TN = WTN / 16;
    constexpr bool PERM = B_KC && TN % 2 == 0;
    constexpr bool KSUM = !A_KC && !B_KC;
    using TA = RingTile<BM, NW, A_KC, false>;
    using TB = RingTile<BN, NW, B_KC, PERM>;
    constexpr int STAGE_BYTES = TA::BYTES + TB::BYTES, L = TA::IPW + TB::IPW;
    static_assert(L * (DEPTH - 1) < 64, "vmcnt is a 6-bit count");

    const int tid = threadIdx.x;
    const int lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wm0 = (wave / WAVES_N) * WTM, wn0 = (wave % WAVES_N) * WTN;
    const int l16 = lane % 16, lq = lane / 16;

    // ---- the work item: a tile of C, of one batch or of one piece of the contraction -----------------------------------
    const int ktiles = (p.k + BK - 1) / BK;
    const int work = xcd_remap(index, p.items);
    const int bidx = work / p.tiles_per_batch, tile = work % p.tiles_per_batch;
    const int gsize = p.group_m * p.tiles_n, first_m = tile / gsize * p.group_m, gm_rows = min(p.tiles_m - first_m, p.group_m);
    const int bm0 = (first_m + (tile % gsize) % gm_rows) * BM, bn0 = ((tile % gsize) / gm_rows) * BN;
    const int batch = p.splits > 1 ? bidx / p.splits : bidx, split = p.splits > 1 ? bidx - batch * p.splits : 0;
    const int it0 = split * p.chunk, iters = min(ktiles * p.kbatches - it0, p.chunk);

    // ---- requests ----------------------------------------------------------------------------------------------------
    const int64_t a_step = A_KC ? BK : (int64_t)BK * p.lda, b_step = B_KC ? BK : (int64_t)BK * p.ldb;
    int f_kb = p.kbatches > 1 ? it0 / ktiles : batch, f_kt = p.kbatches > 1 ? it0 % ktiles : it0, f_left = iters;
    auto a_origin = [&](int kb) { return p.a + (int64_t)(kb / p.nb2) * p.a_b1 + (int64_t)(kb % p.nb2) * p.a_b2 + (A_KC ? (int64_t)bm0 * p.lda : bm0); };
    auto b_origin = [&](int kb) { return p.b + (int64_t)(kb / p.nb2) * p.b_b1 + (int64_t)(kb % p.nb2) * p.b_b2 + (B_KC ? (int64_t)bn0 * p.ldb : bn0); };
    const uint16_t *a_next = a_origin(f_kb) + f_kt * a_step, *b_next = b_origin(f_kb) + f_kt * b_step;
    TA ta;
    TB tb;
    ta.init(p.lda, (A_KC ? p.m : (p.m + 7) & ~7) - bm0, wave, lane);
    tb.init(p.ldb, (B_KC ? p.n : (p.n + 7) & ~7) - bn0, wave, lane);
    const uint32_t smem_addr = (uint32_t)(uintptr_t)(DFDX_LDS const uint8_t *)smem;
    const uint32_t lds_a = __builtin_amdgcn_readfirstlane(TA::wave_base(smem_addr, wave));
    const uint32_t lds_b = __builtin_amdgcn_readfirstlane(TB::wave_base(smem_addr + TA::BYTES, wave));
    auto request_full = [&](uint32_t st) {
        ta.issue(a_next, lds_a + st);
        tb.issue(b_next, lds_b + st);
        --f_left;
        ++f_kt;
        a_next += a_step;
        b_next += b_step;
    };
    auto request = [&](uint32_t st) {  // (st: byte offset of the stage)
        if (f_kt == ktiles) {
            f_kt = 0;
            ++f_kb;
            a_next = a_origin(f_kb);
            b_next = b_origin(f_kb);
        }
        if (f_kt == p.whole) {
            a_next += p.a_last;
            b_next += p.b_last;
        }
        const int k_left = p.k - f_kt * BK;
        if (k_left >= BK) {
            request_full(st);
            return;
        }
        // lane and wave as new values: what the partial tile is addressed by is not carried through the loop
        int f_wave = wave, f_lane = lane;
        asm volatile("" : "+s"(f_wave), "+v"(f_lane));
        ta.template issue_part<0>((const char *)a_next, k_left, f_wave, f_lane, (DFDX_LDS void *)(uintptr_t)(lds_a + st));
        tb.template issue_part<0>((const char *)b_next, k_left, f_wave, f_lane, (DFDX_LDS void *)(uintptr_t)(lds_b + st));
        --f_left;
        ++f_kt;
    };

    // ---- fragments: addresses inside a stage as in gemm_mfma16_dma_kernel -----------------------------------------------
    using FA = std::conditional_t<A_KC, FragK, Frag>;
    using FB = std::conditional_t<B_KC, FragK, Frag>;
    const int tr_k = lq * 8 + l16 / 4, tr_col = 4 * (l16 % 4);
    auto tr_base = [&](auto rows_tag, int col0) -> uint32_t {
        constexpr int ROWS = decltype(rows_tag)::value;
        const int col = col0 + tr_col, c = col / 8, half = (col / 4) % 2;
        return (uint32_t)(tr_k * ROWS * 2 + ((c ^ mc_swizzle<ROWS>(tr_k)) * 16) + half * 8);
    };
    uint32_t a_at[A_KC ? 2 : TM], b_at[B_KC ? 2 : TN];  // along k: per k step; across: per 16 columns
    if constexpr (A_KC) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++) a_at[ks] = (uint32_t)((wm0 + l16) * BK * 2 + (((ks * 4 + lq) ^ ((l16 >> 1) & 7)) * 16));
    } else {
#pragma unroll
        for (int i = 0; i < TM; i++) a_at[i] = tr_base(std::integral_constant<int, BM>{}, wm0 + i * 16);
    }
    if constexpr (B_KC) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
            b_at[ks] = (uint32_t)(TA::BYTES + (wn0 + (PERM ? 8 * (l16 / 4) + l16 % 4 : l16)) * BK * 2 + (((ks * 4 + lq) ^ ((l16 >> 1) & 7)) * 16));
    } else {
#pragma unroll
        for (int j = 0; j < TN; j++) b_at[j] = TA::BYTES + tr_base(std::integral_constant<int, BN>{}, wn0 + j * 16);
    }
    auto read_k = [](FragK &f, uint32_t addr, auto off_tag) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.v) : "v"(addr), "i"(decltype(off_tag)::value));
    };
    auto read_tr = [](Frag &f, uint32_t addr, auto rows_tag, auto ks_tag) {
        constexpr int OFF = decltype(ks_tag)::value * 32 * decltype(rows_tag)::value * 2, HI = 4 * decltype(rows_tag)::value * 2;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.lo) : "v"(addr), "i"(OFF));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.hi) : "v"(addr), "i"(OFF + HI));
    };

    f32x4 acc[TM][TN];
    [[maybe_unused]] f32x4 sums[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        sums[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // the sums of A's rows: one more product, with ones, in the waves that hold the first columns of C
    const bool summing = KSUM && p.ksum && bn0 == 0 && wn0 == 0;

    auto read_step = [&](uint32_t st, auto ks_tag, FA(&fa)[TM], FB(&fb)[TN]) {
        constexpr int ks = decltype(ks_tag)::value;
        auto one_a = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            if constexpr (i < TM) {
                if constexpr (A_KC) read_k(fa[i], st + a_at[ks], std::integral_constant<int, i * 16 * BK * 2>{});
                else read_tr(fa[i], st + a_at[i], std::integral_constant<int, BM>{}, ks_tag);
            }
        };
        auto one_b = [&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            if constexpr (j < TN) {
                if constexpr (B_KC) read_k(fb[j], st + b_at[ks], std::integral_constant<int, (PERM ? (j / 2) * 32 + (j % 2) * 4 : j * 16) * BK * 2>{});
                else read_tr(fb[j], st + b_at[j], std::integral_constant<int, BN>{}, ks_tag);
            }
        };
        static_assert(TM <= 4 && TN <= 4, "fragments listed one by one");
        one_b(std::integral_constant<int, 0>{}); one_b(std::integral_constant<int, 1>{}); one_b(std::integral_constant<int, 2>{}); one_b(std::integral_constant<int, 3>{});
        one_a(std::integral_constant<int, 0>{}); one_a(std::integral_constant<int, 1>{}); one_a(std::integral_constant<int, 2>{}); one_a(std::integral_constant<int, 3>{});
    };
    auto multiply = [&](FA(&fa)[TM], FB(&fb)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++) landed(fa[i]);
#pragma unroll
        for (int j = 0; j < TN; j++) landed(fb[j]);
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int i = 0; i < TM; i++) acc[i][j] = Mma<T>::mfma(operand(fb[j]), operand(fa[i]), acc[i][j]);
        if constexpr (KSUM) {
            if (summing) {
#pragma unroll
                for (int i = 0; i < TM; i++) sums[i] = Mma<T>::mfma(ones<T>(), operand(fa[i]), sums[i]);
            }
        }
    };

    // ---- what the epilogue reads, requested ahead of everything else -------------------------------------------------------
    // A thread finishes the pieces (8 columns of a row) of cells tid, tid + NT, ..; they share their columns.
    constexpr int CPR = BN / 8, CELLS = BM * CPR / NT;
    static_assert(NT % CPR == 0, "a thread's cells lie in the same columns");
    const int cb = p.kbatches > 1 ? 0 : batch;
    uint16_t *const cbase = p.c + (int64_t)(cb / p.nb2) * p.c_b1 + (int64_t)(cb % p.nb2) * p.c_b2;
    const uint16_t *const bias = p.bias + (int64_t)(cb / p.nb2) * p.bias_b1 + (int64_t)(cb % p.nb2) * p.bias_b2;
    const int gn = bn0 + tid % CPR * 8, left = p.n - gn;
    auto piece = [&](const uint16_t *from) -> u32x4 {  // eight columns, zeros beyond the last one
        u32x4 v = {0u, 0u, 0u, 0u};
        if (left >= 8) {
            v = load16<true>(from);
        } else {
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (e < left) v[e / 2] |= (uint32_t)from[e] << (e % 2 * 16);
        }
        return v;
    };
    auto widen = [](u32x4 v, float(&f)[8]) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            f[2 * e] = Mma<T>::to_f32((uint16_t)(v[e] & 0xffffu));
            f[2 * e + 1] = Mma<T>::to_f32((uint16_t)(v[e] >> 16));
        }
    };
    // the old values of C, or the second operand of the op behind the product
    const bool from_with = p.extra == EXTRA_FROM || p.extra == EXTRA_RESIDUAL || p.extra == EXTRA_MASK;
    u32x4 partner[CELLS] = {}, column_bias = {0u, 0u, 0u, 0u};
    if (p.splits <= 1) {
        if (p.bias_mode == BIAS_PER_COL) column_bias = piece(bias + gn);
        if (p.accumulate || from_with) {
            const uint16_t *const base = cbase + (from_with ? p.with - p.c : 0);
#pragma unroll
            for (int q = 0; q < CELLS; q++) {
                const int gm = bm0 + (q * NT + tid) / CPR;
                if (gm < p.m) partner[q] = piece(base + (int64_t)gm * p.ldc + gn);
            }
        }
    }

    // Tile t + 1 is read into registers while tile t is multiplied.
    FA fa[2][2][TM];
    FB fb[2][2][TN];
    for (int s = 0; s < DEPTH && f_left; s++) request((uint32_t)s * STAGE_BYTES);
    uint32_t st = 0;  // stage of the tile in hand
    auto everybody = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto read_tile = [&](FA(&a)[2][TM], FB(&b)[2][TN]) {
        read_step(smem_addr + st, std::integral_constant<int, 0>{}, a[0], b[0]);
        read_step(smem_addr + st, std::integral_constant<int, 1>{}, a[1], b[1]);
    };
    // FULL: the next tile is on its way and DEPTH - 2 behind it, and one more whole tile of the same matrices is to be requested.
    auto step = [&](int t, auto now_tag, auto full_tag) {
        constexpr int now = decltype(now_tag)::value;
        constexpr bool FULL = decltype(full_tag)::value;
        asm volatile("s_waitcnt lgkmcnt(0)");
        const uint32_t done = st;
        const bool more = FULL || t + 1 < iters;
        if (more) {
            if constexpr (FULL) wait_vm<L *(DEPTH - 2)>();
            else wait_tiles<L, DEPTH - 2>(iters - f_left - 2 - t);
            everybody();  // tile t + 1 has landed, tile t is in registers
            st = st == (DEPTH - 1) * STAGE_BYTES ? 0 : st + STAGE_BYTES;
            read_tile(fa[1 - now], fb[1 - now]);
        }
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[now][0], fb[now][0]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (FULL) request_full(done);
        else if (more && f_left) request(done);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[now][1], fb[now][1]);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, 0> EVEN{};
    constexpr std::integral_constant<int, 1> ODD{};
    wait_tiles<L, DEPTH - 1>(iters - f_left - 1);
    everybody();
    read_tile(fa[0], fb[0]);
    for (int t = 0; t < iters; t += 2) {
        for (int whole = min(p.whole - f_kt, f_left); whole >= 2; whole -= 2, t += 2) {
            step(t, EVEN, std::true_type{});
            step(t + 1, ODD, std::true_type{});
        }
        step(t, EVEN, std::false_type{});
        if (t + 1 < iters) step(t + 1, ODD, std::false_type{});
    }

    // ---- epilogue: the tile goes through LDS, so that a thread holds 8 columns of a row whatever the layout --------------------
    // (the last stage's reads are done; the stages hold nothing that is still needed once every wave is here)
    __syncthreads();
    constexpr int PITCH = BN + 4;
    static_assert(BM * PITCH * 4 <= DEPTH * STAGE_BYTES, "the tile of C in f32 fits the stages");
    float *const out = (float *)smem;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
            *(f32x4 *)(out + (wm0 + i * 16 + l16) * PITCH + wn0 + (PERM ? (j / 2) * 32 + lq * 8 + (j % 2) * 4 : j * 16 + lq * 4)) = acc[i][j];
    if constexpr (KSUM) {
        if (summing && lq == 0) {
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int row = bm0 + wm0 + i * 16 + l16;
                if (p.splits > 1) {
                    p.ws_ksum[(int64_t)(batch * p.splits + split) * p.ws_ksum_stride + row] = sums[i][0];  // (rows padded to whole tiles)
                } else if (row < p.m) {
                    const int kb = p.kbatches > 1 ? 0 : batch;
                    uint16_t *dst = p.ksum + (int64_t)(kb / p.nb2) * p.ksum_b1 + (int64_t)(kb % p.nb2) * p.ksum_b2 + row;
                    *dst = Mma<T>::from_f32((p.ksum_accumulate ? Mma<T>::to_f32(*dst) : 0.0f) + sums[i][0]);
                }
            }
        }
    }
    __syncthreads();
    if (p.splits > 1) {
        float *const wbase = p.ws + (int64_t)(batch * p.splits + split) * p.ws_split_stride + (int64_t)bm0 * p.ws_ld + bn0;
#pragma unroll
        for (int q = 0; q < BM * CPR * 2 / NT; q++) {
            const int cell = q * NT + tid, row = cell / (CPR * 2), col = cell % (CPR * 2) * 4;
            *(f32x4 *)(wbase + (int64_t)row * p.ws_ld + col) = *(const f32x4 *)(out + row * PITCH + col);
        }
        return;
    }
    // (stores where the piece lies: handing columns on so that odd rows' pieces lie on words, as the persistent tiles do, has these tiles wait
    // for the lanes' trade at their end -- 512 x 768 x 1487 f16 nt 6.0 -> 6.3 us, 6812 x 1152 x 233 10.7 -> 11.5, 44 products 2.5 % in the mean)
#pragma unroll
    for (int q = 0; q < CELLS; q++) {
        const int row = (q * NT + tid) / CPR, gm = bm0 + row;
        if (gm >= p.m || left <= 0) continue;
        uint16_t *const at = cbase + (int64_t)gm * p.ldc + gn;
        float v[8], w[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) *(f32x4 *)(v + e) = *(const f32x4 *)(out + row * PITCH + tid % CPR * 8 + e);
        if (p.bias_mode == BIAS_PER_COL) {
            widen(column_bias, w);
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] += w[e];
        } else if (p.bias_mode == BIAS_PER_ROW) {
            const float r = Mma<T>::to_f32(bias[gm]);
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] += r;
        }
        widen(partner[q], w);
        if (p.accumulate) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] += w[e];
        }
        if (p.extra != EXTRA_NONE && p.extra != EXTRA_FROM) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float r = Mma<T>::to_f32(Mma<T>::from_f32(v[e]));  // the value that the op behind the product would have read
                v[e] = p.extra == EXTRA_RELU ? fmaxf(r, 0.0f) : p.extra == EXTRA_RESIDUAL ? r + w[e] : w[e] > 0.0f ? r : 0.0f;
            }
        }
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = Mma<T>::pack2(v[2 * e], v[2 * e + 1]);
        if (left >= 8) {
            *(u32x4_any *)at = o;
        } else {
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (e < left) at[e] = (uint16_t)(o[e / 2] >> (e % 2 * 16));
        }
    }
}

template <typename T, int BM, int BN, int WM, int WN, int DEPTH, bool A_KC, bool B_KC>
__global__ __launch_bounds__(WM *WN * 64, 2) void gemm_mfma16_ring_kernel(const RingParams p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    ring_tile<T, BM, BN, WM, WN, DEPTH, A_KC, B_KC>(p, blockIdx.x, smem);
}

// The two products of a backward pass, which share nothing but what they read: one launch where neither fills the chip by itself, and
// none of the gaps between short launches.  The longer items go first; each product keeps its own order over the XCDs (workgroups
// behind the items of the first one, up to the next multiple of eight, have nothing to do).  f16, traced kernels: a Linear layer's
// backward of 400 x 1024 to 256 7.5 + 6.2 -> 7.7 us, 529 x 768 to 768 6.9 + 7.6 -> 8.7, 1344 x 768 to 3072 18.9 + 19.9 -> 32.4; a
// training step of the block of 4 x 100 tokens, d 256, 25 -> 19 launches, 137 -> 118 us.
template <typename T, int BM, int BN, int WM, int WN, int DEPTH, bool B_KC>
__global__ __launch_bounds__(WM *WN * 64, 2) void gemm_mfma16_ring_two_kernel(const RingParams p, const RingParams q, const int q_first) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int front = q_first ? q.items : p.items, at = (int)blockIdx.x, behind = at - ((front + 7) & ~7);
    if (behind < 0 && at >= front) return;
    if ((behind >= 0) == (q_first != 0)) ring_tile<T, BM, BN, WM, WN, DEPTH, true, B_KC>(p, behind >= 0 ? behind : at, smem);
    else ring_tile<T, BM, BN, WM, WN, DEPTH, false, false>(q, behind >= 0 ? behind : at, smem);
}

template <int LDS, typename Kernel, typename... Args> hipError_t start(PerDevice &ready, Kernel kern, int blocks, int threads, hipStream_t stream, const Args &...args) {
    std::atomic<int> &known = ready.here();
    if (!known.load(std::memory_order_acquire)) {
        if (hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS); e != hipSuccess) return e;
        known.store(1, std::memory_order_release);
    }
    kern<<<dim3((unsigned)blocks), dim3((unsigned)threads), LDS, stream>>>(args...);
    return hipGetLastError();
}

template <typename T, int BM, int BN, int WM, int WN, int DEPTH>
hipError_t launch_tile(const RingParams &p, const RingParams *q, bool a_kc, bool b_kc, hipStream_t stream) {
    constexpr int LDS = DEPTH * (BM + BN) * BK * 2, NT = WM * WN * 64;
    static PerDevice ready[6];
    if (q) {
        const int q_first = (q->k + BK - 1) / BK * q->kbatches > (p.k + BK - 1) / BK * p.kbatches;  // the longer items go first
        const int front = q_first ? q->items : p.items, blocks = ((front + 7) & ~7) + (q_first ? p.items : q->items);
        if (b_kc) return start<LDS>(ready[4], gemm_mfma16_ring_two_kernel<T, BM, BN, WM, WN, DEPTH, true>, blocks, NT, stream, p, *q, q_first);
        return start<LDS>(ready[5], gemm_mfma16_ring_two_kernel<T, BM, BN, WM, WN, DEPTH, false>, blocks, NT, stream, p, *q, q_first);
    }
    if (a_kc && b_kc) return start<LDS>(ready[0], gemm_mfma16_ring_kernel<T, BM, BN, WM, WN, DEPTH, true, true>, p.items, NT, stream, p);
    if (a_kc) return start<LDS>(ready[1], gemm_mfma16_ring_kernel<T, BM, BN, WM, WN, DEPTH, true, false>, p.items, NT, stream, p);
    if (b_kc) return start<LDS>(ready[2], gemm_mfma16_ring_kernel<T, BM, BN, WM, WN, DEPTH, false, true>, p.items, NT, stream, p);
    return start<LDS>(ready[3], gemm_mfma16_ring_kernel<T, BM, BN, WM, WN, DEPTH, false, false>, p.items, NT, stream, p);
}

template <typename T> hipError_t launch_variant(int ring, const RingParams &p, const RingParams *q, bool a_kc, bool b_kc, hipStream_t s) {
    switch (ring) {
#define X(id, bm, bn, wm, wn, depth) \
    case id: return launch_tile<T, bm, bn, wm, wn, depth>(p, q, a_kc, b_kc, s);
        DFDX_MFMA16_RING_VARIANTS(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_mfma16_ring(int ring, int dtype, const RingParams &p, bool a_kc, bool b_kc, hipStream_t stream) {
    return dtype == DT_F16 ? launch_variant<_Float16>(ring, p, nullptr, a_kc, b_kc, stream) : launch_variant<__bf16>(ring, p, nullptr, a_kc, b_kc, stream);
}
hipError_t launch_mfma16_ring_two(int ring, int dtype, const RingParams &p, const RingParams &q, bool p_b_kc, hipStream_t stream) {
    return dtype == DT_F16 ? launch_variant<_Float16>(ring, p, &q, true, p_b_kc, stream) : launch_variant<__bf16>(ring, p, &q, true, p_b_kc, stream);
}

}  // namespace dfdx_rocm
