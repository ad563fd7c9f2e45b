// MFMA GEMM for 16-bit inputs (f16 / bf16), f32 accumulate, gfx950 (CDNA4): the fast path for
// K % 64 == 0.  v_mfma_f32_16x16x32_{f16,bf16}; BM x BN x 64 tile per workgroup of 8 waves.
//
// Data movement
//   * A and B tiles go from global memory straight into LDS with 16 B-per-lane LDS-DMA loads
//     (global_load_lds_dwordx4): no VGPR staging, no ds_write.  One wave instruction fills 1 KB of
//     LDS contiguously; WHICH 16 B chunk of the tile a lane fetches is chosen so that the tile lands
//     XOR-swizzled and every fragment read is bank-conflict free (measured: SQ_LDS_BANK_CONFLICT = 0).
//   * k-contiguous operand (A row-major, or B stored [N][K]): LDS holds [row][64 k], chunk c of row r at
//     position c ^ ((r >> 1) & 7); fragments are read with ds_read_b128.
//   * m/n-contiguous operand (A stored [K][M], or B row-major [K][N]): LDS holds [k][rows] exactly as in
//     memory (no transpose anywhere); fragments are read with the transposing ds_read_b64_tr_b16, two per
//     fragment.  Chunk c of k-row k sits at c ^ swz(k) (see mc_swizzle).
//   * Two LDS stages.  Tile t+1 is requested right after the barrier that retires tile t-1 and has one
//     full k step of MFMAs to arrive.
// Schedule per k step (32 wide, two per tile): the A fragments are single buffered in two halves, the B
// fragments double buffered; the reads for the next step are issued in the middle of the MFMAs of the
// current one, into registers that are already free, so each read has >= a quarter step of MFMAs to land.
// One s_barrier per tile.  Stage hand-over uses explicit s_waitcnt vmcnt/lgkmcnt + s_barrier.
//
// Rows/columns past the matrix edge are clamped onto valid addresses (they only feed C entries that are
// never stored).  There is no k tail here: K % 64 != 0 is served by gemm_mfma16_ring.hip, whose tiles are planned here too, and by the
// register-staged kernel.
#include "gemm_mfma16_dma.h"
#include "gemm_mfma16_ring.h"
#include "../../include/dfdx_rocm.h"
#include <algorithm>
#include <array>
#include <cmath>

namespace dfdx_rocm {
namespace {

// ------------------------------------------------------------------ host side --

struct Variant {
    const char *name;
    int bm, bn, waves_m, waves_n;
    bool ring;  // a tile of gemm_mfma16_ring.hip
};

// Ids are those of the two lists, which count through both: a caller may ask for a tile by its id, so new ones go behind.
#define X(...) +1
constexpr int kNumVariants = 0 DFDX_MFMA16_DMA_VARIANTS(X) DFDX_MFMA16_RING_VARIANTS(X);
#undef X
constexpr std::array<Variant, kNumVariants> kVariants = [] {
    std::array<Variant, kNumVariants> v{};
#define X(id, bm, bn, wm, wn) v[id - 1] = {"dma_" #bm "x" #bn "x64_w" #wm "x" #wn, bm, bn, wm, wn, false};
    DFDX_MFMA16_DMA_VARIANTS(X)
#undef X
#define X(id, bm, bn, wm, wn, depth) v[id - 1] = {"ring_" #bm "x" #bn "x64_w" #wm "x" #wn "_s" #depth, bm, bn, wm, wn, true};
    DFDX_MFMA16_RING_VARIANTS(X)
#undef X
    return v;
}();
inline bool is_ring(int variant) { return kVariants[variant - 1].ring; }

template <typename T, int BM, int BN, int WM, int WN>
hipError_t launch_layout(Params p, int compute_units, bool a_kc, bool b_kc, hipStream_t stream) {
    constexpr int NT = WM * WN * 64;
    constexpr size_t lds = (size_t)STAGES * (BM + BN) * BK * 2;
    const bool edge = needs_edge_form<BM, BN>(p);
    if (p.ws_ksum) {  // row sums of A: compiled for the layout of weight gradients only (ksum_supported)
        if (a_kc || b_kc) return hipErrorInvalidValue;
        if (edge) DFDX_LAUNCH(false, false, true, true);
        else DFDX_LAUNCH(false, false, false, true);
    } else if (edge) {
        if (a_kc && b_kc) DFDX_LAUNCH(true, true, true);
        else if (a_kc && !b_kc) DFDX_LAUNCH(true, false, true);
        else if (!a_kc && b_kc) DFDX_LAUNCH(false, true, true);
        else DFDX_LAUNCH(false, false, true);
    } else {
        if (a_kc && b_kc) DFDX_LAUNCH(true, true, false);
        else if (a_kc && !b_kc) DFDX_LAUNCH(true, false, false);
        else if (!a_kc && b_kc) DFDX_LAUNCH(false, true, false);
        else DFDX_LAUNCH(false, false, false);
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_variant(int variant, const Params &p, int compute_units, bool a_kc, bool b_kc, hipStream_t s) {
    switch (variant) {
#define X(id, bm, bn, wm, wn) \
    case id: return launch_layout<T, bm, bn, wm, wn>(p, compute_units, a_kc, b_kc, s);
        DFDX_MFMA16_DMA_VARIANTS(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

struct OperandLayout {
    bool ok, kc;
    int64_t ld;
};
// `ragged`: rows that lie along memory may end off the grid of eight (GemmProblem::ragged: what follows them is readable)
inline OperandLayout classify(int64_t rows, int64_t kdim, int64_t row_stride, int64_t k_stride, bool ragged = false) {
    OperandLayout r{false, false, 0};
    if (ragged && row_stride == 1 && k_stride % 8 == 0 && k_stride >= ((rows + 7) & ~(int64_t)7)) {
        r.ok = true; r.kc = false; r.ld = k_stride;
    } else if (k_stride == 1 && kdim % 8 == 0 && (rows == 1 || (row_stride % 8 == 0 && row_stride >= kdim))) {
        r.ok = true; r.kc = true; r.ld = rows == 1 ? kdim : row_stride;
    } else if (row_stride == 1 && rows % 8 == 0 && (kdim == 1 || (k_stride % 8 == 0 && k_stride >= rows))) {
        r.ok = true; r.kc = false; r.ld = kdim == 1 ? rows : k_stride;
    }
    return r;
}

// The epilogue stores whole 16 B (8 B for the 16-column wave tile) pieces of C rows and nothing narrower; the instances for
// everything else are in gemm_mfma16_dma_ragged.hip.
inline bool c_on_grid(const GemmProblem &p, const Variant &v) {
    const int vecw = (v.bn / v.waves_n) % 32 == 0 ? 8 : 4;
    const int64_t ldc = p.m == 1 ? p.n : p.c_rs;
    const uintptr_t mask = (uintptr_t)vecw * 2 - 1;
    if (p.n % vecw || ldc % vecw || ((uintptr_t)p.c & mask) || p.c_b1 % vecw || p.c_b2 % vecw) return false;
    return !p.bias || !((uintptr_t)p.bias & mask);
}
// Does every row of C start on a whole 128-byte line?  Stores past the caches (stream16) are the faster ones where it does; lines that two
// workgroups write in part have to be put together in a cache: 16384 x 64 x 1032 f16 18.6 -> 13.8 us, 8192 x 256 x 2056 27.9 -> 21.1, 8192 x
// 1024 x 8200 144 -> 124, 2048 x 1024 x 50264 229 -> 210, 8192 x 1024 x 1032 27.3 and 27.7.
inline bool c_on_lines(const GemmProblem &p) {
    const int64_t ldc = p.m == 1 ? p.n : p.c_rs;
    return !(ldc % 64 || ((uintptr_t)p.c & 127u) || p.c_b1 % 64 || p.c_b2 % 64);
}

}  // namespace

bool mfma16dma_takes_any_k(int variant) { return is_ring(variant); }
int mfma16dma_variant_count() { return kNumVariants; }
const char *mfma16dma_variant_name(int v) { return (v >= 1 && v <= kNumVariants) ? kVariants[v - 1].name : "?"; }

// What the family asks of a product whatever the tile (a planner looks at it once); the operands' layouts are left in `la` and `lb`.
static bool takes(const GemmProblem &p, OperandLayout *la, OperandLayout *lb) {
    if (p.dtype != DT_F16 && p.dtype != DT_BF16) return false;
    if (p.m < 1 || p.n < 1 || p.k < 1) return false;
    if (p.m > (1 << 30) || p.n > (1 << 30) || p.k > (1 << 30)) return false;
    if (p.c_cs != 1 && p.n != 1) return false;
    if (p.n > 1 && p.m > 1 && p.c_rs < p.n) return false;
    *la = classify(p.m, p.k, p.a_rs, p.a_cs, p.ragged);
    *lb = classify(p.n, p.k, p.b_cs, p.b_rs, p.ragged);
    if (!la->ok || !lb->ok) return false;
    if (!aligned16(p.a) || !aligned16(p.b)) return false;
    if (p.batch_count() > 1) {
        if (p.a_b1 % 8 || p.a_b2 % 8 || p.b_b1 % 8 || p.b_b2 % 8) return false;
        if (!p.batches && (p.a_b1 < 0 || p.a_b2 < 0 || p.b_b1 < 0 || p.b_b2 < 0)) return false;
        if (p.bias_b1 % 8 || p.bias_b2 % 8) return false;
    }
    if (p.batch_count() >= (1ll << 31)) return false;
    if (p.last_apart && (p.batch_count() != 1 || p.k % BK)) return false;
    if (p.k * (p.reduce ? p.batch_count() : 1) >= (1ll << 31)) return false;
    return true;
}
static int64_t tile_count(const GemmProblem &p, const Variant &v) {
    return ((p.m + v.bm - 1) / v.bm) * ((p.n + v.bn - 1) / v.bn);
}
static bool takes_on(const GemmProblem &p, int variant, const OperandLayout &la, const OperandLayout &lb) {
    const Variant &v = kVariants[variant - 1];
    if (!is_ring(variant) && p.k % BK != 0) return false;
    if (la.ld * (la.kc ? v.bm : BK) >= (1ll << 30) || lb.ld * (lb.kc ? v.bn : BK) >= (1ll << 30)) return false;
    // (wave tiles of 96 columns store half lines: beside a C off the grid the others are ahead, and their instances have no odd rows)
    const int wave_columns = v.bn / v.waves_n;
    if (!is_ring(variant) && !c_on_grid(p, v) && !(p.ragged && wave_columns % 32 == 0 && wave_columns != 96)) return false;
    return tile_count(p, v) * (p.reduce ? 1 : p.batch_count()) < (1ll << 31);
}

bool mfma16dma_supported(const GemmProblem &p, int variant) {
    OperandLayout la, lb;
    return variant >= 1 && variant <= kNumVariants && takes(p, &la, &lb) && takes_on(p, variant, la, lb);
}

int mfma16dma_pick_variant(const GemmProblem &p, int compute_units) {
    // Largest tile that still gives every compute unit a workgroup; BN = 64 tiles only for narrow outputs.
    const int64_t nbatch = p.reduce ? 1 : p.batch_count();
    const int wide[] = {1, 2, 3}, narrow[] = {4, 5};
    if (p.n <= 64) {
        for (int v : narrow) {
            if (!mfma16dma_supported(p, v)) continue;
            const Variant &t = kVariants[v - 1];
            const int64_t blocks = ((p.m + t.bm - 1) / t.bm) * ((p.n + t.bn - 1) / t.bn) * nbatch;
            if (blocks >= compute_units || v == 5) return v;
        }
        return 0;
    }
    for (int v : wide) {
        if (!mfma16dma_supported(p, v)) continue;
        const Variant &t = kVariants[v - 1];
        const int64_t blocks = ((p.m + t.bm - 1) / t.bm) * ((p.n + t.bn - 1) / t.bn) * nbatch;
        if (blocks >= compute_units || v == 3) return v;
    }
    return 0;
}

// Cost model of the planner (seconds), fitted to timings of this kernel family on a 256-CU MI355X.
//   * a compute unit sustains rate1 / rate2 flop/s on a variant's k tiles when the chip is full; the 128-row tiles
//     only get there with two workgroups resident per compute unit, and lightly loaded chips clock higher;
//   * a work item also moves (operands mostly from L2) + (C tile) bytes at the compute unit's share of HBM;
//   * every work item pays a fixed hand-over cost, every launch a first-load latency and a last C tile;
//   * split-k adds the workspace round trip, which stays in the last-level cache while it is small.
namespace {
struct VariantModel {
    int per_cu;           // workgroups resident per compute unit (LDS and register limits)
    double rate1, rate2;  // flop/s of a compute unit with 1 / with >= 2 resident workgroups
};
constexpr VariantModel kModel[kNumVariants] = {
    {1, 5.50e12, 5.50e12},  // 256x256
    {1, 4.40e12, 4.40e12},  // 256x128
    {2, 3.00e12, 4.25e12},  // 128x128
    {1, 3.60e12, 3.60e12},  // 256x64
    {2, 2.20e12, 2.90e12},  // 128x64
    {}, {}, {}, {},         // (ring tiles)
    {1, 5.00e12, 5.00e12},  // 256x192
};
constexpr double kItemOverhead = 2.0e-6, kLaunchLatency = 2e-6, kCuBandwidth = 24e9, kOperandWeight = 0.32;
constexpr double kIdleBoost = 0.146, kWsBandwidthCached = 9.5e12, kWsBandwidthHbm = 6.1e12, kWsCached = 128e6;
constexpr double kSplitLaunch = 7e-6, kSplitPerPiece = 0.25e-6;  // 1024^3: 12.4 us unsplit, 15.9 / 18.0 us in 2 / 4 pieces
// That model ranks its own tiles and split counts; on products of a few microseconds it runs 1 - 2 us above the clock, and 8 us
// above it for a split plan.
constexpr double kAboveClock = 1.0e-6, kAboveClockSplit = 6.5e-6;

// The ring tiles: microseconds per k tile with 1 .. 3 workgroups on a compute unit, per work item, per launch.  Fitted to forced
// timings of 600 products of m, n = 64 .. 4096 and k = 17 .. 8192 in three layouts (standard deviation 6 %, split plans 10 %).
// They are taken only where every work item has a place at once: behind a first round the persistent tiles with their larger
// steps are ahead (1344 x 768 x 3072 f16: 1008 items of 64 x 64 16.9 us, the 256 x 128 tile 15.4; 3072 x 3072 x 128 14.6 and 9.3).
// Nor over more than 96 k tiles, where the larger tiles' fewer LDS reads have caught up (256 items of 128 x 128 x 4096 f16 36.7 us, the
// best of the persistent tiles 43.4; x 8192 75.7 and 75.9).
// kRingAcross is no line between two speeds: weight gradients over 4096 rows and more (both operands stored across k, whole k tiles) keep
// the split plans of the persistent tiles, so that those which carry a layer's bias gradient along (ksum) stay reached and tested at the
// sizes they were built for (test_gpu_linear.py names them); the ring takes 17.8 us for 23.7 at 1024 x 4096 x 1024 and 29.3 for 32.4 at 1024 x 8192 x
// 1024, and has not been measured beyond 8192 rows.
// Over the 600, launched again and again on operands that the last-level cache holds, the plan is 1.3 % from the fastest of all tiles and
// split counts; the plan without the ring was 19 % from it.  In a chain of launches the operands may come from memory: behind the launch that
// writes its first operand, 3152 x 3072 x 768 f16 takes 34 us on the 128 x 128 tile for an estimate of 25.
// 192 x 64 and 256 x 192 are there for the grids that the powers of two leave half empty (256 compute units, 150 tiles of 128 x 128 or 156 of 256 x
// 256): 3152 x 3072 x 768 f16 nt 26.8 -> 24.3 us, 2080 x 3968 x 1472 nn 36.1 -> 32.5, 512 x 4480 x 5440 tn 40.8 -> 37.2; 3152 x 768 x 3072 25.2 ->
// 20.0, 2432 x 1344 x 3712 38.0 -> 32.6, 2048 x 896 x 5864 31.3 -> 26.0.  Of 796 products 124 changed plans, to 1.10 times the speed (geometric
// mean); the largest loss was 11 % (3016 x 768 x 5696 tn, added to C).  192 x 64 is fitted like its neighbour, 7 % under the clock on a
// full chip, and 4 % above that fit: of 298 products that took it at the fit 17 had been faster by more than 3 % on another tile (most of
// them on 64 x 64 ones, at level estimates), 6 so, at the same speed in the mean.  What a split plan takes above its parts (`split`) grows
// with the tile: 2.1 - 3.1 us on 64 x 64, 3.9 on 128 x 64, 6.4 on 128 x 128 and 5.3 on 192 x 64 in the middle of 250 forced timings.
// `cold` is a k tile of a workgroup that has its compute unit to itself and walks kCold of them or more: on operands that the launch in
// front has written, which come from beyond the L2 caches, the two tiles that three stages have on their way do not cover what one takes.
// 128 x 64, 0.31 us on operands launched again and again, 0.53 in an encoder block's forward: its second product of 1752 x 3072 x 768 f16
// 27.7 us where 128 x 128 in three pieces takes 16.7 + 1.8 more in the launch behind, 2007 x 4096 x 1024 34.8 and 25.0 + 1.3.  One plan has to do
// for both (the block leaves the bits of its ops), so the figure lies between, just where that product changes tiles; on fewer k tiles it
// would send products to 128 x 64 in three pieces, which are slower (1833 x 2112 x 640 14.7 -> 18.9).
struct RingModel {
    int per_cu;
    double k_tile[4], item, launch, split, cold;
};
constexpr int64_t kRingChunk = 96, kRingAcross = 64, kCold = 48;
constexpr double kSecondRound = 2.0;  // see mfma16_ring_pair_plan (microseconds)
constexpr double kSecondLaunch = 3.5e-6, kLastRound = 0.6, kShortRound = 12e-6;  // see plan_tail
constexpr RingModel kRing[kNumVariants] = {
    {}, {}, {}, {}, {},                               // (persistent tiles)
    {2, {0.0, 0.187, 0.390, 0.0}, 2.75, 0.9, 2.6},    // 64 x 64, four stages
    {3, {0.0, 0.234, 0.394, 0.572}, 3.30, 0.2, 2.6},  // 64 x 64, three
    {2, {0.0, 0.305, 0.610, 0.0}, 4.10, 0.1, 2.6, 0.35},  // 128 x 64
    {1, {0.0, 0.414, 0.0, 0.0}, 4.80, 0.1, 5.8},      // 128 x 128
    {},                                               // (256 x 192)
    {1, {0.0, 0.363, 0.0, 0.0}, 5.20, 0.1, 5.2},      // 192 x 64
};
inline double ring_time(const RingModel &r, int cus, int64_t items, int64_t total, bool whole, int64_t chunk, bool a_kc, bool b_kc, int splits, double out_elems,
                        int64_t longest = kRingChunk) {
    if (items > (int64_t)cus * r.per_cu || chunk > longest || (!a_kc && !b_kc && whole && total >= kRingAcross)) return 1e300;
    const double layout = a_kc && b_kc ? 0.97 : !a_kc && !b_kc ? 1.1 : 1.0;
    const double k_tile = items <= cus && chunk >= kCold ? std::max(r.cold, r.k_tile[1]) : r.k_tile[(items + cus - 1) / cus];
    double us = r.launch + r.item + (double)chunk * k_tile * layout + out_elems * 2.0 / 8e6;
    if (splits > 1) us += r.split + 0.2 * splits + splits * out_elems * 4.0 / 9.5e6;
    return us * 1e-6;
}
}  // namespace

// The tiles of a product that has more of them than the chip has places are walked in rounds, and a last round of few tiles leaves
// the chip idle for as long as a full one takes (0.6 of it: what runs there has the clock and the caches to itself).  Where the ring
// tiles finish what is left over sooner, the product is cut behind the last full round, along its rows or its columns, into two
// launches; every 16-bit tile sums in the same order, the bits are the same.  Before, such products took smaller tiles throughout.
// f16, whole -> cut: 4224^3 177 -> 134 us, 4096 x 2048 x 4352 93 -> 66, 4608 x 1024 x 4096 51 -> 43, 4400 x 8192 x 4096 362 -> 257 (four
// k pieces before), 8192 x 1024 x 4352 83 -> 69; 50257 x 2048 x 1024 (both across k) 220 -> 200.
// Not for short rounds (16384 x 256 x 1100 25.7 us whole, 27.0 cut), nor for the tiles of which two share a compute unit, whose rounds
// have no sharp end; and an uncut plan within 5 % is taken, as the model knows no better (12800 x 3072 x 768: 256 x 256 tiles 73 us, 256
// x 128 cut 85).
namespace {
struct Tail {
    GemmCut cut;
    double gain = 0.0;  // seconds less than with a last round as long as a full one (what the model takes it for)
};
GemmProblem part_of(const GemmProblem &p, int64_t m0, int64_t m1, int64_t n0, int64_t n1) {
    GemmProblem q = p;
    const int64_t es = 2, c_off = (m0 * p.c_rs + n0 * p.c_cs) * es;
    q.m = m1 - m0;
    q.n = n1 - n0;
    q.ksum = nullptr;
    q.ksum_of = KSUM_NONE;
    q.cut = {};
    q.a = (const char *)p.a + m0 * p.a_rs * es;
    q.b = (const char *)p.b + n0 * p.b_cs * es;
    q.c = (char *)p.c + c_off;
    if (p.with) q.with = (const char *)p.with + c_off;
    if (p.bias) q.bias = (const char *)p.bias + (p.bias_mode == BIAS_PER_ROW ? m0 : n0) * es;
    return q;
}
Tail plan_tail(const GemmProblem &p, int variant, int compute_units) {
    Tail best;
    if (is_ring(variant) || kModel[variant - 1].per_cu > 1 || p.c_cs != 1 || (p.batch_count() != 1 && !p.reduce)) return best;
    const Variant &t = kVariants[variant - 1];
    const int cus = std::max(1, compute_units);
    const int64_t places = cus;
    const int64_t tm = (p.m + t.bm - 1) / t.bm, tn = (p.n + t.bn - 1) / t.bn, rounds = tm * tn / places;
    if (rounds < 1 || tm * tn % places == 0) return best;
    const int64_t steps = (p.k + BK - 1) / BK * (p.reduce ? p.batch_count() : 1);
    const bool a_kc = classify(p.m, p.k, p.a_rs, p.a_cs, p.ragged).kc, b_kc = classify(p.n, p.k, p.b_cs, p.b_rs, p.ragged).kc;
    const double round_seconds = (double)steps * (2.0 * t.bm * t.bn * BK) / kModel[variant - 1].rate1 + kItemOverhead;
    if (round_seconds < kShortRound) return best;
    double soonest = kLastRound * round_seconds;
    for (int along_n = 0; along_n < 2; along_n++) {
        const int64_t keep = rounds * places / (along_n ? tm : tn);  // whole rows (columns) of tiles in the full rounds
        if (keep < 1 || keep >= (along_n ? tn : tm)) continue;
        const int64_t cut = keep * (along_n ? t.bn : t.bm);
        const GemmProblem rest = along_n ? part_of(p, 0, p.m, cut, p.n) : part_of(p, cut, p.m, 0, p.n);
        for (int v = 1; v <= kNumVariants; v++) {
            if (!is_ring(v) || !mfma16dma_supported(rest, v) || (p.extra != EXTRA_NONE && !mfma16dma_extra_supported(rest, v, 1))) continue;
            const Variant &r = kVariants[v - 1];
            const int64_t items = ((rest.m + r.bm - 1) / r.bm) * ((rest.n + r.bn - 1) / r.bn);
            const double after = ring_time(kRing[v - 1], cus, items, 0, true, steps, a_kc, b_kc, 1, (double)rest.m * (double)rest.n, steps) +
                                 kSecondLaunch;
            if (after < soonest) {
                soonest = after;
                best = {{v, along_n ? 0 : cut, along_n ? cut : 0}, round_seconds - after};
            }
        }
    }
    return best;
}
}  // namespace

double mfma16dma_least_time() { return kItemOverhead + kLaunchLatency - kAboveClock; }

void mfma16dma_plan_split(const GemmProblem &p, int compute_units, int forced_variant, int forced_splits, int *variant,
                          int *splits, double *seconds, GemmCut *cut) {
    GemmCut best_cut;
    *variant = 0;
    *splits = 1;
    if (cut) *cut = {};
    if (seconds) *seconds = 1e300;
    OperandLayout la, lb;
    if (!takes(p, &la, &lb)) return;
    const int cus = std::max(1, compute_units);
    const int64_t nbatch = p.reduce ? 1 : p.batch_count();
    const bool may_split = (nbatch == 1 || p.batches > 0) && p.c_cs == 1;
    const int64_t total_iters = ((p.k + BK - 1) / BK) * (p.reduce ? p.batch_count() : 1);
    const bool a_kc = la.kc, b_kc = lb.kc;
    const double elem = 2.0, out_elems = (double)p.m * p.n * nbatch;
    double best = 1e300, best_ring = 1e300;
    int ring = 0, ring_splits = 1;
    // candidates 1..16, 20..32, 40..64 (filter gradients of convolutions: a handful of tiles, thousands of k steps), with their k steps
    struct Pieces {
        int splits;
        int64_t chunk;
    } pieces[32];
    int count = 0;
    {
        int forced_s = forced_splits > 0 ? (int)std::min<int64_t>(forced_splits, total_iters) : 0;
        while (forced_s > 1 && (forced_s - 1) * ((total_iters + forced_s - 1) / forced_s) >= total_iters) forced_s--;  // no empty split
        for (int s = forced_s ? forced_s : 1; s <= (forced_s ? forced_s : 64); s += (s < 16 ? 1 : s < 32 ? 4 : 8)) {
            if (s > 1 && (!may_split || (forced_splits == 0 && total_iters < 4 * (int64_t)s))) break;
            const int64_t chunk = (total_iters + s - 1) / s;
            if ((s - 1) * chunk >= total_iters) continue;  // an empty split
            pieces[count++] = {s, chunk};
        }
    }
    for (int v = 1; v <= kNumVariants; v++) {
        if (forced_variant > 0 && v != forced_variant) continue;
        if (!takes_on(p, v, la, lb)) continue;
        const Variant &t = kVariants[v - 1];
        const VariantModel &vm = kModel[v - 1];
        // narrow outputs take the BN = 64 tiles; wide ones may take the small 128 x 64 tile (more workgroups for a
        // problem of a few tiles), never the 256 x 64 one
        if (forced_variant == 0 && !is_ring(v) && (p.n <= 64 ? t.bn > 64 : (t.bn <= 64 && t.bm > 128))) continue;
        // (256 x 192: measured on operands and results in place)
        if (forced_variant == 0 && !is_ring(v) && t.bn == 192 && (p.last_apart || p.ragged)) continue;
        const int64_t tiles = tile_count(p, t) * nbatch;
        const double layout = (a_kc && b_kc) ? 1.0 : (!a_kc && !b_kc) ? 0.98 : 0.99;  // transposing LDS reads cost a little
        for (int i = 0; i < count; i++) {
            const int s = pieces[i].splits;
            const int64_t chunk = pieces[i].chunk, items = tiles * s;
            // (256 x 192 with no more partial sums than the entry point that allocates nothing has space for: the plans that it stands in for fit)
            if (!is_ring(v) && t.bn == 192 && s > 1 && forced_splits == 0 && mfma16dma_workspace_bytes(p, v, s) > (size_t)DFDX_ROCM_NOALLOC_SCRATCH_BYTES) break;
            if (is_ring(v)) {
                if (forced_variant == 0 && items > (int64_t)cus * kRing[v - 1].per_cu) break;
                const double time = ring_time(kRing[v - 1], cus, items, total_iters, p.k % BK == 0, chunk, a_kc, b_kc, s, out_elems);
                if (time < best_ring || (forced_variant == v && ring == 0)) {
                    best_ring = time;
                    ring = v;
                    ring_splits = s;
                }
                continue;
            }
            const int grid = (int)std::min<int64_t>(items, (int64_t)cus * vm.per_cu), conc = (grid + cus - 1) / cus;
            const int64_t items_per_wg = items == grid ? 1 : (items + grid - 1) / grid;
            const double active = (double)std::min<int64_t>(grid, cus) / cus;
            const double cu_rate = (conc >= 2 ? vm.rate2 : vm.rate1) * layout * (1.0 + kIdleBoost * (1.0 - active));
            const double t_mma = chunk * (2.0 * t.bm * t.bn * BK) / (cu_rate / conc);
            // (half lines, which the wave tiles of 96 columns store, leave a compute unit more slowly: 7640 x 64 x 9536 f16 nt 50 us, 256 x 256 tiles 36)
            const double out_bytes = (double)t.bm * t.bn * (s > 1 ? 4.0 : elem * (1 + p.accumulate) * (t.bn == 192 && !p.accumulate ? 1.5 : 1.0));
            const double t_mem = (kOperandWeight * (t.bm + t.bn) * BK * elem * chunk + out_bytes) / (kCuBandwidth / conc);
            double time = items_per_wg * (std::max(t_mma, t_mem) + kItemOverhead) + kLaunchLatency +
                          out_bytes / (kCuBandwidth / conc);
            if (s > 1) {
                const double ws = s * out_elems * 4.0;
                // second launch + the reduce kernel's chain of s dependent partial-tile reads, then the workspace round trip
                time += kSplitLaunch + kSplitPerPiece * s +
                        (ws + out_elems * elem * (1 + p.accumulate)) / (ws <= kWsCached ? kWsBandwidthCached : kWsBandwidthHbm);
            }
            Tail tail;
            if (s == 1 && forced_variant == 0)
                if (tail = plan_tail(p, v, cus); tail.cut.variant) time = 1.05 * (time - tail.gain);
            if (time < best) {
                best = time;
                best_cut = tail.cut;
                *variant = v;
                *splits = s;
            }
        }
    }
    if (best < 1e300) best -= *splits > 1 ? kAboveClockSplit : kAboveClock;
    // A large C behind a few k tiles is bound by its stores, which the persistent tiles overlap with the next item: the ring's estimate lacks
    // up to 1.2 us there, theirs is 0.9 too high (7040 x 64 x 512 f16 5.1 us and 6.5 for estimates of 6.2 and 5.7, 512 x 256 x 5248 6.7 and
    // 8.0; 30 such products 1.05 - 1.26 times as long; where C is added to the two are level, and below 2.2 million values the ring is ahead).
    const double stores = p.k <= 6 * BK && !p.accumulate && out_elems >= 2.2e6 ? 1.5e-6 : 0.0;
    if (ring && (best_ring + stores < best || *variant == 0)) {
        best = best_ring;
        best_cut = {};
        *variant = ring;
        *splits = ring_splits;
    }
    if (cut) *cut = best_cut;
    if (seconds) *seconds = best;
}

// layout of the split-k workspace: [splits][tiles_m * BM][tiles_n * BN] f32, then -- row sums of A asked for --
// [splits * (BM / 64) * 8][tiles_m * BM] f32
static void ws_layout(const GemmProblem &p, int variant, int64_t *ld, int64_t *split_stride, int64_t *ksum_stride = nullptr) {
    const Variant &v = kVariants[variant - 1];
    *ld = ((p.n + v.bn - 1) / v.bn) * v.bn;
    *split_stride = *ld * (((p.m + v.bm - 1) / v.bm) * v.bm);
    if (ksum_stride) *ksum_stride = ((p.m + v.bm - 1) / v.bm) * v.bm;
}
// Workspace slots of the row sums: one per split, sharing tile column and wave.
static int ksum_slots(int variant, int splits) { return is_ring(variant) ? splits : splits * (kVariants[variant - 1].bm / 64) * 8; }

size_t mfma16dma_workspace_bytes(const GemmProblem &p, int variant, int splits) {
    if (splits <= 1) return 0;
    int64_t ld, stride, ks;
    ws_layout(p, variant, &ld, &stride, &ks);
    const int64_t slots = p.ksum ? ksum_slots(variant, splits) : 0;
    return (size_t)(stride * splits + ks * slots) * (size_t)(p.reduce ? 1 : p.batch_count()) * sizeof(float);
}

// The sums of A's rows ride along only where A and B are both stored contraction-major (m- and n-contiguous: the
// weight gradient grad_out^T . x after the output transposition) and the contraction is split (the partial sums are
// combined by the reduce kernel that runs then anyway).
bool mfma16dma_ksum_supported(const GemmProblem &p, int variant, int splits) {
    if (!p.ksum || p.ksum_of != KSUM_OF_A || (splits <= 1 && !is_ring(variant)) || !mfma16dma_supported(p, variant)) return false;
    if (!p.reduce && p.batch_count() != 1 && !p.batches) return false;
    if ((uintptr_t)p.ksum & 1u) return false;
    const Variant &v = kVariants[variant - 1];
    if (!is_ring(variant) && (p.n + v.bn - 1) / v.bn < v.bm / 64) return false;  // too few tile columns to share a tile's pieces
    return !classify(p.m, p.k, p.a_rs, p.a_cs, p.ragged).kc && !classify(p.n, p.k, p.b_cs, p.b_rs, p.ragged).kc;
}

bool mfma16dma_extra_supported(const GemmProblem &p, int variant, int splits) {
    if ((p.accumulate != 0) != (p.extra == EXTRA_FROM) || (p.batch_count() != 1 && !p.reduce) || !mfma16dma_supported(p, variant)) return false;
    if (p.extra != EXTRA_RELU && (!p.with || !aligned16(p.with))) return false;
    if (p.cut.variant && !mfma16dma_extra_supported(part_of(p, p.cut.m, p.m, p.cut.n, p.n), p.cut.variant, 1)) return false;
    if (splits > 1 || is_ring(variant)) return true;  // (split: the reduce kernel applies it)
    const bool a_kc = classify(p.m, p.k, p.a_rs, p.a_cs, p.ragged).kc, b_kc = classify(p.n, p.k, p.b_cs, p.b_rs, p.ragged).kc;
    return a_kc && b_kc == (p.extra == EXTRA_RELU || p.extra == EXTRA_RESIDUAL);
}

static hipError_t ring_params(const GemmProblem &g, int variant, RingParams &p, bool *a_kc, bool *b_kc) {
    const Variant &v = kVariants[variant - 1];
    const OperandLayout la = classify(g.m, g.k, g.a_rs, g.a_cs, g.ragged);
    const OperandLayout lb = classify(g.n, g.k, g.b_cs, g.b_rs, g.ragged);
    *a_kc = la.kc;
    *b_kc = lb.kc;
    p.a = (const uint16_t *)g.a; p.b = (const uint16_t *)g.b; p.c = (uint16_t *)g.c; p.bias = (const uint16_t *)g.bias;
    p.with = (const uint16_t *)g.with; p.ksum = (uint16_t *)g.ksum;
    p.m = (int)g.m; p.n = (int)g.n; p.k = (int)g.k;
    p.lda = (int)la.ld; p.ldb = (int)lb.ld;
    p.ldc = g.m == 1 ? g.n : g.c_rs;
    p.a_b1 = g.a_b1; p.a_b2 = g.a_b2; p.b_b1 = g.b_b1; p.b_b2 = g.b_b2; p.c_b1 = g.c_b1; p.c_b2 = g.c_b2;
    p.bias_b1 = g.bias_b1; p.bias_b2 = g.bias_b2; p.ksum_b1 = g.ksum_b1; p.ksum_b2 = g.ksum_b2;
    p.nb2 = (int)g.nb2;
    const int nbatch = (int)g.batch_count();
    p.kbatches = g.reduce ? nbatch : 1;
    p.tiles_m = (int)((g.m + v.bm - 1) / v.bm);
    p.tiles_n = (int)((g.n + v.bn - 1) / v.bn);
    p.tiles_per_batch = p.tiles_m * p.tiles_n;
    const int outputs = g.reduce ? 1 : nbatch, total_iters = (p.k + BK - 1) / BK * p.kbatches;
    p.accumulate = g.accumulate; p.bias_mode = g.bias ? g.bias_mode : BIAS_NONE;
    p.extra = g.extra; p.ksum_accumulate = g.ksum_accumulate;
    p.whole = (int)(g.k / BK) - (g.last_apart ? 1 : 0); p.a_last = g.a_last; p.b_last = g.b_last;
    p.group_m = 4;
    p.splits = std::max(1, g.splits); p.chunk = total_iters; p.ws = p.ws_ksum = nullptr; p.ws_ld = p.ws_split_stride = 0; p.ws_ksum_stride = 0;
    if (g.ksum && !mfma16dma_ksum_supported(g, variant, g.splits)) return hipErrorInvalidValue;
    if (g.extra != EXTRA_NONE && !mfma16dma_extra_supported(g, variant, g.splits)) return hipErrorInvalidValue;
    if (p.splits > 1) {
        if (!g.workspace || (outputs != 1 && !g.batches)) return hipErrorInvalidValue;
        p.chunk = (total_iters + p.splits - 1) / p.splits;
        if ((int64_t)(p.splits - 1) * p.chunk >= total_iters) return hipErrorInvalidValue;
        p.ws = g.workspace;
        int64_t ks_stride = 0;
        ws_layout(g, variant, &p.ws_ld, &p.ws_split_stride, &ks_stride);
        p.ws_ksum = g.workspace + p.ws_split_stride * p.splits * outputs;
        p.ws_ksum_stride = (int)ks_stride;
    }
    p.items = p.tiles_per_batch * outputs * p.splits;
    return hipSuccess;
}

static hipError_t launch_ring(const GemmProblem &g, int variant, hipStream_t stream) {
    RingParams p;
    bool a_kc, b_kc;
    if (hipError_t e = ring_params(g, variant, p, &a_kc, &b_kc); e != hipSuccess) return e;
    const hipError_t e = launch_mfma16_ring(variant, g.dtype, p, a_kc, b_kc, stream);
    if (e != hipSuccess || p.splits <= 1) return e;
    return launch_splitk_reduce(g, p.ws_ld, p.ws_split_stride, stream, g.ksum ? p.ws_ksum : nullptr, p.ws_ksum_stride, ksum_slots(variant, p.splits));
}

// When the last of `longer` items of `t_longer`, which go first, and `shorter` ones of `t_shorter` ends, of more items than places and at
// most twice as many.
static double two_rounds(double longer, double shorter, double t_longer, double t_shorter, double places) {
    if (longer >= places) return longer > places ? 2.0 * t_longer : t_longer + t_shorter;
    const double free = places - longer;  // short items go there twice before a long one ends
    return shorter <= 2.0 * free ? std::max(t_longer, 2.0 * t_shorter) : t_longer + t_shorter;
}

// Work items of both products share the places on the chip; they are handed out as places fall free.  With one place a compute unit the rounds
// have a sharp end, and the average says too little: 39 x (448 x 80 . 80 x 448) bf16, 312 items, 17.4 us apart and 19.2 joined.
int mfma16_ring_pair_plan(const GemmProblem &p, const GemmProblem &q, int compute_units, double *seconds) {
    const int cus = std::max(1, compute_units);
    int tile = 0;
    *seconds = 1e300;
    for (int v = 1; v <= kNumVariants; v++) {
        if (!is_ring(v) || !mfma16dma_supported(p, v) || !mfma16dma_supported(q, v)) continue;
        const OperandLayout pa = classify(p.m, p.k, p.a_rs, p.a_cs, p.ragged), pb = classify(p.n, p.k, p.b_cs, p.b_rs, p.ragged);
        if (!pa.kc || classify(q.m, q.k, q.a_rs, q.a_cs, q.ragged).kc || classify(q.n, q.k, q.b_cs, q.b_rs, q.ragged).kc) return 0;
        if (q.ksum && !mfma16dma_ksum_supported(q, v, 1)) return 0;
        const Variant &t = kVariants[v - 1];
        // (not in 192 x 64 tiles: an estimate that ranks single products of theirs has 2048 x 768 . 768 x 768 and its weight gradient at less than
        // 14.9 us, the time of 64 x 64 tiles; they take 22.9)
        if (t.bm == 192) continue;
        const RingModel &r = kRing[v - 1];
        auto items = [&](const GemmProblem &g) {
            return (double)((g.m + t.bm - 1) / t.bm) * (double)((g.n + t.bn - 1) / t.bn) * (double)(g.reduce ? 1 : g.batch_count());
        };
        auto steps = [&](const GemmProblem &g) { return (double)((g.k + BK - 1) / BK) * (double)(g.reduce ? g.batch_count() : 1); };
        const double np = items(p), nq = items(q), places = (double)cus * r.per_cu;
        if (np + nq > 2.0 * places || std::max(steps(p), steps(q)) > kRingChunk) continue;
        const double k_tile = r.k_tile[(int)std::min((double)r.per_cu, std::ceil((np + nq) / cus))];
        const double tp = steps(p) * k_tile * (pb.kc ? 0.97 : 1.0) + r.item, tq = steps(q) * k_tile * 1.1 + r.item, longest = std::max(tp, tq);
        double us = np + nq <= places ? longest : std::max(longest, (np * tp + nq * tq) / places + 0.4 * longest);
        if (r.per_cu == 1 && np + nq > places) us = std::max(us, two_rounds(tp >= tq ? np : nq, tp >= tq ? nq : np, longest, std::min(tp, tq), places) + kSecondRound);
        us += r.launch + 2.0 * ((double)p.m * p.n * (p.reduce ? 1 : p.batch_count()) + (double)q.m * q.n * (q.reduce ? 1 : q.batch_count())) / 8e6;
        if (us * 1e-6 < *seconds) {
            *seconds = us * 1e-6;
            tile = v;
        }
    }
    return tile;
}

hipError_t launch_mfma16_ring_pair(const GemmProblem &p, const GemmProblem &q, int tile, hipStream_t stream) {
    if (!is_ring(tile) || p.dtype != q.dtype || !mfma16dma_supported(p, tile) || !mfma16dma_supported(q, tile)) return hipErrorInvalidValue;
    RingParams rp, rq;
    bool pa, pb, qa, qb;
    GemmProblem whole[2] = {p, q};
    whole[0].splits = whole[1].splits = 1;
    if (hipError_t e = ring_params(whole[0], tile, rp, &pa, &pb); e != hipSuccess) return e;
    if (hipError_t e = ring_params(whole[1], tile, rq, &qa, &qb); e != hipSuccess) return e;
    if (!pa || qa || qb) return hipErrorInvalidValue;
    return launch_mfma16_ring_two(tile, p.dtype, rp, rq, pb, stream);
}

hipError_t launch_mfma16dma(const GemmProblem &g, int variant, hipStream_t stream) {
    if (!mfma16dma_supported(g, variant)) return hipErrorInvalidValue;
    if (is_ring(variant)) return launch_ring(g, variant, stream);
    if (g.cut.variant) {
        const GemmProblem rest = part_of(g, g.cut.m, g.m, g.cut.n, g.n);
        if (g.splits > 1 || g.ksum || !is_ring(g.cut.variant) || !mfma16dma_supported(rest, g.cut.variant) ||
            (g.extra != EXTRA_NONE && !mfma16dma_extra_supported(rest, g.cut.variant, 1)))
            return hipErrorInvalidValue;
        const hipError_t e = launch_mfma16dma(part_of(g, 0, g.cut.m ? g.cut.m : g.m, 0, g.cut.n ? g.cut.n : g.n), variant, stream);
        return e != hipSuccess ? e : launch_ring(rest, g.cut.variant, stream);
    }
    const Variant &v = kVariants[variant - 1];
    const OperandLayout la = classify(g.m, g.k, g.a_rs, g.a_cs, g.ragged);
    const OperandLayout lb = classify(g.n, g.k, g.b_cs, g.b_rs, g.ragged);
    Params p;
    p.a = (const uint16_t *)g.a; p.b = (const uint16_t *)g.b; p.c = (uint16_t *)g.c; p.bias = (const uint16_t *)g.bias;
    p.m = (int)g.m; p.n = (int)g.n; p.k = (int)g.k;
    p.lda = (int)la.ld; p.ldb = (int)lb.ld;
    p.ldc = g.m == 1 ? g.n : g.c_rs;
    p.a_b1 = g.a_b1; p.a_b2 = g.a_b2; p.b_b1 = g.b_b1; p.b_b2 = g.b_b2; p.c_b1 = g.c_b1; p.c_b2 = g.c_b2;
    p.nb2 = (int)g.nb2;
    p.bias_b1 = g.bias_b1; p.bias_b2 = g.bias_b2;
    const int nbatch = (int)(g.batch_count());
    p.kbatches = g.reduce ? nbatch : 1;
    p.tiles_m = (int)((g.m + v.bm - 1) / v.bm);
    p.tiles_n = (int)((g.n + v.bn - 1) / v.bn);
    p.tiles_per_batch = p.tiles_m * p.tiles_n;
    p.total_blocks = p.tiles_per_batch * (g.reduce ? 1 : nbatch);
    p.accumulate = g.accumulate; p.bias_mode = g.bias ? g.bias_mode : BIAS_NONE;
    p.group_m = 4;
    const int total_iters = (p.k / BK) * p.kbatches;
    p.splits = 1; p.chunk = total_iters; p.ws = nullptr; p.ws_ld = 0; p.ws_split_stride = 0;
    p.ws_ksum = nullptr; p.ws_ksum_stride = 0;
    if (g.ksum && !mfma16dma_ksum_supported(g, variant, g.splits)) return hipErrorInvalidValue;
    if (g.splits > 1) {
        if (!g.workspace || (p.total_blocks != p.tiles_per_batch && !g.batches)) return hipErrorInvalidValue;
        p.splits = g.splits;
        p.chunk = (total_iters + g.splits - 1) / g.splits;
        if ((int64_t)(g.splits - 1) * p.chunk >= total_iters) return hipErrorInvalidValue;
        p.ws = g.workspace;
        int64_t ks_stride = 0;
        ws_layout(g, variant, &p.ws_ld, &p.ws_split_stride, &ks_stride);
        if (g.ksum) {
            p.ws_ksum = g.workspace + p.ws_split_stride * g.splits * (g.reduce ? 1 : nbatch);
            p.ws_ksum_stride = (int)ks_stride;
        }
        p.total_blocks *= g.splits;
    }
    p.steps = total_iters;
    if (g.last_apart && p.k == BK) {
        p.a += g.a_last;
        p.b += g.b_last;
    } else if (g.last_apart) {
        // a last k tile that lies apart is one more batch of the contraction, of one tile (a test of the kernel's own for it, once a tile,
        // cost products of short contractions 0.4 - 0.8 %)
        p.k -= BK;
        p.kbatches = p.nb2 = 2;
        p.a_b2 = (la.kc ? p.k : (int64_t)p.k * p.lda) + g.a_last;
        p.b_b2 = (lb.kc ? p.k : (int64_t)p.k * p.ldb) + g.b_last;
    }
    p.grid = 0;  // set per kernel instantiation at launch
    p.with = (const uint16_t *)g.with;
    if (g.extra != EXTRA_NONE && !mfma16dma_extra_supported(g, variant, g.splits)) return hipErrorInvalidValue;
    if (g.extra != EXTRA_NONE && g.splits <= 1) return launch_mfma16dma_extra(variant, g.dtype, g.extra, p, g.compute_units, stream);
    const bool through_caches = !c_on_lines(g) && !g.accumulate && g.extra == EXTRA_NONE && !g.ksum && (v.bn / v.waves_n) % 32 == 0;
    if (g.splits <= 1 && (through_caches || !c_on_grid(g, v))) return launch_mfma16dma_ragged(variant, g.dtype, p, g.compute_units, la.kc, lb.kc, stream);
    hipError_t e = (g.dtype == DT_F16) ? launch_variant<_Float16>(variant, p, g.compute_units, la.kc, lb.kc, stream)
                                       : launch_variant<__bf16>(variant, p, g.compute_units, la.kc, lb.kc, stream);
    if (e != hipSuccess || g.splits <= 1) return e;
    return launch_splitk_reduce(g, p.ws_ld, p.ws_split_stride, stream, p.ws_ksum, p.ws_ksum_stride, ksum_slots(variant, g.splits));
}

}  // namespace dfdx_rocm
