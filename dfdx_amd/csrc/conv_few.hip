// Convolutions of images with one or three channels: square filters of 3, 5 or 7 with half-size padding, stride 1 or 2,
// f16 / bf16, f32 sums.  The first layer of a network.
//
// What bounds it: HBM.  The output (or its gradient) is read or written once -- 103 MB for 64 images of 3 x 224 x 224 and 64
// filters of 7 x 7 at stride 2 -- and the products, 15 GFLOP a direction, are a few microseconds of matrix cores.  Through a patch
// matrix the same layer writes and reads 236 MB of patches three times and rounds the image gradient's 147 terms to the element
// type one by one.  Here the patch matrix exists in registers only: a band of the image (or of grad_out) is staged in LDS and every
// operand is read from there at the offset of its tap.  Each kernel is described where it stands.
//
// Padded slots of an operand are zero on BOTH sides, so that an infinite pixel reaches the outputs that read it and no others.
#include "conv_few.h"

#include <algorithm>
#include <type_traits>

#include "gemm_internal.h"

namespace dfdx_rocm {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T> struct Mma;
template <> struct Mma<_Float16> {
    static constexpr uint32_t EXP = 0x7c007c00u, EXP_ULP = 0x04000400u;
    static __device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)v); }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, h2));
    }
};
template <> struct Mma<__bf16> {
    static constexpr uint32_t EXP = 0x7f807f80u, EXP_ULP = 0x00800080u;
    static __device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint32_t v) { return __uint_as_float(v << 16); }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, b2));
    }
};
// bits 15 and 31: the half holds an infinity or a NaN
template <typename T> __device__ __forceinline__ uint32_t not_finite(uint32_t pair) { return ((pair & Mma<T>::EXP) + Mma<T>::EXP_ULP) & 0x80008000u; }
__device__ __forceinline__ uint32_t low_halves(uint32_t first, uint32_t second) { return __builtin_amdgcn_perm(second, first, 0x05040100u); }
__device__ __forceinline__ uint32_t high_halves(uint32_t first, uint32_t second) { return __builtin_amdgcn_perm(second, first, 0x07060302u); }

struct Params {
    const uint16_t *img, *filters, *go;
    uint16_t *out, *grad_img, *grad_filters;
    float *ws;
    int batch, chan_out, h_in, w_in, h_out, w_out;
    int band, bands, items;  // output rows per item, items per image, items in all
    int fresh;
};

// ---- forward -------------------------------------------------------------------------------------------------------
// out[64 channels][32 pixels] per wave and round, v_mfma_f32_32x32x16: the pixels are the product's rows, the filters its
// columns.  The contraction runs over (channel, filter row) with the filter's columns padded to eight slots: a lane's operand is
// ONE run of eight neighbouring image elements in LDS, starting at its window, and 3 x 7 such rows make 11 steps.  At stride 2
// the windows start on even elements when the run begins one element early (SHIFT), so that the run is whole words; at stride 1
// odd windows are shifted into place.  The filters stay in registers for all bands that a workgroup walks.  Neighbouring lanes read
// neighbouring words: no bank conflicts.
template <typename T, int C, int K, int S>
__global__ __launch_bounds__(256, 3) void conv_few_forward_kernel(const Params p) {
    constexpr int KK = K * K, ROWS = C * K, STEPS = (ROWS + 1) / 2, PAD = K / 2;
    constexpr int LEAD = S == 2 ? (PAD + 1) / 2 * 2 : PAD, SHIFT = LEAD - PAD;  // elements the run starts before the window's middle / its first tap
    constexpr int WORDS = (SHIFT + K + 1) / 2;                                  // words of a run that hold taps
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, h = lane / 32, l32 = lane % 32;
    const int o0 = blockIdx.y * 64, channels = min(64, p.chan_out - o0);
    const int in_max = (p.band - 1) * S + K, pitch = p.w_in + 16;
    for (int i = tid; i < channels * C * KK; i += 256) lds[i] = p.filters[(int64_t)o0 * C * KK + i];
    __syncthreads();
    u32x4 f[STEPS][2];
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
        for (int ob = 0; ob < 2; ob++) {
            const int row = 2 * s + h, o = ob * 32 + l32;
            const bool ok = row < ROWS && o < channels;
            const uint16_t *src = lds + (ok ? o * C * KK + row * K : 0);
#pragma unroll
            for (int w = 0; w < 4; w++) {
                uint32_t v = 0;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int k2 = 2 * w + e - SHIFT;
                    if (k2 >= 0 && k2 < K) v |= (uint32_t)(ok ? src[k2] : 0) << (16 * e);
                }
                f[s][ob][w] = v;
            }
        }
    int row_off[STEPS];  // element offset of the step's image row (per half of the wave)
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int r0 = 2 * s, r1 = 2 * s + 1 < ROWS ? 2 * s + 1 : 2 * s;
        row_off[s] = (h ? r1 / K * in_max + r1 % K : r0 / K * in_max + r0 % K) * pitch;
    }
    const int octs = p.w_in / 8;
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const int b = item / p.bands, first = item % p.bands * p.band, rows = min(p.band, p.h_out - first);
        const int in_rows = (rows - 1) * S + K, y0 = first * S - PAD, pixels = rows * p.w_out;
        __syncthreads();  // the last item's reads (or those of the filters) are done
        for (int u = tid; u < C * in_rows * (octs + 2); u += 256) {
            const int line = u / (octs + 2), oct = u - line * (octs + 2) - 1, c = line / in_rows, r = line - c * in_rows, y = y0 + r;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (oct >= 0 && oct < octs && y >= 0 && y < p.h_in)
                v = *(const u32x4 *)(p.img + ((int64_t)(b * C + c) * p.h_in + y) * p.w_in + oct * 8);
            *(u32x4 *)(lds + (c * in_max + r) * pitch + 8 + oct * 8) = v;
        }
        __syncthreads();
        for (int tile = wave; tile * 32 < pixels; tile += 4) {
            const int px = min(tile * 32 + l32, pixels - 1), oh = px / p.w_out, ow = px - oh * p.w_out;
            const int at = oh * S * pitch + 8 - LEAD + ow * S;
            f32x16 acc[2];
#pragma unroll
            for (int i = 0; i < 16; i++) acc[0][i] = acc[1][i] = 0.0f;
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                const int e = at + row_off[s];
                u32x4 a = {0u, 0u, 0u, 0u};
                if constexpr (S == 2) {
                    const uint32_t *q = (const uint32_t *)(lds + e);
#pragma unroll
                    for (int w = 0; w < WORDS; w++) a[w] = q[w];
                } else {
                    const uint32_t *q = (const uint32_t *)(lds + (e & ~1));
                    const uint32_t sh = (uint32_t)(e & 1) * 16u;
                    uint32_t d[WORDS + 1];
#pragma unroll
                    for (int w = 0; w <= WORDS; w++) d[w] = q[w];
#pragma unroll
                    for (int w = 0; w < WORDS; w++) a[w] = __builtin_amdgcn_alignbit(d[w + 1], d[w], sh);
                }
                if constexpr (SHIFT == 1) a[0] &= 0xffff0000u;
                if constexpr ((SHIFT + K) % 2 == 1) a[WORDS - 1] &= 0xffffu;
                if (2 * s + 1 >= ROWS) {
#pragma unroll
                    for (int w = 0; w < 4; w++) a[w] = h ? 0u : a[w];
                }
                acc[0] = Mma<T>::mfma32(a, f[s][0], acc[0]);
                acc[1] = Mma<T>::mfma32(a, f[s][1], acc[1]);
            }
            // Lane = channel l32, the accumulators hold pixels 8 (i / 4) + 4 h + i % 4.  The halves of the wave trade so that a lane
            // has eight neighbouring pixels, the 16-lane rows so that a store covers 64 bytes of each of 16 channels.
#pragma unroll
            for (int ob = 0; ob < 2; ob++) {
                u32x4 o[2];
#pragma unroll
                for (int m = 0; m < 2; m++)
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const uint32_t x = Mma<T>::pack2(acc[ob][8 * m + 2 * e], acc[ob][8 * m + 2 * e + 1]);
                        const uint32_t y = Mma<T>::pack2(acc[ob][8 * m + 4 + 2 * e], acc[ob][8 * m + 4 + 2 * e + 1]);
                        const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
                        o[m][e] = r[0];
                        o[m][2 + e] = r[1];
                    }
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const auto r = __builtin_amdgcn_permlane16_swap(o[0][e], o[1][e], false, false);
                    o[0][e] = r[0];
                    o[1][e] = r[1];
                }
                const int lr = lane / 16;  // after the trades: pixels 16 (lr & 1) + 8 (lr / 2) .. + 7 of channels lane % 16 and 16 + lane % 16
                const int at_px = tile * 32 + (lr & 1) * 16 + (lr >> 1) * 8;
                uint16_t *dst = p.out + ((int64_t)(b * p.chan_out + o0 + ob * 32 + lane % 16) * p.h_out + first) * p.w_out + at_px;
                if (at_px < pixels) {
                    if (ob * 32 + lane % 16 < channels) *(u32x4 *)dst = o[0];
                    if (ob * 32 + 16 + lane % 16 < channels) *(u32x4 *)(dst + (int64_t)16 * p.h_out * p.w_out) = o[1];
                }
            }
        }
    }
}

// ---- image gradient --------------------------------------------------------------------------------------------------
// In cells of 2 x 2 pixels: the 4 C pixels of a cell (all channels) are the 16 rows of v_mfma_f32_16x16x32, 16 neighbouring cells
// its columns, 32 output channels one step; every position of grad_out that any pixel of a cell reads -- WIN x WIN of them, 4 x 4
// for 7 x 7 filters at stride 2 -- is one product with its own filter matrix (zero where a pixel has no tap there).  grad_out is
// transposed on its way into LDS, [pixel][32 channels], so that a lane's operand is 16 bytes at any shift of the window.  All sums in
// f32, one rounding.  No single unit bounds it: LDS and the vector ALU are each busy a third of the time (74 us at the size above)
// and the phases between barriers -- transpose, products -- do not overlap inside a workgroup.  XORing slots and pieces of the LDS
// tile against bank conflicts of the stores measured level (73.7 us).
// Where a tile or the filters hold an infinity or a NaN, which those zeros would spread over its cell, the products are added position by
// position: 147 -> 211 us for the whole backward at the size above with one infinite filter value (18.3 ms with plain sums of all taps).
template <int C, int K, int S> struct GradImg {
    static constexpr int PAD = K / 2, Q = 2 / S;                                // positions of grad_out per cell
    static constexpr int WIN = S == 2 ? (K + 1) / 2 : K + 1, D0 = S == 2 ? -((K - 1 - PAD) / 2) : PAD - K + 1;  // window size, first offset
    static constexpr int CELLS = S == 2 ? 64 : 32, ROWS = S == 2 ? 8 : K == 3 ? 4 : 2;  // cells of a tile
    static constexpr int TILES = ROWS * CELLS / 16, PER_WAVE = TILES / 4;
    static constexpr int GO_ROWS = Q * (ROWS - 1) + WIN, GO_COLS = Q * (CELLS - 1) + WIN;
    static constexpr int UNITS = (GO_ROWS * ((GO_COLS + 7) / 8 + 1) * 4 + 255) / 256;  // per thread, see the kernel
    static constexpr int HALF = (GO_COLS + 1) / 2, LINE = Q == 2 ? 2 * HALF : GO_COLS;  // Q = 2: even positions, then odd ones
    static constexpr int F_BYTES = WIN * WIN * 1024;                            // filter matrices of 32 channels
    static constexpr int KEEP = 2 * F_BYTES + GO_ROWS * LINE * 64 <= 81920 ? 2 : 1;
    static constexpr int LDS = KEEP * F_BYTES + GO_ROWS * LINE * 64;
    static_assert(LDS <= 81920 && 32 * C * K * K * 2 <= GO_ROWS * LINE * 64, "two workgroups per compute unit");
};

template <typename T, int C, int K, int S>
__global__ __launch_bounds__(256, 2) void conv_few_grad_img_kernel(const Params p) {
    using G = GradImg<C, K, S>;
    constexpr int KK = K * K;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t *const go_lds = smem + G::KEEP * G::F_BYTES;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, l16 = lane % 16, lq = lane / 16;
    const int chunks = (p.chan_out + 31) / 32, cells_w = p.w_in / 2, groups_w = (cells_w + G::CELLS - 1) / G::CELLS;
    const int groups_h = ((p.h_in + 1) / 2 + G::ROWS - 1) / G::ROWS;
    const int64_t plane = (int64_t)p.h_out * p.w_out;
    struct Place {
        int b, cy0, cx0, row0, col0, oct0, octs;  // image, first cell, first position of grad_out in the tile, its pieces of eight
    };
    auto place = [&](int item) -> Place {
        Place t;
        t.b = item / (groups_w * groups_h);
        const int in_img = item - t.b * groups_w * groups_h;
        t.cy0 = in_img / groups_w * G::ROWS;
        t.cx0 = in_img % groups_w * G::CELLS;
        t.row0 = G::Q * t.cy0 + G::D0;
        t.col0 = G::Q * t.cx0 + G::D0;
        t.oct0 = (t.col0 >= 0 ? t.col0 : t.col0 - 7) / 8;
        t.octs = (t.col0 + G::GO_COLS - 1) / 8 - t.oct0 + 1;
        return t;
    };
    // A unit is 8 positions x 8 channels; positions outside grad_out and channels past the last are zeros.  The units of the next
    // 32 channels are loaded while the products of these run.
    u32x4 next[G::UNITS][8];
    auto fetch = [&](const Place &t, int o0) {
        int id = tid;
        asm volatile("" : "+v"(id));  // (what is formed of it is formed here, not kept in registers under the products)
#pragma unroll
        for (int n = 0; n < G::UNITS; n++) {
            const int u = n * 256 + id, g = u % 4, rest = u / 4, r = rest / t.octs, oct = t.oct0 + rest - r * t.octs, y = t.row0 + r;
            const bool ok = r < G::GO_ROWS && y >= 0 && y < p.h_out && oct >= 0 && oct * 8 < p.w_out;
            const uint16_t *src = p.go + ((int64_t)t.b * p.chan_out + o0 + g * 8) * plane + (int64_t)y * p.w_out + oct * 8;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                next[n][j] = u32x4{0u, 0u, 0u, 0u};
                if (ok && o0 + g * 8 + j < p.chan_out) next[n][j] = *(const u32x4 *)(src + j * plane);
            }
        }
    };
    bool bad_filters = false;
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const Place at = place(item);
        const int b = at.b, cy0 = at.cy0, cx0 = at.cx0;
        if (item == (int)blockIdx.x) fetch(at, 0);
        f32x4 acc[G::PER_WAVE];
#pragma unroll
        for (int t = 0; t < G::PER_WAVE; t++) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int ch = 0; ch < chunks; ch++) {
            uint8_t *const f_lds = smem + (ch % G::KEEP) * G::F_BYTES;
            const int o0 = ch * 32;
            __syncthreads();  // the last chunk's reads are done
            if (chunks > G::KEEP || item == (int)blockIdx.x) {
                uint16_t *raw = (uint16_t *)go_lds;
                uint32_t nf = 0;
                constexpr int PIECES = 32 * C * KK / 8;  // 16 bytes each, all of a thread's in flight: element by element the kernel took 88 us instead of 82
                const int have = min(32, p.chan_out - o0) * C * KK;
                const uint16_t *src = p.filters + (int64_t)o0 * C * KK;
                u32x4 piece[(PIECES + 255) / 256];
#pragma unroll
                for (int n = 0; n < (PIECES + 255) / 256; n++) {
                    const int i = (n * 256 + tid) * 8;
                    piece[n] = u32x4{0u, 0u, 0u, 0u};
                    if (i + 8 <= have) {
                        piece[n] = *(const u32x4_any *)(src + i);
                    } else {
#pragma unroll
                        for (int e = 0; e < 7; e++)
                            if (i + e < have) piece[n][e / 2] |= (uint32_t)src[i + e] << (e % 2 * 16);
                    }
                }
#pragma unroll
                for (int n = 0; n < (PIECES + 255) / 256; n++) {
#pragma unroll
                    for (int w = 0; w < 4; w++) nf |= not_finite<T>(piece[n][w]);
                    if (n * 256 + tid < PIECES) *(u32x4 *)(raw + (n * 256 + tid) * 8) = piece[n];
                }
                bad_filters |= __syncthreads_or(nf != 0) != 0;
                for (int e = tid; e < G::WIN * G::WIN * 256; e += 256) {  // words: [position][lane][channel pair]
                    const int pos = e / 256, ln = e / 4 % 64, m = ln % 16, c = m / 4, o = 8 * (ln / 16) + 2 * (e % 4);
                    const int k1 = m / 2 % 2 + G::PAD - S * (G::D0 + pos / G::WIN), k2 = m % 2 + G::PAD - S * (G::D0 + pos % G::WIN);
                    uint32_t v = 0;
                    if (c < C && k1 >= 0 && k1 < K && k2 >= 0 && k2 < K) {
                        const int tap = (c * K + k1) * K + k2;
                        v = raw[o * C * KK + tap] | (uint32_t)raw[(o + 1) * C * KK + tap] << 16;
                    }
                    ((uint32_t *)f_lds)[e] = v;
                }
                __syncthreads();
            }
            uint32_t nf = 0;
            int id = tid;
            asm volatile("" : "+v"(id));  // (as in fetch)
#pragma unroll
            for (int n = 0; n < G::UNITS; n++) {
                const int u = n * 256 + id, g = u % 4, rest = u / 4, r = rest / at.octs, oct = at.oct0 + rest - r * at.octs;
#pragma unroll
                for (int j = 0; j < 8; j++)
#pragma unroll
                    for (int w = 0; w < 4; w++) nf |= not_finite<T>(next[n][j][w]);
                if (r >= G::GO_ROWS) continue;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int s = oct * 8 + i - at.col0;
                    if (s < 0 || s >= G::GO_COLS) continue;
                    u32x4 q;
#pragma unroll
                    for (int w = 0; w < 4; w++)
                        q[w] = i % 2 ? high_halves(next[n][2 * w][i / 2], next[n][2 * w + 1][i / 2]) : low_halves(next[n][2 * w][i / 2], next[n][2 * w + 1][i / 2]);
                    const int slot = G::Q == 2 ? (s & 1) * G::HALF + (s >> 1) : s;
                    *(u32x4 *)(go_lds + (r * G::LINE + slot) * 64 + g * 16) = q;
                }
            }
            const bool masked = __syncthreads_or(nf != 0) != 0 || bad_filters;
            if (ch + 1 < chunks) fetch(at, o0 + 32);
            else if (item + (int)gridDim.x < p.items) fetch(place(item + gridDim.x), 0);
            // Fully unrolled with every address a constant away from one of the lane: tiles in different rows read the same operands
            // one filter row apart, and the compiler keeps them (LDS reads 2.5 -> 1.8 million, 82 -> 74 us at 7 x 7, stride 2).
            constexpr int TW = G::CELLS / 16;
            const int row = wave * G::PER_WAVE / TW, tile0 = wave * G::PER_WAVE % TW;
            const uint8_t *const go_at = go_lds + (G::Q * row * G::LINE + tile0 * 16 + l16) * 64 + lq * 16;
            if (__builtin_expect(!masked, 1)) {
#pragma unroll
                for (int u = 0; u < G::WIN; u++)
#pragma unroll
                    for (int v = 0; v < G::WIN; v++) {
                        const u32x4 f = *(const u32x4 *)(f_lds + ((u * G::WIN + v) * 64 + lane) * 16);
                        const int slot = G::Q == 2 ? (v & 1) * G::HALF + (v >> 1) : v;
#pragma unroll
                        for (int t = 0; t < G::PER_WAVE; t++)
                            acc[t] = Mma<T>::mfma16(f, *(const u32x4 *)(go_at + ((u + G::Q * (t / TW)) * G::LINE + slot + t % TW * 16) * 64), acc[t]);
                    }
            } else {
                // An infinity or a NaN in the tile: every position's product by itself, added where a pixel has a tap at a position of
                // grad_out, so that neither the zeros of the filter matrices nor those around grad_out meet it.
#pragma unroll 1
                for (int pos = 0; pos < G::WIN * G::WIN; pos++) {
                    const int u = pos / G::WIN, v = pos % G::WIN;
                    const u32x4 f = *(const u32x4 *)(f_lds + (pos * 64 + lane) * 16);
                    const int slot = G::Q == 2 ? (v & 1) * G::HALF + (v >> 1) : v;
                    const int k1 = G::PAD - S * (G::D0 + u), k2 = G::PAD - S * (G::D0 + v);  // taps of a cell's first pixel
                    int y0 = at.row0 + G::Q * row + u, x0 = at.col0 + G::Q * (tile0 * 16 + l16) + v;
                    asm volatile("" : "+v"(y0), "+v"(x0));  // (formed here, not kept: the registers are the other loop's)
#pragma unroll
                    for (int t = 0; t < G::PER_WAVE; t++) {
                        const f32x4 one = Mma<T>::mfma16(f, *(const u32x4 *)(go_at + ((u + G::Q * (t / TW)) * G::LINE + slot + t % TW * 16) * 64), f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                        const int y = y0 + G::Q * (t / TW), x = x0 + G::Q * 16 * (t % TW);
                        const bool inside = y >= 0 && y < p.h_out && x >= 0 && x < p.w_out;
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (inside && k1 + i / 2 >= 0 && k1 + i / 2 < K && k2 + i % 2 >= 0 && k2 + i % 2 < K) acc[t][i] += one[i];
                    }
                }
            }
        }
        // lane: channel lq of cell l16 of every tile, its four pixels in the accumulator
#pragma unroll
        for (int t = 0; t < G::PER_WAVE; t++) {
            const int tile = wave * G::PER_WAVE + t, cy = cy0 + tile / (G::CELLS / 16), cx = cx0 + tile % (G::CELLS / 16) * 16 + l16;
            if (lq >= C || cx >= cells_w) continue;
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const int y = 2 * cy + a;
                if (y >= p.h_in) continue;
                float v[2] = {acc[t][2 * a], acc[t][2 * a + 1]};
                uint32_t *dst = (uint32_t *)(p.grad_img + ((int64_t)(b * C + lq) * p.h_in + y) * p.w_in + 2 * cx);
                if (!p.fresh) {
                    const uint32_t old = *dst;
                    v[0] += Mma<T>::to_f32(old & 0xffffu);
                    v[1] += Mma<T>::to_f32(old >> 16);
                }
                *dst = Mma<T>::pack2(v[0], v[1]);
            }
        }
    }
}

constexpr int GO_UNITS = 14, IMG_UNITS = 6;  // 16-byte pieces per thread: the host chooses bands that fit

// ---- filter gradient -------------------------------------------------------------------------------------------------
// grad_filters[64 channels][taps] over the pixels, v_mfma_f32_32x32x16: grad_out's rows are the product's rows, the C K K taps its
// columns, 16 pixels one step; two waves share a block of 32 channels.  A band of grad_out lies in LDS as it does in memory; the image is split into even and odd columns
// there (stride 2), so that the eight pixels of a lane's tap are one run of elements, shifted into place where it starts on an odd
// one.  Every wave keeps the sums of its share of the steps in registers over all bands of its workgroup;
// they meet in LDS in wave order, and the workgroups' sums in a second kernel in theirs: the same bits on every run.
template <typename T, int C, int K, int S>
__global__ __launch_bounds__(256, 2) void conv_few_grad_filters_kernel(const Params p) {
    constexpr int KK = K * K, TAPS = C * KK, NB = (TAPS + 31) / 32, PAD = K / 2;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, h = lane / 32, l32 = lane % 32, ob = wave / 2;
    const int channels = p.chan_out;  // at most 64
    const int in_max = (p.band - 1) * S + K, plane_pitch = S == 2 ? p.w_in / 2 + 8 : p.w_in + 16, pitch = S * plane_pitch;
    const int go_pitch = p.band * p.w_out + 8, octs_row = p.w_out / 8, octs_line = p.w_in / 8 + 2;
    uint16_t *const go_lds = (uint16_t *)smem, *const img_lds = go_lds + 64 * go_pitch;
    f32x16 acc[NB];
    int base[NB];       // element offset of the lane's tap, window at pixel 0, on a word
    uint32_t shift[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int tap = min(nb * 32 + l32, TAPS - 1), c = tap / KK, k1 = tap / K % K, k2 = tap % K;
        const int x = k2 - PAD + 8, d = S == 2 ? x >> 1 : x;
        base[nb] = (c * in_max + k1) * pitch + (S == 2 ? (x & 1) * plane_pitch : 0) + (d & ~1);
        shift[nb] = (uint32_t)(d & 1) * 16u;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[nb][i] = 0.0f;
    }
    // The pieces of an item, GO of grad_out and IM of the image per thread, are loaded while the item before it is computed.
    struct Place {
        int b, first, rows, octs;
    };
    auto place = [&](int item) -> Place {
        Place t;
        t.b = item / p.bands;
        t.first = (item - t.b * p.bands) * p.band;
        t.rows = min(p.band, p.h_out - t.first);
        t.octs = t.rows * octs_row;
        return t;
    };
    u32x4 go_next[GO_UNITS], img_next[IMG_UNITS];
    auto fetch = [&](const Place &t) {
#pragma unroll
        for (int n = 0; n < GO_UNITS; n++) {
            const int u = n * 256 + tid, o = u / t.octs, oct = u - o * t.octs;
            if (o < channels) go_next[n] = *(const u32x4 *)(p.go + ((int64_t)(t.b * channels + o) * p.h_out + t.first) * p.w_out + oct * 8);
        }
        const int in_rows = (t.rows - 1) * S + K, y0 = t.first * S - PAD;
#pragma unroll
        for (int n = 0; n < IMG_UNITS; n++) {
            const int u = n * 256 + tid, line = u / octs_line, oct = u - line * octs_line - 1, c = line / in_rows, y = y0 + line - c * in_rows;
            img_next[n] = u32x4{0u, 0u, 0u, 0u};
            if (c < C && oct >= 0 && oct < octs_line - 2 && y >= 0 && y < p.h_in)
                img_next[n] = *(const u32x4 *)(p.img + ((int64_t)(t.b * C + c) * p.h_in + y) * p.w_in + oct * 8);
        }
    };
    if ((int)blockIdx.x < p.items) fetch(place(blockIdx.x));
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const Place at = place(item);
        const int in_rows = (at.rows - 1) * S + K, octs = at.octs;
        __syncthreads();  // the last item's reads are done
#pragma unroll
        for (int n = 0; n < GO_UNITS; n++) {
            const int u = n * 256 + tid, o = u / octs, oct = u - o * octs;
            if (o < channels) *(u32x4 *)(go_lds + o * go_pitch + oct * 8) = go_next[n];
        }
#pragma unroll
        for (int n = 0; n < IMG_UNITS; n++) {
            const int u = n * 256 + tid, line = u / octs_line, oct = u - line * octs_line - 1, c = line / in_rows;
            if (c >= C) continue;
            uint16_t *dst = img_lds + (c * in_max + line - c * in_rows) * pitch;
            const u32x4 v = img_next[n];
            if constexpr (S == 2) {
                *(u32x2 *)(dst + 4 + oct * 4) = u32x2{low_halves(v[0], v[1]), low_halves(v[2], v[3])};
                *(u32x2 *)(dst + plane_pitch + 4 + oct * 4) = u32x2{high_halves(v[0], v[1]), high_halves(v[2], v[3])};
            } else {
                *(u32x4 *)(dst + 8 + oct * 8) = v;
            }
        }
        __syncthreads();
        if (item + (int)gridDim.x < p.items) fetch(place(item + gridDim.x));
        for (int step = wave % 2; 2 * step < octs; step += 2) {
            const bool ok = 2 * step + h < octs;
            const int oct = ok ? 2 * step + h : octs - 1, oh = oct / octs_row, ow = (oct - oh * octs_row) * 8;
            u32x4 a = *(const u32x4 *)(go_lds + (ob * 32 + l32) * go_pitch + oct * 8);
#pragma unroll
            for (int w = 0; w < 4; w++) a[w] = ok ? a[w] : 0u;
            const int at_px = oh * S * pitch + ow;
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                const uint32_t *q = (const uint32_t *)(img_lds + base[nb] + at_px);
                uint32_t d[5];
#pragma unroll
                for (int w = 0; w < 5; w++) d[w] = q[w];
                u32x4 t;
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    t[w] = __builtin_amdgcn_alignbit(d[w + 1], d[w], shift[nb]);
                    t[w] = ok ? t[w] : 0u;
                }
                acc[nb] = Mma<T>::mfma32(a, t, acc[nb]);
            }
        }
    }
    // lane: tap 32 nb + l32, the accumulators hold channels 32 ob + 8 (i / 4) + 4 h + i % 4
    float *const sums = (float *)smem;  // [64][32 NB]
    for (int w = 0; w < 2; w++) {
        __syncthreads();
        if (wave % 2 == w) {
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float *s = sums + (ob * 32 + 8 * (i / 4) + 4 * h + i % 4) * (32 * NB) + nb * 32 + l32;
                    *s = (w ? *s : 0.0f) + acc[nb][i];
                }
        }
    }
    __syncthreads();
    float *ws = p.ws + (int64_t)blockIdx.x * 64 * TAPS;
    for (int i = tid; i < channels * TAPS; i += 256) ws[i] = sums[i / TAPS * (32 * NB) + i % TAPS];
}

// 32 sums per workgroup, the workgroups' shares in eight runs, in order.
template <typename T>
__global__ __launch_bounds__(256) void conv_few_grad_filters_add_kernel(const float *ws, int shares, int taps, int chan_out, uint16_t *grad_filters, int fresh) {
    __shared__ float part[8][32];
    const int lane = threadIdx.x % 32, run = threadIdx.x / 32, i = blockIdx.x * 32 + lane, n = chan_out * taps;
    const float *src = ws + min(i, n - 1);
    const int per = (shares + 7) / 8, s1 = min(shares, (run + 1) * per);
    float sum = 0.0f;
    int s = run * per;
    for (; s + 8 <= s1; s += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = src[(int64_t)(s + u) * 64 * taps];
#pragma unroll
        for (int u = 0; u < 8; u++) sum += v[u];
    }
    for (; s < s1; s++) sum += src[(int64_t)s * 64 * taps];
    part[run][lane] = sum;
    __syncthreads();
    if (run == 0 && i < n) {
#pragma unroll
        for (int r = 1; r < 8; r++) sum += part[r][lane];
        uint16_t *dst = grad_filters + i;
        *dst = (uint16_t)Mma<T>::pack2(fresh ? sum : Mma<T>::to_f32(*dst) + sum, 0.0f);
    }
}

// ---- host side -------------------------------------------------------------------------------------------------------
constexpr int kLds = 81920;  // two workgroups per compute unit

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }
bool shape_ok(const ConvFew &c) {
    return (c.dtype == DT_F16 || c.dtype == DT_BF16) && (c.kernel == 3 || c.kernel == 5 || c.kernel == 7) && (c.stride == 1 || c.stride == 2) &&
           (c.chan_in == 1 || c.chan_in == 3) && c.chan_out >= 1 && c.batch >= 1 && c.h_in >= 1 && c.w_in >= 16 && c.w_in <= 1024 &&
           c.w_in % (8 * c.stride) == 0 && c.w_out == c.w_in / c.stride && c.h_out == (c.h_in + c.stride - 1) / c.stride &&
           (int64_t)c.batch * c.chan_out < (1 << 30) && (int64_t)c.h_out * c.w_out < (1 << 28) && (int64_t)c.h_in * c.w_in < (1 << 28) &&
           (int64_t)c.batch * (c.h_out + 1) < (1 << 30) && aligned16(c.img);
}
size_t forward_lds(const ConvFew &c, int band) {
    const size_t rows = (size_t)c.chan_in * ((band - 1) * c.stride + c.kernel) * (c.w_in + 16) * 2;
    return std::max(rows, (size_t)64 * c.chan_in * c.kernel * c.kernel * 2);
}
// Output rows of a band: three workgroups fit a compute unit and walk the bands in rounds, a band costs its rows and about a
// row and a half for the image rows it shares with its neighbours and for its two barriers.
int forward_band(const ConvFew &c) {
    int best = 1;
    double least = 1e300;
    for (int band = 1; band <= 16 && band <= c.h_out && (band == 1 || forward_lds(c, band) <= (size_t)kLds * 2 / 3); band++) {
        const int64_t items = (int64_t)c.batch * ((c.h_out + band - 1) / band), rounds = (items + 3 * c.compute_units - 1) / (3 * c.compute_units);
        const double cost = (double)rounds * (band + 1.5);
        if (cost < least) {
            least = cost;
            best = band;
        }
    }
    return best;
}
size_t grad_filters_lds(const ConvFew &c, int band) {
    const size_t go = (size_t)64 * (band * c.w_out + 8) * 2, img = (size_t)c.chan_in * ((band - 1) * c.stride + c.kernel) * (c.w_in + 16) * 2;
    const size_t sums = (size_t)64 * ((c.chan_in * c.kernel * c.kernel + 31) / 32) * 32 * 4;
    return std::max(go + img, sums);
}
int grad_filters_band(const ConvFew &c) {
    auto fits = [&](int band) {
        return grad_filters_lds(c, band) <= (size_t)kLds && 64 * band * (c.w_out / 8) <= 256 * GO_UNITS &&
               c.chan_in * ((band - 1) * c.stride + c.kernel) * (c.w_in / 8 + 2) <= 256 * IMG_UNITS;
    };
    int band = 0;
    while (band < c.h_out && fits(band + 1)) band++;
    return band;
}
int grad_filters_shares(const ConvFew &c) {
    const int band = std::max(1, grad_filters_band(c));
    return (int)std::min<int64_t>((int64_t)c.batch * ((c.h_out + band - 1) / band), 2 * (int64_t)std::max(1, c.compute_units));
}
Params params_of(const ConvFew &c, int band) {
    Params p{};
    p.img = (const uint16_t *)c.img; p.filters = (const uint16_t *)c.filters; p.go = (const uint16_t *)c.grad_out;
    p.out = (uint16_t *)c.out; p.grad_img = (uint16_t *)c.grad_img; p.grad_filters = (uint16_t *)c.grad_filters;
    p.batch = c.batch; p.chan_out = c.chan_out; p.h_in = c.h_in; p.w_in = c.w_in; p.h_out = c.h_out; p.w_out = c.w_out;
    p.band = band; p.bands = (c.h_out + band - 1) / band; p.items = p.bands * c.batch;
    p.fresh = c.fresh_img;
    return p;
}
template <auto KERN> hipError_t allow_lds(size_t bytes) {
    static PerDevice known;
    std::atomic<int> &k = known.here();
    if ((size_t)k.load(std::memory_order_acquire) >= bytes) return hipSuccess;
    const hipError_t e = hipFuncSetAttribute((const void *)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e == hipSuccess) k.store(kLds, std::memory_order_release);
    return e;
}
template <typename T, int C, int K, int S> hipError_t forward_run(const ConvFew &c, hipStream_t stream) {
    const Params p = params_of(c, forward_band(c));
    const size_t lds = forward_lds(c, p.band);
    if (hipError_t e = allow_lds<conv_few_forward_kernel<T, C, K, S>>(lds)) return e;
    const dim3 grid((unsigned)std::min<int64_t>(p.items, 3 * (int64_t)c.compute_units), (unsigned)((c.chan_out + 63) / 64));
    conv_few_forward_kernel<T, C, K, S><<<grid, 256, lds, stream>>>(p);
    return hipGetLastError();
}
template <typename T, int C, int K, int S> hipError_t backward_run(const ConvFew &c, void *workspace, hipStream_t stream) {
    {
        using G = GradImg<C, K, S>;
        Params p = params_of(c, 1);
        const int64_t items = (int64_t)c.batch * ((c.w_in / 2 + G::CELLS - 1) / G::CELLS) * (((c.h_in + 1) / 2 + G::ROWS - 1) / G::ROWS);
        p.items = (int)items;
        if (hipError_t e = allow_lds<conv_few_grad_img_kernel<T, C, K, S>>(G::LDS)) return e;
        conv_few_grad_img_kernel<T, C, K, S><<<(unsigned)std::min<int64_t>(items, 2 * (int64_t)c.compute_units), 256, G::LDS, stream>>>(p);
        if (hipError_t e = hipGetLastError()) return e;
    }
    Params p = params_of(c, grad_filters_band(c));
    p.ws = (float *)workspace;
    const size_t lds = grad_filters_lds(c, p.band);
    if (hipError_t e = allow_lds<conv_few_grad_filters_kernel<T, C, K, S>>(lds)) return e;
    const int shares = grad_filters_shares(c), taps = C * K * K;
    conv_few_grad_filters_kernel<T, C, K, S><<<(unsigned)shares, 256, lds, stream>>>(p);
    if (hipError_t e = hipGetLastError()) return e;
    conv_few_grad_filters_add_kernel<T><<<(unsigned)((c.chan_out * taps + 31) / 32), 256, 0, stream>>>(p.ws, shares, taps, c.chan_out, p.grad_filters, c.fresh_filters);
    return hipGetLastError();
}

// f(element type, channels, kernel, stride as compile-time values) for the instance that `c` asks for
template <typename F> hipError_t with_instance(const ConvFew &c, F f) {
    using std::integral_constant;
    auto kernels = [&](auto t, auto ch, auto s) -> hipError_t {
        if (c.kernel == 3) return f(t, ch, integral_constant<int, 3>{}, s);
        if (c.kernel == 5) return f(t, ch, integral_constant<int, 5>{}, s);
        return f(t, ch, integral_constant<int, 7>{}, s);
    };
    auto strides = [&](auto t, auto ch) -> hipError_t {
        return c.stride == 2 ? kernels(t, ch, integral_constant<int, 2>{}) : kernels(t, ch, integral_constant<int, 1>{});
    };
    auto channels = [&](auto t) -> hipError_t {
        return c.chan_in == 3 ? strides(t, integral_constant<int, 3>{}) : strides(t, integral_constant<int, 1>{});
    };
    return c.dtype == DT_F16 ? channels((_Float16)0) : channels((__bf16)0.0f);
}

}  // namespace

bool conv_few_forward_supported(const ConvFew &c) {
    return shape_ok(c) && aligned16(c.out) && forward_lds(c, 1) <= (size_t)kLds * 2 / 3;
}

hipError_t launch_conv_few_forward(const ConvFew &c, hipStream_t stream) {
    if (!conv_few_forward_supported(c)) return hipErrorInvalidValue;
    return with_instance(c, [&](auto t, auto ch, auto k, auto s) -> hipError_t {
        return forward_run<decltype(t), decltype(ch)::value, decltype(k)::value, decltype(s)::value>(c, stream);
    });
}

// (7 x 7 filters at unit stride have 64 window positions, whose filter matrices leave no room for grad_out; with more than 64
// channels the filter matrices change with every 32 of them: 64 x 3 x 64 x 64 images, 256 filters of 3 x 3: 147 us against 117
// through the patch matrix)
bool conv_few_backward_supported(const ConvFew &c) {
    return shape_ok(c) && !(c.kernel == 7 && c.stride == 1) && c.chan_out <= 64 && aligned16(c.grad_out) && ((uintptr_t)c.grad_img & 3u) == 0 && grad_filters_band(c) > 0;
}
size_t conv_few_workspace_bytes(const ConvFew &c) {
    return (size_t)grad_filters_shares(c) * 64 * c.chan_in * c.kernel * c.kernel * sizeof(float);
}

hipError_t launch_conv_few_backward(const ConvFew &c, void *workspace, hipStream_t stream) {
    if (!conv_few_backward_supported(c)) return hipErrorInvalidValue;
    return with_instance(c, [&](auto t, auto ch, auto k, auto s) -> hipError_t {
        constexpr int K = decltype(k)::value, S = decltype(s)::value;
        if constexpr (K == 7 && S == 1) return hipErrorInvalidValue;
        else return backward_run<decltype(t), decltype(ch)::value, K, S>(c, workspace, stream);
    });
}

}  // namespace dfdx_rocm
