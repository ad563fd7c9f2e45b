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
typedef short v4i16 __attribute__((ext_vector_type(4)));
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
__device__ __align__(16) uint32_t few_zeros[4];  // what a lane beyond the image loads
#define DFDX_LDS __attribute__((address_space(3)))
#define DFDX_GLB __attribute__((address_space(1)))

// u / d and u % d for u = first, first + STEP, ..: one division, then sums (a division for every piece of a band was 28 of 103 thousand
// cycles of the filter gradient's kernel).
template <int STEP> struct Walk {
    int d, dq, dr, q, r;
    __device__ __forceinline__ Walk(int first, int d) : d(d), dq(STEP / d), dr(STEP % d), q(first / d), r(first - q * d) {}
    __device__ __forceinline__ void next() {
        q += dq;
        r += dr;
        if (r >= d) {
            r -= d;
            ++q;
        }
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
// neighbouring words: no bank conflicts.  The image rows come by LDS-DMA, on their way while the filters pass through LDS in pieces of 16
// bytes: with the rows through registers and the filters element by element a workgroup's start took a third of the launch (64 x 3 x 224 x 224,
// 64 filters of 7 x 7 at stride 2: 40.2 -> 32.1 us; filters from memory straight into the lanes' operands, a line for each: 42.4).
template <typename T, int C, int K, int S>
__global__ __launch_bounds__(256, 3) void conv_few_forward_kernel(const Params p) {
    constexpr int KK = K * K, ROWS = C * K, STEPS = (ROWS + 1) / 2, PAD = K / 2;
    constexpr int LEAD = S == 2 ? (PAD + 1) / 2 * 2 : PAD, SHIFT = LEAD - PAD;  // elements the run starts before the window's middle / its first tap
    constexpr int WORDS = (SHIFT + K + 1) / 2;                                  // words of a run that hold taps
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), h = lane / 32, l32 = lane % 32;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(DFDX_LDS const uint16_t *)lds;
    const int o0 = blockIdx.y * 64, channels = min(64, p.chan_out - o0);
    const int in_max = (p.band - 1) * S + K, pitch = p.w_in + 16;
    const int octs = p.w_in / 8, units = C * in_max * (octs + 2);
    // The image rows of an item, zeros around them, straight into LDS: a row there is octs + 2 pieces of 16 bytes, one behind the other.
    auto request = [&](int item) {
        const int b = item / p.bands, y0 = item % p.bands * p.band * S - PAD;
        const uint16_t *const img = p.img + (int64_t)b * C * p.h_in * p.w_in;
        Walk<256> at(tid, octs + 2);
        for (int i = wave * 64; i < units; i += 256, at.next()) {  // (the last instruction's lanes behind the rows fill the allocation's last KB)
            const int c = at.q >= in_max ? at.q >= 2 * in_max ? 2 : 1 : 0, y = y0 + at.q - c * in_max, oct = at.r - 1;
            const void *from = few_zeros;
            if (at.q < C * in_max && oct >= 0 && oct < octs && y >= 0 && y < p.h_in) from = img + ((int64_t)c * p.h_in + y) * p.w_in + oct * 8;
            __builtin_amdgcn_global_load_lds((const DFDX_GLB void *)from, (DFDX_LDS void *)(uintptr_t)(lds_base + (uint32_t)i * 16u), 16, 0, 0);
        }
    };
    if ((int)blockIdx.x < p.items) request(blockIdx.x);
    // The filters pass through LDS behind the rows, 32 at a time.  A lane's row of taps lies in four words there (five where it starts on the
    // upper half of one).
    constexpr int HALF = 32 * C * KK, PIECES = (HALF / 8 + 255) / 256;
    uint32_t *const raw = (uint32_t *)(lds + (units + 63) / 64 * 512);
    u32x4 f[STEPS][2], piece[2][PIECES];
#pragma unroll
    for (int ob = 0; ob < 2; ob++)
#pragma unroll
        for (int n = 0; n < PIECES; n++) {
            const int i = (n * 256 + tid) * 8, have = (channels - ob * 32) * C * KK;
            const uint16_t *src = p.filters + (int64_t)(o0 + ob * 32) * C * KK + i;
            piece[ob][n] = u32x4{0u, 0u, 0u, 0u};
            if (i + 8 <= min(have, HALF)) {
                piece[ob][n] = *(const u32x4_any *)src;
            } else {
#pragma unroll
                for (int e = 0; e < 7; e++)
                    if (i + e < min(have, HALF)) piece[ob][n][e / 2] |= (uint32_t)src[e] << (e % 2 * 16);
            }
        }
#pragma unroll
    for (int ob = 0; ob < 2; ob++) {
        if (ob) __syncthreads();  // the first half's reads are done
#pragma unroll
        for (int n = 0; n < PIECES; n++)
            if (n * 256 + tid < HALF / 8) *(u32x4 *)(raw + (n * 256 + tid) * 4) = piece[ob][n];
        __syncthreads();
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            const int row = min(2 * s + h, ROWS - 1), e = l32 * C * KK + row * K;
            const bool ok = 2 * s + h < ROWS, odd = e & 1;
            uint32_t d[5];
#pragma unroll
            for (int w = 0; w < 5; w++) d[w] = raw[e / 2 + w];
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const int lo = 2 * w - SHIFT, hi = lo + 1;  // taps of the two slots
                const uint32_t even_word = SHIFT == 0 ? d[w] : w == 0 ? d[0] << 16 : __builtin_amdgcn_alignbit(d[w], d[w - 1], 16u);
                const uint32_t odd_word = SHIFT == 0 ? __builtin_amdgcn_alignbit(d[w + 1], d[w], 16u) : d[w];
                f[s][ob][w] = ok ? (odd ? odd_word : even_word) & ((lo >= 0 && lo < K ? 0xffffu : 0u) | (hi >= 0 && hi < K ? 0xffff0000u : 0u)) : 0u;
            }
        }
    }
    int row_off[STEPS];  // element offset of the step's image row (per half of the wave)
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int r0 = 2 * s, r1 = 2 * s + 1 < ROWS ? 2 * s + 1 : 2 * s;
        row_off[s] = (h ? r1 / K * in_max + r1 % K : r0 / K * in_max + r0 % K) * pitch;
    }
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const int b = item / p.bands, first = item % p.bands * p.band, rows = min(p.band, p.h_out - first), pixels = rows * p.w_out;
        if (item != (int)blockIdx.x) {
            __syncthreads();  // the last item's reads are done
            request(item);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's requests are in LDS
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

// ---- image gradient: unit stride, and rows too long for the kernel behind this one ----------------------------------------
// In cells of 2 x 2 pixels: the 4 C pixels of a cell (all channels) are the 16 rows of v_mfma_f32_16x16x32, 16 neighbouring cells
// its columns, 32 output channels one step; every position of grad_out that any pixel of a cell reads -- WIN x WIN of them, 4 x 4
// for 7 x 7 filters at stride 2 -- is one product with its own filter matrix (zero where a pixel has no tap there).  grad_out is
// transposed on its way into LDS, [pixel][32 channels], so that a lane's operand is 16 bytes at any shift of the window.  All sums in
// f32, one rounding.  No single unit bounds it: LDS and the vector ALU are each busy a third of the time (70 us for 7 x 7 filters at the size
// above, which the kernel behind it takes now) and the phases between barriers -- transpose, products -- do not overlap inside a workgroup.  XORing slots and pieces of the LDS
// tile against bank conflicts of the stores measured level (73.7 us).
// Where a tile or the filters hold an infinity or a NaN, which those zeros would spread over its cell, the products are added position by
// position: twice the kernel's time (18.3 ms instead of 147 us for the whole backward at the size above with plain sums of all taps).
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

// ---- image gradient at stride 2, rows of up to 112 positions ------------------------------------------------------------------
// The same cells in another order: a wave owns one row of cells and sums, for every column offset v of the window apart,
//     S_v[n] = sum over the window's rows u and the channels of F[u, v] . grad_out[.][row + u][n]        n: the columns of grad_out
// in its registers (T tiles of 16 columns, WIN of them); a cell's result is the sum of S_v[its column + v], formed once, at the end, from
// neighbouring lanes.  The operand of a row and tile then serves all v and lies on whole tiles: grad_out goes into LDS as it is in memory, by
// LDS-DMA, 16 channels of the next rows under the products of these, and is read by the transposing reads; a step of the contraction is 16
// channels of two window rows.  Against the kernel above, 64 x 3 x 224 x 224, 64 filters of 7 x 7: 69.5 -> 49.7 us (56 with 32 channels of one
// window row a step and one stage; a word of every line of the next chunk loaded ahead, to have it in the XCD's cache: 63).  The vector ALU is
// what is left: the requests' addresses and the sums of the S_v (61 us before the former were formed once a wave, the latter once an item).
//   LDS, grad_out [2 stages][row][16 channels][TW tiles of 16 columns]: tile t of channel ch in slot t ^ spread(ch), which puts the channels
//   that a transposing read touches at once on different banks;
//   LDS, filters [16 channels][pair of window rows][v][lane row][4 C rows][8 channels]: rows of the product that no pixel has are not kept (their
//   lanes repeat others).
// The zeros of the filter matrices spread an infinity or a NaN of grad_out, or of the filters, over a cell: results that are not finite, and all
// of them where a filter is not, are formed position by position, added where a pixel has a tap at a position of grad_out (the whole backward
// at the size above with one infinite filter value: 160 us for 105).
template <int C, int K, int T> struct GradRows {
    static constexpr int PAD = K / 2, WIN = (K + 1) / 2, PAIRS = (WIN + 1) / 2, D0 = -((K - 1 - PAD) / 2), ROWS = 4, GO_ROWS = ROWS + 2 * PAIRS - 1;
    static constexpr int TW = T > 4 ? 8 : 4, ROW_BYTES = 16 * TW * 32, STAGE = GO_ROWS * ROW_BYTES, F_CHUNK = PAIRS * WIN * 4 * 4 * C * 16;
    static constexpr int REQUESTS = (STAGE / 1024 + 3) / 4;                    // of a wave
    static constexpr int VOTES = T < TW ? T * 32 : 2 * STAGE + 4 * F_CHUNK;    // a word of each wave: in a slot that no tile has (either stage's), or behind
    static constexpr int LDS = 2 * STAGE + 4 * F_CHUNK + (T < TW ? 0 : 16);
    static_assert(T <= TW && LDS <= 81920 && 64 * C * K * K * 2 + 16 <= 2 * STAGE && ROW_BYTES % 1024 == 0, "two workgroups per compute unit");
    static __device__ __forceinline__ int spread(int ch) {
        return TW == 8 ? (ch & 3) | (ch >> 3 & 1) << 2 : (ch >> 1 & 1) | (ch >> 3 & 1) << 1;
    }
};
// x of the lane BY places to the right in a row of 16 columns that goes on in `after` (BY < 0: to the left, in `before`)
template <int BY> __device__ __forceinline__ float neighbour(float before, float x, float after) {
    if constexpr (BY == 0) return x;
    constexpr int N = BY > 0 ? BY : -BY;
    constexpr int SHIFT = BY > 0 ? 0x100 + N : 0x110 + N, ROTATE = 0x120 + (BY > 0 ? 16 - N : N);  // row_shl / row_shr, row_ror
    const int rest = __builtin_amdgcn_update_dpp(0, __float_as_int(BY > 0 ? after : before), ROTATE, 0xF, 0xF, false);
    return __int_as_float(__builtin_amdgcn_update_dpp(rest, __float_as_int(x), SHIFT, 0xF, 0xF, false));
}

// Transposing reads of N tiles at byte offset OFF, complete when they return (issued from asm: the compiler would wait for every LDS-DMA load in
// front of them).
template <int OFF> __device__ __forceinline__ void read_columns(const uint32_t (&lo)[4], const uint32_t (&hi)[4], u32x2 (&l)[4], u32x2 (&h)[4]) {
    asm volatile("ds_read_b64_tr_b16 %0, %8 offset:%16\n\tds_read_b64_tr_b16 %1, %9 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %2, %10 offset:%16\n\tds_read_b64_tr_b16 %3, %11 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %4, %12 offset:%16\n\tds_read_b64_tr_b16 %5, %13 offset:%16\n\t"
                 "ds_read_b64_tr_b16 %6, %14 offset:%16\n\tds_read_b64_tr_b16 %7, %15 offset:%16\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(l[0]), "=&v"(h[0]), "=&v"(l[1]), "=&v"(h[1]), "=&v"(l[2]), "=&v"(h[2]), "=&v"(l[3]), "=&v"(h[3])
                 : "v"(lo[0]), "v"(hi[0]), "v"(lo[1]), "v"(hi[1]), "v"(lo[2]), "v"(hi[2]), "v"(lo[3]), "v"(hi[3]), "i"(OFF)
                 : "memory");
}

template <typename T_, int C, int K, int T>
__global__ __launch_bounds__(256, 2) void conv_few_grad_img_rows_kernel(const Params p) {
    using G = GradRows<C, K, T>;
    constexpr int KK = K * K, WIN = G::WIN;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    uint8_t *const f_lds = smem + 2 * G::STAGE;
    const uint32_t go_base = (uint32_t)(uintptr_t)(DFDX_LDS const uint8_t *)smem;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), l16 = lane % 16, lq = lane / 16;
    const int chunks = (p.chan_out + 15) / 16, groups = (p.h_out + G::ROWS - 1) / G::ROWS;
    const int64_t plane = (int64_t)p.h_out * p.w_out;

    bool bad_filters;
    {   // the filter matrices, by way of the filters as they lie in memory
        uint16_t *const raw = (uint16_t *)smem;
        const int have = p.chan_out * C * KK;
        uint32_t nf = 0;
        for (int i = tid * 8; i < have; i += 2048) {
            u32x4 piece = {0u, 0u, 0u, 0u};
            if (i + 8 <= have) {
                piece = *(const u32x4_any *)(p.filters + i);
            } else {
#pragma unroll
                for (int e = 0; e < 7; e++)
                    if (i + e < have) piece[e / 2] |= (uint32_t)p.filters[i + e] << (e % 2 * 16);
            }
            *(u32x4 *)(raw + i) = piece;  // (the stages are larger than the filters and their last piece)
#pragma unroll
            for (int w = 0; w < 4; w++) nf |= not_finite<T_>(piece[w]);
        }
        __syncthreads();
        if (tid < 64 * C) {  // a word of every matrix
            const int w = tid % 4, m = tid / 4 % (4 * C), q = tid / (16 * C), o = 8 * (q % 2) + 2 * w;
            const int a = m / 2 % 2 + G::PAD - 2 * (G::D0 + q / 2), c = m % 2 + G::PAD - 2 * G::D0;  // its tap at the first window row of a pair and v = 0
            uint32_t *to = (uint32_t *)f_lds + tid;
            for (int ch = 0; ch < chunks; ch++) {
                const uint16_t *const from = raw + ((ch * 16 + o) * C + m / 4) * KK;
                const bool one = ch * 16 + o < p.chan_out, two = ch * 16 + o + 1 < p.chan_out;
#pragma unroll
                for (int at = 0; at < G::PAIRS * WIN; at++, to += 64 * C) {
                    const int k1 = a - 4 * (at / WIN), k2 = c - 2 * (at % WIN);
                    const bool tap = k1 >= 0 && k1 < K && k2 >= 0 && k2 < K;
                    uint32_t pair = 0;
                    if (tap && one) pair = from[k1 * K + k2];
                    if (tap && two) pair |= (uint32_t)from[C * KK + k1 * K + k2] << 16;
                    *to = pair;
                }
            }
        }
        __syncthreads();
        uint32_t *const votes = (uint32_t *)smem;
        const bool bad = __any(nf != 0);
        if (lane == 0) votes[wave] = bad;
        __syncthreads();
        bad_filters = (votes[0] | votes[1] | votes[2] | votes[3]) != 0;
        __syncthreads();
    }
    // A wave instruction fills 1 KB: 4 (TW = 8) or 8 channels of a row, the same ones in every row for a wave.
    constexpr int CH = 1024 / (G::TW * 32), PER_ROW = 16 / CH;
    static_assert(4 % PER_ROW == 0, "a wave's channels");
    const int my_ch = wave % PER_ROW * CH + lane / (G::TW * 2), my_col = ((lane % (G::TW * 2) / 2) ^ G::spread(my_ch)) * 16 + lane % 2 * 8;
    const int64_t my_place = my_ch * plane + my_col;
    auto request = [&](int item, int ch, int stage) {
        const int b = item / groups, row0 = item % groups * G::ROWS + G::D0;
        const uint16_t *const from0 = p.go + ((int64_t)b * p.chan_out + ch * 16) * plane;
        const bool mine = my_col < p.w_out && ch * 16 + my_ch < p.chan_out;
#pragma unroll
        for (int j = 0; j < G::REQUESTS; j++) {
            const int i = min(j * 4 + wave, G::STAGE / 1024 - 4 + wave);  // (as many for every wave: the last one twice)
            const int r = row0 + i / PER_ROW;
            const void *from = from0 + (int64_t)r * p.w_out + my_place;
            if (!mine || r < 0 || r >= p.h_out) from = few_zeros;
            __builtin_amdgcn_global_load_lds((const DFDX_GLB void *)from, (DFDX_LDS void *)(uintptr_t)(go_base + (uint32_t)(stage * G::STAGE + i * 1024)), 16, 0, 0);
        }
    };
    // the lane's share of a transposing read: four columns of channel 8 (lq % 2) + l16 / 4, and of the one four behind, in the wave's row or the next
    const int ch0 = 8 * (lq % 2) + l16 / 4;
    uint32_t lo_at[8], hi_at[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const uint32_t row = go_base + (uint32_t)((wave + lq / 2) * G::ROW_BYTES + l16 % 4 * 8);
        lo_at[t] = row + (uint32_t)(ch0 * G::TW * 32 + ((min(t, T - 1) ^ G::spread(ch0)) * 32));
        hi_at[t] = row + (uint32_t)((ch0 + 4) * G::TW * 32 + ((min(t, T - 1) ^ G::spread(ch0 + 4)) * 32));
    }
    auto column_operands = [&](int stage, auto pair_tag, u32x4(&g)[T]) {
        constexpr int OFF = decltype(pair_tag)::value * 2 * G::ROW_BYTES;
#pragma unroll
        for (int t0 = 0; t0 < T; t0 += 4) {
            uint32_t lo[4], hi[4];
            u32x2 l[4], h[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                lo[t] = lo_at[t0 + t] + (uint32_t)(stage * G::STAGE);
                hi[t] = hi_at[t0 + t] + (uint32_t)(stage * G::STAGE);
            }
            read_columns<OFF>(lo, hi, l, h);
#pragma unroll
            for (int t = 0; t < 4; t++)
                if (t0 + t < T) g[t0 + t] = u32x4{l[t][0], l[t][1], h[t][0], h[t][1]};
        }
    };
    const uint8_t *const f_lane = f_lds + (lq * 4 * C + l16 % (4 * C)) * 16;
    auto filter_operand = [&](int ch, int at) -> u32x4 { return *(const u32x4 *)(f_lane + ch * G::F_CHUNK + at * (4 * 4 * C * 16)); };

    f32x4 sum[T][WIN];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int v = 0; v < WIN; v++) sum[t][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    auto result = [&](int t, int i) -> float {  // of pixel i of the lane's cell in tile t
        auto column = [&](auto v_tag) -> float {
            constexpr int V = decltype(v_tag)::value;
            if constexpr (V < WIN) return neighbour<G::D0 + V>(t > 0 ? sum[t > 0 ? t - 1 : 0][V][i] : 0.0f, sum[t][V][i], t + 1 < T ? sum[t + 1 < T ? t + 1 : t][V][i] : 0.0f);
            else return 0.0f;
        };
        float x = column(std::integral_constant<int, 0>{}) + column(std::integral_constant<int, 1>{});
        if constexpr (WIN > 2) x += column(std::integral_constant<int, 2>{});
        if constexpr (WIN > 3) x += column(std::integral_constant<int, 3>{});
        return x;
    };
    auto multiply = [&](int ch, int stage) {
        auto pair = [&](auto pair_tag) {
            constexpr int PAIR = decltype(pair_tag)::value;
            if constexpr (PAIR < G::PAIRS) {
                u32x4 f[WIN], g[T];
#pragma unroll
                for (int v = 0; v < WIN; v++) f[v] = filter_operand(ch, PAIR * WIN + v);
                column_operands(stage, pair_tag, g);
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int v = 0; v < WIN; v++) sum[t][v] = Mma<T_>::mfma16(f[v], g[t], sum[t][v]);
            }
        };
        pair(std::integral_constant<int, 0>{});
        pair(std::integral_constant<int, 1>{});
    };
    // Position by position: the other window row's share is zero on both sides, and what a position gives is added where a pixel has a tap there.
    auto multiply_masked = [&](int ch, int stage, int cy) {
        auto pair = [&](auto pair_tag) {
            constexpr int PAIR = decltype(pair_tag)::value;
            if constexpr (PAIR < G::PAIRS) {
                u32x4 g[T];
                column_operands(stage, pair_tag, g);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    constexpr int U0 = 2 * PAIR;
                    const int y = cy + G::D0 + U0 + h;
                    if (y < 0 || y >= p.h_out) continue;
#pragma unroll
                    for (int v = 0; v < WIN; v++) {
                        u32x4 f = filter_operand(ch, PAIR * WIN + v);
                        if (lq / 2 != h) f = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                        for (int t = 0; t < T; t++) {
                            u32x4 one_g = g[t];
                            if (lq / 2 != h) one_g = u32x4{0u, 0u, 0u, 0u};
                            const f32x4 one = Mma<T_>::mfma16(f, one_g, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                const int k1 = i / 2 + G::PAD - 2 * (G::D0 + U0 + h), k2 = i % 2 + G::PAD - 2 * (G::D0 + v);
                                if (k1 >= 0 && k1 < K && k2 >= 0 && k2 < K && t * 16 + l16 < p.w_out) sum[t][v][i] += one[i];
                            }
                        }
                    }
                }
            }
        };
        pair(std::integral_constant<int, 0>{});
        pair(std::integral_constant<int, 1>{});
    };

    auto item_at = [&](int n) { return n * (int)gridDim.x + xcd_remap(blockIdx.x, gridDim.x); };  // (neighbouring rows share grad_out in an XCD's cache)
    int n = 0, item = item_at(0), ch = 0, stage = 0;
    auto form_masked = [&](int item, int stage, float(&out)[T][4]) {
        clear();
        for (int again = 0; again < chunks; again++) {
            __syncthreads();  // what the stage held has been read
            request(item, again, stage);
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
            multiply_masked(again, stage, item % groups * G::ROWS + wave);
        }
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) out[t][i] = result(t, i);
    };
    auto store = [&](int item, const float(&out)[T][4]) {  // lane: channel lq of the cells l16 of every tile, their four pixels
        const int b = item / groups, cy = item % groups * G::ROWS + wave;
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int cx = t * 16 + l16;
            if (lq >= C || cx >= p.w_out || cy >= p.h_out) continue;
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const int y = 2 * cy + a;
                if (y >= p.h_in) continue;
                float v[2] = {out[t][2 * a], out[t][2 * a + 1]};
                uint32_t *dst = (uint32_t *)(p.grad_img + ((int64_t)(b * C + lq) * p.h_in + y) * p.w_in + 2 * cx);
                if (!p.fresh) {
                    const uint32_t old = *dst;
                    v[0] += Mma<T_>::to_f32(old & 0xffffu);
                    v[1] += Mma<T_>::to_f32(old >> 16);
                }
                *dst = Mma<T_>::pack2(v[0], v[1]);
            }
        }
    };
    if (__builtin_expect(bad_filters, 0)) {
        for (; item < p.items; item = item_at(++n)) {
            float out[T][4];
            form_masked(item, 0, out);
            store(item, out);
        }
        return;
    }
    if (item < p.items) request(item, 0, 0);
    clear();
    while (item < p.items) {
        const bool last = ch + 1 == chunks;
        const int next_item = last ? item_at(n + 1) : item, next_ch = last ? 0 : ch + 1;
        if (next_item < p.items) {
            request(next_item, next_ch, stage ^ 1);
            __builtin_amdgcn_s_waitcnt((G::REQUESTS & 15) | ((G::REQUESTS >> 4) << 14) | 0x0F70);  // this chunk's requests are in LDS
        } else {
            __builtin_amdgcn_s_waitcnt(0x0F70);
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        multiply(ch, stage);
        if (last) {
            float out[T][4];
            uint32_t nf = 0;
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    out[t][i] = result(t, i);
                    nf |= (__float_as_uint(out[t][i]) & 0x7f800000u) + 0x00800000u;
                }
            uint32_t *const votes = (uint32_t *)(smem + G::VOTES + (T < G::TW ? stage * G::STAGE : 0));  // (__syncthreads_or has LDS of its own, for which there is no room)
            const bool bad = __any((nf & 0x80000000u) != 0);
            if (lane == 0) votes[wave] = bad;
            __syncthreads();
            if (__builtin_expect((votes[0] | votes[1] | votes[2] | votes[3]) != 0, 0)) {
                form_masked(item, stage, out);
            }
            store(item, out);
            clear();
            n++;
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();  // this chunk has been read
        asm volatile("" ::: "memory");
        item = next_item;
        ch = next_ch;
        stage ^= 1;
    }
}

constexpr int GO_UNITS = 14, IMG_UNITS = 6;  // 16-byte pieces per thread: the host chooses bands that fit

// ---- filter gradient -------------------------------------------------------------------------------------------------
// grad_filters[64 channels][taps] over the pixels, v_mfma_f32_32x32x16: grad_out's rows are the product's rows, the C K K taps its
// columns, 16 pixels one step; two waves share a block of 32 channels.  A band of grad_out lies in LDS as it does in memory; the image is split into even and odd columns
// there (stride 2), so that the eight pixels of a lane's tap are one run of elements, shifted into place where it starts on an odd
// one.  Every wave keeps the sums of its share of the steps in registers over all bands of its workgroup;
// they meet in LDS in wave order, and the workgroups' sums in a second kernel in theirs: the same bits on every run.  The vector ALU bounds it
// (shifting the taps' runs into place, addresses): 52.5 -> 45.8 us with one division for all pieces of a thread (Walk) and the last step apart.
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
        Walk<256> go(tid, t.octs);
        const uint16_t *const src = p.go + ((int64_t)t.b * channels * p.h_out + t.first) * p.w_out;
#pragma unroll
        for (int n = 0; n < GO_UNITS; n++, go.next())
            if (go.q < channels) go_next[n] = *(const u32x4 *)(src + (int64_t)go.q * p.h_out * p.w_out + go.r * 8);
        const int in_rows = (t.rows - 1) * S + K, y0 = t.first * S - PAD;
        const uint16_t *const img = p.img + (int64_t)t.b * C * p.h_in * p.w_in;
        Walk<256> im(tid, octs_line);
#pragma unroll
        for (int n = 0; n < IMG_UNITS; n++, im.next()) {
            const int c = im.q >= in_rows ? im.q >= 2 * in_rows ? 2 : 1 : 0, y = y0 + im.q - c * in_rows, oct = im.r - 1;
            img_next[n] = u32x4{0u, 0u, 0u, 0u};
            if (im.q < C * in_rows && oct >= 0 && oct < octs_line - 2 && y >= 0 && y < p.h_in)
                img_next[n] = *(const u32x4 *)(img + ((int64_t)c * p.h_in + y) * p.w_in + oct * 8);
        }
    };
    if ((int)blockIdx.x < p.items) fetch(place(blockIdx.x));
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const Place at = place(item);
        const int in_rows = (at.rows - 1) * S + K, octs = at.octs;
        __syncthreads();  // the last item's reads are done
        Walk<256> go(tid, octs);
#pragma unroll
        for (int n = 0; n < GO_UNITS; n++, go.next())
            if (go.q < channels) *(u32x4 *)(go_lds + go.q * go_pitch + go.r * 8) = go_next[n];
        Walk<256> im(tid, octs_line);
#pragma unroll
        for (int n = 0; n < IMG_UNITS; n++, im.next()) {
            const int c = im.q >= in_rows ? im.q >= 2 * in_rows ? 2 : 1 : 0, oct = im.r - 1;
            if (im.q >= C * in_rows) continue;
            uint16_t *dst = img_lds + (c * in_max + im.q - c * in_rows) * pitch;
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
        // CUT: the upper half's pixels lie behind the last ones (zero on both sides: an infinity there meets no zero)
        auto multiply = [&](int step, auto cut_tag) {
            constexpr bool CUT = decltype(cut_tag)::value;
            const bool ok = !CUT || 2 * step + h < octs;
            const int oct = ok ? 2 * step + h : octs - 1, oh = oct / octs_row, ow = (oct - oh * octs_row) * 8;
            u32x4 a = *(const u32x4 *)(go_lds + (ob * 32 + l32) * go_pitch + oct * 8);
            if constexpr (CUT) {
#pragma unroll
                for (int w = 0; w < 4; w++) a[w] = ok ? a[w] : 0u;
            }
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
                    if constexpr (CUT) t[w] = ok ? t[w] : 0u;
                }
                acc[nb] = Mma<T>::mfma32(a, t, acc[nb]);
            }
        };
        int step = wave % 2;
        for (; 2 * step + 1 < octs; step += 2) multiply(step, std::false_type{});
        if (2 * step < octs) multiply(step, std::true_type{});
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
    const size_t half = (size_t)32 * c.chan_in * c.kernel * c.kernel * 2;  // 32 filters, and the four bytes behind them that a row's fifth word may be
    return (rows + 1023) / 1024 * 1024 + half + 16;                          // (rows come in whole instructions of 1 KB)
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
template <typename T, int C, int K, int TILES> hipError_t grad_img_rows_run(const ConvFew &c, hipStream_t stream) {
    using G = GradRows<C, K, TILES>;
    Params p = params_of(c, 1);
    p.items = c.batch * ((c.h_out + G::ROWS - 1) / G::ROWS);
    if (hipError_t e = allow_lds<conv_few_grad_img_rows_kernel<T, C, K, TILES>>(G::LDS)) return e;
    conv_few_grad_img_rows_kernel<T, C, K, TILES><<<(unsigned)std::min<int64_t>(p.items, 2 * (int64_t)c.compute_units), 256, G::LDS, stream>>>(p);
    return hipGetLastError();
}
template <typename T, int C, int K, int S> hipError_t backward_run(const ConvFew &c, void *workspace, hipStream_t stream) {
    bool rows = false;
    if constexpr (S == 2) {
        // Rows of up to seven tiles: with eight, filters of 7 x 7 on three channels leave no room for the votes (81920 + 16 bytes, and two
        // workgroups share 160 KB).  Smaller filters and one channel would fit with eight; rows beyond 112 were not measured for them and
        // take the kernel below, as all rows did before.
        if (c.w_out <= 112) {
            rows = true;
            if (hipError_t e = c.w_out <= 64 ? grad_img_rows_run<T, C, K, 4>(c, stream) : grad_img_rows_run<T, C, K, 7>(c, stream)) return e;
        }
    }
    if (!rows) {
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
