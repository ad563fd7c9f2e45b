// softmax(scale * Q . K^T) . V per head and its gradients without the (seq, seq) matrices: f16 / bf16, head dimensions of
// 32, 64 and 128, any sequence length.  One launch forward, two backward (one on few rows).
//
// What bounds it: written out as ops, attention moves the (seq, seq) scores and probabilities through HBM ten times a
// training step.  Here they exist in registers only, and the vector ALU (one exp2 and about five other instructions per
// score) and the matrix cores share the time.
//
// Shape of all three kernels: a workgroup of four waves owns 128 rows of one head (queries, or keys for dK / dV), 32 per
// wave, in registers; the other side passes through LDS in tiles of 64 rows, double buffered, staged through registers
// (the next tile's loads are in flight under this tile's MFMAs), one barrier per tile.  v_mfma_f32_32x32x16: the result
// tile has the wave's own row in `lane % 32`, so a softmax row lies inside one lane and its partner 32 lanes away, and
// the 16 values a lane holds are, eight by eight, exactly one lane's share of the B operand of the product that follows
// -- P and dS go from accumulator to operand by rounding alone, the contraction index merely takes the order
//     slot (h, j) of step g  <->  row 16 g + 8 (j / 4) + 4 h + j % 4,       h = lane / 32,
// which the A operand read beside it (rows of the LDS tile transposed by ds_read_b64_tr_b16) reproduces for free.
// The LDS tiles are XOR-swizzled so that both kinds of read touch every bank once (see `swizzle`).
//
// Measured over rotating buffers, bf16, (batch, seq, heads, dim), forward and backward, against the ops it replaces
// (scores, softmax, P . V, reshape and their backward, whose (seq, seq) matrices run at 5 TB/s): (16, 512, 16, 64)
// 120 -> 34 us and 212 -> 95 us; (8, 1024, 16, 64) 56 and 147 us; (16, 197, 12, 64) forward 51 -> 14 us.  The vector ALU
// is what is left: the matrix cores are busy a third of the time.  Multiplying the next tile's scores under this tile's
// exponentials inside one wave (two waves per SIMD instead of three) measured level in the forward (56 us at
// (8, 1024, 16, 64), 18 -> 26 us with 128-wide heads) and is left out there; in the backward, where the halves of a tile
// overlap that way, the dQ kernel gains 9 % (69 -> 63 us).
//
// No sum depends on timing: dK / dV are summed over the queries by the wave that owns the keys, dQ over the keys by the
// wave that owns the queries (the scores are formed once more for that instead of adding dQ with atomics).
#include "ctx_internal.h"
#include "gemm_internal.h"
#include <type_traits>
#include <utility>

namespace dfdx_rocm {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#define DFDX_LDS __attribute__((address_space(3)))

template <typename T> struct Mma;
template <> struct Mma<_Float16> {
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)v); }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, h2));
    }
};
template <> struct Mma<__bf16> {
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float to_f32(uint32_t v) { return __uint_as_float(v << 16); }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, b2));
    }
};

constexpr int WAVES = 4, ROWS = 32 * WAVES, TILE = 64;  // rows a workgroup owns; rows of a staged tile

struct Params {
    const uint16_t *q, *k, *v, *o, *go;
    uint16_t *out, *gq, *gk, *gv;
    float *lse, *delta;  // per (batch, head, row): log2 of the softmax denominator (with the maximum), sum of out * grad_out
    int64_t in_b, in_h, out_b, out_h, grad_b, grad_h;  // batch and head strides in elements of q, k, v / out, grad_out / gq, gk, gv
    int in_r, out_r, grad_r;                           // row strides
    int heads, seq, blocks, total;                     // row blocks per head, workgroups
    float scale, c;                                    // scale; scale * log2(e)
    int add_q, add_k, add_v;                           // gradients are added to what is there / stored
};

// XOR applied to the 16-byte piece index of row r of a [64][D] tile.  b128 reads: eight consecutive rows, one piece
// each.  Transposing reads: four consecutive rows, four consecutive pieces each.  Both cover the 256 bytes of the banks
// exactly once.
template <int D> __device__ __forceinline__ int swizzle(int r) {
    if constexpr (D == 128) return ((r & 3) << 2) | ((r >> 2) & 3);
    else if constexpr (D == 64) return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    else return (r >> 2) & 3;
}

// One [64][D] tile: 16-byte pieces, D / 32 of them per thread, held in registers between the load and the LDS store.
template <int D, bool ZERO = false> struct Stage {
    static constexpr int CPR = D / 8, N = TILE * CPR / 256, BYTES = TILE * D * 2;
    static constexpr int OUTSIDE = 0x7ffffff0;  // past every offset in a tile: see walkable
    u32x4 piece[N];
    // Rows past the end repeat the last one, or are ZERO: what the second products take meets probabilities of 0 there, and 0 times an
    // infinity is not 0.  What the scores are formed of repeats: zeros would make NaN of a key's infinity where its rows make -infinity.
    __device__ __forceinline__ void load(const uint16_t *base, int row_stride, int row0, int rows) {
        // (a buffer descriptor reads zeros at offsets past its end)
        const auto tile = __builtin_amdgcn_make_buffer_rsrc((void *)(base + (int64_t)row0 * row_stride), 0, OUTSIDE, 0x00020000);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int slot = i * 256 + (int)threadIdx.x, r = ZERO ? slot / CPR : min(slot / CPR, rows - row0 - 1);
            const int at = (r * row_stride + slot % CPR * 8) * 2;
            piece[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(tile, !ZERO || r < rows - row0 ? at : OUTSIDE, 0, 0));
        }
    }
    __device__ __forceinline__ void store(uint8_t *lds) const {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int slot = i * 256 + (int)threadIdx.x;
            const int r = slot / CPR;
            *(u32x4 *)(lds + r * D * 2 + ((slot % CPR) ^ swizzle<D>(r)) * 16) = piece[i];
        }
    }
};

// A operand with the tile's rows as the product's rows: rows r0 .. r0 + 31, elements 16 ks + 8 h .. + 7 of each.
template <int D> __device__ __forceinline__ u32x4 frag_rows(const uint8_t *lds, int r0, int ks) {
    const int lane = threadIdx.x % 64, r = r0 + lane % 32, h = lane / 32;
    return *(const u32x4 *)(lds + r * D * 2 + ((ks * 2 + h) ^ swizzle<D>(r)) * 16);
}
// A operand with the tile's columns as the product's rows: columns 32 dt .. + 31, the contraction over rows
// r0 + 8 (j / 4) + 4 h + j % 4.
template <int D> __device__ __forceinline__ u32x4 frag_cols(const uint8_t *lds, int r0, int dt) {
    const int lane = threadIdx.x % 64, h = lane / 32, l = lane % 16;
    const int col = dt * 32 + (lane / 16 % 2) * 16 + 4 * (l % 4);
    u32x4 f;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int r = r0 + 8 * j + 4 * h + l / 4;
        const uint8_t *p = lds + r * D * 2 + ((col / 8) ^ swizzle<D>(r)) * 16 + (col / 4 % 2) * 8;
        const v4i16 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((DFDX_LDS v4i16 *)(DFDX_LDS uint8_t *)p);
        const u32x2 u = __builtin_bit_cast(u32x2, t);
        f[2 * j] = u[0];
        f[2 * j + 1] = u[1];
    }
    return f;
}
// B operand of step g from 16 accumulator values.
template <typename T> __device__ __forceinline__ u32x4 as_operand(const f32x16 &v, int g) {
    u32x4 f;
#pragma unroll
    for (int j = 0; j < 4; j++) f[j] = Mma<T>::pack2(v[8 * g + 2 * j], v[8 * g + 2 * j + 1]);
    return f;
}
// The wave's own rows as B operand: row lane % 32, elements 16 ks + 8 h .. + 7.
template <int D> __device__ __forceinline__ void own_rows(const uint16_t *base, int row_stride, int row, u32x4 (&f)[D / 16]) {
    const int h = threadIdx.x % 64 / 32;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++) f[ks] = *(const u32x4 *)(base + (int64_t)row * row_stride + ks * 16 + h * 8);
}

__device__ __forceinline__ float both_halves_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_halves_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Stores acc^T * f: lane % 32 is the row (the pointer's), the accumulators hold columns 32 dt + 8 (i / 4) + 4 h + i % 4.
// Neighbouring groups of four columns trade halves of the wave so that a lane writes 16 contiguous bytes.
template <typename T, int D> __device__ __forceinline__ void store_rows(uint16_t *row, bool ok, const f32x16 (&acc)[D / 32], float f, bool add) {
    const int h = threadIdx.x % 64 / 32;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int m = 0; m < 2; m++) {
            uint32_t x[2][2];  // [column group 2m / 2m + 1][pairs]
            float y[2][4];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) y[t][e] = acc[dt][8 * m + 4 * t + e] * f;
            u32x4 o;
            uint16_t *p = row + dt * 32 + m * 16 + h * 8;
            if (!add) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int e = 0; e < 2; e++) x[t][e] = Mma<T>::pack2(y[t][2 * e], y[t][2 * e + 1]);
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const auto r = __builtin_amdgcn_permlane32_swap(x[0][e], x[1][e], false, false);
                    o[e] = r[0];
                    o[2 + e] = r[1];
                }
            } else {
                float z[8];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[0][e]), __float_as_uint(y[1][e]), false, false);
                    z[e] = __uint_as_float(r[0]);
                    z[4 + e] = __uint_as_float(r[1]);
                }
                u32x4 old = {0u, 0u, 0u, 0u};
                if (ok) old = *(const u32x4 *)p;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    o[e] = Mma<T>::pack2(z[2 * e] + Mma<T>::to_f32(old[e] & 0xffffu), z[2 * e + 1] + Mma<T>::to_f32(old[e] >> 16));
            }
            if (ok) *(u32x4 *)p = o;
        }
}

struct Block {
    int64_t head_row;  // first row of the head in lse / delta
    int64_t in, out, grad;
    int row0;
};
// Workgroups that share a head are neighbours on one XCD: its keys and values stay in that L2.
__device__ __forceinline__ Block my_block(const Params &p, int block) {
    const int w = xcd_remap(block, p.total), bh = w / p.blocks, b = bh / p.heads, hd = bh % p.heads;
    return {(int64_t)bh * p.seq, b * p.in_b + hd * p.in_h, b * p.out_b + hd * p.out_h, b * p.grad_b + hd * p.grad_h, w % p.blocks * ROWS};
}

// ---- forward: rows are queries -------------------------------------------------------------------------------------
// The running maximum is only moved when a row's new maximum exceeds it by more than RAISE (in log2): until then the
// exponentials stay below 2^RAISE, which f32 sums and the 16-bit operands hold at full relative precision, and the
// accumulators need no rescaling.
template <typename T, int D> __global__ __launch_bounds__(256, D == 128 ? 2 : 3) void attention_forward_kernel(const Params p) {
    constexpr float RAISE = 8.0f;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2][2][Stage<D>::BYTES];
    const Block b = my_block(p, blockIdx.x);
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, h = lane / 32;
    const int row = b.row0 + wave * 32 + lane % 32;
    const bool row_ok = row < p.seq;
    u32x4 qf[D / 16];
    own_rows<D>(p.q + b.in, p.in_r, min(row, p.seq - 1), qf);
    Stage<D> sk;
    Stage<D, true> sv;
    sk.load(p.k + b.in, p.in_r, 0, p.seq);
    sv.load(p.v + b.in, p.in_r, 0, p.seq);
    f32x16 acc[D / 32];
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[dt][i] = 0.0f;
    float m = -__FLT_MAX__, l = 0.0f;  // (finite: where all scores so far are -infinity the exponentials are 0, not NaN)
    sk.store(smem[0][0]);
    sv.store(smem[0][1]);
    __syncthreads();
    const int tiles = (p.seq + TILE - 1) / TILE;
    for (int t = 0; t < tiles; t++) {
        const uint8_t *kt = smem[t & 1][0], *vt = smem[t & 1][1];
        const bool more = t + 1 < tiles;
        if (more) {
            sk.load(p.k + b.in, p.in_r, (t + 1) * TILE, p.seq);
            sv.load(p.v + b.in, p.in_r, (t + 1) * TILE, p.seq);
        }
        f32x16 s[2];
#pragma unroll
        for (int n = 0; n < 2; n++) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[n][i] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < D / 16; ks++) s[n] = Mma<T>::mfma(frag_rows<D>(kt, n * 32, ks), qf[ks], s[n]);
        }
        if (t * TILE + TILE > p.seq) {  // the last tile: keys past the end take no part
#pragma unroll
            for (int n = 0; n < 2; n++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (t * TILE + n * 32 + 8 * (i / 4) + 4 * h + i % 4 >= p.seq) s[n][i] = -INFINITY;
        }
        float top = -INFINITY;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int i = 0; i < 16; i += 2) top = fmaxf(top, fmaxf(s[n][i], s[n][i + 1]));
        top = both_halves_max(top) * p.c;
        if (__any(top > m + RAISE)) {
            const float up = fmaxf(m, top), f = __builtin_amdgcn_exp2f(m - up);
            m = up;
            l *= f;
#pragma unroll
            for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[dt][i] *= f;
        }
        float part = 0.0f;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                s[n][i] = __builtin_amdgcn_exp2f(fmaf(s[n][i], p.c, -m));
                part += s[n][i];
            }
        l += part;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int g = 0; g < 2; g++) {
                const u32x4 pf = as_operand<T>(s[n], g);
#pragma unroll
                for (int dt = 0; dt < D / 32; dt++) acc[dt] = Mma<T>::mfma(frag_cols<D>(vt, n * 32 + g * 16, dt), pf, acc[dt]);
            }
        if (more) {
            sk.store(smem[(t + 1) & 1][0]);
            sv.store(smem[(t + 1) & 1][1]);
        }
        __syncthreads();
    }
    l = both_halves_sum(l);
    if (p.lse && row_ok && h == 0) p.lse[b.head_row + row] = m + __log2f(l);
    store_rows<T, D>(p.out + b.out + (int64_t)min(row, p.seq - 1) * p.out_r, row_ok, acc, 1.0f / l, false);
}

// ---- backward, rows are queries: dQ, and the row sums delta = sum(out * grad_out) that dS = P * (dP - delta) needs -----
template <int D> using Stages = uint8_t[2][2][Stage<D>::BYTES];
typedef float Stats[2][2][TILE];
template <typename T, int D> __device__ __forceinline__ void backward_q(const Params &p, int block, Stages<D> &smem) {
    const Block b = my_block(p, block);
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, h = lane / 32;
    const int row = b.row0 + wave * 32 + lane % 32, rowc = min(row, p.seq - 1);
    const bool row_ok = row < p.seq;
    Stage<D> sv;
    Stage<D, true> sk;
    sk.load(p.k + b.in, p.in_r, 0, p.seq);
    sv.load(p.v + b.in, p.in_r, 0, p.seq);
    u32x4 qf[D / 16], gf[D / 16];
    own_rows<D>(p.q + b.in, p.in_r, rowc, qf);
    own_rows<D>(p.go + b.out, p.out_r, rowc, gf);
    float delta = 0.0f;
    {
        u32x4 of[D / 16];
        own_rows<D>(p.o + b.out, p.out_r, rowc, of);
#pragma unroll
        for (int ks = 0; ks < D / 16; ks++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                delta += Mma<T>::to_f32(of[ks][e] & 0xffffu) * Mma<T>::to_f32(gf[ks][e] & 0xffffu) +
                         Mma<T>::to_f32(of[ks][e] >> 16) * Mma<T>::to_f32(gf[ks][e] >> 16);
    }
    delta = both_halves_sum(delta);
    if (row_ok && h == 0) p.delta[b.head_row + row] = delta;
    const float lse = p.lse[b.head_row + rowc];
    f32x16 acc[D / 32];
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[dt][i] = 0.0f;
    f32x16 minus_delta;
#pragma unroll
    for (int i = 0; i < 16; i++) minus_delta[i] = -delta;
    sk.store(smem[0][0]);
    sv.store(smem[0][1]);
    __syncthreads();
    const int tiles = (p.seq + TILE - 1) / TILE;
    auto step = [&](int t, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        const uint8_t *kt = smem[t & 1][0], *vt = smem[t & 1][1];
        if constexpr (!LAST) {
            sk.load(p.k + b.in, p.in_r, (t + 1) * TILE, p.seq);
            sv.load(p.v + b.in, p.in_r, (t + 1) * TILE, p.seq);
        }
        f32x16 s[2], dp[2];  // both halves of the tile: the second one's products run under the first one's exponentials
#pragma unroll
        for (int n = 0; n < 2; n++) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[n][i] = 0.0f;
            dp[n] = minus_delta;
#pragma unroll
            for (int ks = 0; ks < D / 16; ks++) {
                s[n] = Mma<T>::mfma(frag_rows<D>(kt, n * 32, ks), qf[ks], s[n]);
                dp[n] = Mma<T>::mfma(frag_rows<D>(vt, n * 32, ks), gf[ks], dp[n]);
            }
        }
#pragma unroll
        for (int n = 0; n < 2; n++) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                s[n][i] = __builtin_amdgcn_exp2f(fmaf(s[n][i], p.c, -lse)) * dp[n][i];
                if constexpr (LAST) {
                    if (t * TILE + n * 32 + 8 * (i / 4) + 4 * h + i % 4 >= p.seq) s[n][i] = 0.0f;
                }
            }
#pragma unroll
            for (int g = 0; g < 2; g++) {
                const u32x4 sf = as_operand<T>(s[n], g);
#pragma unroll
                for (int dt = 0; dt < D / 32; dt++) acc[dt] = Mma<T>::mfma(frag_cols<D>(kt, n * 32 + g * 16, dt), sf, acc[dt]);
            }
        }
        if constexpr (!LAST) {
            sk.store(smem[(t + 1) & 1][0]);
            sv.store(smem[(t + 1) & 1][1]);
            __syncthreads();
        }
    };
    for (int t = 0; t + 1 < tiles; t++) step(t, std::false_type{});
    step(tiles - 1, std::true_type{});
    store_rows<T, D>(p.gq + b.grad + (int64_t)rowc * p.grad_r, row_ok, acc, p.scale, p.add_q != 0);
}

// ---- backward, rows are keys: dK and dV; runs behind the one above, which leaves delta, or beside it (OWN) -----------
// The queries' lse and delta pass through LDS beside their tiles; past the last query lse is +inf, whose P is 0.
// OWN: delta is formed here, four threads to a row of `out` and grad_out.
template <typename T, int D, bool OWN> __device__ __forceinline__ void backward_kv(const Params &p, int block, Stages<D> &smem, Stats &stats) {
    const Block b = my_block(p, block);
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, h = lane / 32;
    const int row = b.row0 + wave * 32 + lane % 32, rowc = min(row, p.seq - 1);
    const bool row_ok = row < p.seq;
    Stage<D> sq;
    Stage<D, true> sg;
    float st = 0.0f;
    [[maybe_unused]] u32x4 o_part[D / 32], g_part[D / 32];
    [[maybe_unused]] bool past = false;
    auto load_stats = [&](int row0) {  // threads 0..63: lse, 64..127: -delta
        if constexpr (OWN) {
            const int64_t at = b.out + (int64_t)min(row0 + (int)threadIdx.x / 4, p.seq - 1) * p.out_r + threadIdx.x % 4 * (D / 4);
#pragma unroll
            for (int i = 0; i < D / 32; i++) {
                o_part[i] = *(const u32x4 *)(p.o + at + i * 8);
                g_part[i] = *(const u32x4 *)(p.go + at + i * 8);
            }
            past = row0 + (int)threadIdx.x / 4 >= p.seq;
            const int r = row0 + (int)threadIdx.x;
            if (threadIdx.x < TILE) st = r < p.seq ? p.lse[b.head_row + r] : INFINITY;
            return;
        }
        if (threadIdx.x < 2 * TILE) {
            const int r = row0 + (int)threadIdx.x % TILE;
            st = (threadIdx.x < TILE ? p.lse : p.delta)[b.head_row + min(r, p.seq - 1)];
            if (threadIdx.x >= TILE) st = -st;
            if (r >= p.seq) st = threadIdx.x < TILE ? INFINITY : 0.0f;
        }
    };
    auto store_stats = [&](int stage) {
        if constexpr (OWN) {
            float delta = 0.0f;
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    delta += Mma<T>::to_f32(o_part[i][e] & 0xffffu) * Mma<T>::to_f32(g_part[i][e] & 0xffffu) +
                             Mma<T>::to_f32(o_part[i][e] >> 16) * Mma<T>::to_f32(g_part[i][e] >> 16);
            delta += __shfl_xor(delta, 1, 64);
            delta += __shfl_xor(delta, 2, 64);
            if (threadIdx.x % 4 == 0) stats[stage][1][threadIdx.x / 4] = past ? 0.0f : -delta;
            if (threadIdx.x < TILE) stats[stage][0][threadIdx.x] = st;
            return;
        }
        if (threadIdx.x < 2 * TILE) stats[stage][threadIdx.x / TILE][threadIdx.x % TILE] = st;
    };
    sq.load(p.q + b.in, p.in_r, 0, p.seq);
    sg.load(p.go + b.out, p.out_r, 0, p.seq);
    load_stats(0);
    u32x4 kf[D / 16], vf[D / 16];
    own_rows<D>(p.k + b.in, p.in_r, rowc, kf);
    own_rows<D>(p.v + b.in, p.in_r, rowc, vf);
    f32x16 ak[D / 32], av[D / 32];
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) ak[dt][i] = av[dt][i] = 0.0f;
    sq.store(smem[0][0]);
    sg.store(smem[0][1]);
    store_stats(0);
    __syncthreads();
    const int tiles = (p.seq + TILE - 1) / TILE;
    for (int t = 0; t < tiles; t++) {
        const uint8_t *qt = smem[t & 1][0], *gt = smem[t & 1][1];
        const bool more = t + 1 < tiles;
        if (more) {
            sq.load(p.q + b.in, p.in_r, (t + 1) * TILE, p.seq);
            sg.load(p.go + b.out, p.out_r, (t + 1) * TILE, p.seq);
            load_stats((t + 1) * TILE);
        }
        f32x16 s[2], dp[2];  // both halves of the tile, see the kernel above
#pragma unroll
        for (int n = 0; n < 2; n++) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[n][i] = 0.0f;
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const f32x4 minus_delta = *(const f32x4 *)&stats[t & 1][1][n * 32 + 8 * i4 + 4 * h];
#pragma unroll
                for (int e = 0; e < 4; e++) dp[n][4 * i4 + e] = minus_delta[e];
            }
#pragma unroll
            for (int ks = 0; ks < D / 16; ks++) {
                s[n] = Mma<T>::mfma(frag_rows<D>(qt, n * 32, ks), kf[ks], s[n]);
                dp[n] = Mma<T>::mfma(frag_rows<D>(gt, n * 32, ks), vf[ks], dp[n]);
            }
        }
#pragma unroll
        for (int n = 0; n < 2; n++) {
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const f32x4 lse = *(const f32x4 *)&stats[t & 1][0][n * 32 + 8 * i4 + 4 * h];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s[n][4 * i4 + e] = __builtin_amdgcn_exp2f(fmaf(s[n][4 * i4 + e], p.c, -lse[e]));
                    dp[n][4 * i4 + e] *= s[n][4 * i4 + e];
                }
            }
#pragma unroll
            for (int g = 0; g < 2; g++) {
                const u32x4 pf = as_operand<T>(s[n], g), df = as_operand<T>(dp[n], g);
#pragma unroll
                for (int dt = 0; dt < D / 32; dt++) {
                    av[dt] = Mma<T>::mfma(frag_cols<D>(gt, n * 32 + g * 16, dt), pf, av[dt]);
                    ak[dt] = Mma<T>::mfma(frag_cols<D>(qt, n * 32 + g * 16, dt), df, ak[dt]);
                }
            }
        }
        if (more) {
            sq.store(smem[(t + 1) & 1][0]);
            sg.store(smem[(t + 1) & 1][1]);
            store_stats((t + 1) & 1);
        }
        __syncthreads();
    }
    const int64_t at = b.grad + (int64_t)rowc * p.grad_r;
    store_rows<T, D>(p.gk + at, row_ok, ak, p.scale, p.add_k != 0);
    store_rows<T, D>(p.gv + at, row_ok, av, 1.0f, p.add_v != 0);
}

template <typename T, int D> __global__ __launch_bounds__(256, D == 128 ? 1 : 2) void attention_backward_q_kernel(const Params p) {
    __shared__ __attribute__((aligned(1024))) Stages<D> smem;
    backward_q<T, D>(p, blockIdx.x, smem);
}
template <typename T, int D> __global__ __launch_bounds__(256, D == 128 ? 1 : 2) void attention_backward_kv_kernel(const Params p) {
    __shared__ __attribute__((aligned(1024))) Stages<D> smem;
    __shared__ __attribute__((aligned(16))) Stats stats;
    backward_kv<T, D, false>(p, blockIdx.x, smem, stats);
}
// Both in one launch, for few rows: the second launch and the chain of latencies that it would start with cost more there than the
// row sums formed once more.  (4, 100, 4, 64) bf16 6.6 + 6.9 -> 7.0 us, the training step of that block 109.1 -> 105.5.
template <typename T, int D> __global__ __launch_bounds__(256, D == 128 ? 1 : 2) void attention_backward_both_kernel(const Params p) {
    __shared__ __attribute__((aligned(1024))) Stages<D> smem;
    __shared__ __attribute__((aligned(16))) Stats stats;
    if ((int)blockIdx.x < p.total) backward_q<T, D>(p, blockIdx.x, smem);
    else backward_kv<T, D, true>(p, (int)blockIdx.x - p.total, smem, stats);
}

// ---- host side ------------------------------------------------------------------------------------------------------
inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }
// strides of (batch, head, row): what 16-byte pieces of a head's row can walk; offsets in a tile of 64 rows stay below 2^31 bytes
inline bool walkable(const int64_t s[3]) { return s[0] >= 0 && s[1] >= 0 && s[2] > 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 && s[2] < (1ll << 24); }
// What is written through these strides: two workgroups that share a row would store (or load, add and store) it without order.
// Sorted by stride, every axis has to step past all that the shorter ones reach.
bool rows_apart(int64_t batch, int64_t heads, int64_t seq, int64_t dim, const int64_t s[3]) {
    int64_t ext[3] = {batch, heads, seq}, str[3] = {s[0], s[1], s[2]}, reach = dim;
    for (int i = 0; i < 3; i++) {
        int low = i;
        for (int j = i + 1; j < 3; j++)
            if (str[j] < str[low]) low = j;
        std::swap(ext[i], ext[low]);
        std::swap(str[i], str[low]);
        if (ext[i] == 1) continue;
        if (str[i] < reach) return false;
        reach += (ext[i] - 1) * str[i];
    }
    return true;
}
// Does a row of one of two such views meet a row of the other, which lies `delta` elements behind?  What is left of the distance once the
// longer strides are taken out lies less than a stride from zero, on either side of it: rows_apart holds.
bool rows_meet(int64_t batch, int64_t heads, int64_t seq, int64_t dim, const int64_t s[3], int64_t delta) {
    const int64_t ext[3] = {batch, heads, seq};
    auto meet = [&](auto &&self, int left, int64_t apart) -> bool {  // `left`: a bit for each axis not taken out yet
        int top = -1;
        for (int i = 0; i < 3; i++)
            if ((left >> i & 1) && ext[i] > 1 && (top < 0 || s[i] > s[top])) top = i;
        if (top < 0) return apart > -dim && apart < dim;
        const int64_t steps = apart / s[top] - (apart % s[top] < 0);
        for (int64_t d = steps; d <= steps + 1; d++)
            if (d > -ext[top] && d < ext[top] && self(self, left & ~(1 << top), apart - d * s[top])) return true;
        return false;
    };
    return meet(meet, 7, delta);
}

}  // namespace

bool attention_supported(int dtype, int64_t batch, int64_t heads, int64_t seq, int64_t dim) {
    return (dtype == DT_F16 || dtype == DT_BF16) && (dim == 32 || dim == 64 || dim == 128) && batch >= 1 && heads >= 1 && seq >= 1 &&
           seq < (1ll << 30) && batch < (1ll << 24) && heads < (1ll << 24) && batch * heads < (1ll << 24) &&
           batch * heads * ((seq + ROWS - 1) / ROWS) < (1ll << 24);  // (workgroups of 256: a launch holds fewer than 2^32 threads)
}

namespace {
int fill(Params &p, int dtype, int64_t batch, int64_t heads, int64_t seq, int64_t dim, const void *q, const void *k, const void *v,
         const int64_t in[3], float scale, const int64_t out[3]) {
    if (dtype < DT_F32 || dtype > DT_F64 || batch < 0 || heads < 0 || seq < 0 || dim < 0 || !in || !out) return DFDX_ROCM_ERR_INVALID_ARG;
    if (!q || !k || !v) return DFDX_ROCM_ERR_INVALID_ARG;
    if (!attention_supported(dtype, batch, heads, seq, dim) || !(scale > 0.0f)) return DFDX_ROCM_ERR_UNSUPPORTED;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !walkable(in) || !walkable(out)) return DFDX_ROCM_ERR_UNSUPPORTED;
    p = Params{};
    p.q = (const uint16_t *)q; p.k = (const uint16_t *)k; p.v = (const uint16_t *)v;
    p.in_b = in[0]; p.in_h = in[1]; p.in_r = (int)in[2];
    p.out_b = out[0]; p.out_h = out[1]; p.out_r = (int)out[2];
    p.heads = (int)heads; p.seq = (int)seq;
    p.blocks = (int)((seq + ROWS - 1) / ROWS);
    p.total = (int)(batch * heads * p.blocks);
    p.scale = scale;
    p.c = scale * 1.44269504088896340736f;
    return DFDX_ROCM_OK;
}
}  // namespace
}  // namespace dfdx_rocm

using namespace dfdx_rocm;

extern "C" {

int dfdx_rocm_attention_forward(dfdx_rocm_ctx *ctx, int dtype, int64_t batch, int64_t heads, int64_t seq, int64_t dim, const void *q,
                                const void *k, const void *v, const int64_t strides[3], float scale, void *out,
                                const int64_t out_strides[3], float *lse) {
    if (int e = bind(ctx)) return e;
    Params p;
    if (batch == 0 || heads == 0 || seq == 0) return DFDX_ROCM_OK;
    if (int e = fill(p, dtype, batch, heads, seq, dim, q, k, v, strides, scale, out_strides)) return e;
    if (!out || !aligned16(out)) return out ? DFDX_ROCM_ERR_UNSUPPORTED : DFDX_ROCM_ERR_INVALID_ARG;
    if (!rows_apart(batch, heads, seq, dim, out_strides)) return DFDX_ROCM_ERR_ALIASED_OUTPUT;
    for (const void *ptr : {q, k, v})
        if (int e = settle(ctx, ptr)) return e;
    const int64_t ext[4] = {batch, heads, seq, dim}, str[4] = {out_strides[0], out_strides[1], out_strides[2], 1};
    if (int e = settle_output(ctx, out, dense_bytes(4, ext, str, 2), false, nullptr)) return e;
    if (int e = settle_output(ctx, lse, (size_t)(batch * heads * seq) * sizeof(float), false, nullptr)) return e;
    p.out = (uint16_t *)out;
    p.lse = lse;
    const dim3 grid((unsigned)p.total), block(256);
#define DFDX_RUN(KERNEL)                                                                     \
    do {                                                                                     \
        if (dtype == DT_F16) {                                                               \
            if (dim == 32) KERNEL<_Float16, 32><<<grid, block, 0, ctx->stream>>>(p);         \
            else if (dim == 64) KERNEL<_Float16, 64><<<grid, block, 0, ctx->stream>>>(p);    \
            else KERNEL<_Float16, 128><<<grid, block, 0, ctx->stream>>>(p);                  \
        } else {                                                                             \
            if (dim == 32) KERNEL<__bf16, 32><<<grid, block, 0, ctx->stream>>>(p);           \
            else if (dim == 64) KERNEL<__bf16, 64><<<grid, block, 0, ctx->stream>>>(p);      \
            else KERNEL<__bf16, 128><<<grid, block, 0, ctx->stream>>>(p);                    \
        }                                                                                    \
    } while (0)
    DFDX_RUN(attention_forward_kernel);
    return (int)hipGetLastError();
}

int dfdx_rocm_attention_backward(dfdx_rocm_ctx *ctx, int dtype, int64_t batch, int64_t heads, int64_t seq, int64_t dim, const void *q,
                                 const void *k, const void *v, const int64_t strides[3], float scale, const void *out,
                                 const void *grad_out, const int64_t out_strides[3], const float *lse, void *grad_q, void *grad_k,
                                 void *grad_v) {
    if (int e = bind(ctx)) return e;
    if (batch == 0 || heads == 0 || seq == 0) return DFDX_ROCM_OK;
    Params p;
    if (int e = fill(p, dtype, batch, heads, seq, dim, q, k, v, strides, scale, out_strides)) return e;
    if (!out || !grad_out || !lse || !grad_q || !grad_k || !grad_v) return DFDX_ROCM_ERR_INVALID_ARG;
    for (const void *ptr : {out, grad_out, (const void *)grad_q, (const void *)grad_k, (const void *)grad_v})
        if (!aligned16(ptr)) return DFDX_ROCM_ERR_UNSUPPORTED;
    if (!rows_apart(batch, heads, seq, dim, strides)) return DFDX_ROCM_ERR_ALIASED_OUTPUT;  // the gradients have the inputs' strides
    CtxLock lock(ctx->mu);  // delta lives in the shared workspace between the two launches
    if (int e = ensure_workspace(ctx, (size_t)(batch * heads * seq) * sizeof(float))) return e;
    for (const void *ptr : {q, k, v, out, grad_out, (const void *)lse})
        if (int e = settle(ctx, ptr)) return e;
    const int64_t ext[4] = {batch, heads, seq, dim}, str[4] = {strides[0], strides[1], strides[2], 1};
    const size_t dense = dense_bytes(4, ext, str, 2);
    bool fresh[3];
    void *const grads[3] = {grad_q, grad_k, grad_v};
    for (int i = 0; i < 3; i++)
        if (int e = settle_output(ctx, grads[i], dense, true, &fresh[i])) return e;
    p.o = (const uint16_t *)out; p.go = (const uint16_t *)grad_out;
    p.lse = const_cast<float *>(lse);
    p.delta = (float *)ctx->workspace;
    p.gq = (uint16_t *)grad_q; p.gk = (uint16_t *)grad_k; p.gv = (uint16_t *)grad_v;
    p.grad_b = p.in_b; p.grad_h = p.in_h; p.grad_r = p.in_r;
    p.add_q = !fresh[0]; p.add_k = !fresh[1]; p.add_v = !fresh[2];
    dim3 grid((unsigned)p.total);
    const dim3 block(256);
    // In one launch where the workgroups of both have a place at once and neither writes what the other reads or writes (packed
    // gradients interleave without meeting; one that two operands share is added to by one launch behind the other).
    auto end = [&](const void *from, const int64_t st[3]) { return (uintptr_t)from + (size_t)((batch - 1) * st[0] + (heads - 1) * st[1] + (seq - 1) * st[2] + dim) * 2; };
    bool apart = 2 * (int64_t)p.total <= (int64_t)ctx->compute_units * (dim == 128 ? 1 : 2);
    for (const void *ptr : {grad_k, grad_v})
        apart = apart && !rows_meet(batch, heads, seq, dim, strides, ((intptr_t)ptr - (intptr_t)grad_q) / 2);
    for (int i = 0; i < 3 && apart; i++) {
        const uintptr_t lo = (uintptr_t)grads[i], hi = end(grads[i], strides);
        auto meets = [&](const void *from, uintptr_t to) { return lo < to && (uintptr_t)from < hi; };
        for (const void *ptr : {q, k, v}) apart = apart && !meets(ptr, end(ptr, strides));
        for (const void *ptr : {out, grad_out}) apart = apart && !meets(ptr, end(ptr, out_strides));
        apart = apart && !meets(lse, (uintptr_t)(lse + batch * heads * seq));
    }
    if (apart) {
        grid.x *= 2;
        DFDX_RUN(attention_backward_both_kernel);
        return (int)hipGetLastError();
    }
    DFDX_RUN(attention_backward_q_kernel);
    if (hipError_t e = hipGetLastError()) return (int)e;
    DFDX_RUN(attention_backward_kv_kernel);
    return (int)hipGetLastError();
}

}  // extern "C"
