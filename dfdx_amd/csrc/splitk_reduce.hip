// Combines split-k partial sums: C = (accumulate ? C : 0) + bias + sum over splits of the f32 partial tiles,
// splits added in ascending order (deterministic), one rounding to the storage type on store.
#include "gemm_internal.h"

#include <type_traits>

namespace dfdx_rocm {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Cvt;
template <> struct Cvt<float> {
    static __device__ __forceinline__ float load(const float *p) { return *p; }
    static __device__ __forceinline__ void store(float *p, float v) { *p = v; }
};
template <> struct Cvt<_Float16> {
    static __device__ __forceinline__ float load(const _Float16 *p) { return (float)*p; }
    static __device__ __forceinline__ void store(_Float16 *p, float v) { *p = (_Float16)v; }
};
template <> struct Cvt<__bf16> {
    static __device__ __forceinline__ float load(const __bf16 *p) { return __uint_as_float((uint32_t)(*(const uint16_t *)p) << 16); }
    static __device__ __forceinline__ void store(__bf16 *p, float v) { *p = (__bf16)v; }  // RNE, quiet NaNs (v_cvt_pk_bf16_f32)
};

// Where beta = 1 reads the old values, and what else is done to a finished value (EXTRA_RELU and on); both laid out like C.
struct Beyond {
    const void *c_old, *with;
    int extra;
};
// `x` is a finished value, rounded to the element type; `w` its partner
__device__ __forceinline__ float apply_extra(int extra, float x, float w) {
    return extra == EXTRA_RELU ? fmaxf(x, 0.0f) : extra == EXTRA_RESIDUAL ? x + w : w > 0.0f ? x : 0.0f;
}

// The row sums that ride along with a split product (`ksum`, one value per row of C, `slots` partial sums each, stored
// [slot][row]).  The first `blocks` workgroups of grid row 0 do nothing else: each takes 16 rows; thread t adds the
// slots t / 16, t / 16 + 16, ... of row t % 16 in ascending order, four loads in flight at a time; the 16 partial sums
// of a row are added in a fixed order through LDS, then the old value unless the gradient is fresh.
struct KsumParts {
    const float *ws;   // null = none
    int64_t stride;
    void *out;
    int accumulate, slots, blocks;
};
constexpr int KSUM_ROWS = 16, KSUM_GROUPS = 256 / KSUM_ROWS;
template <typename T> __device__ __forceinline__ void combine_ksum(const KsumParts &ks, int m) {
    __shared__ float part[KSUM_GROUPS][KSUM_ROWS];
    const int r = threadIdx.x % KSUM_ROWS, g = threadIdx.x / KSUM_ROWS;
    const int row = min((int)blockIdx.x * KSUM_ROWS + r, m - 1);  // rows past the end repeat the last one, unused
    const float *src = ks.ws + row;
    float v = 0.0f;
    int s = g;
    for (; s + 3 * KSUM_GROUPS < ks.slots; s += 4 * KSUM_GROUPS) {
        const float a = src[(int64_t)s * ks.stride], b = src[(int64_t)(s + KSUM_GROUPS) * ks.stride];
        const float c = src[(int64_t)(s + 2 * KSUM_GROUPS) * ks.stride], d = src[(int64_t)(s + 3 * KSUM_GROUPS) * ks.stride];
        v = (((v + a) + b) + c) + d;
    }
    for (; s < ks.slots; s += KSUM_GROUPS) v += src[(int64_t)s * ks.stride];
    part[g][r] = v;
    __syncthreads();
    if (g == 0 && (int)blockIdx.x * KSUM_ROWS + r < m) {
#pragma unroll
        for (int q = 1; q < KSUM_GROUPS; q++) v += part[q][r];
        T *dst = (T *)ks.out + row;
        const float old = ks.accumulate ? Cvt<T>::load(dst) : 0.0f;
        Cvt<T>::store(dst, old + v);
    }
}

// Where the results of batch blockIdx.z lie (elements): several split products in one launch (GemmProblem::batches).
struct Batches {
    int nb2, splits;
    int64_t c_b1, c_b2, k_b1, k_b2;
};
// What the kernels below take for a product with either; the plain ones take None and read no argument for it (the loads of the
// launch's size and of these addresses stood in front of everything else: 256 x 8192 x 384 f16 in 13 pieces 14.5 us with them, 14.4
// without, 259 x 8192 x 381 in 8 14.8 and 14.7).
struct More {
    Beyond bd;
    Batches bt;
};
struct None {};
template <typename T> __device__ __forceinline__ void to_batch(const Batches &bt, const float *&ws, int64_t ws_split_stride, T *&c, KsumParts &ks, Beyond &bd) {
    if (gridDim.z == 1) return;
    const int z = blockIdx.z, z1 = z / bt.nb2, z2 = z - z1 * bt.nb2;
    const int64_t off = z1 * bt.c_b1 + z2 * bt.c_b2;
    ws += (int64_t)z * bt.splits * ws_split_stride;
    c += off;
    bd.c_old = (const T *)bd.c_old + off;
    bd.with = (const T *)bd.with + off;
    ks.ws = ks.ws ? ks.ws + (int64_t)z * ks.slots * ks.stride : nullptr;
    ks.out = (T *)ks.out + (z1 * bt.k_b1 + z2 * bt.k_b2);
}

// one thread: 4 consecutive columns of one row
template <typename T, typename M>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *ws, int splits, int64_t ws_ld, int64_t ws_split_stride,
                                                            T *c, int64_t c_rs, int m, int n, int accumulate, int bias_mode,
                                                            const T *bias, int vec4, KsumParts ks, M more) {
    constexpr bool PLAIN = std::is_same_v<M, None>;
    if constexpr (!PLAIN) to_batch<T>(more.bt, ws, ws_split_stride, c, ks, more.bd);
    if (ks.ws && (int)blockIdx.x < ks.blocks) {   // uniform over the workgroup
        if (blockIdx.y == 0) combine_ksum<T>(ks, m);
        return;   // the same block index in the other grid rows has no work
    }
    const int col = (blockIdx.y * 64 + threadIdx.x % 64) * 4;   // rows along grid.x: its limit is 2^31, grid.y's 65535
    const int row = ((int)blockIdx.x - (ks.ws ? ks.blocks : 0)) * 4 + threadIdx.x / 64;
    if (row >= m || col >= n) return;
    const float *src = ws + (int64_t)row * ws_ld + col;
    // eight partial sums requested at a time (a tail repeats the last one, unused), added in ascending order: one round
    // trip to memory per eight splits instead of one per split
    f32x4 v;
    for (int s0 = 0; s0 < splits; s0 += 8) {
        f32x4 part[8];
#pragma unroll
        for (int u = 0; u < 8; u++) part[u] = *(const f32x4 *)(src + (int64_t)min(s0 + u, splits - 1) * ws_split_stride);
        if (s0 == 0) v = part[0];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s0 + u < splits && s0 + u > 0) v += part[u];
    }
    T *dst = c + (int64_t)row * c_rs + col;
    const T *from = dst;
    if constexpr (!PLAIN) from = (const T *)more.bd.c_old + (dst - c);
    // value `e` of the thread's columns with what is done to it
    [[maybe_unused]] auto beyond = [&](float x, int e) -> float {
        if constexpr (!PLAIN) {
            if (more.bd.extra) x = apply_extra(more.bd.extra, x, more.bd.extra == EXTRA_RELU ? 0.0f : Cvt<T>::load((const T *)more.bd.with + (dst - c) + e));
        }
        return x;
    };
    const float rb = (bias_mode == BIAS_PER_ROW) ? Cvt<T>::load(bias + row) : 0.0f;
    if constexpr (sizeof(T) == 4) {
        if (vec4 && col + 3 < n) {   // f32 rows aligned to 16 B: one load of the old values, one store
            f32x4 x = v + rb;
            if (bias_mode == BIAS_PER_COL) x += *(const f32x4 *)(bias + col);
            if (accumulate) x += *(const f32x4 *)from;
            if constexpr (!PLAIN) {
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = beyond(x[e], e);
            }
            *(f32x4 *)dst = x;
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (col + e >= n) break;
        float x = v[e] + rb;
        if (bias_mode == BIAS_PER_COL) x += Cvt<T>::load(bias + col + e);
        if (accumulate) x += Cvt<T>::load(from + e);
        if constexpr (!PLAIN) {
            T rounded;
            Cvt<T>::store(&rounded, x);
            x = beyond(Cvt<T>::load(&rounded), e);
        }
        Cvt<T>::store(dst + e, x);
    }
}

// 16-bit outputs whose rows are 16 B-aligned: one thread owns 8 consecutive columns of one row -- two 16 B loads per
// split, requested four splits at a time, the old C values (beta = 1) requested before the first partial arrives, one
// 16 B store.  Same order of additions per element as the general kernel: splits ascending, row bias, column bias, old C.
template <typename T> struct Bits16;
template <> struct Bits16<_Float16> {
    static __device__ __forceinline__ float widen(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
    static __device__ __forceinline__ uint16_t narrow(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
};
template <> struct Bits16<__bf16> {
    static __device__ __forceinline__ float widen(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
    static __device__ __forceinline__ uint16_t narrow(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }  // RNE, quiet NaNs
};
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T, typename M>
__global__ __launch_bounds__(256) void splitk_reduce16_kernel(const float *ws, int splits, int64_t ws_ld, int64_t ws_split_stride,
                                                              uint16_t *c, int64_t c_rs, int m, int n, int accumulate,
                                                              int bias_mode, const uint16_t *bias, KsumParts ks, M more) {
    constexpr bool PLAIN = std::is_same_v<M, None>;
    if constexpr (!PLAIN) to_batch<uint16_t>(more.bt, ws, ws_split_stride, c, ks, more.bd);
    if (ks.ws && (int)blockIdx.x < ks.blocks) {   // uniform over the workgroup
        if (blockIdx.y == 0) combine_ksum<T>(ks, m);
        return;   // the same block index in the other grid rows has no work
    }
    const int col = (blockIdx.y * 64 + threadIdx.x % 64) * 8;
    const int row = ((int)blockIdx.x - (ks.ws ? ks.blocks : 0)) * 4 + threadIdx.x / 64;
    if (row >= m || col >= n) return;   // n is a multiple of 8: a thread's 8 columns are all inside or all outside
    const float *src = ws + (int64_t)row * ws_ld + col;
    uint16_t *dst = c + (int64_t)row * c_rs + col;
    u32x4 old = {0u, 0u, 0u, 0u}, cb = {0u, 0u, 0u, 0u};
    [[maybe_unused]] u32x4 with = {0u, 0u, 0u, 0u};
    if constexpr (PLAIN) {
        if (accumulate) old = *(const u32x4 *)dst;
    } else {
        if (accumulate) old = *(const u32x4 *)((const uint16_t *)more.bd.c_old + (dst - c));
        if (more.bd.extra > EXTRA_RELU) with = *(const u32x4 *)((const uint16_t *)more.bd.with + (dst - c));
    }
    if (bias_mode == BIAS_PER_COL) cb = *(const u32x4 *)(bias + col);
    // eight splits requested at a time (a tail repeats the last one, unused) and added in ascending order: with the old
    // C values and the bias that is ONE round trip to memory for up to eight splits (a loop that waited for split after
    // split paid five for eight splits: 9.2 us for the 1024 x 1024 weight gradients)
    f32x4 lo, hi;
    for (int s0 = 0; s0 < splits; s0 += 8) {
        f32x4 a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float *q = src + (int64_t)min(s0 + u, splits - 1) * ws_split_stride;
            a[u] = *(const f32x4 *)q;
            b[u] = *(const f32x4 *)(q + 4);
        }
        if (s0 == 0) {
            lo = a[0];
            hi = b[0];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s0 + u < splits && s0 + u > 0) {
                lo += a[u];
                hi += b[u];
            }
    }
    const float rb = (bias_mode == BIAS_PER_ROW) ? Bits16<T>::widen(bias[row]) : 0.0f;
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        float x = (e < 4 ? lo[e] : hi[e - 4]) + rb;
        const int sh = (e & 1) * 16;
        if (bias_mode == BIAS_PER_COL) x += Bits16<T>::widen((uint16_t)(cb[e / 2] >> sh));
        if (accumulate) x += Bits16<T>::widen((uint16_t)(old[e / 2] >> sh));
        uint32_t bits = Bits16<T>::narrow(x);
        if constexpr (!PLAIN) {
            if (more.bd.extra) bits = Bits16<T>::narrow(apply_extra(more.bd.extra, Bits16<T>::widen((uint16_t)bits), Bits16<T>::widen((uint16_t)(with[e / 2] >> sh))));
        }
        out[e / 2] = (e & 1) ? (out[e / 2] | (bits << 16)) : bits;
    }
    *(u32x4 *)dst = out;
}

}  // namespace

// C of `p` must have unit column stride and no batch (the planner only splits such problems), or `batches`.
hipError_t launch_splitk_reduce(const GemmProblem &p, int64_t ws_ld, int64_t ws_split_stride, hipStream_t stream,
                                const float *ws_ksum, int64_t ws_ksum_stride, int ksum_slots) {
    const bool with_ksum = p.ksum && ws_ksum;
    const KsumParts ks{with_ksum ? ws_ksum : nullptr, ws_ksum_stride, p.ksum, p.ksum_accumulate, ksum_slots,
                       with_ksum ? (int)((p.m + KSUM_ROWS - 1) / KSUM_ROWS) : 0};
    const bool from = p.extra == EXTRA_FROM;
    const Beyond bd{from ? p.with : p.c, p.with, from ? EXTRA_NONE : p.extra};
    const unsigned products = p.reduce ? 1u : (unsigned)p.batch_count();
    const Batches bt{products > 1 ? (int)p.nb2 : 1, p.splits, p.c_b1, p.c_b2, p.ksum_b1, p.ksum_b2};
    dim3 grid((unsigned)((p.m + 3) / 4 + ks.blocks), (unsigned)((p.n + 255) / 256), products), block(256);
    if ((p.n + 255) / 256 > 65535) return hipErrorInvalidValue;  // 16.7 M columns: no planner splits such a product
    const int64_t c_rs = p.m == 1 ? p.n : p.c_rs;
    const int bias_mode = p.bias ? p.bias_mode : BIAS_NONE;
    const bool is16 = p.dtype == DT_F16 || p.dtype == DT_BF16;
    const bool rows16 = is16 && p.n % 8 == 0 && c_rs % 8 == 0 && (products == 1 || (p.c_b1 % 8 == 0 && p.c_b2 % 8 == 0)) && ws_ld % 4 == 0 && ws_split_stride % 4 == 0 &&
                        ((uintptr_t)p.c & 15u) == 0 && ((uintptr_t)p.workspace & 15u) == 0 && (((uintptr_t)bd.c_old | (uintptr_t)bd.with) & 15u) == 0 &&
                        (bias_mode != BIAS_PER_COL || ((uintptr_t)p.bias & 15u) == 0);
    const int vec4 = p.dtype == DT_F32 && c_rs % 4 == 0 && ((uintptr_t)p.c & 15u) == 0 && ws_ld % 4 == 0 && ws_split_stride % 4 == 0 &&
                     (((uintptr_t)p.workspace | (uintptr_t)bd.c_old) & 15u) == 0 && (bias_mode != BIAS_PER_COL || ((uintptr_t)p.bias & 15u) == 0);
    auto any_rows = [&](auto type, auto more) -> hipError_t {
        typedef decltype(type) T;
        splitk_reduce_kernel<T><<<grid, block, 0, stream>>>(p.workspace, p.splits, ws_ld, ws_split_stride, (T *)p.c, c_rs, (int)p.m, (int)p.n,
                                                            p.accumulate, bias_mode, (const T *)p.bias, vec4, ks, more);
        return hipGetLastError();
    };
    auto half_type = [&](auto type, auto more) -> hipError_t {
        if (!rows16) return any_rows(type, more);
        const dim3 grid16((unsigned)((p.m + 3) / 4 + ks.blocks), (unsigned)((p.n + 511) / 512), products);
        splitk_reduce16_kernel<decltype(type)><<<grid16, block, 0, stream>>>(p.workspace, p.splits, ws_ld, ws_split_stride, (uint16_t *)p.c, c_rs, (int)p.m,
                                                                             (int)p.n, p.accumulate, bias_mode, (const uint16_t *)p.bias, ks, more);
        return hipGetLastError();
    };
    auto run = [&](auto more) -> hipError_t {
        switch (p.dtype) {
        case DT_F32: return any_rows(0.0f, more);
        case DT_F16: return half_type((_Float16)0, more);
        case DT_BF16: return half_type((__bf16)0.0f, more);
        default: return hipErrorInvalidValue;
        }
    };
    return products == 1 && p.extra == EXTRA_NONE ? run(None{}) : run(More{bd, bt});
}

}  // namespace dfdx_rocm
