// C ABI of the dfdx ROCm matmul backend: context, storage helpers, GEMM dispatch.
#include "ctx_internal.h"
#include "gemm_internal.h"

#include <algorithm>
#include <cstdio>
#include <cstring>

using namespace dfdx_rocm;

namespace dfdx_rocm {

int bind(dfdx_rocm_ctx *ctx) {
    if (!ctx) return DFDX_ROCM_ERR_INVALID_ARG;
    HIP_TRY(hipSetDevice(ctx->device));
    return DFDX_ROCM_OK;
}

// Frees the buffers that `grow` replaced.  The caller has drained the stream.
static hipError_t free_retired(dfdx_rocm_ctx *ctx) {
    hipError_t first = hipSuccess;
    for (void *p : ctx->retired) {
        const hipError_t e = hipFree(p);
        if (first == hipSuccess) first = e;
    }
    ctx->retired.clear();
    ctx->retired_bytes = 0;
    ctx->copies_refused = SIZE_MAX;  // (there may be room again)
    return first;
}

// The stream is not drained here: work already queued keeps the old buffer, which is retired, and the call in hand
// gets a new one.  (Drained all the same: when an allocation fails, which then is tried once more with everything retired freed, and
// when the retired buffers hold kRetiredBytes.)  A buffer grows by half of itself at least, up to kGrowthBytes more than asked for, so that
// sizes that rise step by step do not leave a buffer behind at every step.
static int grow(dfdx_rocm_ctx *ctx, void **buf, size_t *have, size_t bytes) {
    constexpr size_t kRetiredBytes = size_t(1) << 30, kGrowthBytes = size_t(256) << 20, kMb = size_t(1) << 20;
    CtxLock lock(ctx->mu);
    if (bytes <= *have) return DFDX_ROCM_OK;
    bytes = (bytes + kMb - 1) & ~(kMb - 1);
    const size_t roomy = std::max(bytes, std::min(*have + *have / 2, bytes + kGrowthBytes) & ~(kMb - 1));
    if (*buf) {
        ctx->retired.push_back(*buf);
        ctx->retired_bytes += *have;
        *buf = nullptr;
        *have = 0;
    }
    if (ctx->retired_bytes >= kRetiredBytes) {
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        (void)free_retired(ctx);
    }
    size_t got = roomy;
    hipError_t e = hipMalloc(buf, got);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        if (!ctx->retired.empty()) {
            HIP_TRY(hipStreamSynchronize(ctx->stream));
            (void)free_retired(ctx);
        }
        got = bytes;
        e = hipMalloc(buf, got);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();  // the failed allocation must not surface again in the next launch check
        *buf = nullptr;
        return (int)e;
    }
    *have = got;
    return DFDX_ROCM_OK;
}

static std::map<uintptr_t, size_t>::iterator pending_holding(dfdx_rocm_ctx *ctx, uintptr_t p) {
    auto it = ctx->pending_zero.upper_bound(p);
    if (it == ctx->pending_zero.begin()) return ctx->pending_zero.end();
    --it;
    return p < it->first + it->second ? it : ctx->pending_zero.end();
}

static int fill_and_drop(dfdx_rocm_ctx *ctx, std::map<uintptr_t, size_t>::iterator it) {
    const hipError_t e = launch_zero_fill((void *)it->first, it->second, ctx->compute_units, ctx->stream);
    if (e != hipSuccess) return (int)e;
    ctx->pending_zero.erase(it);
    ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
    return DFDX_ROCM_OK;
}

int settle(dfdx_rocm_ctx *ctx, const void *ptr) {
    if (!ptr || ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    CtxLock lock(ctx->mu);
    auto it = pending_holding(ctx, (uintptr_t)ptr);
    return it == ctx->pending_zero.end() ? DFDX_ROCM_OK : fill_and_drop(ctx, it);
}

int settle_output(dfdx_rocm_ctx *ctx, void *ptr, size_t bytes, bool accumulates, bool *fresh) {
    if (fresh) *fresh = false;
    if (!ptr || ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    CtxLock lock(ctx->mu);
    auto it = pending_holding(ctx, (uintptr_t)ptr);
    if (it == ctx->pending_zero.end()) return DFDX_ROCM_OK;
    const bool covered = bytes && it->first == (uintptr_t)ptr && it->second == bytes;
    if (covered && (!accumulates || fresh)) {  // every byte is stored without being read first: no fill needed
        ctx->pending_zero.erase(it);
        ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
        if (fresh) *fresh = accumulates;
        return DFDX_ROCM_OK;
    }
    return fill_and_drop(ctx, it);
}

// Runs every deferred fill that overlaps [ptr, ptr + bytes) (a read of that range follows).
static int settle_range(dfdx_rocm_ctx *ctx, const void *ptr, size_t bytes) {
    if (!ptr || ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    CtxLock lock(ctx->mu);
    const uintptr_t lo = (uintptr_t)ptr, hi = lo + bytes;
    auto first = pending_holding(ctx, lo);
    if (first != ctx->pending_zero.end())
        if (int e = fill_and_drop(ctx, first)) return e;
    for (auto it = ctx->pending_zero.lower_bound(lo); it != ctx->pending_zero.end() && it->first < hi;
         it = ctx->pending_zero.lower_bound(lo))
        if (int e = fill_and_drop(ctx, it)) return e;
    return DFDX_ROCM_OK;
}

// Forgets (without filling) every deferred fill that lies wholly inside [ptr, ptr + bytes); one that straddles an end is run.
static int drop_pending_inside(dfdx_rocm_ctx *ctx, const void *ptr, size_t bytes) {
    if (!ptr || ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    CtxLock lock(ctx->mu);
    const uintptr_t lo = (uintptr_t)ptr, hi = lo + bytes;
    auto first = pending_holding(ctx, lo);
    if (first != ctx->pending_zero.end() && first->first < lo)
        if (int e = fill_and_drop(ctx, first)) return e;
    for (auto it = ctx->pending_zero.lower_bound(lo); it != ctx->pending_zero.end() && it->first < hi;) {
        if (it->first + it->second > hi) {
            if (int e = fill_and_drop(ctx, it)) return e;
            break;
        }
        it = ctx->pending_zero.erase(it);
    }
    ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
    return DFDX_ROCM_OK;
}

int settle_all(dfdx_rocm_ctx *ctx) {
    if (ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    CtxLock lock(ctx->mu);
    while (!ctx->pending_zero.empty())
        if (int e = fill_and_drop(ctx, ctx->pending_zero.begin())) return e;
    return DFDX_ROCM_OK;
}

size_t dense_bytes(int rank, const int64_t *extents, const int64_t *strides, size_t elem_bytes) {
    int64_t ext[8], str[8];
    int n = 0;
    if (rank > 8) return 0;
    for (int i = 0; i < rank; i++) {
        if (extents[i] == 0) return 0;
        if (extents[i] == 1) continue;
        if (strides[i] <= 0) return 0;
        int j = n++;
        for (; j > 0 && str[j - 1] > strides[i]; j--) {  // insertion sort by stride
            ext[j] = ext[j - 1];
            str[j] = str[j - 1];
        }
        ext[j] = extents[i];
        str[j] = strides[i];
    }
    int64_t run = 1;
    for (int i = 0; i < n; i++) {
        if (str[i] != run) return 0;
        run *= ext[i];
    }
    return (size_t)run * elem_bytes;
}

int ensure_workspace(dfdx_rocm_ctx *ctx, size_t bytes) { return grow(ctx, &ctx->workspace, &ctx->workspace_bytes, bytes); }
int ensure_patches(dfdx_rocm_ctx *ctx, size_t bytes) { return grow(ctx, &ctx->patches, &ctx->patches_bytes, bytes); }

}  // namespace dfdx_rocm

namespace {

// Scratch of dfdx_rocm_gemm_noalloc: partial sums of split reductions for callers that may not allocate.  Every device
// the library runs on holds its own copy of this array, at its own address, until the process ends.  In host code the
// array's NAME is only a handle for hipGetSymbolAddress: the address a kernel may use is looked up once per device in
// dfdx_rocm_create (with that device current) and kept in `scratch_of_device` / the context.
__device__ __align__(256) __attribute__((used)) static unsigned char scratch[DFDX_ROCM_NOALLOC_SCRATCH_BYTES];
constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
void *scratch_of_device[kMaxDevices];  // guarded by scratch_mu

// The calling thread's current device must be `ordinal`.
int scratch_address(int ordinal, void **out) {
    if (ordinal < 0 || ordinal >= kMaxDevices) return DFDX_ROCM_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_of_device[ordinal]) {
        void *ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return (int)hipErrorInvalidSymbol;
        scratch_of_device[ordinal] = ptr;
    }
    *out = scratch_of_device[ordinal];
    return DFDX_ROCM_OK;
}

// Validates `d` and produces the canonical problem (row-major C whenever the view allows it).
// `colsum_b` (may be null): where the caller would like the sums of B over the contraction; it stays in the problem only
// when the problem is the plain one (no aliased output axis).
int make_problem(const dfdx_rocm_gemm_desc *d, GemmProblem *out, void *colsum_b = nullptr) {
    if (!d) return DFDX_ROCM_ERR_INVALID_ARG;
    if (d->dtype < DFDX_ROCM_F32 || d->dtype > DFDX_ROCM_F64) return DFDX_ROCM_ERR_INVALID_ARG;
    if (d->m < 0 || d->n < 0 || d->k < 0 || d->batch1 < 1 || d->batch2 < 1) return DFDX_ROCM_ERR_INVALID_ARG;
    if (d->m == 0 || d->n == 0) {
        out->m = 0;
        return DFDX_ROCM_OK;
    }
    if (!d->c || (d->k > 0 && (!d->a || !d->b))) return DFDX_ROCM_ERR_INVALID_ARG;
    if (d->c_rs < 0 || d->c_cs < 0 || d->c_b1 < 0 || d->c_b2 < 0) return DFDX_ROCM_ERR_INVALID_ARG;
    if (!d->reduce_batch && ((d->batch1 > 1 && d->c_b1 == 0) || (d->batch2 > 1 && d->c_b2 == 0)))
        return DFDX_ROCM_ERR_ALIASED_OUTPUT;
    // An output view with a zero stride along a matrix axis maps a whole row (or column) of logical elements to one
    // address: the gradient of an operand that was broadcast along that axis (matmul/mod.rs:318-320 lets such views
    // in).  The elements that share an address are SUMMED, which is the gradient of a broadcast (the reference's Cpu
    // path lets them overwrite each other, its Cuda path reads past the buffer).  The aliased axis becomes a batch axis
    // of a product with one row (or column), reduced over the batch.
    const bool rows_alias = d->m > 1 && d->c_rs == 0, cols_alias = d->n > 1 && d->c_cs == 0;
    if (rows_alias || cols_alias) {
        if (d->batch1 * d->batch2 != 1 || d->reduce_batch || d->bias) return DFDX_ROCM_ERR_ALIASED_OUTPUT;
        dfdx_rocm_gemm_desc r = *d;
        r.reduce_batch = 1;
        r.c_b1 = r.c_b2 = 0;
        if (rows_alias) {  // C[j] += sum_i sum_k A[i,k] B[k,j]: the rows become batch 1
            r.m = 1;
            r.batch1 = d->m;
            r.a_b1 = d->a_rs;
            r.b_b1 = 0;
            r.c_rs = cols_alias ? 1 : d->n * (d->c_cs > 0 ? d->c_cs : 1);
        }
        if (cols_alias) {  // C[i] += sum_j sum_k A[i,k] B[k,j]: the columns become batch 2
            r.n = 1;
            r.batch2 = d->n;
            r.a_b2 = 0;
            r.b_b2 = d->b_cs;
            r.c_cs = 1;
        }
        r.flags |= DFDX_ROCM_GEMM_NO_SPLIT_K;
        return make_problem(&r, out);
    }
    GemmProblem p;
    p.dtype = d->dtype;
    p.accumulate = d->accumulate != 0;
    p.reduce = d->reduce_batch != 0 && d->batch1 * d->batch2 > 1;
    p.bias_mode = d->bias ? BIAS_PER_COL : BIAS_NONE;
    p.m = d->m; p.n = d->n; p.k = d->k;
    p.nb1 = d->batch1; p.nb2 = d->batch2;
    p.a = d->a; p.a_rs = d->a_rs; p.a_cs = d->a_cs; p.a_b1 = d->a_b1; p.a_b2 = d->a_b2;
    p.b = d->b; p.b_rs = d->b_rs; p.b_cs = d->b_cs; p.b_b1 = d->b_b1; p.b_b2 = d->b_b2;
    p.c = d->c; p.c_rs = d->c_rs; p.c_cs = d->c_cs;
    p.c_b1 = p.reduce ? 0 : d->c_b1; p.c_b2 = p.reduce ? 0 : d->c_b2;
    p.bias = d->bias;
    p.ksum = colsum_b;
    p.ksum_of = colsum_b ? KSUM_OF_B : KSUM_NONE;
    p.ksum_accumulate = 1;
    p.splits = 1;
    p.workspace = nullptr;
    p.compute_units = 0;
    // column-major C (a permuted operand's gradient): compute C^T = B^T A^T instead
    if (p.c_cs != 1 && p.c_rs == 1 && p.n > 1) p = transposed(p);
    *out = p;
    return DFDX_ROCM_OK;
}

// Frees every buffer the cache holds.  Work that may still use them is drained first.
int drop_cache(dfdx_rocm_ctx *ctx) {
    CtxLock lock(ctx->mu);
    if (ctx->cache.empty()) return DFDX_ROCM_OK;
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    hipError_t first = free_retired(ctx);
    for (auto &kv : ctx->cache)
        for (void *p : kv.second) {
            const hipError_t e = hipFree(p);
            if (first == hipSuccess) first = e;
        }
    ctx->cache.clear();
    ctx->cache_bytes = 0;
    return (int)first;
}

struct Plan;
size_t partials_bytes(const GemmProblem &p, const Plan &plan, Realign *ra = nullptr);

struct Plan {
    int kernel, variant, splits;
    // An LDS-DMA variant on copies of the operands that are off its grid (realign.hip).  Where the copies cannot have their space the
    // register-staged tile `staged` runs on the operands as they lie, with the same splits: every 16-bit tile walks the
    // contraction in the same order, so it leaves the same bits.  Where its partial sums have no space either: the plain plan.
    bool realign = false;
    int staged = 0;
    int plain_kernel = 0, plain_variant = 0, plain_splits = 1;
    GemmCut cut;
    bool pieces_asked = false;  // the caller asked for this number of pieces
};

// Rank-1 updates and k = 2 stream their rows on the vector ALUs; from k = 3 on the matrix-core form of the thin
// contraction is the faster one wherever it applies (f32 4096 x 8 x 4096: 42.5 against 16.7 us; at k = 2 the vector ALUs
// are level or up to 10 % ahead).
inline bool use_rank1(const GemmProblem &p) {
    return rank1_supported(p) && !(p.k >= 3 && thin_mfma_supported(p));
}

// The bandwidth-bound kernels (`Plan::variant` of a DFDX_ROCM_KERNEL_GEMV plan).
enum { BW_NONE = 0, BW_RANK1 = 1, BW_GEMV_MULTI = 2, BW_GEMV = 3, BW_THIN_MFMA = 4, BW_ROWS = 5 };

// Which of them takes `p`, if any.  `plain_order`: the caller asked for the contraction order of the tiled kernels
// (DFDX_ROCM_GEMM_NO_SPLIT_K: the broadcast-rhs forward and grad_lhs, whose results must equal those of the batched
// product of the same slices bit for bit, matmul/mod.rs:460-473).  The vector-product kernels cut k into grid slices
// and sum inside a slice in an order of their own, and the vector-ALU form of the thin contraction sums by fused
// multiply-adds, so none of them qualifies; a rank-1 update has nothing to order, and the matrix-core form of the thin
// contraction walks k exactly as the tiles do.
int bandwidth_kernel(const GemmProblem &p, bool plain_order) {
    if (plain_order) {
        if (p.k == 1 && rank1_supported(p)) return BW_RANK1;
        return thin_mfma_supported(p) ? BW_THIN_MFMA : BW_NONE;
    }
    if (use_rank1(p)) return BW_RANK1;
    if (gemv_multi_supported(p)) return BW_GEMV_MULTI;
    if (gemv_supported(p)) return BW_GEMV;
    return thin_mfma_supported(p) ? BW_THIN_MFMA : BW_NONE;
}

// The same with the rows form of gemv_multi.hip among them.  Of the forms for several vectors those that keep their sums in the vector ALUs
// are weighed against the rows form and the matrix-core plans by estimated time (the tiles stream a large [k][n] matrix faster); the rows
// form has no rival (1 - 16 vectors against 512 - 16384 rows and columns, 245 products: 1.47 times as fast as the best plan
// without it in the mean, 4 x 4091 x 4093 f16 36.5 -> 10.1 us, f32 36.9 -> 15.7, 8 x 4288 x 4288 bf16 14 -> 11) but the
// small-product kernel, by estimated time, on rows that lie on the 16-byte grid of a matrix below 8 MB (up to 11 % there, either
// way: 8 x 520 x 2635 bf16 3.7 and 4.2 us, 16 x 2048 x 2048 7.0 and 6.8), and but the LDS-DMA tiles (`tiles_only`) on such rows of a larger one in
// 16 bits, which a vector more costs nothing (16 x 14208 x 8384 bf16 84 us and 52, 16 x 10304 x 4355 f16 43 and 22, 8 x 7680 x 8960 36 and 30; 57
// products of 1 - 16 rows: 1.11 times the better of the two on this form alone, 1.02 with 0.85 of its estimate against theirs, 0.95 from 96 MB on); the
// others have none.
// `seconds`: the estimate where it has rivals, else 0.
int bandwidth_plan(const GemmProblem &p, bool plain_order, bool may_rows, double *seconds, bool *tiles_only) {
    *seconds = 0.0;
    *tiles_only = false;
    const int bw = bandwidth_kernel(p, plain_order);
    if (bw == BW_GEMV_MULTI) *seconds = gemv_multi_time(p);
    if ((bw != BW_NONE && bw != BW_GEMV_MULTI) || !may_rows || !gemv_rows_supported(p)) return bw;
    // (the other forms take 1.1 times their estimate, 4 x 2048 x 2048 f32 10.2 us and 8.6 as rows, but on matrices that no cache
    // holds: 8 x 16384 x 16384 f32 218 and 240; in 16 bits they are ahead of all others there, 2 x 12920 x 12288 f16 57 us, 68 as rows, 71 on the ring
    // tiles, 8 x 11008 x 16768 89, 103 and 101)
    const double t = gemv_rows_time(p), bytes = (double)std::max(p.m, p.n) * (double)p.k * (double)dtype_size(p.dtype);
    if (bw == BW_GEMV_MULTI && bytes >= 268435456.0 && dtype_size(p.dtype) == 2) {
        *seconds = 0.0;
        return bw;
    }
    if (bw == BW_GEMV_MULTI && t >= (bytes < 268435456.0 ? 1.1 : 1.0) * *seconds) return bw;
    *tiles_only = bytes >= 8e6 && mfma16dma_supported(p, mfma16dma_variant_count());
    *seconds = *tiles_only ? (bytes < 96e6 ? 0.85 : 0.95) * t : bytes < 8e6 && p.k * (int64_t)dtype_size(p.dtype) % 16 == 0 ? t : 0.0;
    return BW_ROWS;
}

const char *bandwidth_kernel_name(const GemmProblem &p, int which) {
    switch (which) {
    case BW_RANK1: return p.k == 1 ? "rank1" : "thin_k";
    case BW_GEMV_MULTI: return "gemv_multi";
    case BW_GEMV: return "gemv";
    case BW_THIN_MFMA: return "thin_k_mfma";
    case BW_ROWS: return "gemv_rows";
    default: return "none";
    }
}

// `seconds` (may be null): the estimate behind an automatic plan of a 16-bit product that the matrix-core tiles take, else 0.
int make_plan(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *d, const GemmProblem &p, Plan *plan, double *seconds = nullptr) {
    if (seconds) *seconds = 0.0;
    const bool is16 = p.dtype == DT_F16 || p.dtype == DT_BF16;
    const bool is32 = p.dtype == DT_F32, is64 = p.dtype == DT_F64;
    // split-k: 1 = never (NO_SPLIT_K), n = forced by the caller, 0 = let the planner decide
    const int forced_splits = (d->flags & DFDX_ROCM_GEMM_NO_SPLIT_K) ? 1 : ((d->flags >> 8) & 0xff);
    switch (d->kernel) {
    case DFDX_ROCM_KERNEL_GENERIC:
        *plan = {DFDX_ROCM_KERNEL_GENERIC, 0, 1};
        return DFDX_ROCM_OK;
    case DFDX_ROCM_KERNEL_GEMV: {  // the bandwidth-bound kernels, forced: the caller's choice outranks the order flag
        // (the rows form by its id, or where no other form takes the product)
        const int other = bandwidth_kernel(p, false), bw = (!other || d->variant == BW_ROWS) && gemv_rows_supported(p) ? BW_ROWS : other;
        if (!bw) return DFDX_ROCM_ERR_UNSUPPORTED;
        *plan = {DFDX_ROCM_KERNEL_GEMV, bw, 1};
        return DFDX_ROCM_OK;
    }
    case DFDX_ROCM_KERNEL_MFMA: {
        int v = d->variant;
        if (is16 && (v == 0 || (v >= mfma16_dma_first_variant() && v != mfma16_small_variant()))) {  // LDS-DMA family: tile and split count together
            int dv = 0, splits = 1;
            GemmCut cut;
            mfma16dma_plan_split(p, ctx->compute_units, v ? v - mfma16_dma_first_variant() + 1 : 0, forced_splits, &dv, &splits, nullptr, &cut);
            if (dv) {
                *plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits};
                plan->cut = cut;
                return DFDX_ROCM_OK;
            }
            if (v) return DFDX_ROCM_ERR_UNSUPPORTED;
        }
        if (v == 0)
            v = is16 ? mfma16_pick_variant(p, ctx->compute_units)
                     : is32 ? mfma32_pick_variant(p, ctx->compute_units, forced_splits) : is64 ? mfma64_pick_variant(p, ctx->compute_units) : 0;
        const bool ok = is16 ? mfma16_supported(p, v) : is32 ? mfma32_supported(p, v) : is64 ? mfma64_supported(p, v) : false;
        if (!ok) return DFDX_ROCM_ERR_UNSUPPORTED;
        *plan = {DFDX_ROCM_KERNEL_MFMA, v,
                 is32 ? mfma32_plan_splits(p, v, ctx->compute_units, forced_splits)
                      : is16 ? mfma16_plan_splits(p, v, ctx->compute_units, forced_splits) : 1};
        return DFDX_ROCM_OK;
    }
    case DFDX_ROCM_KERNEL_AUTO:
        break;
    default:
        return DFDX_ROCM_ERR_INVALID_ARG;
    }
    // The bandwidth-bound kernels first.
    double t_bw = 1e300;
    bool tiles_only = false;
    const int bw = bandwidth_plan(p, (d->flags & DFDX_ROCM_GEMM_NO_SPLIT_K) != 0, !forced_splits, &t_bw, &tiles_only);
    if (tiles_only) {
        // what the tiles' estimates lack on few rows: the matrix streams past the caches once (238 MB 52 us for an estimate of 32)
        const double t_stream = 3.0e-6 + (double)(p.m + p.n) * (double)p.k * (double)dtype_size(p.dtype) / 4.6e12;
        int dv = 0, splits = 1;
        double t_dma = 1e300;
        GemmCut cut;
        mfma16dma_plan_split(p, ctx->compute_units, 0, 0, &dv, &splits, &t_dma, &cut);
        *plan = {DFDX_ROCM_KERNEL_GEMV, bw, 1};
        if (dv && std::max(t_dma, t_stream) < t_bw) {
            *plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits};
            plan->cut = cut;
        }
        return DFDX_ROCM_OK;
    }
    if (bw && t_bw == 0.0) {
        *plan = {DFDX_ROCM_KERNEL_GEMV, bw, 1};
        return DFDX_ROCM_OK;
    }
    if (!bw) t_bw = 1e300;
    const Plan bw_plan = {DFDX_ROCM_KERNEL_GEMV, bw, 1};
    // The small-product kernel where its estimate beats the family's (the f32 family weighs it among its own variants);
    // not where the caller fixed the order of the contraction.
    const bool may_small = forced_splits == 0 && (is16 || is64) && small_supported(p);
    const double t_small = may_small ? small_time(p, ctx->compute_units) : 1e300;
    // Against the ring tiles: a short contraction that four waves share takes less than the estimate, which is of long ones, most of all where
    // values that lie across k are gathered (512 x 208 x 200 tn f16 4.2 us for 4.9, the ring 5.1 for 4.5; 104 x 64 x 384 tn 3.3 and 4.0, 256 x 96 x
    // 1971 nt 3.9 and 4.6; of 82 products that the ring had taken from this kernel 15 were slower there by 4 - 24 %, all of them such; none that
    // adds to C).
    const double t_short = is16 && p.k < 256 && !p.accumulate ? (p.a_cs != 1 || p.b_rs != 1 ? 1.0e-6 : 0.4e-6) : 0.0;
    const Plan small_plan = {DFDX_ROCM_KERNEL_MFMA, is16 ? mfma16_small_variant() : mfma64_small_variant(), 1};
    Plan ring_plan = {};
    double t_ring = 1e300;
    bool narrow = false;
    if (is16) {
        int dv = 0, splits = 1;
        double t_dma = 1e300;
        GemmCut cut;
        mfma16dma_plan_split(p, ctx->compute_units, 0, forced_splits, &dv, &splits, &t_dma, &cut);
        bool only_ring = dv && mfma16dma_takes_any_k(dv);
        for (int v = 1; only_ring && v <= mfma16dma_variant_count(); v++) only_ring = mfma16dma_takes_any_k(v) || !mfma16dma_supported(p, v);
        // (a C on the 8-byte grid only: of the persistent tiles one stores it as it is, the 128 x 64 one; all others with the
        // element-aligned stores of the plans below.  2048 x 1024 x 50260 f16 342 us and 208, 4096 x 1024 x 4092 51 and 36.)
        const int64_t ldc = p.m == 1 ? p.n : p.c_rs;
        narrow = dv && (p.n % 8 || ldc % 8 || ((uintptr_t)p.c & 15u) || p.c_b1 % 8 || p.c_b2 % 8);
        if (only_ring || narrow) {  // (k off the tile or C off the grid: weighed against the families below, copies among them)
            t_ring = t_dma;
            ring_plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits};
            ring_plan.cut = cut;
            int skinny_splits = 1;
            double t_skinny = 1e300;
            const int sv = !only_ring ? mfma16_skinny_plan(p, ctx->compute_units, forced_splits, &skinny_splits, &t_skinny) : 0;
            if (sv && t_skinny < t_ring) {
                t_ring = t_skinny;
                ring_plan = {DFDX_ROCM_KERNEL_MFMA, sv, skinny_splits};
            }
        } else if (dv) {
            *plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits};
            plan->cut = cut;
            if (t_small - (mfma16dma_takes_any_k(dv) ? t_short : 0.0) < t_dma) *plan = small_plan;
            double t_best = std::min(t_small, t_dma);
            int skinny_splits = 1;
            double t_skinny = 1e300;
            if (const int sv = mfma16_skinny_plan(p, ctx->compute_units, forced_splits, &skinny_splits, &t_skinny)) {
                if (t_skinny < t_best) {
                    *plan = {DFDX_ROCM_KERNEL_MFMA, sv, skinny_splits};
                    t_best = t_skinny;
                }
            }
            if (t_bw < t_best) *plan = bw_plan;
            if (seconds) *seconds = std::min(t_best, t_bw);
            return DFDX_ROCM_OK;
        }
    }
    double t_family = 1e300;
    int v = is16 ? mfma16_pick_variant(p, ctx->compute_units)
                 : is32 ? mfma32_pick_variant(p, ctx->compute_units, forced_splits, &t_family) : is64 ? mfma64_pick_variant(p, ctx->compute_units) : 0;
    if (v > 0) {
        *plan = {DFDX_ROCM_KERNEL_MFMA, v,
                 is32 ? mfma32_plan_splits(p, v, ctx->compute_units, forced_splits)
                      : is16 ? mfma16_plan_splits(p, v, ctx->compute_units, forced_splits) : 1};
        if (!is32) t_family = is16 ? mfma16_staged_time(p, v, plan->splits, ctx->compute_units) : mfma64_time(p, v, ctx->compute_units);
        Realign ra;
        ra.off_grid = ra.off_grid_k = 0;
        const bool realignable = is16 && plan_realign(p, &ra);
        // The small-product kernel's estimate holds for rows on the 16-byte grid; an operand stored along k whose rows are off it
        // is gathered value by value (f16, 76 x 6298 x 100, both such: 62 us for an estimate of 13, 13 us in 64 x 64 tiles;
        // 118 x 2413 x 481, one such: 20 against 13 us).
        const double t_small_here = realignable && ra.off_grid_k ? 2.5e-6 + (t_small - 2.5e-6) * (1.0 + 1.9 * ra.off_grid_k) : t_small;
        if (may_small && t_small_here < t_family) *plan = small_plan;
        if (t_bw < std::min(t_small_here, t_family)) *plan = bw_plan;
        // Operands off the grid of the LDS-DMA kernels: copies of them and those kernels, where the two together are expected
        // to be faster.  The register-staged family's estimate ranks its own tiles; against the clock the 64 x 64 tile runs at
        // 0.6 of it with operands on the 16-byte grid and at 0.9 - 1.6 off it, the larger tiles at about 1 and 1.4 - 3, and those
        // write a large C at 2.2 TB/s.  f16, staged and on copies: 2048 x 50257 x 1024 563 and 325 us, 4095^3 293 and 143, 1315 x
        // 2340 x 3033 150 and 52, 530 x 3231 x 1057 84 and 28, 6928 x 106 x 7330 80 and 43; and where the line leaves the
        // staged kernels: 1000^3 12.0 and 18.8, 304 x 611 x 4120 11.0 and 16.4, 448 x 315 x 4890 13.2 and 14.5.  In pieces the larger tiles
        // take 1.45 of the estimate on the grid and 2.1 - 2.9 off it (84 products; 3778 x 7038 x 256 bf16 nn 104 us for 37, 43 on copies), and
        // 2.2 - 3.5 where only C is off it (2304 x 576 x 8188 f16 nt + C 70 us for 29, the 128 x 64 LDS-DMA tile 40).
        double t_copies = 1e300;
        const bool small_tile = v == mfma16_skinny_variant();
        const bool large_pieces = is16 && !small_tile && mfma16_plan_splits(p, v, ctx->compute_units, forced_splits) > 1;
        const double t_staged = t_family * (small_tile ? (ra.off_grid ? 1.0 : 0.6) : large_pieces ? (ra.off_grid ? 2.4 : 1.45) : narrow ? 2.2 : ra.off_grid ? 1.4 : 0.95) +
                                (small_tile ? 0.0 : 2.0 * (double)p.m * (double)p.n * (double)(p.reduce ? 1 : p.nb1 * p.nb2) / 2.2e12);
        const double t_uncopied = std::min(std::min(t_small_here, t_staged), t_bw);
        if (realignable && ra.seconds + mfma16dma_least_time() < t_uncopied) {
            int dv = 0, splits = 1;
            GemmCut cut;
            mfma16dma_plan_split(ra.problem, ctx->compute_units, 0, forced_splits, &dv, &splits, &t_copies, &cut);
            // (a product whose plan without copies fits the fixed scratch array fits it in this form too: see dfdx_rocm_gemm_noalloc)
            const size_t piece = mfma16_workspace_bytes(p, v, 2) / 2, most = DFDX_ROCM_NOALLOC_SCRATCH_BYTES;
            if (dv && splits > 1 && !forced_splits && piece * (size_t)splits > most && partials_bytes(p, *plan) <= most)
                mfma16dma_plan_split(ra.problem, ctx->compute_units, 0, (int)std::max<size_t>(1, most / piece), &dv, &splits, &t_copies, &cut);
            // (copies are not taken for a gain within the estimates' error)
            t_copies = dv ? t_copies + ra.seconds + (mfma16dma_takes_any_k(dv) ? 0.0 : splits > 1 ? 6.5e-6 : 1.0e-6) : 1e300;
            if (t_copies < t_uncopied) {
                const Plan plain = *plan;
                *plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits, true, v, plain.kernel, plain.variant, plain.splits, cut};
            }
        }
        // (on operands in place with k off 64 the staged tiles run at 0.83 - 1.06 of the estimate: 528 x 1024 x 1325 f16 21.4 us for 25.6,
        // 2304 x 128 x 1534 in three pieces 16.2 for 15.3; the ring 9.4 both; not so the larger ones in pieces, nor where C alone
        // is off the grid)
        const double t_place = large_pieces || (narrow && !small_tile) ? t_staged : 0.85 * t_family;
        const double t_plan = plan->realign ? t_copies : plan->kernel == DFDX_ROCM_KERNEL_GEMV ? t_bw : plan->variant == v ? t_place : t_small_here - t_short;
        if (t_ring <= t_plan) *plan = ring_plan;
        if (seconds && is16) *seconds = std::min(t_ring, t_plan);
        return DFDX_ROCM_OK;
    }
    if (t_ring < std::min(t_small - t_short, t_bw)) {
        *plan = ring_plan;
        return DFDX_ROCM_OK;
    }
    if (bw) {  // no tiled kernel takes these strides, the multi-vector kernel does
        *plan = t_small < t_bw ? small_plan : bw_plan;
        return DFDX_ROCM_OK;
    }
    // no tiled kernel takes these strides: the small-product kernel takes any, up to the size where 16 x 16 tiles pay
    if (may_small && (double)p.m * (double)p.n * (double)p.k <= 134217728.0) {
        *plan = small_plan;
        return DFDX_ROCM_OK;
    }
    *plan = {DFDX_ROCM_KERNEL_GENERIC, 0, 1};
    return DFDX_ROCM_OK;
}

// Where the partial sums of a split plan go: the context's own buffer (grown on demand), or -- `static_scratch` --
// the device's fixed scratch array, in which case nothing is allocated and a plan that needs more is refused.
int partials_buffer(dfdx_rocm_ctx *ctx, size_t need, bool static_scratch, float **out) {
    if (static_scratch) {
        if (need > (size_t)DFDX_ROCM_NOALLOC_SCRATCH_BYTES) return DFDX_ROCM_ERR_SCRATCH_TOO_SMALL;
        if (!ctx->static_scratch) return DFDX_ROCM_ERR_INVALID_ARG;
        *out = (float *)ctx->static_scratch;
        return DFDX_ROCM_OK;
    }
    if (int rc = ensure_workspace(ctx, need)) return rc;
    *out = (float *)ctx->workspace;
    return DFDX_ROCM_OK;
}

// The f32 partial sums `plan` needs for `p`, in bytes (0: none), and, behind them, the copies of its operands.
size_t partials_bytes(const GemmProblem &p, const Plan &plan, Realign *ra) {
    if (plan.realign) {
        Realign here;
        if (!ra) ra = &here;
        if (!plan_realign(p, ra)) return 0;
        return ((mfma16dma_workspace_bytes(ra->problem, plan.variant - mfma16_dma_first_variant() + 1, plan.splits) + 255) & ~(size_t)255) +
               ra->a_bytes + ra->b_bytes;
    }
    if (plan.kernel == DFDX_ROCM_KERNEL_MFMA && plan.splits > 1)
        return p.dtype == DT_F32 ? mfma32_workspace_bytes(p, plan.variant, plan.splits)
               : plan.variant < mfma16_dma_first_variant()
                   ? mfma16_workspace_bytes(p, plan.variant, plan.splits)
                   : mfma16dma_workspace_bytes(p, plan.variant - mfma16_dma_first_variant() + 1, plan.splits);
    if (plan.kernel == DFDX_ROCM_KERNEL_GEMV && plan.variant == BW_GEMV_MULTI) return gemv_multi_workspace_bytes(p);
    if (plan.kernel == DFDX_ROCM_KERNEL_GEMV && plan.variant == BW_GEMV) return gemv_workspace_bytes(p);
    if (plan.kernel == DFDX_ROCM_KERNEL_GEMV && plan.variant == BW_ROWS) return plan.splits ? gemv_rows_workspace_bytes(p) : 0;  // (0: in one piece)
    return 0;
}

// Space that the call could do without is not asked for while the stream is being captured into a graph, nor where as much has been
// refused since memory was last freed.
bool capturing(dfdx_rocm_ctx *ctx) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &status) != hipSuccess) (void)hipGetLastError();
    return status != hipStreamCaptureStatusNone;
}
bool grow_for_copies(dfdx_rocm_ctx *ctx, int (*ensure)(dfdx_rocm_ctx *, size_t), size_t bytes) {
    if (bytes >= ctx->copies_refused || capturing(ctx)) return false;
    if (ensure(ctx, bytes) == DFDX_ROCM_OK) return true;
    ctx->copies_refused = bytes;
    return false;
}

// Makes sure the partial sums of `plan` have a place, BEFORE the caller resolves pending zero fills among the operands:
// a call that is refused here (scratch too small, out of memory) must leave every declaration as it found it.
// A plan with copies of operands that cannot have their space -- they do not fit the fixed scratch array, memory has run out, or
// the stream is being captured -- is changed to one without them (see Plan).
int reserve_partials(dfdx_rocm_ctx *ctx, const GemmProblem &problem, Plan &plan, bool static_scratch) {
    GemmProblem p = problem;
    p.compute_units = ctx->compute_units;
    float *unused = nullptr;
    if (plan.realign) {
        CtxLock lock(ctx->mu);
        auto room = [&](size_t need) {
            if (static_scratch) return need <= (size_t)DFDX_ROCM_NOALLOC_SCRATCH_BYTES;
            return need <= ctx->workspace_bytes || grow_for_copies(ctx, ensure_workspace, need);
        };
        if (room(partials_bytes(p, plan))) return DFDX_ROCM_OK;
        const Plan plain = {plan.plain_kernel, plan.plain_variant, plan.plain_splits};
        plan = {DFDX_ROCM_KERNEL_MFMA, plan.staged, plan.splits};
        if (room(partials_bytes(p, plan))) return DFDX_ROCM_OK;
        plan = plain;
    }
    const size_t need = partials_bytes(p, plan);
    // Products that kernels without partial sums had before the ring tiles and the rows form, and any that f32 tiles are planned to take in
    // pieces: captured with no space they run in one piece.  An f32 product keeps the pieces that the caller asked for.
    const bool ring = plan.kernel == DFDX_ROCM_KERNEL_MFMA &&
                      (p.dtype == DT_F32 || ((p.dtype == DT_F16 || p.dtype == DT_BF16) && plan.variant >= mfma16_dma_first_variant() &&
                                             plan.variant != mfma16_small_variant() && mfma16dma_takes_any_k(plan.variant - mfma16_dma_first_variant() + 1)));
    const bool rows = plan.kernel == DFDX_ROCM_KERNEL_GEMV && plan.variant == BW_ROWS;
    if (need && !static_scratch && (ring || rows)) {
        CtxLock lock(ctx->mu);
        if (need > ctx->workspace_bytes && capturing(ctx)) {
            if (plan.pieces_asked && p.dtype == DT_F32) return DFDX_ROCM_ERR_SCRATCH_TOO_SMALL;
            plan.splits = ring ? 1 : 0;
            return DFDX_ROCM_OK;
        }
    }
    return need ? partials_buffer(ctx, need, static_scratch, &unused) : DFDX_ROCM_OK;
}

int run_plan(dfdx_rocm_ctx *ctx, const GemmProblem &problem, const Plan &plan, bool static_scratch = false) {
    CtxLock lock(ctx->mu);  // a split plan is two launches around the shared workspace
    GemmProblem p = problem;
    p.splits = 1;
    p.workspace = nullptr;
    p.compute_units = ctx->compute_units;
    Realign ra;
    if (const size_t need = partials_bytes(p, plan, &ra)) {
        if (int rc = partials_buffer(ctx, need, static_scratch, &p.workspace)) return rc;
        if (plan.realign) {
            ra.problem.workspace = p.workspace;
            HIP_TRY(launch_realign(p, &ra, (char *)p.workspace + (need - ra.a_bytes - ra.b_bytes), ctx->stream));
        }
    }
    if (plan.realign) p = ra.problem;
    if (plan.kernel == DFDX_ROCM_KERNEL_MFMA && plan.splits > 1) p.splits = plan.splits;
    p.cut = plan.cut;
    hipError_t e;
    switch (plan.kernel) {
    case DFDX_ROCM_KERNEL_GENERIC: e = launch_generic(p, ctx->stream); break;
    case DFDX_ROCM_KERNEL_GEMV:
        e = plan.variant == BW_RANK1 ? launch_rank1(p, ctx->stream)
            : plan.variant == BW_GEMV_MULTI ? launch_gemv_multi(p, ctx->stream)
            : plan.variant == BW_GEMV ? launch_gemv(p, ctx->stream)
            : plan.variant == BW_ROWS ? launch_gemv_rows(p, ctx->stream)
            : plan.variant == BW_THIN_MFMA ? launch_thin_mfma(p, ctx->stream) : hipErrorInvalidValue;
        break;
    case DFDX_ROCM_KERNEL_MFMA:
        e = (p.dtype == DT_F32) ? launch_mfma32(p, plan.variant, ctx->stream)
                                : (p.dtype == DT_F64) ? launch_mfma64(p, plan.variant, ctx->stream) : launch_mfma16(p, plan.variant, ctx->stream);
        break;
    default: return DFDX_ROCM_ERR_INVALID_ARG;
    }
    return (int)e;
}

// Deferred zero fills among the operands: inputs are filled now; an accumulation that covers the whole of a pending C
// becomes a plain store (`may_overwrite`), which leaves the same bits as 0 + value.
int settle_operands(dfdx_rocm_ctx *ctx, GemmProblem *p, bool may_overwrite) {
    if (ctx->pending_count.load(std::memory_order_acquire) == 0) return DFDX_ROCM_OK;
    if (p->k > 0) {
        if (int e = settle(ctx, p->a)) return e;
        if (int e = settle(ctx, p->b)) return e;
    }
    if (int e = settle(ctx, p->bias)) return e;
    if (int e = settle(ctx, p->with)) return e;
    const int64_t ext[4] = {p->reduce ? 1 : p->nb1, p->reduce ? 1 : p->nb2, p->m, p->n};
    const int64_t str[4] = {p->c_b1, p->c_b2, p->c_rs, p->c_cs};
    const size_t es = p->dtype == DT_F64 ? 8 : p->dtype == DT_F32 ? 4 : 2;
    bool fresh = false;
    if (int e = settle_output(ctx, p->c, dense_bytes(4, ext, str, es), p->accumulate, may_overwrite ? &fresh : nullptr)) return e;
    if (fresh) p->accumulate = false;
    return DFDX_ROCM_OK;
}

}  // namespace

namespace {
// Which plans apply p.extra on the way into C.
bool extra_supported(const GemmProblem &p, const Plan &plan) {
    if (p.extra == EXTRA_NONE) return true;
    if (plan.realign) return false;
    if (plan.kernel != DFDX_ROCM_KERNEL_MFMA || p.nb1 * p.nb2 != 1) return false;
    const bool is16 = p.dtype == DT_F16 || p.dtype == DT_BF16;
    if (is16 && plan.variant == mfma16_small_variant()) return true;
    if (p.dtype == DT_F64 && plan.variant == mfma64_small_variant()) return true;
    if (is16 && plan.variant >= mfma16_dma_first_variant()) {
        GemmProblem whole = p;
        whole.cut = plan.cut;
        return mfma16dma_extra_supported(whole, plan.variant - mfma16_dma_first_variant() + 1, plan.splits);
    }
    return plan.splits > 1;  // the reduce kernel does it
}

// A product with its plan made: space, pending fills, launches.
int run_planned(dfdx_rocm_ctx *ctx, GemmProblem &p, Plan &plan, bool static_scratch = false) {
    if (int e = reserve_partials(ctx, p, plan, static_scratch)) return e;
    if (int e = settle_operands(ctx, &p, /*may_overwrite=*/true)) return e;
    return run_plan(ctx, p, plan, static_scratch);
}

// The same with the sums that `p` asks for (ksum) where the plan can take them along: *fused.
int run_with_colsum(dfdx_rocm_ctx *ctx, GemmProblem &p, Plan &plan, bool *fused) {
    if (int e = reserve_partials(ctx, p, plan, false)) return e;
    if (int e = settle_operands(ctx, &p, /*may_overwrite=*/true)) return e;
    bool can = p.ksum && plan.kernel == DFDX_ROCM_KERNEL_MFMA && !plan.realign;
    if (can && (p.dtype == DT_F16 || p.dtype == DT_BF16))
        can = plan.variant == mfma16_small_variant()
                  ? small_ksum_supported(p)
                  : plan.variant >= mfma16_dma_first_variant() &&
                        mfma16dma_ksum_supported(p, plan.variant - mfma16_dma_first_variant() + 1, plan.splits);
    else if (can && p.dtype == DT_F32)
        can = plan.splits <= 1 && mfma32_ksum_supported(p, plan.variant);
    else if (can && p.dtype == DT_F64)
        can = plan.variant == mfma64_small_variant() && small_ksum_supported(p);
    else
        can = false;
    if (can) {
        bool fresh = false;
        const int64_t len = p.ksum_of == KSUM_OF_A ? p.m : p.n;
        if (int e = settle_output(ctx, p.ksum, (size_t)len * dtype_size(p.dtype), true, &fresh)) return e;
        p.ksum_accumulate = !fresh;
        *fused = true;
    } else {
        p.ksum = nullptr;
        p.ksum_of = KSUM_NONE;
    }
    return run_plan(ctx, p, plan);
}

}  // namespace

namespace dfdx_rocm {

// What gemm_beyond asks of a product: C and `with` are one contiguous matrix each, which the separate ops walk.
static bool beyond_ok(const GemmProblem &p, int extra, const void *with) {
    return p.nb1 * p.nb2 == 1 && p.c_cs == 1 && p.c_rs == p.n && (!extra || (p.accumulate != 0) == (extra == EXTRA_FROM)) && (extra <= EXTRA_RELU || with);
}

static int run_beyond(dfdx_rocm_ctx *ctx, GemmProblem &p, Plan &plan, int extra, const void *with) {
    if (int e = reserve_partials(ctx, p, plan, false)) return e;
    p.extra = extra;
    p.with = with;
    const int64_t len = p.m * p.n;
    const bool whole = extra_supported(p, plan);
    if (!whole) {
        if (extra == EXTRA_FROM)
            if (int e = dfdx_rocm_copy_d2d(ctx, p.c, with, (size_t)len * dtype_size(p.dtype))) return e;
        p.extra = EXTRA_NONE;
    }
    if (int e = settle_operands(ctx, &p, /*may_overwrite=*/extra != EXTRA_FROM)) return e;
    if (int e = run_plan(ctx, p, plan)) return e;
    if (whole) return DFDX_ROCM_OK;
    switch (extra) {
    case EXTRA_RELU: return dfdx_rocm_relu_forward(ctx, p.dtype, len, p.c, p.c);
    case EXTRA_RESIDUAL: return dfdx_rocm_add_forward(ctx, p.dtype, len, p.c, with, p.c);
    case EXTRA_MASK: return relu_mask(ctx, p.dtype, len, with, p.c);
    default: return DFDX_ROCM_OK;
    }
}

int gemm_beyond(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc, int extra, const void *with) {
    if (int e = bind(ctx)) return e;
    GemmProblem p;
    if (int e = make_problem(desc, &p)) return e;
    if (p.m == 0) return DFDX_ROCM_OK;
    if (!beyond_ok(p, extra, with)) return DFDX_ROCM_ERR_INVALID_ARG;
    Plan plan;
    if (int e = make_plan(ctx, desc, p, &plan)) return e;
    return run_beyond(ctx, p, plan, extra, with);
}

// Bytes that the matrices of one operand span, matrix by matrix where they lie anywhere (`batches`), else together.
struct Spans {
    uintptr_t lo[3], hi[3];
    int count = 0;
    void add(const void *ptr, size_t es, int64_t rows, int64_t rs, int64_t cols, int64_t cs, const GemmProblem &p, int64_t b1, int64_t b2) {
        if (!ptr) return;
        const int64_t apart = p.batches > 0 ? p.batches : 1;
        for (int64_t i = 0; i < apart && i < 3; i++) {
            int64_t from = p.batches > 0 ? (i / p.nb2) * b1 + (i % p.nb2) * b2 : 0, to = from;
            auto axis = [&](int64_t n, int64_t stride) { (stride < 0 ? from : to) += (n - 1) * stride; };
            axis(rows, rs);
            axis(cols, cs);
            if (p.batches <= 0) {
                axis(p.nb1, b1);
                axis(p.nb2, b2);
            }
            lo[count] = (uintptr_t)ptr + (uintptr_t)(from * (int64_t)es);
            hi[count++] = (uintptr_t)ptr + (uintptr_t)((to + 1) * (int64_t)es);
        }
    }
    bool meets(const Spans &o) const {
        for (int i = 0; i < count; i++)
            for (int j = 0; j < o.count; j++)
                if (lo[i] < o.hi[j] && o.lo[j] < hi[i]) return true;
        return false;
    }
};

// May the two products run side by side?  Nothing that one writes may be read or written by the other.
static bool independent(const GemmProblem &p, const GemmProblem &q) {
    auto written = [](const GemmProblem &g, Spans(&s)[2]) {
        const size_t es = dtype_size(g.dtype);
        s[0].add(g.c, es, g.m, g.c_rs, g.n, g.c_cs, g, g.reduce ? 0 : g.c_b1, g.reduce ? 0 : g.c_b2);
        s[1].add(g.ksum, es, 1, 0, g.ksum_of == KSUM_OF_B ? g.n : g.m, 1, g, g.ksum_b1, g.ksum_b2);
    };
    auto read = [](const GemmProblem &g, Spans(&s)[4]) {
        const size_t es = dtype_size(g.dtype);
        s[0].add(g.a, es, g.m, g.a_rs, g.k, g.a_cs, g, g.a_b1, g.a_b2);
        s[1].add(g.b, es, g.k, g.b_rs, g.n, g.b_cs, g, g.b_b1, g.b_b2);
        s[2].add(g.with, es, g.m, g.c_rs, g.n, g.c_cs, g, g.reduce ? 0 : g.c_b1, g.reduce ? 0 : g.c_b2);
        s[3].add(g.bias, es, 1, 0, g.bias_mode == BIAS_PER_ROW ? g.m : g.n, 1, g, g.bias_b1, g.bias_b2);
    };
    Spans wp[2], wq[2], rp[4], rq[4];
    written(p, wp);
    written(q, wq);
    read(p, rp);
    read(q, rq);
    for (const Spans &w : wp) {
        for (const Spans &o : wq)
            if (w.meets(o)) return false;
        for (const Spans &o : rq)
            if (w.meets(o)) return false;
    }
    for (const Spans &w : wq)
        for (const Spans &o : rp)
            if (w.meets(o)) return false;
    return true;
}

// A call's product and its plan, which is made once, when it is first asked for.
struct Product {
    const dfdx_rocm_gemm_desc *desc;
    GemmProblem p;
    Plan plan;
    double seconds = 0.0;
    bool planned = false;
    int need_plan(dfdx_rocm_ctx *ctx) {
        if (planned) return DFDX_ROCM_OK;
        if (int e = make_plan(ctx, desc, p, &plan, &seconds)) return e;
        planned = true;
        return DFDX_ROCM_OK;
    }
};

// The tile on which the two products of a backward pass run faster as one launch than as two, 0 if there is none.  Decided from the
// shapes and layouts alone, so that a call that joins more of them (the encoder block's) and the calls it stands for agree.
static int ring_pair_tile(dfdx_rocm_ctx *ctx, Product &one, Product &two) {
    if ((one.p.dtype != DT_F16 && one.p.dtype != DT_BF16) || one.desc->kernel != DFDX_ROCM_KERNEL_AUTO || two.desc->kernel != DFDX_ROCM_KERNEL_AUTO) return 0;
    double together = 1e300;
    const int tile = mfma16_ring_pair_plan(one.p, two.p, ctx->compute_units, &together);
    if (!tile) return 0;
    double t1 = 0.0;
    if (one.p.accumulate) {
        if (one.need_plan(ctx)) return 0;
        t1 = one.seconds;
    } else {  // (the ops that a product with one thing more stands for accumulate)
        GemmProblem added = one.p;
        added.accumulate = 1;
        Plan unused;
        if (make_plan(ctx, one.desc, added, &unused, &t1)) return 0;
    }
    if (two.need_plan(ctx)) return 0;
    // (the second launch and the gap in front of it are not in the estimates)
    return t1 > 0.0 && two.seconds > 0.0 && together < t1 + two.seconds + 1.0e-6 ? tile : 0;
}

// Would the call run on the small-product kernel?  Products that do and share nothing but what they read are one launch
// (launch_small_many), with the bits of several.
static bool plans_small(dfdx_rocm_ctx *ctx, Product &x) {
    if (x.desc->kernel != DFDX_ROCM_KERNEL_AUTO || !small_supported(x.p)) return false;
    if (x.need_plan(ctx) || x.plan.kernel != DFDX_ROCM_KERNEL_MFMA || x.plan.realign) return false;
    const int small = x.p.dtype == DT_F32 ? mfma32_variant_count() : x.p.dtype == DT_F64 ? mfma64_small_variant() : mfma16_small_variant();
    return x.plan.variant == small && (!x.p.ksum || small_ksum_supported(x.p));
}

// Two independent products in one launch: pending fills, then the launch.  `sums` of the second one ride along.
// `tile`: of the ring, 0: the small-product kernel.
static int run_pair(dfdx_rocm_ctx *ctx, GemmProblem p, GemmProblem q, int tile, bool may_overwrite) {
    CtxLock lock(ctx->mu);
    if (int e = settle_operands(ctx, &p, may_overwrite)) return e;
    if (int e = settle_operands(ctx, &q, /*may_overwrite=*/true)) return e;
    if (q.ksum) {
        bool fresh = false;
        if (int e = settle_output(ctx, q.ksum, (size_t)(q.ksum_of == KSUM_OF_A ? q.m : q.n) * dtype_size(q.dtype), true, &fresh)) return e;
        q.ksum_accumulate = !fresh;
    }
    p.compute_units = q.compute_units = ctx->compute_units;
    if (tile) return (int)launch_mfma16_ring_pair(p, q, tile, ctx->stream);
    const GemmProblem both[2] = {p, q};
    return (int)launch_small_many(both, 2, ctx->stream);
}

// Both products as one launch where that is expected to be faster: *done.  When not, nothing has been touched.
static int join_two(dfdx_rocm_ctx *ctx, Product &one, int extra, const void *with, Product &two, bool colsum, bool *done) {
    *done = false;
    if (one.p.m == 0 || two.p.m == 0 || (colsum && !two.p.ksum)) return DFDX_ROCM_OK;
    const int tile = ring_pair_tile(ctx, one, two);
    if (!tile && !(plans_small(ctx, one) && plans_small(ctx, two))) return DFDX_ROCM_OK;
    GemmProblem p = one.p;
    p.extra = extra;
    p.with = with;
    if (!independent(p, two.p)) return DFDX_ROCM_OK;
    *done = true;
    return run_pair(ctx, p, two.p, tile, extra != EXTRA_FROM);
}

// One behind the other.
static int run_apart(dfdx_rocm_ctx *ctx, Product &one, int extra, const void *with, Product &two, bool *fused) {
    if (one.p.m) {
        if (int e = one.need_plan(ctx)) return e;
        if (int e = extra == EXTRA_NONE ? run_planned(ctx, one.p, one.plan) : run_beyond(ctx, one.p, one.plan, extra, with)) return e;
    }
    if (!two.p.m) return DFDX_ROCM_OK;
    if (int e = two.need_plan(ctx)) return e;
    return run_with_colsum(ctx, two.p, two.plan, fused);
}

int gemm_two(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *first, int extra, const void *with, const dfdx_rocm_gemm_desc *second, void *colsum, bool *fused) {
    *fused = false;
    if (int e = bind(ctx)) return e;
    Product one{first}, two{second};
    if (int e = make_problem(first, &one.p)) return e;
    if (int e = make_problem(second, &two.p, colsum)) return e;
    if (one.p.m && extra != EXTRA_NONE && !beyond_ok(one.p, extra, with)) return DFDX_ROCM_ERR_INVALID_ARG;
    bool done = false;
    if (int e = join_two(ctx, one, extra, with, two, colsum != nullptr, &done)) return e;
    if (!done) return run_apart(ctx, one, extra, with, two, fused);
    *fused = colsum != nullptr;
    return DFDX_ROCM_OK;
}

int gemm_pair(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *first, const dfdx_rocm_gemm_desc *second, const void *grad_out, int64_t rows, int64_t cols,
              void *colsum, bool *fused) {
    bool taken = false;  // (without `fused` no sums are asked for)
    if (!fused) {
        fused = &taken;
        colsum = nullptr;
    }
    *fused = false;
    if (int e = bind(ctx)) return e;
    Product x[2] = {{first}, {second}};
    if (int e = make_problem(first, &x[0].p)) return e;
    if (int e = make_problem(second, &x[1].p, colsum)) return e;
    bool done = false;
    if (int e = join_two(ctx, x[0], EXTRA_NONE, nullptr, x[1], colsum != nullptr, &done)) return e;
    if (done) {
        *fused = colsum != nullptr;
        return DFDX_ROCM_OK;
    }
    auto apart = [&]() { return run_apart(ctx, x[0], EXTRA_NONE, nullptr, x[1], fused); };
    // (a copy of less than 4 MB costs little more than its launch)
    const bool off = cols % 64 || rows % 64 || ((uintptr_t)grad_out & 15u);
    if ((first->dtype != DFDX_ROCM_F16 && first->dtype != DFDX_ROCM_BF16) || !off || (double)rows * (double)cols < 2097152.0) return apart();
    Realign ra;
    bool both = true;
    for (Product &i : x) {
        if (i.p.m == 0) {
            both = false;
            continue;
        }
        if (int e = i.need_plan(ctx)) return e;
        // (one matrix each: the batches that a broadcast gradient is summed over step through grad_out by strides of their own)
        both = both && i.plan.realign && i.p.nb1 * i.p.nb2 == 1 && i.p.a != i.p.b && plan_realign(i.p, &ra) && (i.p.a == grad_out ? ra.a || ra.a_last : ra.b || ra.b_last);
    }
    CtxLock lock(ctx->mu);  // the copy lives in the patch buffer until the second product has been launched
    int64_t ld = 0;
    const size_t bytes = realign_shared_bytes(rows, cols, &ld);
    if (!both || bytes == 0 || (bytes > ctx->patches_bytes && !grow_for_copies(ctx, ensure_patches, bytes))) return apart();
    // each product with grad_out replaced by the copy: the space of its own copy is not asked for
    GemmProblem q[2] = {x[0].p, x[1].p};
    for (int i = 0; i < 2; i++) {
        q[i].ksum = nullptr;
        q[i].ksum_of = KSUM_NONE;
        if (q[i].a == grad_out) {
            (q[i].a_rs == 1 ? q[i].a_cs : q[i].a_rs) = ld;
            q[i].a = ctx->patches;
            q[i].a_laid = true;
        } else {
            (q[i].b_cs == 1 ? q[i].b_rs : q[i].b_cs) = ld;
            q[i].b = ctx->patches;
            q[i].b_laid = true;
        }
        Plan reserved = x[i].plan;
        if (int e = reserve_partials(ctx, q[i], reserved, false)) return e;
        if (!reserved.realign) return apart();
    }
    const size_t sums_bytes = colsum ? bias_backward_copy_partials(ctx->compute_units, rows, cols, ld) : 0;
    const bool sums = sums_bytes > 0 && (sums_bytes <= ctx->workspace_bytes || grow_for_copies(ctx, ensure_workspace, sums_bytes));
    if (int e = settle(ctx, grad_out)) return e;
    if (sums) {  // on the way into the copy; their partials are done with the workspace before the products write it
        bool fresh = false;
        if (int e = settle_output(ctx, colsum, (size_t)cols * dtype_size(first->dtype), true, &fresh)) return e;
        HIP_TRY(launch_bias_backward_copy(first->dtype, ctx->compute_units, rows, cols, grad_out, ctx->patches, ld, (rows + 63) / 64 * 64, colsum, fresh,
                                          (float *)ctx->workspace, ctx->stream));
        *fused = true;
    } else {
        HIP_TRY(launch_realign_shared(grad_out, rows, cols, ctx->patches, ctx->stream));
    }
    for (int i = 0; i < 2; i++) {
        if (int e = settle_operands(ctx, &q[i], /*may_overwrite=*/true)) return e;
        if (int e = run_plan(ctx, q[i], x[i].plan)) return e;
    }
    return DFDX_ROCM_OK;
}

// Deferred zero fills, as settle_operands, for three products in one.
static int settle_three(dfdx_rocm_ctx *ctx, GemmProblem *problem) {
    const GemmProblem p = *problem;
    const size_t es = dtype_size(p.dtype), c_bytes = (size_t)(p.m * p.n) * es, k_bytes = (size_t)p.m * es;
    auto at = [&](const void *ptr, int64_t b1, int64_t b2, int i) -> char * {
        return ptr ? (char *)ptr + (i == 1 ? b2 : i == 2 ? b1 : 0) * (int64_t)es : nullptr;
    };
    if (int e = settle(ctx, p.with)) return e;
    bool fresh[2][3] = {};
    for (int i = 0; i < 3; i++) {
        if (int e = settle(ctx, at(p.a, p.a_b1, p.a_b2, i))) return e;
        if (int e = settle(ctx, at(p.b, p.b_b1, p.b_b2, i))) return e;
        if (int e = settle(ctx, at(p.bias, p.bias_b1, p.bias_b2, i))) return e;
        if (i > 0 && p.reduce) continue;
        if (int e = settle_output(ctx, at(p.c, p.c_b1, p.c_b2, i), c_bytes, p.accumulate, p.extra == EXTRA_FROM ? nullptr : &fresh[0][i])) return e;
        if (p.ksum)
            if (int e = settle_output(ctx, at(p.ksum, p.ksum_b1, p.ksum_b2, i), k_bytes, true, &fresh[1][i])) return e;
    }
    // gradients are stored where all three count as zero; a mixture is filled after all
    for (int r = 0; r < 2; r++) {
        const bool all = fresh[r][0] && fresh[r][1] && fresh[r][2];
        if (all && r == 0) problem->accumulate = 0;
        if (all && r == 1) problem->ksum_accumulate = 0;
        for (int i = 0; i < 3 && !all; i++)
            if (fresh[r][i])
                HIP_TRY(launch_zero_fill(r == 0 ? at(p.c, p.c_b1, p.c_b2, i) : at(p.ksum, p.ksum_b1, p.ksum_b2, i), r == 0 ? c_bytes : k_bytes,
                                         ctx->compute_units, ctx->stream));
    }
    return DFDX_ROCM_OK;
}

int gemm_three(dfdx_rocm_ctx *ctx, const GemmProblem &problem, bool *done) {
    *done = false;
    GemmProblem p = problem;
    p.compute_units = ctx->compute_units;
    if (!p.reduce && p.extra == EXTRA_NONE) {
        GemmProblem one[3] = {p, p, p};
        const int64_t es = (int64_t)dtype_size(p.dtype);
        dfdx_rocm_gemm_desc plain;
        std::memset(&plain, 0, sizeof(plain));  // (an automatic plan)
        bool small = true;
        for (int i = 0; i < 3; i++) {
            auto at = [&](const void *ptr, int64_t b1, int64_t b2) { return ptr ? (char *)ptr + (i == 1 ? b2 : i == 2 ? b1 : 0) * es : nullptr; };
            GemmProblem &q = one[i];
            q.batches = 0;
            q.nb1 = q.nb2 = 1;
            q.a = at(p.a, p.a_b1, p.a_b2);
            q.b = at(p.b, p.b_b1, p.b_b2);
            q.c = at(p.c, p.c_b1, p.c_b2);
            q.bias = at(p.bias, p.bias_b1, p.bias_b2);
            q.ksum = at(p.ksum, p.ksum_b1, p.ksum_b2);
            if (!small) continue;
            Product x{&plain, q};
            small = plans_small(ctx, x);
        }
        if (small && independent(one[0], one[1]) && independent(one[0], one[2]) && independent(one[1], one[2])) {
            *done = true;
            CtxLock lock(ctx->mu);
            if (int e = settle_three(ctx, &p)) return e;
            for (GemmProblem &q : one) {
                q.accumulate = p.accumulate;
                q.ksum_accumulate = p.ksum_accumulate;
            }
            return (int)launch_small_many(one, 3, ctx->stream);
        }
    }
    if (p.dtype != DT_F16 && p.dtype != DT_BF16) return DFDX_ROCM_OK;
    int dv = 0, splits = 1, dv1 = 0, splits1 = 1;
    double t3 = 1e300, t1 = 1e300;
    GemmCut cut;
    mfma16dma_plan_split(p, ctx->compute_units, 0, 0, &dv, &splits, &t3, &cut);
    if (!dv || (p.ksum && !mfma16dma_ksum_supported(p, dv, splits)) || (p.extra != EXTRA_NONE && !mfma16dma_extra_supported(p, dv, splits)))
        return DFDX_ROCM_OK;
    GemmProblem q = p;
    q.batches = 0;
    q.nb1 = q.nb2 = 1;
    q.reduce = 0;
    mfma16dma_plan_split(q, ctx->compute_units, 0, 0, &dv1, &splits1, &t1);
    const double t_small = small_supported(q) ? small_time(q, ctx->compute_units) : 1e300;
    // Results that replace those of three calls have the bits of those: the order of the contraction is that of the tiles, so the
    // small kernel and split plans are no match.  (Sums that join what three calls round one by one are free of that.)
    if ((!p.accumulate || p.k % 64) && (t_small < t1 || splits1 > 1 || splits > 1)) return DFDX_ROCM_OK;
    if (t3 >= 3.0 * std::min(t1, t_small)) return DFDX_ROCM_OK;
    Plan plan = {DFDX_ROCM_KERNEL_MFMA, dv + mfma16_dma_first_variant() - 1, splits};
    plan.cut = cut;
    if (int e = reserve_partials(ctx, p, plan, false)) return e;
    if (int e = settle_three(ctx, &p)) return e;
    *done = true;
    return run_plan(ctx, p, plan);
}

int gemm_three_two(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *first, const dfdx_rocm_gemm_desc *second, void *colsum, const GemmProblem &sum,
                   const GemmProblem &apart, bool *done) {
    *done = false;
    if (int e = bind(ctx)) return e;
    Product one{first}, two{second};
    if (int e = make_problem(first, &one.p)) return e;
    if (int e = make_problem(second, &two.p, colsum)) return e;
    if (one.p.m == 0 || two.p.m == 0 || !two.p.ksum) return DFDX_ROCM_OK;
    if (!ring_pair_tile(ctx, one, two)) return DFDX_ROCM_OK;  // (what the calls that this one stands for would do)
    GemmProblem p = sum, q = apart;
    double seconds = 0.0;
    const int tile = mfma16_ring_pair_plan(p, q, ctx->compute_units, &seconds);
    if (!tile || !independent(p, q)) return DFDX_ROCM_OK;
    *done = true;
    CtxLock lock(ctx->mu);
    if (int e = settle_three(ctx, &p)) return e;
    if (int e = settle_three(ctx, &q)) return e;
    p.compute_units = q.compute_units = ctx->compute_units;
    return (int)launch_mfma16_ring_pair(p, q, tile, ctx->stream);
}

int gemm_with_colsum(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc, void *colsum_b, bool *fused) {
    *fused = false;
    if (int e = bind(ctx)) return e;
    GemmProblem p;
    if (int e = make_problem(desc, &p, colsum_b)) return e;
    if (p.m == 0) return DFDX_ROCM_OK;
    Plan plan;  // from the product as the caller states it: a pending zero fill of C must not change which kernel runs
    if (int e = make_plan(ctx, desc, p, &plan)) return e;
    return run_with_colsum(ctx, p, plan, fused);
}

}  // namespace dfdx_rocm

extern "C" {

int dfdx_rocm_create(int ordinal, void *stream, dfdx_rocm_ctx **out) {
    if (!out || ordinal < 0) return DFDX_ROCM_ERR_INVALID_ARG;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || ordinal >= count) return DFDX_ROCM_ERR_NO_DEVICE;
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, ordinal));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return DFDX_ROCM_ERR_NO_DEVICE;  // code objects are gfx950 only
    HIP_TRY(hipSetDevice(ordinal));
    void *static_scratch = nullptr;
    if (int e = scratch_address(ordinal, &static_scratch)) return e;
    dfdx_rocm_ctx *ctx = new (std::nothrow) dfdx_rocm_ctx();
    if (!ctx) return (int)hipErrorOutOfMemory;
    ctx->static_scratch = static_scratch;
    ctx->device = ordinal;
    ctx->stream = (hipStream_t)stream;
    ctx->compute_units = prop.multiProcessorCount;
    ctx->clock_mhz = prop.clockRate / 1000;
    std::snprintf(ctx->name, sizeof(ctx->name), "%s (%s)", prop.name, prop.gcnArchName);
    *out = ctx;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_destroy(dfdx_rocm_ctx *ctx) {
    if (!ctx) return DFDX_ROCM_OK;
    if (ctx->workspace || ctx->patches || !ctx->retired.empty() || !ctx->cache.empty() || ctx->pending_count.load()) {
        (void)hipSetDevice(ctx->device);
        (void)settle_all(ctx);  // the caller's buffers outlive the context: they must hold the zeros they were promised
        (void)hipStreamSynchronize(ctx->stream);
        (void)free_retired(ctx);
        if (ctx->workspace) (void)hipFree(ctx->workspace);
        if (ctx->patches) (void)hipFree(ctx->patches);
        (void)drop_cache(ctx);
    }
    delete ctx;
    return DFDX_ROCM_OK;
}

const char *dfdx_rocm_strerror(int code) {
    switch (code) {
    case DFDX_ROCM_OK: return "ok";
    case DFDX_ROCM_ERR_INVALID_ARG: return "dfdx_rocm: invalid argument";
    case DFDX_ROCM_ERR_UNSUPPORTED: return "dfdx_rocm: no kernel for this request";
    case DFDX_ROCM_ERR_NO_DEVICE: return "dfdx_rocm: no usable gfx950 device";
    case DFDX_ROCM_ERR_ALIASED_OUTPUT: return "dfdx_rocm: output view aliases itself (zero stride)";
    case DFDX_ROCM_ERR_SCRATCH_TOO_SMALL:
        return "dfdx_rocm: the split reduction of this product needs more than the fixed scratch of the no-allocation entry";
    default: break;
    }
    if (code > 0) return hipGetErrorString((hipError_t)code);
    return "dfdx_rocm: unknown error";
}

int dfdx_rocm_device_info(dfdx_rocm_ctx *ctx, char *name, size_t name_len, int *compute_units, int *clock_mhz) {
    if (!ctx) return DFDX_ROCM_ERR_INVALID_ARG;
    if (name && name_len) std::snprintf(name, name_len, "%s", ctx->name);
    if (compute_units) *compute_units = ctx->compute_units;
    if (clock_mhz) *clock_mhz = ctx->clock_mhz;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_alloc(dfdx_rocm_ctx *ctx, size_t bytes, int zeroed, void **out) {
    if (!out) return DFDX_ROCM_ERR_INVALID_ARG;
    *out = nullptr;
    if (int e = bind(ctx)) return e;
    if (bytes == 0) bytes = 16;
    void *p = nullptr;
    bool recycled = false;
    {   // a cached buffer of exactly this size, if the cache is on and has one (cache.rs:105-149)
        CtxLock lock(ctx->mu);
        if (ctx->cache_enabled) {
            auto it = ctx->cache.find(bytes);
            if (it != ctx->cache.end()) {
                p = it->second.back();
                it->second.pop_back();
                if (it->second.empty()) ctx->cache.erase(it);
                ctx->cache_bytes -= bytes;
                recycled = true;
            }
        }
    }
    if (!recycled) {
        const hipError_t e = hipMalloc(&p, bytes);
        if (e == hipErrorOutOfMemory) {
            // once more with everything the context can give back: the cached buffers and the outgrown workspaces
            (void)hipGetLastError();
            (void)dfdx_rocm_empty_cache(ctx);
            {
                CtxLock lock(ctx->mu);
                if (!ctx->retired.empty()) {
                    HIP_TRY(hipStreamSynchronize(ctx->stream));
                    (void)free_retired(ctx);
                }
            }
            const hipError_t again = hipMalloc(&p, bytes);
            if (again != hipSuccess) {
                (void)hipGetLastError();
                return (int)again;
            }
        } else if (e != hipSuccess) {
            (void)hipGetLastError();
            return (int)e;
        }
        CtxLock lock(ctx->mu);
        ctx->sizes[p] = bytes;
    }
    if (zeroed == DFDX_ROCM_ZERO_DEFERRED) {
        CtxLock lock(ctx->mu);
        ctx->pending_zero[(uintptr_t)p] = bytes;
        ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
    } else if (zeroed) {
        hipError_t e = launch_zero_fill(p, bytes, ctx->compute_units, ctx->stream);
        if (e != hipSuccess) {
            (void)dfdx_rocm_free(ctx, p);
            return (int)e;
        }
    }
    *out = p;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_free(dfdx_rocm_ctx *ctx, void *ptr) {
    if (int e = bind(ctx)) return e;
    if (!ptr) return DFDX_ROCM_OK;
    {
        CtxLock lock(ctx->mu);
        auto it = ctx->sizes.find(ptr);
        if (ctx->pending_count.load(std::memory_order_acquire)) {  // a fill nobody waited for is not run
            if (it != ctx->sizes.end()) {
                if (int e = drop_pending_inside(ctx, ptr, it->second)) return e;
            } else if (ctx->pending_zero.erase((uintptr_t)ptr)) {
                ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
            }
        }
        if (it != ctx->sizes.end() && ctx->cache_enabled) {
            // Kept for the next allocation of this size.  No synchronisation: whoever gets the buffer next uses it
            // through this context's stream, behind the work that still reads it.
            ctx->cache[it->second].push_back(ptr);
            ctx->cache_bytes += it->second;
            return DFDX_ROCM_OK;
        }
        if (it != ctx->sizes.end()) ctx->sizes.erase(it);
    }
    HIP_TRY(hipStreamSynchronize(ctx->stream));  // pending kernels may still use the buffer
    HIP_TRY(hipFree(ptr));
    CtxLock lock(ctx->mu);
    HIP_TRY(free_retired(ctx));  // the stream is drained: nothing uses the outgrown workspaces either
    return DFDX_ROCM_OK;
}

int dfdx_rocm_enable_cache(dfdx_rocm_ctx *ctx) {
    if (!ctx) return DFDX_ROCM_ERR_INVALID_ARG;
    CtxLock lock(ctx->mu);
    ctx->cache_enabled = true;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_disable_cache(dfdx_rocm_ctx *ctx) {
    if (int e = bind(ctx)) return e;
    {
        CtxLock lock(ctx->mu);
        ctx->cache_enabled = false;
    }
    return dfdx_rocm_empty_cache(ctx);
}

int dfdx_rocm_empty_cache(dfdx_rocm_ctx *ctx) {
    if (int e = bind(ctx)) return e;
    CtxLock lock(ctx->mu);
    for (auto &kv : ctx->cache)
        for (void *p : kv.second) ctx->sizes.erase(p);
    return drop_cache(ctx);
}

int dfdx_rocm_cache_stats(dfdx_rocm_ctx *ctx, size_t *buffers, size_t *bytes) {
    if (!ctx) return DFDX_ROCM_ERR_INVALID_ARG;
    CtxLock lock(ctx->mu);
    size_t n = 0;
    for (auto &kv : ctx->cache) n += kv.second.size();
    if (buffers) *buffers = n;
    if (bytes) *bytes = ctx->cache_bytes;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_memset_zero(dfdx_rocm_ctx *ctx, void *ptr, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if (!ptr && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    if (bytes) {
        if (int e = drop_pending_inside(ctx, ptr, bytes)) return e;
        HIP_TRY(launch_zero_fill(ptr, bytes, ctx->compute_units, ctx->stream));
    }
    return DFDX_ROCM_OK;
}

int dfdx_rocm_zero_deferred(dfdx_rocm_ctx *ctx, void *ptr, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if (!ptr && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    if (!bytes) return DFDX_ROCM_OK;
    if (int e = drop_pending_inside(ctx, ptr, bytes)) return e;  // earlier declarations inside the range are replaced
    CtxLock lock(ctx->mu);
    if (pending_holding(ctx, (uintptr_t)ptr) != ctx->pending_zero.end())  // still inside a larger pending buffer
        return DFDX_ROCM_OK;                                             // which already stands for these zeros
    ctx->pending_zero[(uintptr_t)ptr] = bytes;
    ctx->pending_count.store((int)ctx->pending_zero.size(), std::memory_order_release);
    return DFDX_ROCM_OK;
}

int dfdx_rocm_settle_zeros(dfdx_rocm_ctx *ctx) {
    if (int e = bind(ctx)) return e;
    return settle_all(ctx);
}

int dfdx_rocm_forget_zeros(dfdx_rocm_ctx *ctx, void *ptr, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if (!ptr && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    return bytes ? drop_pending_inside(ctx, ptr, bytes) : DFDX_ROCM_OK;
}

int dfdx_rocm_copy_h2d(dfdx_rocm_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if ((!dst || !src) && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    if (bytes) {
        if (int e = drop_pending_inside(ctx, dst, bytes)) return e;
        HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));  // the host buffer may be reused on return
        CtxLock lock(ctx->mu);
        HIP_TRY(free_retired(ctx));
    }
    return DFDX_ROCM_OK;
}

int dfdx_rocm_copy_d2h(dfdx_rocm_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if ((!dst || !src) && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    if (bytes) {
        if (int e = settle_range(ctx, src, bytes)) return e;
        HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(hipStreamSynchronize(ctx->stream));
        CtxLock lock(ctx->mu);
        HIP_TRY(free_retired(ctx));
    }
    return DFDX_ROCM_OK;
}

int dfdx_rocm_copy_d2d(dfdx_rocm_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (int e = bind(ctx)) return e;
    if ((!dst || !src) && bytes) return DFDX_ROCM_ERR_INVALID_ARG;
    if (bytes) {
        if (int e = settle_range(ctx, src, bytes)) return e;
        if (int e = drop_pending_inside(ctx, dst, bytes)) return e;
        HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    }
    return DFDX_ROCM_OK;
}

int dfdx_rocm_synchronize(dfdx_rocm_ctx *ctx) {
    if (int e = bind(ctx)) return e;
    if (int e = settle_all(ctx)) return e;  // whoever reads the memory after this call must find the zeros
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    CtxLock lock(ctx->mu);
    HIP_TRY(free_retired(ctx));  // workspaces outgrown since the last call: nothing on the stream uses them any more
    return DFDX_ROCM_OK;
}

int dfdx_rocm_gemm(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc) {
    if (int e = bind(ctx)) return e;
    GemmProblem p;
    if (int e = make_problem(desc, &p)) return e;
    if (p.m == 0) return DFDX_ROCM_OK;
    Plan plan;  // from the product as the caller states it: a pending zero fill of C must not change which kernel runs
    if (int e = make_plan(ctx, desc, p, &plan)) return e;
    plan.pieces_asked = ((desc->flags >> 8) & 0xff) != 0;
    return run_planned(ctx, p, plan);
}

int dfdx_rocm_gemm_noalloc(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc) {
    if (int e = bind(ctx)) return e;
    GemmProblem p;
    if (int e = make_problem(desc, &p)) return e;
    if (p.m == 0) return DFDX_ROCM_OK;
    Plan plan;  // from the product as the caller states it: a pending zero fill of C must not change which kernel runs
    if (int e = make_plan(ctx, desc, p, &plan)) return e;
    return run_planned(ctx, p, plan, /*static_scratch=*/true);
}

int dfdx_rocm_gemm_plan(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc, int *kernel, int *variant, char *name,
                        size_t name_len) {
    if (!ctx) return DFDX_ROCM_ERR_INVALID_ARG;
    GemmProblem p;
    if (int e = make_problem(desc, &p)) return e;
    Plan plan = {DFDX_ROCM_KERNEL_GENERIC, 0, 1};
    if (p.m != 0)
        if (int e = make_plan(ctx, desc, p, &plan)) return e;
    if (kernel) *kernel = plan.kernel;
    // (a tile variant; of the bandwidth kernels, which the shape and the layout choose, one beside another has an id)
    if (variant) *variant = plan.kernel == DFDX_ROCM_KERNEL_GEMV && plan.variant != BW_ROWS ? 0 : plan.variant;
    if (name && name_len) {
        const bool ring = plan.realign && mfma16dma_takes_any_k(plan.variant - mfma16_dma_first_variant() + 1);  // one of the LDS-DMA kernels too
        const char *const copied = !plan.realign ? "" : ring ? "_dma_realigned" : "_realigned";
        if (plan.kernel == DFDX_ROCM_KERNEL_MFMA && plan.splits > 1)
            std::snprintf(name, name_len, "%s_%s%s_splitk%d", p.dtype == DT_F32 ? "mfma32" : "mfma16",
                          p.dtype == DT_F32 ? mfma32_variant_name(plan.variant) : mfma16_variant_name(plan.variant), copied, plan.splits);
        else if (plan.kernel == DFDX_ROCM_KERNEL_MFMA && p.dtype == DT_F64)
            std::snprintf(name, name_len, "mfma64_%s", mfma64_variant_name(plan.variant));
        else if (plan.kernel == DFDX_ROCM_KERNEL_MFMA)
            std::snprintf(name, name_len, "%s_%s%s", p.dtype == DT_F32 ? "mfma32" : "mfma16",
                          p.dtype == DT_F32 ? mfma32_variant_name(plan.variant) : mfma16_variant_name(plan.variant), copied);
        else
            std::snprintf(name, name_len, "%s", plan.kernel != DFDX_ROCM_KERNEL_GEMV ? "generic" : bandwidth_kernel_name(p, plan.variant));
        if (plan.cut.variant) {
            const size_t at = std::strlen(name);
            std::snprintf(name + at, name_len - at, "+%s", mfma16dma_variant_name(plan.cut.variant));
        }
    }
    return DFDX_ROCM_OK;
}

int dfdx_rocm_mfma_variant_count(int dtype) {
    if (dtype == DFDX_ROCM_F16 || dtype == DFDX_ROCM_BF16) return mfma16_variant_count();
    if (dtype == DFDX_ROCM_F32) return mfma32_variant_count();
    if (dtype == DFDX_ROCM_F64) return mfma64_variant_count();
    return 0;
}

int dfdx_rocm_gemm_time_rotating(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *descs, int count, int warmup, int iters,
                                 float *avg_ms) {
    if (!avg_ms || !descs || count < 1 || iters < 1 || warmup < 0) return DFDX_ROCM_ERR_INVALID_ARG;
    if (int e = bind(ctx)) return e;
    std::vector<GemmProblem> problems((size_t)count);
    std::vector<Plan> plans((size_t)count);
    for (int i = 0; i < count; i++) {
        if (int e = make_problem(&descs[i], &problems[(size_t)i])) return e;
        if (problems[(size_t)i].m == 0) {   // an empty product launches nothing: there is no time to report
            *avg_ms = 0.0f;
            return DFDX_ROCM_OK;
        }
        if (int e = make_plan(ctx, &descs[i], problems[(size_t)i], &plans[(size_t)i])) return e;
        if (int e = reserve_partials(ctx, problems[(size_t)i], plans[(size_t)i], false)) return e;
        if (int e = settle_operands(ctx, &problems[(size_t)i], /*may_overwrite=*/false)) return e;
    }
    for (int i = 0; i < warmup; i++)
        if (int e = run_plan(ctx, problems[(size_t)(i % count)], plans[(size_t)(i % count)])) return e;
    hipEvent_t t0, t1;
    HIP_TRY(hipEventCreate(&t0));
    HIP_TRY(hipEventCreate(&t1));
    int rc = DFDX_ROCM_OK;
    hipError_t he = hipEventRecord(t0, ctx->stream);
    for (int i = 0; i < iters && rc == DFDX_ROCM_OK && he == hipSuccess; i++)
        rc = run_plan(ctx, problems[(size_t)(i % count)], plans[(size_t)(i % count)]);
    if (he == hipSuccess) he = hipEventRecord(t1, ctx->stream);
    if (he == hipSuccess) he = hipEventSynchronize(t1);
    float ms = 0.0f;
    if (he == hipSuccess) he = hipEventElapsedTime(&ms, t0, t1);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    if (rc != DFDX_ROCM_OK) return rc;
    if (he != hipSuccess) return (int)he;
    *avg_ms = ms / (float)iters;
    return DFDX_ROCM_OK;
}

int dfdx_rocm_gemm_time(dfdx_rocm_ctx *ctx, const dfdx_rocm_gemm_desc *desc, int warmup, int iters, float *avg_ms) {
    return dfdx_rocm_gemm_time_rotating(ctx, desc, desc ? 1 : 0, warmup, iters, avg_ms);
}

}  // extern "C"
