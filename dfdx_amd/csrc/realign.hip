// Operands of a 16-bit product copied into the layout that the LDS-DMA kernels load: addresses and leading dimensions on the
// 16-byte grid, the contraction padded with zeros to whole k tiles.
//
// What bounds it: HBM, one read and one write of the operand.  The product behind it is bound by the matrix cores, and the
// register-staged kernels that take any layout feed them at 0.3 - 0.6 of the LDS-DMA kernels' rate once both are large.
// An operand on the grid whose rows lie along memory lacks the padding only: its last k tile is copied, with the leading dimension that
// it has, and the kernels go there for it (2048 x 50257 . 50257 x 1024 f16, the copy 47 -> 6 us).
// Both operands go in one launch; a thread moves four 16-byte pieces (element-aligned loads, aligned stores) that lie 256
// pieces apart, so that every wave access is contiguous and four loads are in flight.
#include "gemm_internal.h"
#include <algorithm>

namespace dfdx_rocm {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));

struct Side {
    const uint16_t *src;
    uint16_t *dst;
    int64_t ld, b1, b2;      // elements between source rows and batches
    uint32_t rows, cols;     // of the source
    uint32_t rows_out, pieces;  // of the copy: rows, 16-byte pieces per row
    uint32_t n2, total;      // batches of the second axis; pieces in all
};
struct Sides {
    Side s[2];
    uint32_t first_blocks;   // workgroups of s[0]
};
constexpr int PER_THREAD = 4, PER_BLOCK = 256 * PER_THREAD;

__global__ __launch_bounds__(256) void realign_kernel(const Sides both) {
    const bool second = blockIdx.x >= both.first_blocks;
    const Side &s = both.s[second ? 1 : 0];
    const uint32_t first = (blockIdx.x - (second ? both.first_blocks : 0u)) * PER_BLOCK + threadIdx.x;
    u32x4 v[PER_THREAD];
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
        const uint32_t at = first + u * 256;
        v[u] = u32x4{0u, 0u, 0u, 0u};
        if (at >= s.total) continue;
        const uint32_t line = at / s.pieces, col = (at - line * s.pieces) * 8;
        const uint32_t b = line / s.rows_out, row = line - b * s.rows_out;
        if (row >= s.rows || col >= s.cols) continue;
        const uint16_t *src = s.src + (int64_t)(b / s.n2) * s.b1 + (int64_t)(b % s.n2) * s.b2 + (int64_t)row * s.ld + col;
        if (col + 8 <= s.cols) {
            v[u] = *(const u32x4_any *)src;
        } else {
#pragma unroll
            for (uint32_t e = 0; e < 7; e++)
                if (col + e < s.cols) v[u][e / 2] |= (uint32_t)src[e] << (e % 2 * 16);
        }
    }
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
        const uint32_t at = first + u * 256;
        if (at < s.total) *(u32x4 *)(s.dst + (int64_t)at * 8) = v[u];
    }
}

inline int64_t up(int64_t v, int64_t to) { return (v + to - 1) / to * to; }

// One operand: `rows` of the product (m or n), strides of it and of the contraction, batch strides.
struct Operand {
    bool kc, copy, off, last;  // last: of the last k tile only
    int64_t lines, lines_out, cols, ld_out, src_ld, n1, n2;  // as the copy walks it
    int64_t pieces() const { return n1 * n2 * lines_out * (ld_out / 8); }
};
// False where no stride is 1 or the copy would be out of range.
bool operand(const void *ptr, int64_t rows, int64_t k, int64_t row_stride, int64_t k_stride, int64_t b1, int64_t b2, int64_t nb1, int64_t nb2, bool laid, Operand *o) {
    const int64_t kp = up(k, 64);
    if (b1 < 0 || b2 < 0 || row_stride < 0 || k_stride < 0) return false;
    if (k_stride == 1 && (rows == 1 || row_stride >= k)) {
        o->kc = true;
        o->lines = o->lines_out = rows;
        o->cols = k;
        o->ld_out = kp;
        o->src_ld = rows == 1 ? k : row_stride;
    } else if (row_stride == 1 && k_stride >= rows) {
        o->kc = false;
        o->lines = k;
        o->lines_out = kp;
        o->cols = rows;
        o->ld_out = up(rows, 64);
        o->src_ld = k_stride;
    } else {
        return false;
    }
    o->n1 = b1 == 0 ? 1 : nb1;  // an operand that the batches share is copied once
    o->n2 = b2 == 0 ? 1 : nb2;
    o->off = o->src_ld % 8 != 0 || (!o->kc && rows % 8 != 0) || ((uintptr_t)ptr & 15u) != 0 || (o->n1 > 1 && b1 % 8 != 0) || (o->n2 > 1 && b2 % 8 != 0);
    o->copy = o->off || kp != k;
    if (laid) o->off = o->copy = false;
    // (one matrix; rows far apart in a view would be a copy of what lies between them)
    o->last = o->copy && !o->off && !o->kc && nb1 * nb2 == 1 && o->src_ld <= 2 * o->ld_out;
    if (o->last) {
        o->lines = k - (kp - 64);
        o->lines_out = 64;
        o->ld_out = o->src_ld;
    }
    return !o->copy || (o->pieces() < (1ll << 31) && o->lines_out < (1ll << 31) && o->ld_out < (1ll << 31));
}
void describe(const Operand &o, const void *src, void *dst, int64_t b1, int64_t b2, Side *s) {
    s->src = (const uint16_t *)src;
    s->dst = (uint16_t *)dst;
    s->ld = o.src_ld;
    s->b1 = o.n1 > 1 ? b1 : 0;
    s->b2 = o.n2 > 1 ? b2 : 0;
    s->rows = (uint32_t)o.lines;
    s->cols = (uint32_t)o.cols;
    s->rows_out = (uint32_t)o.lines_out;
    s->pieces = (uint32_t)(o.ld_out / 8);
    s->n2 = (uint32_t)o.n2;
    s->total = o.copy ? (uint32_t)o.pieces() : 0;
}
// strides of the copy in the product's terms
void strides(const Operand &o, int64_t *row_stride, int64_t *k_stride, int64_t *b1, int64_t *b2) {
    const int64_t matrix = o.lines_out * o.ld_out;
    *row_stride = o.kc ? o.ld_out : 1;
    *k_stride = o.kc ? 1 : o.ld_out;
    *b2 = o.n2 > 1 ? matrix : 0;
    *b1 = o.n1 > 1 ? matrix * o.n2 : 0;
}

}  // namespace

bool plan_realign(const GemmProblem &p, Realign *r) {
    if ((p.dtype != DT_F16 && p.dtype != DT_BF16) || p.k < 1 || p.extra != EXTRA_NONE) return false;
    Operand a, b;
    if (!operand(p.a, p.m, p.k, p.a_rs, p.a_cs, p.a_b1, p.a_b2, p.nb1, p.nb2, p.a_laid, &a)) return false;
    if (!operand(p.b, p.n, p.k, p.b_cs, p.b_rs, p.b_b1, p.b_b2, p.nb1, p.nb2, p.b_laid, &b)) return false;
    r->a = a.copy && !a.last;
    r->b = b.copy && !b.last;
    r->a_last = a.last;
    r->b_last = b.last;
    r->problem = p;
    GemmProblem &q = r->problem;
    q.ragged = true;
    q.ksum = nullptr;
    q.ksum_of = KSUM_NONE;
    q.k = up(p.k, 64);
    r->a_bytes = r->b_bytes = 0;
    // (planning looks at the addresses' alignment only)
    q.last_apart = a.last || b.last;
    if (r->a) {
        strides(a, &q.a_rs, &q.a_cs, &q.a_b1, &q.a_b2);
        q.a = (const void *)256;
    }
    if (r->b) {
        strides(b, &q.b_cs, &q.b_rs, &q.b_b1, &q.b_b2);
        q.b = (const void *)256;
    }
    if (a.copy) r->a_bytes = (size_t)up(a.pieces() * 16, 256);
    if (b.copy) r->b_bytes = (size_t)up(b.pieces() * 16, 256);
    if (r->a_bytes + r->b_bytes > REALIGN_MAX_BYTES) return false;
    r->off_grid = a.off + b.off;
    r->off_grid_k = (a.off && a.kc) + (b.off && b.kc);
    // a launch and the gap behind it, a read and a write (2048 x 50257 and 50257 x 1024: 140 us)
    r->seconds = (a.copy || b.copy) ? 6.0e-6 + 2.0 * (double)(r->a_bytes + r->b_bytes) / 4.5e12 : 0.0;
    return true;
}

size_t realign_shared_bytes(int64_t rows, int64_t cols, int64_t *ld) {
    *ld = up(cols, 64);
    const int64_t pieces = up(rows, 64) * (*ld / 8);
    return pieces < (1ll << 31) && (size_t)pieces * 16 <= REALIGN_MAX_BYTES ? (size_t)pieces * 16 : 0;
}

hipError_t launch_realign_shared(const void *src, int64_t rows, int64_t cols, void *dst, hipStream_t stream) {
    Sides both{};
    Side &s = both.s[0];
    s.src = (const uint16_t *)src;
    s.dst = (uint16_t *)dst;
    s.ld = cols;
    s.rows = (uint32_t)rows;
    s.cols = (uint32_t)cols;
    s.rows_out = (uint32_t)up(rows, 64);
    s.pieces = (uint32_t)(up(cols, 64) / 8);
    s.n2 = 1;
    s.total = s.rows_out * s.pieces;
    both.first_blocks = (s.total + PER_BLOCK - 1) / PER_BLOCK;
    realign_kernel<<<dim3(both.first_blocks), dim3(256), 0, stream>>>(both);
    return hipGetLastError();
}

hipError_t launch_realign(const GemmProblem &p, Realign *r, void *space, hipStream_t stream) {
    Operand a, b;
    if (!operand(p.a, p.m, p.k, p.a_rs, p.a_cs, p.a_b1, p.a_b2, p.nb1, p.nb2, p.a_laid, &a) ||
        !operand(p.b, p.n, p.k, p.b_cs, p.b_rs, p.b_b1, p.b_b2, p.nb1, p.nb2, p.b_laid, &b) || (a.copy && !a.last) != r->a || (b.copy && !b.last) != r->b || a.last != r->a_last || b.last != r->b_last)
        return hipErrorInvalidValue;
    Sides both{};
    char *const a_to = (char *)space, *const b_to = a_to + r->a_bytes;
    const int64_t first = p.k - 1 - (p.k - 1) % 64;  // of the last k tile
    const uint16_t *const a_from = (const uint16_t *)p.a + (a.last ? first * a.src_ld : 0), *const b_from = (const uint16_t *)p.b + (b.last ? first * b.src_ld : 0);
    describe(a, a_from, a_to, p.a_b1, p.a_b2, &both.s[0]);
    describe(b, b_from, b_to, p.b_b1, p.b_b2, &both.s[1]);
    r->problem.a = r->a ? a_to : p.a;
    r->problem.b = r->b ? b_to : p.b;
    r->problem.a_last = a.last ? ((intptr_t)a_to - (intptr_t)a_from) / 2 : 0;
    r->problem.b_last = b.last ? ((intptr_t)b_to - (intptr_t)b_from) / 2 : 0;
    both.first_blocks = (both.s[0].total + PER_BLOCK - 1) / PER_BLOCK;
    const uint32_t blocks = both.first_blocks + (both.s[1].total + PER_BLOCK - 1) / PER_BLOCK;
    if (blocks == 0) return hipSuccess;
    realign_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(both);
    return hipGetLastError();
}

}  // namespace dfdx_rocm
