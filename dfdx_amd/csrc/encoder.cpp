// A transformer encoder block as one call forward and one backward: the sequence of entry points that the block's ops map
// to, strung together on the host side of the library, and the passes between them that the products can do on the way.
//
// TransformerEncoderBlock (dfdx/src/nn/layers/transformer.rs:24-48) over MultiHeadAttention (multi_head_attention.rs:
// 105-146), Linear, LayerNorm1D and ResidualAdd, with the tape's backward.  What the reference does in ops of their own:
//   - ReLU and the residual adds ride on the store of the product in front of them (gemm_beyond), values rounded where the
//     op would have read them rounded; the pre-activation is not kept, the ReLU's output tells the gradient what it needs;
//   - the gradient of ReLU masks the store of the input gradient behind it;
//   - a gradient with two contributions starts as the first one (read from where it is) instead of as zeros plus a copy.
// Everything else is the public entry point it names.
#include "ctx_internal.h"
#include "gemm_internal.h"

#include <cmath>
#include <cstring>

using namespace dfdx_rocm;

namespace dfdx_rocm {
bool attention_supported(int dtype, int64_t batch, int64_t heads, int64_t seq, int64_t dim);
}

namespace {

enum { WQ, BQ, WK, BK_, WV, BV, WO, BO, G1, BE1, W1, B1, W2, B2, G2, BE2, PARAM_COUNT };
static_assert(PARAM_COUNT == DFDX_ROCM_ENCODER_PARAMS, "parameter order of the header");

struct Shape {
    int dtype;
    int64_t B, S, d, H, D, ff, T;
    size_t es;
    bool fused;    // attention without the (seq, seq) matrices
    double scale;  // 1 / sqrt(D)
    bool folded;   // the softmax entry's float scale is exact enough (f64: only when the value is)
    int64_t token[3];
};

int shape_of(const dfdx_rocm_encoder *e, Shape *s) {
    if (!e || e->dtype < DFDX_ROCM_F32 || e->dtype > DFDX_ROCM_F64) return DFDX_ROCM_ERR_INVALID_ARG;
    if (e->batch < 0 || e->seq < 0 || e->d_model < 1 || e->heads < 1 || e->d_ff < 1 || e->d_model % e->heads) return DFDX_ROCM_ERR_INVALID_ARG;
    s->dtype = e->dtype;
    s->B = e->batch; s->S = e->seq; s->d = e->d_model; s->H = e->heads; s->ff = e->d_ff;
    s->D = s->d / s->H;
    s->T = s->B * s->S;
    s->es = dtype_size(s->dtype);
    s->fused = attention_supported(s->dtype, s->B, s->H, s->S, s->D) && s->d < (1ll << 24);  // (the rows it walks are d_model apart)
    s->scale = 1.0 / std::sqrt((double)s->D);
    s->folded = s->dtype != DFDX_ROCM_F64 || (double)(float)s->scale == s->scale;
    s->token[0] = s->S * s->d; s->token[1] = s->D; s->token[2] = s->d;
    return DFDX_ROCM_OK;
}

int64_t param_size(const Shape &s, int i) {
    switch (i) {
    case WQ: case WK: case WV: case WO: return s.d * s.d;
    case W1: case W2: return s.ff * s.d;
    case B1: return s.ff;
    default: return s.d;
    }
}

// Pieces of one buffer, each on a 256-byte boundary.
struct Pieces {
    size_t at = 0;
    size_t take(size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    }
};

void saved_layout(const Shape &s, dfdx_rocm_encoder_layout *l) {
    Pieces p;
    const size_t tok = (size_t)(s.T * s.d) * s.es, mat = (size_t)(s.B * s.H * s.S * s.S) * s.es;
    l->q = p.take(tok); l->k = p.take(tok); l->v = p.take(tok); l->tok = p.take(tok);
    l->h1 = p.take(tok); l->n1 = p.take(tok); l->h2 = p.take(tok);
    l->r1 = p.take((size_t)(s.T * s.ff) * s.es);
    l->lse = s.fused ? p.take((size_t)(s.B * s.H * s.S) * sizeof(float)) : 0;
    l->probs = s.fused ? 0 : p.take(mat);
    l->tokens = s.fused ? 0 : p.take(tok);
    l->saved_bytes = p.at;
    l->fused_attention = s.fused;
    // scratch of the forward: the scores; of the backward: the gradients that the caller does not get
    Pieces f, b;
    if (!s.fused) f.take(mat);
    b.take((size_t)(s.T * s.ff) * s.es);
    for (int i = 0; i < 7; i++) b.take(tok);
    if (!s.fused) {
        b.take(tok);
        b.take(mat);
        b.take(mat);
        if (!s.folded) b.take(mat);
    }
    l->forward_scratch_bytes = f.at;
    l->backward_scratch_bytes = b.at;
}

dfdx_rocm_gemm_desc product(int dtype, int64_t m, int64_t k, int64_t n, const void *a, int64_t a_rs, int64_t a_cs, const void *b,
                            int64_t b_rs, int64_t b_cs, void *c, const void *bias = nullptr) {
    dfdx_rocm_gemm_desc g;
    std::memset(&g, 0, sizeof(g));
    g.dtype = dtype;
    g.m = m; g.k = k; g.n = n;
    g.batch1 = g.batch2 = 1;
    g.a = a; g.a_rs = a_rs; g.a_cs = a_cs;
    g.b = b; g.b_rs = b_rs; g.b_cs = b_cs;
    g.c = c; g.c_rs = n; g.c_cs = 1;
    g.bias = bias;
    return g;
}
// y (T, o) = x (T, i) . w^T + bias; w is (o, i)
dfdx_rocm_gemm_desc linear(const Shape &s, int64_t i, int64_t o, const void *x, const void *w, const void *bias, void *y) {
    return product(s.dtype, s.T, i, o, x, i, 1, w, 1, i, y, bias);
}
// grad_x (T, i) = grad_y (T, o) . w
dfdx_rocm_gemm_desc input_grad(const Shape &s, int64_t i, int64_t o, const void *gy, const void *w, void *gx) {
    return product(s.dtype, s.T, o, i, gy, o, 1, w, i, 1, gx);
}
// grad_w (o, i) and grad_b (o) from x and grad_y, both stored; the sums of grad_y come out of the product where they can
dfdx_rocm_gemm_desc weight_product(const Shape &s, int64_t i, int64_t o, const void *x, const void *gy, void *gw) {
    dfdx_rocm_gemm_desc g = product(s.dtype, i, s.T, o, x, 1, i, gy, o, 1, gw);
    g.accumulate = 1;
    g.c_rs = 1; g.c_cs = i;
    return g;
}
int weight_grad(dfdx_rocm_ctx *ctx, const Shape &s, int64_t i, int64_t o, const void *x, const void *gy, void *gw, void *gb) {
    dfdx_rocm_gemm_desc g = weight_product(s, i, o, x, gy, gw);
    bool done = false;
    if (int e = gemm_with_colsum(ctx, &g, gb, &done)) return e;
    return done ? DFDX_ROCM_OK : dfdx_rocm_bias_backward(ctx, s.dtype, s.T, o, gy, gb);
}
// A Linear layer's backward: `gx` is its input gradient with one thing more on the way into it.
int linear_backward(dfdx_rocm_ctx *ctx, const Shape &s, const dfdx_rocm_gemm_desc &gx, int extra, const void *with, int64_t i, int64_t o, const void *x,
                    const void *gy, void *gw, void *gb) {
    const dfdx_rocm_gemm_desc w = weight_product(s, i, o, x, gy, gw);
    bool done = false;
    if (int e = gemm_two(ctx, &gx, extra, with, &w, gb, &done)) return e;
    return done ? DFDX_ROCM_OK : dfdx_rocm_bias_backward(ctx, s.dtype, s.T, o, gy, gb);
}

// The products of the query, key and value projections as one launch: same shapes, matrices wherever they are (addresses from
// the first to the second and to the third).  False where the distances are not whole elements.
bool apart(const void *first, const void *second, const void *third, size_t es, int64_t *b1, int64_t *b2) {
    const int64_t to2 = (const char *)second - (const char *)first, to3 = (const char *)third - (const char *)first;
    *b2 = to2 / (int64_t)es;
    *b1 = to3 / (int64_t)es;
    return to2 % (int64_t)es == 0 && to3 % (int64_t)es == 0;
}
GemmProblem three(int dtype, int64_t m, int64_t k, int64_t n, const void *a, int64_t a_rs, int64_t a_cs, const void *b, int64_t b_rs, int64_t b_cs, void *c) {
    GemmProblem p{};
    p.dtype = dtype;
    p.m = m; p.k = k; p.n = n;
    p.nb1 = p.nb2 = 2;
    p.batches = 3;
    p.a = a; p.a_rs = a_rs; p.a_cs = a_cs;
    p.b = b; p.b_rs = b_rs; p.b_cs = b_cs;
    p.c = c; p.c_rs = n; p.c_cs = 1;
    p.splits = 1;
    return p;
}

#define TRY(call)                \
    do {                         \
        if (int e__ = (call)) return e__; \
    } while (0)

int forward(dfdx_rocm_ctx *ctx, const Shape &s, const dfdx_rocm_encoder *e, const dfdx_rocm_encoder_layout &l, const void *x, void *out,
            char *saved, char *scratch) {
    const void *const *p = e->params;
    void *q = saved + l.q, *k = saved + l.k, *v = saved + l.v, *tok = saved + l.tok, *h1 = saved + l.h1, *n1 = saved + l.n1,
         *h2 = saved + l.h2, *r1 = saved + l.r1;
    const int64_t row[2] = {s.d, 1};
    bool done = false;
    GemmProblem all = three(s.dtype, s.T, s.d, s.d, x, s.d, 1, p[WQ], 1, s.d, q);
    all.bias = p[BQ];
    all.bias_mode = BIAS_PER_COL;
    if (apart(p[WQ], p[WK], p[WV], s.es, &all.b_b1, &all.b_b2) && apart(p[BQ], p[BK_], p[BV], s.es, &all.bias_b1, &all.bias_b2) &&
        apart(q, k, v, s.es, &all.c_b1, &all.c_b2))
        TRY(gemm_three(ctx, all, &done));
    if (!done) {
        TRY(dfdx_rocm_linear_forward(ctx, s.dtype, s.T, s.d, s.d, x, row, p[WQ], p[BQ], q));
        TRY(dfdx_rocm_linear_forward(ctx, s.dtype, s.T, s.d, s.d, x, row, p[WK], p[BK_], k));
        TRY(dfdx_rocm_linear_forward(ctx, s.dtype, s.T, s.d, s.d, x, row, p[WV], p[BV], v));
    }
    if (s.fused) {
        TRY(dfdx_rocm_attention_forward(ctx, s.dtype, s.B, s.H, s.S, s.D, q, k, v, s.token, (float)s.scale, tok, s.token, (float *)(saved + l.lse)));
    } else {
        void *scores = scratch, *probs = saved + l.probs, *tokens = saved + l.tokens;
        const int64_t qs[4] = {s.token[0], s.D, s.d, 1}, ks[4] = {s.token[0], s.D, 1, s.d};
        const int64_t ps[4] = {s.H * s.S * s.S, s.S * s.S, s.S, 1}, shape[4] = {s.B, s.S, s.H, s.D}, ts[4] = {s.H * s.S * s.D, s.D, s.S * s.D, 1};
        TRY(dfdx_rocm_matmat_batch4_forward(ctx, s.dtype, s.B, s.H, s.S, s.D, s.S, q, qs, k, ks, scores));
        if (!s.folded) TRY(dfdx_rocm_scalar_mul_forward(ctx, s.dtype, s.B * s.H * s.S * s.S, scores, s.scale, scores));
        TRY(dfdx_rocm_softmax_forward(ctx, s.dtype, s.B * s.H * s.S, s.S, scores, s.folded ? (float)s.scale : 1.0f, probs));
        TRY(dfdx_rocm_matmat_batch4_forward(ctx, s.dtype, s.B, s.H, s.S, s.S, s.D, probs, ps, v, qs, tokens));
        TRY(dfdx_rocm_reshape_forward(ctx, s.dtype, 4, shape, ts, tokens, tok));
    }
    dfdx_rocm_gemm_desc g = linear(s, s.d, s.d, tok, p[WO], p[BO], h1);
    TRY(gemm_beyond(ctx, &g, EXTRA_RESIDUAL, x));
    TRY(dfdx_rocm_layer_norm_forward(ctx, s.dtype, s.T, s.d, h1, p[G1], p[BE1], 1e-5, n1));
    g = linear(s, s.d, s.ff, n1, p[W1], p[B1], r1);
    TRY(gemm_beyond(ctx, &g, EXTRA_RELU, nullptr));
    g = linear(s, s.ff, s.d, r1, p[W2], p[B2], h2);
    TRY(gemm_beyond(ctx, &g, EXTRA_RESIDUAL, n1));
    return dfdx_rocm_layer_norm_forward(ctx, s.dtype, s.T, s.d, h2, p[G2], p[BE2], 1e-5, out);
}

int backward(dfdx_rocm_ctx *ctx, const Shape &s, const dfdx_rocm_encoder *e, const dfdx_rocm_encoder_layout &l, const void *x,
             const char *saved, const void *grad_out, void *const *grads, void *grad_x, char *scratch) {
    const void *const *p = e->params;
    const void *q = saved + l.q, *k = saved + l.k, *v = saved + l.v, *tok = saved + l.tok, *h1 = saved + l.h1, *n1 = saved + l.n1,
               *h2 = saved + l.h2, *r1 = saved + l.r1;
    const size_t act = (size_t)(s.T * s.d) * s.es, mat = (size_t)(s.B * s.H * s.S * s.S) * s.es;
    Pieces at;
    void *gf1 = scratch + at.take((size_t)(s.T * s.ff) * s.es);
    void *gh2 = scratch + at.take(act), *gn1 = scratch + at.take(act), *gh1 = scratch + at.take(act), *gtok = scratch + at.take(act),
         *gq = scratch + at.take(act), *gk = scratch + at.take(act), *gv = scratch + at.take(act);
    // what the entry points below accumulate into counts as zero: every one of these is stored by its first use
    for (int i = 0; i < PARAM_COUNT; i++) TRY(dfdx_rocm_zero_deferred(ctx, grads[i], (size_t)param_size(s, i) * s.es));
    for (void *g : {gh2, gh1, gtok, gq, gk, gv}) TRY(dfdx_rocm_zero_deferred(ctx, g, act));

    TRY(dfdx_rocm_layer_norm_backward(ctx, s.dtype, s.T, s.d, h2, p[G2], 1e-5, gh2, grads[G2], grads[BE2], grad_out));
    // h2 = Linear2(r1) + n1: gh2 is the gradient of both
    dfdx_rocm_gemm_desc g = input_grad(s, s.ff, s.d, gh2, p[W2], gf1);
    TRY(linear_backward(ctx, s, g, EXTRA_MASK, r1, s.ff, s.d, r1, gh2, grads[W2], grads[B2]));
    g = input_grad(s, s.d, s.ff, gf1, p[W1], gn1);
    g.accumulate = 1;
    TRY(linear_backward(ctx, s, g, EXTRA_FROM, gh2, s.d, s.ff, n1, gf1, grads[W1], grads[B1]));
    TRY(dfdx_rocm_layer_norm_backward(ctx, s.dtype, s.T, s.d, h1, p[G1], 1e-5, gh1, grads[G1], grads[BE1], gn1));
    // h1 = Linear_o(tok) + x: gh1 is the gradient of both
    g = input_grad(s, s.d, s.d, gh1, p[WO], gtok);
    TRY(linear_backward(ctx, s, g, EXTRA_NONE, nullptr, s.d, s.d, tok, gh1, grads[WO], grads[BO]));
    if (s.fused) {
        TRY(dfdx_rocm_attention_backward(ctx, s.dtype, s.B, s.H, s.S, s.D, q, k, v, s.token, (float)s.scale, tok, gtok, s.token,
                                         (const float *)(saved + l.lse), gq, gk, gv));
    } else {
        const void *probs = saved + l.probs;
        void *gtokens = scratch + at.take(act), *gp = scratch + at.take(mat), *gscores = scratch + at.take(mat);
        void *gscaled = s.folded ? gscores : scratch + at.take(mat);
        TRY(dfdx_rocm_zero_deferred(ctx, gtokens, act));
        TRY(dfdx_rocm_zero_deferred(ctx, gp, mat));
        TRY(dfdx_rocm_zero_deferred(ctx, gscores, mat));
        if (!s.folded) TRY(dfdx_rocm_zero_deferred(ctx, gscaled, mat));
        const int64_t qs[4] = {s.token[0], s.D, s.d, 1}, ks[4] = {s.token[0], s.D, 1, s.d};
        const int64_t ps[4] = {s.H * s.S * s.S, s.S * s.S, s.S, 1}, shape[4] = {s.B, s.S, s.H, s.D}, ts[4] = {s.H * s.S * s.D, s.D, s.S * s.D, 1};
        TRY(dfdx_rocm_reshape_backward(ctx, s.dtype, 4, shape, ts, gtokens, gtok));
        TRY(dfdx_rocm_matmat_batch4_backward(ctx, s.dtype, s.B, s.H, s.S, s.S, s.D, probs, ps, gp, v, qs, gv, gtokens));
        TRY(dfdx_rocm_softmax_backward(ctx, s.dtype, s.B * s.H * s.S, s.S, probs, s.folded ? (float)s.scale : 1.0f, gscaled, gp));
        if (!s.folded) TRY(dfdx_rocm_scalar_mul_backward(ctx, s.dtype, s.B * s.H * s.S * s.S, s.scale, gscores, gscaled));
        TRY(dfdx_rocm_matmat_batch4_backward(ctx, s.dtype, s.B, s.H, s.S, s.D, s.S, q, qs, gq, k, ks, gk, gscores));
    }
    // x feeds the three projections and the residual: grad_x is one sum over their 3 d columns, rounded once
    bool summed = false, weights = false;
    GemmProblem sum = three(s.dtype, s.T, s.d, s.d, gq, s.d, 1, p[WQ], s.d, 1, grad_x);
    sum.reduce = 1;
    sum.accumulate = 1;
    sum.extra = EXTRA_FROM;
    sum.with = gh1;
    const bool may_sum = apart(gq, gk, gv, s.es, &sum.a_b1, &sum.a_b2) && apart(p[WQ], p[WK], p[WV], s.es, &sum.b_b1, &sum.b_b2);
    GemmProblem all = three(s.dtype, s.d, s.T, s.d, gq, 1, s.d, x, s.d, 1, grads[WQ]);  // weight (o, i) += grad_y^T . x, bias += sums of grad_y
    all.accumulate = 1;
    all.ksum = grads[BQ];
    all.ksum_of = KSUM_OF_A;
    all.ksum_accumulate = 1;
    const bool may_join = apart(gq, gk, gv, s.es, &all.a_b1, &all.a_b2) && apart(grads[WQ], grads[WK], grads[WV], s.es, &all.c_b1, &all.c_b2) &&
                          apart(grads[BQ], grads[BK_], grads[BV], s.es, &all.ksum_b1, &all.ksum_b2);
    if (may_sum && may_join) {
        g = input_grad(s, s.d, s.d, gq, p[WQ], grad_x);
        const dfdx_rocm_gemm_desc w = weight_product(s, s.d, s.d, x, gq, grads[WQ]);
        TRY(gemm_three_two(ctx, &g, &w, grads[BQ], sum, all, &summed));
        weights = summed;
    }
    if (may_sum && !summed) TRY(gemm_three(ctx, sum, &summed));
    if (may_join && !weights) TRY(gemm_three(ctx, all, &weights));
    for (int i = 0; i < 3; i++) {
        const int w = i == 0 ? WQ : i == 1 ? WK : WV;
        const void *gy = i == 0 ? gq : i == 1 ? gk : gv;
        if (!summed) {
            g = input_grad(s, s.d, s.d, gy, p[w], grad_x);
            g.accumulate = 1;
            TRY(gemm_beyond(ctx, &g, i == 0 ? EXTRA_FROM : EXTRA_NONE, i == 0 ? gh1 : nullptr));
        }
        if (!weights) TRY(weight_grad(ctx, s, s.d, s.d, x, gy, grads[w], grads[w + 1]));
    }
    return DFDX_ROCM_OK;
}

}  // namespace

extern "C" {

int dfdx_rocm_encoder_plan(dfdx_rocm_ctx *ctx, const dfdx_rocm_encoder *e, dfdx_rocm_encoder_layout *layout) {
    if (!ctx || !layout) return DFDX_ROCM_ERR_INVALID_ARG;
    Shape s;
    TRY(shape_of(e, &s));
    saved_layout(s, layout);
    return DFDX_ROCM_OK;
}

int dfdx_rocm_encoder_forward(dfdx_rocm_ctx *ctx, const dfdx_rocm_encoder *e, const void *x, void *out, void *saved, void *scratch) {
    TRY(bind(ctx));
    Shape s;
    TRY(shape_of(e, &s));
    dfdx_rocm_encoder_layout l;
    saved_layout(s, &l);
    if (s.T == 0) return DFDX_ROCM_OK;  // an empty batch has an empty result
    if (!x || !out || !saved || (l.forward_scratch_bytes && !scratch)) return DFDX_ROCM_ERR_INVALID_ARG;
    for (int i = 0; i < PARAM_COUNT; i++)
        if (!e->params[i]) return DFDX_ROCM_ERR_INVALID_ARG;
    return forward(ctx, s, e, l, x, out, (char *)saved, (char *)scratch);
}

int dfdx_rocm_encoder_backward(dfdx_rocm_ctx *ctx, const dfdx_rocm_encoder *e, const void *x, const void *saved, const void *grad_out,
                               void *const grads[DFDX_ROCM_ENCODER_PARAMS], void *grad_x, void *scratch) {
    TRY(bind(ctx));
    Shape s;
    TRY(shape_of(e, &s));
    dfdx_rocm_encoder_layout l;
    saved_layout(s, &l);
    if (!grads || (s.T && (!x || !saved || !grad_out || !grad_x || !scratch))) return DFDX_ROCM_ERR_INVALID_ARG;
    for (int i = 0; i < PARAM_COUNT; i++)
        if (!e->params[i] || !grads[i]) return DFDX_ROCM_ERR_INVALID_ARG;
    if (s.T == 0) {  // sums over no token
        for (int i = 0; i < PARAM_COUNT; i++) TRY(dfdx_rocm_memset_zero(ctx, grads[i], (size_t)param_size(s, i) * s.es));
        return DFDX_ROCM_OK;
    }
    const int rc = backward(ctx, s, e, l, x, (const char *)saved, grad_out, grads, grad_x, (char *)scratch);
    if (rc) {  // refused in mid-pass: no declaration made here outlives the call
        for (int i = 0; i < PARAM_COUNT; i++) (void)dfdx_rocm_forget_zeros(ctx, grads[i], (size_t)param_size(s, i) * s.es);
        (void)dfdx_rocm_forget_zeros(ctx, scratch, l.backward_scratch_bytes);
    }
    return rc;
}

}  // extern "C"
