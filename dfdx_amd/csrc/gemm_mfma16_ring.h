// The interface of gemm_mfma16_ring.hip to the planner of the LDS-DMA kernels (gemm_mfma16_dma.hip), whose last variants these are.
#pragma once
#include "gemm_internal.h"

namespace dfdx_rocm {

struct RingParams {
    const uint16_t *a, *b, *bias, *with;
    uint16_t *c, *ksum;
    float *ws, *ws_ksum;  // f32 partial tiles [batch * splits + split][tiles_m * BM][tiles_n * BN] and row sums [batch * splits + split][tiles_m * BM]
    int64_t ldc;
    int64_t a_b1, a_b2, b_b1, b_b2, c_b1, c_b2, bias_b1, bias_b2, ksum_b1, ksum_b2;
    int64_t ws_ld, ws_split_stride;
    int m, n, k, lda, ldb;
    int nb2, kbatches;
    int tiles_m, tiles_n, tiles_per_batch, items;
    int accumulate, bias_mode, extra, ksum_accumulate;
    int group_m, splits, chunk, ws_ksum_stride;
    int whole;               // k tiles in front of a last one that is not whole, or lies apart: a_last, b_last elements from its place
    int64_t a_last, b_last;
};

// X(id, BM, BN, WAVES_M, WAVES_N, stages); ids go on behind and between those of gemm_mfma16_dma.h.
#define DFDX_MFMA16_RING_VARIANTS(X) \
    X(6, 64, 64, 2, 2, 4)            \
    X(7, 64, 64, 2, 2, 3)            \
    X(8, 128, 64, 2, 2, 3)           \
    X(9, 128, 128, 2, 4, 4)          \
    X(11, 192, 64, 4, 2, 4)

// A backward pass: `p` with A stored along k, `q` with both operands stored across k, in one launch.
hipError_t launch_mfma16_ring_two(int ring, int dtype, const RingParams &p, const RingParams &q, bool p_b_kc, hipStream_t stream);
hipError_t launch_mfma16_ring(int ring, int dtype, const RingParams &p, bool a_kc, bool b_kc, hipStream_t stream);

}  // namespace dfdx_rocm
