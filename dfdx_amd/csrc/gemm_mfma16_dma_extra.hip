// The instances of the LDS-DMA kernel that do one thing more to a finished value on its way into C (EXTRA_* in
// gemm_internal.h), for the two operand layouts that ask for it: a Linear layer's forward (both operands stored along k:
// RELU, RESIDUAL) and its input gradient (the weight stored across k: MASK, FROM).  They save the pass over C that the op behind
// the product would make: 8192 x 4096 bf16 (67 MB) costs ReLU 23 us forward and 34 us backward as a kernel of its own.
#include "gemm_mfma16_dma.h"

namespace dfdx_rocm {
namespace {

template <typename T, int BM, int BN, int WM, int WN> hipError_t launch_extra(Params p, int extra, int compute_units, hipStream_t stream) {
    constexpr int NT = WM * WN * 64;
    constexpr size_t lds = (size_t)STAGES * (BM + BN) * BK * 2;
    const bool edge = needs_edge_form<BM, BN>(p);
    switch (extra) {
    case EXTRA_RELU:
        if (edge) DFDX_LAUNCH(true, true, true, false, EXTRA_RELU);
        else DFDX_LAUNCH(true, true, false, false, EXTRA_RELU);
        break;
    case EXTRA_RESIDUAL:
        if (edge) DFDX_LAUNCH(true, true, true, false, EXTRA_RESIDUAL);
        else DFDX_LAUNCH(true, true, false, false, EXTRA_RESIDUAL);
        break;
    case EXTRA_MASK:
        if (edge) DFDX_LAUNCH(true, false, true, false, EXTRA_MASK);
        else DFDX_LAUNCH(true, false, false, false, EXTRA_MASK);
        break;
    case EXTRA_FROM:
        if (edge) DFDX_LAUNCH(true, false, true, false, EXTRA_FROM);
        else DFDX_LAUNCH(true, false, false, false, EXTRA_FROM);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T> hipError_t launch_variant(int variant, int extra, const Params &p, int compute_units, hipStream_t s) {
    switch (variant) {
#define X(id, bm, bn, wm, wn) \
    case id: return launch_extra<T, bm, bn, wm, wn>(p, extra, compute_units, s);
        DFDX_MFMA16_DMA_VARIANTS(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_mfma16dma_extra(int variant, int dtype, int extra, const DmaParams &p, int compute_units, hipStream_t stream) {
    return dtype == DT_F16 ? launch_variant<_Float16>(variant, extra, p, compute_units, stream)
                           : launch_variant<__bf16>(variant, extra, p, compute_units, stream);
}

}  // namespace dfdx_rocm
