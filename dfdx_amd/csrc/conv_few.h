// Convolutions of images with one or three channels (conv_few.hip): the first layer of a network, f16 / bf16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dfdx_rocm {

struct ConvFew {
    int dtype, kernel, stride;
    int batch, chan_in, chan_out, h_in, w_in, h_out, w_out;
    const void *img, *filters, *grad_out;
    void *out, *grad_img, *grad_filters;
    int fresh_img, fresh_filters;         // that gradient is stored instead of added to
    int compute_units;
};

bool conv_few_forward_supported(const ConvFew &c);
hipError_t launch_conv_few_forward(const ConvFew &c, hipStream_t stream);
bool conv_few_backward_supported(const ConvFew &c);
size_t conv_few_workspace_bytes(const ConvFew &c);  // partial sums of the filter gradient
hipError_t launch_conv_few_backward(const ConvFew &c, void *workspace, hipStream_t stream);

}  // namespace dfdx_rocm
