// 3 x 3, unit-stride, padding-1 convolution forward for the 16-bit types without a patch matrix (conv3x3.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace dfdx_rocm {

struct Conv3x3Problem {
    int dtype;                 // DT_F16 / DT_BF16
    int batch, chan_in, chan_out, h, w;
    const void *img;           // [batch][chan_in][h][w]
    const void *filters;       // [chan_out][chan_in][3][3]; `transposed_filters`: [chan_in][chan_out][3][3], applied turned
                               // by 180 degrees (the image gradient of a convolution with these filters: img = its grad_out)
    void *out;                 // [batch][chan_out][h][w]
    int accumulate = 0;        // out += ... instead of out = ...
    int transposed_filters = 0;
    void *wt;                  // scratch for the filters as [chan_out][9][chan_in]: conv3x3_filter_bytes(), 16-byte aligned
};

bool conv3x3_supported(const Conv3x3Problem &c);
size_t conv3x3_filter_bytes(const Conv3x3Problem &c);
// hipErrorNotSupported when the shape does not fit (the caller then takes another path).  `laid`: c.wt is filled already.
hipError_t launch_conv3x3(const Conv3x3Problem &c, hipStream_t stream, bool laid = false);

// How c.filters become c.wt: wt[o][tap][c] = filters[o][c][tap] -- or, `transposed` (the image gradient: a convolution of grad_out
// with the filters turned by 180 degrees, input and output channels trading places), wt[c][tap][o] = filters[o][c][8 - tap].
// `inner` = the extent of wt's last axis without its padding with zeros (`padded`), `outer` = that of its first.
struct Conv3x3Filters {
    const void *filters;
    void *wt;
    int inner, padded, outer, transposed, total;
};
Conv3x3Filters conv3x3_filters(const Conv3x3Problem &c);
template <typename E> __device__ __forceinline__ void conv3x3_lay(const Conv3x3Filters &a, int i) {
    if (i >= a.total) return;
    const E *f = (const E *)a.filters;
    const int c = i % a.padded, tap = (i / a.padded) % 9, o = i / (9 * a.padded);
    ((E *)a.wt)[i] = c >= a.inner ? (E)0 : a.transposed ? f[((int64_t)c * a.outer + o) * 9 + (8 - tap)] : f[((int64_t)o * a.inner + c) * 9 + tap];
}

// The filter gradient of the same convolution without a patch matrix (conv3x3_wgrad.hip).  `c` as above with `out` =
// grad_out [batch][chan_out][h][w] and `filters` = grad_filters, added to (`accumulate`) or stored; `workspace`: f32 shares of the
// sums, conv3x3_wgrad_workspace_bytes(), 16-byte aligned.
bool conv3x3_wgrad_supported(const Conv3x3Problem &c, int compute_units);
size_t conv3x3_wgrad_workspace_bytes(const Conv3x3Problem &c, int compute_units);
// `next` (may be null): a convolution whose filters are laid beside the adding up of the shares.
hipError_t launch_conv3x3_wgrad(const Conv3x3Problem &c, int compute_units, void *workspace, hipStream_t stream, const Conv3x3Problem *next);

}  // namespace dfdx_rocm
