// K2 streaming path, bilinear batches whose source rows start at any byte phase (images of odd widths packed without padding, or
// padded to an odd width), and interleaved fp32 outputs of whole groups: body in rmx_kernels_resize_dma_impl.h, form PHASED.
// Replaces a kernel that staged windows through registers (16-byte loads, realignment to one dword per pixel, LDS stores:
// about 25 instructions per 4 source pixels) and, for destinations that are no whole aligned groups, the general kernel. Measured,
// kernel alone: 128 packed RandomResizedCrop images to 224 x 224 fp16 23.9 -> 19.7 us (staged before); 13 frames of 585 x 1831 to
// 276 x 863 fp32 planes 107 -> 27.8 us, 20 images of 247 x 207 to 156 x 156 fp16 12.8 -> 6.7 us (general kernel before).
#include "rmx_kernels_resize_dma_impl.h"

namespace rmx {

template <typename T, int LAYOUT, bool NORM, bool QUANT, int CHAIN>
__global__ void __launch_bounds__(256) rmx_resize_fast_kernel(RmxKArgs a) {
    resize_stream<T, LAYOUT, NORM, QUANT, CHAIN, false, true, false>(a);
}

// Interleaved fp32 of whole groups at 16-byte aligned rows, source rows at any phase: bound by its stores, and a row's runs leave as
// whole 16-byte pieces without a head, a tail or a loop over them (128 windows to 224 x 224 from rows at one phase / at any: the form for
// any destination 40.1 / 34.4 us a launch, this one 34.0 / 28.7).
template <bool NORM, bool QUANT, int CHAIN>
__global__ void __launch_bounds__(256) rmx_resize_runs_kernel(RmxKArgs a) {
    resize_stream<float, RMX_NHWC, NORM, QUANT, CHAIN, true, true, false>(a);
}

static KernelFn pick_runs(bool norm, bool quant, int chain) {
    if (norm && quant && chain == CHAIN_LINEAR) return (KernelFn)rmx_resize_runs_kernel<true, true, CHAIN_LINEAR>;
    if (norm && quant && chain == CHAIN_TWIST) return (KernelFn)rmx_resize_runs_kernel<true, true, CHAIN_TWIST>;
    if (norm && quant) return (KernelFn)rmx_resize_runs_kernel<true, true, CHAIN_NONE>;
    if (norm) return (KernelFn)rmx_resize_runs_kernel<true, false, CHAIN_NONE>;
    return (KernelFn)rmx_resize_runs_kernel<false, false, CHAIN_NONE>;
}

template <typename T, int LAYOUT>
static KernelFn pick3(bool norm, bool quant, int chain) {
    if (norm && quant && chain == CHAIN_LINEAR) return (KernelFn)rmx_resize_fast_kernel<T, LAYOUT, true, true, CHAIN_LINEAR>;
    if (norm && quant && chain == CHAIN_TWIST) return (KernelFn)rmx_resize_fast_kernel<T, LAYOUT, true, true, CHAIN_TWIST>;
    if (norm && quant) return (KernelFn)rmx_resize_fast_kernel<T, LAYOUT, true, true, CHAIN_NONE>;
    if (norm) return (KernelFn)rmx_resize_fast_kernel<T, LAYOUT, true, false, CHAIN_NONE>;
    return (KernelFn)rmx_resize_fast_kernel<T, LAYOUT, false, false, CHAIN_NONE>;
}

// chain: 0 none, 1 linear colour node, 2 colour twist between resize and normalisation (only with norm and quant)
// aligned: whole groups and 16-byte aligned rows
KernelFn select_resize_fast_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool aligned, const char **name) {
    *name = "rmx_resize_fast_kernel";
    if (layout == RMX_NCHW) {
        switch (dtype) {
            case RMX_FP32: return pick3<float, RMX_NCHW>(norm, quant, chain);
            case RMX_FP16: return pick3<__half, RMX_NCHW>(norm, quant, chain);
            default: return pick3<uint8_t, RMX_NCHW>(norm, quant, chain);
        }
    }
    switch (dtype) {
        case RMX_FP32: return aligned ? pick_runs(norm, quant, chain) : pick3<float, RMX_NHWC>(norm, quant, chain);
        case RMX_FP16: return pick3<__half, RMX_NHWC>(norm, quant, chain);
        default: return pick3<uint8_t, RMX_NHWC>(norm, quant, chain);
    }
}

}  // namespace rmx
