// K2 streaming path, bilinear batches whose source rows all start at one byte phase (row strides that are multiples of 4): body
// in rmx_kernels_resize_dma_impl.h.
#include "rmx_kernels_resize_dma_impl.h"

namespace rmx {

template <typename T, int LAYOUT, bool NORM, bool QUANT, int CHAIN, bool ALIGNED>
__global__ void __launch_bounds__(256) rmx_resize_dma_kernel(RmxKArgs a) {
    resize_stream<T, LAYOUT, NORM, QUANT, CHAIN, ALIGNED, false, false>(a);
}

template <typename T, int LAYOUT, bool ALIGNED>
static KernelFn pick3(bool norm, bool quant, int chain) {
    if (norm && quant && chain == CHAIN_LINEAR) return (KernelFn)rmx_resize_dma_kernel<T, LAYOUT, true, true, CHAIN_LINEAR, ALIGNED>;
    if (norm && quant && chain == CHAIN_TWIST) return (KernelFn)rmx_resize_dma_kernel<T, LAYOUT, true, true, CHAIN_TWIST, ALIGNED>;
    if (norm && quant) return (KernelFn)rmx_resize_dma_kernel<T, LAYOUT, true, true, CHAIN_NONE, ALIGNED>;
    if (norm) return (KernelFn)rmx_resize_dma_kernel<T, LAYOUT, true, false, CHAIN_NONE, ALIGNED>;
    return (KernelFn)rmx_resize_dma_kernel<T, LAYOUT, false, false, CHAIN_NONE, ALIGNED>;
}

// aligned: the form for whole groups and 16-byte aligned rows; null for interleaved fp32, which is bound by its stores and has
// one such form for rows at any phase (rmx_resize_runs_kernel).
KernelFn select_resize_dma_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool aligned, const char **name) {
    *name = "rmx_resize_dma_kernel";
    if (!aligned) {
        if (layout == RMX_NCHW) {
            switch (dtype) {
                case RMX_FP32: return pick3<float, RMX_NCHW, false>(norm, quant, chain);
                case RMX_FP16: return pick3<__half, RMX_NCHW, false>(norm, quant, chain);
                default: return pick3<uint8_t, RMX_NCHW, false>(norm, quant, chain);
            }
        }
        switch (dtype) {
            case RMX_FP32: return pick3<float, RMX_NHWC, false>(norm, quant, chain);
            case RMX_FP16: return pick3<__half, RMX_NHWC, false>(norm, quant, chain);
            default: return pick3<uint8_t, RMX_NHWC, false>(norm, quant, chain);
        }
    }
    if (layout == RMX_NCHW) {
        switch (dtype) {
            case RMX_FP32: return pick3<float, RMX_NCHW, true>(norm, quant, chain);
            case RMX_FP16: return pick3<__half, RMX_NCHW, true>(norm, quant, chain);
            default: return pick3<uint8_t, RMX_NCHW, true>(norm, quant, chain);
        }
    }
    switch (dtype) {
        case RMX_FP32: return nullptr;
        case RMX_FP16: return pick3<__half, RMX_NHWC, true>(norm, quant, chain);
        default: return pick3<uint8_t, RMX_NHWC, true>(norm, quant, chain);
    }
}

}  // namespace rmx
