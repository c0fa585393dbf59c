// K2 streaming path for batches that leave wavefront slots of the chip idle: several wavefronts share the x-tiles of a window (body in
// rmx_kernels_resize_dma_impl.h, form SPLIT), instead of one that works through them and waits for every tile's source pixels anew; when
// the host takes it, and what that gives, stands there (plan_resize, rmx_api.hip). Such launches wait for memory, so the
// form for rows at any phase and any destination serves all of them. Kernels of their own: the few scalar instructions in front of every
// wavefront's first load, in the kernels that the other batches take, cost those up to 1.4 % (100 windows to 173 x 173 interleaved fp32 19.2 ->
// 19.5 us).
#include "rmx_kernels_resize_dma_impl.h"

namespace rmx {

template <typename T, int LAYOUT, bool NORM, bool QUANT, int CHAIN, bool NEAREST>
__global__ void __launch_bounds__(256) rmx_resize_split_kernel(RmxKArgs a) {
    resize_stream<T, LAYOUT, NORM, QUANT, CHAIN, false, true, NEAREST, true>(a);
}

template <typename T, int LAYOUT>
static KernelFn pick(bool norm, bool quant, int chain, bool nearest) {
    if (nearest) return norm ? (KernelFn)rmx_resize_split_kernel<T, LAYOUT, true, false, CHAIN_NONE, true> : (KernelFn)rmx_resize_split_kernel<T, LAYOUT, false, false, CHAIN_NONE, true>;
    if (norm && quant && chain == CHAIN_LINEAR) return (KernelFn)rmx_resize_split_kernel<T, LAYOUT, true, true, CHAIN_LINEAR, false>;
    if (norm && quant && chain == CHAIN_TWIST) return (KernelFn)rmx_resize_split_kernel<T, LAYOUT, true, true, CHAIN_TWIST, false>;
    if (norm && quant) return (KernelFn)rmx_resize_split_kernel<T, LAYOUT, true, true, CHAIN_NONE, false>;
    if (norm) return (KernelFn)rmx_resize_split_kernel<T, LAYOUT, true, false, CHAIN_NONE, false>;
    return (KernelFn)rmx_resize_split_kernel<T, LAYOUT, false, false, CHAIN_NONE, false>;
}

KernelFn select_resize_split_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool nearest) {
    const bool planar = layout == RMX_NCHW;
    switch (dtype) {
        case RMX_FP32: return planar ? pick<float, RMX_NCHW>(norm, quant, chain, nearest) : pick<float, RMX_NHWC>(norm, quant, chain, nearest);
        case RMX_FP16: return planar ? pick<__half, RMX_NCHW>(norm, quant, chain, nearest) : pick<__half, RMX_NHWC>(norm, quant, chain, nearest);
        default: return planar ? pick<uint8_t, RMX_NCHW>(norm, quant, chain, nearest) : pick<uint8_t, RMX_NHWC>(norm, quant, chain, nearest);
    }
}

}  // namespace rmx
