// K2 streaming path, nearest-pixel resize from source rows at any byte phase to any destination: body in
// rmx_kernels_resize_dma_impl.h, forms PHASED and NEAREST. Bound by the memory system: 64 images of 384 x 512 to 256 x 256 bytes, of
// which 38 MB move, 11.6 us (the general kernel, which stages every row of a window through registers and gathers from a ring of
// rows: 22.0 us).
// Bytes to interleaved bytes are moved, not converted (see BYTES there): without its loads and stores the kernel still took 27 of 42 us on 144
// images of 410 x 417 to 433 x 284, half of it conversions to float and back. Whole batches: that one 39.0 -> 34.4 us, 64 images of 384 x
// 512 to 256 x 256 10.3 -> 9.5, 94 of 308 x 389 to 489 x 352 29.0 -> 25.7. (Windows of eight rows, whose taps are shared by more rows, leave
// fewer wavefronts: 37.9, 9.4 and 30.9.)
#include "rmx_kernels_resize_dma_impl.h"

namespace rmx {

template <typename T, int LAYOUT, bool NORM>
__global__ void __launch_bounds__(256) rmx_resize_near_kernel(RmxKArgs a) {
    resize_stream<T, LAYOUT, NORM, false, CHAIN_NONE, false, true, true>(a);
}

template <typename T>
static KernelFn pick(int layout, bool norm) {
    if (layout == RMX_NCHW) return norm ? (KernelFn)rmx_resize_near_kernel<T, RMX_NCHW, true> : (KernelFn)rmx_resize_near_kernel<T, RMX_NCHW, false>;
    return norm ? (KernelFn)rmx_resize_near_kernel<T, RMX_NHWC, true> : (KernelFn)rmx_resize_near_kernel<T, RMX_NHWC, false>;
}

// (the nearest pixel is a byte already: quantising it changes nothing)
KernelFn select_resize_near_kernel(int dtype, int layout, bool norm, const char **name) {
    *name = "rmx_resize_near_kernel";
    switch (dtype) {
        case RMX_FP32: return pick<float>(layout, norm);
        case RMX_FP16: return pick<__half>(layout, norm);
        default: return pick<uint8_t>(layout, norm);
    }
}

}  // namespace rmx
