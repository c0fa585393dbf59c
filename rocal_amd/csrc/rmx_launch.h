// Host-side kernel selection: each kernel family exports a selector that maps the static
// node configuration to one template instantiation.
#pragma once
#include "rmx_common.h"

namespace rmx {
typedef void (*KernelFn)(RmxKArgs);

// norm: 0 plain values, 1 the row's scale and bias, 2 constants from the sample's own moments (Normalize)
KernelFn select_cmn_kernel(int dtype, int layout, int norm, int mode, const char **name);
KernelFn select_resize_linear_kernel(int dtype, int layout, bool norm, bool quant, int chain, const char **name);
KernelFn select_resize_fast_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool aligned, const char **name);
KernelFn select_resize_dma_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool aligned, const char **name);
// Whether a streaming resize kernel's lanes exchange their fp32 runs through LDS before storing (and how it is built: rmx_kernels_resize_dma_impl.h).
// The plan makes room for the exchange where this says so and nowhere else: 2 KB more than a full slice of 10 are three of sixteen
// wavefronts per CU. fp32 planes from rows at any phase, without room / with room that their kernel does not use: 96 windows to 160 x 160
// 16.0 / 18.4 us, 64 to 224 x 224 14.0 / 14.9, 100 to 200 x 200 15.9 / 16.5; 128 to 224 x 224, whose stores fewer wavefronts in
// flight disturb less, 32.5 / 31.3.
constexpr bool resize_exchanges(bool fp32, bool planes, bool aligned, bool twist) { return fp32 && (!planes || aligned || twist); }
KernelFn select_resize_near_kernel(int dtype, int layout, bool norm, const char **name);
KernelFn select_resize_split_kernel(int dtype, int layout, bool norm, bool quant, int chain, bool nearest);
KernelFn select_resize_nearest_kernel(int dtype, int layout, bool norm, bool quant, const char **name);
KernelFn select_resize_tri_kernel(int dtype, int layout, bool norm, bool quant, const char **name);
KernelFn select_resize_tri_down_kernel(int dtype, int layout, bool norm, bool quant, int columns_per_lane, const char **name);
KernelFn select_resize_tri_dma_kernel(int dtype, int layout, bool norm, bool quant, int rows_in_flight, const char **name);
KernelFn select_resize_tri_adj_kernel(int dtype, int layout, bool norm, bool quant, bool any_phase);
KernelFn select_color_kernel(int kind, int dtype, int layout, int mode, const char **name);
KernelFn select_point_kernel(int kind, int dtype, int layout, int mode, const char **name);
KernelFn select_transpose_kernel(int dtype, int layout, const char **name);
KernelFn select_warp_kernel(int interp, int dtype, int layout, bool raw, const char **name);
// Warps to interleaved bytes: how rows leave (see warp_body, rmx_kernels_warp.hip)
enum { RMX_WARP_LANES = 0, RMX_WARP_TILES = 1, RMX_WARP_TEAMS = 2 };
constexpr int kWarpTeam = 4, kWarpTileBytes = 32 * 32 * 3;  // tiles of a team; bytes of a tile's rows, of which a wavefront's slice must have room
KernelFn select_warp_rows_kernel(int interp, bool raw, int rows);
// Normalize: integer moments of every sample's window, 1 << log2_parts shares of six 64-bit numbers per sample, each made by a workgroup
// of `threads` (whole wavefronts, at most 512)
void launch_moments(hipStream_t stream, const RmxKArgs &a, unsigned long long *parts, int log2_parts, int threads);
void launch_copy(hipStream_t stream, const void *src, void *dst, size_t nbytes, int num_cus);
// mode 0 copy, 1 read only, 2 write only; groups_per_cu 0 = the default (16)
void launch_stream(hipStream_t stream, int mode, const void *src, void *dst, size_t nbytes, int num_cus, int groups_per_cu);
}  // namespace rmx
