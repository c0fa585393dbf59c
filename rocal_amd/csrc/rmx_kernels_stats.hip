// Normalize (mean / standard deviation over the image axes of each sample): the pass in front of the streaming one.
//   rmx_moments_kernel  1 to RMX_MOMENT_PARTS workgroups per sample, each a share of the window's rows: per-channel sum and sum of
//                       squares as exact integers (bytes: no rounding, so the order of the additions does not matter), six
//                       64-bit numbers per workgroup, written to a workspace of the op.
// The streaming pass is the CropMirrorNormalize kernel in its form NORM_OWN: every wavefront adds its sample's shares up, makes
// mean and population standard deviation in double from the exact integer moments and from them its FMA constants
// a = scale / sigma, b = shift - mean * a (sigma = 0: a = 0, b = shift).
// What bounds this pass is the read of the batch. Bytes are sorted into one dword per channel (two v_perm per dword) and summed
// four at a time by v_dot4_u32_u8: one instruction per byte where extracting, adding and multiplying byte by byte took four and
// made the pass an arithmetic one (64 images of 300 x 400, 23 MB: 24.8 us, now 6 us). Shares instead of atomic counters
// take the launch that cleared the counters with them, and the constants made by the streaming wavefronts the launch that
// wrote them into the table (zero 3.3 + moments 24.8 + constants 4.6 us before).
#include "rmx_device.h"
#include "rmx_launch.h"

namespace rmx {

constexpr int MOM_THREADS = 512;  // at most
constexpr int MOM_WAVES = MOM_THREADS / RMX_WAVE;

// sum over the wavefront, in lane 63 (row shifts inside rows of 16 lanes, then the broadcasts of their last lanes)
RMX_DEV uint32_t wave_sum_lane63(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, true);  // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, true);  // row_bcast:31 into rows 2 and 3
    return v;
}

// WHOLE: workgroups of MOM_THREADS (told by the type: 64 images of 300 x 400 lose 0.1 us to a size that is read first)
template <bool WHOLE>
__global__ void __launch_bounds__(MOM_THREADS) rmx_moments_kernel(RmxKArgs a, unsigned long long *parts, int log2_parts) {
    __shared__ unsigned long long wave_sums[MOM_WAVES][6];
    const int s = (int)(blockIdx.x >> log2_parts), part = (int)(blockIdx.x & ((1u << log2_parts) - 1u));
    const int threads = WHOLE ? MOM_THREADS : (int)blockDim.x;
    const RmxSample P = load_sample<RMX_C_WINDOW | RMX_C_DST>(a, s);
    const int w = max(P.dst_w, 0), h = max(P.dst_h, 0);
    const int r0 = (int)(((long long)h * part) >> log2_parts), r1 = (int)(((long long)h * (part + 1)) >> log2_parts);
    uint32_t row_stride;
    const uint8_t *simg = sample_base(a, s, row_stride);
    const uint8_t *first = simg + (size_t)P.src_y * row_stride + (size_t)P.src_x * 3;
    const uint8_t *buf_end = a.src + a.src_bytes;

    // groups of 8 pixels, row after row, dealt to the threads
    const int groups = (w + PX - 1) / PX;
    const int dr = groups ? threads / groups : 0, dg = threads - dr * groups;
    int r = r0 + (groups ? (int)threadIdx.x / groups : 0), g = groups ? (int)threadIdx.x % groups : 0;
    if (groups == 0) r = r1;
    unsigned long long total[6] = {};
    while (r < r1) {
        // (32-bit sums inside a block of 1024 groups per thread: 8 x 1024 x 255^2 < 2^32)
        uint32_t sum[3] = {0, 0, 0}, sq[3] = {0, 0, 0};
        constexpr int NI = 4;  // groups whose loads are in flight together
        for (int k = 0; k < 1024 / NI && r < r1; k++) {
            uint32_t d[NI][6];
            int cnt[NI];
#pragma unroll
            for (int i = 0; i < NI; i++) {
                cnt[i] = r < r1 ? min(PX, w - g * PX) : 0;
                const int rr = min(r, r1 - 1);
                load_realigned<7>(first + (size_t)rr * row_stride + (size_t)g * (PX * 3), buf_end, d[i]);
                r += dr;
                g += dg;
                if (g >= groups) {
                    g -= groups;
                    r++;
                }
            }
#pragma unroll
            for (int i = 0; i < NI; i++) {
                if (cnt[i] < PX) {
                    const int nb = 3 * cnt[i];
#pragma unroll
                    for (int j = 0; j < 6; j++) {
                        const int have = nb - 4 * j;  // bytes of this dword that belong to the window
                        d[i][j] = have >= 4 ? d[i][j] : (have <= 0 ? 0u : d[i][j] & ((1u << (8 * have)) - 1u));
                    }
                }
#pragma unroll
                for (int j = 0; j < 6; j += 3) {
                    const uint32_t w0 = d[i][j], w1 = d[i][j + 1], w2 = d[i][j + 2];
                    // bytes 0 3 6 9 | 1 4 7 10 | 2 5 8 11 of the twelve (selectors 0..3 take the second operand, 4..7 the first, 12 is zero)
                    const uint32_t c[3] = {__builtin_amdgcn_perm(w2, __builtin_amdgcn_perm(w1, w0, 0x0c060300u), 0x05020100u),
                                           __builtin_amdgcn_perm(w2, __builtin_amdgcn_perm(w1, w0, 0x0c070401u), 0x06020100u),
                                           __builtin_amdgcn_perm(w2, __builtin_amdgcn_perm(w1, w0, 0x0c0c0502u), 0x07040100u)};
#pragma unroll
                    for (int ch = 0; ch < 3; ch++) {
                        sum[ch] = __builtin_amdgcn_udot4(c[ch], 0x01010101u, sum[ch], false);
                        sq[ch] = __builtin_amdgcn_udot4(c[ch], c[ch], sq[ch], false);
                    }
                }
            }
        }
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            total[ch] += sum[ch];
            total[3 + ch] += sq[ch];
        }
    }
    const bool small = (long long)(r1 - r0) * w <= 65536;  // (65536 x 255^2 < 2^32: the sums of the whole workgroup are 32-bit)
#pragma unroll
    for (int k = 0; k < 6; k++) {
        if (small) {
            total[k] = wave_sum_lane63((uint32_t)total[k]);
        } else {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) total[k] += __shfl_xor(total[k], off, RMX_WAVE);
        }
        if ((threadIdx.x & (RMX_WAVE - 1)) == RMX_WAVE - 1) wave_sums[threadIdx.x / RMX_WAVE][k] = total[k];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned long long t = 0;
#pragma unroll
        for (int v = 0; v < MOM_WAVES; v++) t += v * RMX_WAVE < threads ? wave_sums[v][threadIdx.x] : 0ull;
        parts[(((size_t)s * 6 + threadIdx.x) << log2_parts) + part] = t;
    }
}

void launch_moments(hipStream_t stream, const RmxKArgs &a, unsigned long long *parts, int log2_parts, int threads) {
    hipLaunchKernelGGL(threads == MOM_THREADS ? rmx_moments_kernel<true> : rmx_moments_kernel<false>, dim3((unsigned)a.n << log2_parts), dim3(threads), 0, stream, a, parts, log2_parts);
}

}  // namespace rmx
