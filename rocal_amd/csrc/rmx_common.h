// Shared host/device definitions of the MI355X augmentation library: the per-sample row of
// the per-batch parameter table, kernel launch arguments and host-side bookkeeping.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "../../include/rocal_mi355x.h"

// One row per sample; the whole batch's table is uploaded once per update and every
// workgroup reads its sample's row with scalar loads (the row index is wave-uniform).
struct __attribute__((aligned(16))) RmxSample {
    int32_t src_x, src_y, src_w, src_h;  // source window in pixels (ROI or crop), XYWH
    int32_t dst_w, dst_h;                // valid output size written for this sample
    int32_t pc_x, pc_y;                  // offset of the written window inside the virtual resized image
    int32_t rs_w, rs_h;                  // virtual resized size (== dst when there is no post-crop)
    uint32_t flags;                      // RMX_S_*
    int32_t strip_rows;                  // output rows per wave strip for this sample; Normalize: shares of its moments (log2)
    float rx, ry;                        // src_len / rs_len, the IEEE quotient
    float fsx, fsy;                      // triangular: ratio > 1 ? 1/ratio : 1
    float scale[3], bias[3];             // normalisation: out = v*scale + bias
    union {
        float color[4];                  // colour twist: alpha, beta, hue shift in sextants [0,6], saturation
        int32_t plan[4];                 // [1] x-tile width of the streaming resize kernels; triangular: RMX_TRI_FOUR / RMX_TRI_EIGHT, [2] the row's sample
    };
    float m[6];                          // warp: destination -> source affine about the centres
};
static_assert(sizeof(RmxSample) == 128, "parameter table row must stay 128 bytes");

// Where a sample's image lies when the source is not one padded [N,Hmax,Wmax,3] tensor: tightly packed images of
// different sizes, one after the other (or anywhere) in one buffer.
struct RmxSrcLayout {
    uint64_t offset;      // bytes from the source base to the sample's first pixel
    uint32_t row_stride;  // bytes per image row
    uint32_t rows;        // image height
};
static_assert(sizeof(RmxSrcLayout) == 16, "source layout entry must stay 16 bytes");

enum : uint32_t {
    RMX_S_HFLIP = 1u,
    RMX_S_VFLIP = 2u,
    RMX_S_CHREV = 4u,    // output channel k reads source channel 2-k
    RMX_S_OWN_MEAN = 16u,  // Normalize: the mean / the deviation is the window's own (else m[0..2] / m[3..5]), one per channel or one
    RMX_S_OWN_STD = 32u,   // for all three; color[0] and color[1] are scale and shift
    RMX_S_PER_CHANNEL = 64u,
    RMX_S_EDGE_REF = 8u  // bilinear: both neighbours clamp to the window's last-but-one column / row (RMX_F_EDGE_REF)
};

// A batch whose rows differ in little (crop windows and mirror flags, colour factors, a matrix) travels in the kernel's
// arguments: one row of what all samples share and a few dwords per sample, from which load_sample() (rmx_device.h) makes the
// row again. A table in device memory costs a launch of its own in front of every batch's kernel (the upload, 3 - 4 us on the
// GPU and, with the event that guards its slot, 8 us of the host), the arguments 1 us of the host. A kernel launched again and again on
// the rows of one update is 0.1 - 0.8 us longer with them than with a table that stays in the caches (256 windows 40.5 -> 40.8 us, bytes
// 21.9 -> 22.3, 128 windows with antialiasing 41.2 -> 41.9). Whole batches, one update and launch after the other: 256 RandomResizedCrop windows to 224 x 224 fp16
// 37.4 -> 31.5 us, 128 crops of 224 x 224 to fp32 planes 22.2 -> 16.8 us, 14 small crops 16.9 -> 11.0 us. What a sample's dwords hold, in this order:
enum : uint32_t {
    RMX_C_ON = 1u,        // the rows are in the arguments
    RMX_C_WINDOW = 2u,    // two dwords: x, y, w, h in 14 bits each, mirror flags, the x-tile width's code (see compact_rows, rmx_api.hip)
    RMX_C_DST = 4u,       // (nothing stored) the written size is the window's
    RMX_C_RATIO = 8u,     // (nothing stored) rx, ry, fsx, fsy are quotients of the sizes
    RMX_C_COLOR0 = 16u,   // color[0..3], one dword each, those that differ between samples (four bits from here)
    RMX_C_M4 = 256u,      // m[0..3]
    RMX_C_M6 = 512u,      // m[0..5]
    RMX_C_ORDER = 1024u,  // the sample this row belongs to (plan[2])
    RMX_C_CROP = 4096u,   // two dwords behind the window's: a resize whose samples write windows of their own (pc_x, pc_y, dst_w, dst_h)
    RMX_C_LAYOUT = 2048u  // two dwords, of the sample and not of the row: source offset (40 bits) and row stride (24 bits)
};
constexpr int RMX_C_WORDS = 768;  // 3 KB of the 4 KB that arguments may take: 384 windows, 256 with their order, 192 colour twists, 128 matrices
constexpr int RMX_C_PAD = 4;      // (load_sample reads this many dwords from a record's start, however many it has)
constexpr int RMX_C_TILE_WHOLE = 512;  // code k of an x-tile width: 0 the whole row (up to this many pixels), else this >> k
// Output rows that a source row of the sample may enter, in the streaming triangular kernel with eight accumulator sets (as x-tile
// widths, so that a record holds them as it holds those).
constexpr int RMX_TRI_FOUR = RMX_C_TILE_WHOLE >> 1, RMX_TRI_EIGHT = RMX_C_TILE_WHOLE >> 2;

struct RmxKArgs {
    const uint8_t *src;      // batch base, u8 NHWC
    void *dst;               // batch base
    const RmxSample *table;  // device table, n rows
    uint64_t src_bytes;      // total bytes of the source batch (bounds the wide loads)
    int32_t n;
    int32_t src_h, src_w;    // padded source dims (pixels); row stride = src_w*3
    int32_t dst_h, dst_w;    // padded destination dims
    int32_t strips;          // wave strips per sample (grid = n*strips waves)
    int32_t lds_bytes;       // dynamic LDS per wave
    int32_t aux0, aux1;
    int32_t wpb;             // wavefronts per workgroup of this launch
    uint32_t nblocks;        // workgroups of this launch
    const RmxSrcLayout *layout;  // per-sample source placement, or null: sample s starts at s*src_h*src_w*3
    const uint8_t *src2;         // second source batch of the same shape (Blend), else null
    const uint8_t *extra;        // per-sample side table behind the layout entries (Gamma: 256 bytes per sample), else null
    // wavefront -> (sample, strip) without a division, and samples dealt round-robin to the XCDs (see wave_to_sample)
    uint32_t inv_strips;         // ceil(2^32 / strips), or 0: divide
    uint32_t per_xcd, inv_per_xcd;  // samples per XCD (n / 8) and ceil(2^32 / per_xcd); per_xcd 0: samples in batch order
    uint32_t compact;            // RMX_C_*: 0 when the rows are in `table`
    uint32_t compact_words;      // dwords per sample in `rec`
    RmxSample shared;            // what every sample's row holds
    uint32_t rec[RMX_C_WORDS + RMX_C_PAD];
};
static_assert(sizeof(RmxKArgs) <= 4096, "kernel arguments are limited to 4 KB");

// a / b, correctly rounded, for whole numbers a and b of up to 14 bits and recip = 1 / b correctly rounded: the product with the
// reciprocal is off by an ulp at most, its remainder is exact, and one correction of the quotient by it rounds as the
// division does (Markstein, IBM J. Res. Dev. 34, 1990; every pair is checked by tests/test_quotients_cpu.py).
__host__ __device__ inline float ratio_of(float a, float b, float recip) {
    const float q = a * recip;
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), recip, q);
}

#define RMX_WAVE 64
#define RMX_MOMENT_PARTS 64  // workgroups per sample of the moments pass (Normalize) at most

// Hue shift of a sample in sextants (ColorTwist, Hue, Saturation). A pixel's hue before it is brought back into [0, 6] lies in
// [shift - 1.0000002, shift + 5.0000002]; below RMX_HUE_SHIFT_LOW it can never reach 6, from RMX_HUE_SHIFT_HIGH on never fall
// below 0, and one comparison brings it back. The host picks the twist kernel with the single comparison for batches in
// which every sample's shift is on one side or the other; the kernel tells the sides apart with the same comparison.
#define RMX_HUE_SHIFT_LOW 0.99998f
#define RMX_HUE_SHIFT_HIGH 1.00002f
