// Where the pieces of a warp's boxes come from, for windows of one to four rows and columns at the corners and inside of images at both
// ends of a batch buffer, at every byte phase, and maps that put tiles on every side of the window: no piece that is loaded
// without a look at the buffer's ends lies outside of it, and none lands outside the wavefront's LDS slice. Built and run by
// tests/test_warp_box_cpu.py.
#include <math.h>
#include <stdio.h>

#include "rmx_warp_box.h"

static long boxes, unchecked, outside, slice;

// start: byte of the buffer at which the image begins (the buffer itself begins at a dword), bytes: the buffer's length
template <bool NEAREST, bool RAW>
static void walk(long start, long bytes, uint32_t row_stride, const int *win, int dw, int dh, const float *m, int passes) {
    const int lds_bytes = 16 * 1024;
    const uint32_t skew = (uint32_t)(start & 3);
    const long base4 = start - skew;
    for (int Y0 = 0; Y0 < dh; Y0 += rmx::WTH * passes)
        for (int X0 = 0; X0 < dw; X0 += rmx::WTW) {
            const rmx::WarpBox b = rmx::warp_box<NEAREST, RAW>(win[0], win[1], win[2], win[3], dw, dh, m[0], m[1], m[2], m[3], m[4], m[5], X0, Y0, passes, skew, row_stride, lds_bytes);
            if (!b.use_lds) continue;
            boxes++;
            slice += 16 * b.total > lds_bytes || (b.bh - 1) * b.pitch_b + b.ph + 3 * (b.bw + 1) > lds_bytes;
            if (!rmx::warp_box_inside<RAW>(b, row_stride, (uint64_t)(bytes - base4))) continue;
            unchecked++;
            const float inv = 1.0f / (float)(RAW ? b.ppr : b.pitch_b);
            for (int i = 0; i < b.total; i++) {
                const long at = base4 + (long)(uint32_t)rmx::warp_piece<RAW>(b, row_stride, i, inv);
                if (at < 0 || at + 16 > bytes) {
                    if (!outside++) printf("first: buffer of %ld, image at %ld, window %d %d %d %d, tile %d %d: piece %d at %ld\n", bytes, start, win[0], win[1], win[2], win[3], X0, Y0, i, at);
                    break;
                }
            }
        }
}

int main() {
    for (int w : {200, 201, 64, 37})
        for (int h : {1, 2, 3, 50}) {
            const uint32_t row_stride = 3u * w;
            const long image = (long)row_stride * h;
            for (long start : {0l, 1l, image}) {  // (the first image at a dword and off it, the last of two)
                const long bytes = start + image;
                for (int ww : {1, 2, 4, w})
                    for (int wh : {1, 2, 3, h}) {
                        if (ww > w || wh > h) continue;
                        for (int corner = 0; corner < 4; corner++) {
                            const int win[4] = {(corner & 1) ? w - ww : 0, (corner & 2) ? h - wh : 0, ww, wh};
                            for (float angle : {0.0f, 0.1f, 0.7853982f, 1.5707964f, -0.5f, 3.1415927f})
                                for (float scale : {1.0f, 1.1f, 0.5f}) {
                                    const float c = scale * cosf(angle), s = scale * sinf(angle);
                                    for (float sx : {0.0f, -60.5f, 25.0f})
                                        for (float sy : {0.0f, -0.5f, 0.25f, 1.0f, 25.0f, -25.5f, 40.75f}) {
                                            const float m[6] = {c, s, sx, -s, c, sy};
                                            const int dw = w, dh = h < 48 ? 48 : h;
                                            if (row_stride % 4 == 0) {
                                                walk<false, true>(start, bytes, row_stride, win, dw, dh, m, 2);
                                                walk<true, true>(start, bytes, row_stride, win, dw, dh, m, 1);
                                            }
                                            walk<false, false>(start, bytes, row_stride, win, dw, dh, m, 2);
                                            walk<true, false>(start, bytes, row_stride, win, dw, dh, m, 1);
                                        }
                                }
                        }
                    }
            }
        }
    printf("%ld boxes, %ld loaded unchecked, %ld of them leave the buffer, %ld leave the slice\n", boxes, unchecked, outside, slice);
    return outside != 0 || slice != 0 || unchecked == 0 || unchecked == boxes;
}
