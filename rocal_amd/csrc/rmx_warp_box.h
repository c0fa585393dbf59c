// The box of source pixels that one tile of a warp reads: its bounds, how its rows lie in LDS, where its 16-byte pieces come from, and
// whether they all lie inside the batch buffer. Numbers only, shared by the kernel and by tests/cpp/warp_box.cpp, which walks the
// pieces of windows at the ends of a buffer: a byte read outside of it never reaches an output, so no comparison of values shows it.
#pragma once
#include "rmx_common.h"

namespace rmx {

#define RMX_BOX __host__ __device__ inline

constexpr int WTW = 32, WTH = 16;      // destination tile: 4 lanes x 8 px wide, 16 rows per pass
constexpr int kWarpRawPieces = 10;     // LDS pitch, in 16-byte pieces, at which every box that fits it is staged

RMX_BOX int box_min(int x, int y) { return x < y ? x : y; }
RMX_BOX int box_max(int x, int y) { return x > y ? x : y; }
RMX_BOX int box_mul24(int x, int y) {  // (numbers of up to 24 bits)
#ifdef __HIP_DEVICE_COMPILE__
    return __mul24(x, y);
#else
    return x * y;
#endif
}

struct WarpBox {
    int xlo, ylo, xhi, yhi;  // the window (inclusive)
    int bx0, bx1, by0, by1;  // the box: the tile's image with the right and lower neighbours, clipped to the window
    int bw, bh;
    int nr;                  // rows in LDS: bh, and one more where a tap can lie in the box's last row
    int ppr;                 // RAW: 16-byte pieces per row
    int pitch_b;             // LDS bytes per row
    int ph;                  // LDS byte of the box's first pixel
    int total;               // 16-byte pieces
    uint32_t colb;           // byte of column bx0 in a source row, from the dword that holds the image's first byte
    bool empty;              // no pixel of the tile lies in the window
    bool all_in;             // all of them do
    bool use_lds;            // the box fits the slice
};

// P: window and written size, m: destination -> source, (X0, Y0): the tile; skew: byte phase of the image's first pixel in its dword.
template <bool NEAREST, bool RAW>
RMX_BOX WarpBox warp_box(int src_x, int src_y, int src_w, int src_h, int dw, int dh, float m0, float m1, float m2, float m3, float m4, float m5,
                         int X0, int Y0, int passes, uint32_t skew, uint32_t row_stride, int lds_bytes) {
    WarpBox b;
    b.xlo = src_x;
    b.ylo = src_y;
    b.xhi = src_x + src_w - 1;
    b.yhi = src_y + src_h - 1;
    const float dcx = (float)(dw >> 1), dcy = (float)(dh >> 1);
    const float scx = (float)(src_x + (src_w >> 1)), scy = (float)(src_y + (src_h >> 1));
    const int X1 = box_min(X0 + WTW, dw) - 1, Y1 = box_min(Y0 + WTH * passes, dh) - 1;
    float bxmin = 3.0e38f, bxmax = -3.0e38f, bymin = 3.0e38f, bymax = -3.0e38f;
    bool corners_ok = true;
#pragma unroll
    for (int cy = 0; cy < 2; cy++)
#pragma unroll
        for (int cx = 0; cx < 2; cx++) {
            const float xr = (float)(cx ? X1 : X0) - dcx, yr = (float)(cy ? Y1 : Y0) - dcy;
            float sx = __builtin_fmaf(xr, m0, __builtin_fmaf(yr, m1, m2)) + scx;
            float sy = __builtin_fmaf(xr, m3, __builtin_fmaf(yr, m4, m5)) + scy;
            if constexpr (NEAREST) {
                sx += 0.5f;
                sy += 0.5f;
            }
            bxmin = __builtin_fminf(bxmin, sx); bxmax = __builtin_fmaxf(bxmax, sx);
            bymin = __builtin_fminf(bymin, sy); bymax = __builtin_fmaxf(bymax, sy);
            corners_ok = corners_ok && sx == sx && sy == sy;
        }
    // every pixel of the tile maps between the corner extremes: when those lie inside the window no pixel needs a test
    b.all_in = corners_ok && bxmin >= (float)b.xlo && bymin >= (float)b.ylo && bxmax < (float)(b.xhi + 1) && bymax < (float)(b.yhi + 1);
    // keep the float->int conversions in range for degenerate matrices
    bxmin = __builtin_fmaxf(bxmin, -1.0e6f); bxmax = __builtin_fminf(bxmax, 1.0e6f);
    bymin = __builtin_fmaxf(bymin, -1.0e6f); bymax = __builtin_fminf(bymax, 1.0e6f);
    b.bx0 = box_max((int)__builtin_floorf(bxmin), b.xlo);
    b.bx1 = box_min((int)__builtin_floorf(bxmax) + 1, b.xhi);
    b.by0 = box_max((int)__builtin_floorf(bymin), b.ylo);
    b.by1 = box_min((int)__builtin_floorf(bymax) + 1, b.yhi);
    b.bw = b.bx1 - b.bx0 + 1;
    b.bh = b.by1 - b.by0 + 1;
    b.empty = b.bw <= 0 || b.bh <= 0;
    // staged box: bw columns + the repeated last one, bh rows + the last one again where a tap can lie in it: it is the window's last
    // row, or (a tile above the window, whose pixels are clamped to it and replaced) its first one. The row behind it in the source is
    // not loaded in its place: warp_box_inside() answers for rows up to by1 alone.
    b.nr = b.bh + (int)(bymax >= (float)b.yhi || bymax < (float)b.ylo);
    // RAW: a row is ppr 16-byte pieces from the dword that holds pixel bx0 (byte phase ph inside it). Boxes of at most kWarpRawPieces pieces
    // per row (every tile of a map that minifies by less than a tenth or so) and those of one piece more are staged at a pitch known to
    // the compiler: the row below is an offset inside the read instruction.
    b.colb = (uint32_t)box_max(b.bx0, 0) * 3u + skew;
    const int ppr_box = ((int)(b.colb & 3u) + 3 * (box_max(b.bw, 0) + 1) + 15) >> 4;
    b.ppr = box_max(ppr_box, kWarpRawPieces);
    // Any phase: rows at a pitch that leaves the same remainder mod 4 as the row stride, so that a row's bytes keep their place
    // within a dword on the way into LDS; at least 16 bytes between two rows' data, so that no piece holds data of both.
    const int need = 3 * box_max(b.bw, 0) + 16;
    b.pitch_b = RAW ? b.ppr * 16 : box_max(kWarpRawPieces * 16, (need + 3) & ~3) + (int)(row_stride & 3u);
    b.ph = (int)((RAW ? b.colb : b.colb + (uint32_t)box_max(b.by0, 0) * row_stride) & 3u);
    b.total = RAW ? b.nr * b.ppr : (int)(((int64_t)b.ph + (int64_t)(b.bh - 1) * b.pitch_b + 3 * b.bw + 15) >> 4);
    // (RAW: the three dwords read for the last tap of the last row may reach 8 bytes behind the box)
    b.use_lds = !b.empty && (!RAW || b.total <= 16 * RMX_WAVE) && (uint64_t)b.nr * (uint32_t)b.pitch_b + (RAW ? 16 : 32) <= (uint64_t)lds_bytes;
    return b;
}

// Where piece idx of the box comes from, in bytes from the dword that holds the image's first byte. RAW: piece c of row r, rows one after
// the other. Any phase: LDS byte i belongs to row r of the box (r * pitch_b + ph is the row's first pixel) and holds the source
// byte at the same distance from that row's first pixel; a piece is the row's that its last byte lies in (what a piece holds in front
// of a row is never read). Pitch and stride agree mod 4 and the box's first dword is a source dword, so every piece is loaded from a
// dword. inv: 1 / ppr (RAW), 1 / pitch_b; (x + 0.5) / n is at least 0.5 / n away from an integer, so the truncations are exact.
template <bool RAW>
RMX_BOX int64_t warp_piece(const WarpBox &b, uint32_t row_stride, int idx, float inv) {
    if constexpr (RAW) {
        const int r = (int)(((float)idx + 0.5f) * inv);
        const int c = idx - box_mul24(r, b.ppr);
        return (int64_t)(uint32_t)((uint32_t)box_min(b.by0 + r, b.by1) * row_stride + (b.colb & ~3u) + 16u * (uint32_t)c);
    } else {
        const int r = box_min((int)(((float)(16 * idx + 15 - b.ph) + 0.5f) * inv), b.bh - 1);
        return (int64_t)b.by0 * row_stride + b.colb - b.ph + 16 * idx + (int64_t)r * ((int64_t)row_stride - b.pitch_b);
    }
}

// Every piece of the box lies inside the batch buffer, which ends `left` bytes behind the dword of the image's first byte (the last rows of
// the last image may not, nor, at any phase, the first rows of the first one, where a piece starts up to 15 bytes in front of its row).
template <bool RAW>
RMX_BOX bool warp_box_inside(const WarpBox &b, uint32_t row_stride, uint64_t left) {
    const uint64_t last = (uint64_t)b.by1 * row_stride + b.colb;
    if constexpr (RAW) return last + 16u * (uint32_t)b.ppr <= left;
    else return last + (uint32_t)b.pitch_b + 32u <= left && (b.bh == 1 || (uint32_t)b.by0 * row_stride + b.colb - (uint32_t)b.ph + row_stride >= 16u);
}

}  // namespace rmx
