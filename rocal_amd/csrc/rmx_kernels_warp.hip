// K4: inverse-map affine warp (WarpAffine / Rotate), bilinear or nearest, constant-0 outside
// the source ROI; u8 NHWC in, T/LAYOUT out.
//
// A wavefront owns a destination tile of 32 columns x (16 x passes) rows. The tile's corners are pushed
// through the affine map to get the source bounding box (every pixel of the tile maps inside it: each
// step of the coordinate law is monotone in x and in y, also after rounding), which is staged into the
// wavefront's LDS slice with all loads of the box in flight together; one extra
// column and row repeat the ROI's last column / row, so the right and lower neighbours of a tap are always
// at +3 bytes and +pitch. Each lane then produces 8 adjacent destination pixels of one row per pass, branch-free:
// taps of pixels that fall outside the ROI are read from wherever their (meaningless) address points inside
// the slice and the result is replaced by 0. When the box does not fit the slice (strong minification) the
// wavefront gathers from global memory instead.
//
// The box travels from global memory straight into LDS as packed bytes (global_load_lds_dwordx4, 16 bytes per lane: no vector
// register, no unpacking, no LDS store), three bytes per pixel, and a tap pair (two packed pixels, 6 bytes at any byte phase) is
// read as three aligned dwords and realigned with two v_alignbyte. Two forms:
//   RAW    every source row starts at the same byte phase (row strides multiples of 4): piece i of the box, rows one after the
//          other, is loaded by lane i & 63 of load instruction i >> 6;
//   any    rows at any byte phase (299 pixels are 897 bytes; images packed without padding): a load starts at a dword, so bytes
//          keep their place within a dword on the way into LDS. The LDS pitch therefore leaves the same remainder mod 4 as the row
//          stride: a tap's address stays linear in its coordinates, and the only cost in the loop is that the lower row's address
//          is masked by itself (two instructions per pixel). Against staging through registers with one dword per pixel (111 registers,
//          13 KB): 64 rotations of 299 x 299, bytes, with the wide stores below, 18.4 -> 15.1 us per batch. Rows at one phase keep RAW:
//          its loop has the masks' two instructions less, of 58.
// Interleaved bytes leave by whole rows of a tile, or of four tiles side by side (ROWS): stored by each lane as they
// came, 24 bytes in two pieces, every cache line was written by up to six instructions with part of it each, and that, not the bytes, made loads
// and stores wait for one another (nearest pixel, 128 images of 512 x 512, in a trace: 60 us, without stores 38, without loads 36). 128 images
// of 512 x 512, whole batches: nearest pixel 57.3 -> 48.6 us by tiles -> 43.4 by four tiles as streaming stores (these cost the stores of
// single lanes 8 us: part of a line at a time, they go to memory before their neighbours come); bilinear 63.4 -> 61.0.
// The nearest pixel's bytes are moved, not converted to float and back (BYTES): 43.4 -> 42.7, 86 turned images of 151 x 447 10.7 -> 10.2.
// Bound by how many wavefronts are there to compute while others wait for their box: 128 images of 512 x 512 take 58 - 61 us; with the
// lanes' own stores, 61 - 63 then, without the box's loads 47, without the stores 52, without both 42, with taps that meet no bank conflict
// the same; the bytes are 36 at the rate of a large copy. The LDS slice therefore holds the box and nothing besides: no pixel of margin (the corners bound it exactly), the
// repeated row only where it is read, rows of 10 pieces where they fit instead of 11 (a batch turned by up to 30 degrees and scaled by a
// tenth: 9.4 -> 7.7 KB a wavefront, 20 of them per CU instead of 16; a seventh fewer pieces to load): 63.2 - 64.0 -> 60.9 - 63.1 us on
// several inputs, in turn. Fewer instructions alone (taps widened inside v_fma_mix_f32: a fifth fewer) measured the same beside it.
#include "rmx_device.h"
#include "rmx_launch.h"
#include "rmx_warp_box.h"

#include <type_traits>

#ifndef RMX_WARP_NT
#define RMX_WARP_NT false
#endif

namespace rmx {

extern __shared__ uint32_t rmx_lds_warp[];
typedef __attribute__((address_space(3))) uint32_t lds_u32;  // explicit LDS pointers: 32-bit address arithmetic

typedef uint32_t u32x2_l __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_l __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_b __attribute__((ext_vector_type(4), aligned(1)));  // (global memory takes any address)
typedef __attribute__((address_space(3))) u32x2_l lds_u32x2;
typedef __attribute__((address_space(3))) u32x4_l lds_u32x4_l;

constexpr int WRP = kWarpRawPieces;
constexpr int WTEAM = kWarpTeam;                 // tiles side by side whose wavefronts store their rows together
constexpr int WROW = WTW * 3;                    // bytes of a tile's row, u8
constexpr int WTILE_BYTES = 2 * WTH * WROW;      // of a tile of two passes
static_assert(WTILE_BYTES == kWarpTileBytes, "the host gives a slice room for a tile");

RMX_DEV uint32_t load_px_global(const uint8_t *p) {
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16);
}

// floor(x) as an integer in one instruction (saturating; 0 for NaN)
RMX_DEV int floor_i32(float x) {
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

template <typename T, int LAYOUT, bool NEAREST, bool RAW, int ROWS>
RMX_DEV void warp_body(const RmxKArgs &a) {
    const int lane = threadIdx.x & (RMX_WAVE - 1);
    const int wib = threadIdx.x / RMX_WAVE;
    const uint32_t nwaves = (uint32_t)a.n * (uint32_t)a.strips;
    uint32_t wave = xcd_swizzle(blockIdx.x, a.nblocks) * (uint32_t)a.wpb + wib;
    wave = __builtin_amdgcn_readfirstlane(wave);
    if (wave >= nwaves) return;
    int s, tile;
    wave_to_sample(a, wave, s, tile);
    const int tiles_x = a.aux0;
    const int passes = a.aux1 >> 8;
    const int ty = tile / tiles_x, tx = tile - ty * tiles_x;
    // the whole table row in one round trip
    const RmxSample P = load_sample<RMX_C_WINDOW | RMX_C_M6>(a, s);
    asm volatile("" : : "s"(P.src_x), "s"(P.dst_w), "s"(P.flags), "s"(P.m[0]), "s"(P.m[5]));
    const int dw = P.dst_w, dh = P.dst_h;
    const int X0 = tx * WTW, Y0 = ty * (WTH * passes);
    if (X0 >= dw || Y0 >= dh) return;

    const float m0 = P.m[0], m1 = P.m[1], m2 = P.m[2], m3 = P.m[3], m4 = P.m[4], m5 = P.m[5];
    const float dcx = (float)(dw >> 1), dcy = (float)(dh >> 1);
    const float scx = (float)(P.src_x + (P.src_w >> 1)), scy = (float)(P.src_y + (P.src_h >> 1));

    uint32_t row_stride;
    const uint8_t *simg = sample_base(a, s, row_stride);
    const uint8_t *buf_end = a.src + a.src_bytes;
    T *dimg = reinterpret_cast<T *>(a.dst) + (size_t)s * 3 * a.dst_h * a.dst_w;
    uint32_t *lds = rmx_lds_warp + (size_t)wib * (a.lds_bytes >> 2);

    // source bounding box of the tile (wave-uniform)
    const uint32_t skew = (uint32_t)((uintptr_t)simg & 3u);
    const WarpBox box = warp_box<NEAREST, RAW>(P.src_x, P.src_y, P.src_w, P.src_h, dw, dh, m0, m1, m2, m3, m4, m5, X0, Y0, passes, skew, row_stride, a.lds_bytes);
    const int xlo = box.xlo, ylo = box.ylo, xhi = box.xhi, yhi = box.yhi;
    const int bx0 = box.bx0, by0 = box.by0, bw = box.bw, bh = box.bh, nr = box.nr;
    const int ppr = box.ppr, pitch_b = box.pitch_b, ph = box.ph, total = box.total;
    const bool empty = box.empty, all_in = box.all_in;

    // ROWS: a tile's groups wait in registers until both its passes are done, change places through the slice, and rows leave as 16-byte
    // pieces that lie one behind the other in memory (a tile of fewer than 32 columns keeps the lanes' own stores); RMX_WARP_TEAMS: the
    // rows of the workgroup's four tiles side by side, 128 pixels, whole cache lines, as streaming stores.
    const bool together = ROWS != RMX_WARP_LANES && dw - X0 >= WTW;
    // (the same in all wavefronts of the workgroup: none of them leaves early then, and all reach the barrier)
    const bool team = ROWS == RMX_WARP_TEAMS && dw - (X0 - wib * WTW) >= WTEAM * WTW;
    [[maybe_unused]] PackedGroup<T> upper, lower;
    const int lr = lane >> 2, g = lane & 3;
    int x0 = X0 + g * PX;
    // The short last group of a row moves left until it is whole (its pixels belong to this tile): it recomputes pixels of the group
    // before it and stores the same values to the same places. Only a tile narrower than 8 pixels keeps a short group.
    if (x0 < dw) x0 = max(min(x0, dw - PX), X0);
    const int cnt = min(PX, dw - x0);
    // Whole groups leave as wide stores at the alignment of an element (the same instructions as for aligned rows).
    auto store_run = [&](int pass, int y, const PackedGroup<T> &packed) {
        if (ROWS != RMX_WARP_LANES && together) {
            if (pass == 0) upper = packed;
            else lower = packed;
        } else {
            store_packed<T, LAYOUT, RMX_WARP_NT, true>(dimg, a.dst_h, a.dst_w, y, x0, packed);
        }
    };
    auto store = [&](int pass, int y, const float (&v)[3][PX]) {
        if ((ROWS != RMX_WARP_LANES && together) || cnt == PX) {
            PackedGroup<T> packed;
            pack_group_dir<T, LAYOUT, false>(v, packed);
            store_run(pass, y, packed);
        } else {
            store_group<T, LAYOUT>(dimg, a.dst_h, a.dst_w, y, x0, cnt, v, false);
        }
    };
    // Nearest bytes to interleaved bytes are moved, not converted: a pixel in the low three bytes of each dword
    constexpr bool BYTES = NEAREST && sizeof(T) == 1 && LAYOUT == RMX_NHWC;
    auto store_bytes = [&](int pass, int y, const uint32_t (&px)[PX]) {
        PackedGroup<T> packed;
        if constexpr (BYTES) {
#pragma unroll
            for (int k = 0; k < PX / 4; k++) {
                packed.w[3 * k] = __builtin_amdgcn_perm(px[4 * k + 1], px[4 * k], 0x04020100u);
                packed.w[3 * k + 1] = __builtin_amdgcn_perm(px[4 * k + 2], px[4 * k + 1], 0x05040201u);
                packed.w[3 * k + 2] = __builtin_amdgcn_perm(px[4 * k + 3], px[4 * k + 2], 0x06050402u);
            }
        }
        if (cnt == PX) store_run(pass, y, packed);
        else store_packed_part<T, LAYOUT>(dimg, a.dst_h, a.dst_w, y, x0, 0, cnt, packed);
    };
    const float xr0 = (float)x0 - dcx;
    lds_u8 *ldsb = (lds_u8 *)(lds_ptr_t)rmx_lds_warp + (uint32_t)to_sgpr((int)((uint32_t)wib * (uint32_t)a.lds_bytes));
    auto leave = [&]() {
        if constexpr (ROWS != RMX_WARP_LANES) {
            if (!together) return;
            wave_sync();  // (the box has been read for the last time)
            lds_u8 *mine = ldsb + lr * WROW + g * (PX * 3);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                *(lds_u32x2 *)(mine + 8 * k) = (u32x2_l){upper.w[2 * k], upper.w[2 * k + 1]};
                *(lds_u32x2 *)(mine + WTH * WROW + 8 * k) = (u32x2_l){lower.w[2 * k], lower.w[2 * k + 1]};
            }
            // (A team's lanes store the same piece of every second row, 48 of them, so that their places are made once: 62.4 -> 61.1 us; a
            // tile's ten rows at a time, 60 lanes, gain nothing, 62.6 -> 63.3)
            uint8_t *out = reinterpret_cast<uint8_t *>(dimg) + ((size_t)Y0 * a.dst_w + X0) * 3;
            constexpr int PCS = WROW / 16;  // pieces of a tile's row
            const uint32_t pitch = (uint32_t)a.dst_w * 3u;
            if (ROWS == RMX_WARP_TEAMS && team) {
                __syncthreads();
                constexpr int PCT = WTEAM * PCS, AT_ONCE = 2, PART = 2 * WTH / WTEAM;  // (a wavefront stores a quarter of the rows)
                const int rr = lane >= PCT ? 1 : 0, c = lane - rr * PCT, t = c / PCS, row = wib * PART + rr;
                const lds_u8 *from = (lds_u8 *)(lds_ptr_t)rmx_lds_warp + t * a.lds_bytes + row * WROW + (c - t * PCS) * 16;
                const uint32_t to = (uint32_t)row * pitch + (uint32_t)c * 16u;
                out -= wib * WROW;
                if (lane < AT_ONCE * PCT) {
#pragma unroll
                    for (int k = 0; k < PART / AT_ONCE; k++) {
                        const u32x4_l v = *(const lds_u32x4_l *)(from + k * AT_ONCE * WROW);
                        if (Y0 + row + k * AT_ONCE < dh) __builtin_nontemporal_store(u32x4_b(v), reinterpret_cast<u32x4_b *>(out + (size_t)(k * AT_ONCE) * pitch + to));
                    }
                }
                return;
            }
            wave_sync();
#pragma unroll
            for (int k = 0; k < WTILE_BYTES / 16 / RMX_WAVE; k++) {
                const int idx = k * RMX_WAVE + lane, row = idx / PCS;
                const u32x4_l v = *(const lds_u32x4_l *)(ldsb + 16 * idx);
                if (Y0 + row < dh) *reinterpret_cast<u32x4_b *>(out + ((uint32_t)row * pitch + (uint32_t)(idx - row * PCS) * 16u)) = v;
            }
        }
    };

    if (empty) {
        // every pixel of the tile maps outside the ROI: the fill value
        float z[3][PX];
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int k = 0; k < PX; k++) z[c][k] = 0.0f;
        for (int pass = 0; pass < passes; pass++) {
            const int y = Y0 + pass * WTH + lr;
            if (y < dh && cnt > 0) store(pass, y, z);
        }
        return leave();
    }
    if (!box.use_lds) {
        // a box too large for the slice: per-pixel gathers from global memory
        for (int pass = 0; pass < passes; pass++) {
            const int y = Y0 + pass * WTH + lr;
            if (y >= dh || cnt <= 0) continue;
            const float yr = (float)y - dcy;
            float v[3][PX];
#pragma unroll
            for (int k = 0; k < PX; k++) {
                const float xr = (float)(x0 + k) - dcx;
                const float sx = __builtin_fmaf(xr, m0, __builtin_fmaf(yr, m1, m2)) + scx;
                const float sy = __builtin_fmaf(xr, m3, __builtin_fmaf(yr, m4, m5)) + scy;
                float fx, fy;
                if constexpr (NEAREST) {
                    fx = floorf(sx + 0.5f);
                    fy = floorf(sy + 0.5f);
                } else {
                    fx = floorf(sx);
                    fy = floorf(sy);
                }
                const bool oob = empty || fx < (float)xlo || fy < (float)ylo || fx > (float)xhi || fy > (float)yhi || !(fx == fx) || !(fy == fy);
                float o0 = 0.0f, o1 = 0.0f, o2 = 0.0f;
                if (!oob) {
                    const int ix0 = (int)fx, iy0 = (int)fy;
                    const int ix1 = min(ix0 + 1, xhi), iy1 = min(iy0 + 1, yhi);
                    const uint32_t tl = load_px_global(simg + (size_t)iy0 * row_stride + (size_t)ix0 * 3);
                    if constexpr (NEAREST) {
                        o0 = ubyte0(tl); o1 = ubyte1(tl); o2 = ubyte2(tl);
                    } else {
                        const uint32_t tr = load_px_global(simg + (size_t)iy0 * row_stride + (size_t)ix1 * 3);
                        const uint32_t bl = load_px_global(simg + (size_t)iy1 * row_stride + (size_t)ix0 * 3);
                        const uint32_t br = load_px_global(simg + (size_t)iy1 * row_stride + (size_t)ix1 * 3);
                        const float wx = sx - fx, wy = sy - fy;
                        const float omx = 1.0f - wx, omy = 1.0f - wy;
                        const float w00 = omy * omx, w01 = omy * wx, w10 = wy * omx;
                        o0 = __builtin_fmaf(ubyte0(tl), w00, __builtin_fmaf(ubyte0(tr), w01, __builtin_fmaf(ubyte0(bl), w10, ubyte0(br) * wy * wx)));
                        o1 = __builtin_fmaf(ubyte1(tl), w00, __builtin_fmaf(ubyte1(tr), w01, __builtin_fmaf(ubyte1(bl), w10, ubyte1(br) * wy * wx)));
                        o2 = __builtin_fmaf(ubyte2(tl), w00, __builtin_fmaf(ubyte2(tr), w01, __builtin_fmaf(ubyte2(bl), w10, ubyte2(br) * wy * wx)));
                    }
                }
                v[0][k] = o0; v[1][k] = o1; v[2][k] = o2;
            }
            store(pass, y, v);
        }
        return leave();
    }

    const uint8_t *base4 = simg - skew;
    // ---- the box straight into LDS: piece idx lands at byte 16 idx of the slice
    const uint64_t left = (uint64_t)(buf_end - base4);
    const float inv = 1.0f / (float)(RAW ? ppr : pitch_b);
    if (warp_box_inside<RAW>(box, row_stride, left)) {
        for (int j0 = 0; j0 < total; j0 += RMX_WAVE) {
            const int idx = j0 + lane;
            const uint32_t off = (uint32_t)warp_piece<RAW>(box, row_stride, idx, inv);
            if (idx < total) __builtin_amdgcn_global_load_lds((glb_ptr_t)(base4 + off), (lds_ptr_t)(ldsb + 16 * j0), 16, 0, RMX_LDS_LOAD_AUX);
        }
    } else {
        // the box touches the ends of the batch buffer: the pieces that leave it are stored by their lanes
        for (int j0 = 0; j0 < total; j0 += RMX_WAVE) {
            const int idx = j0 + lane;
            const int64_t off = warp_piece<RAW>(box, row_stride, idx, inv);
            if (idx < total && off >= 0 && off + 16 <= (int64_t)left) __builtin_amdgcn_global_load_lds((glb_ptr_t)(base4 + off), (lds_ptr_t)(ldsb + 16 * j0), 16, 0, RMX_LDS_LOAD_AUX);
            else if (idx < total) {
                const uint4 v = load_piece_bounded<int64_t>(base4, off, (int64_t)left);
                *(lds_u32x4 *)(ldsb + 16 * idx) = (u32x4_a4){v.x, v.y, v.z, v.w};
            }
        }
    }
    // the compiler does not order LDS reads behind loads into LDS: await them explicitly
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    wave_sync();
    // the column behind the box repeats its last column where that is the ROI's last column, and (rows at any phase) the row below
    // the box its last row where a tap can lie in that (only then are they read; RAW has loaded that row)
    if (box.bx1 == xhi) {
        for (int r = lane; r < (RAW ? nr : bh); r += RMX_WAVE) {
            lds_u8 *px = ldsb + r * pitch_b + ph + 3 * (bw - 1);
            px[3] = px[0];
            px[4] = px[1];
            px[5] = px[2];
        }
        wave_sync();
    }
    if (!RAW && !NEAREST && nr > bh) {
        lds_u8 *last = ldsb + (bh - 1) * pitch_b + ph;
        for (int b = lane; b < 3 * (bw + 1); b += RMX_WAVE) last[pitch_b + b] = last[b];
        wave_sync();
    }

    // ---- gather and blend, branch-free
    // LDS byte address of the first byte of source pixel (0, 0), three bytes per pixel: the slice's base minus the box origin (may
    // lie below the slice)
    const int lbase0 = (int)(uint32_t)(uintptr_t)(lds_u32 *)lds + ph - (by0 * pitch_b + 3 * bx0);
    // pixels whose floor lies inside the ROI: xlo <= s < xhi + 1 (and not NaN), tested on the clamped coordinate
    // (upper bounds: the float just below xhi + 1, a positive number, so one step down in its bit pattern)
    const float cx_lo = (float)xlo, cx_hi = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, (float)(xhi + 1)) - 1u);
    const float cy_lo = (float)ylo, cy_hi = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, (float)(yhi + 1)) - 1u);
    int lbase_v = lbase0;  // the same in a vector register: the multiply-add takes only one scalar operand
    asm volatile("" : "+v"(lbase_v));
    auto gather = [&](auto chk, auto fix) {
        constexpr bool CHECK = decltype(chk)::value;
        constexpr int PITCH = decltype(fix)::value;  // 16-byte pieces, 0: not known before
        constexpr bool FIXED = PITCH != 0;
        for (int pass = 0; pass < passes; pass++) {
            const int y = Y0 + pass * WTH + lr;
            if (y >= dh || cnt <= 0) continue;
            const float yr = (float)y - dcy;
            const float cxy = __builtin_fmaf(yr, m1, m2), cyy = __builtin_fmaf(yr, m4, m5);
            float v[3][PX];
            [[maybe_unused]] uint32_t bytes[PX];
            // A pixel in two steps: fetch (coordinates, tap address, the LDS reads of its taps) and blend. The reads of pixel
            // k + 1 are issued before pixel k is blended, so that a wavefront waits for LDS once per row instead of once per
            // pixel (left to the compiler's order, every pixel's reads were followed at once by the wait for them): 65.6 -> 64.1 us
            // on 128 images of 512 x 512.
            typedef uint32_t u32x2_r __attribute__((ext_vector_type(2)));
            struct Taps {
                u32x2_r top, bot;   // the first two dwords of the upper and of the lower row
                uint32_t t2, b2;    // the third dword of each row
                float sx, sy;
                uint32_t tph, bph;  // addresses of the tap pairs: their two low bits are the phase inside the first dword
                bool inb;
            };
            // RAW bilinear taps at the fixed pitch: the reads are written out (one address register for both rows, the row
            // below at an offset inside the instruction) and awaited by a count, so that the reads of the next pixel stay in
            // flight while this one is blended; the compiler's own bookkeeping would wait for every outstanding read.
            constexpr bool BY_HAND = RAW && FIXED && !NEAREST;
            auto fetch = [&](int k) {
                Taps t;
                const float xr = xr0 + (float)k;  // == (float)(x0 + k) - dcx: small integers, exact
                float sx = __builtin_fmaf(xr, m0, cxy) + scx;
                float sy = __builtin_fmaf(xr, m3, cyy) + scy;
                if constexpr (NEAREST) {
                    sx += 0.5f;
                    sy += 0.5f;
                }
                t.inb = true;
                if constexpr (CHECK) {
                    // Clamped into the ROI (a NaN becomes the lower bound): equal to the coordinate exactly when the pixel is
                    // inside, and an address inside the staged box also when it is not (the box holds the ROI's border
                    // wherever the tile reaches beyond it).
                    const float qx = __builtin_fminf(__builtin_fmaxf(sx, cx_lo), cx_hi);
                    const float qy = __builtin_fminf(__builtin_fmaxf(sy, cy_lo), cy_hi);
                    t.inb = qx == sx && qy == sy;
                    sx = qx;
                    sy = qy;
                }
                t.sx = sx;
                t.sy = sy;
                const int ix0 = floor_i32(sx), iy0 = floor_i32(sy);
                // byte address: a 24-bit multiply-add of the row onto the slice base, another of the column
                uint32_t rowb, adr;
                if constexpr (FIXED) asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(rowb) : "v"(iy0), "s"(PITCH * 16), "v"(lbase_v));
                else asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(rowb) : "v"(iy0), "s"(pitch_b), "v"(lbase_v));
                asm("v_mad_i32_i24 %0, %1, 3, %2" : "=v"(adr) : "v"(ix0), "v"(rowb));
                const uint32_t adr1 = adr + (uint32_t)pitch_b;
                t.tph = adr;
                t.bph = RAW ? adr : adr1;
                const lds_u32 *t0p = (const lds_u32 *)(adr & ~3u);
                const lds_u32 *t1p = FIXED ? t0p + PITCH * 4 : (const lds_u32 *)(adr1 & ~3u);
                if constexpr (BY_HAND) {
                    static_assert(PITCH * 4 + 2 < 256, "the row below must be reachable by the 8-bit dword offsets of ds_read2_b32");
                    // (the values are taken apart only behind the wait: nothing may copy a register before its data has arrived)
                    asm volatile("ds_read2_b32 %0, %4 offset1:1\n\tds_read_b32 %1, %4 offset:8\n\t"
                                 "ds_read2_b32 %2, %4 offset0:%5 offset1:%6\n\tds_read_b32 %3, %4 offset:%7"
                                 : "=&v"(t.top), "=&v"(t.t2), "=&v"(t.bot), "=&v"(t.b2)
                                 : "v"((uint32_t)(uintptr_t)t0p), "n"(PITCH * 4), "n"(PITCH * 4 + 1), "n"(PITCH * 16 + 8));
                    return t;
                }
                t.top = (u32x2_r){t0p[0], t0p[1]};
                t.bot = (u32x2_r){0u, 0u};
                t.t2 = t.b2 = 0u;
                if constexpr (!NEAREST) {
                    t.t2 = t0p[2];
                    t.bot = (u32x2_r){t1p[0], t1p[1]};
                    t.b2 = t1p[2];
                }
                return t;
            };
            // BY_HAND: the taps of a pixel have arrived when at most `behind` younger read instructions are outstanding
            // (LDS operations of a wavefront complete in issue order); everything that reads the taps comes behind this.
            auto arrived = [&](Taps &t, auto behind) {
                if constexpr (BY_HAND)
                    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(t.top), "+v"(t.t2), "+v"(t.bot), "+v"(t.b2) : "n"(decltype(behind)::value));
            };
            auto blend = [&](int k, const Taps &tp) {
                struct { uint32_t tl, tr, t2, bl, br, b2; float sx, sy; uint32_t tph, bph; bool inb; } t = {tp.top.x, tp.top.y, tp.t2, tp.bot.x, tp.bot.y, tp.b2, tp.sx, tp.sy, tp.tph, tp.bph, tp.inb};
                float o0, o1, o2;
                if constexpr (NEAREST) {
                    const uint32_t tl = __builtin_amdgcn_alignbyte(t.tr, t.tl, t.tph);
                    if constexpr (BYTES) {
                        bytes[k] = t.inb ? tl : 0u;
                        return;
                    }
                    o0 = ubyte0(tl); o1 = ubyte1(tl); o2 = ubyte2(tl);
                } else {
                    // s - floor(s): exact for the non-negative coordinates of pixels inside the ROI
                    const float wx = __builtin_amdgcn_fractf(t.sx), wy = __builtin_amdgcn_fractf(t.sy);
                    const float omx = 1.0f - wx, omy = 1.0f - wy;
                    const float w00 = omy * omx, w01 = omy * wx, w10 = wy * omx;
                    // six bytes from byte tph on: TL in bytes 0..2 of the first realigned dword, TR from its byte 3 on
                    const uint32_t tlo = __builtin_amdgcn_alignbyte(t.tr, t.tl, t.tph), thi = __builtin_amdgcn_alignbyte(t.t2, t.tr, t.tph);
                    const uint32_t blo = __builtin_amdgcn_alignbyte(t.br, t.bl, t.bph), bhi = __builtin_amdgcn_alignbyte(t.b2, t.br, t.bph);
                    o0 = __builtin_fmaf(ubyte0(tlo), w00, __builtin_fmaf(ubyte3(tlo), w01, __builtin_fmaf(ubyte0(blo), w10, ubyte3(blo) * wy * wx)));
                    o1 = __builtin_fmaf(ubyte1(tlo), w00, __builtin_fmaf(ubyte0(thi), w01, __builtin_fmaf(ubyte1(blo), w10, ubyte0(bhi) * wy * wx)));
                    o2 = __builtin_fmaf(ubyte2(tlo), w00, __builtin_fmaf(ubyte1(thi), w01, __builtin_fmaf(ubyte2(blo), w10, ubyte1(bhi) * wy * wx)));
                }
                v[0][k] = t.inb ? o0 : 0.0f;
                v[1][k] = t.inb ? o1 : 0.0f;
                v[2][k] = t.inb ? o2 : 0.0f;
            };
            // (one pixel ahead; two ahead, with eight reads outstanding, measured the same: 64.1 us on 128 images of 512 x 512)
            Taps cur = fetch(0);
#pragma unroll
            for (int k = 0; k < PX; k++) {
                Taps nxt = cur;
                if (k + 1 < PX) {
                    nxt = fetch(k + 1);
                    arrived(cur, std::integral_constant<int, 4>{});  // (the four read instructions of the next pixel may be outstanding)
                    __builtin_amdgcn_sched_barrier(0);               // (the next pixel's reads stay in front of this pixel's arithmetic)
                } else {
                    arrived(cur, std::integral_constant<int, 0>{});
                }
                blend(k, cur);
                cur = nxt;
            }
            if constexpr (BYTES) store_bytes(pass, y, bytes);
            else store(pass, y, v);
        }
    };
    auto run = [&](auto fix) {
        if (all_in) gather(std::false_type{}, fix);
        else gather(std::true_type{}, fix);
    };
    if (RAW && ppr == WRP) run(std::integral_constant<int, RAW ? WRP : 0>{});
    else if (RAW && ppr == WRP + 1) run(std::integral_constant<int, RAW ? WRP + 1 : 0>{});
    else run(std::integral_constant<int, 0>{});
    leave();
}

template <typename T, int LAYOUT, bool NEAREST, bool RAW>
__global__ void __launch_bounds__(256) rmx_warp_kernel(RmxKArgs a) {
    warp_body<T, LAYOUT, NEAREST, RAW, RMX_WARP_LANES>(a);
}

template <bool NEAREST, bool RAW, int ROWS>
__global__ void __launch_bounds__(256) rmx_warp_rows_kernel(RmxKArgs a) {
    warp_body<uint8_t, RMX_NHWC, NEAREST, RAW, ROWS>(a);
}

template <bool NEAREST, bool RAW>
static KernelFn pick(int dtype, int layout) {
    if (layout == RMX_NCHW) {
        switch (dtype) {
            case RMX_FP32: return (KernelFn)rmx_warp_kernel<float, RMX_NCHW, NEAREST, RAW>;
            case RMX_FP16: return (KernelFn)rmx_warp_kernel<__half, RMX_NCHW, NEAREST, RAW>;
            default: return (KernelFn)rmx_warp_kernel<uint8_t, RMX_NCHW, NEAREST, RAW>;
        }
    }
    switch (dtype) {
        case RMX_FP32: return (KernelFn)rmx_warp_kernel<float, RMX_NHWC, NEAREST, RAW>;
        case RMX_FP16: return (KernelFn)rmx_warp_kernel<__half, RMX_NHWC, NEAREST, RAW>;
        default: return (KernelFn)rmx_warp_kernel<uint8_t, RMX_NHWC, NEAREST, RAW>;
    }
}

// raw: the form for source rows that all start at the same byte phase
KernelFn select_warp_kernel(int interp, int dtype, int layout, bool raw, const char **name) {
    *name = raw ? "rmx_warp_kernel(raw)" : "rmx_warp_kernel";
    if (raw) return interp == RMX_INTERP_NEAREST ? pick<true, true>(dtype, layout) : pick<false, true>(dtype, layout);
    return interp == RMX_INTERP_NEAREST ? pick<true, false>(dtype, layout) : pick<false, false>(dtype, layout);
}

template <bool NEAREST, bool RAW>
static KernelFn pick_rows(int rows) {
    return rows == RMX_WARP_TEAMS ? (KernelFn)rmx_warp_rows_kernel<NEAREST, RAW, RMX_WARP_TEAMS> : (KernelFn)rmx_warp_rows_kernel<NEAREST, RAW, RMX_WARP_TILES>;
}

KernelFn select_warp_rows_kernel(int interp, bool raw, int rows) {
    if (raw) return interp == RMX_INTERP_NEAREST ? pick_rows<true, true>(rows) : pick_rows<false, true>(rows);
    return interp == RMX_INTERP_NEAREST ? pick_rows<true, false>(rows) : pick_rows<false, false>(rows);
}

}  // namespace rmx
