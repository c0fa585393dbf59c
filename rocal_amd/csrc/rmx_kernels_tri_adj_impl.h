// K2t streaming path, second form: triangular (antialiased) resize in both directions, from source rows at any byte phase. As in
// rmx_resize_tri_dma_kernel (rmx_kernels_tri_dma_impl.h) a wavefront owns 128 output columns and a strip of output rows, its source
// rows travel straight into a ring in LDS, and the arithmetic is the ring kernel's (rmx_kernels_tri.hip), operation for operation. What differs:
//   * a lane owns two neighbouring columns, and a row leaves as three stores of a pair (interleaved: one run of six elements) instead of six
//     of an element. The kernel's memory operations, not its arithmetic, are what it waits for: of 46 us for 256 RandomResizedCrop windows
//     to 224 x 224 fp16 with single elements (a trace), 37 are left without the stores, 40 without the loads, 37 without either, 43
//     without the arithmetic. (Rows gathered in LDS and stored as 16-byte pieces: 45.1 against 43.5 with single elements and 42.2 us
//     with pairs: what an element costs on its way through LDS is more than its store. A ring of six rows, loads two steps ahead: 44.5
//     against 43.6. Six wavefronts per SIMD: no change.)
//   * a sample that grows vertically (two taps per output row) makes its output rows from the last two filtered rows, 12 multiply-adds per
//     output row, whatever its ratio; eight accumulator sets took 48 per source row, 119 registers and no more than eight rows in flight.
//   * a sample that shrinks has two accumulator sets for every ratio and not for whole and half ones only, half the vertical multiply-adds
//     of four sets: see `run`.
//   * ANY: rows at any byte phase. A row is loaded from the dword that holds its first byte, so every LDS row has a phase of its own, which
//     a tap's address carries (two instructions per column and row).
// Whole batches, before -> after: 256 RandomResizedCrop windows of 640 x 640 to 224 x 224 fp16 45.1 -> 42.5 us (before: eight accumulator
// sets). Rows at any phase, or windows that grow by more than 3.8, which the ring kernel took: 182 windows to 160 x 160 fp16 81.2 -> 32.2,
// 101 to 189 x 189 58.0 -> 24.0, 219 packed ones to 224 x 224 interleaved fp32 94.1 -> 57.9; and frames of 985 pixels to 464 (shrinking
// alone, staged through registers before) 24.4 -> 19.9.
#pragma once
#include "rmx_kernels_tri_dma_impl.h"

// (called from several places, the kernel's lambdas would become functions, and everything they share would live in scratch memory)
#define TS_INLINE __attribute__((always_inline))

namespace rmx {

typedef __attribute__((address_space(3))) f32x2 lds_f32x2;

constexpr int TS_GROW = 4;  // output rows made behind one another without going back, from two rows of a sample that grows

// Six accumulators to h * c (c 0: to 0) when idx == M, the branch inside the statement as in zero_if. h is a sum of products that are not
// negative: with c 0 this is +0.
template <int M>
RMX_DEV void start_over_if(int idx, float (&acc)[3][2], const float (&h)[3][2], float c) {
    asm("s_cmp_lg_u32 %6, %7\n\ts_cbranch_scc1 .Lkeep%=\n\tv_mul_f32 %0, %8, %9\n\tv_mul_f32 %1, %8, %10\n\tv_mul_f32 %2, %8, %11\n\tv_mul_f32 %3, %8, %12\n\tv_mul_f32 %4, %8, %13\n\tv_mul_f32 %5, %8, %14\n.Lkeep%=:"
        : "+&v"(acc[0][0]), "+&v"(acc[0][1]), "+&v"(acc[1][0]), "+&v"(acc[1][1]), "+&v"(acc[2][0]), "+&v"(acc[2][1])
        : "s"(idx), "n"(M), "s"(c), "v"(h[0][0]), "v"(h[0][1]), "v"(h[1][0]), "v"(h[1][1]), "v"(h[2][0]), "v"(h[2][1])
        : "scc");
}

template <int DWORDS>
struct PairDwords {
    uint32_t w[2][DWORDS];
    uint32_t at[2];  // the first tap's byte
    f32x2 cv;        // the row's vertical coefficients
};

// Two neighbouring pixels of an output row, byte `at` of the plane or image: planar, one store per plane; interleaved, one run of six
// elements. At the alignment of an element, which global memory takes.
template <typename T, int LAYOUT>
RMX_DEV void store_pair(uint8_t *d, size_t plane_bytes, uint32_t at, const float (&v)[3][2]) {
    typedef uint32_t w3 __attribute__((ext_vector_type(3), aligned(1)));
    typedef uint32_t w2 __attribute__((ext_vector_type(2), aligned(1)));
    typedef uint32_t w1 __attribute__((aligned(1)));
    typedef uint16_t h1 __attribute__((aligned(1)));
    if constexpr (LAYOUT == RMX_NCHW) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            uint8_t *p = d + c * plane_bytes + at;
            if constexpr (sizeof(T) == 4) *reinterpret_cast<w2 *>(p) = (w2{elem_bits<T>(v[c][0]), elem_bits<T>(v[c][1])});
            else if constexpr (sizeof(T) == 2) *reinterpret_cast<w1 *>(p) = elem_bits<T>(v[c][0]) | elem_bits<T>(v[c][1]) << 16;
            else *reinterpret_cast<h1 *>(p) = (h1)__builtin_amdgcn_cvt_pk_u8_f32(v[c][1], 1, __builtin_amdgcn_cvt_pk_u8_f32(v[c][0], 0, 0));
        }
    } else {
        uint8_t *p = d + at;
        if constexpr (sizeof(T) == 4) {
            *reinterpret_cast<w3 *>(p) = (w3{elem_bits<T>(v[0][0]), elem_bits<T>(v[1][0]), elem_bits<T>(v[2][0])});
            *reinterpret_cast<w3 *>(p + 12) = (w3{elem_bits<T>(v[0][1]), elem_bits<T>(v[1][1]), elem_bits<T>(v[2][1])});
        } else if constexpr (sizeof(T) == 2) {
            *reinterpret_cast<w3 *>(p) = (w3{elem_bits<T>(v[0][0]) | elem_bits<T>(v[1][0]) << 16, elem_bits<T>(v[2][0]) | elem_bits<T>(v[0][1]) << 16,
                                             elem_bits<T>(v[1][1]) | elem_bits<T>(v[2][1]) << 16});
        } else {
            uint32_t w = __builtin_amdgcn_cvt_pk_u8_f32(v[0][0], 0, 0);
            w = __builtin_amdgcn_cvt_pk_u8_f32(v[1][0], 1, w);
            w = __builtin_amdgcn_cvt_pk_u8_f32(v[2][0], 2, w);
            *reinterpret_cast<w1 *>(p) = __builtin_amdgcn_cvt_pk_u8_f32(v[0][1], 3, w);
            *reinterpret_cast<h1 *>(p + 4) = (h1)__builtin_amdgcn_cvt_pk_u8_f32(v[2][1], 1, __builtin_amdgcn_cvt_pk_u8_f32(v[1][1], 0, 0));
        }
    }
}

template <typename T, int LAYOUT, bool NORM, bool QUANT, bool ANY>
__global__ void __launch_bounds__(256, 5) rmx_resize_tri_adj_kernel(RmxKArgs a) {
    constexpr int TPX = 2;               // columns per lane, side by side
    constexpr int TTW = RMX_WAVE * TPX;  // output columns per wave tile
    const int lane = threadIdx.x & (RMX_WAVE - 1);
    const int wib = threadIdx.x / RMX_WAVE;
    const uint32_t nwaves = (uint32_t)a.n * (uint32_t)a.strips;
    uint32_t wave = xcd_swizzle(blockIdx.x, a.nblocks) * (uint32_t)a.wpb + wib;
    wave = __builtin_amdgcn_readfirstlane(wave);
    if (wave >= nwaves) return;
    int s, part;
    wave_to_sample(a, wave, s, part);
    const int tiles_x = a.aux1;
    const int strip = part / tiles_x, tx = part - strip * tiles_x;
    // the whole table row in one round trip
    const RmxSample P = load_sample<RMX_C_WINDOW | RMX_C_RATIO | RMX_C_ORDER>(a, s);
    asm volatile("" : : "s"(P.src_x), "s"(P.dst_w), "s"(P.pc_x), "s"(P.flags), "s"(P.rx), "s"(P.scale[0]), "s"(P.bias[2]), "s"(P.fsx));
    s = P.plan[2];  // (the host may have put the rows in another order: the row names its sample)

    const int dw = P.dst_w, dh = P.dst_h;
    const int srows = a.aux0;
    const int r0 = strip * srows;
    int xt = tx * TTW;
    if (r0 >= dh || xt >= dw) return;
    // (a last tile of one column takes the column before it too: the host keeps rows of one pixel from this kernel)
    if (dw - xt == 1) xt--;
    const int r1 = min(r0 + srows, dh);
    const int tw = min(TTW, dw - xt);
    const bool hf = (P.flags & RMX_S_HFLIP) != 0;
    const int xlo = P.src_x, ylo = P.src_y;
    const int xhi = xlo + P.src_w - 1, yhi = ylo + P.src_h - 1;
    const int pcx = P.pc_x, pcy = P.pc_y;
    const TriAxis ax = tri_axis(P.rx, P.fsx), ay = tri_axis(P.ry, P.fsy);
    const int kx = to_sgpr(ax.ksize), ky = to_sgpr(ay.ksize);

    // (a sample is smaller than 4 GiB: the host checks it, so offsets inside a sample are 32-bit)
    uint32_t row_stride_v;
    const uint8_t *simg_v = sample_base(a, s, row_stride_v);
    const uint32_t row_stride = (uint32_t)to_sgpr((int)row_stride_v);
    const uint8_t *simg = reinterpret_cast<const uint8_t *>(((uint64_t)(uint32_t)to_sgpr((int)((uintptr_t)simg_v >> 32)) << 32) |
                                                            (uint32_t)to_sgpr((int)(uint32_t)(uintptr_t)simg_v));
    const uint32_t skew = (uint32_t)((uintptr_t)simg & 3u);
    const uint8_t *base4 = simg - skew;  // dword-aligned base below the sample
    const uint64_t left = (uint64_t)((a.src + a.src_bytes) - base4);
    const uint32_t lim = left > 0xffffffffull ? 0xffffffffu : (uint32_t)left;  // bytes of the batch buffer from base4 on
    T *dimg = reinterpret_cast<T *>(a.dst) + (size_t)s * 3 * a.dst_h * a.dst_w;
    // (the wavefront's index inside its workgroup comes from a lane id: wave-uniform, but only a scalar register says so)
    const uint32_t slice_off = (uint32_t)to_sgpr((int)((uint32_t)wib * (uint32_t)a.lds_bytes));
    lds_u8 *bufb = (lds_u8 *)(lds_ptr_t)rmx_lds_tdma + slice_off;

    float sc[3], bi[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        sc[c] = P.scale[c];
        bi[c] = P.bias[c];
        if constexpr (NORM) asm("" : "+v"(bi[c]), "+v"(sc[c]));  // (a multiply-add takes one scalar operand: the other would be moved for every output row)
    }

    // ---- the tile's source columns and the layout of an LDS row (all wave-uniform)
    int l_first, l_last;
    {
        int lf, ll;
        float w0;
        tri_loc(ax, pcx + xt, (float)xlo, lf, w0);
        tri_loc(ax, pcx + xt + tw - 1, (float)xlo, ll, w0);
        l_first = to_sgpr(lf);
        l_last = to_sgpr(ll);
    }
    const int cs = max(min(l_first, xhi), xlo);
    const int ce = max(min(l_last + kx - 1, xhi), xlo);
    const int nrep_l = max(cs - l_first, 0), nrep_r = max(l_last + kx - 1 - ce, 0);
    const uint32_t colb = (uint32_t)cs * 3u + skew;  // byte offset (from base4) of pixel cs, within a row
    // Byte phase of pixel cs inside its dword: the same in every row, or (ANY) each row's own, up to 3
    const int ph = ANY ? 0 : (int)(colb & 3u);
    const int ph_max = ANY ? 3 : ph;
    const int nd = (ph_max + 3 * (ce - cs + 1) + 15) >> 4;  // data pieces of a row
    const int lm = ((3 * nrep_l + 15) >> 4) << 4;           // margin bytes in front of the data
    // data, right replicas, and the bytes the widest tap read (8 taps from the last column's first tap) may touch
    const int body = max(ph_max + 3 * (l_last + 8 - cs) + 8, 16 * nd);
    const int pitch = lm + (((body + 15) >> 4) << 4);
    const int ppr = pitch >> 4;  // pieces per row
    const int tab_off = a.lds_bytes - 2 * (TS_TAB + TS_EDGE) * 4;  // the tables of vertical coefficients
    // (the host sizes the slice for four rows of the widest tile; a tile that does not fit is left alone)
    if (2 * TS_RPS * pitch > tab_off || ppr > TS_NCH * RMX_WAVE || 3 * (nrep_l + nrep_r) > RMX_WAVE) return;

    // ---- output rows of the strip, one per lane (a strip has at most 64 rows): first tap row and its weight offset;
    // wave-uniform code fetches a row's entry with v_readlane
    int oloc_v;
    float ow0_v;
    tri_loc(ay, pcy + min(r0 + lane, r1 - 1), (float)ylo, oloc_v, ow0_v);
    auto row_loc = [&](int r) { return __builtin_amdgcn_readlane(oloc_v, r - r0); };
    auto row_w0 = [&](int r) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ow0_v), r - r0)); };
    const int y_first = max(min(row_loc(r0), yhi), ylo);
    const int y_last = max(min(row_loc(r1 - 1) + ky - 1, yhi), ylo);

    // ---- load plan of the tile: piece c of an LDS row is loaded by lane c & 63 of load instruction c >> 6. Margin pieces
    // and pieces behind the data repeat a neighbouring data piece (their content is never read before a replica is written
    // over it), so no load leaves the row's own bytes.
    auto piece_off = [&](int c) TS_INLINE { return 16u * (uint32_t)max(min(c - (lm >> 4), nd - 1), 0); };
    const uint32_t lane_off = piece_off(lane);
    // Rows from y_lanes on are stored by the lanes, with bounds-checked loads: those whose last piece would leave the batch
    // buffer, which only the last row of the last sample of the buffer can be (a row's pieces end less than 16 bytes behind
    // the row); should even the row before it not fit, every row goes that way.
    const uint32_t tail = (ANY ? colb : colb & ~3u) + 16u * (uint32_t)nd;
    int y_lanes = y_last + 1;
    if ((uint64_t)((uint32_t)y_last * row_stride) + tail > (uint64_t)lim)
        y_lanes = (y_last > y_first && (uint64_t)((uint32_t)(y_last - 1) * row_stride) + tail <= (uint64_t)lim) ? y_last : y_first;

    // Starts the transfer of the next two source rows (rows behind the last repeat it) into the two slots of one half of the
    // ring; y_next / rb_next (the byte of the row's pixel cs) walk down the rows. Returns whether a row was stored by the lanes.
    int y_next = y_first;
    uint32_t rb_next = (uint32_t)y_first * row_stride + colb;
    auto issue = [&](lds_u8 *half_base) TS_INLINE {
        if (y_next + 1 < y_lanes) {
            // both rows are there and come by loads into LDS
            const uint32_t rb2 = rb_next + row_stride;
            auto two_rows = [&](uint32_t off, int k) TS_INLINE {
                asm volatile("" : "+v"(off));  // (or it would be kept as a 64-bit number, and added to the row's address by the vector unit)
                __builtin_amdgcn_global_load_lds((glb_ptr_t)(base4 + (rb_next & ~3u) + off), (lds_ptr_t)(half_base + k * RMX_WAVE * 16), 16, 0, RMX_LDS_LOAD_AUX);
                __builtin_amdgcn_global_load_lds((glb_ptr_t)(base4 + (rb2 & ~3u) + off), (lds_ptr_t)(half_base + pitch + k * RMX_WAVE * 16), 16, 0, RMX_LDS_LOAD_AUX);
            };
            if (lane < ppr) two_rows(lane_off, 0);
            if (ppr > RMX_WAVE) {
                int c = RMX_WAVE + lane;
                asm volatile("" : "+v"(c));
                if (c < ppr) two_rows(piece_off(c), 1);
            }
            y_next += TS_RPS;
            rb_next = rb2 + row_stride;
            return false;
        }
        bool by_lanes = false;
#pragma unroll 1
        for (int q = 0; q < TS_RPS; q++) {
            const uint32_t roff = rb_next & ~3u;
            lds_u8 *slot = half_base + q * pitch;
            if (y_next < y_lanes) {
                const uint8_t *rowp = base4 + roff;
                for (int k = 0; k < TS_NCH; k++) {
                    const int c = k * RMX_WAVE + lane;
                    if (c < ppr) __builtin_amdgcn_global_load_lds((glb_ptr_t)(rowp + piece_off(c)), (lds_ptr_t)(slot + k * RMX_WAVE * 16), 16, 0, RMX_LDS_LOAD_AUX);
                }
            } else {
                by_lanes = true;
                for (int c = lane; c < ppr; c += RMX_WAVE) {
                    const uint4 v = load_piece_bounded<uint32_t>(base4, roff + 16u * (uint32_t)max(min(c - (lm >> 4), nd - 1), 0), lim);
                    *(lds_u32x4 *)(slot + 16 * c) = (u32x4_a4){v.x, v.y, v.z, v.w};
                }
            }
            if (y_next < y_last) {
                y_next++;
                rb_next += row_stride;
            }
        }
        return by_lanes;
    };

    // The first two rows are asked for here, ahead of the coefficient set-up below (some hundred instructions that need no
    // memory): they travel while it runs.
    const bool first_by_lanes = issue(bufb);

    // ---- per-lane columns: taps, coefficients (registers), column sums, destination column (mirrored if asked)
    // (a lane whose columns lie beyond the row takes the last two again and stores the same values to the same places: every
    // wavefront issues every store instruction, which the count in the wait below relies on)
    uint32_t xoff = 0, tap[TPX];
    float colsum[TPX] = {}, creg[TPX][8] = {};
    int locx[TPX];
    float w0x[TPX];
#pragma unroll
    for (int i = 0; i < TPX; i++) {
        // (in the order of the destination; at an odd width the last of them moves left by one column)
        const int colc = xt + min(2 * lane, tw - 2) + (hf ? 1 - i : i);
        if (i == 0) xoff = (uint32_t)(hf ? (dw - 1 - colc) : colc) * (uint32_t)(LAYOUT == RMX_NCHW ? sizeof(T) : 3 * sizeof(T));
        tri_loc(ax, pcx + colc, (float)xlo, locx[i], w0x[i]);
    }
    // (the host admits at most eight taps; a wavefront-wide branch per tap, so that only those there are cost anything)
#pragma unroll
    for (int k = 0; k < 8; k++) {
        if (k < kx) {
#pragma unroll
            for (int i = 0; i < TPX; i++) {
                creg[i][k] = tri_coeff(w0x[i], ax.radius, k, ax.fscale);
                colsum[i] += creg[i][k];
            }
        }
    }
    const bool lead = !(creg[0][0] == 0.0f) || !(creg[1][0] == 0.0f);  // some column's first tap has a coefficient other than 0
#pragma unroll
    for (int i = 0; i < TPX; i++) colsum[i] = (colsum[i] == 0.0f) ? 1.0f : colsum[i];
    // When the first tap of every column of the tile has coefficient 0 (ratios 1 and 3, the odd whole numbers: the first tap then
    // lies a whole radius from the centre), the horizontal pass starts one pixel on with one tap less: fma(p, 0, 0) is the 0
    // the accumulation starts from anyway. Wave-uniform.
    const int skip = (kx > 1 && __builtin_amdgcn_ballot_w64(lead) == 0) ? 1 : 0;
    const int kx_run = kx - skip;
    if (skip) {
#pragma unroll
        for (int i = 0; i < TPX; i++)
#pragma unroll
            for (int k = 0; k < 8; k++) creg[i][k] = k < 7 ? creg[i][k + 1] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < TPX; i++) {
        // the first tap's byte inside an LDS row (a tap left of the window reads a replica in or behind the margin), from the row's
        // phase on where each row has its own
        tap[i] = (uint32_t)(lm + ph + 3 * (locx[i] + skip - cs));
    }
    // Of output row r0 + lane: the sum of its vertical coefficients, taps ascending, and the source rows of its first and last
    // coefficient other than 0. Whoever needs a row's entry fetches it from the lane that holds it.
    float rsum_v = 0.0f;
    int ylast_v = max(min(oloc_v + ky - 1, yhi), ylo);
    // Output row r + 2 takes the set of row r when that has been stored. Its source rows lie behind row r's, but for one that both may have:
    // rounding can leave its first tap and row r's last one a coefficient other than 0 in one source row. Row r's is then in the
    // table, and the other one, kept here by row r's lane, starts the set that row r leaves (see `run`).
    float late_v = 0.0f;
    if (ky == 2) {
        rsum_v = rsum_v + tri_coeff(ow0_v, ay.radius, 0, ay.fscale) + tri_coeff(ow0_v, ay.radius, 1, ay.fscale);
    } else {
        int jb = 0;
        for (int j = 0; j < ky; j++) {
            const float c = tri_coeff(ow0_v, ay.radius, j, ay.fscale);
            rsum_v += c;
            if (c > 0.0f) jb = j;
        }
        ylast_v = max(min(oloc_v + jb, yhi), ylo);
        const int below = __builtin_amdgcn_ds_bpermute(4 * (lane + 2), oloc_v);  // (of the output row two below)
        const float below_w0 = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (lane + 2), __builtin_bit_cast(int, ow0_v)));
        if (lane + 2 < r1 - r0 && below <= ylast_v) late_v = tri_coeff(below_w0, ay.radius, 0, ay.fscale);
    }
    rsum_v = (rsum_v == 0.0f) ? 1.0f : rsum_v;
    auto last_tap_row = [&](int r) { return __builtin_amdgcn_readlane(ylast_v, r - r0); };

    // ---- clamp-to-edge columns: byte e of the replicas (left ones first) is copied by lane e from the first / last pixel
    const int nrep_b = 3 * (nrep_l + nrep_r);
    auto replicate = [&](lds_u8 *half_base, int nr, uint32_t rb) TS_INLINE {
        if (nrep_b > 0) {
            if (lane < nrep_b) {
                int e = lane;
                asm volatile("" : "+v"(e));  // (made again for every step of the tiles at the window's edge, the places take no registers in the others)
                const bool is_l = e < 3 * nrep_l;
                const int er = is_l ? e : e - 3 * nrep_l;
                const int j = er / 3, c = er - 3 * j;
                const uint32_t src = (uint32_t)(lm + ph + (is_l ? 0 : 3 * (ce - cs)) + c);
                const uint32_t dst = (uint32_t)(lm + ph + (is_l ? -3 * (j + 1) : 3 * (ce - cs + 1 + j)) + c);
                for (int q = 0; q < nr; q++) {
                    lds_u8 *slot = half_base + q * pitch + (ANY ? (rb + q * row_stride) & 3u : 0u);
                    slot[dst] = slot[src];
                }
            }
            wave_sync();
        }
    };

    // ---- output rows in flight. rq is the oldest one, qlast its last tap row (wave-uniform state).
    int rq = r0;
    int qlast = last_tap_row(r0);
    int emitted = 0;  // output rows stored since the loads that were started last

    // ---- vertical coefficients by source row, a table of 64 rows x the two sets in the tail of the LDS slice: entry (l, k) is
    // the coefficient with which source row ytab + l enters the output row of set k (0: none; fma(h, 0, acc) == acc for
    // the finite h a filtered row is, so both sets take every row and no branch is needed). Lane r writes the taps of output row
    // r0 + r, in their order: where a first tap's source row is the last one of the output row two above (late_v), that one stays; the
    // filter loop reads a source row's entry with one broadcast read. Rebuilt every 64 source rows. The first and the last row of the window serve several taps of a row
    // each (clamped tap indices) and take their own path below.
    // (Written by source rows instead, lane l going through all the strip's output rows for row l's coefficients, the table
    // and the coefficients of the columns, made twice, were a third of the instructions in front of the row loop: 256 RandomResizedCrop windows to
    // 224 x 224 fp16 47.8 -> 45.3 us.)
    lds_f32 *cftab = (lds_f32 *)(bufb + tab_off);
    const lds_f32x2 *cv_next = (const lds_f32x2 *)cftab;  // the table entry of the next source row
    int ytab = y_first;
    auto build_table = [&]() TS_INLINE {
        *(lds_f32x2 *)(cftab + 2 * lane) = f32x2{};
        wave_sync();
        int loc = oloc_v, row = lane;
        float w0 = ow0_v;
        asm volatile("" : "+v"(loc), "+v"(w0), "+v"(row));  // (or the taps' coefficients and places would be kept in registers from one table to the next)
        const int l0 = loc - ytab;
        lds_f32 *mine = cftab + 2 * l0 + (row & 1);
        const bool on = row < r1 - r0;
#pragma unroll 1
        for (int j = 0; j < ky; j++) {
            const float c = tri_coeff(w0, ay.radius, j, ay.fscale);
            if (on && c > 0.0f && (uint32_t)(l0 + j) < (uint32_t)TS_TAB) mine[2 * j] = c;
        }
        wave_sync();
    };

    // An output row whose last tap row has been added: normalise, epilogue, store. out_row, the row's byte in its plane (planar) or image,
    // walks down the output rows and is added to the lanes' columns: the planes' addresses stay as they are. (The host sees to it that
    // a sample's output is smaller than 4 GiB.)
    const size_t plane = (size_t)a.dst_h * a.dst_w;
    const uint32_t out_step = (uint32_t)a.dst_w * (uint32_t)(LAYOUT == RMX_NCHW ? sizeof(T) : 3 * sizeof(T));
    uint32_t out_row = (uint32_t)r0 * out_step;
    int rsum_idx = 0;
    // 1 / (row sum x column sum) is kept from one output row to the next: rows of an integer ratio all have the same sum
    int rsum_bits_prev = 0;  // (no row sum is +0: a zero sum is replaced by 1)
    float inv_c[TPX];
#pragma unroll
    for (int i = 0; i < TPX; i++) inv_c[i] = 0.0f;
    auto row_sums = [&]() TS_INLINE {
        const int rsum_bits = __builtin_amdgcn_readlane(__builtin_bit_cast(int, rsum_v), rsum_idx);
        if (rsum_bits != rsum_bits_prev) {
            rsum_bits_prev = rsum_bits;
            const float rsum = __builtin_bit_cast(float, rsum_bits);
#pragma unroll
            for (int i = 0; i < TPX; i++) inv_c[i] = recip(rsum * colsum[i]);
        }
    };
    auto emit = [&](const float (&sum)[3][TPX]) TS_INLINE {
        float v[3][TPX];
#pragma unroll
        for (int i = 0; i < TPX; i++)
#pragma unroll
            for (int ch = 0; ch < 3; ch++) {
                float t = sum[ch][i] * inv_c[i];
                if constexpr (QUANT) t = round_u8(t);
                if constexpr (NORM) t = __builtin_fmaf(t, sc[ch], bi[ch]);
                v[ch][i] = t;
            }
        store_pair<T, LAYOUT>(reinterpret_cast<uint8_t *>(dimg), plane * sizeof(T), xoff + out_row, v);
    };
    auto next_output_row = [&]() TS_INLINE {
        rq++;
        rsum_idx++;
        out_row += out_step;
        emitted++;
        qlast = rq < r1 ? last_tap_row(rq) : 0x7fffffff;  // (behind the last row: no source row completes anything)
    };

    // A source row's part of a lane: the dwords that hold the taps of its two columns (rb: the byte of the row's pixel cs, whose phase the
    // row's bytes keep in LDS) and, where a table is used, the row's vertical coefficients.
    auto fetch_row = [&](auto nt, auto table, const lds_u8 *srow, uint32_t rb) TS_INLINE {
        constexpr int NT = decltype(nt)::value;
        constexpr bool TABLE = decltype(table)::value;
        PairDwords<(3 * NT + 3) / 4 + 1> f;
        if constexpr (TABLE) f.cv = *cv_next++;
#pragma unroll
        for (int i = 0; i < TPX; i++) {
            f.at[i] = ANY ? tap[i] + (rb & 3u) : tap[i];
            const lds_u32 *p0 = (const lds_u32 *)(srow + (f.at[i] & ~3u));
#pragma unroll
            for (int j = 0; j < (3 * NT + 3) / 4 + 1; j++) f.w[i][j] = p0[j];
        }
        return f;
    };

    // The horizontal pass of a source row. NT = taps of the unrolled pass (2, 3, 4, 5, 6 or 8 >= the taps that are run): taps beyond
    // those carry coefficient 0 (fma(p, 0, a) == a for the finite p an unpacked byte always is), so no bound test is needed
    // inside. A column's 3 NT bytes start at byte at & 3 of the first dword read: NE + 1 dwords are read and realigned into NE.
    auto filter_row = [&](auto nt, const auto &f, float (&h)[3][TPX]) TS_INLINE {
        constexpr int NT = decltype(nt)::value;
        constexpr int NE = (3 * NT + 3) / 4;
#pragma unroll
        for (int i = 0; i < TPX; i++) {
            uint32_t e[NE];
#pragma unroll
            for (int j = 0; j < NE; j++) e[j] = __builtin_amdgcn_alignbyte(f.w[i][j + 1], f.w[i][j], f.at[i]);
            float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
            tri_taps<NT, NE>(e, creg[i], a0, a1, a2);
            h[0][i] = a0;
            h[1][i] = a1;
            h[2][i] = a2;
        }
    };

    // Two rows per step. The loads of a step were started a step earlier; the compiler does not order LDS reads behind
    // loads into LDS, so their arrival is awaited explicitly, between two wavefront fences. Memory operations of a wavefront
    // complete in issue order, loads and stores on one counter: the wait names a number of store instructions that have been issued
    // since those loads (see store_pair), so it waits for none of these. The next step's loads are
    // started right behind the wait (the slots they fill were read for the last time in the step before).
    constexpr int NS = LAYOUT == RMX_NCHW ? 3 : 1;  // store instructions per output row, at least
    lds_u8 *half_cur = bufb, *half_nxt = bufb + TS_RPS * pitch;
    uint32_t rb_cur = (uint32_t)y_first * row_stride + colb;
    bool by_lanes = first_by_lanes;
    auto step_in = [&](int y, int nr) TS_INLINE {
        if (by_lanes || emitted == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the lanes' own loads, or no store behind the loads)
        else if (emitted == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NS) : "memory");
        else if (emitted < 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NS) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * NS) : "memory");
        wave_sync();
        emitted = 0;
        by_lanes = (y + TS_RPS <= y_last) ? issue(half_nxt) : false;
        replicate(half_cur, nr, rb_cur);
    };
    auto step_out = [&]() TS_INLINE {
        wave_sync();  // the slots are reused two steps on
        lds_u8 *t = half_cur;
        half_cur = half_nxt;
        half_nxt = t;
        rb_cur += TS_RPS * row_stride;
    };

    // ---- samples that shrink vertically. A source row has a coefficient other than 0 in two output rows, so two accumulator sets do:
    // output row r accumulates in set (r - r0) & 1 until its last such row has been added. Rounding can give that row to output row r + 2
    // as well (late_v): the set then starts over from it instead of from 0. The rows two apart lie two radii apart, so no other row can be in both,
    // and that one is neither the window's first nor its last (tests/test_tri_rows_cpu.py; the host keeps windows whose coordinates
    // are no longer exact to half a row from this kernel). How many output rows are so is the ratio's doing: one strip in 400 of random
    // ones, but half of them at 11 / 7. (Such strips done in two goes, the even pairs of their output rows and then the odd ones: 96 images
    // of 550 x 550 to 350 x 350 fp16 69.2 us instead of 43.2, 192 of 476 x 476 to
    // 140 x 140 94.8 instead of 55.5; with four accumulator sets 48.9 and 56.7.)
    auto run = [&](auto nt) TS_INLINE {
        float acc[2][3][TPX];
        // The row in work is source row yy: filter it and add it to the output rows in flight.
        auto process_row = [&](const auto &f, int yy) TS_INLINE {
            // A row inside the window is one tap of every output row that reads it: one pass, coefficients from the table. The
            // first / last row of the window is also read by every tap index that leaves the window: one pass per such tap, in
            // tap order, coefficients computed here by lane p for pass p (rare: twice per image column of strips at most).
            f32x2 cv = f.cv;
            int more = 0;
            const lds_f32x2 *cvp = nullptr;
            if ((uint32_t)(yy - ylo - 1) >= (uint32_t)(yhi - ylo - 1)) {  // yy == ylo or yy == yhi (rows lie inside the window)
                float ec[2];
                int npass = 0;
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    const int r = (rsum_idx & 1) == m ? rq : rq + 1;  // the row in flight that lives in set m
                    ec[m] = 0.0f;
                    if (r < r1) {
                        const int loc = row_loc(r);
                        const int jlo = max((yy == ylo) ? 0 : yy - loc, 0);
                        const int jhi = min((yy == yhi) ? ky - 1 : yy - loc, ky - 1);
                        npass = max(npass, jhi - jlo + 1);
                        const int j = jlo + lane;
                        const float c = tri_coeff(row_w0(r), ay.radius, j, ay.fscale);
                        if (j <= jhi) ec[m] = c;
                    }
                }
                lds_f32 *etab = cftab + 2 * TS_TAB;
                if (lane < TS_EDGE) *(lds_f32x2 *)(etab + 2 * lane) = f32x2{ec[0], ec[1]};
                wave_sync();
                cvp = (const lds_f32x2 *)etab;
                cv = *cvp;
                more = npass - 1;
            }
            float h[3][TPX];
            filter_row(nt, f, h);
            // every pass adds the filtered row to both sets with that pass's coefficients (0: none)
            auto add_row = [&]() TS_INLINE {
#pragma unroll
                for (int m = 0; m < 2; m++)
#pragma unroll
                    for (int ch = 0; ch < 3; ch++)
#pragma unroll
                        for (int i = 0; i < TPX; i++) fmac_inplace(acc[m][ch][i], h[ch][i], cv[m]);
            };
            add_row();
            for (; more > 0; more--) {
                cv = *++cvp;
                add_row();
            }
            // rows whose last tap was this source row
            while (qlast <= yy) {
                row_sums();
                if (rsum_idx & 1) emit(acc[1]);
                else emit(acc[0]);
                const float late = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, late_v), rsum_idx));
                start_over_if<0>(rsum_idx & 1, acc[0], h, late);
                start_over_if<1>(rsum_idx & 1, acc[1], h, late);
                next_output_row();
            }
        };
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int i = 0; i < TPX; i++) acc[m][c][i] = 0.0f;
        build_table();  // (under the round trip of the first loads)
        for (int y = y_first; y <= y_last; y += TS_RPS) {
            const int nr = min(TS_RPS, y_last - y + 1);
            if (y + nr - ytab > RMX_WAVE) {
                ytab = y;
                cv_next = (const lds_f32x2 *)cftab;
                build_table();
            }
            step_in(y, nr);
            auto row = fetch_row(nt, std::true_type{}, half_cur, rb_cur);
            // Both rows' reads are started before the first row is filtered (the second row's slot holds a row also where
            // the window ends with the first one) where the registers allow it.
            constexpr bool AHEAD = decltype(nt)::value <= 4;
            auto second = row;
            if constexpr (AHEAD) second = fetch_row(nt, std::true_type{}, half_cur + pitch, rb_cur + row_stride);
            process_row(row, y);
            if (nr > 1) {
                if constexpr (!AHEAD) second = fetch_row(nt, std::true_type{}, half_cur + pitch, rb_cur + row_stride);
                process_row(second, y + 1);
            }
            step_out();
        }
    };

    // ---- samples that grow vertically: two taps per output row, one or more output rows per source row. The last two filtered rows are
    // kept and every output row is made from them when its second tap row has been filtered: c0 * row + c1 * next row, what an
    // accumulator that starts at 0 would hold (the products are not negative), whatever the ratio. Clamped taps read the window's first or last
    // row twice: the row before is then that row itself.
    auto run_grow = [&](auto nt) TS_INLINE {
        float c0_v = tri_coeff(ow0_v, ay.radius, 0, ay.fscale), c1_v = tri_coeff(ow0_v, ay.radius, 1, ay.fscale);
        float h[TS_RPS][3][TPX] = {};
        auto one_row = [&](float (&prev)[3][TPX], const float (&cur)[3][TPX], int yy) TS_INLINE {
            if (max(row_loc(rq), ylo) != yy - 1) {
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int i = 0; i < TPX; i++) prev[c][i] = cur[c][i];
            }
            // (in vector registers: a multiply-add takes a scalar operand at half its rate)
            float c0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c0_v), rsum_idx));
            float c1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c1_v), rsum_idx));
            asm("" : "+v"(c0), "+v"(c1));
            row_sums();
            float sum[3][TPX];
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int i = 0; i < TPX; i++) sum[c][i] = __builtin_fmaf(cur[c][i], c1, prev[c][i] * c0);
            emit(sum);
            next_output_row();
        };
        auto rows_of = [&](float (&prev)[3][TPX], const float (&cur)[3][TPX], int yy) TS_INLINE {
            while (qlast <= yy) {
#pragma unroll
                for (int k = 0; k < TS_GROW; k++) {
                    if (qlast > yy) break;
                    one_row(prev, cur, yy);
                }
            }
        };
        for (int y = y_first; y <= y_last; y += TS_RPS) {
            const int nr = min(TS_RPS, y_last - y + 1);
            step_in(y, nr);
            constexpr bool AHEAD = decltype(nt)::value <= 4;
            const auto first = fetch_row(nt, std::false_type{}, half_cur, rb_cur);
            auto second = first;
            if constexpr (AHEAD) second = fetch_row(nt, std::false_type{}, half_cur + pitch, rb_cur + row_stride);
            filter_row(nt, first, h[0]);
            rows_of(h[1], h[0], y);
            if (nr > 1) {
                if constexpr (!AHEAD) second = fetch_row(nt, std::false_type{}, half_cur + pitch, rb_cur + row_stride);
                filter_row(nt, second, h[1]);
                rows_of(h[0], h[1], y + 1);
            }
            step_out();
        }
    };

    auto by_taps = [&](auto go) TS_INLINE {
        if (kx_run <= 2) go(std::integral_constant<int, 2>{});
        else if (kx_run == 3) go(std::integral_constant<int, 3>{});
        else if (kx_run == 4) go(std::integral_constant<int, 4>{});
        else if (kx_run == 5) go(std::integral_constant<int, 5>{});
        else if (kx_run == 6) go(std::integral_constant<int, 6>{});
        else go(std::integral_constant<int, 8>{});
    };
    if (ky == 2) by_taps(run_grow);
    else by_taps(run);
}

#define RMX_TADJ_UNIT(LAYOUT, ANY, NAME)                                                             \
    template <typename T>                                                                            \
    static KernelFn pick_tadj(bool norm, bool quant) {                                               \
        if (norm && quant) return (KernelFn)rmx_resize_tri_adj_kernel<T, LAYOUT, true, true, ANY>;   \
        if (norm) return (KernelFn)rmx_resize_tri_adj_kernel<T, LAYOUT, true, false, ANY>;           \
        return (KernelFn)rmx_resize_tri_adj_kernel<T, LAYOUT, false, false, ANY>;                    \
    }                                                                                                \
    KernelFn NAME(int dtype, bool norm, bool quant) {                                                \
        switch (dtype) {                                                                             \
            case RMX_FP32: return pick_tadj<float>(norm, quant);                                     \
            case RMX_FP16: return pick_tadj<__half>(norm, quant);                                    \
            default: return pick_tadj<uint8_t>(norm, quant);                                         \
        }                                                                                            \
    }

}  // namespace rmx
