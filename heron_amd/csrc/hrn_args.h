// What hrn_api.cpp hands to the kernels of mfma_gemm_template.hip, and the whole-number arithmetic the kernels do with it.  Both
// include this file; without HIP it is plain C++.
#ifndef HRN_ARGS_H
#define HRN_ARGS_H
#include <stdint.h>

#ifdef __HIP__
#define HRN_BOTH __host__ __device__ __forceinline__
#else
#define HRN_BOTH inline
#endif

// n / d for 0 <= n < 2^31 and 1 <= d < 2^31 by a multiplication: with L = ceil(log2 d) and m = ceil(2^(31+L) / d), which fits into
// 32 bits, n*m / 2^(31+L) exceeds n / d by less than 1 / d (Granlund and Montgomery, Division by Invariant Integers).
// Kernels divide by what is fixed for a launch.  A division proper is some 30 instructions, and a kernel starts with four
// (GEMM) to eight of them, each waiting for the one before, in front of its first load: 194 instructions to it instead of 127 (u8 64x128
// tiles), 435 instead of 283 (fp16 im2col 128x128) when the multipliers came.
struct HrnDiv {
    uint32_t m, shift;
    HrnDiv() = default;
    explicit HrnDiv(uint32_t d) : shift(d > 1 ? 32 - __builtin_clz(d - 1) : 0) { m = (uint32_t)(((1ull << (31 + shift)) + d - 1) / d); }
    HRN_BOTH uint32_t operator()(uint32_t n) const {
#ifdef __HIP_DEVICE_COMPILE__
        return __umulhi(n << 1, m) >> shift;
#else
        return (uint32_t)((uint64_t)(n << 1) * m >> 32) >> shift;
#endif
    }
};

// What every launch hands over, and all of it for a product
struct HrnKArgs {
    const void* A;
    const void* B;
    void* C;
    int32_t M, N, K;            // K in elements
    int32_t lda, ldb, ldc;      // elements
    int64_t sA, sB, sC;         // batch strides, elements
    int32_t tiles_m, tiles_n, group_m, batch;
    int32_t split, kt_per_slice;         // split-K: number of K slices and k-tiles per slice
    const void* bsum;                    // uint8 path: per batch entry N column sums of B (sum_k B[n,k], int32), or null
    // split-K: the result and what tells the last slice of a tile to add them all up; arrivals null: a kernel behind this one does
    void* out;
    int64_t out_stride;                  // batch stride of the result, elements
    uint64_t* arrivals;                  // one word per output tile, of any content
    uint64_t ticket;                     // of this launch, its low 16 bits zero
    int32_t out_ld;
    // divisors of the launch: K slices, output tiles of a batch entry, of a raster group, rows of a group and of the last one
    HrnDiv by_split, by_tiles, by_group, by_gm, by_gm_last;
};

// What a conv's launch adds; a product's does without
struct HrnConvArgs : HrnKArgs {
    int32_t H, W, CI, HO, WO, KH, KW, cstride, cpad, cdil;
    int32_t cstride_w, cpad_w, cdil_w;   // the width-direction values (cstride/cpad/cdil are the height ones)
    int32_t out_plane;                   // CHW kernels: row m, column n of the result goes to C[m / out_plane][n][m % out_plane]
    int32_t expand_shift;                // EXPAND kernels: the H x W input is not in memory: pixel (y, x) of the in_h x in_w
    int32_t in_h, in_w, top, left;       // one that is stands at (top + (y << shift), left + (x << shift)), zeros elsewhere
    // divisors of the launch: elements of a filter row and of a tap, output pixels of an image and of a row, 16-byte pieces of a pixel, pixels
    // of a plane (out_plane)
    HrnDiv by_kwci, by_ci, by_hw, by_wo, by_cpp, by_plane;
    // im2col (hrn_walk_args): the bytes of a pixel; the width of all taps; whether taps are carried along K (CI, or 0); what a byte offset
    // changes by, beyond the step itself, where K goes on to the next tap and filter row; the step from one row of A that a lane
    // loads to the next in output pixels, input pixels and bytes, and what changes where it leaves a row or an image of the result.  Modulo
    // 2^32, as the kernel adds them: pads, strides and dilations may be of any size, and only what lies inside an image is used.
    uint32_t px, kw_end, tap_bytes, taprow_bytes;
    int32_t carry_ci;
    uint32_t d_ox, d_oy, x_step, y_step, off_step, x_row, row_bytes, y_img, img_bytes;
};

// The (output tile, K slice) pair of a split-K workgroup, slices fastest: workgroup i runs on XCD i % 8, and each XCD has an eighth of
// the pairs in their order, the first XCDs one more where 8 does not divide them.
HRN_BOTH int hrn_pair_of(int block, int pairs) {
    const int xcd = block & 7, more = pairs & 7;
    return xcd * (pairs >> 3) + (xcd < more ? xcd : more) + (block >> 3);
}

// What the walks below need of a launch whose conv fields are set; `rows`: output pixels from one load of a lane to its next.
// expanded: the input in memory is the in_h x in_w one.
inline void hrn_walk_args(HrnConvArgs* k, int es, int rows, bool expanded) {
    const uint32_t px = (uint32_t)k->CI * es, H = k->H, W = k->W, sh = k->cstride, sw = k->cstride_w, hw = (uint32_t)k->HO * k->WO;
    const uint32_t images = rows / hw, rest = rows % hw;
    k->px = px;
    k->tap_bytes = ((uint32_t)k->cdil_w - 1u) * px;
    k->kw_end = (uint32_t)k->KW * k->cdil_w;
    k->carry_ci = (uint64_t)k->KW * k->cdil_w >> 32 ? 0 : k->CI;      // (then no other tap of a row is where the row ends)
    k->taprow_bytes = ((uint32_t)k->cdil * W - k->kw_end) * px;
    k->d_oy = rest / k->WO; k->d_ox = rest % k->WO;
    k->x_step = k->d_ox * sw; k->y_step = k->d_oy * sh;
    k->x_row = k->WO * sw; k->y_img = k->HO * sh;
    k->row_bytes = (sh * W - k->x_row) * px;
    if (expanded) {
        k->img_bytes = (uint32_t)k->in_h * k->in_w * px;
        k->off_step = images * k->img_bytes;
    } else {
        k->img_bytes = (H - k->y_img) * W * px;
        k->off_step = ((images * H + k->y_step) * W + k->x_step) * px;
    }
}

// Where a row of A begins: the output pixel, the input position of tap (0, 0), which may lie in the padding, and its byte offset
// modulo 2^32 (EXPAND: that of the image).  Rows follow one another by carry: each sum is less than twice its modulus.
struct HrnRow {
    uint32_t oy, ox;
    int32_t y, x;
    uint32_t off;
};

template <bool EXPAND>
HRN_BOTH HrnRow hrn_row_at(const HrnConvArgs& a, int m) {
    HrnRow r;
    const uint32_t img = a.by_hw((uint32_t)m), rem = (uint32_t)m - img * ((uint32_t)a.HO * a.WO);
    r.oy = a.by_wo(rem);
    r.ox = rem - r.oy * a.WO;
    r.y = (int)(r.oy * a.cstride - a.cpad);
    r.x = (int)(r.ox * a.cstride_w - a.cpad_w);
    r.off = EXPAND ? img * a.img_bytes : ((img * a.H + (uint32_t)r.y) * a.W + (uint32_t)r.x) * a.px;
    return r;
}

template <bool EXPAND>
HRN_BOTH void hrn_next_row(const HrnConvArgs& a, HrnRow& r) {
    r.ox += a.d_ox;
    r.oy += a.d_oy;
    r.x = (int)((uint32_t)r.x + a.x_step);
    r.y = (int)((uint32_t)r.y + a.y_step);
    r.off += a.off_step;
    const bool row = r.ox >= (uint32_t)a.WO;
    r.ox -= row ? a.WO : 0;
    r.oy += row ? 1 : 0;
    r.x = (int)((uint32_t)r.x - (row ? a.x_row : 0u));
    r.y = (int)((uint32_t)r.y + (row ? a.cstride : 0));
    if (!EXPAND) r.off += row ? a.row_bytes : 0u;
    const bool image = r.oy >= (uint32_t)a.HO;
    r.oy -= image ? a.HO : 0;
    r.y = (int)((uint32_t)r.y - (image ? a.y_img : 0u));
    r.off += image ? a.img_bytes : 0u;
}

// Where a lane's chunk is in K: its channel, its tap in input pixels from tap (0, 0), and that and the channel as a byte offset
// modulo 2^32.  Past the end of K it means nothing.
struct HrnTap {
    int32_t c, dy, dx;
    uint32_t off;
};

HRN_BOTH HrnTap hrn_tap_at(const HrnConvArgs& a, int ke, int in_w, int es) {
    HrnTap t;
    const int r = (int)a.by_kwci((uint32_t)ke);
    ke -= r * (a.KW * a.CI);
    const int s = (int)a.by_ci((uint32_t)ke);
    t.c = ke - s * a.CI;
    t.dy = (int)((uint32_t)r * a.cdil);
    t.dx = (int)((uint32_t)s * a.cdil_w);
    t.off = ((uint32_t)t.dy * in_w + (uint32_t)t.dx) * a.px + (uint32_t)t.c * es;
    return t;
}

// ELEMS further along K, to element ke.  Carried where a step goes one tap further at most and a filter row's end shows in dx; a count of the
// taps instead costs 2 - 12 % (fp16 3x3 32x7x7x512 -> 512 27.7 us, 31.0 with the count).  The compiler is told which branch is taken so that
// the division lies outside the k-loop (26.8 -> 26.3 there, 9x46x49x240 -> 64 18.1 -> 17.9, 5x5, stride 2, 2x54x54x352 -> 368 49.3 -> 48.1).
template <int ELEMS, int ES>
HRN_BOTH void hrn_next_tap(const HrnConvArgs& a, HrnTap& t, int ke, int in_w) {
    if (__builtin_expect(a.carry_ci >= ELEMS, 1)) {
        t.c += ELEMS;
        const bool tap = t.c >= a.CI;
        t.c -= tap ? a.CI : 0;
        t.dx = (int)((uint32_t)t.dx + (tap ? a.cdil_w : 0));
        t.off += ELEMS * ES + (tap ? a.tap_bytes : 0u);
        const bool row = (uint32_t)t.dx == a.kw_end;
        t.dx = row ? 0 : t.dx;
        t.dy = (int)((uint32_t)t.dy + (row ? a.cdil : 0));
        t.off += row ? a.taprow_bytes : 0u;
    } else {
        t = hrn_tap_at(a, ke, in_w, ES);
    }
}

#endif
