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
// tiles), 435 instead of 283 (fp16 im2col 128x128).
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

struct HrnKArgs {
    const void* A;
    const void* B;
    void* C;
    int32_t M, N, K;            // K in elements
    int32_t lda, ldb, ldc;      // elements
    int64_t sA, sB, sC;         // batch strides, elements
    int32_t tiles_m, tiles_n, group_m, batch;
    // conv
    int32_t H, W, CI, HO, WO, KH, KW, cstride, cpad, cdil;
    int32_t cstride_w, cpad_w, cdil_w;   // conv: the width-direction values (cstride/cpad/cdil are the height ones)
    int32_t split, kt_per_slice;         // split-K: number of K slices and k-tiles per slice
    const void* bsum;                    // uint8 path: per batch entry N column sums of B (sum_k B[n,k], int32), or null
    int32_t out_plane;                   // CHW kernels: row m, column n of the result goes to C[m / out_plane][n][m % out_plane]
    int32_t expand_shift;                // EXPAND kernels: the H x W input is not in memory: pixel (y, x) of the in_h x in_w
    int32_t in_h, in_w, top, left;       // one that is stands at (top + (y << shift), left + (x << shift)), zeros elsewhere
    // split-K: the result and what tells the last slice of a tile to add them all up; arrivals null: a kernel behind this one does
    void* out;
    int64_t out_stride;                  // batch stride of the result, elements
    uint64_t* arrivals;                  // one word per output tile, of any content
    uint64_t ticket;                     // of this launch, its low 16 bits zero
    int32_t out_ld;
    // divisors of the launch: K slices, output tiles of a batch entry, of a raster group, rows of a group and of the last one, conv: elements of
    // a filter row and of a tap, output pixels of an image and of a row, 16-byte pieces of a pixel, pixels of a plane (out_plane)
    HrnDiv by_split, by_tiles, by_group, by_gm, by_gm_last, by_kwci, by_ci, by_hw, by_wo, by_cpp, by_plane;
    // conv, im2col: extents of all taps (dilated) and of the result (times the stride) in input pixels, the bytes of a pixel, and what
    // a byte offset changes by beyond the step itself where K goes on to the next tap and filter row, the pixels to the next row and image
    int32_t kw_end, kh_end, x_row, y_img, px;
    uint32_t tap_bytes, taprow_bytes, row_bytes, img_bytes;
};

// The (output tile, K slice) pair of a split-K workgroup, slices fastest: workgroup i runs on XCD i % 8, and each XCD has an eighth of
// the pairs in their order, the first XCDs one more where 8 does not divide them.
HRN_BOTH int hrn_pair_of(int block, int pairs) {
    const int xcd = block & 7, more = pairs & 7;
    return xcd * (pairs >> 3) + (xcd < more ? xcd : more) + (block >> 3);
}

#endif
