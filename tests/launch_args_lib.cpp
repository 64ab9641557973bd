// What tests call of hrn_args.h, the arithmetic that launches and kernels share.
#include <type_traits>
#include <vector>

#include "../heron_amd/csrc/hrn_args.h"

namespace {

using i64 = long long;

// im2col loads of an instance (`row_bytes` of K in a tile row, `rows` of a tile a load of every wave, `loads` a lane) over a conv: how many
// (row, K position) pairs find another address, or another answer to whether it is in the image, than the definition gives.
template <int ELEMS, int ES, bool EXPAND>
i64 walk_errors(HrnConvArgs a, int images, int rows, int loads, const int* starts, int n_starts) {
    const int hw = a.HO * a.WO, M = images * hw, K = a.KH * a.KW * a.CI, kts = (K + ELEMS - 1) / ELEMS, tile = rows * loads;
    const int in_w = EXPAND ? a.in_w : a.W, in_h = EXPAND ? a.in_h : a.H;
    a.by_kwci = HrnDiv((uint32_t)(a.KW * a.CI)); a.by_ci = HrnDiv((uint32_t)a.CI);
    a.by_hw = HrnDiv((uint32_t)hw); a.by_wo = HrnDiv((uint32_t)a.WO);
    hrn_walk_args(&a, ES, rows, EXPAND);
    struct Want { HrnRow row; i64 y, x, img; };
    std::vector<Want> want;
    for (int m0 : {0, (M / tile / 2) * tile, ((M - 1) / tile) * tile})
        for (int r0 = 0; r0 < rows; ++r0) {
            HrnRow row = hrn_row_at<EXPAND>(a, m0 + r0);
            for (int i = 0; i < loads; ++i) {
                const int m = m0 + r0 + i * rows;
                if (m < M) {
                    const i64 img = m / hw, oy = m % hw / a.WO, ox = m % a.WO;
                    want.push_back({row, oy * a.cstride - a.cpad, ox * a.cstride_w - a.cpad_w, img});
                }
                hrn_next_row<EXPAND>(a, row);
            }
        }
    i64 errors = 0;
    for (int z = 0; z < n_starts; ++z)
        for (int chunk = 0; chunk < ELEMS * ES / 16; ++chunk) {
            HrnTap t = hrn_tap_at(a, chunk * (16 / ES) + starts[z] * ELEMS, in_w, ES);
            for (int kt = starts[z]; kt < kts; ++kt) {
                const i64 k = (i64)kt * ELEMS + chunk * (16 / ES);
                if (kt > starts[z]) hrn_next_tap<ELEMS, ES>(a, t, (int)k, in_w);
                if (k >= K) break;
                const i64 r = k / (a.KW * a.CI), s = k / a.CI % a.KW, c = k % a.CI;
                for (const Want& w : want) {
                    const i64 iy = w.y + r * a.cdil, ix = w.x + s * a.cdil_w;
                    const bool in = iy >= 0 && iy < a.H && ix >= 0 && ix < a.W;
                    const uint32_t ky = (uint32_t)w.row.y + t.dy, kx = (uint32_t)w.row.x + t.dx;
                    bool ok = in == (ky < (uint32_t)a.H && kx < (uint32_t)a.W) && t.c == c;
                    if (ok && in && EXPAND) ok = ky == (uint32_t)iy && kx == (uint32_t)ix && w.row.off == (uint32_t)(w.img * in_h * in_w * a.CI * ES);
                    if (ok && in && !EXPAND) ok = w.row.off + t.off == (uint32_t)((((w.img * a.H + iy) * a.W + ix) * a.CI + c) * ES);
                    errors += !ok;
                }
            }
        }
    return errors;
}

}  // namespace

extern "C" {

// quotients of ns by d as the kernels compute them
void div_all(const uint32_t* ns, uint32_t* out, int count, uint32_t d) {
    const HrnDiv by(d);
    for (int i = 0; i < count; ++i) out[i] = by(ns[i]);
}

// conv: images, H, W, CI, HO, WO, KH, KW, then (stride, pad, dilation) of the height and of the width, then in_h, in_w (0: not expanded)
long long conv_walk_errors(const int* conv, int es, int row_bytes, int rows, int loads, const int* starts, int n_starts) {
    HrnConvArgs a = {};
    a.H = conv[1]; a.W = conv[2]; a.CI = conv[3]; a.HO = conv[4]; a.WO = conv[5]; a.KH = conv[6]; a.KW = conv[7];
    a.cstride = conv[8]; a.cpad = conv[9]; a.cdil = conv[10];
    a.cstride_w = conv[11]; a.cpad_w = conv[12]; a.cdil_w = conv[13];
    a.in_h = conv[14]; a.in_w = conv[15];
    auto run = [&](auto elems, auto size) -> long long {
        return a.in_h ? walk_errors<decltype(elems)::value, decltype(size)::value, true>(a, conv[0], rows, loads, starts, n_starts)
                      : walk_errors<decltype(elems)::value, decltype(size)::value, false>(a, conv[0], rows, loads, starts, n_starts);
    };
    using std::integral_constant;
    switch (row_bytes * 4 + es) {
        case 64 * 4 + 1: return run(integral_constant<int, 64>{}, integral_constant<int, 1>{});
        case 128 * 4 + 1: return run(integral_constant<int, 128>{}, integral_constant<int, 1>{});
        case 256 * 4 + 1: return run(integral_constant<int, 256>{}, integral_constant<int, 1>{});
        case 64 * 4 + 2: return run(integral_constant<int, 32>{}, integral_constant<int, 2>{});
        case 128 * 4 + 2: return run(integral_constant<int, 64>{}, integral_constant<int, 2>{});
        case 256 * 4 + 2: return run(integral_constant<int, 128>{}, integral_constant<int, 2>{});
    }
    return -1;
}

int args_bytes(int conv) { return conv ? (int)sizeof(HrnConvArgs) : (int)sizeof(HrnKArgs); }

int pair_of(int block, int pairs) { return hrn_pair_of(block, pairs); }
}
