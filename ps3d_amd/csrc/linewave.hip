// linewave.hip -- wave line passes (linewave.hpp) of the powers of two from 64, and the
// dispatch over all built lengths.
#include "linewave.hpp"

namespace ps3d {

// layouts of the transform-only passes (Y) and of those that hold several fields (M)
template <> struct LwLay<64> { using Y = Lay<64, 8, 8, 8, 1>; using M = Y; };
template <> struct LwLay<128> { using Y = Lay<128, 16, 8, 16, 1>; using M = Lay<128, 8, 8, 4, 4>; };
template <> struct LwLay<256> { using Y = Lay<256, 16, 16, 16, 1>; using M = Lay<256, 8, 8, 8, 4>; };
// (8 elements per lane, one level pair per wave: the held passes are 1.5-1.7x slower)
template <> struct LwLay<512> { using Y = Lay<512, 16, 8, 8, 8>; using M = Y; };
#define SIZES(X) X(64) X(128) X(256) X(512)
PS3D_LW_SET(pow2, SIZES)

static bool find_set(int n, LwSet &set) {
    static LwSet (*const sets[])() = {lw_set_pow2, lw_set_a, lw_set_b, lw_set_c, lw_set_d, lw_set_e};
    for (auto f : sets) {
        set = f();
        if (set.levels(n)) return true;
    }
    return false;
}

// Whether a mode has a wave kernel for the line length.  (Of the x products pass, see below;
// at 512 points it holds six fields of 16 elements per lane, one wave per SIMD: 13.9 ms per
// 512^3 step against 13.2 of the tile pass, which it keeps.)
bool linewave_ok(int n, int mode) {
    if (mode == LM_DIFF || (mode == LM_XMAIN && n == 512)) return false;
    LwSet s;
    return find_set(n, s);
}
// Whether the x products pass takes its wave kernel.  A wave does nine transforms one after
// the other, so a grid with less than about a wave per SIMD waits for that chain, where a
// tile's block shares it among its threads: tiles up to 200 thousand points for the short
// lines (4 to 8 elements per lane), up to 450 thousand from 96 points (8 to 16).  Only against
// tiles with a compile-time plan; the run-time plans are twice as slow as the waves at any
// size.  us per pass, waves | tiles: 32^3 16.3 | 12.4, two and four instances 2.5 more on
// waves, eight 5.5 less; 48^3 17.6 | 16.0, two instances 6.8 less on waves; 64x64x32 4.7 more,
// 64^3 2.1 less; 96x64x48 8.6 more, 96^3 34.0 | 33.5; 128x64x32 3.4 more, 128x64x64 2.8 less;
// 256x32x32 5.8 more, 256x64x64 3.5 less; 384x32x32 16.6 more.
// With physical input (ps3d_gpu_source) only three transforms are left, and from 192 points
// the tiles stay ahead: source() of 256^3 820 | 775, 192^3 499 | 486, 128^3 106 | 110.
bool linewave_xmain(int n, size_t points, bool phys_in) {
    if (!linewave_ok(n, LM_XMAIN)) return false;
    if (!line_reg_ok(n, 512)) return true;
    return points > (n < 96 ? 200000u : 450000u) && !(phys_in && n > 128);
}
int linewave_blocks(int n, int nz) {
    LwSet s;
    if (!find_set(n, s)) return 0;
    const int zc = s.levels(n);
    return (nz + 1 + zc - 1) / zc;
}
hipError_t launch_linewave(const LineArgs &a, hipStream_t stream) {
    LwSet s;
    return find_set(a.n, s) ? s.launch(a, stream) : hipErrorInvalidValue;
}

}  // namespace ps3d
