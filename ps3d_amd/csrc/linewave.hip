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

// Whether a mode has a wave kernel for the line length.  (The x products pass of 512 points
// holds six fields of 16 elements per lane, one wave per SIMD: 13.9 ms per 512^3 step
// against 13.2 of the tile pass, which it keeps.)
bool linewave_ok(int n, int mode) {
    if (mode == LM_DIFF || (mode == LM_XMAIN && n == 512)) return false;
    LwSet s;
    return find_set(n, s);
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
