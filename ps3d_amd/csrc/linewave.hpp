// linewave.hpp -- horizontal line passes with the lines in the registers of one wave.
//
// A wave owns G line pairs of one line set: lane = l*G + g holds elements l + L q (q < E)
// of the complex line g, whose real and imaginary parts are the z levels 2g and 2g+1.
// Two layouts of this form are used, one for the coefficients (LI lanes of EI elements) and
// one for the physical values (LO lanes of EO).  Engines:
//   Lay   n = R0 R1 (R2), E a multiple of every radix: a Stockham pass of radix R | E reads
//         its butterflies from the lane's own registers and the last pass leaves its result
//         in the same layout (L = n/E), both layouts are one;
//   Two   n = A B, one butterfly per lane and pass: radix A from the coefficients' layout
//         (LI = B, EI = A), radix B into the physical one (LO = A, EO = B).  Any n with
//         factors up to 25 this way, the lanes beyond 64/max(A, B) lines idle.
// Either way a transform needs one exchange between two passes -- through a slice of LDS
// that only this wave uses: no block barrier, and loads, transforms and stores of different
// waves overlap freely.  Global accesses are 16 bytes a lane, 16 G bytes in a
// row; waves of one block take neighbouring z ranges, so that whole 128-byte lines are used
// by one CU.  Against the tiles in LDS of linepass.hip, a field goes through LDS four times
// instead of eight to ten, and the index arithmetic (two thirds of the instructions there)
// is gone: addresses are a lane offset plus constants.
//
// The Hermitian real form of stafft (src/fft/stafft.f90:55-58, 196-403) pairs slots k and
// n-k: element l + L q pairs with lane L - l, register E-1-q (lane 0: E-q), one more
// exchange ("mirror").  A derivative along the line (sta3dfft.f90:304-377) is a factor
// +-i k on the paired coefficients.
//
// Measured per step against the tile passes (256^3; 128^3): y inverse 1.17 -> 1.11, 0.181 ->
// 0.119 ms; x products 1.47 -> 1.36, 0.27 -> 0.20; y forward 0.40 -> 0.35, 0.084 -> 0.068; adapt
// stage along y 0.93 -> 0.58, 0.18 -> 0.062, and along x 0.75 -> 0.54, 0.155 -> 0.092.  The
// transform-only passes run at 4.4 to 5.1 TB/s (a plain copy: 5.0).
// The two-butterfly engine, whole RK4 steps: 96^3 0.65 -> 0.53 ms, 100^3 1.80 -> 0.63, 160^3
// 5.40 -> 2.22, 200^3 10.2 -> 4.5, 320^3 39.7 -> 21.0, 384^3 41.6 -> 33.3; 32^3 0.223 -> 0.167,
// with the products pass on tiles, as on small grids in general (linewave_xmain).  At 90 points
// and above the passes that hold several fields run one wave per SIMD.
//
// Exchanges move real and imaginary parts one after the other through half the LDS, which
// leaves room for four waves per SIMD.
#pragma once
#include "kernels.hpp"
#include "lfft.hpp"

namespace ps3d {

namespace {

// Line layout: length, elements per lane, radices (R2 = 1: two passes).
template <int N_, int E_, int R0_, int R1_, int R2_>
struct Lay {
    static constexpr int N = N_, E = E_, R0 = R0_, R1 = R1_, R2 = R2_;
    static constexpr int L = N / E, G = 64 / L;
    static constexpr int SK = R0 == 16 ? 4 : 3;     // one pad slot after every R0 elements
    static_assert(R0 * R1 * R2 == N && (R0 == 16 || R0 == 8) && L % (1 << SK) == 0 && 64 % L == 0, "line layout");
    static constexpr int sl(int x) { return x + (x >> SK); }
    // line stride: slots 0..n, and the G lines a 16-lane group touches start 16/G slots apart
    // (mod 16), so that its 8-byte accesses fall on different banks
    static constexpr int LS0 = sl(N) + 1;
    static constexpr int LS = LS0 + ((16 / G) - LS0 % 16 + 16) % 16;
    // twiddle tables of the second and third pass
    static constexpr int S1 = R0, S2 = R0 * R1;
    static constexpr int B1 = S1 <= L ? 1 : E / R1, B2 = S2 <= L ? 1 : E / R2;
    static constexpr int T1 = B1 * (R1 - 1) * L, T2 = R2 > 1 ? B2 * (R2 - 1) * L : 0;
    static constexpr int LEV = 2 * G;               // z levels per wave
    static constexpr bool TWO = false;
    static constexpr int EI = E, EO = E, LI = L, LO = L, TW = T1 + T2;
};
constexpr int kLwWaves = 4;

constexpr int lw_imax(int a, int b) { return a > b ? a : b; }

// n = A B, one butterfly per lane.  The exchange is the transpose of a matrix of A (inverse:
// B rows; forward: A rows of B) with an odd row stride; the mirror takes the elements in order.
template <int A_, int B_>
struct Two {
    static constexpr int A = A_, B = B_, N = A * B;
    static constexpr bool TWO = true;
    static constexpr int EI = A, LI = B, EO = B, LO = A;
    static constexpr int LL = lw_imax(A, B), G = 64 / LL, LEV = 2 * G;
    static constexpr int PA = A | 1, PB = B | 1;     // row strides of the transposes
    static constexpr int LS0 = lw_imax(lw_imax(B * PA, A * PB), N + 1);
    static constexpr int LS = LS0 + ((16 / (G > 16 ? 16 : G)) - LS0 % 16 + 16) % 16;
    static constexpr int TS = B + 1, TW = A * TS;    // table w^(a b), row stride B + 1
};

template <class Y>
constexpr size_t lw_lds() {
    constexpr size_t b = sizeof(double2) * Y::TW + sizeof(double) * kLwWaves * Y::G * Y::LS;
    static_assert(b <= 64 * 1024, "dynamic LDS a kernel may use without asking");
    return b;
}

// ---------------------------------------------------------------------------
// radices beyond lfft.hpp's: Good-Thomas for coprime factors (no twiddles), 9 and 25 as
// 3 x 3 and 5 x 5
// ---------------------------------------------------------------------------
// R = P Q, P and Q coprime: input (Q p + P q) mod R, output (KP p + KQ q) mod R with KP = 1
// mod P and 0 mod Q, KQ the other way round
template <int P, int Q, int KP, int KQ>
__device__ inline void pfa(double2 *u, int dir) {
    constexpr int R = P * Q;
    static_assert(KP % P == 1 % P && KP % Q == 0 && KQ % Q == 1 && KQ % P == 0, "Good-Thomas indices");
    double2 x[R];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        double2 v[P];
#pragma unroll
        for (int p = 0; p < P; ++p) v[p] = u[(Q * p + P * q) % R];
        butterfly(P, v, dir);
#pragma unroll
        for (int p = 0; p < P; ++p) x[q * P + p] = v[p];
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        double2 v[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = x[q * P + p];
        if constexpr (Q == 9) {
            // 3 x 3: w9^(a b)
            const double c1 = 0.76604444311897803520239265055541668, s1 = 0.64278760968653932632264340990726343;
            const double c2 = 0.17364817766693034885171662676931479, s2 = 0.98480775301220805936674302458952301;
            const double c4 = -0.93969262078590838405410927732473147, s4 = 0.34202014332566873304409961468225958;
            const double sg = dir < 0 ? -1.0 : 1.0;
            double2 z[9];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                double2 w[3] = {v[a], v[a + 3], v[a + 6]};
                butterfly(3, w, dir);
#pragma unroll
                for (int b = 0; b < 3; ++b) z[a + 3 * b] = w[b];
            }
            z[4] = cmul(z[4], make_double2(c1, sg * s1));
            z[7] = cmul(z[7], make_double2(c2, sg * s2));
            z[5] = cmul(z[5], make_double2(c2, sg * s2));
            z[8] = cmul(z[8], make_double2(c4, sg * s4));
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                double2 w[3] = {z[3 * b], z[3 * b + 1], z[3 * b + 2]};
                butterfly(3, w, dir);
#pragma unroll
                for (int a = 0; a < 3; ++a) v[b + 3 * a] = w[a];
            }
        } else {
            butterfly(Q, v, dir);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) u[(KP * p + KQ * q) % R] = v[q];
    }
}
// w25^m
__device__ inline double2 w25(int m, double sg) {
    constexpr double c[17] = {1.0000000000000000000000000, 0.9685831611286311194901684, 0.8763066800438635873081159,
                              0.7289686274214115231467303, 0.5358267949789966182713088, 0.3090169943749474241022934,
                              0.0627905195293133760761782, -0.1873813145857246305425507, -0.4257792915650726488625024,
                              -0.6374239897486897101767128, -0.8090169943749474241022934, -0.9297764858882514036609426,
                              -0.9921147013144778310497930, -0.9921147013144778310497930, -0.9297764858882514036609426,
                              -0.8090169943749474241022934, -0.6374239897486897101767128};
    constexpr double s[17] = {0E-25, 0.2486898871648547882422837, 0.4817536741017152749871915,
                              0.6845471059286886737322834, 0.8443279255020150785485581, 0.9510565162951535721164393,
                              0.9980267284282715619523368, 0.9822872507286886810856417, 0.9048270524660195277136686,
                              0.7705132427757892308030096, 0.5877852522924731291687060, 0.3681245526846779591569471,
                              0.1253332335643042453731188, -0.1253332335643042453731188, -0.3681245526846779591569471,
                              -0.5877852522924731291687060, -0.7705132427757892308030096};
    return make_double2(c[m], sg * s[m]);
}
template <int R>
__device__ inline void rad(double2 *u, int dir) {
    if constexpr (R == 6)
        pfa<2, 3, 3, 4>(u, dir);
    else if constexpr (R == 9)
        pfa<1, 9, 0, 1>(u, dir);
    else if constexpr (R == 10)
        pfa<2, 5, 5, 6>(u, dir);
    else if constexpr (R == 12)
        pfa<4, 3, 9, 4>(u, dir);
    else if constexpr (R == 15)
        pfa<3, 5, 10, 6>(u, dir);
    else if constexpr (R == 18)
        pfa<2, 9, 9, 10>(u, dir);
    else if constexpr (R == 20)
        pfa<4, 5, 5, 16>(u, dir);
    else if constexpr (R == 24)
        pfa<8, 3, 9, 16>(u, dir);
    else if constexpr (R == 25) {
        const double sg = dir < 0 ? -1.0 : 1.0;
        double2 z[25];
#pragma unroll
        for (int a = 0; a < 5; ++a) {
            double2 w[5] = {u[a], u[a + 5], u[a + 10], u[a + 15], u[a + 20]};
            butterfly(5, w, dir);
#pragma unroll
            for (int b = 0; b < 5; ++b) z[5 * b + a] = a * b == 0 ? w[b] : cmul(w[b], w25(a * b, sg));
        }
#pragma unroll
        for (int b = 0; b < 5; ++b) {
            double2 w[5] = {z[5 * b], z[5 * b + 1], z[5 * b + 2], z[5 * b + 3], z[5 * b + 4]};
            butterfly(5, w, dir);
#pragma unroll
            for (int a = 0; a < 5; ++a) u[b + 5 * a] = w[a];
        }
    } else {
        bfly<R>(u, dir);
    }
}

// Orders a wave's LDS accesses for the compiler (the LDS runs them in order).
__device__ inline void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Butterfly i = l + L b of a pass with span S: its twiddle index k = i mod S and the
// position of its output t = 0 (output t: + t S).
template <class Y, int S>
__device__ inline int pass_k(int l, int b) {
    if constexpr (S <= Y::L)
        return l % S;
    else
        return l + Y::L * (b % (S / Y::L));
}
template <class Y, int R, int S>
__device__ inline int pass_j(int l, int b) {
    const int i = l + Y::L * b, k = pass_k<Y, S>(l, b);
    return (i - k) * R + k;
}

// The tables w^(k t N / (S R)) of one block, laid out [b][t - 1][l].
template <class Y, int R, int S, int B>
__device__ inline void fill_tw(double2 *dst, const double2 *__restrict__ tw) {
    for (int e = threadIdx.x; e < B * (R - 1) * Y::L; e += blockDim.x) {
        const int l = e % Y::L, t = e / Y::L % (R - 1) + 1, b = e / (Y::L * (R - 1));
        dst[e] = tw[pass_k<Y, S>(l, b) * t * (Y::N / (S * R))];
    }
}

struct LwCtx {
    int l, lo, g;           // lane of the coefficients' and of the physical layout
    double *w;              // the wave's line g in LDS
    const double2 *tw;      // twiddle tables
};

template <class Y, int R, int S, int DIR, bool LAST>
__device__ inline void lw_pass(double2 (&x)[Y::E], const LwCtx &c, const double2 *tw) {
    constexpr int B = Y::E / R;
    constexpr bool SHARED = S <= Y::L;   // one set of twiddles for all butterflies of a lane
#pragma unroll
    for (int b = 0; b < B; ++b) {
        double2 u[R];
#pragma unroll
        for (int t = 0; t < R; ++t) {
            u[t] = x[b + t * B];
            if (S > 1 && t > 0) {
                const double2 w = tw[((SHARED ? 0 : b) * (R - 1) + t - 1) * Y::L + c.l];
                u[t] = DIR < 0 ? cmul(u[t], w) : cmulc(u[t], w);
            }
        }
        bfly<R>(u, DIR);
#pragma unroll
        for (int t = 0; t < R; ++t) x[b + t * B] = u[t];
    }
    if constexpr (!LAST) {
        const int nat = Y::sl(c.l);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const int j = pass_j<Y, R, S>(c.l, b);
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    // S = 1: the R = R0 outputs share a padded group; else S is a multiple of it
                    const int a = S == 1 ? Y::sl(j) + t : Y::sl(j) + Y::sl(t * S);
                    c.w[a] = h ? x[b + t * B].y : x[b + t * B].x;
                }
            }
            lds_order();
#pragma unroll
            for (int q = 0; q < Y::E; ++q) (h ? x[q].y : x[q].x) = c.w[nat + Y::sl(Y::L * q)];
            lds_order();
        }
    }
}

// Unscaled complex DFT of the wave's lines in a Lay layout.
template <class Y, int DIR>
__device__ inline void lw_fft(double2 (&x)[Y::EI], const LwCtx &c) {
    lw_pass<Y, Y::R0, 1, DIR, false>(x, c, nullptr);
    lw_pass<Y, Y::R1, Y::S1, DIR, Y::R2 == 1>(x, c, c.tw);
    if constexpr (Y::R2 > 1) lw_pass<Y, Y::R2, Y::S2, DIR, true>(x, c, c.tw + Y::T1);
}

// Inverse: coefficients x -> physical values y; forward: physical x -> coefficients y.
template <class Y>
__device__ inline void lw_inv(double2 (&x)[Y::EI], double2 (&y)[Y::EO], const LwCtx &c) {
    if constexpr (!Y::TWO) {
#pragma unroll
        for (int q = 0; q < Y::EI; ++q) y[q] = x[q];
        lw_fft<Y, +1>(y, c);
    } else {
        rad<Y::A>(x, +1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < Y::A; ++t) c.w[c.l * Y::PA + t] = h ? x[t].y : x[t].x;
            lds_order();
#pragma unroll
            for (int t = 0; t < Y::B; ++t) (h ? y[t].y : y[t].x) = c.w[t * Y::PA + c.lo];
            lds_order();
        }
#pragma unroll
        for (int t = 1; t < Y::B; ++t) y[t] = cmulc(y[t], c.tw[c.lo * Y::TS + t]);
        rad<Y::B>(y, +1);
    }
}
template <class Y>
__device__ inline void lw_fwd(double2 (&x)[Y::EO], double2 (&y)[Y::EI], const LwCtx &c) {
    if constexpr (!Y::TWO) {
#pragma unroll
        for (int q = 0; q < Y::EI; ++q) y[q] = x[q];
        lw_fft<Y, -1>(y, c);
    } else {
        rad<Y::B>(x, -1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < Y::B; ++t) c.w[c.lo * Y::PB + t] = h ? x[t].y : x[t].x;
            lds_order();
#pragma unroll
            for (int t = 0; t < Y::A; ++t) (h ? y[t].y : y[t].x) = c.w[t * Y::PB + c.l];
            lds_order();
        }
#pragma unroll
        for (int t = 1; t < Y::A; ++t) y[t] = cmul(y[t], c.tw[t * Y::TS + c.l]);
        rad<Y::A>(y, -1);
    }
}

// LDS slot of element l + LI q for the mirror, and of its partner n - l - LI q
template <class Y>
__device__ inline int lw_slot(int l, int q) {
    if constexpr (Y::TWO)
        return l + Y::LI * q;
    else
        return Y::sl(l) + Y::sl(Y::L * q);
}

// Part h of every element into the wave's line, and the slot of element n - k of
// k = l + L q there (k = 0: itself) by lw_mir.
template <class Y>
__device__ inline void lw_put(const double2 (&x)[Y::EI], const LwCtx &c, int h) {
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) c.w[lw_slot<Y>(c.l, q)] = h ? x[q].y : x[q].x;
    if (c.l == 0) c.w[lw_slot<Y>(0, Y::EI)] = h ? x[0].y : x[0].x;   // element n is element 0
    lds_order();
}
template <class Y>
__device__ inline double lw_mir(const LwCtx &c, int q) {
    return c.w[lw_slot<Y>(Y::LI - c.l, Y::EI - 1 - q)];
}
// Element l + LI q against n/2: -1 below, +1 above, 0 at 0 or n/2 (their own partners).
// EI even: the half lies between the registers (and at lane 0); odd: inside the middle one.
template <class Y>
__device__ inline int lw_side(const LwCtx &c, int q) {
    if ((Y::EI & 1) && q == Y::EI / 2) {
        const int k2 = 2 * c.l;   // k - n/2 = l - LI/2
        return k2 < Y::LI ? -1 : (k2 > Y::LI ? 1 : 0);
    }
    if ((q == 0 || (!(Y::EI & 1) && q == Y::EI / 2)) && c.l == 0) return 0;
    return q < (Y::EI + 1) / 2 && !(!(Y::EI & 1) && q >= Y::EI / 2) ? -1 : 1;
}

// Hermitian real spectra of two levels -> the complex line's spectrum, times sc.
template <class Y>
__device__ inline void lw_herm_in(double2 (&x)[Y::EI], const LwCtx &c, double sc) {
    double my[Y::EI];
    lw_put<Y>(x, c, 1);
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) my[q] = lw_mir<Y>(c, q);
    lds_order();
    lw_put<Y>(x, c, 0);
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) {
        // k < n/2: s_k + i s_(n-k); k > n/2: s_(n-k) - i s_k; k = 0, n/2: s_k
        const double mx = lw_mir<Y>(c, q);
        const int side = lw_side<Y>(c, q);
        double2 z = side < 0 ? make_double2(x[q].x - my[q], x[q].y + mx) : make_double2(mx + x[q].y, my[q] - x[q].x);
        if (side == 0) z = x[q];
        x[q] = make_double2(sc * z.x, sc * z.y);
    }
    lds_order();
}

// Complex spectrum -> Hermitian real spectra of the two levels, times sc.
template <class Y>
__device__ inline void lw_herm_out(double2 (&x)[Y::EI], const LwCtx &c, double sc) {
    double my[Y::EI];
    lw_put<Y>(x, c, 1);
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) my[q] = lw_mir<Y>(c, q);
    lds_order();
    lw_put<Y>(x, c, 0);
    sc *= 0.5;
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) {
        const double mx = lw_mir<Y>(c, q);
        double2 lo = make_double2(x[q].x + mx, x[q].y + my[q]);
        const double2 hi = make_double2(my[q] - x[q].y, x[q].x - mx);
        if (lw_side<Y>(c, q) > 0) lo = hi;
        x[q] = make_double2(sc * lo.x, sc * lo.y);
    }
    lds_order();
}

// Tile of a wave: z range, line set, addresses.  Lanes beyond a layout's (l >= LI, lo >= LO)
// repeat its last lane: they load and exchange the same values and store and count nothing.
template <class Y>
struct LwTile {
    int l, lo, g, z0, other, tile;
    bool any, full;         // the wave has levels; all of them (else lanes are masked)
    bool v0, v1;            // this lane's levels exist
    bool oni, ono;          // the lane holds a line element of its own in the layout
    bool c0, c1;            // physical layout: the lane's levels count
    long base;              // wave-uniform element offset of (line element 0, level z0)
    unsigned lani, lano;    // lane's element offset
    long stepi, stepo;      // element offset from register to register
};
template <class Y>
__device__ inline LwTile<Y> lw_tile(const LineArgs &a) {
    LwTile<Y> t;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int l = lane / Y::G;
    t.g = lane % Y::G;
    t.oni = l < Y::LI;
    t.ono = l < Y::LO;
    t.l = t.oni ? l : Y::LI - 1;
    t.lo = t.ono ? l : Y::LO - 1;
    // XCD-contiguous tile ranges, as linepass.hip's tile_index
    const int B = gridDim.x, i = blockIdx.x, qn = B >> 3, r = B & 7, xc = i & 7, k = i >> 3;
    t.tile = xc < r ? xc * (qn + 1) + k : r * (qn + 1) + (xc - r) * qn + k;
    const int nz1 = a.g.nz + 1;
    t.z0 = ((t.tile % a.nzt) * kLwWaves + wv) * Y::LEV;
    t.other = t.tile / a.nzt;
    if (t.other >= a.osplit) t.other += a.oshift;
    t.any = t.z0 < nz1;
    t.full = t.z0 + Y::LEV <= nz1;
    t.v0 = t.z0 + 2 * t.g < nz1;
    t.v1 = t.z0 + 2 * t.g + 1 < nz1;
    t.c0 = t.v0 && t.ono;
    t.c1 = t.v1 && t.ono;
    t.base = (long)blockIdx.y * a.bt.vol + (long)t.other * a.ostride + t.z0;
    t.lani = (unsigned)(t.l * a.estride + 2 * t.g);
    t.lano = (unsigned)(t.lo * a.estride + 2 * t.g);
    t.stepi = (long)Y::LI * a.estride;
    t.stepo = (long)Y::LO * a.estride;
    return t;
}
// O: physical layout, else the coefficients'
template <class Y, bool O, int E>
__device__ inline void lw_load(const LwTile<Y> &t, const double *__restrict__ src, double2 (&x)[E]) {
    static_assert(E == (O ? Y::EO : Y::EI), "layout");
    const double *p = src + t.base;
    const long step = O ? t.stepo : t.stepi;
    const unsigned lane = O ? t.lano : t.lani;
    if (t.full) {
#pragma unroll
        for (int q = 0; q < E; ++q, p += step) x[q] = *reinterpret_cast<const double2 *>(p + lane);
    } else {
        // a pair whose second level is beyond the lid reads the column's padding (columns
        // are padded to 16 levels); the level is zeroed, as it shares a complex line
#pragma unroll
        for (int q = 0; q < E; ++q, p += step) {
            x[q] = make_double2(0.0, 0.0);
            if (t.v0) x[q] = *reinterpret_cast<const double2 *>(p + lane);
            if (!t.v1) x[q].y = 0.0;
        }
    }
}
// coefficients: only slots of wavenumber index <= kb
template <class Y, bool O, int E>
__device__ inline void lw_store(const LwTile<Y> &t, double *__restrict__ dst, const double2 (&x)[E], int kb) {
    static_assert(E == (O ? Y::EO : Y::EI), "layout");
    double *p = dst + t.base;
    const long step = O ? t.stepo : t.stepi;
    const unsigned lane = O ? t.lano : t.lani;
#pragma unroll
    for (int q = 0; q < E; ++q, p += step) {
        bool on = (t.full || t.v0) && (O ? t.ono : t.oni);
        if (!O) {
            const int j = t.l + Y::LI * q;
            on = on && (j <= kb || j >= Y::N - kb);
        }
        if (!on) continue;
        if (t.full || t.v1)
            *reinterpret_cast<double2 *>(p + lane) = x[q];
        else
            p[lane] = x[q].x;
    }
}

template <class Y>
__device__ inline LwCtx lw_ctx(const LwTile<Y> &t, double2 *smem, const LineArgs &a) {
    LwCtx c;
    c.l = t.l;
    c.lo = t.lo;
    c.g = t.g;
    c.tw = smem;
    double *w = reinterpret_cast<double *>(smem + Y::TW);
    c.w = w + ((threadIdx.x >> 6) * Y::G + t.g) * Y::LS;
    if constexpr (Y::TWO) {
        for (int e = threadIdx.x; e < Y::A * Y::B; e += blockDim.x)
            smem[(e / Y::B) * Y::TS + e % Y::B] = a.tw[(e / Y::B) * (e % Y::B)];
    } else {
        fill_tw<Y, Y::R1, Y::S1, Y::B1>(smem, a.tw);
        if constexpr (Y::R2 > 1) fill_tw<Y, Y::R2, Y::S2, Y::B2>(smem + Y::T1, a.tw);
    }
    __syncthreads();   // the only one: the tables are read by every wave
    return c;
}

// waves per SIMD of the transform-only passes: what their registers allow without spills
template <class Y>
constexpr int lw_occ() {
    return lw_imax(Y::EI, Y::EO) <= 8 ? 4 : lw_imax(Y::EI, Y::EO) <= 16 ? 3 : 2;
}
// Whether a pass over several fields loads them all before the first transform: with at
// most 8 elements per lane they fit the registers, and such short lines have too few waves
// to hide a load per field (32^3: products pass 71 -> 66 us per step); longer ones spill.
template <class Y>
constexpr bool lw_pre() {
    return Y::TWO && Y::EI <= 8;
}
// and of the passes that hold several fields of EO elements
template <class Y>
constexpr int lw_occ_held() {
    return Y::EO <= 8 ? 2 : 1;
}

// nf fields forward (FWD) or inverse, one per block (blockIdx.z): a wave that loops over
// the fields leaves the last round of waves nearly empty (256^3: 8.3 waves per SIMD; 1.47
// against 1.11 ms per step).  Three waves per SIMD: at four the 16 elements per lane spill
// (1.16 ms).
template <class Y, bool FWD>
__global__ void __launch_bounds__(64 * kLwWaves) __attribute__((amdgpu_waves_per_eu(lw_occ<Y>(), 8)))
k_lw_lines(LineArgs a) {
    extern __shared__ double2 lwsm[];
    if (gated_off(a.g.gate)) return;
    const LwTile<Y> t = lw_tile<Y>(a);
    const LwCtx c = lw_ctx<Y>(t, lwsm, a);
    if (!t.any) return;
    const double sc = 1.0 / sqrt((double)Y::N);
    const int f = blockIdx.z;
    double2 x[Y::EI], y[Y::EO];
    if constexpr (FWD) {
        lw_load<Y, true>(t, a.in[f], y);
        lw_fwd<Y>(y, x, c);
        lw_herm_out<Y>(x, c, sc);
        lw_store<Y, false>(t, a.out[f], x, a.kb);
    } else {
        lw_load<Y, false>(t, a.in[f], x);
        lw_herm_in<Y>(x, c, sc);
        lw_inv<Y>(x, y, c);
        lw_store<Y, true>(t, a.out[f], y, 0);
    }
}

// closure input: channel ch of the bf16 tensor [p][16], p = (ix*ny + iy)*(nz+1) + iz
template <class Y>
__device__ inline void lw_export(const LwTile<Y> &t, const LineArgs &a, const double2 (&x)[Y::EO], int ch) {
    if (!a.nn_in) return;
    const float s = a.nn_scale[ch];
#pragma unroll
    for (int q = 0; q < Y::EO; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (!(h ? t.c1 : t.c0)) continue;
            const long p = ((long)(t.lo + Y::LO * q) * a.g.ny + t.other) * (a.g.nz + 1) + t.z0 + 2 * t.g + h;
            uint32_t u = __builtin_bit_cast(uint32_t, (float)(h ? x[q].y : x[q].x) * s);
            u += 0x7fffu + ((u >> 16) & 1u);
            a.nn_in[p * 16 + ch] = (uint16_t)(u >> 16);
        }
}

// Coefficients of element k times i k (derivative along the line), zero at 0 and n/2.
template <class Y>
__device__ inline void lw_deriv(double2 (&x)[Y::EI], const LwCtx &c, const double *__restrict__ rk) {
#pragma unroll
    for (int q = 0; q < Y::EI; ++q) {
        const int side = lw_side<Y>(c, q);
        double r = rk[c.l + Y::LI * q];
        r = side < 0 ? r : (side > 0 ? -r : 0.0);
        x[q] = make_double2(-r * x[q].y, r * x[q].x);
    }
}

// Adapt stage along y: nf fields inverse and, of the first three, the inverse of the
// derivative too (out[9 + f]).  The second reading of a tile goes past the L2 again: 1.51 GB
// fetched at 256^3 for the 0.86 of six padded volumes, 578 us.
template <class Y>
__global__ void __launch_bounds__(64 * kLwWaves) __attribute__((amdgpu_waves_per_eu(lw_occ<Y>() > 3 ? 3 : lw_occ<Y>(), 8)))
k_lw_inv_d(LineArgs a) {
    extern __shared__ double2 lwsm[];
    if (gated_off(a.g.gate)) return;
    const LwTile<Y> t = lw_tile<Y>(a);
    const LwCtx c = lw_ctx<Y>(t, lwsm, a);
    if (!t.any) return;
    const double sc = 1.0 / sqrt((double)Y::N);
    const int f = blockIdx.z;
    for (int d = f < 3 ? 1 : 0; d >= 0; --d) {
        double2 x[Y::EI], y[Y::EO];
        lw_load<Y, false>(t, a.in[f], x);
        lw_herm_in<Y>(x, c, sc);
        if (d) lw_deriv<Y>(x, c, a.rk);
        lw_inv<Y>(x, y, c);
        lw_store<Y, true>(t, a.out[d ? 9 + f : f], y, 0);
    }
}

template <class Y>
__device__ inline double lw_max(const LwTile<Y> &t, const double2 (&x)[Y::EO]) {
    double m = -INFINITY;
#pragma unroll
    for (int q = 0; q < Y::EO; ++q) {
        if (t.c0) m = fmax(m, x[q].x);
        if (t.c1) m = fmax(m, x[q].y);
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) m = fmax(m, __shfl_xor(m, s));
    return m;
}

// x products pass: r = u eta - v xi, q = w xi - u zeta, p = v zeta - w eta with
// omega + f_cor (inversion.f90:316-352).  The fields come in the order u, eta, w, xi, v,
// zeta, around the cycle of the six products, so that at most five are held while the sixth
// is transformed: 250 VGPRs at eight elements per lane, two waves per SIMD.  (Measured:
// loading each field during the transform before it spills 30 registers and is slower,
// 1.47 against 1.36 ms per 256^3 step.)
template <class Y>
__global__ void __launch_bounds__(64 * kLwWaves) __attribute__((amdgpu_waves_per_eu(lw_occ_held<Y>(), 8)))
k_lw_xmain(LineArgs a) {
    constexpr int E = Y::EO;
    extern __shared__ double2 lwsm[];
    if (gated_off(a.g.gate)) return;
    const LwTile<Y> t = lw_tile<Y>(a);
    const LwCtx c = lw_ctx<Y>(t, lwsm, a);
    const double sc = 1.0 / sqrt((double)Y::N);
    const bool pm = a.part != nullptr;
    __shared__ double red[kLwWaves][RM_N];
    auto put_max = [&](double um, double vm, double wm) {   // adapt stage: signed maxima (advance.f90:319-321)
        if (!pm) return;
        if ((threadIdx.x & 63) == 0) {
            red[threadIdx.x >> 6][RM_UMAX] = um;
            red[threadIdx.x >> 6][RM_VMAX] = vm;
            red[threadIdx.x >> 6][RM_WMAX] = wm;
        }
        __syncthreads();
        if (threadIdx.x < RM_N) {
            double v = red[0][threadIdx.x];
#pragma unroll
            for (int w = 1; w < kLwWaves; ++w) v = fmax(v, red[w][threadIdx.x]);
            a.part[(size_t)blockIdx.y * a.bt.part + (size_t)t.tile * RM_N + threadIdx.x] = v;
        }
    };
    if (!t.any) {
        put_max(-INFINITY, -INFINITY, -INFINITY);
        return;
    }
    // short lines: all six fields are loaded at once (registers allow it), as their grids have
    // few waves per SIMD to cover one load after the other
    constexpr bool PRE = lw_pre<Y>();
    double2 pre[PRE ? 6 : 1][Y::EI];
    if (PRE && !a.phys_in)
#pragma unroll
        for (int f = 0; f < 6; ++f) lw_load<Y, false>(t, a.in[f], pre[f % (PRE ? 6 : 1)]);
    auto phys = [&](int f, double2(&x)[E]) {
        if (a.phys_in) {
            lw_load<Y, true>(t, a.in[f], x);
        } else if constexpr (PRE) {
            lw_herm_in<Y>(pre[f], c, sc);
            lw_inv<Y>(pre[f], x, c);
        } else {
            double2 s[Y::EI];
            lw_load<Y, false>(t, a.in[f], s);
            lw_herm_in<Y>(s, c, sc);
            lw_inv<Y>(s, x, c);
        }
        lw_export<Y>(t, a, x, f);
    };
    auto fwd = [&](double2(&x)[E], int f) {
        double2 s[Y::EI];
        lw_fwd<Y>(x, s, c);
        lw_herm_out<Y>(s, c, sc);
        lw_store<Y, false>(t, a.out[f], s, a.kb);
    };
    auto add = [&](double2(&x)[E], double f) {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i] = make_double2(x[i].x + f, x[i].y + f);
    };
    double2 u[E], r[E], p[E], q[E], s[E], v[E];
    phys(0, u);
    const double um = pm ? lw_max<Y>(t, u) : 0.0;
    phys(4, s);            // eta
    add(s, a.fcor[1]);
#pragma unroll
    for (int i = 0; i < E; ++i) r[i] = make_double2(u[i].x * s[i].x, u[i].y * s[i].y);
    phys(2, v);            // w
    const double wm = pm ? lw_max<Y>(t, v) : 0.0;
#pragma unroll
    for (int i = 0; i < E; ++i) p[i] = make_double2(-v[i].x * s[i].x, -v[i].y * s[i].y);
    phys(3, q);            // xi
    add(q, a.fcor[0]);
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const double2 xi = q[i];
        q[i] = make_double2(v[i].x * xi.x, v[i].y * xi.y);
        v[i] = xi;
    }
    phys(1, s);            // v
    const double vm = pm ? lw_max<Y>(t, s) : 0.0;
#pragma unroll
    for (int i = 0; i < E; ++i) r[i] = make_double2(r[i].x - s[i].x * v[i].x, r[i].y - s[i].y * v[i].y);
    fwd(r, 0);
    phys(5, v);            // zeta
    add(v, a.fcor[2]);
#pragma unroll
    for (int i = 0; i < E; ++i) {
        p[i] = make_double2(s[i].x * v[i].x + p[i].x, s[i].y * v[i].y + p[i].y);
        q[i] = make_double2(q[i].x - u[i].x * v[i].x, q[i].y - u[i].y * v[i].y);
    }
    fwd(q, 1);
    fwd(p, 2);
    put_max(um, vm, wm);
}

// Largest |eigenvalue| of a traceless symmetric matrix from p^2 = tr(S^2)/6 and its
// determinant.  The roots of the characteristic cubic are 2 p cos((acos r + 2 pi j) / 3) with
// r = det / (2 p^3) (Smith, CACM 4(4), 1961); the largest in modulus is 2 p y with
// 4 y^3 - 3 y = |r|, y in [sqrt(3)/2, 1]: a simple root with derivative 12 y^2 - 3 >= 6, so
// Newton's iteration gives it to rounding.  Three steps in 32 bits, two with 64-bit
// residuals and the 32-bit slope (error 1e-7, then 1e-14, then rounding).
__device__ inline double eig_absmax0(double p2, double det) {
    if (!(p2 > 0.0)) return 0.0;
    const double p = sqrt(p2);
    const double r = fmin(1.0, 0.5 * fabs(det) / (p2 * p));
    const float rf = (float)r;
    float yf = 0.8660254f + 0.1339746f * rf;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float y2 = yf * yf;
        yf -= (yf * (4.0f * y2 - 3.0f) - rf) * __builtin_amdgcn_rcpf(12.0f * y2 - 3.0f);
    }
    double y = (double)yf;
    const double s = (double)__builtin_amdgcn_rcpf(12.0f * yf * yf - 3.0f);
#pragma unroll
    for (int i = 0; i < 2; ++i) y -= (y * (4.0 * y * y - 3.0) - r) * s;
    return 2.0 * p * y;
}

// x adapt pass (advance.f90:171-289): max |omega|, the largest |eigenvalue| of the
// symmetrised strain, its lid maxima, and the sums of the characteristic vorticity; velocity
// maxima where the products pass has not taken them.  S11 = u_x, S12 = u_y + zeta/2,
// S13 = w_x + eta/2, S22 = v_y, S23 = w_y - xi/2, S33 = -(u_x + v_y) (225-257): the vorticity
// comes first and the strain is built in its place, so that five fields are held at most.
// The z-midpoint vorticity (field_diagnostics.f90:501-545) is formed here, from the level
// below the wave's tile as one more line pair, instead of going through the z and y passes
// as three more fields.  Eigenvalues lie between sqrt(3) p and 2 p, so only points with
// p^2 >= 3/4 of the wave's largest are evaluated.  Five fields and the sums spill 264 to 392
// bytes a lane at most lengths, 0.33 GB written at 256^3: 520 us, 2.05 TB/s of the eight fields.
template <class Y>
__global__ void __launch_bounds__(64 * kLwWaves) __attribute__((amdgpu_waves_per_eu(lw_occ_held<Y>(), 8)))
k_lw_xadapt(LineArgs a) {
    constexpr int E = Y::EO;
    extern __shared__ double2 lwsm[];
    if (gated_off(a.g.gate)) return;
    const LwTile<Y> t = lw_tile<Y>(a);
    const LwCtx c = lw_ctx<Y>(t, lwsm, a);
    const double sc = 1.0 / sqrt((double)Y::N);
    const int nz = a.g.nz;
    double res[RX_N] = {0.0, 2.220446049250313e-16, 0.0, 0.0, -INFINITY, -INFINITY, -INFINITY, 0.0, 0.0};
    if (t.any) {
        auto inv = [&](double2(&s)[Y::EI], double2(&x)[E]) {
            lw_herm_in<Y>(s, c, sc);
            lw_inv<Y>(s, x, c);
        };
        auto phys = [&](int f, double2(&x)[E]) {
            if (a.phys_in) {
                lw_load<Y, true>(t, a.in[f], x);
            } else {
                double2 s[Y::EI];
                lw_load<Y, false>(t, a.in[f], s);
                inv(s, x);
            }
        };
        auto deriv = [&](int f, double2(&x)[E]) {
            double2 s[Y::EI];
            if (a.phys_in) {   // the complex line's spectrum as it is
                lw_load<Y, true>(t, a.in[f], x);
                lw_fwd<Y>(x, s, c);
            } else {
                lw_load<Y, false>(t, a.in[f], s);
                lw_herm_in<Y>(s, c, sc);
            }
            lw_deriv<Y>(s, c, a.rk);
            lw_inv<Y>(s, x, c);
            if (a.phys_in)
#pragma unroll
                for (int q = 0; q < E; ++q) x[q] = make_double2(x[q].x * (1.0 / Y::N), x[q].y * (1.0 / Y::N));
        };
        double2 s1[E], s2[E], s3[E], s4[E], s5[E];
        if (!a.velmax_given) {
            for (int f = 0; f < 3; ++f) {
                phys(f, s1);
                res[RX_UMAX + f] = lw_max<Y>(t, s1);
            }
        }
        phys(3, s1);   // xi
        phys(4, s2);   // eta
        phys(5, s3);   // zeta
        {
            // the level below: (xi, eta) in the first line, zeta in the second (the halo
            // values then sit in lanes g = 0 and 1)
            static_assert(Y::G > 1, "two lines for the level below");
            double2 hx[E];
            auto halo = [&](auto &h, int l, long step) {
                const long zb = t.base - 1 + (long)l * a.estride;
#pragma unroll
                for (int q = 0; q < (int)(sizeof(h) / sizeof(h[0])); ++q) {
                    h[q] = make_double2(0.0, 0.0);
                    if (t.z0 > 0 && t.g == 0) h[q] = make_double2(a.in[3][zb + q * step], a.in[4][zb + q * step]);
                    if (t.z0 > 0 && t.g == 1) h[q].x = a.in[5][zb + q * step];
                }
            };
            if (a.phys_in) {
                halo(hx, t.lo, t.stepo);
            } else {
                double2 s[Y::EI];
                halo(s, t.l, t.stepi);
                inv(s, hx);
            }
            const double vortrms = a.scal[(size_t)blockIdx.y * SC_NSCAL + SC_VORTRMS];
            double w2 = 0.0, l1 = 0.0, l2 = 0.0;
#pragma unroll
            for (int q = 0; q < E; ++q) {
                // level below 2g: the upper level of the pair below, or the halo
                double p1 = hx[q].x, p2 = hx[q].y, p3 = __shfl_down(hx[q].x, 1);
                const double u1 = __shfl_up(s1[q].y, 1), u2 = __shfl_up(s2[q].y, 1), u3 = __shfl_up(s3[q].y, 1);
                if (t.g > 0) {
                    p1 = u1;
                    p2 = u2;
                    p3 = u3;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (!(h ? t.c1 : t.c0)) continue;
                    const double o1 = h ? s1[q].y : s1[q].x, o2 = h ? s2[q].y : s2[q].x, o3 = h ? s3[q].y : s3[q].x;
                    w2 = fmax(w2, o1 * o1 + o2 * o2 + o3 * o3);
                    if (h == 0 && t.z0 + 2 * t.g == 0) continue;
                    const double t1 = fabs(0.5 * ((h ? s1[q].x : p1) + o1)), t2 = fabs(0.5 * ((h ? s2[q].x : p2) + o2)),
                                 t3 = fabs(0.5 * ((h ? s3[q].x : p3) + o3));
                    if (t1 + t2 + t3 > vortrms) {
                        l1 += t1 + t2 + t3;
                        l2 += t1 * t1 + t2 * t2 + t3 * t3;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // one element at a time (registers)
            }
            res[RX_W2MAX] = w2;
            res[RX_L1] = l1;
            res[RX_L2] = l2;
        }
        auto into = [&](double2(&s)[E], const double2(&d)[E], double f) {   // s = d + f s
#pragma unroll
            for (int q = 0; q < E; ++q) s[q] = make_double2(d[q].x + f * s[q].x, d[q].y + f * s[q].y);
        };
            phys(8, s4);         // dw/dy
        into(s1, s4, -0.5);  // S23
        phys(6, s4);         // du/dy
        into(s3, s4, 0.5);   // S12
        deriv(2, s4);        // dw/dx
        into(s2, s4, 0.5);   // S13
        deriv(0, s5);        // du/dx
        phys(7, s4);         // dv/dy
        // p^2 of point (q, h); evaluated again where it is needed, to hold fewer registers
#define C_(V) (h ? (V).y : (V).x)
        auto psq = [&](int q, int h) {
            const double x = C_(s5[q]), y = C_(s4[q]), z = x + y, b = C_(s3[q]), d = C_(s2[q]), e = C_(s1[q]);
            return ((x * x + y * y + z * z) + 2.0 * (b * b + d * d + e * e)) * (1.0 / 6.0);
        };
        double pmax = 0.0;
#pragma unroll
        for (int q = 0; q < E; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (h ? t.c1 : t.c0) pmax = fmax(pmax, psq(q, h));
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) pmax = fmax(pmax, __shfl_xor(pmax, m));
        const double cut = 0.75 * (1.0 - 1.0e-6) * pmax;
        const bool lids = t.z0 == 0 || t.z0 + Y::LEV > nz;   // the tile has a lid (wave-uniform)
        double gg = 2.220446049250313e-16, us = 0.0, ls = 0.0;
#pragma unroll
        for (int q = 0; q < E; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int z = t.z0 + 2 * t.g + h;
                const bool lid = lids && (z == 0 || z == nz);
                const double p2 = psq(q, h);
                if (!((h ? t.c1 : t.c0) && (p2 >= cut || lid))) continue;
                const double x = C_(s5[q]), y = C_(s4[q]), b = C_(s3[q]), d = C_(s2[q]), e = C_(s1[q]);
                const double w = -(x + y);
                const double lam = eig_absmax0(p2, x * (y * w - e * e) - b * (b * w - e * d) + d * (b * e - y * d));
                gg = fmax(gg, lam);
                if (z == nz) us = fmax(us, lam);
                if (z == 0) ls = fmax(ls, lam);
                __builtin_amdgcn_sched_barrier(0);   // one point at a time (registers)
            }
#undef C_
        res[RX_GG] = gg;
        res[RX_USGG] = us;
        res[RX_LSGG] = ls;
    }
    // the block's partial; velocity maxima are the wave's already
    __shared__ double red[kLwWaves][RX_N];
#pragma unroll
    for (int k = 0; k < RX_N; ++k) {
        const bool add = k == RX_L1 || k == RX_L2;
        if (k != RX_UMAX && k != RX_VMAX && k != RX_WMAX)
#pragma unroll
            for (int m = 32; m >= 1; m >>= 1) {
                const double o = __shfl_xor(res[k], m);
                res[k] = add ? res[k] + o : fmax(res[k], o);
            }
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = res[k];
    }
    __syncthreads();
    if (threadIdx.x < RX_N) {
        const int k = threadIdx.x;
        double v = red[0][k];
#pragma unroll
        for (int w = 1; w < kLwWaves; ++w) v = (k == RX_L1 || k == RX_L2) ? v + red[w][k] : fmax(v, red[w][k]);
        a.part[(size_t)blockIdx.y * a.bt.part + (size_t)t.tile * RX_N + k] = v;
    }
}

template <class Y>
LineArgs lw_args(const LineArgs &a) {
    LineArgs b = a;
    b.ZC = Y::LEV * kLwWaves;
    b.nzt = (a.g.nz + 1 + b.ZC - 1) / b.ZC;
    return b;
}
template <class Y, bool FWD>
hipError_t go_lines(const LineArgs &a, hipStream_t stream) {
    const LineArgs b = lw_args<Y>(a);
    hipLaunchKernelGGL((k_lw_lines<Y, FWD>), dim3(b.nother * b.nzt, b.bt.nb > 1 ? b.bt.nb : 1, b.nf),
                       dim3(64 * kLwWaves), lw_lds<Y>(), stream, b);
    return hipGetLastError();
}
template <class Y>
hipError_t go_held(const LineArgs &a, hipStream_t stream) {
    const LineArgs b = lw_args<Y>(a);
    const dim3 grid(b.nother * b.nzt, b.bt.nb > 1 ? b.bt.nb : 1), block(64 * kLwWaves);
    if (a.mode == LM_XMAIN)
        hipLaunchKernelGGL((k_lw_xmain<Y>), grid, block, lw_lds<Y>(), stream, b);
    else
        hipLaunchKernelGGL((k_lw_xadapt<Y>), grid, block, lw_lds<Y>(), stream, b);
    return hipGetLastError();
}
template <class Y>
hipError_t go_inv_d(const LineArgs &a, hipStream_t stream) {
    const LineArgs b = lw_args<Y>(a);
    hipLaunchKernelGGL((k_lw_inv_d<Y>), dim3(b.nother * b.nzt, b.bt.nb > 1 ? b.bt.nb : 1, 6), dim3(64 * kLwWaves),
                       lw_lds<Y>(), stream, b);
    return hipGetLastError();
}
// transform-only passes in layout Y, those that hold several fields in layout M
template <class Y, class M>
hipError_t go(const LineArgs &a, hipStream_t stream) {
    switch (a.mode) {
        case LM_FWD: return go_lines<Y, true>(a, stream);
        case LM_INV: return go_lines<Y, false>(a, stream);
        case LM_INV_Y1: return go_inv_d<Y>(a, stream);
        case LM_XMAIN:
        case LM_XADAPT: return go_held<M>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// The built lengths of one source file: z levels of a block of the held passes (0: not
// built), launch.
struct LwSet {
    int (*levels)(int n);
    hipError_t (*launch)(const LineArgs &a, hipStream_t stream);
};
#define PS3D_LW_SET(NAME_, SIZES_)                                                                       \
    static int levels_##NAME_(int n) {                                                                   \
        switch (n) { SIZES_(PS3D_LW_LEV) default: return 0; }                                            \
    }                                                                                                    \
    static hipError_t launch_##NAME_(const LineArgs &a, hipStream_t stream) {                            \
        switch (a.n) { SIZES_(PS3D_LW_GO) default: return hipErrorInvalidValue; }                        \
    }                                                                                                    \
    LwSet lw_set_##NAME_() { return {levels_##NAME_, launch_##NAME_}; }
#define PS3D_LW_LEV(N_, ...) case N_: return LwLay<N_>::M::LEV * kLwWaves;
#define PS3D_LW_GO(N_, ...) case N_: return go<LwLay<N_>::Y, LwLay<N_>::M>(a, stream);
LwSet lw_set_a();
LwSet lw_set_b();
LwSet lw_set_c();
LwSet lw_set_d();
LwSet lw_set_e();
template <int N> struct LwLay;
#define PS3D_LW_TWO(N_, A_, B_)                            \
    template <>                                            \
    struct LwLay<N_> {                                     \
        using Y = Two<A_, B_>;                             \
        using M = Two<A_, B_>;                             \
        static_assert(Y::N == N_, "factors of the length"); \
    };

}  // namespace ps3d
