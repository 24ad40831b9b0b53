// Register-resident DFTs of the periodic passes: radix R in one lane.
//
// dft_reg<R>(v, DIR) transforms v[0..R) in natural order (DIR = -1 forward,
// +1 backward, not normalised).  Composite radices are split R = A B inside the
// lane with constant twiddles, so a line of length R1 R2 takes one exchange
// through LDS instead of one per factor 2, 3, 4, 5, 8.  Products are written as
// explicit fused multiply-adds: a transform rounds the same way in every
// kernel that it is inlined into.
#pragma once
#include "cf_device.h"

namespace cf {

// cos and sin of 2 pi t / R, correctly rounded
template <int R> struct RegTwiddle;
template <> struct RegTwiddle<3> {
    static constexpr double c[3] = {1.0, -0.5, -0.5};
    static constexpr double s[3] = {0.0, 0.8660254037844386, -0.8660254037844386};
};
template <> struct RegTwiddle<5> {
    static constexpr double c[5] = {1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475,
        0.30901699437494745};
    static constexpr double s[5] = {0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731,
        -0.9510565162951535};
};
template <> struct RegTwiddle<6> {
    static constexpr double c[6] = {1.0, 0.5, -0.5, -1.0, -0.5, 0.5};
    static constexpr double s[6] = {0.0, 0.8660254037844386, 0.8660254037844386, 0.0, -0.8660254037844386,
        -0.8660254037844386};
};
template <> struct RegTwiddle<7> {
    static constexpr double c[7] = {1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191,
        -0.9009688679024191, -0.2225209339563144, 0.6234898018587335};
    static constexpr double s[7] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581,
        -0.4338837391175581, -0.9749279121818236, -0.7818314824680298};
};
template <> struct RegTwiddle<8> {
    static constexpr double c[8] = {1.0, 0.7071067811865476, 0.0, -0.7071067811865476, -1.0,
        -0.7071067811865476, 0.0, 0.7071067811865476};
    static constexpr double s[8] = {0.0, 0.7071067811865476, 1.0, 0.7071067811865476, 0.0, -0.7071067811865476,
        -1.0, -0.7071067811865476};
};
template <> struct RegTwiddle<9> {
    static constexpr double c[9] = {1.0, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084,
        -0.9396926207859084, -0.5, 0.17364817766693036, 0.766044443118978};
    static constexpr double s[9] = {0.0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386,
        0.3420201433256687, -0.3420201433256687, -0.8660254037844386, -0.984807753012208, -0.6427876096865394};
};
template <> struct RegTwiddle<10> {
    static constexpr double c[10] = {1.0, 0.8090169943749475, 0.30901699437494745, -0.30901699437494745,
        -0.8090169943749475, -1.0, -0.8090169943749475, -0.30901699437494745, 0.30901699437494745,
        0.8090169943749475};
    static constexpr double s[10] = {0.0, 0.5877852522924731, 0.9510565162951535, 0.9510565162951535,
        0.5877852522924731, 0.0, -0.5877852522924731, -0.9510565162951535, -0.9510565162951535,
        -0.5877852522924731};
};
template <> struct RegTwiddle<12> {
    static constexpr double c[12] = {1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0,
        -0.8660254037844386, -0.5, 0.0, 0.5, 0.8660254037844386};
    static constexpr double s[12] = {0.0, 0.5, 0.8660254037844386, 1.0, 0.8660254037844386, 0.5, 0.0, -0.5,
        -0.8660254037844386, -1.0, -0.8660254037844386, -0.5};
};
template <> struct RegTwiddle<14> {
    static constexpr double c[14] = {1.0, 0.9009688679024191, 0.6234898018587335, 0.2225209339563144,
        -0.2225209339563144, -0.6234898018587335, -0.9009688679024191, -1.0, -0.9009688679024191,
        -0.6234898018587335, -0.2225209339563144, 0.2225209339563144, 0.6234898018587335, 0.9009688679024191};
    static constexpr double s[14] = {0.0, 0.4338837391175581, 0.7818314824680298, 0.9749279121818236,
        0.9749279121818236, 0.7818314824680298, 0.4338837391175581, 0.0, -0.4338837391175581,
        -0.7818314824680298, -0.9749279121818236, -0.9749279121818236, -0.7818314824680298,
        -0.4338837391175581};
};
template <> struct RegTwiddle<15> {
    static constexpr double c[15] = {1.0, 0.9135454576426009, 0.6691306063588582, 0.30901699437494745,
        -0.10452846326765347, -0.5, -0.8090169943749475, -0.9781476007338057, -0.9781476007338057,
        -0.8090169943749475, -0.5, -0.10452846326765347, 0.30901699437494745, 0.6691306063588582,
        0.9135454576426009};
    static constexpr double s[15] = {0.0, 0.4067366430758002, 0.7431448254773942, 0.9510565162951535,
        0.9945218953682733, 0.8660254037844386, 0.5877852522924731, 0.20791169081775934, -0.20791169081775934,
        -0.5877852522924731, -0.8660254037844386, -0.9945218953682733, -0.9510565162951535, -0.7431448254773942,
        -0.4067366430758002};
};
template <> struct RegTwiddle<16> {
    static constexpr double c[16] = {1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0,
        -0.3826834323650898, -0.7071067811865476, -0.9238795325112867, -1.0, -0.9238795325112867,
        -0.7071067811865476, -0.3826834323650898, 0.0, 0.3826834323650898, 0.7071067811865476,
        0.9238795325112867};
    static constexpr double s[16] = {0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867, 1.0,
        0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0, -0.3826834323650898,
        -0.7071067811865476, -0.9238795325112867, -1.0, -0.9238795325112867, -0.7071067811865476,
        -0.3826834323650898};
};
template <> struct RegTwiddle<18> {
    static constexpr double c[18] = {1.0, 0.9396926207859084, 0.766044443118978, 0.5, 0.17364817766693036,
        -0.17364817766693036, -0.5, -0.766044443118978, -0.9396926207859084, -1.0, -0.9396926207859084,
        -0.766044443118978, -0.5, -0.17364817766693036, 0.17364817766693036, 0.5, 0.766044443118978,
        0.9396926207859084};
    static constexpr double s[18] = {0.0, 0.3420201433256687, 0.6427876096865394, 0.8660254037844386,
        0.984807753012208, 0.984807753012208, 0.8660254037844386, 0.6427876096865394, 0.3420201433256687, 0.0,
        -0.3420201433256687, -0.6427876096865394, -0.8660254037844386, -0.984807753012208, -0.984807753012208,
        -0.8660254037844386, -0.6427876096865394, -0.3420201433256687};
};
template <> struct RegTwiddle<20> {
    static constexpr double c[20] = {1.0, 0.9510565162951535, 0.8090169943749475, 0.5877852522924731,
        0.30901699437494745, 0.0, -0.30901699437494745, -0.5877852522924731, -0.8090169943749475,
        -0.9510565162951535, -1.0, -0.9510565162951535, -0.8090169943749475, -0.5877852522924731,
        -0.30901699437494745, 0.0, 0.30901699437494745, 0.5877852522924731, 0.8090169943749475,
        0.9510565162951535};
    static constexpr double s[20] = {0.0, 0.30901699437494745, 0.5877852522924731, 0.8090169943749475,
        0.9510565162951535, 1.0, 0.9510565162951535, 0.8090169943749475, 0.5877852522924731,
        0.30901699437494745, 0.0, -0.30901699437494745, -0.5877852522924731, -0.8090169943749475,
        -0.9510565162951535, -1.0, -0.9510565162951535, -0.8090169943749475, -0.5877852522924731,
        -0.30901699437494745};
};
template <> struct RegTwiddle<21> {
    static constexpr double c[21] = {1.0, 0.9555728057861407, 0.8262387743159949, 0.6234898018587335,
        0.36534102436639504, 0.07473009358642425, -0.2225209339563144, -0.5, -0.7330518718298263,
        -0.9009688679024191, -0.9888308262251285, -0.9888308262251285, -0.9009688679024191, -0.7330518718298263,
        -0.5, -0.2225209339563144, 0.07473009358642425, 0.36534102436639504, 0.6234898018587335,
        0.8262387743159949, 0.9555728057861407};
    static constexpr double s[21] = {0.0, 0.2947551744109042, 0.5633200580636221, 0.7818314824680298,
        0.9308737486442042, 0.9972037971811801, 0.9749279121818236, 0.8660254037844386, 0.6801727377709194,
        0.4338837391175581, 0.14904226617617444, -0.14904226617617444, -0.4338837391175581, -0.6801727377709194,
        -0.8660254037844386, -0.9749279121818236, -0.9972037971811801, -0.9308737486442042, -0.7818314824680298,
        -0.5633200580636221, -0.2947551744109042};
};
template <> struct RegTwiddle<24> {
    static constexpr double c[24] = {1.0, 0.9659258262890683, 0.8660254037844386, 0.7071067811865476, 0.5,
        0.25881904510252074, 0.0, -0.25881904510252074, -0.5, -0.7071067811865476, -0.8660254037844386,
        -0.9659258262890683, -1.0, -0.9659258262890683, -0.8660254037844386, -0.7071067811865476, -0.5,
        -0.25881904510252074, 0.0, 0.25881904510252074, 0.5, 0.7071067811865476, 0.8660254037844386,
        0.9659258262890683};
    static constexpr double s[24] = {0.0, 0.25881904510252074, 0.5, 0.7071067811865476, 0.8660254037844386,
        0.9659258262890683, 1.0, 0.9659258262890683, 0.8660254037844386, 0.7071067811865476, 0.5,
        0.25881904510252074, 0.0, -0.25881904510252074, -0.5, -0.7071067811865476, -0.8660254037844386,
        -0.9659258262890683, -1.0, -0.9659258262890683, -0.8660254037844386, -0.7071067811865476, -0.5,
        -0.25881904510252074};
};
template <> struct RegTwiddle<32> {
    static constexpr double c[32] = {1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025452,
        0.7071067811865476, 0.5555702330196022, 0.3826834323650898, 0.19509032201612828, 0.0,
        -0.19509032201612828, -0.3826834323650898, -0.5555702330196022, -0.7071067811865476,
        -0.8314696123025452, -0.9238795325112867, -0.9807852804032304, -1.0, -0.9807852804032304,
        -0.9238795325112867, -0.8314696123025452, -0.7071067811865476, -0.5555702330196022, -0.3826834323650898,
        -0.19509032201612828, 0.0, 0.19509032201612828, 0.3826834323650898, 0.5555702330196022,
        0.7071067811865476, 0.8314696123025452, 0.9238795325112867, 0.9807852804032304};
    static constexpr double s[32] = {0.0, 0.19509032201612828, 0.3826834323650898, 0.5555702330196022,
        0.7071067811865476, 0.8314696123025452, 0.9238795325112867, 0.9807852804032304, 1.0, 0.9807852804032304,
        0.9238795325112867, 0.8314696123025452, 0.7071067811865476, 0.5555702330196022, 0.3826834323650898,
        0.19509032201612828, 0.0, -0.19509032201612828, -0.3826834323650898, -0.5555702330196022,
        -0.7071067811865476, -0.8314696123025452, -0.9238795325112867, -0.9807852804032304, -1.0,
        -0.9807852804032304, -0.9238795325112867, -0.8314696123025452, -0.7071067811865476, -0.5555702330196022,
        -0.3826834323650898, -0.19509032201612828};
};

// R = A B; primes and 4, 8 are written out
template <int R> struct RegSplit { static constexpr int A = 0, B = 0; };
template <> struct RegSplit<6> { static constexpr int A = 2, B = 3; };
template <> struct RegSplit<9> { static constexpr int A = 3, B = 3; };
template <> struct RegSplit<10> { static constexpr int A = 2, B = 5; };
template <> struct RegSplit<12> { static constexpr int A = 4, B = 3; };
template <> struct RegSplit<14> { static constexpr int A = 2, B = 7; };
template <> struct RegSplit<15> { static constexpr int A = 3, B = 5; };
template <> struct RegSplit<16> { static constexpr int A = 4, B = 4; };
template <> struct RegSplit<18> { static constexpr int A = 6, B = 3; };
template <> struct RegSplit<20> { static constexpr int A = 4, B = 5; };
template <> struct RegSplit<21> { static constexpr int A = 3, B = 7; };
template <> struct RegSplit<24> { static constexpr int A = 8, B = 3; };
template <> struct RegSplit<32> { static constexpr int A = 8, B = 4; };

__device__ __forceinline__ double2 rot90(double2 a, int dir) { return dir < 0 ? cmulni(a) : cmuli(a); }  // a * exp(dir i pi/2)

// a * exp(dir 2 pi i T / R), T < R
template <int R, int T>
__device__ __forceinline__ double2 reg_twiddle(double2 a, int dir) {
    if constexpr (T == 0) {
        return a;
    } else if constexpr (4 * T == R) {
        return rot90(a, dir);
    } else if constexpr (2 * T == R) {
        return cmk(-a.x, -a.y);
    } else if constexpr (4 * T == 3 * R) {
        return rot90(a, -dir);
    } else {
        const double c = RegTwiddle<R>::c[T], s = dir < 0 ? -RegTwiddle<R>::s[T] : RegTwiddle<R>::s[T];
        return cmk(fma(a.x, c, -(a.y * s)), fma(a.x, s, a.y * c));
    }
}

template <int R>
__device__ __forceinline__ void dft_reg(double2* v, int dir);

// twiddles of sub-transform b: Y_b[p] * exp(dir 2 pi i b p / R), p = P..A-1
template <int R, int A, int B, int b, int P>
__device__ __forceinline__ void reg_twiddle_row(double2 (&y)[B][A], int dir) {
    if constexpr (P < A) {
        y[b][P] = reg_twiddle<R, (b * P) % R>(y[b][P], dir);
        reg_twiddle_row<R, A, B, b, P + 1>(y, dir);
    }
}
template <int R, int A, int B, int b>
__device__ __forceinline__ void reg_twiddle_rows(double2 (&y)[B][A], int dir) {
    if constexpr (b < B) {
        reg_twiddle_row<R, A, B, b, 1>(y, dir);
        reg_twiddle_rows<R, A, B, b + 1>(y, dir);
    }
}

template <int R>
__device__ __forceinline__ void dft_reg(double2* v, int dir) {
    if constexpr (R == 1) {
    } else if constexpr (R == 2) {
        const double2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 3) {
        const double s = dir < 0 ? -0.86602540378443864676 : 0.86602540378443864676;
        const double2 a = v[0], t = cadd(v[1], v[2]), u = csub(v[1], v[2]);
        const double2 m = cfma(-0.5, t, a);
        v[0] = cadd(a, t);
        v[1] = cmk(fma(-s, u.y, m.x), fma(s, u.x, m.y));  // m + i s u
        v[2] = cmk(fma(s, u.y, m.x), fma(-s, u.x, m.y));
    } else if constexpr (R == 4) {
        const double2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]), t2 = cadd(v[1], v[3]);
        const double2 t3 = rot90(csub(v[1], v[3]), dir);
        v[0] = cadd(t0, t2);
        v[1] = cadd(t1, t3);
        v[2] = csub(t0, t2);
        v[3] = csub(t1, t3);
    } else if constexpr (R == 5) {
        const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
        const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
        const double2 a = v[0], b1 = cadd(v[1], v[4]), b2 = cadd(v[2], v[3]), d1 = csub(v[1], v[4]), d2 = csub(v[2], v[3]);
        const double2 m1 = cfma(c1, b1, cfma(c2, b2, a)), m2 = cfma(c2, b1, cfma(c1, b2, a));
        const double2 n1 = rot90(cfma(s1, d1, cscale(d2, s2)), dir), n2 = rot90(cfma(s2, d1, cscale(d2, -s1)), dir);
        v[0] = cadd(a, cadd(b1, b2));
        v[1] = cadd(m1, n1);
        v[4] = csub(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
    } else if constexpr (R == 7) {
        // cos and sin of 2 pi j / 7
        const double c[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
        const double s[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
        const double2 a = v[0];
        double2 b[3], d[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            b[j] = cadd(v[1 + j], v[6 - j]);
            d[j] = csub(v[1 + j], v[6 - j]);
        }
        v[0] = cadd(a, cadd(b[0], cadd(b[1], b[2])));
#pragma unroll
        for (int q = 1; q <= 3; ++q) {
            double2 m = a, n = czero();
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int t = (q * (j + 1)) % 7, f = t <= 3 ? t : 7 - t;  // fold the angle to 1..3
                const double sn = t <= 3 ? s[f - 1] : -s[f - 1];
                m = cfma(c[f - 1], b[j], m);
                n = j == 0 ? cscale(d[j], sn) : cfma(sn, d[j], n);
            }
            n = rot90(n, dir);
            v[q] = cadd(m, n);
            v[7 - q] = csub(m, n);
        }
    } else if constexpr (R == 8) {
        const double h = 0.70710678118654752440;
        double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        dft_reg<4>(e, dir);
        dft_reg<4>(o, dir);
        const double2 r1 = rot90(o[1], dir), r3 = rot90(o[3], dir);
        o[1] = cscale(cadd(o[1], r1), h);  // exp(dir i pi/4) = (1 + dir i) h
        o[2] = rot90(o[2], dir);
        o[3] = cscale(csub(r3, o[3]), h);  // exp(3 dir i pi/4) = (dir i - 1) h
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = cadd(e[k], o[k]);
            v[k + 4] = csub(e[k], o[k]);
        }
    } else {
        // n = B a + b: DFT_A over a, twiddles, DFT_B over b; X[p + A s]
        constexpr int A = RegSplit<R>::A, B = RegSplit<R>::B;
        static_assert(A * B == R, "radix without a split");
        double2 y[B][A];
#pragma unroll
        for (int b = 0; b < B; ++b) {
#pragma unroll
            for (int a = 0; a < A; ++a) y[b][a] = v[B * a + b];
            dft_reg<A>(y[b], dir);
        }
        reg_twiddle_rows<R, A, B, 1>(y, dir);
#pragma unroll
        for (int p = 0; p < A; ++p) {
            double2 t[B];
#pragma unroll
            for (int b = 0; b < B; ++b) t[b] = y[b][p];
            dft_reg<B>(t, dir);
#pragma unroll
            for (int s = 0; s < B; ++s) v[p + A * s] = t[s];
        }
    }
}

// half-length packing of an even R, M = R/2: Z_k = E + i O with E = g_k + conj
// g_{M-k}, O = (g_k - conj g_{M-k}) exp(2 pi i k / R); Z_{M-k} = conj E + i conj O
template <int R, int K>
__device__ __forceinline__ void c2r_pack(const double2* g, double2* z) {
#pragma clang fp contract(off)
    constexpr int M = R / 2;
    if constexpr (2 * K < M) {
        const double2 a = g[K], b = cconj(g[M - K]);
        const double2 e = cadd(a, b), o = reg_twiddle<R, K>(csub(a, b), +1);
        z[K] = cmk(e.x - o.y, e.y + o.x);
        z[M - K] = cmk(e.x + o.y, o.x - e.y);
        c2r_pack<R, K + 1>(g, z);
    } else if constexpr (2 * K == M) {
        z[K] = cmk(2.0 * g[K].x, -2.0 * g[K].y);
    }
}
// its inverse: g_k = (E - i O) / 2 with E = Z_k + conj Z_{M-k}, O = (Z_k - conj
// Z_{M-k}) exp(-2 pi i k / R); g_{M-k} = conj (E + i O) / 2
template <int R, int K>
__device__ __forceinline__ void r2c_unpack(const double2* z, double2* g) {
#pragma clang fp contract(off)
    constexpr int M = R / 2;
    if constexpr (2 * K < M) {
        const double2 a = z[K], b = cconj(z[M - K]);
        const double2 e = cscale(cadd(a, b), 0.5), o = reg_twiddle<R, K>(cscale(csub(a, b), 0.5), -1);
        g[K] = cmk(e.x + o.y, e.y - o.x);
        g[M - K] = cmk(e.x - o.y, -(e.y + o.x));
        r2c_unpack<R, K + 1>(z, g);
    } else if constexpr (2 * K == M) {
        g[K] = cconj(z[K]);
    }
}

// Real DFTs: x real of length R, g its R/2 + 1 lowest coefficients (the others
// are their conjugates).  Every output is a sum over this one line alone, so
// its error is relative to the line's own size and a zero line stays zero.
// Odd R: cosine and sine sums; even R: the complex transform of half the
// length, even points in the real part and odd points in the imaginary part.

// x_s = sum_k g_k exp(2 pi i k s / R); Im g_0, and Im g_{R/2} of an even R, are ignored
template <int R>
__device__ __forceinline__ void c2r_reg(const double2* g, double* x) {
#pragma clang fp contract(off)
    if constexpr (R == 2) {
        x[0] = g[0].x + g[1].x;
        x[1] = g[0].x - g[1].x;
    } else if constexpr (R % 2 == 1) {
        constexpr int H = R / 2;
        double a[H], b[H];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            a[k] = 2.0 * g[1 + k].x;
            b[k] = 2.0 * g[1 + k].y;
        }
        double t = a[0];
#pragma unroll
        for (int k = 1; k < H; ++k) t += a[k];
        x[0] = g[0].x + t;
#pragma unroll
        for (int s = 1; s <= H; ++s) {
            double m = g[0].x, n = b[0] * RegTwiddle<R>::s[s];
#pragma unroll
            for (int k = 1; k <= H; ++k) m = fma(a[k - 1], RegTwiddle<R>::c[(k * s) % R], m);
#pragma unroll
            for (int k = 2; k <= H; ++k) n = fma(b[k - 1], RegTwiddle<R>::s[(k * s) % R], n);
            x[s] = m - n;
            x[R - s] = m + n;
        }
    } else {
        constexpr int M = R / 2;
        double2 z[M];
        z[0] = cmk(g[0].x + g[M].x, g[0].x - g[M].x);
        c2r_pack<R, 1>(g, z);
        dft_reg<M>(z, +1);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            x[2 * m] = z[m].x;
            x[2 * m + 1] = z[m].y;
        }
    }
}

// g_k = sum_s x_s exp(-2 pi i k s / R), k <= R/2
template <int R>
__device__ __forceinline__ void r2c_reg(const double* x, double2* g) {
#pragma clang fp contract(off)
    if constexpr (R == 2) {
        g[0] = cmk(x[0] + x[1], 0.0);
        g[1] = cmk(x[0] - x[1], 0.0);
    } else if constexpr (R % 2 == 1) {
        constexpr int H = R / 2;
        double e[H], d[H];
#pragma unroll
        for (int s = 0; s < H; ++s) {
            e[s] = x[1 + s] + x[R - 1 - s];
            d[s] = x[R - 1 - s] - x[1 + s];
        }
        double t = e[0];
#pragma unroll
        for (int s = 1; s < H; ++s) t += e[s];
        g[0] = cmk(x[0] + t, 0.0);
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            double m = x[0], n = d[0] * RegTwiddle<R>::s[k];
#pragma unroll
            for (int s = 1; s <= H; ++s) m = fma(e[s - 1], RegTwiddle<R>::c[(k * s) % R], m);
#pragma unroll
            for (int s = 2; s <= H; ++s) n = fma(d[s - 1], RegTwiddle<R>::s[(k * s) % R], n);
            g[k] = cmk(m, n);
        }
    } else {
        constexpr int M = R / 2;
        double2 z[M];
#pragma unroll
        for (int m = 0; m < M; ++m) z[m] = cmk(x[2 * m], x[2 * m + 1]);
        dft_reg<M>(z, -1);
        g[0] = cmk(z[0].x + z[0].y, 0.0);
        g[M] = cmk(z[0].x - z[0].y, 0.0);
        r2c_unpack<R, 1>(z, g);
    }
}

}  // namespace cf
