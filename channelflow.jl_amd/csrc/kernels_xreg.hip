// x passes whose padded length splits into two register radices (FP64).
//
// N = Nxp = R1 R2, one real field a line.  The columns j and R2 - j of a line's
// inverse transform are conjugates, and so are the columns p and R2 - p of its
// forward transform, so R2/2 + 1 of them are worked on, for odd and even N
// alike.  A block owns NL consecutive (zp, y) lines; a lane holds one butterfly:
//   A  gather X at j + R2 r from HBM (padding is never stored), radix R1,
//      twiddles, LDS                               (lane: field, line, j <= R2/2)
//   B  real radix R2 of every field at the points q + R1 s; the products of the
//      form at those points in registers; real radix R2 of the products,
//      twiddles, LDS                                             (lane: line, q)
//   C  radix R1, X_k for k < nk to HBM     (lane: output field, line, p <= R2/2)
// The points are never stored, and each transform crosses LDS once.
// No two fields share a transform: an error is relative to its own field and a
// field that is zero stays zero.  (Two fields as one complex line Z = A + i B
// gave each the rounding errors of the larger: N_x 1.80 times as far from its
// value in extended precision as plain FP64 sums, rms over eight states of
// 128x97x128; so 0.97 times.)
//
// The staged form (a wavefront per line, half-length lines in LDS) issued 243
// 16-byte LDS operations a line, about 60 of its 91 us at 128x97x128 at the
// full LDS rate.  Rotating form, us a launch, staged -> here: 32x33x32 11.3 ->
// 4.7, 64x65x64 33.6 -> 13.0, 128x97x128 91 -> 52.2 (3.3 TB/s), 256x257x256
// 1030 -> 566 (3.2 TB/s); 42x49x54, whose odd padded length runs the block-wide
// staged pass, 130 -> 7.0; convective 80x65x96 74.5 -> 33.0.  Bound by HBM at
// 128x97x128 and above (a device copy takes 35 us for those bytes).
#include <algorithm>

#include "cf_kernels.h"
#include "cf_regfft.h"

#ifndef CF_X_PART
#define CF_X_PART 0
#endif

// a product rounds the same way in every kernel that it is inlined into
#pragma clang fp contract(off)

namespace cf {

constexpr int XRNT = 256;  // largest block

// real lines of a round of phase A, of phase C
__host__ __device__ constexpr int xr_in(int mode, int nf) {
    return mode == X_FORWARD ? 0 : (mode == X_INVERSE ? nf : (mode == X_DIVERGENCE ? 3 : 6));
}
__host__ __device__ constexpr int xr_out(int mode, int nf) {
    return mode == X_DIVERGENCE ? 6 : ((mode == X_INVERSE || mode == X_GRADIENT) ? 0 : (mode == X_FORWARD ? nf : 3));
}
__host__ __device__ constexpr int xr_regions(int mode, int nf) {
    return xr_in(mode, nf) > xr_out(mode, nf) ? xr_in(mode, nf) : xr_out(mode, nf);
}
// a line in LDS: R1 rows of the R2/2 + 1 columns, padded to an odd stride, so
// lanes that read whole rows fall on distinct banks
__host__ __device__ constexpr int xr_pitch(int r2) { return (r2 / 2 + 1) | 1; }

// Split N = a b, a = R1 and b = R2: b bounds the registers of phase B (six real
// lines of b points: 192 registers at 16, the largest built), a those of phases
// A and C.  Of the splits with radices built, the one nearest to a = 2 b, where
// the lanes of the phases (3 b + 6, a and 1.5 b + 3 of the rotating form) are
// closest; of two as near, the one with a <= 12, whose kernel needs about half
// the registers, else the larger a.  Steps of Nx x 33 x 96, us, rotating and
// convective: N = 96 as 16 x 6 218 and 242, as 12 x 8 213 and 225; 108 as 18 x 6
// 223 and 256, as 12 x 9 218 and 232; 192 as 24 x 8 261 and 295, as 16 x 12 260
// and 302; 216 as 24 x 9 271 and 308, as 18 x 12 275 and 323.
__host__ __device__ constexpr bool xr_r1(int r) {
    return (r >= 2 && r <= 10) || r == 12 || (r >= 14 && r <= 16) || r == 18 || r == 20 || r == 21 || r == 24;
}
__host__ __device__ constexpr bool xr_r2(int r) { return (r >= 2 && r <= 10) || r == 12 || r == 15 || r == 16; }
__host__ __device__ constexpr int xr_split(int n) {  // R2, 0: none
    int best = 0;
    for (int b = 2; b <= 16; ++b) {
        const int a = n / b;
        if (n % b != 0 || !xr_r2(b) || !xr_r1(a) || a < b || a > 6 * b) continue;
        if (!best) {
            best = b;
            continue;
        }
        // max(a / 2 b, 2 b / a) of both, cross-multiplied
        const int a0 = n / best;
        const long long nu = a > 2 * b ? a : 2 * b, de = a > 2 * b ? 2 * b : a;
        const long long nu0 = a0 > 2 * best ? a0 : 2 * best, de0 = a0 > 2 * best ? 2 * best : a0;
        if (nu * de0 < nu0 * de || (nu * de0 == nu0 * de && a <= 12 && a0 > 12)) best = b;
    }
    return best;
}
// the pairs that some length is split into, and the kernel classes (R2, R1 up
// to 12 or 24) that hold one
__host__ __device__ constexpr bool xr_pair(int r1, int r2) { return xr_r1(r1) && xr_split(r1 * r2) == r2; }
__host__ __device__ constexpr bool xr_class(int r2, int rmax) {
    for (int r1 = rmax > 12 ? 13 : 2; r1 <= rmax; ++r1)
        if (xr_pair(r1, r2)) return true;
    return false;
}

// rows of R1 that hold wavenumbers on one side of the padding (xr_gather)
__host__ __device__ constexpr int xr_rows(int r1) { return r1 % 3 == 0 ? r1 / 3 : r1 / 3 + 1; }

__device__ __forceinline__ double xrfma(double a, double b, double c) { return fma(a, b, c); }

struct XLines {
    const XArgs& a;
    double2* sm;
    int nk, NL, slots;
    unsigned ldk;
    long long gl0, nlines;
    __device__ __forceinline__ XLines(const XArgs& a_, double2* s, unsigned block) : a(a_), sm(s) {
        nk = a.gd.nk;
        ldk = (unsigned)a.gd.ldk;
        NL = a.nl;
        slots = a.r1 * xr_pitch(a.r2);
        gl0 = (long long)block * NL;
        nlines = (long long)a.gd.Nzp * a.gd.Ny;
    }
    __device__ __forceinline__ bool valid(int ln) const { return gl0 + ln < nlines; }
    __device__ __forceinline__ double2* region(int p, int ln) const { return sm + (p * NL + ln) * slots; }
    // line ln of workspace field f
    __device__ __forceinline__ const double2* field(int f, int ln) const {
        return a.in[0] + (size_t)a.gd.Sz * f + (size_t)(gl0 + ln) * ldk;
    }
    __device__ __forceinline__ double2* out(int f, int ln) const {
        return a.out[0] + (size_t)a.gd.Sz * f + (size_t)(gl0 + ln) * ldk;
    }
};

// Line p of a round: workspace field f; dx: its x derivative i alpha k is meant.
//   convective  V_x V_y V_z and the derivatives of V_x, then those of V_y, V_z
//   gradient    the derivatives of V_x and V_y, then those of V_z
template <int MODE, int ROUND>
__device__ __forceinline__ void xr_source(int p, int& f, bool& dx) {
    f = p;
    dx = false;
    if constexpr (MODE == X_CONVECTIVE || MODE == X_GRADIENT) {
        constexpr unsigned F = ROUND ? (MODE == X_GRADIENT ? 0x852u : 0x852741u) : (MODE == X_GRADIENT ? 0x741630u : 0x630210u);
        constexpr unsigned D = ROUND ? (MODE == X_GRADIENT ? 0x1u : 0x9u) : (MODE == X_GRADIENT ? 0x9u : 0x8u);
        f = (F >> (4 * p)) & 15;
        dx = (D >> p) & 1;
    }
}

template <int MODE, int R1, int R2, int ROUND>
__device__ __forceinline__ void xr_gather(const XLines& x, int np) {
    constexpr int H1 = R2 / 2 + 1;
    const int t = threadIdx.x;
    const int j = t % H1, u = t / H1;
    const int p = (int)fast_div((unsigned)u, x.a.mul_nl), ln = u - p * x.NL;
    if (p < np && x.valid(ln)) {
        int f;
        bool dx;
        xr_source<MODE, ROUND>(p, f, dx);
        const double2* A = x.field(f, ln);
        const double alpha = x.a.gd.alpha;
        // Rows r < RP hold wavenumbers k = j + R2 r, rows r >= R1 - RP hold
        // k = N - (j + R2 r), the rows between only padding: nk <= N/3 + 1/3,
        // with nk = N/3 exactly where 3 divides N.  Beyond that a k can reach nk
        // only in the outermost row of each side, where its load is clamped and
        // its value dropped; all other loads are unconditional, so they are
        // issued together.
        constexpr int RP = xr_rows(R1);
        double2 v[R1];
        auto wave = [&](int r, bool& in) {  // k of row r
            const bool neg = r >= R1 - RP, edge = neg ? r == R1 - RP : (r == RP - 1 && R1 % 3 != 0);
            const int k = neg ? R2 - j + R2 * (R1 - 1 - r) : j + R2 * r;
            in = !edge || k < x.nk;
            return edge ? min(k, x.nk - 1) : k;
        };
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            if (r >= RP && r < R1 - RP) {
                v[r] = czero();
                continue;
            }
            bool in;
            const int k = wave(r, in);
            double2 c = A[k];
            if constexpr (MODE == X_CONVECTIVE || MODE == X_GRADIENT) {
                const double s = alpha * k;
                c = cmk(dx ? -(s * c.y) : c.x, dx ? s * c.x : c.y);
            }
            if (r == 0) c.y = k == 0 ? 0.0 : c.y;  // a real field's mean
            v[r] = cmk(in ? c.x : 0.0, in ? (r >= R1 - RP ? -c.y : c.y) : 0.0);
        }
        if constexpr (MODE == X_ROTATIONAL) {
            if (p == 4) {  // Omega_y = field 4 - i alpha k V_z
                const double2* V2 = x.field(2, ln);
#pragma unroll
                for (int r = 0; r < R1; ++r) {
                    if (r >= RP && r < R1 - RP) continue;
                    bool in;
                    const int k = wave(r, in);
                    const double2 w = V2[k];
                    const double s = in ? alpha * k : 0.0;
                    v[r] = cmk(fma(s, w.y, v[r].x), fma(r >= R1 - RP ? s : -s, w.x, v[r].y));
                }
            }
        }
        dft_reg<R1>(v, +1);
        double2* d = x.region(p, ln) + j;
        d[0] = v[0];
#pragma unroll
        for (int q = 1; q < R1; ++q) d[q * xr_pitch(R2)] = cmul(v[q], cconj(x.a.twx[j * q]));
    }
}

// Radix R1 of the forward transform: X[p + R2 s] of output field m.  Of a
// column that has a mirror, the rows past the padding are the mirror's low ones.
template <int MODE, int R1, int R2>
__device__ __forceinline__ void xr_finish(const XLines& x, int nm) {
    constexpr int H1 = R2 / 2 + 1, RP = xr_rows(R1);
    const int t = threadIdx.x;
    const int p = t % H1, u = t / H1;
    const int m = (int)fast_div((unsigned)u, x.a.mul_nl), ln = u - m * x.NL;
    if (m >= nm || !x.valid(ln)) return;
    const double2* d = x.region(m, ln) + p;
    double2 v[R1];
#pragma unroll
    for (int q = 0; q < R1; ++q) v[q] = d[q * xr_pitch(R2)];
    dft_reg<R1>(v, -1);
    double2* o = x.out(m, ln) + p;
    double2* om = x.out(m, ln) + (R2 - p);
    const bool mirror = p != 0 && 2 * p != R2;
#pragma unroll
    for (int s = 0; s < RP; ++s)
        if (s < RP - 1 || R1 % 3 == 0 || p + R2 * s < x.nk) o[R2 * s] = v[s];
#pragma unroll
    for (int s = 0; s < RP; ++s)
        if (mirror && (s < RP - 1 || R1 % 3 == 0 || R2 - p + R2 * s < x.nk)) om[R2 * s] = cconj(v[R1 - 1 - s]);
}

// real radix R2 of one field at the points q + R1 s
template <int R2>
__device__ __forceinline__ void xr_inverse_half(const XLines& x, int p, int ln, int q, double* u) {
    const double2* d = x.region(p, ln) + q * xr_pitch(R2);
    double2 g[R2 / 2 + 1];
#pragma unroll
    for (int j = 0; j <= R2 / 2; ++j) g[j] = d[j];
    c2r_reg<R2>(g, u);
}

// real radix R2 of the forward transform of the points q + R1 s, twiddles, LDS
template <int R2>
__device__ __forceinline__ void xr_forward_half(const XLines& x, int m, int ln, int q, const double* u) {
    double2 g[R2 / 2 + 1];
    r2c_reg<R2>(u, g);
    double2* d = x.region(m, ln) + q * xr_pitch(R2);
    d[0] = g[0];
#pragma unroll
    for (int p = 1; p <= R2 / 2; ++p) d[p] = cmul(g[p], x.a.twx[q * p]);
}

#define CF_XR_SWITCH(X)                                                                                                   \
    switch (a.r1) {                                                                                                       \
        X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16) X(18) X(20) X(21) X(24)                     \
        default: break;                                                                                                   \
    }

// Between the gathers and the finish a lane reads and writes only its own rows
// (line, q) of the regions, so phase B needs no barrier of its own.
template <int MODE, int R2, int RMAX>
__device__ __forceinline__ void xreg_body(const XArgs& a, unsigned block) {
    extern __shared__ double2 smem[];
    XLines x(a, smem, block);
    const int R1 = a.r1, NL = a.nl;
    const int nf = a.nfields, t = threadIdx.x;
    const int np = xr_in(MODE, nf), nm = xr_out(MODE, nf);
    const int ln = (int)fast_div((unsigned)t, a.mul_r1), q = t - ln * R1;
    const bool on = ln < NL && x.valid(ln);
#define CF_XG0(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_gather<MODE, R, R2, 0>(x, np); break;
#define CF_XG1(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_gather<MODE, R, R2, 1>(x, MODE == X_GRADIENT ? 3 : np); break;
#define CF_XF(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_finish<MODE, R, R2>(x, nm); break;
    const size_t nphys = (size_t)a.gd.Nxp * a.gd.Nzp * a.gd.Ny;
    const size_t at = (size_t)(x.gl0 + ln) * a.gd.Nxp + q;  // this lane's first point
    if constexpr (MODE != X_FORWARD) {
        CF_XR_SWITCH(CF_XG0)
        __syncthreads();
    }
    if constexpr (MODE == X_ROTATIONAL) {
        if (on) {
            double u0[R2], u1[R2], u2[R2], w0[R2], w1[R2], w2[R2];
            xr_inverse_half<R2>(x, 0, ln, q, u0);
            xr_inverse_half<R2>(x, 1, ln, q, u1);
            xr_inverse_half<R2>(x, 2, ln, q, u2);
            xr_inverse_half<R2>(x, 3, ln, q, w0);
            xr_inverse_half<R2>(x, 4, ln, q, w1);
            xr_inverse_half<R2>(x, 5, ln, q, w2);
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                const double n0 = xrfma(u1[s], w2[s], -(u2[s] * w1[s]));
                const double n1 = xrfma(u2[s], w0[s], -(u0[s] * w2[s]));
                const double n2 = xrfma(u0[s], w1[s], -(u1[s] * w0[s]));
                u0[s] = n0;
                u1[s] = n1;
                u2[s] = n2;
            }
            xr_forward_half<R2>(x, 0, ln, q, u0);
            xr_forward_half<R2>(x, 1, ln, q, u1);
            xr_forward_half<R2>(x, 2, ln, q, u2);
        }
    } else if constexpr (MODE == X_CONVECTIVE) {
        double u0[R2], u1[R2], u2[R2], n0[R2];
        // (V . grad) of the component whose derivatives are lines p, p + 1, p + 2
        auto advect = [&](int p, double* n) {
            double d[R2];
            xr_inverse_half<R2>(x, p + 1, ln, q, d);
#pragma unroll
            for (int s = 0; s < R2; ++s) n[s] = u1[s] * d[s];
            xr_inverse_half<R2>(x, p, ln, q, d);
#pragma unroll
            for (int s = 0; s < R2; ++s) n[s] = xrfma(u0[s], d[s], n[s]);
            xr_inverse_half<R2>(x, p + 2, ln, q, d);
#pragma unroll
            for (int s = 0; s < R2; ++s) n[s] = xrfma(u2[s], d[s], n[s]);
        };
        if (on) {
            xr_inverse_half<R2>(x, 0, ln, q, u0);
            xr_inverse_half<R2>(x, 1, ln, q, u1);
            xr_inverse_half<R2>(x, 2, ln, q, u2);
            advect(3, n0);
        }
        __syncthreads();  // every lane has read its rows
        CF_XR_SWITCH(CF_XG1)
        __syncthreads();
        if (on) {
            double n1[R2], n2[R2];
            advect(0, n1);
            advect(3, n2);
            xr_forward_half<R2>(x, 0, ln, q, n0);
            xr_forward_half<R2>(x, 1, ln, q, n1);
            xr_forward_half<R2>(x, 2, ln, q, n2);
        }
    } else if constexpr (MODE == X_DIVERGENCE) {
        if (on) {
            double u[3][R2];
#pragma unroll
            for (int c = 0; c < 3; ++c) xr_inverse_half<R2>(x, c, ln, q, u[c]);
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = i; j < 3; ++j) {  // uu, uv, uw, vv, vw, ww
                    double n[R2];
#pragma unroll
                    for (int s = 0; s < R2; ++s) n[s] = u[i][s] * u[j][s];
                    xr_forward_half<R2>(x, i == 0 ? j : i + j + 1, ln, q, n);
                }
        }
    } else if constexpr (MODE == X_INVERSE) {
        if (on) {
            double* o = a.rout[0] + at;
            for (int p = 0; p < np; ++p) {
                double u[R2];
                xr_inverse_half<R2>(x, p, ln, q, u);
#pragma unroll
                for (int s = 0; s < R2; ++s) o[p * nphys + R1 * s] = u[s];
            }
        }
        return;
    } else if constexpr (MODE == X_GRADIENT) {  // component 3 i + d is dV_i/dx_d
        double* o = a.rout[0] + at;
        auto put = [&](int p, int c) {
            double u[R2];
            xr_inverse_half<R2>(x, p, ln, q, u);
#pragma unroll
            for (int s = 0; s < R2; ++s) o[c * nphys + R1 * s] = u[s];
        };
        if (on)
            for (int c = 0; c < 6; ++c) put(c, c);
        __syncthreads();
        CF_XR_SWITCH(CF_XG1)
        __syncthreads();
        if (on)
            for (int c = 0; c < 3; ++c) put(c, 6 + c);
        return;
    } else {  // X_FORWARD
        if (on) {
            const double* f = a.rin[0] + at;
            for (int c = 0; c < nf; ++c) {
                double u[R2];
#pragma unroll
                for (int s = 0; s < R2; ++s) u[s] = f[c * nphys + R1 * s];
                xr_forward_half<R2>(x, c, ln, q, u);
            }
        }
    }
    __syncthreads();
    CF_XR_SWITCH(CF_XF)
#undef CF_XG0
#undef CF_XG1
#undef CF_XF
}

// waves per SIMD that the registers must leave room for: the convective
// products keep the velocity and one component beside a gather of R1 points
__host__ __device__ constexpr int xr_waves(int mode, int r2, int rmax) {
    return (mode == X_CONVECTIVE && (r2 > 8 || rmax > 12)) ? 1 : 2;
}

template <int MODE, int R2, int RMAX>
__global__ void __launch_bounds__(XRNT) __attribute__((amdgpu_waves_per_eu(xr_waves(MODE, R2, RMAX)))) xreg_kernel(XArgs a) {
    xreg_body<MODE, R2, RMAX>(a, xcd_logical(blockIdx.x, gridDim.x));
}
template <int MODE, int R2, int RMAX>
__global__ void __launch_bounds__(XRNT) __attribute__((amdgpu_waves_per_eu(xr_waves(MODE, R2, RMAX))))
xreg_batch_kernel(const XArgs* __restrict__ tab, const unsigned* __restrict__ start, int n) {
    const int i = batch_instance(start, n, blockIdx.x);
    xreg_body<MODE, R2, RMAX>(tab[i], blockIdx.x - start[i]);
}

template <int MODE, int R2, int RMAX>
static hipError_t xr_launch(const XArgs& a, size_t lds, hipStream_t st) {
    const long long nlines = (long long)a.gd.Nzp * a.gd.Ny;
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute((const void*)xreg_kernel<MODE, R2, RMAX>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((xreg_kernel<MODE, R2, RMAX>), dim3((unsigned)((nlines + a.nl - 1) / a.nl)), dim3(a.waves * 64), lds, st, a);
    return hipGetLastError();
}
template <int MODE, int R2, int RMAX>
static hipError_t xr_launch_batch(int waves, const XArgs* tab, const unsigned* start, int n, unsigned nblocks, size_t lds,
                                  hipStream_t st) {
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute((const void*)xreg_batch_kernel<MODE, R2, RMAX>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((xreg_batch_kernel<MODE, R2, RMAX>), dim3(nblocks), dim3(waves * 64), lds, st, tab, start, n);
    return hipGetLastError();
}

// one translation unit per form
#define CF_XR_R2(X)                                                                       \
    X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(15) X(16)
template <int MODE>
hipError_t launch_xreg_mode(const XArgs& a, size_t lds, hipStream_t st);
template <int MODE>
hipError_t launch_xreg_batch_mode(int r2, int rmax, int waves, const XArgs* tab, const unsigned* start, int n, unsigned nblocks,
                                  size_t lds, hipStream_t st);
#if CF_X_PART != 0
template <int MODE>
hipError_t launch_xreg_mode(const XArgs& a, size_t lds, hipStream_t st) {
#define CF_XR1(R)                                                                         \
    if (a.r2 == R) {                                                                      \
        if constexpr (xr_class(R, 12))                                                    \
            if (a.r1 <= 12) return xr_launch<MODE, R, 12>(a, lds, st);                    \
        if constexpr (xr_class(R, 24))                                                    \
            if (a.r1 > 12) return xr_launch<MODE, R, 24>(a, lds, st);                     \
    }
    CF_XR_R2(CF_XR1)
#undef CF_XR1
    return hipErrorInvalidValue;
}
template <int MODE>
hipError_t launch_xreg_batch_mode(int r2, int rmax, int waves, const XArgs* tab, const unsigned* start, int n, unsigned nblocks,
                                  size_t lds, hipStream_t st) {
#define CF_XR1(R)                                                                                                          \
    if (r2 == R) {                                                                                                         \
        if constexpr (xr_class(R, 12))                                                                                     \
            if (rmax <= 12) return xr_launch_batch<MODE, R, 12>(waves, tab, start, n, nblocks, lds, st);                   \
        if constexpr (xr_class(R, 24))                                                                                     \
            if (rmax > 12) return xr_launch_batch<MODE, R, 24>(waves, tab, start, n, nblocks, lds, st);                    \
    }
    CF_XR_R2(CF_XR1)
#undef CF_XR1
    return hipErrorInvalidValue;
}
#endif
#if CF_X_PART == 1
template hipError_t launch_xreg_mode<X_ROTATIONAL>(const XArgs&, size_t, hipStream_t);
#elif CF_X_PART == 2
template hipError_t launch_xreg_batch_mode<X_ROTATIONAL>(int, int, int, const XArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_X_PART == 3
template hipError_t launch_xreg_mode<X_CONVECTIVE>(const XArgs&, size_t, hipStream_t);
#elif CF_X_PART == 4
template hipError_t launch_xreg_batch_mode<X_CONVECTIVE>(int, int, int, const XArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_X_PART == 5
template hipError_t launch_xreg_mode<X_DIVERGENCE>(const XArgs&, size_t, hipStream_t);
#elif CF_X_PART == 6
template hipError_t launch_xreg_mode<X_GRADIENT>(const XArgs&, size_t, hipStream_t);
#elif CF_X_PART == 7
template hipError_t launch_xreg_mode<X_INVERSE>(const XArgs&, size_t, hipStream_t);
template hipError_t launch_xreg_mode<X_FORWARD>(const XArgs&, size_t, hipStream_t);
#endif

#if CF_X_PART == 0
bool x_reg_split(int n, int* r1, int* r2) {
    *r2 = xr_split(n);
    *r1 = *r2 ? n / *r2 : 0;
    return *r2 > 0;
}
// lanes of the busiest phase, a line
static int xr_lanes(const XArgs& a) { return std::max(a.r1, xr_regions(a.mode, a.nfields) * (a.r2 / 2 + 1)); }
// Lines per block: the busiest phase fills the block's lanes, about 53 KB of
// LDS (three blocks share a CU), and a small problem is cut into enough blocks
// to reach every CU.
void x_reg_shape(XArgs& a) {
    const int lanes = xr_lanes(a);
    const size_t line = (size_t)xr_regions(a.mode, a.nfields) * a.r1 * xr_pitch(a.r2) * sizeof(double2);
    const long long nlines = (long long)a.gd.Nzp * a.gd.Ny;
    int nl = std::max(1, std::min(XRNT / lanes, (int)(53 * 1024 / line)));
    while (nl > 1 && (nlines + nl - 1) / nl < 512 && nl * lanes > 64) --nl;
    a.nl = nl;
    a.waves = (nl * lanes + 63) / 64;
    a.mul_nl = recip_mul((unsigned)nl);
    a.mul_r1 = recip_mul((unsigned)a.r1);
}
size_t x_reg_lds(const XArgs& a) {
    return (size_t)xr_regions(a.mode, a.nfields) * a.nl * a.r1 * xr_pitch(a.r2) * sizeof(double2);
}
unsigned x_reg_blocks(const XArgs& a) { return (unsigned)(((long long)a.gd.Nzp * a.gd.Ny + a.nl - 1) / a.nl); }

hipError_t launch_xreg(const XArgs& a, hipStream_t st) {
    if (a.mixed || a.r1 * a.r2 != a.gd.Nxp || !xr_r1(a.r1) || !xr_r2(a.r2) || !xr_pair(a.r1, a.r2) || a.nl < 1 ||
        a.nl * xr_lanes(a) > 64 * a.waves || 64 * a.waves > XRNT)
        return hipErrorInvalidValue;
    const size_t lds = x_reg_lds(a);
    switch (a.mode) {
        case X_ROTATIONAL: return launch_xreg_mode<X_ROTATIONAL>(a, lds, st);
        case X_CONVECTIVE: return launch_xreg_mode<X_CONVECTIVE>(a, lds, st);
        case X_DIVERGENCE: return launch_xreg_mode<X_DIVERGENCE>(a, lds, st);
        case X_GRADIENT: return launch_xreg_mode<X_GRADIENT>(a, lds, st);
        case X_INVERSE: return a.nfields <= 3 ? launch_xreg_mode<X_INVERSE>(a, lds, st) : hipErrorInvalidValue;
        case X_FORWARD: return a.nfields <= 3 ? launch_xreg_mode<X_FORWARD>(a, lds, st) : hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_xreg_batch(int mode, int r2, int rmax, int waves, const XArgs* tab, const unsigned* start, int n,
                             unsigned nblocks, size_t lds, hipStream_t st) {
    if (waves < 1 || 64 * waves > XRNT) return hipErrorInvalidValue;
    if (mode == X_ROTATIONAL) return launch_xreg_batch_mode<X_ROTATIONAL>(r2, rmax, waves, tab, start, n, nblocks, lds, st);
    if (mode == X_CONVECTIVE) return launch_xreg_batch_mode<X_CONVECTIVE>(r2, rmax, waves, tab, start, n, nblocks, lds, st);
    return hipErrorInvalidValue;
}
#endif

}  // namespace cf
