// x passes whose padded length splits into two register radices (FP64).
//
// N = Nxp = R1 R2.  Two real fields travel as one complex line Z = A + i B of
// length N, which serves odd and even N alike (half-length real transforms need
// an even one).  A block owns NL consecutive (zp, y) lines; a lane holds one
// butterfly of one line:
//   A  gather Z at j + R2 r from HBM (padding is never stored), radix R1,
//      twiddles, LDS                              (lane: pair of fields, line, j)
//   B  radix R2 of every pair at the points q + R1 s; the products of the form
//      at those points in registers; radix R2 of the first forward pass, whose
//      inputs are the same points; twiddles, LDS          (lane: line, q)
//   C  radix R1, then X_k for k < nk              (lane: output line, line, p)
// The points are never stored, and each transform crosses LDS once.
//
// The staged form (a wavefront per line, half-length lines in LDS) issued 243
// 16-byte LDS operations a line, about 60 of its 91 us at 128x97x128 at the
// full LDS rate.  Rotating form, us a launch: 32x33x32 11.3 -> 4.8, 64x65x64
// 33.6 -> 13.7, 128x97x128 91 -> 57.8 (3.0 TB/s), 256x257x256 1030 -> 565 (3.2
// TB/s); 42x49x54, whose odd padded length ran the block-wide pass, 130 -> 7.8;
// convective 80x65x96 74.5 -> 45.8.  Bound by HBM at 128x97x128 and above (a
// device copy takes 35 us for those bytes), with three to six wavefronts a CU.
//
// Radix split: R1 near 2.5 R2 gives the three phases about the same number of
// lanes (3 R2, R1 and 2 R2 of the rotating form), and R2 bounds the registers
// of phase B (three complex lines of R2 points).
#include <algorithm>

#include "cf_kernels.h"
#include "cf_regfft.h"

#ifndef CF_X_PART
#define CF_X_PART 0
#endif

namespace cf {

constexpr int XRNT = 256;  // largest block

// complex lines of phase A (a round) and of phase C.  Plain transforms carry
// one field a line: three fields transformed together and one by one give the
// same bits.
__host__ __device__ constexpr int xr_pairs(int mode, int nf) {
    return mode == X_DIVERGENCE ? 2 : (mode == X_INVERSE ? nf : (mode == X_FORWARD ? 0 : 3));
}
__host__ __device__ constexpr int xr_out(int mode, int nf) {
    return mode == X_DIVERGENCE ? 4 : ((mode == X_INVERSE || mode == X_GRADIENT) ? 0 : (mode == X_FORWARD ? nf : 2));
}
__host__ __device__ constexpr int xr_regions(int mode, int nf) {
    return xr_pairs(mode, nf) > xr_out(mode, nf) ? xr_pairs(mode, nf) : xr_out(mode, nf);
}
// LDS elements of one line and region: rows padded to an odd stride, so lanes
// that read whole rows fall on distinct banks
__host__ __device__ constexpr int xr_slots(int r1, int r2) {
    return r1 * (r2 | 1) > r2 * (r1 | 1) ? r1 * (r2 | 1) : r2 * (r1 | 1);
}

__device__ __forceinline__ double xrfma(double a, double b, double c) { return fma(a, b, c); }

struct XLines {
    const XArgs& a;
    double2* sm;
    int N, nk, NL, slots;
    unsigned ldk;
    long long gl0, nlines;
    __device__ __forceinline__ XLines(const XArgs& a_, double2* s, unsigned block) : a(a_), sm(s) {
        N = a.gd.Nxp;
        nk = a.gd.nk;
        ldk = (unsigned)a.gd.ldk;
        NL = a.nl;
        slots = xr_slots(a.r1, a.r2);
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

// The two real fields of complex line `pair`: workspace fields fa, fb (fb < 0:
// none); da: the x derivative i alpha k of field fa is meant.
// A line's rounding errors are relative to the larger of its two fields, so
// fields of like size share one, and no error exceeds eps |u| |omega| in a
// product: wall-normal derivatives, the largest, go together; V_x, of order one
// with the base flow, goes with a field that it multiplies.
//   rotating    (V_x, Omega_y), (V_y, V_z), (Omega_x, Omega_z)
//   convective, (V_x, d_y V_x), (V_y, V_z), (d_x V_x, d_z V_x),
//   gradient    (d_x V_y, d_z V_y), (d_x V_z, d_z V_z), (d_y V_y, d_y V_z)
//   divergence  (V_x), (V_y, V_z)
template <int MODE>
__device__ __forceinline__ void xr_source(int pair, int& fa, int& fb, bool& da) {
    da = false;
    if constexpr (MODE == X_ROTATIONAL) {
        fa = pair + (pair >> 1);
        fb = pair == 0 ? 4 : 3 * pair - 1;
    } else if constexpr (MODE == X_CONVECTIVE || MODE == X_GRADIENT) {
        fa = (0x421010 >> (4 * pair)) & 15;
        fb = (0x587623 >> (4 * pair)) & 15;
        da = (0x1C >> pair) & 1;
    } else if constexpr (MODE == X_DIVERGENCE) {
        fa = pair;
        fb = pair ? 2 : -1;
    } else {
        fa = pair;
        fb = -1;
    }
}

template <int MODE, int R1, int R2, int ROUND>
__device__ __forceinline__ void xr_gather(const XLines& x, int np) {
    const int t = threadIdx.x;
    const int j = t % R2, u = t / R2;
    const int p = (int)fast_div((unsigned)u, x.a.mul_nl), ln = u - p * x.NL;
    if (p < np && x.valid(ln)) {
        int fa, fb;
        bool da;
        xr_source<MODE>(3 * ROUND + p, fa, fb, da);
        const bool two = fb >= 0;
        const double2* A = x.field(fa, ln);
        const double2* B = x.field(two ? fb : fa, ln);
        const double alpha = x.a.gd.alpha;
        // Rows r < RP hold wavenumbers k = j + R2 r, rows r >= R1 - RP hold
        // k = N - (j + R2 r), the rows between only padding: nk <= N/3 + 1/3,
        // with nk = N/3 exactly where 3 divides N.  Beyond that a k can reach nk
        // only in the outermost row of each side, where its load is clamped and
        // its value dropped; all other loads are unconditional, so they are
        // issued together.
        constexpr int RP = R1 % 3 == 0 ? R1 / 3 : R1 / 3 + 1;
        double2 v[R1];
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            if (r >= RP && r < R1 - RP) {
                v[r] = czero();
                continue;
            }
            const bool neg = r >= R1 - RP;
            const bool edge = neg ? r == R1 - RP : (r == RP - 1 && R1 % 3 != 0);
            const int k0 = neg ? x.N - (j + R2 * r) : j + R2 * r;
            const bool in = !edge || k0 < x.nk;
            const int k = edge ? min(k0, x.nk - 1) : k0;
            double2 ca = A[k], cb = czero();
            if constexpr (MODE != X_INVERSE) cb = B[k];
            if constexpr (MODE == X_CONVECTIVE || MODE == X_GRADIENT) {
                const double s = alpha * k;
                ca = cmk(da ? -(s * ca.y) : ca.x, da ? s * ca.x : ca.y);
            }
            if (r == 0) {  // a real field's mean
                ca.y = k == 0 ? 0.0 : ca.y;
                cb.y = k == 0 ? 0.0 : cb.y;
            }
            if constexpr (MODE == X_DIVERGENCE) cb = cmk(two ? cb.x : 0.0, two ? cb.y : 0.0);
            const double2 z = neg ? cmk(ca.x + cb.y, cb.x - ca.y) : cmk(ca.x - cb.y, ca.y + cb.x);  // conj A + i conj B, A + i B
            v[r] = cmk(in ? z.x : 0.0, in ? z.y : 0.0);
        }
        if constexpr (MODE == X_ROTATIONAL) {
            if (p == 0) {  // B is Omega_y = field 4 - i alpha k V_z
                const double2* V2 = x.field(2, ln);
#pragma unroll
                for (int r = 0; r < R1; ++r) {
                    if (r >= RP && r < R1 - RP) continue;
                    const bool neg = r >= R1 - RP;
                    const bool edge = neg ? r == R1 - RP : (r == RP - 1 && R1 % 3 != 0);
                    const int k0 = neg ? x.N - (j + R2 * r) : j + R2 * r;
                    const int k = edge ? min(k0, x.nk - 1) : k0;
                    const double2 w = V2[k];
                    const double s = !edge || k0 < x.nk ? alpha * k : 0.0;
                    v[r] = cmk(fma(neg ? -s : s, w.x, v[r].x), fma(s, w.y, v[r].y));
                }
            }
        }
        dft_reg<R1>(v, +1);
        double2* d = x.region(p, ln) + j;
        d[0] = v[0];
#pragma unroll
        for (int q = 1; q < R1; ++q) {
            const double2 w = cconj(x.a.twx[j * q]);
            d[q * (R2 | 1)] = cmul(v[q], w);
        }
    }
}

// Output fields of complex line m of phase C; fb < 0: a line of one real field,
// whose X_k are its coefficients as they stand
template <int MODE>
__device__ __forceinline__ void xr_target(int m, int& fa, int& fb) {
    if constexpr (MODE == X_ROTATIONAL) {  // (N_x, N_z), (N_y): V_x Omega_z is of order one
        fa = m;
        fb = m ? -1 : 2;
    } else if constexpr (MODE == X_CONVECTIVE) {  // (N_x, N_y), (N_z)
        fa = 2 * m;
        fb = m ? -1 : 1;
    } else if constexpr (MODE == X_DIVERGENCE) {  // (uv, uw), (vv, vw), (uu), (ww)
        fa = m == 0 ? 1 : (m == 1 ? 3 : (m == 2 ? 0 : 5));
        fb = m == 0 ? 2 : (m == 1 ? 4 : -1);
    } else {
        fa = m;
        fb = -1;
    }
}
// radix R1 of the forward transform: X[p + R2 s] of line m; lines of one field
// are stored at once, the others left in LDS in natural order
template <int MODE, int R1, int R2>
__device__ __forceinline__ void xr_finish(const XLines& x, int nm) {
    const int t = threadIdx.x;
    const int p = t % R2, u = t / R2;
    const int m = (int)fast_div((unsigned)u, x.a.mul_nl), ln = u - m * x.NL;
    const bool on = m < nm && x.valid(ln);
    double2 v[R1];
    double2* d = x.region(on ? m : 0, on ? ln : 0);
    int fa, fb;
    xr_target<MODE>(m, fa, fb);
    if (on) {
#pragma unroll
        for (int q = 0; q < R1; ++q) v[q] = d[p * (R1 | 1) + q];
        dft_reg<R1>(v, -1);
    }
    __syncthreads();
    if (on) {
        if (fb < 0) {
            double2* o = x.out(fa, ln);
#pragma unroll
            for (int s = 0; s < R1; ++s)
                if (p + R2 * s < x.nk) o[p + R2 * s] = v[s];
        } else {
#pragma unroll
            for (int s = 0; s < R1; ++s) d[p + R2 * s] = v[s];
        }
    }
}

// radix R2 of the forward transform of the points q + R1 s, twiddles, LDS
template <int R2>
__device__ __forceinline__ void xr_forward_half(const XLines& x, int m, int ln, int q, double2* z) {
    dft_reg<R2>(z, -1);
    double2* d = x.region(m, ln) + q;
    const int R1p = x.a.r1 | 1;
    d[0] = z[0];
#pragma unroll
    for (int p = 1; p < R2; ++p) d[p * R1p] = cmul(z[p], x.a.twx[q * p]);
}

template <int R2>
__device__ __forceinline__ void xr_inverse_half(const XLines& x, int p, int ln, int q, double2* z) {
    const double2* s = x.region(p, ln) + q * (R2 | 1);
#pragma unroll
    for (int j = 0; j < R2; ++j) z[j] = s[j];
    dft_reg<R2>(z, +1);
}

// radices of phase A and C that the kernel of R2 holds
__host__ __device__ constexpr bool xr_pair(int r1, int r2) { return r1 >= r2 && r1 <= 6 * r2 && r1 <= 24; }

#define CF_XR_SWITCH(X)                                                                                                   \
    switch (a.r1) {                                                                                                       \
        X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16) X(18) X(20) X(21) X(24)                     \
        default: break;                                                                                                   \
    }

template <int MODE, int R2, int RMAX>
__device__ __forceinline__ void xreg_body(const XArgs& a, unsigned block) {
    extern __shared__ double2 smem[];
    XLines x(a, smem, block);
    const int R1 = a.r1, NL = a.nl;
    const int nf = a.nfields, t = threadIdx.x;
    const int np = xr_pairs(MODE, nf), nm = xr_out(MODE, nf);
    const int ln = (int)fast_div((unsigned)t, a.mul_r1), q = t - ln * R1;
    const bool on = ln < NL && x.valid(ln);
#define CF_XG0(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_gather<MODE, R, R2, 0>(x, np); break;
#define CF_XG1(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_gather<MODE, R, R2, 1>(x, np); break;
#define CF_XF(R) case R: if constexpr (xr_pair(R, R2) && (RMAX > 12 ? R > 12 : R <= 12)) xr_finish<MODE, R, R2>(x, nm); break;
    const size_t nphys = (size_t)a.gd.Nxp * a.gd.Nzp * a.gd.Ny;
    const size_t at = (size_t)(x.gl0 + ln) * a.gd.Nxp + q;  // this lane's first point
    if constexpr (MODE != X_FORWARD) {
        CF_XR_SWITCH(CF_XG0)
        __syncthreads();
    }
    if constexpr (MODE == X_ROTATIONAL) {
        double2 m0[R2], m1[R2], m2[R2];
        if (on) {
            xr_inverse_half<R2>(x, 0, ln, q, m0);  // V_x, Omega_y
            xr_inverse_half<R2>(x, 1, ln, q, m1);  // V_y, V_z
            xr_inverse_half<R2>(x, 2, ln, q, m2);  // Omega_x, Omega_z
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                const double u0 = m0[s].x, w1 = m0[s].y, u1 = m1[s].x, u2 = m1[s].y, w0 = m2[s].x, w2 = m2[s].y;
                m0[s] = cmk(xrfma(u1, w2, -(u2 * w1)), xrfma(u0, w1, -(u1 * w0)));
                m1[s] = cmk(xrfma(u2, w0, -(u0 * w2)), 0.0);
            }
        }
        __syncthreads();  // every lane has read the inverse halves
        if (on) {
            xr_forward_half<R2>(x, 0, ln, q, m0);
            xr_forward_half<R2>(x, 1, ln, q, m1);
        }
    } else if constexpr (MODE == X_CONVECTIVE) {
        double u0[R2], u1[R2], u2[R2], n0[R2], n1[R2], n2[R2];
        if (on) {
            double2 m[R2];
            xr_inverse_half<R2>(x, 0, ln, q, m);  // V_x, d_y V_x
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                u0[s] = m[s].x;
                n0[s] = m[s].y;
            }
            xr_inverse_half<R2>(x, 1, ln, q, m);  // V_y, V_z
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                u1[s] = m[s].x;
                u2[s] = m[s].y;
                n0[s] *= u1[s];
            }
            xr_inverse_half<R2>(x, 2, ln, q, m);  // d_x V_x, d_z V_x
#pragma unroll
            for (int s = 0; s < R2; ++s) n0[s] = xrfma(u2[s], m[s].y, xrfma(u0[s], m[s].x, n0[s]));
        }
        __syncthreads();
        CF_XR_SWITCH(CF_XG1)
        __syncthreads();
        if (on) {
            double2 m[R2];
            xr_inverse_half<R2>(x, 0, ln, q, m);  // d_x V_y, d_z V_y
#pragma unroll
            for (int s = 0; s < R2; ++s) n1[s] = xrfma(u2[s], m[s].y, u0[s] * m[s].x);
            xr_inverse_half<R2>(x, 1, ln, q, m);  // d_x V_z, d_z V_z
#pragma unroll
            for (int s = 0; s < R2; ++s) n2[s] = xrfma(u2[s], m[s].y, u0[s] * m[s].x);
            xr_inverse_half<R2>(x, 2, ln, q, m);  // d_y V_y, d_y V_z
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                n1[s] = xrfma(u1[s], m[s].x, n1[s]);
                n2[s] = xrfma(u1[s], m[s].y, n2[s]);
            }
        }
        __syncthreads();
        if (on) {
            double2 m[R2];
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(n0[s], n1[s]);
            xr_forward_half<R2>(x, 0, ln, q, m);
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(n2[s], 0.0);
            xr_forward_half<R2>(x, 1, ln, q, m);
        }
    } else if constexpr (MODE == X_DIVERGENCE) {
        double2 m0[R2], m1[R2];
        if (on) {
            xr_inverse_half<R2>(x, 0, ln, q, m0);  // V_x
            xr_inverse_half<R2>(x, 1, ln, q, m1);  // V_y, V_z
        }
        __syncthreads();
        if (on) {
            double2 m[R2];
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(m0[s].x * m1[s].x, m0[s].x * m1[s].y);
            xr_forward_half<R2>(x, 0, ln, q, m);
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(m1[s].x * m1[s].x, m1[s].x * m1[s].y);
            xr_forward_half<R2>(x, 1, ln, q, m);
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(m0[s].x * m0[s].x, 0.0);
            xr_forward_half<R2>(x, 2, ln, q, m);
#pragma unroll
            for (int s = 0; s < R2; ++s) m[s] = cmk(m1[s].y * m1[s].y, 0.0);
            xr_forward_half<R2>(x, 3, ln, q, m);
        }
    } else if constexpr (MODE == X_INVERSE) {
        if (on) {
            double* o = a.rout[0] + at;
            for (int p = 0; p < np; ++p) {
                double2 m[R2];
                xr_inverse_half<R2>(x, p, ln, q, m);
#pragma unroll
                for (int s = 0; s < R2; ++s) o[p * nphys + R1 * s] = m[s].x;
            }
        }
        return;
    } else if constexpr (MODE == X_GRADIENT) {  // component 3 i + d is dV_i/dx_d
        double* o = a.rout[0] + at;
        auto put = [&](int p, int ca, int cb) {
            double2 m[R2];
            xr_inverse_half<R2>(x, p, ln, q, m);
#pragma unroll
            for (int s = 0; s < R2; ++s) {
                if (ca >= 0) o[ca * nphys + R1 * s] = m[s].x;
                o[cb * nphys + R1 * s] = m[s].y;
            }
        };
        if (on) {
            put(0, -1, 1);
            put(2, 0, 2);
        }
        __syncthreads();
        CF_XR_SWITCH(CF_XG1)
        __syncthreads();
        if (on) {
            put(0, 3, 5);
            put(1, 6, 8);
            put(2, 4, 7);
        }
        return;
    } else {  // X_FORWARD
        if (on) {
            const double* f = a.rin[0] + at;
            for (int c = 0; c < nf; ++c) {
                double2 m[R2];
#pragma unroll
                for (int s = 0; s < R2; ++s) m[s] = cmk(f[c * nphys + R1 * s], 0.0);
                xr_forward_half<R2>(x, c, ln, q, m);
            }
        }
    }
    __syncthreads();
    CF_XR_SWITCH(CF_XF)
    if constexpr (MODE != X_FORWARD) {
        __syncthreads();
        // X_k of the two real fields of Z: A_k = (Z_k + conj Z_{N-k}) / 2, B_k = -i (Z_k - conj Z_{N-k}) / 2
        constexpr int NU = MODE == X_DIVERGENCE ? 2 : 1;  // lines of two fields come first
        for (int i = t; i < NU * NL * x.nk; i += blockDim.x) {
            const int u = (int)fast_div((unsigned)i, a.mul_nk), k = i - u * x.nk;
            const int m = (int)fast_div((unsigned)u, a.mul_nl), l = u - m * NL;
            if (!x.valid(l)) continue;
            int fa, fb;
            xr_target<MODE>(m, fa, fb);
            const double2* z = x.region(m, l);
            const double2 zk = z[k], zm = z[k == 0 ? 0 : x.N - k];
            x.out(fa, l)[k] = cmk(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
            x.out(fb, l)[k] = cmk(0.5 * (zk.y + zm.y), 0.5 * (zm.x - zk.x));
        }
    }
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
        if constexpr (R <= 12)                                                            \
            if (a.r1 <= 12) return xr_launch<MODE, R, 12>(a, lds, st);                    \
        if (a.r1 > 12) return xr_launch<MODE, R, 24>(a, lds, st);                         \
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
        if constexpr (R <= 12)                                                                                             \
            if (rmax <= 12) return xr_launch_batch<MODE, R, 12>(waves, tab, start, n, nblocks, lds, st);                   \
        if (rmax > 12) return xr_launch_batch<MODE, R, 24>(waves, tab, start, n, nblocks, lds, st);                        \
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
static bool xr_r2(int r) { return (r >= 2 && r <= 10) || r == 12 || r == 15 || r == 16; }
bool x_reg_split(int n, int* r1, int* r2) {
    *r1 = *r2 = 0;
    double best = 1e30;
    for (int b = 2; b <= 16; ++b) {
        if (!xr_r2(b) || n % b != 0) continue;
        const int a = n / b;
        if (!reg_radix(a) || !xr_pair(a, b)) continue;
        const double ratio = a > 2.5 * b ? a / (2.5 * b) : 2.5 * b / a;
        if (ratio < best) {
            best = ratio;
            *r1 = a;
            *r2 = b;
        }
    }
    return *r1 > 0;
}
// Lines per block: the busiest phase fills the block's lanes, about 53 KB of
// LDS (three blocks share a CU), and a small problem is cut into enough blocks
// to reach every CU.
void x_reg_shape(XArgs& a) {
    const int lanes = std::max(a.r1, std::max(xr_pairs(a.mode, a.nfields), xr_out(a.mode, a.nfields)) * a.r2);
    const size_t line = (size_t)xr_regions(a.mode, a.nfields) * xr_slots(a.r1, a.r2) * sizeof(double2);
    const long long nlines = (long long)a.gd.Nzp * a.gd.Ny;
    int nl = std::max(1, std::min(XRNT / lanes, (int)(53 * 1024 / line)));
    while (nl > 1 && (nlines + nl - 1) / nl < 512 && nl * lanes > 64) --nl;
    a.nl = nl;
    a.waves = (nl * lanes + 63) / 64;
    a.mul_nl = recip_mul((unsigned)nl);
    a.mul_r1 = recip_mul((unsigned)a.r1);
}
size_t x_reg_lds(const XArgs& a) {
    return (size_t)xr_regions(a.mode, a.nfields) * a.nl * xr_slots(a.r1, a.r2) * sizeof(double2);
}
unsigned x_reg_blocks(const XArgs& a) { return (unsigned)(((long long)a.gd.Nzp * a.gd.Ny + a.nl - 1) / a.nl); }

hipError_t launch_xreg(const XArgs& a, hipStream_t st) {
    const int lanes = std::max(a.r1, std::max(xr_pairs(a.mode, a.nfields), xr_out(a.mode, a.nfields)) * a.r2);
    if (a.mixed || a.r1 * a.r2 != a.gd.Nxp || !reg_radix(a.r1) || !xr_r2(a.r2) || !xr_pair(a.r1, a.r2) || a.nl < 1 ||
        a.nl * lanes > 64 * a.waves || 64 * a.waves > XRNT)
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
