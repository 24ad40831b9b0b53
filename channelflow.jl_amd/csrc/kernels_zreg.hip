// z passes whose FFT length splits into two register radices (FP64).
//
// N = Nzp = R1 R2.  A block owns KT consecutive x wavenumbers of one y plane of
// one field.  First half: a lane gathers the R1 points z = j + R2 r of one
// column straight from HBM, transforms them in registers, applies the twiddles
// exp(+-2 pi i j q / N) and leaves them in LDS; second half: a lane gathers the
// R2 values of output residue q and writes z = q + R1 p straight to HBM.  Each
// point crosses LDS once (one 16-byte write, one read); the staged multi-pass
// form moved it through LDS once for the load, three times for a length of
// three factors, and once for the store, with a twiddle read beside each pass.
//
// Bound by HBM.  Against the staged passes, us a launch (algorithmic TB/s):
// inverse, 6 fields out, 128x97x128: 48.7 -> 39.2 (4.6); 256x257x256: 549 ->
// 448 (4.2); forward, 3 fields, 26.6 -> 21.7 (4.5) and 246 -> 219 (4.6); the
// largest inverse launch of a 64-instance ensemble 125 -> 39.  A 2 GiB device
// copy reaches 4.9.
#include <algorithm>

#include "cf_kernels.h"
#include "cf_regfft.h"

namespace cf {

// l of the resolved spectrum held at padded position z (ffts.jl:242-293), or
// -1: padding, or the Nyquist row, which is neither read nor written
struct ZMap {
    int npos, neg0, nyq;  // z < npos: l = z; z >= neg0: l = z - neg0 + npos
    __device__ __forceinline__ explicit ZMap(const GridDims& gd) {
        npos = (gd.Nz >> 1) + 1;
        neg0 = gd.Nzp - (gd.Nz - npos);
        nyq = (gd.Nz % 2 == 0) ? gd.Nz / 2 : -1;
    }
    __device__ __forceinline__ int l(int z) const {
        return z < npos ? (z == nyq ? -1 : z) : (z >= neg0 ? z - neg0 + npos : -1);
    }
};

template <int DIR, int R>
__device__ __forceinline__ void z_store(const GridDims& gd, const ZMap& m, double2* out, int q, int step, const double2* v) {
#pragma unroll
    for (int p = 0; p < R; ++p) {
        const int z = q + step * p;
        if constexpr (DIR > 0) {
            out[(unsigned)(gd.ldk * z)] = v[p];
        } else {
            const int l = m.l(z);
            if (l >= 0) out[(unsigned)(gd.Nxh * l)] = v[p];
        }
    }
}

template <int DIR, int R>
__device__ __forceinline__ void z_first(const ZArgs& a, double2* sm, const double2* in, double2* out, bool dz, int KT, int nk) {
    const GridDims& gd = a.gd;
    const ZMap m(gd);
    const int R2 = a.r2, R2p = R2 | 1;
    for (int t = threadIdx.x; t < KT * R2; t += blockDim.x) {
        const int j = (int)fast_div((unsigned)t, a.mul_kt), kk = t - j * KT;
        double2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int z = j + r * R2;
            v[r] = czero();
            if constexpr (DIR > 0) {
                const int l = m.l(z);
                if (l >= 0 && kk < nk) v[r] = in[(unsigned)(gd.Nxh * l) + kk];
            } else {
                if (kk < nk) v[r] = in[(unsigned)(gd.ldk * z) + kk];
            }
        }
        if (DIR > 0 && dz) {  // d/dz: times i beta l
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int l = m.l(j + r * R2);
                v[r] = cmuli(cscale(v[r], gd.beta * (l <= gd.Nz / 2 ? l : l - gd.Nz)));
            }
        }
        dft_reg<R>(v, DIR);
        if (R2 == 1) {  // the whole line in one lane
            if (kk < nk) z_store<DIR, R>(gd, m, out + kk, 0, 1, v);
            continue;
        }
#pragma unroll
        for (int q = 1; q < R; ++q) {
            double2 w = a.plan.tw[j * q];
            if (DIR > 0) w = cconj(w);
            v[q] = cmul(v[q], w);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) sm[(q * R2p + j) * KT + kk] = v[q];
    }
}

template <int DIR, int R>
__device__ __forceinline__ void z_second(const ZArgs& a, const double2* sm, double2* out, int KT, int nk) {
    const ZMap m(a.gd);
    const int R1 = a.r1, R2p = R | 1;
    for (int t = threadIdx.x; t < KT * R1; t += blockDim.x) {
        const int q = (int)fast_div((unsigned)t, a.mul_kt), kk = t - q * KT;
        double2 v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = sm[(q * R2p + j) * KT + kk];
        dft_reg<R>(v, DIR);
        if (kk < nk) z_store<DIR, R>(a.gd, m, out + kk, q, R1, v);
    }
}

template <int DIR, int RMAX>
__device__ __forceinline__ void zreg_body(const ZArgs& a, unsigned lb) {
    extern __shared__ double2 smem_raw[];
    const GridDims& gd = a.gd;
    const int KT = a.KT;
    const unsigned ntiles = (unsigned)((gd.nk + KT - 1) / KT);
    const unsigned tile = lb % ntiles, plane = lb / ntiles;
    const int y = (int)(plane % (unsigned)gd.Ny), f = (int)(plane / (unsigned)gd.Ny);
    const int k0 = (int)tile * KT, nk = gd.nk - k0;  // columns kk < nk exist
    const size_t rin = DIR > 0 ? (size_t)gd.Nxh * gd.Nz : (size_t)gd.ldk * gd.Nzp;
    const size_t rout = DIR > 0 ? (size_t)gd.ldk * gd.Nzp : (size_t)gd.Nxh * gd.Nz;
    const double2* in = a.in[f] + rin * y + k0;
    double2* out = a.out[f] + rout * y + k0;
    const bool dz = (a.dz_mask >> f) & 1u;
#define CF_ZF(R) case R: z_first<DIR, R>(a, smem_raw, in, out, dz, KT, nk); break;
#define CF_ZS(R) case R: z_second<DIR, R>(a, smem_raw, out, KT, nk); break;
    switch (a.r1) {
        CF_ZF(1) CF_ZF(2) CF_ZF(3) CF_ZF(4) CF_ZF(5) CF_ZF(6) CF_ZF(7) CF_ZF(8) CF_ZF(9) CF_ZF(10) CF_ZF(12)
        default:
            if constexpr (RMAX > 12) switch (a.r1) {
                CF_ZF(14) CF_ZF(15) CF_ZF(16)
                default:
                    if constexpr (RMAX > 16) switch (a.r1) { CF_ZF(18) CF_ZF(20) CF_ZF(21) CF_ZF(24) default: break; }
            }
    }
    if (a.r2 == 1) return;  // uniform
    __syncthreads();
    switch (a.r2) {
        CF_ZS(2) CF_ZS(3) CF_ZS(4) CF_ZS(5) CF_ZS(6) CF_ZS(7) CF_ZS(8) CF_ZS(9) CF_ZS(10) CF_ZS(12)
        default:
            if constexpr (RMAX > 12) switch (a.r2) {
                CF_ZS(14) CF_ZS(15) CF_ZS(16)
                default:
                    if constexpr (RMAX > 16) switch (a.r2) { CF_ZS(18) CF_ZS(20) CF_ZS(21) CF_ZS(24) default: break; }
            }
    }
#undef CF_ZF
#undef CF_ZS
}

constexpr int ZRNT = 512;  // largest block
template <int DIR, int RMAX>
__global__ void __launch_bounds__(ZRNT) zreg_kernel(ZArgs a) {
    zreg_body<DIR, RMAX>(a, xcd_logical(blockIdx.x, gridDim.x));
}
// ensemble launch: logical blocks [start[i], start[i+1]) belong to instance i
template <int DIR, int RMAX>
__global__ void __launch_bounds__(ZRNT) zreg_batch_kernel(const ZArgs* __restrict__ tab, const unsigned* __restrict__ start,
                                                          int n) {
    const unsigned lb = xcd_logical(blockIdx.x, gridDim.x);
    const int i = batch_instance(start, n, lb);
    zreg_body<DIR, RMAX>(tab[i], lb - start[i]);
}

// Split of a line: both radices among those built, the larger as small as
// possible (registers), the larger one first (more HBM loads in flight per
// lane); a line of at most 12 points stays in one lane.  0: no split.
bool reg_radix(int r) { return (r >= 1 && r <= 10) || r == 12 || (r >= 14 && r <= 16) || r == 18 || r == 20 || r == 21 || r == 24; }
bool z_reg_split(int n, int* r1, int* r2) {
    *r1 = *r2 = 0;
    if (n <= 12 && reg_radix(n)) {
        *r1 = n;
        *r2 = 1;
        return true;
    }
    for (int r = 2; r <= 24; ++r)  // r: the larger radix
        if (reg_radix(r) && n % r == 0 && n / r <= r && reg_radix(n / r)) {
            *r1 = r;
            *r2 = n / r;
            return true;
        }
    return false;
}
int z_reg_class(const ZArgs& a) { return a.r1 <= 12 ? 12 : (a.r1 <= 16 ? 16 : 24); }
int z_reg_threads(const ZArgs& a) {
    const int t = a.KT * (a.r1 > a.r2 ? a.r1 : a.r2);
    return std::max(64, std::min(ZRNT, (t + 63) / 64 * 64));
}
size_t z_reg_lds(const ZArgs& a) { return a.r2 == 1 ? 0 : (size_t)a.r1 * (a.r2 | 1) * a.KT * sizeof(double2); }

template <int DIR>
static hipError_t launch_zreg_dir(const ZArgs& a, hipStream_t st) {
    const dim3 grid((unsigned)((a.gd.nk + a.KT - 1) / a.KT) * (unsigned)a.gd.Ny * (unsigned)a.nfields), block(z_reg_threads(a));
    const size_t lds = z_reg_lds(a);
#define CF_ZL(RM)                                                                                                        \
    {                                                                                                                    \
        if (lds > 64 * 1024)                                                                                             \
            (void)hipFuncSetAttribute((const void*)zreg_kernel<DIR, RM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        hipLaunchKernelGGL((zreg_kernel<DIR, RM>), grid, block, lds, st, a);                                             \
        return hipGetLastError();                                                                                        \
    }
    const int c = z_reg_class(a);
    if (c == 12) CF_ZL(12)
    if (c == 16) CF_ZL(16)
    CF_ZL(24)
#undef CF_ZL
}
hipError_t launch_zreg(int dir, const ZArgs& a, hipStream_t st) {
    if (a.mixed || !reg_radix(a.r1) || !reg_radix(a.r2) || a.r1 * a.r2 != a.gd.Nzp) return hipErrorInvalidValue;
    return dir > 0 ? launch_zreg_dir<+1>(a, st) : launch_zreg_dir<-1>(a, st);
}

template <int DIR>
static hipError_t launch_zreg_batch_dir(int cls, int nthreads, const ZArgs* tab, const unsigned* start, int n, unsigned nblocks,
                                        size_t lds, hipStream_t st) {
#define CF_ZL(RM)                                                                                                        \
    {                                                                                                                    \
        if (lds > 64 * 1024)                                                                                             \
            (void)hipFuncSetAttribute((const void*)zreg_batch_kernel<DIR, RM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        hipLaunchKernelGGL((zreg_batch_kernel<DIR, RM>), dim3(nblocks), dim3(nthreads), lds, st, tab, start, n);         \
        return hipGetLastError();                                                                                        \
    }
    if (cls == 12) CF_ZL(12)
    if (cls == 16) CF_ZL(16)
    if (cls == 24) CF_ZL(24)
#undef CF_ZL
    return hipErrorInvalidValue;
}
hipError_t launch_zreg_batch(int dir, int cls, int nthreads, const ZArgs* tab, const unsigned* start, int n, unsigned nblocks,
                             size_t lds, hipStream_t st) {
    if (nthreads < 64 || nthreads > ZRNT || nthreads % 64 != 0) return hipErrorInvalidValue;
    return dir > 0 ? launch_zreg_batch_dir<+1>(cls, nthreads, tab, start, n, nblocks, lds, st)
                   : launch_zreg_batch_dir<-1>(cls, nthreads, tab, start, n, nblocks, lds, st);
}

}  // namespace cf
