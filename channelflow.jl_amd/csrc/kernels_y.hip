// Wall-normal (Chebyshev) pencil kernels.
//
// A block owns M = NT/L consecutive Fourier modes s = ix + Nxh*iz of the
// reference (k,l,n) layout; a group of L lanes owns one mode, lane t holding
// Chebyshev coefficients n = Kt..Kt+K-1 in registers (K = 4, or 6 / 8 when
// Ny exceeds 256 / 384).  HBM rows (fixed n, M
// consecutive modes) are moved through LDS, which also stages the DCT-I
// (REDFT00) as a length-2P Stockham FFT of the even extension.
//
// Reference: CNRK2 stage (src/timesteppers/cnrk2.jl:170-205), Stokes solve
// (src/solvers/stokes.jl:81-108, batchedinfluence.jl:129-159, meanmode.jl:103-150),
// Chebyshev transforms (src/ffts.jl:65-82,151-166, transforms/chebyshev.jl:45-66),
// curl (src/fields/operators.jl:172-190), pressure (src/pressure.jl:196-285).
#include <type_traits>

#include "cf_device.h"
#include "cf_kernels.h"
#include "cf_regfft.h"

// This file is compiled as several translation units so that the layouts
// build in parallel: part 0 (this file on its own) holds the dispatchers and
// the reduction kernels, parts 1-7 (kernels_y_p<n>.hip) each instantiate the
// kernels of some (L, K) layouts; the list is at the end of the file.
#ifndef CF_Y_PART
#define CF_Y_PART 0
#endif

namespace cf {

constexpr int YNT = 256;  // threads per block of every y kernel

struct ModeInfo {
    long long s;
    int ix, iz, l;
    double kx, kz, kappa2;
    bool valid, nyq, mean;
};

__device__ __forceinline__ ModeInfo mode_info(const GridDims& gd, long long s) {
    ModeInfo mi;
    mi.s = s;
    mi.valid = s < gd.B;
    const unsigned ss = mi.valid ? (unsigned)s : 0u;  // B = Nxh*Nz < 2^31
    mi.iz = (int)(ss / (unsigned)gd.Nxh);
    mi.ix = (int)ss - mi.iz * gd.Nxh;
    mi.l = mi.iz <= (gd.Nz >> 1) ? mi.iz : mi.iz - gd.Nz;
    mi.kx = gd.alpha * mi.ix;
    mi.kz = gd.beta * mi.l;
    mi.kappa2 = mi.kx * mi.kx + mi.kz * mi.kz;
    mi.nyq = ((gd.Nx % 2 == 0) && mi.ix == gd.Nx / 2) || ((gd.Nz % 2 == 0) && mi.iz == gd.Nz / 2);
    mi.mean = (ss == 0);
    return mi;
}

// Radices of the register DCT (Tile::dct_*_reg) built for a layout: those that
// split the lengths 2P its Ny range holds, as few as cover the 7-smooth P (the
// largest one sets the kernel's registers).  The layouts without any (K = 8,
// and K = 6 on 32 lanes) keep the staged transforms.
__host__ __device__ constexpr bool y_radix(int L, int K, int r) {
    if (K == 6) return L == 64 && (r == 16 || r == 18 || r == 20 || r == 21 || r == 24 || r == 32);
    if (K != 4) return false;
    if (L == 4) return r >= 2 && r <= 7;
    if (L == 8) return r >= 3 && r <= 10;
    if (L == 16) return (r >= 6 && r <= 10) || r == 12 || r == 14;
    if (L == 32) return (r >= 8 && r <= 10) || r == 12 || (r >= 14 && r <= 16) || r == 18 || r == 20;
    return r == 12 || (r >= 14 && r <= 16) || r == 18 || r == 20 || r == 21 || r == 24;
}
template <int L, int K>
constexpr bool y_has_reg() { return K == 4 || (K == 6 && L == 64); }

// f(radix r as a compile-time constant)
template <int L, int K, int R = 2, typename F>
__device__ __forceinline__ void with_radix(int r, F&& f) {
    if constexpr (R <= 32) {
        if constexpr (y_radix(L, K, R)) {
            if (r == R) {
                f(std::integral_constant<int, R>{});
                return;
            }
        }
        with_radix<L, K, R + 1>(r, f);
    }
}

// LDS slots (double2) of the per-degree table: CHEB_TAB_ARRAYS arrays of K L doubles
template <int L, int K>
__host__ __device__ constexpr int y_table_slots() { return CHEB_TAB_ARRAYS * K * L / 2; }

// ---------------------------------------------------------------------------
// Per-wavefront tile.  Wave w of block b owns the W = 64/L consecutive modes
// starting at b*M + w*W, and a private LDS region holding two FFT lines per
// mode (the DCT-I staging) that also serves as the solve's stash.  Spectral
// rows move between HBM and the group registers directly (lane t of a mode
// reads/writes degrees Kt..Kt+K-1; the W modes of one row are contiguous), so
// no block-level barrier is needed anywhere after the twiddle table load.
// ---------------------------------------------------------------------------
template <int L, int K>
struct Tile {
    static constexpr int M = YNT / L;  // modes per block
    static constexpr int W = 64 / L;   // modes per wavefront
    const GridDims& gd;
    long long s, sw0;  // this group's mode, the wave's first mode
    int lane, mw, ld;
    double2 *bufA, *bufB, *stash, *lines;  // lines: the block's regions as one
    unsigned blk;                          // block index
    const double2* tw;
    // region: LDS slots per wave (y_region_slots); smem starts with the
    // twiddle table of the DCT plan (ntw entries) and the per-degree table
    // (y_table_slots<L>), see load_tables
    const double* tab;
    // block: this block's index within its launch (or within its instance
    // of a batched ensemble launch)
    __device__ __forceinline__ Tile(const GridDims& g_, double2* smem, int ntw, int ld_, int region, unsigned block)
        : gd(g_), ld(ld_) {
        const int tid = threadIdx.x, wave = tid >> 6;
        lane = tid & 63;
        mw = lane / L;
        sw0 = (long long)block * M + wave * W;
        s = sw0 + mw;
        tw = smem;
        tab = reinterpret_cast<const double*>(smem + ntw);
        bufA = smem + ntw + y_table_slots<L, K>() + (size_t)wave * region;
        bufB = bufA + W * ld;
        stash = bufA + mw * 3 * K * L;
        lines = smem + ntw + y_table_slots<L, K>();
        blk = block;
    }
    // Non-Nyquist-first order (YOrder): the wave's first slot sw0 becomes a
    // mode index.  W divides nxr, so the wave's W slots lie in one z row and
    // its modes stay consecutive; a wave past the last non-Nyquist mode is
    // empty (modes >= B: zero loads, no stores).
    __device__ __forceinline__ void order_modes(long long nreg, int nxr, int zskip) {
        if (sw0 >= nreg) {
            sw0 = gd.B;
        } else {
            const unsigned q = (unsigned)sw0 / (unsigned)nxr;
            const int iz = (int)q + ((int)q >= zskip ? 1 : 0);
            sw0 = (long long)iz * gd.Nxh + ((unsigned)sw0 - q * (unsigned)nxr);
        }
        s = sw0 + mw;
    }
    __device__ __forceinline__ void order_modes(const YOrder& o) { order_modes(o.nreg, o.nxr, o.zskip); }
    // spectral field column of this group's mode (zero beyond P / absent mode)
    __device__ __forceinline__ CVec<K> load(const double2* __restrict__ src, const Group<L, K>& g) const {
        CVec<K> v;
        const bool ok = s < gd.B;
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            v.v[e] = (ok && n < gd.Ny) ? src[s + gd.B * n] : czero();
        }
        return v;
    }
    // load of a column that this lane may have stored before (no forwarding of
    // the stored registers: the index is opaque)
    __device__ __forceinline__ CVec<K> reload(const double2* src, const Group<L, K>& g) const {
        CVec<K> v;
        long long i = s + gd.B * (K * g.t);
        asm volatile("" : "+v"(i));
#pragma unroll
        for (int e = 0; e < K; ++e) v.v[e] = (s < gd.B && K * g.t + e < gd.Ny) ? src[i + gd.B * e] : czero();
        return v;
    }
    __device__ __forceinline__ void store(double2* __restrict__ dst, const Group<L, K>& g, const CVec<K>& v) const {
        const bool ok = s < gd.B;
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (ok && n < gd.Ny) dst[s + gd.B * n] = v.v[e];
        }
    }
    // forward Chebyshev transform of y-physical rows (values at y_j, j=0..P):
    // REDFT00, times norm, endpoint 1/2, Nyquist modes zeroed (normalize_forward!).
    // SC: storage of the rows (double2, or float2 widened on load); the
    // transform itself runs in FP64.
    template <typename SC>
    __device__ __forceinline__ CVec<K> dct_forward(const SC* __restrict__ src, const FFTPlan& plan, double norm,
                                                const Group<L, K>& g, bool zero_mode) {
        const int P = gd.P;
        // YLOADS rows' HBM loads in flight before their LDS stores
        constexpr int YLOADS = 4;
        for (int base = lane; base < (P + 1) * W; base += YLOADS * 64) {
            SC r[YLOADS];
#pragma unroll
            for (int b = 0; b < YLOADS; ++b) {
                const int idx = base + b * 64;
                const int n = idx / W, m = idx - n * W;
                const long long sm = sw0 + m;
                r[b] = (idx < (P + 1) * W && sm < gd.B) ? src[sm + gd.B * n] : from_c64<SC>(czero());
            }
#pragma unroll
            for (int b = 0; b < YLOADS; ++b) {
                const int idx = base + b * 64;
                if (idx < (P + 1) * W) {
                    const int n = idx / W, m = idx - n * W;
                    const double2 v = to_c64(r[b]);
                    bufA[m * ld + n] = v;
                    if (n >= 1 && n <= P - 1) bufA[m * ld + 2 * P - n] = v;
                }
            }
        }
        wave_sync();
        double2* res = lds_fft<true, true>(bufA, bufB, plan, tw, W, ld, -1, lane, 64);
        CVec<K> v;
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            double w = (n == 0 || n == P) ? 0.5 * norm : norm;
            v.v[e] = (n <= P && !zero_mode) ? cscale(res[mw * ld + n], w) : czero();
        }
        wave_sync();
        return v;
    }
    // inverse: coefficient registers -> values at y_j (endpoints doubled,
    // REDFT00, x1/2: InverseFFT!'s chebyshev + copy_to_padded! scale).
    // Computed in FP64; SC = float2 rounds the stored values.  INPLACE: one
    // LDS line per mode, transformed in place (8 points per lane).
    template <typename SC, bool INPLACE = false>
    __device__ __forceinline__ void dct_inverse(SC* __restrict__ dst, const FFTPlan& plan, const Group<L, K>& g,
                                                const CVec<K>& a) {
        const int P = gd.P;
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n <= P) {
                double2 x = a.v[e];
                bufA[mw * ld + n] = (n == 0 || n == P) ? cscale(x, 2.0) : x;
                if (n >= 1 && n <= P - 1) bufA[mw * ld + 2 * P - n] = x;
            }
        }
        wave_sync();
        double2* res = bufA;
        if constexpr (INPLACE) lds_fft_inplace<8, true>(bufA, plan, tw, W, ld, -1, lane, 64);
        else res = lds_fft<true, true>(bufA, bufB, plan, tw, W, ld, -1, lane, 64);
        for (int idx = lane; idx < (P + 1) * W; idx += 64) {
            int n = idx / W, m = idx - n * W;
            long long sm = sw0 + m;
            if (sm < gd.B) dst[sm + gd.B * n] = from_c64<SC>(cscale(res[m * ld + n], 0.5));
        }
        wave_sync();
    }

    // ---- DCT-I in two register radices, several fields a pass -------------
    // The even extension has length N = 2P = r1 r2.  Its columns j + r2 r and
    // (r2 - j) + r2 r mirror each other, and so do its output rows q + r1 p and
    // (r1 - q) + r1 p: r2/2 + 1 columns and r1/2 + 1 rows are transformed, half
    // of a length-2P transform.  First half: a lane holds one column of one
    // mode and field, transforms it and leaves it twiddled in LDS, for its
    // mirror column too (row pitch r2|1); second half: a lane gathers one row.
    // One exchange through LDS instead of one per factor.  Bound by the issue of
    // FP64 and LDS instructions beside the solves' scans; against the staged
    // form, us a step: 32x33x32 186 -> 148, 64x65x64 282 -> 245, 128x97x128 824
    // -> 787, 256x257x256 12550 -> 11865, 64-instance ensemble 1429 -> 1340.
    // nf fields travel together so that the columns and rows fill the lanes: at
    // Ny = 97 (12 x 16, two modes a wavefront) one field has 18 columns and 14
    // rows, three have 54 and 42.
    // SHARE: with one mode a wavefront (L = 64) the block's four modes share the
    // work, neighbouring lanes holding neighbouring modes: 64 contiguous bytes a
    // row where a wavefront on its own touches 16, and the address units bound
    // it (256x257x256 step 12.37 -> 11.87 ms).  With two modes and more the
    // block's barriers cost as much as that gains (32x33x32 step 148 us on
    // wavefronts, 158 on blocks; 128x97x128 783 and 785).
    static constexpr bool SHARE = L == 64;
    static constexpr int RM = SHARE ? M : W;  // modes that share lines
    static __device__ __forceinline__ void reg_sync() {
        if constexpr (SHARE) __syncthreads();
        else wave_sync();
    }
    struct RegItem {
        int f, m, c;  // field within the pass, mode of the RM sharing lines, column or row
        bool on;
    };
    __device__ __forceinline__ RegItem reg_item(int per, int nf) const {
        // opaque to the optimiser: the addresses of every radix built would
        // otherwise be hoisted out of the loop over the passes (registers)
        int ln = SHARE ? (int)threadIdx.x : lane;
        asm volatile("" : "+v"(ln));
        const int rest = ln / RM;
        RegItem it;
        it.m = ln - rest * RM;
        it.f = (rest >= per) + (rest >= 2 * per);
        it.c = rest - it.f * per;
        it.on = rest < per * nf;
        return it;
    }
    // mode of slot m of those sharing lines (>= B: none)
    __device__ __forceinline__ long long reg_mode(const YArgs& a, int m) const {
        if constexpr (!SHARE) return sw0 + m;
        const unsigned slot = blk * M + m;
        if (!a.order.on) return slot;
        if (slot >= (unsigned)a.order.nreg) return gd.B;
        const unsigned q = slot / (unsigned)a.order.nxr;
        return (long long)(q + (q >= (unsigned)a.order.zskip ? 1u : 0u)) * gd.Nxh + (slot - q * (unsigned)a.order.nxr);
    }
    __device__ __forceinline__ int line_slot() const { return SHARE ? (int)threadIdx.x / L : mw; }  // this group's m
    __device__ __forceinline__ double2* reg_line(const YArgs& a, int f, int m) const {
        return (SHARE ? lines : bufA) + (f * RM + m) * a.zs;
    }
    // twiddled column of R points -> LDS, and its mirror column
    template <int R>
    __device__ __forceinline__ void reg_column(const YArgs& a, const RegItem& it, double2* z, double2* v) const {
        const int r2 = a.r2, pitch = r2 | 1, c = it.c, mc = r2 - c;
        const bool mir = c > 0 && c != mc;
        dft_reg<R>(v, -1);
        if (!it.on) return;
        z[c] = v[0];
        if (mir) z[mc] = v[0];
#pragma unroll
        for (int q = 1; q <= R / 2; ++q) {
            const double2 w = tw[c * q];
            z[q * pitch + c] = cmul(v[q], w);
            if (mir) z[q * pitch + mc] = cmul(v[R - q], cconj(w));
        }
    }
    template <int R>
    __device__ __forceinline__ void reg_row(const YArgs& a, const RegItem& it, const double2* z, double2* v) const {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = it.on ? z[it.c * (a.r2 | 1) + j] : czero();
        dft_reg<R>(v, -1);
    }
    // output p of row q: its degree, or -1 (a mirrored duplicate)
    __device__ __forceinline__ int reg_out(const YArgs& a, const RegItem& it, int p) const {
        const int k = it.c + a.r1 * p;
        if (k <= gd.P) return it.on ? k : -1;
        return (it.on && it.c != 0 && 2 * it.c != a.r1) ? 2 * gd.P - k : -1;
    }
    // three y-physical fields -> unscaled coefficients in the LDS lines
    // reg_line(a, c, m) (row n at slot n)
    template <typename SC>
    __device__ __forceinline__ void dct_forward_reg(const YArgs& a, const SC* s0, const SC* s1, const SC* s2) {
        const int P = gd.P, r1 = a.r1, r2 = a.r2, nf = a.nf;
#pragma unroll 1
        for (int base = 0; base < 3; base += nf) {
            const int cnt = 3 - base < nf ? 3 - base : nf;
            {
                const RegItem it = reg_item(r2 / 2 + 1, cnt);
                const int f = base + it.f;
                const long long sm = reg_mode(a, it.m);
                const SC* src = (f == 0 ? s0 : (f == 1 ? s1 : s2)) + sm;
                const bool ok = it.on && sm < gd.B;
                double2* z = reg_line(a, f, it.m);
                with_radix<L, K>(r1, [&](auto rc) {
                    constexpr int R = decltype(rc)::value;
                    SC raw[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int k = it.c + r2 * r, n = k <= P ? k : 2 * P - k;
                        raw[r] = ok ? src[gd.B * n] : from_c64<SC>(czero());
                    }
                    double2 v[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) v[r] = to_c64(raw[r]);
                    reg_column<R>(a, it, z, v);
                });
            }
            reg_sync();
            {
                const RegItem it = reg_item(r1 / 2 + 1, cnt);
                double2* z = reg_line(a, base + it.f, it.m);
                with_radix<L, K>(r2, [&](auto rc) {
                    constexpr int R = decltype(rc)::value;
                    double2 v[R];
                    reg_row<R>(a, it, z, v);
                    reg_sync();  // every row is read: the lines are reused
#pragma unroll
                    for (int p = 0; p < R; ++p) {
                        const int n = reg_out(a, it, p);
                        if (n >= 0) z[n] = v[p];
                    }
                });
            }
            reg_sync();
        }
    }
    // fields get(i) (coefficients, i < nfields) -> values at the Lobatto points
    // in dst(i)
    template <typename SC, typename GetF, typename Dst>
    __device__ __forceinline__ void dct_inverse_reg(const YArgs& a, const Group<L, K>& g, int nfields, GetF get, Dst dst) {
        const int P = gd.P, r1 = a.r1, r2 = a.r2, nf = a.nf;
#pragma unroll 1
        for (int base = 0; base < nfields; base += nf) {
            const int cnt = nfields - base < nf ? nfields - base : nf;
#pragma unroll 1
            for (int i = 0; i < cnt; ++i) {
                const CVec<K> x = get(base + i);
                double2* z = reg_line(a, i, line_slot());
#pragma unroll
                for (int e = 0; e < K; ++e) {
                    const int n = K * g.t + e;
                    if (n <= P) z[n] = (n == 0 || n == P) ? cscale(x.v[e], 2.0) : x.v[e];
                }
            }
            reg_sync();
            {
                const RegItem it = reg_item(r2 / 2 + 1, cnt);
                double2* z = reg_line(a, it.f, it.m);
                with_radix<L, K>(r1, [&](auto rc) {
                    constexpr int R = decltype(rc)::value;
                    double2 v[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int k = it.c + r2 * r, n = k <= P ? k : 2 * P - k;
                        v[r] = it.on ? z[n] : czero();
                    }
                    reg_sync();  // every column is read: the lines are reused
                    reg_column<R>(a, it, z, v);
                });
            }
            reg_sync();
            {
                const RegItem it = reg_item(r1 / 2 + 1, cnt);
                double2* z = reg_line(a, it.f, it.m);
                SC* d0 = dst(base);
                SC* d1 = dst(base + 1);
                SC* d2 = dst(base + 2);
                const long long sm = reg_mode(a, it.m);
                SC* d = (it.f == 0 ? d0 : (it.f == 1 ? d1 : d2)) + sm;
                const bool ok = sm < gd.B;
                with_radix<L, K>(r2, [&](auto rc) {
                    constexpr int R = decltype(rc)::value;
                    double2 v[R];
                    reg_row<R>(a, it, z, v);
#pragma unroll
                    for (int p = 0; p < R; ++p) {
                        const int n = reg_out(a, it, p);
                        if (ok && n >= 0) d[gd.B * n] = from_c64<SC>(cscale(v[p], 0.5));
                    }
                });
            }
            reg_sync();
        }
    }
};

// LDS slots of one wave's region: two FFT lines per mode, or the solve's
// stash of three coefficient vectors (K L slots each) per mode.
template <int L, int K>
__host__ __device__ constexpr int y_region_slots(int ld) {
    return (2 * (64 / L) * ld > 3 * K * 64) ? 2 * (64 / L) * ld : 3 * K * 64;
}

// the register DCT's region: `fields` lines per mode, or the stash
template <int L, int K>
__host__ __device__ constexpr int y_reg_slots(int fields, int zs) {
    return (fields * (64 / L) * zs > 3 * K * 64) ? fields * (64 / L) * zs : 3 * K * 64;
}

// Block prologue of every y kernel: the DCT twiddle table and the
// per-degree table into LDS.
template <int L, int K>
__device__ __forceinline__ void load_tables(double2* smem, const YArgs& a) {
    for (int i = threadIdx.x; i < a.dct.n; i += YNT) smem[i] = a.dct.tw[i];
    double* tab = reinterpret_cast<double*>(smem + a.dct.n);
    constexpr int NT = K * L;
    for (int i = threadIdx.x; i < CHEB_TAB_ARRAYS * NT; i += YNT) {
        const int arr = i / NT, n = i - arr * NT;
        tab[i] = a.cheb_tab[arr * a.ntab + n];
    }
    __syncthreads();
}

// Lane-private LDS stash of a coefficient vector (each lane writes and reads
// back only its own four slots, so no barrier is needed between the two).
template <int L, int K>
__device__ __forceinline__ void stash(double2* slot, const Group<L, K>& g, const CVec<K>& v) {
#pragma unroll
    for (int e = 0; e < K; ++e) slot[K * g.t + e] = v.v[e];
}
template <int L, int K>
__device__ __forceinline__ CVec<K> unstash(const double2* slot, const Group<L, K>& g) {
    CVec<K> v;
#pragma unroll
    for (int e = 0; e < K; ++e) v.v[e] = slot[K * g.t + e];
    return v;
}

// coefficient of degree n (broadcast to the group)
template <int L, int K>
__device__ __forceinline__ double2 coef_at(const Group<L, K>& g, const CVec<K>& a, int n) {
    double2 v = czero();
#pragma unroll
    for (int e = 0; e < K; ++e)
        if (K * g.t + e == n) v = a.v[e];
    return g.sum(v);
}

template <int L, int K>
__device__ __forceinline__ void load_fac(const double* __restrict__ f, long long s, int Ny, const Group<L, K>& g,
                                         double out[K]) {
#pragma unroll
    for (int e = 0; e < K; ++e) {
        int n = K * g.t + e;
        out[e] = (n < Ny) ? f[s * Ny + n] : 0.0;
    }
}

// Total velocity V = U + Ub e_x at (0,0) and the y-physical fields each
// nonlinear form needs, at the Lobatto points, into out6:
//   rotating   V, Omega_x, Omega_z of Omega = curl V (nonlinear.jl:173-193,
//              operators.jl:172-190); out6[4] is not written: Omega_y =
//              dV_x/dz - dV_z/dx is formed by the periodic passes (the z
//              inverse emits i beta l V_x from V_x into z field 4, the x pass
//              subtracts i alpha k V_z), one Chebyshev transform fewer
//   convective V, dV/dy            (nonlinear.jl:113-140; x and z derivatives
//                                   are formed by the periodic passes)
//   divergence V                   (nonlinear.jl:146-167)
// get(c) returns U component c: from registers in the stage kernel, from HBM
// in the prologue (loaded where first needed, which shortens live ranges).
template <int L, int K, typename SC, bool INPLACE = false, typename GetU>
__device__ __forceinline__ void inverse_six(Tile<L, K>& tile, const YArgs& a, const Group<L, K>& g, const ModeInfo& mi,
                                            GetU get) {
    SC* out6[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) out6[i] = reinterpret_cast<SC*>(a.out6[i]);
    CVec<K> V0 = get(0);
    if (mi.mean && mi.valid) {
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n < a.gd.Ny) V0.v[e] = cadd(V0.v[e], cmk(a.base[n], 0.0));
        }
    }
    if (a.form != FORM_ROTATING) {
        tile.template dct_inverse<SC, INPLACE>(out6[0], a.dct, g, V0);
        if (a.form == FORM_CONVECTIVE) tile.template dct_inverse<SC, INPLACE>(out6[3], a.dct, g, cheb_deriv(g, V0));
        const CVec<K> V1 = get(1);
        tile.template dct_inverse<SC, INPLACE>(out6[1], a.dct, g, V1);
        if (a.form == FORM_CONVECTIVE) tile.template dct_inverse<SC, INPLACE>(out6[4], a.dct, g, cheb_deriv(g, V1));
        const CVec<K> V2 = get(2);
        tile.template dct_inverse<SC, INPLACE>(out6[2], a.dct, g, V2);
        if (a.form == FORM_CONVECTIVE) tile.template dct_inverse<SC, INPLACE>(out6[5], a.dct, g, cheb_deriv(g, V2));
        return;
    }
    // order chosen so each velocity component dies as early as possible
    const CVec<K> V1 = get(1);
    CVec<K> W;
    tile.template dct_inverse<SC, INPLACE>(out6[0], a.dct, g, V0);
    {
        CVec<K> d1 = cheb_deriv(g, V0);
#pragma unroll
        for (int e = 0; e < K; ++e) W.v[e] = csub(cmuli(cscale(V1.v[e], mi.kx)), d1.v[e]);  // i k V2 - dy V1
    }
    tile.template dct_inverse<SC, INPLACE>(out6[5], a.dct, g, W);
    const CVec<K> V2 = get(2);
    tile.template dct_inverse<SC, INPLACE>(out6[2], a.dct, g, V2);
    {
        CVec<K> d3 = cheb_deriv(g, V2);
#pragma unroll
        for (int e = 0; e < K; ++e) W.v[e] = csub(d3.v[e], cmuli(cscale(V1.v[e], mi.kz)));  // dy V3 - i l V2
    }
    tile.template dct_inverse<SC, INPLACE>(out6[3], a.dct, g, W);
    tile.template dct_inverse<SC, INPLACE>(out6[1], a.dct, g, V1);
}

// inverse_six with the register DCT: the form's fields in passes of a.nf.  The
// velocity is read back from a.U for every field (a stage has just stored it:
// L2), not held in registers across the transforms.
template <int L, int K, typename SC>
__device__ __forceinline__ void inverse_six_reg(Tile<L, K>& tile, const YArgs& a, const Group<L, K>& g, const ModeInfo& mi) {
    const int form = a.form;
    const int nfields = form == FORM_ROTATING ? 5 : (form == FORM_CONVECTIVE ? 6 : 3);
    // field i of the sequence: rotating V0, Omega_z, V2, Omega_x, V1;
    // convective V0, dV0, V1, dV1, V2, dV2; divergence V0, V1, V2
    auto get = [&](int i) {
        const int c = form == FORM_DIVERGENCE ? i : (form == FORM_CONVECTIVE ? i >> 1 : (i < 2 ? 0 : (i < 4 ? 2 : 1)));
        CVec<K> x = tile.reload(c == 0 ? a.U[0] : (c == 1 ? a.U[1] : a.U[2]), g);
        if (c == 0 && mi.mean && mi.valid) {
#pragma unroll
            for (int e = 0; e < K; ++e) {
                const int n = K * g.t + e;
                if (n < a.gd.Ny) x.v[e] = cadd(x.v[e], cmk(a.base[n], 0.0));
            }
        }
        if (form == FORM_DIVERGENCE || !(i & 1)) return x;
        x = cheb_deriv(g, x);
        if (form == FORM_ROTATING) {
            const CVec<K> v1 = tile.reload(a.U[1], g);
#pragma unroll
            for (int e = 0; e < K; ++e) {
                const double2 d = x.v[e];
                x.v[e] = i == 1 ? csub(cmuli(cscale(v1.v[e], mi.kx)), d)   // i k V2 - dy V1
                                : csub(d, cmuli(cscale(v1.v[e], mi.kz)));  // dy V3 - i l V2
            }
        }
        return x;
    };
    auto dst = [&](int i) {
        const int slot = form == FORM_DIVERGENCE ? i
                         : form == FORM_CONVECTIVE ? (i >> 1) + 3 * (i & 1)
                                                   : (i == 1 ? 5 : (i == 4 ? 1 : i));
        double2* d = a.out6[0];
        if (slot == 1) d = a.out6[1];
        if (slot == 2) d = a.out6[2];
        if (slot == 3) d = a.out6[3];
        if (slot == 4) d = a.out6[4];
        if (slot == 5) d = a.out6[5];
        return reinterpret_cast<SC*>(d);
    };
    tile.template dct_inverse_reg<SC>(a, g, nfields, get, dst);
}

// ---------------------------------------------------------------------------
// Stokes solve of one mode given R (re-solve form of the influence + tau
// correction; see the derivation in the library documentation).  Returns
// U[3], P.  mean/nyq modes handled separately by the caller.
// ---------------------------------------------------------------------------
template <int L, int K>
__device__ __forceinline__ void solve_nonzero(const Group<L, K>& g, const YArgs& a, const Bank& bk, const ModeInfo& mi,
                                              const double2* Rs0, const double2* Rs1, const double2* Rs2,
                                              CVec<K> Uout[3], CVec<K>& Pout) {
    const int P = a.gd.P, Ny = a.gd.Ny;
    const double* mc = bk.mconst + mi.s * MC_COUNT;
    const double shift = bk.lambda + bk.nu * mi.kappa2;
    double fp[K], fv[K];
    load_fac(a.facP, mi.s, Ny, g, fp);
    // r = D Ry + i k Rx + i l Rz
    CVec<K> r;
    {
        CVec<K> R1 = unstash(Rs1, g);
        r = cheb_deriv(g, R1);
        CVec<K> R0 = unstash(Rs0, g), R2 = unstash(Rs2, g);
#pragma unroll
        for (int e = 0; e < K; ++e)
            r.v[e] = cadd(r.v[e], cadd(cmuli(cscale(R0.v[e], mi.kx)), cmuli(cscale(R2.v[e], mi.kz))));
    }
    double2 p1P, v1a, v1b, bp, bm;
    {
        CVec<K> p1 = helm_solve(g, P, mi.kappa2, fp, false, r, czero(), czero());
        p1P = coef_at(g, p1, P);
        CVec<K> q = cheb_deriv(g, p1);
        CVec<K> R1 = unstash(Rs1, g);
#pragma unroll
        for (int e = 0; e < K; ++e) q.v[e] = csub(q.v[e], R1.v[e]);
        load_fac(bk.facV, mi.s, Ny, g, fv);
        CVec<K> v1 = helm_solve(g, P, shift, fv, false, q, czero(), czero());
        bp = cscale(wall_deriv_plus(g, v1), -1.0);
        bm = cscale(wall_deriv_minus(g, v1), -1.0);
        v1a = coef_at(g, v1, P - 1);
        v1b = coef_at(g, v1, P);
    }
    double2 dp = cadd(cscale(bp, mc[MC_A11]), cscale(bm, mc[MC_A12]));
    double2 dm = cadd(cscale(bp, mc[MC_A21]), cscale(bm, mc[MC_A22]));
    double2 ra, rb;
    {
        CVec<K> R1 = unstash(Rs1, g);
        ra = coef_at(g, R1, P - 1);
        rb = coef_at(g, R1, P);
    }
    double2 p2P = cadd(p1P, cadd(cscale(dp, mc[MC_PPT]), cscale(dm, mc[MC_PMT])));
    double2 v2a = cadd(v1a, cadd(cscale(dp, mc[MC_VP1]), cscale(dm, mc[MC_VM1])));
    double2 v2b = cadd(v1b, cadd(cscale(dp, mc[MC_VP0]), cscale(dm, mc[MC_VM0])));
    double2 s1 = cscale(csub(cadd(cscale(v2a, shift), cscale(p2P, 2.0 * P)), ra), 1.0 / (1.0 - mc[MC_SIG1]));
    double2 s2 = cscale(csub(cscale(v2b, shift), rb), 1.0 / (1.0 - mc[MC_SIG2]));
    // final pressure: rhs r + s1 D T_{P-1} + s2 D T_P, wall data per parity
#pragma unroll
    for (int e = 0; e < K; ++e) {
        int n = K * g.t + e;
        if (n % 2 == 0) {
            if (n < P - 1) r.v[e] = cfma(n == 0 ? (double)(P - 1) : 2.0 * (P - 1), s1, r.v[e]);
        } else {
            if (n < P) r.v[e] = cfma(2.0 * P, s2, r.v[e]);
        }
    }
    double2 de = cadd(cscale(cadd(dp, dm), 0.5), cscale(s1, 0.5 * (mc[MC_D0P] + mc[MC_D0M])));
    double2 dd = cadd(cscale(csub(dp, dm), 0.5), cscale(s2, 0.5 * (mc[MC_D0P] - mc[MC_D0M])));
    Pout = helm_solve(g, P, mi.kappa2, fp, false, r, de, dd);
    __builtin_amdgcn_sched_barrier(0);
    // the three velocity solves share the operator: one fused solve
    CVec<K> q[3];
    {
        const CVec<K> R0 = unstash(Rs0, g), R2 = unstash(Rs2, g);
#pragma unroll
        for (int e = 0; e < K; ++e) {
            q[0].v[e] = csub(cmuli(cscale(Pout.v[e], mi.kx)), R0.v[e]);
            q[2].v[e] = csub(cmuli(cscale(Pout.v[e], mi.kz)), R2.v[e]);
        }
    }
    q[1] = cheb_deriv(g, Pout);
    {
        const CVec<K> R1 = unstash(Rs1, g);
#pragma unroll
        for (int e = 0; e < K; ++e) q[1].v[e] = csub(q[1].v[e], R1.v[e]);
    }
    const double2 zero3[3] = {czero(), czero(), czero()};
    helm_solve_n<3>(g, P, shift, fv, false, q, zero3, zero3, Uout);
}

// mean mode (meanmode.jl:103-150); returns the new gradients
template <int L, int K>
__device__ __forceinline__ void solve_mean(const Group<L, K>& g, const YArgs& a, const Bank& bk, const double2* Rs0,
                                           const double2* Rs1, const double2* Rs2, CVec<K> Uout[3], CVec<K>& Pout,
                                           double gout[2]) {
    const int P = a.gd.P, Ny = a.gd.Ny;
    const CVec<K> R[3] = {unstash(Rs0, g), unstash(Rs1, g), unstash(Rs2, g)};
    // pressure: integrate Ry through degree P-1, zero bulk mean
    {
        double2 prev3 = g.up1(R[1].v[K - 1]);
        double2 next0 = g.down1(R[1].v[0]);
        CVec<K> r = R[1];
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            double2 rm = (e == 0) ? prev3 : r.v[e - 1];  // r_{n-1}
            double2 rp = (e == K - 1) ? next0 : r.v[e + 1];  // r_{n+1}
            double2 lower = (n == 1) ? rm : cscale(rm, 0.5);
            double2 upper = (n + 1 < P) ? cscale(rp, 0.5) : czero();
            Pout.v[e] = (n >= 1 && n <= P) ? cscale(csub(lower, upper), 1.0 / n) : czero();
        }
        double2 m = bulk_mean(g, Pout);  // p_0 = 0 at this point
        if (g.t == 0) Pout.v[0] = cscale(m, -1.0);
    }
#pragma unroll
    for (int e = 0; e < K; ++e) Uout[1].v[e] = czero();
    double fv[K];
    load_fac(bk.facV, 0, Ny, g, fv);
    for (int c = 0; c < 2; ++c) {
        const CVec<K>& src = R[c == 0 ? 0 : 2];
        CVec<K> f;
#pragma unroll
        for (int e = 0; e < K; ++e) f.v[e] = cscale(src.v[e], -1.0);
        CVec<K> u = helm_solve(g, P, bk.lambda, fv, false, f, czero(), czero());
        double grad;
        if (a.bulk) {
            double target = c == 0 ? a.c0 : a.c1;
            grad = (target - bulk_mean(g, u).x) / bk.resp_mean;
        } else {
            grad = c == 0 ? a.c0 : a.c1;
        }
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n < Ny) u.v[e] = cadd(u.v[e], cmk(grad * bk.resp[n], 0.0));
        }
        Uout[c == 0 ? 0 : 2] = u;
        gout[c] = grad;
    }
}

template <int L, int K>
__device__ __forceinline__ void zero_vec(CVec<K>& v) {
#pragma unroll
    for (int e = 0; e < K; ++e) v.v[e] = czero();
}

// Laplacian D^2 a - kappa^2 a
template <int L, int K>
__device__ __forceinline__ CVec<K> laplacian(const Group<L, K>& g, const CVec<K>& a, double kappa2) {
    CVec<K> d = cheb_deriv(g, cheb_deriv(g, a));
#pragma unroll
    for (int e = 0; e < K; ++e) d.v[e] = cfma(-kappa2, a.v[e], d.v[e]);
    return d;
}

// ---------------------------------------------------------------------------
// Full CNRK2 stage: forward DCT of the nonlinear term, Q update, RHS,
// Stokes solve, state write, inverse transforms for the next stage.
// ---------------------------------------------------------------------------
// SC: storage of the y-physical fields (double2; float2 in the mixed step).
// REG: the DCTs run in two register radices (a.r1, a.r2), all three nonlinear
// terms first (their coefficients wait in the LDS lines).
template <int L, int K, typename SC, bool REG>
__device__ __forceinline__ void ystage_body(const YArgs& a, unsigned block) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, REG ? y_reg_slots<L, K>(3, a.zs) : y_region_slots<L, K>(a.ld), block);
    if (a.order.on) tile.order_modes(a.order);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    const int Ny = a.gd.Ny;
    const bool meanmode = mi.mean && mi.valid;

    // Per component: forward DCT of the nonlinear term, Q = N (stage 1) or
    // A_j Q + N, R_c = lambda U_c + nu Lap U_c - d_c P + (B_j/C_j) Q_c.
    double gold0 = a.c0, gold1 = a.c1;
    if constexpr (REG) {
        if (!a.Ncoef[0])  // the three terms come in one form
            tile.dct_forward_reg(a, reinterpret_cast<const SC*>(a.Nphys[0]), reinterpret_cast<const SC*>(a.Nphys[1]),
                                 reinterpret_cast<const SC*>(a.Nphys[2]));
    }
    CVec<K> Pold = tile.load(a.P, g);
    CVec<K> R[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        CVec<K> Qc;
        if (a.Ncoef[c]) {
            Qc = tile.load(a.Ncoef[c], g);
        } else if constexpr (REG) {
            const double2* line = tile.reg_line(a, c, tile.line_slot());
#pragma unroll
            for (int e = 0; e < K; ++e) {
                const int n = K * g.t + e;
                const double w = ((n == 0 || n == a.gd.P) ? 0.5 * a.norm : a.norm) * a.nl_sign;
                Qc.v[e] = (n < Ny && !mi.nyq) ? cscale(line[n], w) : czero();
            }
        } else {
            Qc = tile.dct_forward(reinterpret_cast<const SC*>(a.Nphys[c]), a.dct, a.norm, g, mi.nyq);
#pragma unroll
            for (int e = 0; e < K; ++e) Qc.v[e] = cscale(Qc.v[e], a.nl_sign);
        }
        if (a.Fcoef[c]) {  // forcing(tstage, U, N): N += F (cnrk2.jl:175)
            const CVec<K> F = tile.load(a.Fcoef[c], g);
#pragma unroll
            for (int e = 0; e < K; ++e) Qc.v[e] = cadd(Qc.v[e], F.v[e]);
        }
        double bN = 0.0;
        if (a.bulk && meanmode && c != 1) bN = bulk_mean(g, Qc).x;
        if (a.stage != 0) {
            CVec<K> Qo = tile.load(a.Q[c], g);
#pragma unroll
            for (int e = 0; e < K; ++e) Qc.v[e] = cfma(a.Aj, Qo.v[e], Qc.v[e]);
        }
        if (a.store_Q) tile.store(a.Q[c], g, Qc);
        CVec<K> U = tile.load(a.U[c], g);
        if (a.bulk && meanmode && c != 1) {  // _bulkpressuregradient, cnrk2.jl:98-107
            double2 sh = csub(wall_deriv_plus(g, U), wall_deriv_minus(g, U));
            double gv = a.nu * sh.x / 2.0 + (c == 0 ? a.nu * a.curv_mean : 0.0) + bN;
            if (c == 0) gold0 = gv; else gold1 = gv;
        }
        CVec<K> lap = laplacian(g, U, mi.kappa2);
        CVec<K> dP;
        if (c == 1) {
            dP = cheb_deriv(g, Pold);
        } else {
            double kk = (c == 0) ? mi.kx : mi.kz;
#pragma unroll
            for (int e = 0; e < K; ++e) dP.v[e] = cmuli(cscale(Pold.v[e], kk));
        }
#pragma unroll
        for (int e = 0; e < K; ++e) {
            double2 x = cscale(U.v[e], a.lambda);
            x = cfma(a.nu, lap.v[e], x);
            x = csub(x, dP.v[e]);
            R[c].v[e] = cfma(a.weight, Qc.v[e], x);
            // materialise R_c here: otherwise the RHS arithmetic is sunk into
            // the solve branches below and every input of all three
            // components stays live until then
            asm volatile("" : "+v"(R[c].v[e].x), "+v"(R[c].v[e].y));
        }
    }
    if (meanmode) {
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n < Ny) R[0].v[e] = cadd(R[0].v[e], cmk(2.0 * a.nu * a.curv[n], 0.0));
        }
        if (g.t == 0) {
            R[0].v[0] = csub(R[0].v[0], cmk(gold0, 0.0));
            R[2].v[0] = csub(R[2].v[0], cmk(gold1, 0.0));
        }
    }
    double2* st = tile.stash;
    if constexpr (REG) tile.reg_sync();  // the stash aliases the lines of the nonlinear terms
    stash(st, g, R[0]);
    stash(st + K * L, g, R[1]);
    stash(st + 2 * K * L, g, R[2]);
    CVec<K> Un[3], Pn;
    if (meanmode) {
        double gnew[2] = {0.0, 0.0};
        solve_mean(g, a, a.bank, st, st + K * L, st + 2 * K * L, Un, Pn, gnew);
        if (g.t == 0 && a.grad_out) {
            a.grad_out[0] = gnew[0];
            a.grad_out[1] = gnew[1];
        }
    } else if (mi.nyq || !mi.valid) {
#pragma unroll
        for (int c = 0; c < 3; ++c) zero_vec<L, K>(Un[c]);
        zero_vec<L, K>(Pn);
    } else {
        solve_nonzero(g, a, a.bank, mi, st, st + K * L, st + 2 * K * L, Un, Pn);
    }
    if constexpr (REG) tile.reg_sync();  // the stash aliases the FFT lines reused below
    else wave_sync();
    tile.store(a.U[0], g, Un[0]);
    tile.store(a.U[1], g, Un[1]);
    tile.store(a.U[2], g, Un[2]);
    tile.store(a.P, g, Pn);
    if (a.out6[0]) {
        if constexpr (REG) inverse_six_reg<L, K, SC>(tile, a, g, mi);
        else inverse_six<L, K, SC>(tile, a, g, mi, [&](int c) { return Un[c]; });
    }
}

// Nyquist modes of a stage under the non-Nyquist-first order, elementwise
// (blk-th of order.nyq_blocks blocks).  The result equals ystage_body's for
// such a mode: the transformed nonlinear term is zero there
// (normalize_forward!), so Q = A_j Q_old + nl_sign*0 (+ F), and U, P and the
// y-physical outputs are zero.  The x Nyquist column ix = Nx/2 (every iz)
// comes first, then the z Nyquist row iz = Nz/2 (ix < nxr).
template <typename SC>
__device__ __forceinline__ void ystage_nyquist(const YArgs& a, unsigned blk) {
    const YOrder& o = a.order;
    const GridDims& gd = a.gd;
    const unsigned nnyq = (unsigned)o.nnyq;
    const unsigned total = nnyq * (unsigned)gd.Ny;
    const unsigned ncol = (gd.Nx % 2 == 0) ? (unsigned)gd.Nz : 0u;
    const bool six = a.out6[0] != nullptr, vort = a.form != FORM_DIVERGENCE;
    for (unsigned e = blk * YNT + threadIdx.x; e < total; e += o.nyq_blocks * YNT) {
        const unsigned n = e / nnyq, q = e - n * nnyq;
        const long long s = q < ncol ? (long long)q * gd.Nxh + gd.Nx / 2 : (long long)(gd.Nz / 2) * gd.Nxh + (q - ncol);
        const long long i = s + gd.B * n;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double2 Qc = a.Ncoef[c] ? a.Ncoef[c][i] : cscale(czero(), a.nl_sign);
            if (a.Fcoef[c]) Qc = cadd(Qc, a.Fcoef[c][i]);
            if (a.stage != 0) Qc = cfma(a.Aj, a.Q[c][i], Qc);
            if (a.store_Q) a.Q[c][i] = Qc;
            a.U[c][i] = czero();
        }
        a.P[i] = czero();
        if (six) {
#pragma unroll
            for (int f = 0; f < 6; ++f)
                if (f < 3 || vort) reinterpret_cast<SC*>(a.out6[f])[i] = from_c64<SC>(czero());
        }
    }
}

template <int L, int K, typename SC, bool REG>
// two waves per SIMD (<= 256 registers per lane): one wave per SIMD leaves
// the wave-serial scans and LDS FFTs unhidden.  K = 6 and 8 (Ny above 256)
// keep 1.5 and 2 times the coefficients per lane and run one wave per SIMD,
// whose larger register budget holds them without scratch (at two waves
// K = 6 spills 160 bytes per lane).
__global__ void __launch_bounds__(YNT) __attribute__((amdgpu_waves_per_eu(K >= 6 ? 1 : 2))) ystage_kernel(YArgs a) {
    if (a.order.on) {  // block-uniform branches
        if (blockIdx.x >= a.order.nyq_first) {
            ystage_nyquist<SC>(a, blockIdx.x - a.order.nyq_first);
            return;
        }
        // z rows of Nxh modes leave the blocks' row segments unaligned to
        // cache lines: neighbouring blocks share lines, so they run on one XCD
        ystage_body<L, K, SC, REG>(a, a.order.xcd ? xcd_logical(blockIdx.x, a.order.nyq_first) : blockIdx.x);
        return;
    }
    ystage_body<L, K, SC, REG>(a, blockIdx.x);
}

// prologue: state U -> six y-physical fields (velocity and vorticity)
template <int L, int K, typename SC, bool REG>
__device__ __forceinline__ void yprologue_body(const YArgs& a, unsigned block) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, REG ? a.nf * (64 / L) * a.zs : y_region_slots<L, K>(a.ld), block);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    if constexpr (REG) {
        inverse_six_reg<L, K, SC>(tile, a, g, mi);
        return;
    }
    inverse_six<L, K, SC>(tile, a, g, mi, [&](int c) { return tile.load(a.U[c], g); });
}

// The single-problem prologue keeps its own copy of the body: passing the
// byval kernel argument by reference to yprologue_body makes the compiler
// materialise part of it in scratch memory.  Under the non-Nyquist-first
// order (a.order.on) the launch has only the regular blocks: the periodic
// passes never read the Nyquist modes' y-physical values, so none are
// written.
// INPLACE: the DCT lines are transformed in place (one line per mode, half
// the LDS of the two-buffer form, so more blocks per CU); the host picks it
// where the plan fits 8 points per lane (fft_inplace_fits)
// REG: the DCTs in two register radices, instead of both
template <int L, int K, typename SC, bool INPLACE = false, bool REG = false>
__global__ void __launch_bounds__(YNT) yprologue_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    // the order's fields are read one by one (a reference to the byval
    // argument, or a copy of the whole struct, lands in scratch)
    const bool ordered = a.order.on != 0;
    const unsigned block = (ordered && a.order.xcd) ? xcd_logical(blockIdx.x, gridDim.x) : blockIdx.x;
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld,
                    REG ? a.nf * (64 / L) * a.zs : (INPLACE ? (64 / L) * a.ld : y_region_slots<L, K>(a.ld)), block);
    if (ordered) tile.order_modes(a.order.nreg, a.order.nxr, a.order.zskip);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    if constexpr (REG) {
        inverse_six_reg<L, K, SC>(tile, a, g, mi);
    } else if constexpr (L == 4) {  // all loads first: the 4-lane build stays within 128 registers so
        CVec<K> U[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) U[c] = tile.load(a.U[c], g);
        inverse_six<L, K, SC, INPLACE>(tile, a, g, mi, [&](int c) { return U[c]; });
    } else {
        inverse_six<L, K, SC, INPLACE>(tile, a, g, mi, [&](int c) { return tile.load(a.U[c], g); });
    }
}

// Batched ensemble launches: instance i owns blocks [start[i], start[i+1])
// of the grid and its own argument block tab[i] (grid, factors, fields).
// All instances of one launch share the group size L.
template <int L, int K, bool REG>
__global__ void __launch_bounds__(YNT) __attribute__((amdgpu_waves_per_eu(2)))
ystage_batch_kernel(const YArgs* __restrict__ tab, const unsigned* __restrict__ start, int n) {
    const int i = batch_instance(start, n, blockIdx.x);
    ystage_body<L, K, double2, REG>(tab[i], blockIdx.x - start[i]);
}

template <int L, int K, bool REG>
__global__ void __launch_bounds__(YNT) yprologue_batch_kernel(const YArgs* __restrict__ tab,
                                                              const unsigned* __restrict__ start, int n) {
    const int i = batch_instance(start, n, blockIdx.x);
    yprologue_body<L, K, double2, REG>(tab[i], blockIdx.x - start[i]);
}

// Stokes solve! of a bank: R (3 spectral) -> U (3), P (stokes.jl:81-108)
template <int L, int K>
__global__ void __launch_bounds__(YNT) ysolve_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    CVec<K> R[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) R[c] = tile.load(a.Rin[c], g);
    CVec<K> Un[3], Pn;
    double gnew[2] = {0.0, 0.0};
    double2* st = tile.stash;
    stash(st, g, R[0]);
    stash(st + K * L, g, R[1]);
    stash(st + 2 * K * L, g, R[2]);
    if (mi.mean && mi.valid) {
        solve_mean(g, a, a.bank, st, st + K * L, st + 2 * K * L, Un, Pn, gnew);
        if (g.t == 0 && a.grad_out) {
            a.grad_out[0] = gnew[0];
            a.grad_out[1] = gnew[1];
        }
    } else if (mi.nyq || !mi.valid) {
        for (int c = 0; c < 3; ++c) zero_vec<L, K>(Un[c]);
        zero_vec<L, K>(Pn);
    } else {
        solve_nonzero(g, a, a.bank, mi, st, st + K * L, st + 2 * K * L, Un, Pn);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) tile.store(a.U[c], g, Un[c]);
    tile.store(a.P, g, Pn);
}

// R = -Laplacian(U) (projection source, pressure.jl:125)
template <int L, int K>
__global__ void __launch_bounds__(YNT) yneglap_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    for (int c = 0; c < 3; ++c) {
        CVec<K> U = tile.load(a.U[c], g);
        CVec<K> lap = laplacian(g, U, mi.kappa2);
#pragma unroll
        for (int e = 0; e < K; ++e) lap.v[e] = cscale(lap.v[e], -1.0);
        tile.store(a.Rout[c], g, lap);
    }
}

// pressure reconstruction (_pressure_poisson, pressure.jl:196-285):
// A (3 spectral accelerations), v = U[1] -> P
template <int L, int K>
__global__ void __launch_bounds__(YNT) ypressure_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    const int P = a.gd.P, Ny = a.gd.Ny;
    CVec<K> A[3];
    for (int c = 0; c < 3; ++c) A[c] = tile.load(a.Rin[c], g);
    CVec<K> v = tile.load(a.U[1], g);
    CVec<K> Pn;
    if (mi.mean && mi.valid) {
        double2 prev3 = g.up1(A[1].v[K - 1]);
        double2 next0 = g.down1(A[1].v[0]);
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            double2 rm = (e == 0) ? prev3 : A[1].v[e - 1];
            double2 rp = (e == K - 1) ? next0 : A[1].v[e + 1];
            double2 lower = (n == 1) ? rm : cscale(rm, 0.5);
            double2 upper = (n + 1 < Ny - 1) ? cscale(rp, 0.5) : czero();
            Pn.v[e] = (n >= 1 && n <= P) ? cscale(csub(lower, upper), 1.0 / n) : czero();
        }
        double2 m = bulk_mean(g, Pn);
        if (g.t == 0) Pn.v[0] = cscale(m, -1.0);
    } else if (mi.nyq || !mi.valid) {
        zero_vec<L, K>(Pn);
    } else {
        // div A
        CVec<K> r = cheb_deriv(g, A[1]);
#pragma unroll
        for (int e = 0; e < K; ++e)
            r.v[e] = cadd(r.v[e], cadd(cmuli(cscale(A[0].v[e], mi.kx)), cmuli(cscale(A[2].v[e], mi.kz))));
        // wall data P_y(+-1) = A_y(+-1) + nu v_yy(+-1)
        double2 up = czero(), lo = czero();
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n < Ny) {
                double nn = n;
                double2 term = cfma(a.nu * (nn * nn * (nn * nn - 1.0) / 3.0), v.v[e], A[1].v[e]);
                up = cadd(up, term);
                lo = (n % 2 == 0) ? cadd(lo, term) : csub(lo, term);
            }
        }
        up = g.sum(up);
        lo = g.sum(lo);
        double fp[K];
        load_fac(a.facPN, mi.s, Ny, g, fp);
        // Neumann parity data: even (g+ - g-)/2, odd (g+ + g-)/2
        Pn = helm_solve(g, P, mi.kappa2, fp, true, r, cscale(csub(up, lo), 0.5), cscale(cadd(up, lo), 0.5));
    }
    tile.store(a.P, g, Pn);
}

// Batched Chebyshev transforms of spectral fields (no group logic).
// dir < 0: y-physical values -> normalised coefficients (normalize_forward!)
// dir > 0: coefficients -> values at the Lobatto points
template <int L, int K>
__global__ void __launch_bounds__(YNT) ydct_kernel(YArgs a, int dir) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    for (int c = 0; c < a.nfields; ++c) {
        if (dir < 0) {
            CVec<K> v = tile.dct_forward(a.Nphys[c], a.dct, a.norm, g, mi.nyq);
#pragma unroll
            for (int e = 0; e < K; ++e) v.v[e] = cscale(v.v[e], a.nl_sign);
            tile.store(a.Rout[c], g, v);
        } else {
            CVec<K> v = tile.load(a.Rin[c], g);
            tile.dct_inverse(a.out6[c], a.dct, g, v);
        }
    }
}

// Divergence form (nonlinear.jl:146-167, div! of the flux tensor): the six
// y-physical products T = (VxVx, VxVy, VxVz, VyVy, VyVz, VzVz) are forward
// transformed and N_i = -(i k T_ix + d/dy T_iy + i l T_iz) is written to Rout.
template <int L, int K>
__global__ void __launch_bounds__(YNT) ydivergence_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    CVec<K> N[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) zero_vec<L, K>(N[c]);
    // tensor entry (i, j) for products p = 0..5
    const int pi[6] = {0, 0, 0, 1, 1, 2}, pj[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        CVec<K> T = tile.dct_forward(a.Nphys[p], a.dct, a.norm, g, mi.nyq);
        CVec<K> dT = cheb_deriv(g, T);
        // contribution to N_i from d_j T_ij and, off the diagonal, to N_j from d_i T_ij
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            if (side == 1 && pi[p] == pj[p]) continue;
            const int i = side == 0 ? pi[p] : pj[p], j = side == 0 ? pj[p] : pi[p];
#pragma unroll
            for (int e = 0; e < K; ++e) {
                double2 d = (j == 1) ? dT.v[e] : cmuli(cscale(T.v[e], j == 0 ? mi.kx : mi.kz));
                N[i].v[e] = csub(N[i].v[e], d);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) tile.store(a.Rout[c], g, N[c]);
}

// Volume inner products (postprocessing.jl:30-60, 87-91).  Per mode,
// Re(u^H M v) with the exact Chebyshev mass matrix
// M_mn = (mu(m+n) + mu(|m-n|)) / 2, mu(k) = 1/(1-k^2) for even k (0 for odd),
// weighted 1 for k = 0 and 2 for k > 0 (conjugate pairs), Nyquist planes
// excluded.  Y_DOT: sum over the three components of U (U) and V (Rin).
// Y_DISSIPATION: u = v = curl U (operators.jl:172-190); the caller scales by nu.
// Each block writes its partial sum to partial[blockIdx.x].
//
// Bound by FP64 issue of the Ny^2/2 products per component.  M is Toeplitz +
// Hankel, so a lane needs mu only at m + n and m - n: with n = K q + f (f
// unrolled) both are entries at a fixed residue mod K and at the quotients
// t + q, t - q, one new entry a residue and iteration (the other is the
// previous iteration's).  The table holds mu/2 by residue, so the lanes of a
// group read consecutive words, and it takes the place of the per-degree
// constants, which this kernel does not use.  The three components share the
// entries.  At 128x97x128: 225 us with two divisions per entry, 38.6 us so.
template <int L, int K>
__global__ void __launch_bounds__(YNT) ydot_kernel(YArgs a, int curl) {
    extern __shared__ double2 smem[];
    constexpr int NT = K * L, LT = 3 * L;  // entries i = -NT .. 2 NT - 1 at [i mod K][i / K + L]
    double* mu = reinterpret_cast<double*>(smem + a.dct.n);
    for (int j = threadIdx.x; j < 3 * NT; j += YNT) {
        const int i = j - NT;
        mu[(j % K) * LT + j / K] = (i % 2 == 0) ? 0.5 / (1.0 - (double)i * i) : 0.0;
    }
    __syncthreads();
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    const int Ny = a.gd.Ny;
    double2* vline = tile.stash;  // this group's copies of v, indexed by degree
    CVec<K> u[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c] = tile.load(a.U[c], g);
    if (curl) {
        const CVec<K> d2 = cheb_deriv(g, u[2]), d0 = cheb_deriv(g, u[0]);
#pragma unroll
        for (int e = 0; e < K; ++e) {
            const double2 w0 = csub(d2.v[e], cmuli(cscale(u[1].v[e], mi.kz)));
            const double2 w1 = cmuli(csub(cscale(u[0].v[e], mi.kz), cscale(u[2].v[e], mi.kx)));
            const double2 w2 = csub(cmuli(cscale(u[1].v[e], mi.kx)), d0.v[e]);
            u[0].v[e] = w0;
            u[1].v[e] = w1;
            u[2].v[e] = w2;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) stash(vline + c * NT, g, u[c]);
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) stash(vline + c * NT, g, tile.load(a.Rin[c], g));
    }
    wave_sync();
    double2 s[3][K];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int e = 0; e < K; ++e) s[c][e] = czero();
    // plus[r] = mu/2 at m + n = K (t + q) + r and K (t + q + 1) + r, minus[r]
    // at m - n = K (t - q - 1) + r and K (t - q) + r (even r)
    double plus[2][K], minus[2][K];
#pragma unroll
    for (int r = 0; r < K; r += 2) {
        plus[0][r] = mu[r * LT + L + g.t];
        minus[1][r] = mu[r * LT + L + g.t];
    }
    const int nq = (Ny + K - 1) / K;
#pragma unroll 1
    for (int q = 0; q < nq; ++q) {
#pragma unroll
        for (int r = 0; r < K; r += 2) {
            plus[1][r] = mu[r * LT + L + g.t + q + 1];
            minus[0][r] = mu[r * LT + L + g.t - q - 1];
        }
#pragma unroll
        for (int f = 0; f < K; ++f) {
            double2 v[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] = vline[c * NT + K * q + f];
#pragma unroll
            for (int e = f & 1; e < K; e += 2) {
                const double Mmn = plus[(e + f) / K][(e + f) % K] + (e >= f ? minus[1][e >= f ? e - f : 0] : minus[0][e >= f ? 0 : K + e - f]);
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c][e] = cfma(Mmn, v[c], s[c][e]);
            }
        }
#pragma unroll
        for (int r = 0; r < K; r += 2) {
            plus[0][r] = plus[1][r];
            minus[1][r] = minus[0][r];
        }
    }
    double acc = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int e = 0; e < K; ++e)  // Re(conj(u_m) (M v)_m); s of the padded degrees may be infinite where u is 0
            if (K * g.t + e < Ny) acc += u[c].v[e].x * s[c][e].x + u[c].v[e].y * s[c][e].y;
    acc = g.sum(acc);
    const bool use = mi.valid && !mi.nyq;
    double* part = reinterpret_cast<double*>(smem);  // twiddle area is free now
    __syncthreads();
    constexpr int M = YNT / L;
    const int mloc = threadIdx.x / L;
    if (g.t == 0) part[mloc] = use ? (mi.ix == 0 ? 1.0 : 2.0) * acc : 0.0;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = 0.0;
        for (int i = 0; i < M; ++i) b += part[i];
        a.partial[blockIdx.x] = b;
    }
}

// Plane statistics of the TOTAL velocity V = U + Ub e_x (examples/mkm590/
// statistics.jl:26-43) at the Lobatto points.  By Parseval on the padded
// grid, the x-z plane mean is the (0,0) mode's y-physical value and the
// plane covariance of a, b is sum over the other modes of
// w_k Re(a(k,l,y) conj(b(k,l,y))) with w = 1 (k = 0), 2 (k > 0), Nyquist
// planes excluded.  partial[block * Ny * 9 + y * 9 + q] (PLANE_STATS_Q
// quantities: means u v w, then uu vv ww uv uw vw).
template <int L, int K>
__global__ void __launch_bounds__(YNT) ystats_kernel(YArgs a) {
    extern __shared__ double2 smem[];
    load_tables<L, K>(smem, a);
    Tile<L, K> tile(a.gd, smem, a.dct.n, a.ld, y_region_slots<L, K>(a.ld), blockIdx.x);
    Group<L, K> g(tile.tab);
    ModeInfo mi = mode_info(a.gd, tile.s);
    const int Ny = a.gd.Ny, P = a.gd.P;
    constexpr int M = YNT / L, W = 64 / L, Q = PLANE_STATS_Q;
    double2 vals[3][K];  // values at y = Kt+e (group layout after the inverse transform)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        CVec<K> U = tile.load(a.U[c], g);
        if (c == 0 && mi.mean && mi.valid) {
#pragma unroll
            for (int e = 0; e < K; ++e) {
                int n = K * g.t + e;
                if (n < Ny) U.v[e] = cadd(U.v[e], cmk(a.base[n], 0.0));
            }
        }
        // inverse Chebyshev transform in the wave's lines, result read back in group layout
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            if (n <= P) {
                double2 x = U.v[e];
                tile.bufA[tile.mw * tile.ld + n] = (n == 0 || n == P) ? cscale(x, 2.0) : x;
                if (n >= 1 && n <= P - 1) tile.bufA[tile.mw * tile.ld + 2 * P - n] = x;
            }
        }
        wave_sync();
        double2* res = lds_fft<true>(tile.bufA, tile.bufB, a.dct, tile.tw, W, tile.ld, -1, tile.lane, 64);
#pragma unroll
        for (int e = 0; e < K; ++e) {
            int n = K * g.t + e;
            vals[c][e] = (n <= P) ? cscale(res[tile.mw * tile.ld + n], 0.5) : czero();
        }
        wave_sync();
    }
    // this mode's contributions at each y of the lane: 9 quantities x K points
    const bool use = mi.valid && !mi.nyq;
    const double wk = (mi.ix == 0) ? 1.0 : 2.0;
    const int pi[6] = {0, 1, 2, 0, 0, 1}, pj[6] = {0, 1, 2, 1, 2, 2};
    __syncthreads();  // tables and wave lines are free: reuse LDS as the block's [Ny][Q] accumulator
    double* red = reinterpret_cast<double*>(smem);
    for (int idx = threadIdx.x; idx < Ny * Q; idx += YNT) red[idx] = 0.0;
    __syncthreads();
    const int mloc = threadIdx.x / L;
    // the block's modes add in a fixed order (deterministic sums)
    for (int m = 0; m < M; ++m) {
        if (mloc == m) {
#pragma unroll
            for (int e = 0; e < K; ++e) {
                const int y = K * g.t + e;
                if (y >= Ny) continue;
#pragma unroll
                for (int c = 0; c < 3; ++c) red[y * Q + c] += (use && mi.mean) ? vals[c][e].x : 0.0;
#pragma unroll
                for (int k = 0; k < 6; ++k) {
                    const double2 u = vals[pi[k]][e], v = vals[pj[k]][e];
                    red[y * Q + 3 + k] += (use && !mi.mean) ? wk * (u.x * v.x + u.y * v.y) : 0.0;
                }
            }
        }
        __syncthreads();
    }
    for (int idx = threadIdx.x; idx < Ny * Q; idx += YNT) a.partial[(size_t)blockIdx.x * Ny * Q + idx] = red[idx];
}

#if CF_Y_PART == 0
// Column sums of the blocks' partials in a fixed order: a block owns 32
// columns, its 32 row groups sum every 32nd row and are added in order.
// Bound by the latency of the loads: one thread per column took 254 us for the
// 1040 x 873 partials of 128x97x128, all rows in one serial chain; 7.6 us so.
constexpr int RCOL = 32, RGRP = 32;
__global__ void __launch_bounds__(RCOL * RGRP) reduce_columns_kernel(const double* part, int nblocks, int nq, double* out) {
    __shared__ double s[RGRP][RCOL];
    const int c = threadIdx.x % RCOL, r = threadIdx.x / RCOL, q = blockIdx.x * RCOL + c;
    double v = 0.0;
    if (q < nq) {
#pragma unroll 8
        for (int b = r; b < nblocks; b += RGRP) v += part[(size_t)b * nq + q];
    }
    s[r][c] = v;
    __syncthreads();
    if (r == 0 && q < nq) {
        for (int i = 1; i < RGRP; ++i) v += s[i][c];
        out[q] = v;
    }
}

hipError_t launch_reduce_columns(const double* part, int nblocks, int nq, double* out, hipStream_t st) {
    hipLaunchKernelGGL(reduce_columns_kernel, dim3((unsigned)((nq + RCOL - 1) / RCOL)), dim3(RCOL * RGRP), 0, st, part,
                       nblocks, nq, out);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) reduce_kernel(const double* part, int n, double* out) {
    __shared__ double s[256];
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) v += part[i];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = s[0];
}

hipError_t launch_reduce(const double* part, int n, double* out, hipStream_t st) {
    hipLaunchKernelGGL(reduce_kernel, dim3(1), dim3(256), 0, st, part, n, out);
    return hipGetLastError();
}
#endif

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
int y_group_lanes(int Ny);
int y_group_k(int Ny);
size_t y_lds_bytes(int Ny, int ld);

template <typename K>
static void allow_lds(K kernel, size_t lds) {
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

// Non-Nyquist-first order of a Y_STAGE launch (YOrder); returns its grid,
// or 0 (plain order) when the grid has no Nyquist modes or a wave's W modes
// would straddle z rows.
template <int L>
static unsigned y_stage_order(YArgs& a) {
    constexpr int M = YNT / L, W = 64 / L;
    const GridDims& gd = a.gd;
    const bool xe = gd.Nx % 2 == 0, ze = gd.Nz % 2 == 0;
    const int nxr = xe ? gd.Nx / 2 : gd.Nxh, nzr = ze ? gd.Nz - 1 : gd.Nz;
    if ((!xe && !ze) || nxr <= 0 || nzr <= 0 || nxr % W != 0) return 0;
    YOrder& o = a.order;
    o.on = 1;
    // XCD-contiguous order when a block's row segment (M modes, 16 B each) is
    // at least one 128 B line.  Measured on MI355X: 128x97x128 (M = 8) 905 ->
    // 930 steps/s, HBM fetch 1.56 -> 1.11 of the algorithmic bytes; at
    // 256x193x256 (M = 4) the same order lost 6 %.
    o.xcd = (M * 16 >= 128) ? 1 : 0;
    o.nxr = nxr;
    o.zskip = ze ? gd.Nz / 2 : gd.Nz;
    o.nreg = (long long)nxr * nzr;
    o.nnyq = (int)(gd.B - o.nreg);
    o.nyq_first = (unsigned)((o.nreg + M - 1) / M);
    const long long elems = (long long)o.nnyq * gd.Ny;  // about four per thread
    o.nyq_blocks = (unsigned)((elems + 4 * YNT - 1) / (4 * YNT));
    if (o.nyq_blocks == 0) o.nyq_blocks = 1;
    return o.nyq_first + o.nyq_blocks;
}

template <int L, int K>
static size_t y_lds_lk(int Ny, int ld) {
    return (2 * (size_t)(Ny - 1) + (size_t)CHEB_TAB_ARRAYS * K * L / 2 + (YNT / 64) * (size_t)y_region_slots<L, K>(ld)) *
           sizeof(double2);
}

template <int L, int K>
hipError_t launch_y_step(int which, const YArgs& a, hipStream_t st);
template <int L, int K>
hipError_t launch_y(int which, const YArgs& a, hipStream_t st);
template <int L>
hipError_t launch_y_batch(int which, bool reg, const YArgs* tab, const unsigned* start, int n, unsigned nblocks, size_t lds,
                          hipStream_t st);

#if CF_Y_PART != 0
template <typename Kern>
static hipError_t y_go(Kern kernel, dim3 grid, size_t lds, const YArgs& a, hipStream_t st) {
    allow_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, grid, dim3(YNT), lds, st, a);
    return hipGetLastError();
}
template <int L, int K>
hipError_t launch_y_step(int which, const YArgs& a, hipStream_t st) {
    constexpr int M = YNT / L;
    if (which != Y_STAGE && which != Y_PROLOGUE) return hipErrorInvalidValue;
    const size_t lds = y_lds_lk<L, K>(a.gd.Ny, a.ld);
    const size_t tables = (2 * (size_t)(a.gd.Ny - 1) + (size_t)CHEB_TAB_ARRAYS * K * L / 2) * sizeof(double2);
    YArgs b = a;
    const unsigned nb = y_stage_order<L>(b);
    // the prologue runs the regular (non-Nyquist) blocks only, see yprologue_kernel
    const dim3 grid(!nb ? (unsigned)((a.gd.B + M - 1) / M) : (which == Y_STAGE ? nb : b.order.nyq_first));
    if constexpr (y_has_reg<L, K>()) {
        y_reg_split(b, L, K);
        if (b.r1) {
            if (which == Y_STAGE)
                return y_go(ystage_kernel<L, K, double2, true>, grid, y_reg_lds(b, L, K), b, st);
            // K = 6: the register prologue runs one wave per SIMD (54 AGPRs), the
            // staged one three (256x257x256: 1087 against 823 us)
            if constexpr (K == 4) {
                const size_t ldsr = tables + (YNT / 64) * (size_t)b.nf * (64 / L) * b.zs * sizeof(double2);
                return y_go(yprologue_kernel<L, K, double2, false, true>, grid, ldsr, b, st);
            }
        }
    }
    if (which == Y_STAGE)
        return a.mixed ? y_go(ystage_kernel<L, K, float2, false>, grid, lds, b, st)
                       : y_go(ystage_kernel<L, K, double2, false>, grid, lds, b, st);
    if (fft_inplace_fits(a.dct, 64 / L, 8, 64)) {
        const size_t ldsi = tables + (YNT / 64) * (size_t)(64 / L) * a.ld * sizeof(double2);
        return a.mixed ? y_go(yprologue_kernel<L, K, float2, true>, grid, ldsi, b, st)
                       : y_go(yprologue_kernel<L, K, double2, true>, grid, ldsi, b, st);
    }
    return a.mixed ? y_go(yprologue_kernel<L, K, float2>, grid, lds, b, st)
                   : y_go(yprologue_kernel<L, K, double2>, grid, lds, b, st);
}

template <int L, int K>
hipError_t launch_y(int which, const YArgs& a, hipStream_t st) {
    if (which == Y_STAGE || which == Y_PROLOGUE) return launch_y_step<L, K>(which, a, st);
    constexpr int M = YNT / L;
    dim3 grid((unsigned)((a.gd.B + M - 1) / M));
    size_t lds = y_lds_lk<L, K>(a.gd.Ny, a.ld);
    allow_lds(ysolve_kernel<L, K>, lds);
    allow_lds(yneglap_kernel<L, K>, lds);
    allow_lds(ypressure_kernel<L, K>, lds);
    allow_lds(ydct_kernel<L, K>, lds);
    allow_lds(ydivergence_kernel<L, K>, lds);
    allow_lds(ydot_kernel<L, K>, lds);
    allow_lds(ystats_kernel<L, K>, lds);
    switch (which) {
        case Y_SOLVE: hipLaunchKernelGGL((ysolve_kernel<L, K>), grid, dim3(YNT), lds, st, a); break;
        case Y_NEGLAP: hipLaunchKernelGGL((yneglap_kernel<L, K>), grid, dim3(YNT), lds, st, a); break;
        case Y_PRESSURE: hipLaunchKernelGGL((ypressure_kernel<L, K>), grid, dim3(YNT), lds, st, a); break;
        case Y_DCT_FWD: hipLaunchKernelGGL((ydct_kernel<L, K>), grid, dim3(YNT), lds, st, a, -1); break;
        case Y_DCT_INV: hipLaunchKernelGGL((ydct_kernel<L, K>), grid, dim3(YNT), lds, st, a, +1); break;
        case Y_DIVERGENCE: hipLaunchKernelGGL((ydivergence_kernel<L, K>), grid, dim3(YNT), lds, st, a); break;
        case Y_DOT: hipLaunchKernelGGL((ydot_kernel<L, K>), grid, dim3(YNT), lds, st, a, 0); break;
        case Y_DISSIPATION: hipLaunchKernelGGL((ydot_kernel<L, K>), grid, dim3(YNT), lds, st, a, 1); break;
        case Y_PLANE_STATS: hipLaunchKernelGGL((ystats_kernel<L, K>), grid, dim3(YNT), lds, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename Kern>
static hipError_t y_go_batch(Kern kernel, const YArgs* tab, const unsigned* start, int n, unsigned nblocks, size_t lds,
                             hipStream_t st) {
    allow_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(YNT), lds, st, tab, start, n);
    return hipGetLastError();
}
template <int L>
hipError_t launch_y_batch(int which, bool reg, const YArgs* tab, const unsigned* start, int n, unsigned nblocks, size_t lds,
                          hipStream_t st) {
    if (which == Y_STAGE)
        return reg ? y_go_batch(ystage_batch_kernel<L, 4, true>, tab, start, n, nblocks, lds, st)
                   : y_go_batch(ystage_batch_kernel<L, 4, false>, tab, start, n, nblocks, lds, st);
    if (which == Y_PROLOGUE)
        return reg ? y_go_batch(yprologue_batch_kernel<L, 4, true>, tab, start, n, nblocks, lds, st)
                   : y_go_batch(yprologue_batch_kernel<L, 4, false>, tab, start, n, nblocks, lds, st);
    return hipErrorInvalidValue;
}

#endif  // CF_Y_PART != 0

#if CF_Y_PART == 0
unsigned y_blocks(const GridDims& gd) {
    const int L = y_group_lanes(gd.Ny);
    if (!L) return 0;
    const long long M = YNT / L;
    return (unsigned)((gd.B + M - 1) / M);
}

// Group layout of a wall-normal size: K = 4 coefficients per lane and the
// smallest L with 4 L >= Ny; above 256 points L = 64 with K = 6 (up to 384)
// or K = 8 (up to 512).
int y_group_lanes(int Ny) {
    int need = (Ny + 3) / 4;
    if (need <= 4) return 4;
    if (need <= 8) return 8;
    if (need <= 16) return 16;
    if (need <= 32) return 32;
    if (need <= 64) return 64;
    if (Ny <= 512) return 64;
    return 0;
}
int y_group_k(int Ny) { return Ny <= 256 ? 4 : (Ny <= 384 ? 6 : (Ny <= 512 ? 8 : 0)); }

// DCT twiddle table (2P entries) followed by one region per wavefront
size_t y_lds_bytes(int Ny, int ld) {
    return y_lds_bytes_layout(Ny, ld, y_group_lanes(Ny), y_group_k(Ny));
}

// Layouts built: K = 4 with L = 4..64 (the defaults up to 256 points), K = 6
// with L = 64 (the default up to 384) and L = 32, and K = 8 with L = 16, 32,
// 64 (the default up to 512); the non-default ones are alternatives the tuner
// may pick for the step's stage and prologue kernels.
size_t y_lds_bytes_layout(int Ny, int ld, int L, int K) {
    if (K * L < Ny) return 0;
    if (K == 4) {
        switch (L) {
            case 4: return y_lds_lk<4, 4>(Ny, ld);
            case 8: return y_lds_lk<8, 4>(Ny, ld);
            case 16: return y_lds_lk<16, 4>(Ny, ld);
            case 32: return y_lds_lk<32, 4>(Ny, ld);
            case 64: return y_lds_lk<64, 4>(Ny, ld);
            default: return 0;
        }
    }
    if (K == 6) return L == 64 ? y_lds_lk<64, 6>(Ny, ld) : (L == 32 ? y_lds_lk<32, 6>(Ny, ld) : 0);
    if (K == 8) {
        switch (L) {
            case 16: return y_lds_lk<16, 8>(Ny, ld);
            case 32: return y_lds_lk<32, 8>(Ny, ld);
            case 64: return y_lds_lk<64, 8>(Ny, ld);
            default: return 0;
        }
    }
    return 0;
}

// The split whose larger radix is smallest (registers), the smaller one first;
// the columns and rows of one field must fit the lanes.  The mixed step keeps
// the staged transforms and their bits: a last-bit difference before the FP32
// rounding of a field flips some of its values by an FP32 ulp, and the register
// form gains nothing there (256x193x256: 7.84 ms staged, 7.95).
void y_reg_split(YArgs& a, int L, int K) {
    const int N = 2 * a.gd.P, W = 64 / L;
    const bool staged = a.r1 < 0;
    a.r1 = a.r2 = a.nf = a.zs = 0;
    if (a.mixed || staged) return;
    for (int r2 = 2; r2 <= 32; ++r2) {
        if (N % r2 != 0 || N / r2 > r2 || !y_radix(L, K, r2) || !y_radix(L, K, N / r2)) continue;
        const int nf = 64 / (W * (r2 / 2 + 1)), lines = (N / r2 / 2 + 1) * (r2 | 1);
        if (nf < 1) return;
        a.r1 = N / r2;
        a.r2 = r2;
        a.nf = nf < 3 ? nf : 3;
        a.zs = (lines > a.gd.Ny ? lines : a.gd.Ny) | 1;
        return;
    }
}
size_t y_reg_lds(const YArgs& a, int L, int K) {
    const int W = 64 / L, lines = 3 * W * a.zs, stash = 3 * K * 64;
    return (2 * (size_t)a.gd.P + (size_t)CHEB_TAB_ARRAYS * K * L / 2 + (YNT / 64) * (size_t)(lines > stash ? lines : stash)) *
           sizeof(double2);
}

hipError_t launch_ykernel_batch(int which, int L, bool reg, const YArgs* tab, const unsigned* start, int n, unsigned nblocks,
                                size_t lds, hipStream_t st) {
    switch (L) {
        case 4: return launch_y_batch<4>(which, reg, tab, start, n, nblocks, lds, st);
        case 8: return launch_y_batch<8>(which, reg, tab, start, n, nblocks, lds, st);
        case 16: return launch_y_batch<16>(which, reg, tab, start, n, nblocks, lds, st);
        case 32: return launch_y_batch<32>(which, reg, tab, start, n, nblocks, lds, st);
        case 64: return launch_y_batch<64>(which, reg, tab, start, n, nblocks, lds, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ykernel(int which, const YArgs& a, hipStream_t st) {
    if ((which == Y_STAGE || which == Y_PROLOGUE) && a.yk != 0 &&
        !(a.yk == y_group_k(a.gd.Ny) && a.yl == y_group_lanes(a.gd.Ny))) {
        if (!y_lds_bytes_layout(a.gd.Ny, a.ld, a.yl, a.yk)) return hipErrorInvalidValue;
        if (a.yk == 6 && a.yl == 32) return launch_y_step<32, 6>(which, a, st);
        if (a.yk == 6 && a.yl == 64) return launch_y_step<64, 6>(which, a, st);
        if (a.yk == 8 && a.yl == 16) return launch_y_step<16, 8>(which, a, st);
        if (a.yk == 8 && a.yl == 32) return launch_y_step<32, 8>(which, a, st);
        if (a.yk == 8 && a.yl == 64) return launch_y_step<64, 8>(which, a, st);
        return hipErrorInvalidValue;
    }
    if (y_group_k(a.gd.Ny) == 6) return launch_y<64, 6>(which, a, st);
    if (y_group_k(a.gd.Ny) == 8) return launch_y<64, 8>(which, a, st);
    switch (y_group_lanes(a.gd.Ny)) {
        case 4: return launch_y<4, 4>(which, a, st);
        case 8: return launch_y<8, 4>(which, a, st);
        case 16: return launch_y<16, 4>(which, a, st);
        case 32: return launch_y<32, 4>(which, a, st);
        case 64: return launch_y<64, 4>(which, a, st);
        default: return hipErrorInvalidValue;
    }
}

#endif  // CF_Y_PART == 0

// Layouts and the translation unit that instantiates each: the default
// layouts (K = 4 on L = 4..64; K = 6 and 8 on L = 64 above 256 and 384
// points) with every kernel, the alternative layouts (K = 8 on 16 and 32
// lanes, K = 6 on 32) with the step's two kernels only, and the ensemble's
// batched kernels on K = 4.
#if CF_Y_PART == 1
template hipError_t launch_y<4, 4>(int, const YArgs&, hipStream_t);
template hipError_t launch_y<8, 4>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_batch<4>(int, bool, const YArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
template hipError_t launch_y_batch<8>(int, bool, const YArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_Y_PART == 2
template hipError_t launch_y<16, 4>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_step<16, 8>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_batch<16>(int, bool, const YArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_Y_PART == 3
template hipError_t launch_y<32, 4>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_batch<32>(int, bool, const YArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_Y_PART == 4
template hipError_t launch_y<64, 4>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_batch<64>(int, bool, const YArgs*, const unsigned*, int, unsigned, size_t, hipStream_t);
#elif CF_Y_PART == 5
template hipError_t launch_y_step<32, 8>(int, const YArgs&, hipStream_t);
#elif CF_Y_PART == 6
template hipError_t launch_y<64, 8>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_step<64, 8>(int, const YArgs&, hipStream_t);
#elif CF_Y_PART == 7
template hipError_t launch_y<64, 6>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_step<64, 6>(int, const YArgs&, hipStream_t);
template hipError_t launch_y_step<32, 6>(int, const YArgs&, hipStream_t);
#endif

}  // namespace cf
