// fft_kernels.hpp - the passes of the dipolar convolution
//   phi = IDFT3( potdd * DFT3( |psi|^2 ) )      (unnormalised)
// over the half spectrum spec[kz][x][y], kz = 0..Nz/2.
//
//   zfwd : reads psi rows [x][y][:], forms |s psi|^2 (s = pending
//          renormalisation), transforms two real rows at once as the real and
//          imaginary parts of one complex line, splits the result into the two
//          half spectra and writes spec[kz][x][y-tile] (coalesced over y).
//   ypass: contiguous y lines of spec, forward or inverse.
//   xconv: x lines of spec (stride Ny, coalesced over y tiles): forward FFT,
//          multiplication by potdd(|kx|, |ky|, kz), inverse FFT, one pass.
//   zinv : rebuilds two Hermitian full spectra per complex line, inverse
//          transform, real and imaginary parts are the two real rows of phi.
//   zinv_nu: zinv fused with calcnu (the composite step).
//   sweepz_zfwd: the z sweep of a step fused with zfwd of the next step.
//
// Included by fft_inst.hip with DBEC_FFT_N set; every kernel is a template on
// the length N, the lines per workgroup L and the real type R of spec.
#pragma once

#include <cstdlib>

#include "fft_launch.hpp"
#include "internal.hpp"
#include "norm_device.hpp"
#include "sweep_device.hpp"

namespace dbec {

// largest divisor of n up to 8: the batches of a loop of n loads
constexpr int batch8(int n) {
    for (int b = 8; b > 1; --b)
        if (n % b == 0) return b;
    return 1;
}

template <typename Pl, int LM = 1, bool HALF = false>
struct FftTile {
    static constexpr int T = Pl::T;
    // lines per workgroup: at least 8, and at least one wavefront of threads,
    // times the tile multiplier LM (wider tiles: longer contiguous HBM runs
    // on the strided side, fewer workgroups per CU)
    static constexpr int L0 = (64 + T - 1) / T;
    static constexpr int L1 = L0 <= 8 ? 8 : (L0 <= 16 ? 16 : (L0 <= 32 ? 32 : 64));
    static constexpr int L = HALF ? LM * L1 / 2 : LM * L1;
    static constexpr int WG = L * T;
};

template <typename R>
__device__ __forceinline__ void stage_twiddles(cpx<R> *tw_s, const cpx<R> *tw_g, int n, int tid, int nthreads) {
    for (int i = tid; i < n; i += nthreads) tw_s[i] = tw_g[i];
}

template <typename P>
struct PsiTraits;
template <>
struct PsiTraits<double> {
    static __device__ __forceinline__ double mod2(double v, double s) {
        double t = v * s;
        return t * t;
    }
};
template <>
struct PsiTraits<float> {
    static __device__ __forceinline__ double mod2(float v, double s) {
        double t = (double)v * s;
        return t * t;
    }
};
// complex psi: x^2 + y^2 as one FMA, as calcnu forms it (the reference's
// cabs(psi)^2 differs by rounding only; the library hypot costs tens of
// instructions per point)
template <>
struct PsiTraits<cpx<double>> {
    static __device__ __forceinline__ double mod2(cpx<double> v, double) { return fma(v.x, v.x, v.y * v.y); }
};
// mixed form: |psi|^2 of complex64 psi in FP32 (the spectrum is FP32 too)
template <>
struct PsiTraits<cpx<float>> {
    static __device__ __forceinline__ double mod2(cpx<float> v, double) { return v.x * v.x + v.y * v.y; }
};

// ---------------------------------------------------------------------------
template <int N, typename R, typename P, int LM>
__global__ void __launch_bounds__((FftTile<FftPlan<N>, LM>::WG))
k_zfwd(Solves v, int Nx, int Ny, const cpx<R> *__restrict__ twg, const double *__restrict__ wx, int tiles) {
    constexpr int L = FftTile<FftPlan<N>, LM>::L, WG = FftTile<FftPlan<N>, LM>::WG;
    using Pl = FftPlan<N>;
    __shared__ cpx<R> buf[N * (L + 1)];
    __shared__ cpx<R> tw[N];
    const SolveAt sr = solve_at(v);
    const P *__restrict__ psi = reinterpret_cast<const P *>(sr.psi);
    cpx<R> *__restrict__ spec = reinterpret_cast<cpx<R> *>(sr.spec);
    const int tid = threadIdx.x;
    const int ytiles = (Ny + 2 * L - 1) / (2 * L);
    const int x = blockIdx.x / ytiles;
    const int y0 = (blockIdx.x % ytiles) * 2 * L;
    const int nrows = min(2 * L, Ny - y0);
    const double s = (v.use_scale && !v.fold) ? sr.scal[SC_SCALE] : 1.0;
    stage_twiddles(tw, twg, N, tid, WG);
    // Rows 2p and 2p+1 of the tile become the real and imaginary parts of
    // line p.  A thread takes VE consecutive z of both rows, so its LDS
    // writes are whole complex slots; all of its loads are issued before the
    // first LDS write.
    constexpr int VE = sizeof(P) == 4 ? 2 : 1, NVR = N / VE, KV = L * NVR / WG;
    static_assert((L * NVR) % WG == 0, "zfwd tile");
    struct alignas(VE * sizeof(P)) Pv {
        P e[VE];
    };
    const P *src = psi + ((long)x * Ny + y0) * N;
    Pv ra[KV], rb[KV];
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        const int iv = tid + k * WG;
        const int p = iv / NVR, zv = iv % NVR;
        ra[k] = *reinterpret_cast<const Pv *>(src + (unsigned)(min(2 * p, nrows - 1) * N + zv * VE));
        rb[k] = *reinterpret_cast<const Pv *>(src + (unsigned)(min(2 * p + 1, nrows - 1) * N + zv * VE));
    }
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        const int iv = tid + k * WG;
        const int p = iv / NVR, zv = iv % NVR;
#pragma unroll
        for (int j = 0; j < VE; ++j) {
            const R va = 2 * p < nrows ? (R)PsiTraits<P>::mod2(ra[k].e[j], s) : R(0);
            const R vb = 2 * p + 1 < nrows ? (R)PsiTraits<P>::mod2(rb[k].e[j], s) : R(0);
            buf[Pl::template at<L, R>(zv * VE + j, p)] = {va, vb};
        }
    }
    __syncthreads();
    Pl::template run<-1, L>(buf, tid % L, tid / L, tw);
    // split Z = A + iB into the spectra of the two real rows:
    //   A[k] = (Z[k] + conj Z[N-k]) / 2,  B[k] = (Z[k] - conj Z[N-k]) / (2i)
    constexpr int nkz = N / 2 + 1;
#pragma unroll
    for (int q = 0; q < (nkz * 2 * L + WG - 1) / WG; ++q) {
        const int i = tid + q * WG;
        const int row = i % (2 * L), k = i / (2 * L);
        if (k < nkz && row < nrows) {
            const int p = row >> 1;
            const cpx<R> z = buf[Pl::template at<L, R>(k, p)];
            const cpx<R> w = buf[Pl::template at<L, R>((N - k) % N, p)];
            cpx<R> o;
            if ((row & 1) == 0) o = {R(0.5) * (z.x + w.x), R(0.5) * (z.y - w.y)};
            else o = {R(0.5) * (z.y + w.y), R(0.5) * (w.x - z.x)};
            spec[(unsigned)((k * Nx + x) * Ny + y0 + row)] = o;
        }
    }
    if (v.fold == 1 && blockIdx.x == 0) {  // the last step's norm, for the x convolution and calcnu
        __syncthreads();
        norm_from_cols<WG>(sr.rows, tiles, wx, Nx, sr.scal, v.shift, reinterpret_cast<double *>(buf));
    }
}

// ---------------------------------------------------------------------------
// The z sweep of one step fused with the forward z pass of the next
// (calcluz, imag3d.cu:1895-1942, then the first transform of calcpsidd2):
// both walk the same contiguous z rows.  A workgroup takes L rows of one x
// plane through the LDS tile of k_sweep_z (partitioned Thomas solve, Simpson
// column partials with COLS), stores psi, then reuses the tile's LDS for the
// |psi|^2 of its rows, two rows per complex line, and runs the forward
// transform and split of k_zfwd on them, so psi is read once for both.  The
// rows transform unscaled: the next step's norm comes from the column
// partials (v.fold == 2, first workgroup of the forward y pass).  The
// transform's plan (FusedPlan) has T = N / 8, so its L / 2 lines of T threads
// are the sweep's L * P threads (P = N / 16 segments per row).
//
// Bound by memory, as long as enough rows are in flight: a CU needs about
// 100 KiB of psi on its way, and what limits that is LDS per workgroup and,
// with complex FP64, registers.  LDS therefore holds, one after the other in
// the same bytes: the tables, which the twiddles overwrite once the solve is
// done; and the tile, the carry exchange while the tile is in registers, and
// the transform buffer after the tile is stored.  Complex rows are twice the
// transform buffer, so (half) they pass through a tile of half the rows in
// two turns, each in registers before the next: 50 instead of 83 KiB a
// workgroup of 16 rows at N = 256 in FP64.  Complex FP32 rows of less than 256 fit often
// enough without, and the two turns' barriers measured 2-8 % slower there.
// Measured (us; before: separate regions for tables, exchange and twiddles,
// whole tiles; -> now; "+" where the two passes ran unfused before):
//   rows    grid          FP64           FP32           complex FP64    complex FP32
//   16    256x384x16      10 + 8 -> 10   9 + 6 -> 8     9 + 10 -> 14    7 + 8 -> 10
//   48    192x320x48      11 + 10 -> 15  7 + 8 -> 10    13 + 22 -> 24   8 + 10 -> 13
//   64    512x192x64      18 + 21 -> 29  11 + 11 -> 15  24 + 39 -> 46   14 + 19 -> 24
//   80    256x384x80      22 + 25 -> 38  13 + 15 -> 23  30 + 47 -> 62   17 + 24 -> 30
//   192   192^3           39 -> 37       21 -> 20       63 -> 58        31 -> 31
//   256   256^3           75 -> 72       38 -> 38       214 -> 142      61 -> 58
//   384   256x256x384     84 + 84 -> 131 38 + 43 -> 61  120 + 160 -> 229 55 + 89 -> 117
//   512   128x256x512     110 -> 84      50 -> 44       279 -> 151      83 -> 72
template <int N, bool HALF>
struct FusedZ {
    static_assert(FusedPlan<N>::T * 8 == N, "fused z plan");
    // row partials of the z integrals: real lines (imaginary time) only
    template <typename S>
    static constexpr bool cols() { return std::is_floating_point<S>::value; }
    // wavefronts per SIMD that the registers have to leave room for (what LDS
    // allows; left to itself the compiler takes more registers than that)
    template <typename S>
    static constexpr int waves() {
        if (!HALF && fused_z_half<S>(N)) return sizeof(S) == 16 ? 2 : 3;
        if (cols<S>()) return sizeof(S) == 8 ? 3 : 6;
        return sizeof(S) == 16 ? 3 : 4;
    }
    template <typename S, int L>
    static constexpr size_t tile_b() {
        return ((size_t)(N + Pk<S>::n) * (HALF ? L / 2 : L) * sizeof(S) + 15) & ~size_t(15);
    }
    // transform buffer swizzled (unpadded) where the padded one does not fit
    // in the tile's region
    template <typename S, typename R, int L>
    static constexpr bool swz() { return (size_t)N * (L / 2 + 1) * sizeof(cpx<R>) > tile_b<S, L>(); }
    // the region of the tile, the exchange and the transform buffer
    template <typename S, typename R, int L>
    static constexpr size_t x_b() {
        constexpr size_t tile = tile_b<S, L>();
        constexpr size_t buf = (size_t)N * (swz<S, R, L>() ? L / 2 : L / 2 + 1) * sizeof(cpx<R>);
        constexpr size_t ex = 2 * (size_t)L * (N / 16) * sizeof(typename Arith<S>::T);
        constexpr size_t m = tile > buf ? tile : buf;
        return ((m > ex ? m : ex) + 15) & ~size_t(15);
    }
    // tables (or twiddles), last elements, row partials, then the region
    template <typename S, typename R>
    static constexpr size_t tab_b() {
        using A = typename Arith<S>::T;
        constexpr size_t t = 4 * (size_t)SweepShared<A, 16>::tab_len(N) * sizeof(A), w = (size_t)N * sizeof(cpx<R>);
        return ((t > w ? t : w) + 15) & ~size_t(15);
    }
    template <typename S, int L>
    static constexpr size_t exl_b() { return ((size_t)L * sizeof(typename Arith<S>::T) + 15) & ~size_t(15); }
    template <typename S, int L>
    static constexpr size_t exn_b() {
        return cols<S>() ? ((size_t)L * (N / 16) * sizeof(double) + 15) & ~size_t(15) : 0;
    }
    template <typename S, typename R, int L>
    static constexpr size_t x_off() { return tab_b<S, R>() + exl_b<S, L>() + exn_b<S, L>(); }
    template <typename S, typename R, int L>
    static constexpr size_t lds() { return x_off<S, R, L>() + x_b<S, R, L>(); }
    // the kernel exists for rows L: at most 512 threads, LDS within 160 KiB,
    // half tiles only of the rows that are to take them
    template <typename S, typename R, int L>
    static constexpr bool fits() {
        return L * (N / 16) <= 512 && lds<S, R, L>() <= 160 * 1024 && (!HALF || fused_z_half<S>(N));
    }
    // workgroups that a CU holds at once by LDS and registers; 0: no kernel
    template <typename S, typename R, int L>
    static constexpr int per_cu() {
        constexpr int by_lds = (int)(160 * 1024 / lds<S, R, L>()), by_reg = 4 * waves<S>() / ((L * (N / 16) + 63) / 64);
        return !fits<S, R, L>() ? 0 : (by_lds < by_reg ? by_lds : by_reg);
    }
};

// Whether the workgroups run from the largest x down, for psi of `bytes` (all
// solves of the launch).  The y sweep before it ends with the planes of the
// largest x, and 256 MiB of last-level cache hold the latest of them: complex
// psi of 176 MiB or more, which does not stay there as a whole beside the
// spectrum, is taken from that end (us a step, from the smallest x -> from the
// largest: complex FP32 482 -> 445 at 256x256x384, 456 -> 420 at 384x256x256,
// but 361 -> 365 at 512x512x80, 160 MiB; complex FP64 921 -> 901, 917 -> 891,
// 745 -> 735 at 512x256x160, 574 -> 574 at 256^3).  Real psi of these sizes
// gains nothing (604 -> 605 at 256x256x384 FP64).
inline bool z_reversed(bool real, long bytes) { return !real && bytes >= (176L << 20); }

template <int N, typename S, typename R, int L, bool COLS, bool HALF>
__global__ void __launch_bounds__(L *(N / 16), (FusedZ<N, HALF>::template waves<S>()))
k_sweepz_zfwd(Solves v, int Nx, int Ny, SweepTab<typename Arith<S>::T> tab, SweepConst<typename Arith<S>::T> k,
              const double *__restrict__ wz, const double *__restrict__ wy, const cpx<R> *__restrict__ twg, bool reversed) {
    using A = typename Arith<S>::T;
    using F = FusedZ<N, HALF>;
    using Pl = FusedPlan<N>;
    // psi tile rows of N + VE elements: 16-byte aligned, and consecutive rows
    // 4 banks apart, so the packet accesses below are conflict-free
    constexpr int M = 16, VE = Pk<S>::n, KV = M / VE;
    constexpr int P = N / M, WG = L * P, LF = L / 2, RS = N + VE;
    // turns through the tile, rows and threads of each
    constexpr int NH = HALF ? 2 : 1, LH = L / NH, TH = WG / NH;
    static_assert(Pl::T * LF == WG && KV % NH == 0 && TH * NH == WG, "one transform thread per sweep thread");
    static_assert(COLS == F::template cols<S>(), "z integrals for real lines");
    constexpr size_t X_OFF = F::template x_off<S, R, L>(), X_B = F::template x_b<S, R, L>();
    constexpr size_t TAB_B = F::template tab_b<S, R>(), EXL_B = F::template exl_b<S, L>();
    constexpr bool SWZ = F::template swz<S, R, L>();  // swizzled transform buffer
    static_assert(X_B >= (size_t)RS * LH * sizeof(S) && X_B >= (size_t)N * (SWZ ? LF : LF + 1) * sizeof(cpx<R>),
                  "fused z LDS");
    __shared__ __align__(16) char smem[F::template lds<S, R, L>()];
    const SolveAt sr = solve_at(v);
    S *__restrict__ psi = reinterpret_cast<S *>(sr.psi);
    cpx<R> *__restrict__ spec = reinterpret_cast<cpx<R> *>(sr.spec);
    SweepShared<A, M> sh(smem, N, WG, L);
    sh.exa = reinterpret_cast<A *>(smem + X_OFF);  // in the tile region while the tile is in registers
    sh.exb = sh.exa + WG;
    sh.exl = reinterpret_cast<A *>(smem + TAB_B);
    sh.exn = reinterpret_cast<double *>(smem + TAB_B + EXL_B);
    cpx<R> *tw = reinterpret_cast<cpx<R> *>(smem);  // over the tables, after the solve
    S *tile = reinterpret_cast<S *>(smem + X_OFF);
    cpx<R> *buf = reinterpret_cast<cpx<R> *>(smem + X_OFF);  // after the tile is stored
    const int tid = threadIdx.x;
    const int hh = HALF ? tid / TH : 0, th = HALF ? tid % TH : tid;
    const int l = hh * LH + th % LH, s = th / LH;
    // a complex FP64 segment is 256 bytes, so the 16 lanes that one LDS cycle
    // serves (LH rows of 16 / LH segments) would meet in the same banks: the
    // segments that share a cycle take their packets in different orders
    const auto at = [](int row, int e) {
        if constexpr (HALF && sizeof(S) == 16) e ^= ((e >> 4) & (16 / (LH < 16 ? LH : 16) - 1)) * (LH < 16 ? LH : 0);
        return row * RS + e;
    };
    const int yt = (Ny + L - 1) / L;
    const int bid = !COLS && reversed ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
    const int xrow = bid / yt, tno = bid % yt, y0 = tno * L;
    const int nl = min(L, Ny - y0);
    const long base = ((long)xrow * Ny + y0) * N;
    const A zero = m_zero(k.A);
    const int npk = nl * N / VE;
    const int e0 = s * M;
    const bool act = l < nl;
    A vv[M], hl, hr;
    const CoefPre<A> cp = coef_pre(tab, N, tid);
    // the twiddles wait in registers until the tables are free
    constexpr int KT = (N + WG - 1) / WG;
    R twx[KT], twy[KT];
    {
        typename Pk<S>::type r[KV];
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const int iv = tid + q * WG;
            r[q] = ld_pk(psi + base + (unsigned)((iv < npk ? iv : 0) * VE));
        }
#pragma unroll
        for (int q = 0; q < KT; ++q) {
            const int i = tid + q * WG;
            const cpx<R> w = twg[i < N ? i : 0];
            twx[q] = w.x;
            twy[q] = w.y;
        }
        coef_put(sh, cp, tab, N, tid, WG);
        if constexpr (NH == 1) {
#pragma unroll
            for (int q = 0; q < KV; ++q) {
                const int iv = tid + q * WG;
                if (iv < npk) {
                    const int e = (iv * VE) % N, row = (iv * VE) / N;
                    st_pk(tile + row * RS + e, r[q]);
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if (h) __syncthreads();  // the last pass's rows are in registers
#pragma unroll
                for (int q = h * (KV / NH); q < (h + 1) * (KV / NH); ++q) {
                    const int iv = tid + q * WG;
                    if (iv < npk) {
                        const int e = (iv * VE) % N, row = (iv * VE) / N;
                        st_pk(tile + at(row - h * LH, e), r[q]);
                    }
                }
                __syncthreads();
                if (hh == h) {
                    const int row = l - h * LH;
                    hl = hr = zero;
#pragma unroll
                    for (int m = 0; m < KV; ++m) {
                        const typename Pk<S>::type pk = ld_pk(tile + at(row, e0 + m * VE));
#pragma unroll
                        for (int j = 0; j < VE; ++j) vv[m * VE + j] = act ? to_a(pk.e[j]) : zero;
                    }
                    if (act && e0 > 0) hl = to_a(tile[at(row, e0 - 1)]);
                    if (act && e0 + M < N) hr = to_a(tile[at(row, e0 + M)]);
                }
            }
        }
    }
    if constexpr (NH == 1) {
        __syncthreads();
        const S *row = tile + l * RS;
#pragma unroll
        for (int m = 0; m < KV; ++m) {
            const typename Pk<S>::type pk = ld_pk(row + e0 + m * VE);
#pragma unroll
            for (int j = 0; j < VE; ++j) vv[m * VE + j] = act ? to_a(pk.e[j]) : zero;
        }
        hl = (act && e0 > 0) ? to_a(row[e0 - 1]) : zero;
        hr = (act && e0 + M < N) ? to_a(row[e0 + M]) : zero;
    }
    {
        __syncthreads();  // the tile is in registers; its region takes the carry exchange
        const double acc = seg_solve<A, M, COLS, true>(vv, hl, hr, e0, N, s, l, L, P, sh, k, wz);
        __syncthreads();  // every carry is read; the region holds the tile again
        const auto put = [&](int row) {
#pragma unroll
            for (int m = 0; m < KV; ++m) {
                typename Pk<S>::type o;
#pragma unroll
                for (int j = 0; j < VE; ++j) o.e[j] = from_a<S>(vv[m * VE + j]);
                st_pk(tile + at(row, e0 + m * VE), o);
            }
        };
        if (act && (NH == 1 || hh == 0)) put(l);
        if constexpr (COLS) {
            sh.exn[s * L + l] = acc;
            __syncthreads();
            if (tid < 64) {
                double w = 0.0;
                if (tid < L && tid < nl) {
                    double rsum = 0.0;
                    for (int t = 0; t < P; ++t) rsum += sh.exn[t * L + tid];
                    w = wy[y0 + tid] * rsum;
                }
                w = wave_sum(w);
                if (tid == 0) sr.rows[(long)tno * Nx + xrow] = w;
            }
        } else {
            __syncthreads();
        }
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            if (h) {
                __syncthreads();  // the first rows are stored
                if (act && hh == h) put(l - h * LH);
                __syncthreads();
            }
#pragma unroll
            for (int q = h * (KV / NH); q < (h + 1) * (KV / NH); ++q) {
                const int iv = tid + q * WG;
                if (iv < npk) {
                    const int e = (iv * VE) % N, row = (iv * VE) / N;
                    st_pk(psi + base + (unsigned)(iv * VE), ld_pk(tile + at(row - h * LH, e)));
                }
            }
        }
    }
    __syncthreads();  // the tile is stored; its LDS becomes the transform buffer (and the tables the twiddles)
#pragma unroll
    for (int q = 0; q < KT; ++q) {
        const int i = tid + q * WG;
        if (i < N) tw[i] = {twx[q], twy[q]};
    }
    // |psi|^2 of the new rows (zero past the plane's last row): row 2p is the
    // real part, row 2p + 1 the imaginary part of line p
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const R m2 = act ? (R)PsiTraits<S>::mod2(from_a<S>(vv[j]), 1.0) : R(0);
        R *slot = reinterpret_cast<R *>(&buf[Pl::template at<LF, R, SWZ>(e0 + j, l >> 1)]);
        slot[l & 1] = m2;
    }
    __syncthreads();
    Pl::template run<-1, LF, SWZ>(buf, tid % LF, tid / LF, tw);
    // split Z = A + iB into the spectra of the two real rows (as k_zfwd)
    constexpr int nkz = N / 2 + 1;
#pragma unroll
    for (int q = 0; q < (nkz * L + WG - 1) / WG; ++q) {
        const int i = tid + q * WG;
        const int row = i % L, kz = i / L;
        if (kz < nkz && row < nl) {
            const int p = row >> 1;
            const cpx<R> z = buf[Pl::template at<LF, R, SWZ>(kz, p)];
            const cpx<R> w = buf[Pl::template at<LF, R, SWZ>((N - kz) % N, p)];
            cpx<R> o;
            if ((row & 1) == 0) o = {R(0.5) * (z.x + w.x), R(0.5) * (z.y - w.y)};
            else o = {R(0.5) * (z.y + w.y), R(0.5) * (w.x - z.x)};
            spec[(unsigned)((kz * Nx + xrow) * Ny + y0 + row)] = o;
        }
    }
}

// ---------------------------------------------------------------------------
// With v.fold == 2 (the forward z pass ran fused with the last z sweep) the
// first workgroup of each solve's forward pass also forms the last step's
// norm from the z sweep's column partials, for the x convolution and calcnu.
template <int N, int DIR, typename R, int LM, typename Pl>
__global__ void __launch_bounds__((FftTile<Pl, LM>::WG))
k_ypass(Solves v, long nlines, const cpx<R> *__restrict__ twg, const double *__restrict__ wx, int tiles, int Nx) {
    constexpr int L = FftTile<Pl, LM>::L, WG = FftTile<Pl, LM>::WG;
    __shared__ cpx<R> buf[N * (L + 1)];
    __shared__ cpx<R> tw[N];
    cpx<R> *__restrict__ spec = reinterpret_cast<cpx<R> *>(solve_at(v).spec);
    const int tid = threadIdx.x;
    stage_twiddles(tw, twg, N, tid, WG);
    const long line0 = (long)blockIdx.x * L;
    const int nl = (int)min((long)L, nlines - line0);
    cpx<R> *g = spec + line0 * N;
    constexpr int K = L * N / WG;
    static_assert((L * N) % WG == 0, "ypass tile");
    cpx<R> r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = tid + k * WG;
        r[k] = g[i < nl * N ? i : 0];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = tid + k * WG;
        buf[Pl::template at<L, R>(i % N, i / N)] = r[k];
    }
    __syncthreads();
    Pl::template run<DIR, L>(buf, tid % L, tid / L, tw);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = tid + k * WG;
        if (i < nl * N) g[i] = buf[Pl::template at<L, R>(i % N, i / N)];
    }
    if (DIR < 0 && v.fold == 2 && blockIdx.x == 0) {
        const SolveAt sr = solve_at(v);
        __syncthreads();  // buf becomes the reduction scratch
        norm_from_cols<WG>(sr.rows, tiles, wx, Nx, sr.scal, v.shift, reinterpret_cast<double *>(buf));
    }
}

// ---------------------------------------------------------------------------
// PL: the spectrum's rows come from the plane kernels (digit order along y,
// yq = Ny / 8; the norm from one partial per x with v.fold == 3); a template
// parameter, so the other grids' kernel stays as lean as without it.
template <int N, typename R, int LM, bool PL, typename Pl>
__global__ void __launch_bounds__((FftTile<Pl, LM>::WG))
k_xconv(Solves v, const R *__restrict__ potddq, int Ny, const cpx<R> *__restrict__ twg, const double *__restrict__ wx,
        int yq) {
    constexpr int L = FftTile<Pl, LM>::L, WG = FftTile<Pl, LM>::WG;
    constexpr int T = Pl::T, K = N / T;  // x values per thread
    static_assert(L * T == WG, "xconv tile");
    constexpr int NXH = N / 2 + 1;
    __shared__ cpx<R> buf[N * (L + 1)];
    __shared__ cpx<R> tw[N];
    const SolveAt sr = solve_at(v);
    cpx<R> *__restrict__ spec = reinterpret_cast<cpx<R> *>(sr.spec);
    // folded norm: |psi|^2 was transformed unscaled, so potdd takes 1/norm^2
    R s2 = (!PL && v.fold) ? (R)(sr.scal[SC_SCALE] * sr.scal[SC_SCALE]) : R(1);
    const int tid = threadIdx.x;
    const int ytiles = (Ny + L - 1) / L;
    const int kz = blockIdx.x / ytiles;
    // y tiles of one kz: the first half in order, the second half reversed,
    // so tile t and its mirror tile (ytiles - 1 - t, the same |ky| table
    // rows) are h workgroups apart.  Workgroups go to the 8 XCDs round
    // robin; with h a multiple of 8 (256 lines in tiles of 16) the pair runs
    // on one XCD at about the same time and the second reads the table rows
    // from that XCD's L2.
    const int p = blockIdx.x % ytiles, h = (ytiles + 1) / 2;
    const int y0 = (p < h ? p : ytiles - 1 - (p - h)) * L;
    const int nl = min(L, Ny - y0);
    stage_twiddles(tw, twg, N, tid, WG);
    // Thread (l, t) holds x = t + k T of y line l, lanes along y (coalesced
    // rows of L values): the layout in which the transforms take and leave
    // their line in registers, so the potdd product is applied in registers.
    const int l = tid % L, t = tid / L;
    const int y = y0 + (l < nl ? l : 0);
    cpx<R> *g = spec + (long)kz * N * Ny + y;
    cpx<R> r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) r[k] = g[(unsigned)((t + k * T) * Ny)];
    // potdd(|kx|, |ky|, kz): the table rows [kz][|ky|] are contiguous in |kx|
    const int Ny2 = Ny / 2;
    const int ky = PL ? y / yq + 8 * (y % yq) : y, ka = ky <= Ny2 ? ky : Ny - ky;
    const int tq = PL && pot_digit_rows<R>() ? yq : 0;
    const R *pk = potddq + ((long)kz * pot_rows(Ny, tq) + pot_row(ka, tq)) * NXH;
    R pw[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int e = t + k * T;
        pw[k] = pk[e <= N / 2 ? e : N - e];
    }
    if (PL && v.fold) {  // one partial per x: every workgroup forms the norm, the first one stores it
        static_assert(sizeof(buf) >= WG * sizeof(double), "norm scratch");
        const double sc = norm_from_cols<WG>(sr.rows, 1, wx, N, sr.scal, v.shift, reinterpret_cast<double *>(buf),
                                             blockIdx.x == 0);
        s2 = (R)(sc * sc);
        __syncthreads();  // the scratch becomes the transform buffer
    }
    Pl::template run_reg<-1, L>(buf, l, t, tw, r);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const R w = pw[k] * s2;
        r[k] = {r[k].x * w, r[k].y * w};
    }
    __syncthreads();  // the forward transform's last LDS reads are done
    Pl::template run_reg<+1, L>(buf, l, t, tw, r);
    if (l < nl) {
#pragma unroll
        for (int k = 0; k < K; ++k) g[(unsigned)((t + k * T) * Ny)] = r[k];
    }
}

// ---------------------------------------------------------------------------
// Inverse z transform of two real rows per complex line: line p holds
//   Z[k] = A[k] + i B[k] (k <= N/2) and Z[N-k] = conj A[k] + i conj B[k],
// A, B the half spectra of the rows; the imaginary parts of the
// self-conjugate bins k = 0, N/2 are dropped.  SpecIdx(p, k, &ia, &ib) sets
// the spec indices of A and B and returns which of them exist (bit 0: A,
// bit 1: B); a missing one reads as zero.  All loads are issued before the
// first LDS write.
template <int N, typename Pl, int L, int WG, bool SWZ, typename R, typename SpecIdx>
__device__ __forceinline__ void load_hermitian_pairs(cpx<R> *buf, const cpx<R> *__restrict__ spec, int tid,
                                                     const SpecIdx &idx) {
    constexpr int nkz = N / 2 + 1;
    constexpr int K = (nkz * L + WG - 1) / WG;
    cpx<R> ra[K], rb[K];
    int m[K];
#pragma unroll
    for (int q = 0; q < K; ++q) {
        const int i = tid + q * WG;
        const int p = i % L, k = i / L;
        unsigned ia = 0, ib = 0;
        m[q] = i < nkz * L ? idx(p, k, ia, ib) : 0;
        ra[q] = spec[(m[q] & 1) ? ia : 0u];
        rb[q] = spec[(m[q] & 2) ? ib : 0u];
    }
#pragma unroll
    for (int q = 0; q < K; ++q) {
        const int i = tid + q * WG;
        const int p = i % L, k = i / L;
        if (i < nkz * L) {
            cpx<R> a = ra[q], b = rb[q];
            if (!(m[q] & 1)) a = {R(0), R(0)};
            if (!(m[q] & 2)) b = {R(0), R(0)};
            if (k == 0 || k == N / 2) {
                a.y = R(0);
                b.y = R(0);
            }
            buf[Pl::template at<L, R, SWZ>(k, p)] = {a.x - b.y, a.y + b.x};
            if (k > 0 && k < N / 2) buf[Pl::template at<L, R, SWZ>(N - k, p)] = {a.x + b.y, b.x - a.y};
        }
    }
}

// The same pairs straight into the registers of the first transform pass:
// v[r] = Z[t + r T] of line p = l (T threads per line), each bin above N/2
// formed from the spectrum rows of its mirror N - k.
template <int N, typename Pl, typename R, typename SpecIdx>
__device__ __forceinline__ void load_hermitian_reg(cpx<R> *v, const cpx<R> *__restrict__ spec, int l, int t,
                                                   const SpecIdx &idx) {
    constexpr int T = Pl::T, K = N / T;
    cpx<R> ra[K], rb[K];
    int m[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const int k = t + r * T, kk = k <= N / 2 ? k : N - k;
        unsigned ia = 0, ib = 0;
        m[r] = idx(l, kk, ia, ib);
        ra[r] = spec[(m[r] & 1) ? ia : 0u];
        rb[r] = spec[(m[r] & 2) ? ib : 0u];
    }
#pragma unroll
    for (int r = 0; r < K; ++r) {
        const int k = t + r * T, kk = k <= N / 2 ? k : N - k;
        cpx<R> a = ra[r], b = rb[r];
        if (!(m[r] & 1)) a = {R(0), R(0)};
        if (!(m[r] & 2)) b = {R(0), R(0)};
        if (kk == 0 || kk == N / 2) {
            a.y = R(0);
            b.y = R(0);
        }
        v[r] = k <= N / 2 ? cpx<R>{a.x - b.y, a.y + b.x} : cpx<R>{a.x + b.y, b.x - a.y};
    }
}

// k_zinv also makes the periodic face copies of the potential
// (calcpsidd2_kernel2a/2b, imag3d.cu:1491-1505, 1591-1625, at one rank):
//   A: phi[Nx-1][j][k] = phi[0][j][k]  (j < Ny-1, k < Nz-1)
//   B: phi[i][Ny-1][k] = phi[i][0][k]  (i < Nx-1, k < Nz-1)
//   C: phi[i][j][Nz-1] = phi[i][j][0]  (i < Nx-1, j < Ny-1)
// The source row's workgroup writes both places of A and B, the face row's own
// one leaves those elements alone, so each is written once.  Against a launch
// of their own, calcpsidd2 in us: 25.2 -> 22.7 at 32x160x32, 57.6 -> 55.8 at
// 96x160x96, 234 -> 228 at 256^3 (FP64); 22.7 -> 20.6, 40.8 -> 38.6, 125.4 ->
// 123.3 (FP32 spectra).
template <int N, typename R, int LM>
__global__ void __launch_bounds__((FftTile<FftPlan<N>, LM>::WG))
k_zinv(const cpx<R> *__restrict__ spec, R *__restrict__ phi, int Nx, int Ny, const cpx<R> *__restrict__ twg) {
    constexpr int L = FftTile<FftPlan<N>, LM>::L, WG = FftTile<FftPlan<N>, LM>::WG;
    using Pl = FftPlan<N>;
    __shared__ cpx<R> buf[N * (L + 1)];
    __shared__ cpx<R> tw[N];
    const int tid = threadIdx.x;
    const int ytiles = (Ny + 2 * L - 1) / (2 * L);
    const int x = blockIdx.x / ytiles;
    const int y0 = (blockIdx.x % ytiles) * 2 * L;
    const int nrows = min(2 * L, Ny - y0);
    stage_twiddles(tw, twg, N, tid, WG);
    load_hermitian_pairs<N, Pl, L, WG, false>(buf, spec, tid, [&](int p, int k, unsigned &ia, unsigned &ib) {
        ia = (unsigned)((k * Nx + x) * Ny + y0 + 2 * p);
        ib = ia + 1;
        return (2 * p < nrows ? 1 : 0) | (2 * p + 1 < nrows ? 2 : 0);
    });
    __syncthreads();
    Pl::template run<+1, L>(buf, tid % L, tid / L, tw);
    R *dst = phi + ((long)x * Ny + y0) * N;
    constexpr int Q = 2 * L * N / WG;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + q * WG;
        const int z = i % N, row = i / N;
        if (row < nrows) {
            const int y = y0 + row;
            const bool xl = x == Nx - 1, yl = y == Ny - 1, zl = z == N - 1;
            const cpx<R> c = buf[Pl::template at<L, R>(!xl && !yl && zl ? 0 : z, row >> 1)];
            const R v = (row & 1) ? c.y : c.x;
            if (zl || xl == yl) dst[(unsigned)(row * N + z)] = v;
            if (!zl && x == 0 && !yl) phi[((long)(Nx - 1) * Ny + y) * N + z] = v;
            if (!zl && y == 0 && !xl) phi[((long)x * Ny + Ny - 1) * N + z] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// zinv fused with calcnu (calcnu_kernel, imag3d.cu:1759-1783; real3d.cu
// 1856-1883).  Blocks [0, nfaceb) take the face rows x = Nx-1 or y = Ny-1,
// whose phi comes from other rows after the periodic face copies
// (calcpsidd2_kernel2a/2b, imag3d.cu:1591-1625):
//   row (Nx-1, y):          z < Nz-1 and y < Ny-1 from row (0, y), else own
//   row (x, Ny-1), x<Nx-1:  z < Nz-1 from row (x, 0), z = Nz-1 own.
// A face row is transformed together with its source row as the real and
// imaginary parts of one complex line; face f < Ny is (Nx-1, f), face f >= Ny
// is (f - Ny, Ny-1).  They go first so that they overlap the interior
// blocks instead of trailing them.  The remaining blocks take the interior
// rows x < Nx-1, y < Ny-1: within such a row the face copy of
// calcpsidd2_kernel2b (imag3d.cu:1618-1624) takes phi[.][.][Nz-1] from
// phi[.][.][0] of the same row, so the row's potential never leaves the chip.
// The tile's psi is fetched into registers before the transform when it is at
// most 256 bytes per thread (every plan with T = N / 8 or N / 4), so its
// latency overlaps the spectrum load and the passes; otherwise after it in
// batches of 8.  The per-row and per-z parts of the trap
// potential (trap_xy, trap_z) are staged in LDS.  With ZREG the spectrum
// pairs go straight into the registers of the first transform pass
// (load_hermitian_reg) instead of through LDS; with SWZ the transform buffer
// is the swizzled one (lds_at).  Neither changes the results.
template <int N, typename R, typename P, int LM, bool ZREG, bool SWZ, typename Pl>
__global__ void __launch_bounds__((FftTile<Pl, LM, kZHalf<N, P>>::WG))
k_zinv_nu(Solves v, const double *__restrict__ sq, NuConst nc, int Nx, int Ny, int nfaceb,
          const cpx<R> *__restrict__ twg) {
    constexpr int L = FftTile<Pl, LM, kZHalf<N, P>>::L, WG = FftTile<Pl, LM, kZHalf<N, P>>::WG;
    constexpr int Q = 2 * L * N / WG;  // psi elements per thread (interior rows)
    // the tile's psi (at most 256 bytes per thread) is fetched before the
    // transform, so its latency overlaps the spectrum load and the passes
    constexpr bool PREFETCH = Q * sizeof(P) <= 256;
    constexpr int C = PREFETCH ? Q : batch8(Q);  // psi batch
    static_assert((2 * L * N) % WG == 0 && Q % C == 0, "zinv_nu tile");
    __shared__ cpx<R> buf[N * lds_slots_per_row<L, SWZ>()];
    // complex FP64 psi with the swizzled buffer: the passes read the
    // twiddles from the global table (L1 / L2), which leaves LDS for a third
    // workgroup per CU
    constexpr bool TWG = SWZ && std::is_same<P, cpx<double>>::value;
    __shared__ cpx<R> tw_s[TWG ? 1 : N];
    const cpx<R> *tw = TWG ? twg : tw_s;
    __shared__ double sqz[N];      // trap_z of each z
    __shared__ double sqr[2 * L];  // trap_xy of the tile's rows (faces: of each face row)
    const SolveAt sr = solve_at(v);
    const cpx<R> *__restrict__ spec = reinterpret_cast<const cpx<R> *>(sr.spec);
    P *__restrict__ psi = reinterpret_cast<P *>(sr.psi);
    const TrapConst tc = sr.p.tc;
    nc.g = sr.p.g;
    nc.gd = sr.p.gd;
    nc.shift = v.shift ? sr.scal[SC_SHIFT] : 0.0;
    nc.cap = v.shift;
    nc.capped = sr.scal + SC_CAPPED;
    nu_prepare(nc);
    const int tid = threadIdx.x;
    const double s = v.use_scale ? sr.scal[SC_SCALE] : 1.0;
    if constexpr (!TWG) stage_twiddles(tw_s, twg, N, tid, WG);
    for (int i = tid; i < N; i += WG) sqz[i] = trap_z(tc, sq[Nx + Ny + i]);
    if ((int)blockIdx.x >= nfaceb) {
        const int b = (int)blockIdx.x - nfaceb;
        const int ytiles = (Ny + 2 * L - 1) / (2 * L);
        const int x = b / ytiles;  // x < Nx - 1
        const int y0 = (b % ytiles) * 2 * L;
        const int nrows = min(2 * L, Ny - y0);
        P *dst = psi + ((long)x * Ny + y0) * N;
        // 2L rows; a workgroup of L * T threads covers them in one pass when
        // T >= 2, in two when T = 1 (N = 16)
        for (int r = tid; r < 2 * L; r += WG) sqr[r] = trap_xy(tc, sq[x], sq[Nx + min(y0 + r, Ny - 1)]);
        P pv[C];
        if constexpr (PREFETCH) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int i = tid + q * WG;
                pv[q] = dst[(unsigned)(min(i / N, nrows - 1) * N + i % N)];
            }
        }
        const auto idx = [&](int p, int k, unsigned &ia, unsigned &ib) {
            ia = (unsigned)((k * Nx + x) * Ny + y0 + 2 * p);
            ib = ia + 1;
            return (2 * p < nrows ? 1 : 0) | (2 * p + 1 < nrows ? 2 : 0);
        };
        if constexpr (ZREG) {
            cpx<R> zv[N / Pl::T];
            load_hermitian_reg<N, Pl>(zv, spec, tid % L, tid / L, idx);
            Pl::template run_from_reg<+1, L, SWZ>(buf, tid % L, tid / L, tw, zv);
        } else {
            load_hermitian_pairs<N, Pl, L, WG, SWZ>(buf, spec, tid, idx);
            __syncthreads();
            Pl::template run<+1, L, SWZ>(buf, tid % L, tid / L, tw);
        }
#pragma unroll
        for (int q0 = 0; q0 < Q; q0 += C) {
            if constexpr (!PREFETCH) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int i = tid + (q0 + c) * WG;
                    pv[c] = dst[(unsigned)(min(i / N, nrows - 1) * N + i % N)];
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int i = tid + (q0 + c) * WG;
                const int z = i % N, row = i / N;
                if (row < nrows && y0 + row < Ny - 1) {
                    const cpx<R> cv = buf[Pl::template at<L, R, SWZ>(z == N - 1 ? 0 : z, row >> 1)];
                    const R phi = (row & 1) ? cv.y : cv.x;
                    const double pot = trap_sum(tc, sqr[row], sqz[z]);
                    dst[(unsigned)(row * N + z)] = nu_apply(pv[PREFETCH ? q0 + c : c], s, phi, pot, nc);
                }
            }
        }
        return;
    }
    // face rows
    const int nface = Ny + Nx - 1;
    const int f0 = (int)blockIdx.x * L;
    const int nl = min(L, nface - f0);
    if (tid < L) {
        const int f = f0 + min(tid, nl - 1);
        sqr[tid] = trap_xy(tc, sq[f < Ny ? Nx - 1 : f - Ny], sq[Nx + (f < Ny ? f : Ny - 1)]);
    }
    const auto fidx = [&](int p, int k, unsigned &ia, unsigned &ib) {
        if (p >= nl) return 0;
        const int f = f0 + p;
        int xo, yo, xs, ys;
        if (f < Ny) { xo = Nx - 1; yo = f; xs = 0; ys = f; }
        else { xo = f - Ny; yo = Ny - 1; xs = f - Ny; ys = 0; }
        ia = (unsigned)((k * Nx + xo) * Ny + yo);
        ib = (unsigned)((k * Nx + xs) * Ny + ys);
        return 3;
    };
    if constexpr (ZREG) {
        cpx<R> zv[N / Pl::T];
        load_hermitian_reg<N, Pl>(zv, spec, tid % L, tid / L, fidx);
        Pl::template run_from_reg<+1, L, SWZ>(buf, tid % L, tid / L, tw, zv);
    } else {
        load_hermitian_pairs<N, Pl, L, WG, SWZ>(buf, spec, tid, fidx);
        __syncthreads();
        Pl::template run<+1, L, SWZ>(buf, tid % L, tid / L, tw);
    }
    constexpr int QF = L * N / WG;
    constexpr int CF = PREFETCH ? QF : batch8(QF);
    static_assert((L * N) % WG == 0 && QF % CF == 0, "zinv_nu face tile");
#pragma unroll
    for (int q0 = 0; q0 < QF; q0 += CF) {
        P fv[CF];
        unsigned fn[CF];
#pragma unroll
        for (int c = 0; c < CF; ++c) {
            const int i = tid + (q0 + c) * WG;
            const int z = i % N, f = f0 + min(i / N, nl - 1);
            const int xo = f < Ny ? Nx - 1 : f - Ny, yo = f < Ny ? f : Ny - 1;
            fn[c] = (unsigned)((xo * Ny + yo) * N + z);
            fv[c] = psi[fn[c]];
        }
#pragma unroll
        for (int c = 0; c < CF; ++c) {
            const int i = tid + (q0 + c) * WG;
            const int z = i % N, p = i / N;
            if (p < nl) {
                const int f = f0 + p;
                const bool from_src = (f < Ny) ? (f < Ny - 1) && (z < N - 1) : (z < N - 1);
                const cpx<R> cv = buf[Pl::template at<L, R, SWZ>(z, p)];
                const R phi = from_src ? cv.y : cv.x;
                const double pot = trap_sum(tc, sqr[p], sqz[z]);
                psi[fn[c]] = nu_apply(fv[c], s, phi, pot, nc);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Launchers for one length.  Each pass has a tile multiplier LM (1 or 2)
// chosen per precision and plan from measurements; the environment variables
// DBEC_FFT_LM_{ZFWD,YPASS,XCONV,FUSED}{64,32} override them (tuning runs).
inline int fft_lm(const char *name, int dflt) {
    const char *e = getenv(name);
    if (!e) return dflt;
    int v = atoi(e);
    return (v == 1 || v == 2) ? v : dflt;
}
// DBEC_FFT_ZINV_SWZ: transform buffer layout of the FP64 fused inverse pass
// (0 padded, 1 swizzled); -1 when unset
inline int fft_swz_env() {
    const char *e = getenv("DBEC_FFT_ZINV_SWZ");
    if (!e) return -1;
    const int v = atoi(e);
    return (v == 0 || v == 1) ? v : -1;
}

template <int N>
struct FftLaunchImpl {
    // Plans whose workgroup at LM = 1 has fewer than 192 threads take LM = 2
    // where wide tiles measured faster (FP32 passes, FP64 fused with real
    // psi); plans of 192 threads or more keep LM = 1 there (measured at
    // 256^3 and 192^3).  FP32 xconv always takes LM = 2, the other FP64
    // passes LM = 1.
    template <typename Pl>
    static constexpr int wide() { return FftTile<Pl, 1>::WG < 192 ? 2 : 1; }

    template <int LM>
    static hipError_t zfwd_t(const FftArgs &a) {
        using Tl = FftTile<FftPlan<N>, LM>;
        const int ytiles = (int)((a.Ny + 2 * Tl::L - 1) / (2 * Tl::L));
        dim3 grid((unsigned)(a.Nx * ytiles), (unsigned)a.v.nb), block(Tl::WG);
        const int Nx = (int)a.Nx, Ny = (int)a.Ny;
        if (!a.fp32) {
            auto *tw = static_cast<const cpx<double> *>(a.tw);
            if (a.cpsi) k_zfwd<N, double, cpx<double>, LM><<<grid, block, 0, a.stream>>>(a.v, Nx, Ny, tw, a.wx, a.tiles);
            else k_zfwd<N, double, double, LM><<<grid, block, 0, a.stream>>>(a.v, Nx, Ny, tw, a.wx, a.tiles);
        } else {
            auto *tw = static_cast<const cpx<float> *>(a.tw);
            if (a.cpsi) k_zfwd<N, float, cpx<float>, LM><<<grid, block, 0, a.stream>>>(a.v, Nx, Ny, tw, a.wx, a.tiles);
            else k_zfwd<N, float, float, LM><<<grid, block, 0, a.stream>>>(a.v, Nx, Ny, tw, a.wx, a.tiles);
        }
        return hipGetLastError();
    }
    // The tile multiplier of a pass: the environment variable, else the
    // context's tuned choice, else the rule.
    static int pick_lm(const FftArgs &a, int env, int pass, int rule) {
        if (env) return env;
        return a.tune.lm[pass] ? a.tune.lm[pass] : rule;
    }
    static hipError_t zfwd(const FftArgs &a) {
        static const int l64 = fft_lm("DBEC_FFT_LM_ZFWD64", 0), l32 = fft_lm("DBEC_FFT_LM_ZFWD32", 0);
        return pick_lm(a, a.fp32 ? l32 : l64, 0, a.fp32 ? wide<FftPlan<N>>() : 1) == 2 ? zfwd_t<2>(a) : zfwd_t<1>(a);
    }
    // FP32 spectra use tiles twice as wide, so every strided access still
    // moves 128-256 contiguous bytes.

    template <typename R, int LM, typename Pl = YPlan<N, R>>
    static hipError_t ypass_t(int dir, const FftArgs &a) {
        if constexpr (kF32<R> && !std::is_same<Pl, FftPlan<N>>::value)
            if (a.phi_plans) return ypass_t<R, LM, FftPlan<N>>(dir, a);
        using Tl = FftTile<Pl, LM>;
        const long nlines = a.Nkz * a.Nx;
        dim3 grid((unsigned)((nlines + Tl::L - 1) / Tl::L), (unsigned)a.v.nb), block(Tl::WG);
        auto *tw = static_cast<const cpx<R> *>(a.tw);
        if (dir < 0) k_ypass<N, -1, R, LM, Pl><<<grid, block, 0, a.stream>>>(a.v, nlines, tw, a.wx, a.tiles, (int)a.Nx);
        else k_ypass<N, +1, R, LM, Pl><<<grid, block, 0, a.stream>>>(a.v, nlines, tw, a.wx, a.tiles, (int)a.Nx);
        return hipGetLastError();
    }
    static hipError_t ypass(int dir, const FftArgs &a) {
        static const int l64 = fft_lm("DBEC_FFT_LM_YPASS64", 0), l32 = fft_lm("DBEC_FFT_LM_YPASS32", 0);
        const bool two = pick_lm(a, a.fp32 ? l32 : l64, 1, a.fp32 ? wide<YPlan<N, float>>() : 1) == 2;
        if (a.fp32) return two ? ypass_t<float, 2>(dir, a) : ypass_t<float, 1>(dir, a);
        return two ? ypass_t<double, 2>(dir, a) : ypass_t<double, 1>(dir, a);
    }

    template <typename R, int LM, typename Pl = XPlan<N, R>>
    static hipError_t xconv_t(const FftArgs &a) {
        if constexpr ((kF32<R> || kXPlanLines<N, R> > 0) && !std::is_same<Pl, FftPlan<N>>::value)
            if ((kF32<R> && a.phi_plans) || a.Nkz * a.Ny <= kXPlanLines<N, R>) return xconv_t<R, LM, FftPlan<N>>(a);
        using Tl = FftTile<Pl, LM>;
        const int ytiles = (int)((a.Ny + Tl::L - 1) / Tl::L);
        dim3 grid((unsigned)(a.Nkz * ytiles), (unsigned)a.v.nb), block(Tl::WG);
        const auto launch = [&](auto planes) {
            k_xconv<N, R, LM, decltype(planes)::value, Pl><<<grid, block, 0, a.stream>>>(
                a.v, static_cast<const R *>(a.potddq), (int)a.Ny, static_cast<const cpx<R> *>(a.tw), a.wx, a.yq);
        };
        if (a.yq) launch(std::true_type{});
        else launch(std::false_type{});
        return hipGetLastError();
    }
    static hipError_t xconv(const FftArgs &a) {
        static const int l64 = fft_lm("DBEC_FFT_LM_XCONV64", 0), l32 = fft_lm("DBEC_FFT_LM_XCONV32", 0);
        const bool two = pick_lm(a, a.fp32 ? l32 : l64, 2, a.fp32 ? 2 : 1) == 2;
        if (a.fp32) return two ? xconv_t<float, 2>(a) : xconv_t<float, 1>(a);
        return two ? xconv_t<double, 2>(a) : xconv_t<double, 1>(a);
    }

    template <typename S, typename R, bool COLS, int L, bool HALF>
    static hipError_t sweepz_zfwd_t(const FftArgs &a) {
        using A = typename Arith<S>::T;
        if constexpr (!FusedZ<N, HALF>::template fits<S, R, L>()) {
            return hipErrorInvalidValue;
        } else {
            const int yt = (int)((a.Ny + L - 1) / L);
            dim3 grid((unsigned)(a.Nx * yt), (unsigned)a.v.nb), block(L * (N / 16));
            using TT = typename TabOf<A>::T;
            const SweepTab<A> tab{static_cast<const TT *>(a.ztab[0]), static_cast<const TT *>(a.ztab[1]),
                                  static_cast<const TT *>(a.ztab[2]), static_cast<const TT *>(a.ztab[3])};
            SweepConst<A> k;
            zconst(a, k);
            const bool reversed = z_reversed(COLS, (long)a.v.nb * a.Nx * a.Ny * N * (long)sizeof(S));
            k_sweepz_zfwd<N, S, R, L, COLS, HALF><<<grid, block, 0, a.stream>>>(
                a.v, (int)a.Nx, (int)a.Ny, tab, k, a.wz, a.wy, static_cast<const cpx<R> *>(a.tw), reversed);
            return hipGetLastError();
        }
    }
    static void zconst(const FftArgs &a, SweepConst<double> &k) {
        k.A0r = a.zk[0][0];
        k.A = a.zk[1][0];
        k.mA = a.zk[2][0];
    }
    static void zconst(const FftArgs &a, SweepConst<float> &k) {
        k.A0r = (float)a.zk[0][0];
        k.A = (float)a.zk[1][0];
        k.mA = (float)a.zk[2][0];
    }
    static void zconst(const FftArgs &a, SweepConst<cpx<double>> &k) {
        k.A0r = {a.zk[0][0], a.zk[0][1]};
        k.A = {a.zk[1][0], a.zk[1][1]};
        k.mA = {a.zk[2][0], a.zk[2][1]};
    }
    static void zconst(const FftArgs &a, SweepConst<cpx<float>> &k) {
        k.A0r = {(float)a.zk[0][0], (float)a.zk[0][1]};
        k.A = {(float)a.zk[1][0], (float)a.zk[1][1]};
        k.mA = {(float)a.zk[2][0], (float)a.zk[2][1]};
    }
    template <typename S, typename R, bool COLS, bool HALF>
    static hipError_t sweepz_zfwd_rows(const FftArgs &a, int rows) {
        switch (rows) {
        case 64: return sweepz_zfwd_t<S, R, COLS, 64, HALF>(a);
        case 32: return sweepz_zfwd_t<S, R, COLS, 32, HALF>(a);
        case 16: return sweepz_zfwd_t<S, R, COLS, 16, HALF>(a);
        case 8: return sweepz_zfwd_t<S, R, COLS, 8, HALF>(a);
        default: return hipErrorInvalidValue;
        }
    }
    template <typename S, typename R, bool HALF>
    static int per_cu(int zrows) {
        switch (zrows) {
        case 64: return FusedZ<N, HALF>::template per_cu<S, R, 64>();
        case 32: return FusedZ<N, HALF>::template per_cu<S, R, 32>();
        case 16: return FusedZ<N, HALF>::template per_cu<S, R, 16>();
        case 8: return FusedZ<N, HALF>::template per_cu<S, R, 8>();
        default: return 0;
        }
    }
    // Whole or half tiles (of complex rows that have both; the results are the
    // same).  Half tiles put more rows on a CU, but each row takes two turns
    // more at the barriers: whole ones serve a launch that needs no more
    // rounds of the chip with them, in FP64 up to two rounds, in FP32 one.
    // Measured, half / whole (us): complex FP64 64x32x160 13.4 / 11.0,
    // 48x160x160 17.6 / 15.0, 48x160x320 35.0 / 31.3 (one, one and two rounds
    // with either), 160x64x160 21.2 / 22.2, 96x160x256 34.6 / 41.8 (one with
    // half, two with whole tiles); complex FP32 160x64x256 15.3 / 14.0,
    // 96x160x256 18.1 / 20.7, and two rounds with either at 160x64x512
    // 28.5 / 30.3, 96x160x384 31.5 / 32.6.
    template <typename S, typename R, bool COLS>
    static hipError_t sweepz_zfwd_tile(const FftArgs &a) {
        const int kw = per_cu<S, R, false>(a.zrows), kh = per_cu<S, R, true>(a.zrows_half);
        const auto rounds = [&](int rows, int k) {
            const long wgs = (long)a.v.nb * a.Nx * ((a.Ny + rows - 1) / rows), all = 256L * k;
            return (wgs + all - 1) / all;
        };
        bool half = kw == 0;
        if (kw && kh) {
            const long w = rounds(a.zrows, kw);
            half = w > rounds(a.zrows_half, kh) || w > (sizeof(R) == 8 ? 2 : 1);
        }
        if (!half) return sweepz_zfwd_rows<S, R, COLS, false>(a, a.zrows);
        if constexpr (fused_z_half<S>(N)) return sweepz_zfwd_rows<S, R, COLS, true>(a, a.zrows_half);
        else return hipErrorInvalidValue;
    }
    static hipError_t sweepz_zfwd(const FftArgs &a) {
        if (!a.fp32) return a.cpsi ? sweepz_zfwd_tile<cpx<double>, double, false>(a) : sweepz_zfwd_tile<double, double, true>(a);
        return a.cpsi ? sweepz_zfwd_tile<cpx<float>, float, false>(a) : sweepz_zfwd_tile<float, float, true>(a);
    }
    template <typename S, typename R>
    static bool has_rows(int whole, int half) { return per_cu<S, R, false>(whole) || per_cu<S, R, true>(half); }
    static bool fusable(bool fp32, bool cpsi, int rows, int rows_half) {
        if (!fp32) return cpsi ? has_rows<cpx<double>, double>(rows, rows_half) : has_rows<double, double>(rows, rows_half);
        return cpsi ? has_rows<cpx<float>, float>(rows, rows_half) : has_rows<float, float>(rows, rows_half);
    }

    // single solve: spectrum of `one` -> phi
    static hipError_t zinv(const FftArgs &a) {
        using Tl = FftTile<FftPlan<N>, 1>;
        const int ytiles = (int)((a.Ny + 2 * Tl::L - 1) / (2 * Tl::L));
        dim3 grid((unsigned)(a.Nx * ytiles)), block(Tl::WG);
        if (!a.fp32)
            k_zinv<N, double, 1><<<grid, block, 0, a.stream>>>(static_cast<const cpx<double> *>(a.v.spec),
                                                               static_cast<double *>(a.phi), (int)a.Nx, (int)a.Ny,
                                                               static_cast<const cpx<double> *>(a.tw));
        else
            k_zinv<N, float, 1><<<grid, block, 0, a.stream>>>(static_cast<const cpx<float> *>(a.v.spec),
                                                              static_cast<float *>(a.phi), (int)a.Nx, (int)a.Ny,
                                                              static_cast<const cpx<float> *>(a.tw));
        return hipGetLastError();
    }

    template <typename P, typename R, int LM, typename Pl = ZPlan<N, P>>
    static hipError_t fused_t(const FftArgs &a) {
        if constexpr (kZPlanRows<N, P> > 0 && !std::is_same<Pl, FftPlan<N>>::value)
            if (a.Nx * a.Ny <= kZPlanRows<N, P>) return fused_t<P, R, LM, FftPlan<N>>(a);
        using Tl = FftTile<Pl, LM, kZHalf<N, P>>;
        const auto *tw = static_cast<const cpx<R> *>(a.tw);
        const int ytiles = (int)((a.Ny + 2 * Tl::L - 1) / (2 * Tl::L));
        const int nmain = (int)((a.Nx - 1) * ytiles);
        const int nfaceb = (int)((a.Ny + a.Nx - 1 + Tl::L - 1) / Tl::L);
        dim3 grid((unsigned)(nmain + nfaceb), (unsigned)a.v.nb), block(Tl::WG);
        // FP32 spectra load straight into the first pass's registers (faster at
        // every measured size); FP64 ones through LDS (the extra registers
        // cost more occupancy than the LDS round trip saves).  FP64 has both
        // transform buffer layouts (swizzled: real psi faster at 256, slower
        // at 160 and 192; complex psi, twiddles from the global table, 234 ->
        // 215 us at 256x256x384, slower at 192): the environment variable,
        // else the tuned choice, else padded.
        constexpr bool ZREG = std::is_same<R, float>::value;
        if constexpr (std::is_same<R, double>::value) {
            static const int env = fft_swz_env();
            if (env >= 0 ? env == 1 : a.tune.zinv_swz == 1) {
                k_zinv_nu<N, R, P, LM, ZREG, true, Pl><<<grid, block, 0, a.stream>>>(a.v, a.sq, a.nc, (int)a.Nx,
                                                                                      (int)a.Ny, nfaceb, tw);
                return hipGetLastError();
            }
        }
        k_zinv_nu<N, R, P, LM, ZREG, false, Pl><<<grid, block, 0, a.stream>>>(a.v, a.sq, a.nc, (int)a.Nx, (int)a.Ny,
                                                                               nfaceb, tw);
        return hipGetLastError();
    }
    template <int LM>
    static hipError_t fused_lm(const FftArgs &a) {
        if (!a.fp32) return a.cpsi ? fused_t<cpx<double>, double, LM>(a) : fused_t<double, double, LM>(a);
        return a.cpsi ? fused_t<cpx<float>, float, LM>(a) : fused_t<float, float, LM>(a);
    }
    static hipError_t fused(const FftArgs &a) {
        // FP64: narrow tiles for complex psi
        static const int l64 = fft_lm("DBEC_FFT_LM_FUSED64", 0), l32 = fft_lm("DBEC_FFT_LM_FUSED32", 0);
        const int rule = !a.fp32 ? (a.cpsi ? 1 : wide<ZPlan<N, double>>())
                                 : (a.cpsi ? wide<ZPlan<N, cpx<float>>>() : wide<ZPlan<N, float>>());
        const int lm = pick_lm(a, a.fp32 ? l32 : l64, 3, rule);
        return lm == 2 ? fused_lm<2>(a) : fused_lm<1>(a);
    }
};

template <int N>
hipError_t FftLaunch<N>::zfwd(const FftArgs &a) { return FftLaunchImpl<N>::zfwd(a); }
template <int N>
hipError_t FftLaunch<N>::ypass(int dir, const FftArgs &a) { return FftLaunchImpl<N>::ypass(dir, a); }
template <int N>
hipError_t FftLaunch<N>::xconv(const FftArgs &a) { return FftLaunchImpl<N>::xconv(a); }
template <int N>
hipError_t FftLaunch<N>::zinv(const FftArgs &a) { return FftLaunchImpl<N>::zinv(a); }
template <int N>
hipError_t FftLaunch<N>::fused(const FftArgs &a) { return FftLaunchImpl<N>::fused(a); }
template <int N>
hipError_t FftLaunch<N>::sweepz_zfwd(const FftArgs &a) { return FftLaunchImpl<N>::sweepz_zfwd(a); }
template <int N>
bool FftLaunch<N>::fusable(bool fp32, bool cpsi, int rows, int rows_half) {
    return FftLaunchImpl<N>::fusable(fp32, cpsi, rows, rows_half);
}

}  // namespace dbec
