// plane.hip - split-step kernels that hold a whole (y, z) plane of one x in
// LDS, for grids whose planes are small enough (plane_ok).
//
//   k_plane_fwd : y sweep, z sweep, Simpson partial of the plane, then
//                 |psi|^2 and its z and y transforms: the end of one step and
//                 the start of the next one's convolution in one launch;
//                 also without the sweeps (start of a dbec_step call) and
//                 without the transforms (its end).
//   k_plane_inv : inverse y and z transforms, then calcnu on psi (or phi
//                 itself, for the standalone calcpsidd2), with the periodic
//                 face copies.
//
// With the x convolution and the x sweep a step is four launches instead of
// eight (seven where the z sweep fuses with the next forward z pass), and the
// half spectrum crosses HBM four times instead of eight, psi six times
// instead of eight.  At these sizes a launch is bound by its own start and the
// latency of its chain of loads, barriers and recurrences (4-8 us each at
// 64^3 and 128x96x80 whatever its bytes), so the number of launches decides.
// One workgroup of Ny Nz / 16 threads per x plane and solve: each thread holds
// one 16-point segment of a line in the sweeps, as in the other sweep kernels,
// and one butterfly per pass in the transforms (the real bins 0 and Nz/2 share
// a complex line, or one pass in eight would run a second round for the last
// line).  With one or two wavefronts per SIMD the vector unit's own rate
// counts: index arithmetic is in 24-bit multiplies and no array may land in
// scratch memory (plane_inv at 64^3 FP64 14.5 us with the staged spectrum there,
// 10 without).  Measured at 64^3 FP64: fwd 12.5 us for the y sweep, z sweep,
// forward z and y passes (4.3 + 6.0 + 5.0 + 4.6 us apart), inv 10 us (4.3 + 6.5
// apart); steps at plane_ok.
//
// The spectrum between the two kernels is in digit order along y (fft_slot):
// the x convolution only has to know which |ky| a slot holds (FftArgs::yq).
#include <algorithm>
#include <atomic>

#include "ops.hpp"
#include "plane_device.hpp"
#include "sweep_device.hpp"

namespace dbec {

namespace {

// psi's |psi|^2 as the forward z passes form it (fft_kernels.hpp).
__device__ __forceinline__ double plane_mod2(double v, double s) {
    const double t = v * s;
    return t * t;
}
__device__ __forceinline__ double plane_mod2(float v, double s) {
    const double t = (double)v * s;
    return t * t;
}
__device__ __forceinline__ double plane_mod2(cpx<double> v, double) { return fma(v.x, v.x, v.y * v.y); }
__device__ __forceinline__ double plane_mod2(cpx<float> v, double) { return v.x * v.x + v.y * v.y; }

struct PlaneDims {
    int Nx, Ny, Nz, qy, qz, nt;
    FastDiv dNy, dNyh, dNz, dNzh, dqy;
    // inverse kernel: workgroups per plane, their share of the rows (qy / parts
    // butterflies), and as divisors
    int parts, nj, extra;  // extra: 1 with an extra plane's workgroups
    FastDiv dparts, dnj, dlines;
};

// Workgroups go to the 8 XCDs round robin; block b takes item (b % 8) * per +
// b / 8, so an XCD works on a run of neighbouring planes: their spectrum rows
// differ in the address bits that select its L2 channels (with x = b, the
// planes of one XCD are 8 rows apart, a multiple of 4 KiB at common Ny, and
// crowd a few channels), and the parts of a plane share that L2.
__device__ __forceinline__ int xcd_item(int n) {
    const int per = (n + 7) / 8;
    return (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
}
inline unsigned xcd_blocks(long n) { return (unsigned)((n + 7) / 8 * 8); }

template <typename A>
struct PlaneSweep {
    SweepTab<A> ty, tz;
    SweepConst<A> ky, kz;
    const double *wz, *wy;
};

constexpr size_t up16(size_t b) { return (b + 15) & ~size_t(15); }

// LDS of the plane kernels: small arrays, then the main region that holds in
// turn the carry exchange, the psi tile, the z lines and the half spectrum.
template <typename S, typename R>
struct PlaneLds {
    using A = typename Arith<S>::T;
    size_t ty, tz, twy, twz, exl, red, main, total;
    __host__ __device__ PlaneLds(int Ny, int Nz, int bd, bool sweeps, bool fft) {
        using SH = SweepShared<A, 16>;
        ty = 0;
        tz = ty + (sweeps ? up16(4 * (size_t)SH::tab_len(Ny) * sizeof(A)) : 0);
        twy = tz + (sweeps ? up16(4 * (size_t)SH::tab_len(Nz) * sizeof(A)) : 0);
        twz = twy + (fft ? up16((size_t)Ny * sizeof(cpx<R>)) : 0);
        exl = twz + (fft ? up16((size_t)Nz * sizeof(cpx<R>)) : 0);
        const int m = Ny > Nz ? Ny : Nz;
        red = exl + (sweeps ? up16((size_t)m * sizeof(A)) : 0);
        main = red + 16 * sizeof(double);
        const size_t tile = (size_t)Ny * (Nz + Pk<S>::n) * sizeof(S);
        const size_t zb = (size_t)Nz * (Ny / 2 + 1) * sizeof(cpx<R>);
        const size_t sp = (size_t)Ny * (Nz / 2 + 1) * sizeof(cpx<R>);
        size_t w = 0;
        if (sweeps) {
            w = tile;
            const size_t ex = 2 * (size_t)bd * sizeof(A);
            w = w > ex ? w : ex;
        }
        if (fft) {
            w = w > zb ? w : zb;
            w = w > sp ? w : sp;
        }
        total = main + up16(w);
    }
};

// wavefronts per SIMD a kernel is built for: two workgroups of 640 threads per
// CU in FP32
template <typename R, int MAXT>
constexpr int plane_waves() { return sizeof(R) == 4 && MAXT == 640 ? 6 : 1; }

constexpr int KPSI = 16;  // a plane's points per thread: threads >= Ny Nz / 16
constexpr int KSPEC = 8;  // its spectrum lines' elements per thread

template <typename S, typename R, bool SW, bool FF, int MAXT>
__global__ void __launch_bounds__(MAXT, (plane_waves<R, MAXT>()))
k_plane_fwd(Solves v, PlaneDims g, PlaneSweep<typename Arith<S>::T> k, const cpx<R> *__restrict__ twyg,
            const cpx<R> *__restrict__ twzg) {
    using A = typename Arith<S>::T;
    constexpr int M = 16, VE = Pk<S>::n, KV = M / VE;
    constexpr bool COLS = std::is_floating_point<S>::value;
    extern __shared__ __align__(16) char smem_raw[];
    const int tid = threadIdx.x, bd = blockDim.x;
    const int Ny = g.Ny, Nz = g.Nz, x = xcd_item(g.Nx);
    if (x >= g.Nx) return;
    const PlaneLds<S, R> lay(Ny, Nz, bd, SW, FF);
    const SolveAt sr = solve_at(v);
    S *__restrict__ psi = reinterpret_cast<S *>(sr.psi) + (long)x * Ny * Nz;
    cpx<R> *twy = reinterpret_cast<cpx<R> *>(smem_raw + lay.twy), *twz = reinterpret_cast<cpx<R> *>(smem_raw + lay.twz);
    char *main = smem_raw + lay.main;
    cpx<R> *zb = reinterpret_cast<cpx<R> *>(main);
    const int LP = Ny / 2 + 1, Nyh = Ny / 2, SK = Nz / 2 + 1;
    // Every table entry a thread stages (Ny, Nz <= threads: one of each) is
    // loaded before the plane's data, so writing it to LDS waits for no load
    // issued later.
    cpx<R> wy{}, wz{};
    if constexpr (FF) {
        wy = twyg[tid < Ny ? tid : 0];
        wz = twzg[tid < Nz ? tid : 0];
    }
    const auto put_twiddles = [&] {
        if constexpr (FF) {
            if (tid < Ny) twy[tid] = wy;
            if (tid < Nz) twz[tid] = wz;
        }
    };
    if constexpr (SW) {
        // Threads past the segments repeat the work of thread t (the same
        // values to the same places), so all of them meet the barriers.
        const int t = tid < g.nt ? tid : tid % g.nt;
        const int RS = Nz + VE;
        S *tile = reinterpret_cast<S *>(main);
        const A zero = m_zero(k.ky.A);
        A vv[M];
        {
            int s, l;
            g.dNz.divmod(t, s, l);
            const int e0 = s * M;
            const S *seg = psi + m24(e0, Nz) + l;
            const CoefPre<A> cy = coef_pre(k.ty, Ny, tid), cz = coef_pre(k.tz, Nz, tid);
#pragma unroll
            for (int j = 0; j < M; ++j) vv[j] = to_a(seg[j * Nz]);
            const A hl = e0 > 0 ? to_a(seg[-Nz]) : zero;
            const A hr = e0 + M < Ny ? to_a(seg[M * Nz]) : zero;
            SweepShared<A, M> shy(smem_raw + lay.ty, Ny, bd, 0), shz(smem_raw + lay.tz, Nz, bd, 0);
            coef_put(shy, cy, k.ty, Ny, tid, bd);
            coef_put(shz, cz, k.tz, Nz, tid, bd);
            put_twiddles();
            shy.exa = reinterpret_cast<A *>(main);
            shy.exb = shy.exa + bd;
            shy.exl = reinterpret_cast<A *>(smem_raw + lay.exl);
            __syncthreads();
            seg_solve<A, M, false, true>(vv, hl, hr, e0, Ny, s, l, Nz, Ny / M, shy, k.ky, nullptr);
            __syncthreads();  // carries read: the region takes the tile
#pragma unroll
            for (int j = 0; j < M; ++j) tile[m24(e0, RS) + j * RS + l] = from_a<S>(vv[j]);
        }
        __syncthreads();
        int s, l;
        g.dNy.divmod(t, s, l);
        const int e0 = s * M;
        {
            const S *row = tile + m24(l, RS);
#pragma unroll
            for (int q = 0; q < KV; ++q) {
                const typename Pk<S>::type pk = ld_pk(row + e0 + q * VE);
#pragma unroll
                for (int j = 0; j < VE; ++j) vv[q * VE + j] = to_a(pk.e[j]);
            }
            const A hl = e0 > 0 ? to_a(row[e0 - 1]) : zero;
            const A hr = e0 + M < Nz ? to_a(row[e0 + M]) : zero;
            __syncthreads();  // the tile is in registers
            SweepShared<A, M> shz(smem_raw + lay.tz, Nz, bd, 0);
            shz.exa = reinterpret_cast<A *>(main);
            shz.exb = shz.exa + bd;
            shz.exl = reinterpret_cast<A *>(smem_raw + lay.exl);
            const double acc = seg_solve<A, M, COLS, true>(vv, hl, hr, e0, Nz, s, l, Ny, Nz / M, shz, k.kz, k.wz);
            __syncthreads();  // carries read
            S *orow = tile + m24(l, RS);
#pragma unroll
            for (int q = 0; q < KV; ++q) {
                typename Pk<S>::type o;
#pragma unroll
                for (int j = 0; j < VE; ++j) o.e[j] = from_a<S>(vv[q * VE + j]);
                st_pk(orow + e0 + q * VE, o);
            }
            if constexpr (COLS) {
                double *red = reinterpret_cast<double *>(smem_raw + lay.red);
                const double w = wave_sum(tid < g.nt ? k.wy[l] * acc : 0.0);
                if ((tid & 63) == 0) red[tid >> 6] = w;
            }
        }
        __syncthreads();
        if constexpr (COLS) {
            if (tid == 0) {
                const double *red = reinterpret_cast<const double *>(smem_raw + lay.red);
                double w = 0.0;
                for (int i = 0; i < bd >> 6; ++i) w += red[i];
                sr.rows[x] = w;
            }
        }
        const int npr = Nz / VE;  // packets per row
        for (int i = tid; i < Ny * npr; i += bd) {
            const int e = i * VE, row = g.dNz.div(e);
            st_pk(psi + e, ld_pk(tile + e + row * VE));  // rows of Nz + VE
        }
        if constexpr (FF) {
            __syncthreads();  // the tile is stored: the region takes the z lines
            int r, jq;
            g.dqy.divmod(l, r, jq);
            R *slot = reinterpret_cast<R *>(&zb[m24(e0, LP) + m24(r >> 1, g.qy) + jq]) + (r & 1);
#pragma unroll
            for (int j = 0; j < M; ++j) slot[2 * j * LP] = (R)plane_mod2(from_a<S>(vv[j]), 1.0);
        }
    } else {
        const double sc = v.use_scale ? sr.scal[SC_SCALE] : 1.0;
#pragma unroll 4
        for (int i = tid; i < Nyh * Nz; i += bd) {
            int p, z, t, jq;
            g.dNz.divmod(i, p, z);
            g.dqy.divmod(p, t, jq);
            const S *row = psi + m24(jq + m24(2 * t, g.qy), Nz) + z;  // rows y and y + qy are line p
            const S a = row[0], b = row[m24(g.qy, Nz)];
            zb[m24(z, LP) + p] = {(R)plane_mod2(a, sc), (R)plane_mod2(b, sc)};
        }
        put_twiddles();
    }
    if constexpr (FF) {
        __syncthreads();
        fft_lines<-1>(zb, LP, g.dNyh, g.qz, twz, tid, bd);
        // The spectra of the two rows of a line, A[k] = (Z[k] + conj Z[N-k]) /
        // 2 and B[k] = (Z[k] - conj Z[N-k]) / (2i), go straight into the first
        // pass along y: its butterfly j takes the rows j + qy r, which are the
        // lines t qy + j, t = 0..3.  The bins 0 and Nz/2 are real and run as
        // one complex line (its real and imaginary parts), so there are Nz/2
        // lines, one butterfly per thread.  Through registers, since the
        // spectrum takes the z lines' region.
        const int q = g.qy, h = Nz / 2, i0 = tid;
        cpx<R> o[8];
        int kz0, j0;
        g.dqy.divmod(i0 < g.nt ? i0 : 0, kz0, j0);
        {
            const cpx<R> *zp = zb + m24(fft_slot(kz0, g.qz), LP) + j0, *wp = zb + m24(fft_slot(kz0 ? Nz - kz0 : h, g.qz), LP) + j0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const cpx<R> z = zp[t * q], w = wp[t * q];
                const bool dc = kz0 == 0;
                o[2 * t] = {dc ? z.x : R(0.5) * (z.x + w.x), dc ? w.x : R(0.5) * (z.y - w.y)};
                o[2 * t + 1] = {dc ? z.y : R(0.5) * (z.y + w.y), dc ? w.y : R(0.5) * (w.x - z.x)};
            }
            dft8<-1>(o);
#pragma unroll
            for (int c = 1; c < 8; ++c) o[c] = cmul(o[c], twy[m24(j0, c)]);
        }
        __syncthreads();
        if (i0 < g.nt) {
            cpx<R> *sp = zb + m24(j0, SK) + kz0;
            const int qs = m24(q, SK);
#pragma unroll
            for (int c = 0; c < 8; ++c) sp[c * qs] = o[c];
        }
        __syncthreads();
        passq<-1>(zb, SK, g.dNzh, q, twy, tid, bd);
        __syncthreads();
        cpx<R> *__restrict__ spec = reinterpret_cast<cpx<R> *>(sr.spec) + (long)x * Ny;
        const unsigned plane = (unsigned)(g.Nx * Ny);
        for (int i = tid; i < m24(h, Ny); i += bd) {
            int kz, y;
            g.dNy.divmod(i, kz, y);
            cpx<R> v = zb[m24(y, SK) + kz];
            if (kz == 0) {  // line 0: bin 0 plus i times bin Nz/2, both even under ky -> -ky with conjugation
                int c, d;
                g.dqy.divmod(y, c, d);
                const int ky = c + 8 * d, n = ky ? Ny - ky : 0;
                const cpx<R> w = zb[m24(fft_slot(n, q), SK)];
                spec[__umul24(h, plane) + y] = {R(0.5) * (v.y + w.y), R(0.5) * (w.x - v.x)};
                v = {R(0.5) * (v.x + w.x), R(0.5) * (v.y - w.y)};
            }
            spec[__umul24(kz, plane) + y] = v;
        }
    }
}

// P: psi's type; with PHI the potential goes to phi instead of into calcnu.
// Periodic face copies (calcpsidd2_kernel2a/2b, imag3d.cu:1591-1625).  Plane
// x < Nx-1: row y < Ny-1 takes its point z = Nz-1 from z = 0; row Ny-1 takes
// its points z < Nz-1 from row 0.  Plane Nx-1: the points y < Ny-1, z < Nz-1
// come from plane 0: an extra plane's workgroups transform plane 0 once more
// and write them (g.extra), or plane 0's own do so in a second round, where
// the extra ones would be the ones that do not fit the chip in the first round
// (a 257th workgroup at 256x64x64 FP64: 27 us instead of 21; at 96^3 FP64 the
// second round costs 18 us instead of 14).  The rest of plane Nx-1 comes from
// the plane itself.
//
// A plane's rows may be shared by `parts` workgroups: each does the first pass
// along y of the whole plane, then the rows j + qy r of its own butterflies j.
// Which rows pair into a complex z line does not depend on it, so neither does
// the result.  SPLIT: two parts or more.
template <typename P, typename R, bool PHI, bool SPLIT, int MAXT>
__global__ void __launch_bounds__(MAXT, (plane_waves<R, MAXT>()))
k_plane_inv(Solves v, PlaneDims g, const double *__restrict__ sq, NuConst nc, R *__restrict__ phi,
            const cpx<R> *__restrict__ twyg, const cpx<R> *__restrict__ twzg) {
    constexpr int KG = (SPLIT ? KPSI / 2 : KPSI) / 4;  // groups of 4 points per thread
    constexpr int PRE = SPLIT ? KG : 1;               // of which loaded ahead of the z transform
    extern __shared__ __align__(16) char smem_raw[];
    const int tid = threadIdx.x, bd = blockDim.x;
    const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz, q = g.qy, nj = g.nj;
    int part;
    const int item = xcd_item((Nx + g.extra) * g.parts);
    if (item >= (Nx + g.extra) * g.parts) return;
    int x;
    g.dparts.divmod(item, x, part);
    const bool extra = x == Nx;
    if (extra) x = 0;
    const int j0 = part * nj;
    const int nl = 4 * nj, LP = nl + 1, h = Nz / 2, SK = h + 1;  // nl: z lines of this part
    double *sqz = reinterpret_cast<double *>(smem_raw), *sqr = sqz + Nz;  // trap_z, trap_xy of the plane and of plane Nx-1
    cpx<R> *twy = reinterpret_cast<cpx<R> *>(sqr + 2 * Ny), *twz = twy + Ny;
    cpx<R> *zb = twz + Nz;
    const SolveAt sr = solve_at(v);
    const cpx<R> *__restrict__ spec = reinterpret_cast<const cpx<R> *>(sr.spec) + x * Ny;
    const unsigned plane = (unsigned)(Nx * Ny);
    // small tables first (Ny, Nz <= threads), then everything else in flight
    // at once: the first wait is for the oldest loads only
    const cpx<R> wy = twyg[tid < Ny ? tid : 0], wz = twzg[tid < Nz ? tid : 0];
    double x2 = 0.0, xf2 = 0.0, y2 = 0.0, z2 = 0.0;
    if constexpr (!PHI) {
        x2 = sq[x];
        xf2 = sq[Nx - 1];
        y2 = sq[Nx + (tid < Ny ? tid : 0)];
        z2 = sq[Nx + Ny + (tid < Nz ? tid : 0)];
    }
    const int se = m24(h, Ny);
    R rx[KSPEC], ry[KSPEC];  // (an array of cpx ended up in scratch memory)
#pragma unroll
    for (int u = 0; u < KSPEC; ++u) {
        const int i = tid + u * bd;
        int kz, y;
        g.dNy.divmod(i < se ? i : 0, kz, y);
        const cpx<R> t = spec[__umul24(kz, plane) + y];
        rx[u] = t.x;
        ry[u] = t.y;
    }
    const cpx<R> sh = spec[__umul24(h, plane) + (tid < Ny ? tid : 0)];  // bin Nz/2
    // The points this workgroup writes: its rows, and for part 0 of a plane x
    // < Nx-1 the points z < Nz-1 of row Ny-1, which take row 0's potential.
    // Their psi is loaded after the first pass along y, in flight during the
    // others.
    const long far = (long)(Nx - 1) * Ny * Nz;
    P *__restrict__ psi = reinterpret_cast<P *>(sr.psi) + (extra ? far : (long)x * Ny * Nz);
    const int points = 8 * nj * Nz;
    const bool rim = !extra && x < Nx - 1 && part == 0 && tid < Nz - 1;
    const auto place = [&](int i, int &lr, int &y, int &z) {
        int r, jj;
        g.dNz.divmod(i, lr, z);
        g.dnj.divmod(lr, r, jj);
        y = j0 + jj + m24(q, r);
    };
    const TrapConst tc = sr.p.tc;
    if (tid < Ny) {
        twy[tid] = wy;
        if constexpr (!PHI) {
            sqr[tid] = trap_xy(tc, x2, y2);
            sqr[Ny + tid] = trap_xy(tc, xf2, y2);
        }
    }
    if (tid < Nz) {
        twz[tid] = wz;
        if constexpr (!PHI) sqz[tid] = trap_z(tc, z2);
    }
    if (tid < Ny) {  // kz = 0: bins 0 and Nz/2 as one line, S0 + i Sh
        rx[0] -= sh.y;
        ry[0] += sh.x;
    }
#pragma unroll
    for (int u = 0; u < KSPEC; ++u) {
        const int i = opaque(tid) + u * bd;
        if (i < se) {
            int kz, y;
            g.dNy.divmod(i, kz, y);
            zb[m24(y, SK) + kz] = {rx[u], ry[u]};
        }
    }
    __syncthreads();
    passq<+1>(zb, SK, g.dNzh, q, twy, tid, bd);
    P pv[KG][4], pr;
    const auto load_psi = [&](int gr) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int i = opaque(tid) + (4 * gr + w) * bd;
            int lr, y, z;
            place(i < points ? i : 0, lr, y, z);
            pv[gr][w] = psi[m24(y, Nz) + z];
        }
    };
    if constexpr (!PHI) {
#pragma unroll
        for (int gr = 0; gr < PRE; ++gr) load_psi(gr);
        pr = psi[(Ny - 1) * Nz + (rim ? tid : 0)];
    }
    __syncthreads();
    // Last pass along y of this part's butterflies, and the complex z lines of
    // its row pairs: Z[k] = A[k] + i B[k], Z[N-k] = conj A[k] + i conj B[k];
    // line 0 holds the (real) bins 0 and Nz/2 in its real and imaginary parts.
    cpx<R> o[8];
    const int items = m24(nj, h);
    int kz0, jj0;
    g.dnj.divmod(tid < items ? tid : 0, kz0, jj0);
    {
        const cpx<R> *sp = zb + m24(j0 + jj0, SK) + kz0;
        const int qs = m24(q, SK);
#pragma unroll
        for (int c = 0; c < 8; ++c) o[c] = sp[c * qs];
        dft8<+1>(o);
    }
    __syncthreads();
    if (tid < items) {
        cpx<R> *zp = zb + m24(fft_slot(kz0, g.qz), LP) + jj0, *wp = zb + m24(fft_slot(kz0 ? Nz - kz0 : h, g.qz), LP) + jj0;
        const bool dc = kz0 == 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const cpx<R> a = o[2 * t], b = o[2 * t + 1];
            zp[t * nj] = {dc ? a.x : a.x - b.y, dc ? b.x : a.y + b.x};
            wp[t * nj] = {dc ? a.y : a.x + b.y, dc ? b.y : b.x - a.y};
        }
    }
    __syncthreads();
    fft_lines<+1>(zb, LP, g.dlines, g.qz, twz, tid, bd);
    double s = 1.0;
    if constexpr (!PHI) {
        nc.g = sr.p.g;
        nc.gd = sr.p.gd;
        nc.shift = v.shift ? sr.scal[SC_SHIFT] : 0.0;
        nc.cap = v.shift;
        nc.capped = sr.scal + SC_CAPPED;
        nu_prepare(nc);
        s = v.use_scale ? sr.scal[SC_SCALE] : 1.0;
    }
    using O = typename std::conditional<PHI, R, P>::type;
    O *__restrict__ out;
    if constexpr (PHI) out = phi + (extra ? far : (long)x * Ny * Nz);
    else out = psi;
    const double *row = extra ? sqr + Ny : sqr;
    const auto value = [&](int y, int z, P p0, R f, bool kept) {
        if constexpr (PHI) return f;
        else return nu_apply(p0, s, f, trap_sum(tc, row[y], sqz[z]), nc, kept);
    };
    if (rim) out[(Ny - 1) * Nz + tid] = value(Ny - 1, tid, pr, zb[m24(tid, LP)].x, true);
    // own: the plane transformed; else the points y < Ny-1, z < Nz-1 of plane Nx-1
#pragma unroll 1
    for (bool own = !extra;; own = false) {
        // in groups of 4 without a branch inside, so that their chains (LDS
        // reads, the exponential) run side by side: with one or two wavefronts
        // per SIMD nothing else hides them
#pragma unroll
        for (int gr = 0; gr < KG; ++gr) {
            if (4 * gr * bd >= points) break;  // uniform
            if constexpr (!PHI)
                if (gr + 1 < KG && gr + 1 >= PRE) load_psi(gr + 1);
            O ov[4];
            int at[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int i = opaque(tid) + (4 * gr + w) * bd;
                int lr, y, z, r, jj;
                place(i < points ? i : 0, lr, y, z);
                g.dnj.divmod(lr, r, jj);
                const bool yl = y == Ny - 1, zl = z == Nz - 1;
                // own plane x < Nx-1: not row Ny-1 below z = Nz-1; plane Nx-1: its
                // rim; not own: all but the rim
                const bool put = i < points && (own ? (x < Nx - 1 ? !(yl && !zl) : (yl || zl)) : !(yl || zl));
                const int zs = (own && x < Nx - 1 && zl && !yl) ? 0 : z;
                const R *c = reinterpret_cast<const R *>(&zb[m24(zs, LP) + m24(r >> 1, nj) + jj]) + (r & 1);
                ov[w] = value(y, z, pv[gr][w], *c, put);
                at[w] = put ? m24(y, Nz) + z : -1;
            }
#pragma unroll
            for (int w = 0; w < 4; ++w)
                if (at[w] >= 0) out[at[w]] = ov[w];
        }
        if (x != 0 || !own || g.extra) return;
        if constexpr (PHI) {
            out = phi + far;
        } else {
            psi = reinterpret_cast<P *>(sr.psi) + far;
            out = psi;
            row = sqr + Ny;
#pragma unroll
            for (int gr = 0; gr < PRE; ++gr) load_psi(gr);
        }
    }
}

template <typename S>
constexpr int max_threads() { return sizeof(S) == 16 ? 512 : 1024; }


template <typename S, typename R>
size_t inv_lds(int Ny, int Nz) {
    const size_t zb = (size_t)Nz * (Ny / 2 + 1), sp = (size_t)Ny * (Nz / 2 + 1);
    return ((size_t)Nz + 2 * Ny) * sizeof(double) + ((size_t)Ny + Nz + std::max(zb, sp)) * sizeof(cpx<R>);
}

// one thread per segment of 16 points: as many as each pass has butterflies
inline int plane_threads(long Ny, long Nz) { return (int)((Ny * Nz / 16 + 63) / 64 * 64); }

constexpr size_t kLdsMax = 160 * 1024;

template <typename S, typename R>
bool fits(long Ny, long Nz) {
    if (Ny * Nz / 16 > max_threads<S>()) return false;
    const int bd = plane_threads(Ny, Nz);
    return PlaneLds<S, R>((int)Ny, (int)Nz, bd, true, true).total <= kLdsMax &&
           inv_lds<S, R>((int)Ny, (int)Nz) <= kLdsMax;
}

// Dynamic LDS beyond 64 KiB is asked for once per kernel and device.
template <typename K>
hipError_t allow_lds(K kernel, size_t bytes, std::atomic<unsigned long> &done) {
    if (bytes <= 65536) return hipSuccess;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long bit = 1ul << (dev & 63);
    if (done.load(std::memory_order_relaxed) & bit) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_relaxed);
    return e;
}

// parts: workgroups per plane of the inverse kernel
PlaneDims dims(const dbec_ctx *c, int parts, int extra = 0) {
    PlaneDims g;
    g.Nx = (int)c->Nx;
    g.Ny = (int)c->Ny;
    g.Nz = (int)c->Nz;
    g.qy = g.Ny / 8;
    g.qz = g.Nz / 8;
    g.nt = g.Ny * g.Nz / 16;
    g.dNy = FastDiv::of(g.Ny);
    g.dNyh = FastDiv::of(g.Ny / 2);
    g.dNz = FastDiv::of(g.Nz);
    g.dNzh = FastDiv::of(g.Nz / 2);
    g.dqy = FastDiv::of(g.qy);
    g.parts = parts;
    g.nj = g.qy / parts;
    g.extra = extra;
    g.dparts = FastDiv::of(parts);
    g.dnj = FastDiv::of(g.nj);
    g.dlines = FastDiv::of(4 * g.nj);
    return g;
}

void sweep_const(const AxisArgs &a, SweepConst<double> &k) { k = {a.k[0][0], a.k[1][0], -a.k[1][0]}; }
void sweep_const(const AxisArgs &a, SweepConst<float> &k) {
    k.A0r = (float)a.k[0][0];
    k.A = (float)a.k[1][0];
    k.mA = -k.A;
}
template <typename Q>
void sweep_const(const AxisArgs &a, SweepConst<cpx<Q>> &k) {
    k.A0r = {(Q)a.k[0][0], (Q)a.k[0][1]};
    k.A = {(Q)a.k[1][0], (Q)a.k[1][1]};
    k.mA = {(Q)a.k[2][0], (Q)a.k[2][1]};
}
template <typename A>
SweepTab<A> sweep_tab(const AxisArgs &a) {
    using T = typename TabOf<A>::T;
    return {static_cast<const T *>(a.tab[0]), static_cast<const T *>(a.tab[1]), static_cast<const T *>(a.tab[2]),
            static_cast<const T *>(a.tab[3])};
}

template <typename S, typename R, bool SW, bool FF, int MAXT>
hipError_t fwd_t(const dbec_ctx *c, const Solves &v) {
    using A = typename Arith<S>::T;
    static std::atomic<unsigned long> done{0};
    const PlaneDims g = dims(c, 1);
    const int bd = plane_threads(g.Ny, g.Nz);
    const size_t lds = PlaneLds<S, R>(g.Ny, g.Nz, bd, SW, FF).total;
    PlaneSweep<A> k;
    const AxisArgs y = sweep_axis_args(c, 1), z = sweep_axis_args(c, 2);
    k.ty = sweep_tab<A>(y);
    k.tz = sweep_tab<A>(z);
    sweep_const(y, k.ky);
    sweep_const(z, k.kz);
    k.wy = c->b.wgt + c->Nx;
    k.wz = k.wy + c->Ny;
    auto *kernel = &k_plane_fwd<S, R, SW, FF, MAXT>;
    hipError_t e = allow_lds(kernel, lds, done);
    if (e != hipSuccess) return e;
    void *const *tw = std::is_same<R, float>::value ? c->b.twf : c->b.tw;
    kernel<<<dim3(xcd_blocks(g.Nx), (unsigned)v.nb), bd, lds, c->stream>>>(
        v, g, k, static_cast<const cpx<R> *>(tw[1]), static_cast<const cpx<R> *>(tw[2]));
    return hipGetLastError();
}
// The variant by workgroup size: 512 (also all of complex FP64), 640, 1024.
template <typename S>
int block_class(const dbec_ctx *c) {
    const int bd = plane_threads(c->Ny, c->Nz);
    return bd <= 512 || max_threads<S>() == 512 ? 512 : (bd <= 640 ? 640 : 1024);
}

template <typename S, typename R, int MAXT>
hipError_t fwd_m(const dbec_ctx *c, const Solves &v, bool sweeps, bool fft) {
    if (sweeps && fft) return fwd_t<S, R, true, true, MAXT>(c, v);
    if (sweeps) return fwd_t<S, R, true, false, MAXT>(c, v);
    return fwd_t<S, R, false, true, MAXT>(c, v);
}
template <typename S, typename R>
hipError_t fwd(const dbec_ctx *c, const Solves &v, bool sweeps, bool fft) {
    if constexpr (max_threads<S>() > 512) {
        if (block_class<S>(c) == 640) return fwd_m<S, R, 640>(c, v, sweeps, fft);
        if (block_class<S>(c) == 1024) return fwd_m<S, R, 1024>(c, v, sweeps, fft);
    }
    return fwd_m<S, R, 512>(c, v, sweeps, fft);
}

// Workgroups per plane of the inverse kernel: as many as divide the
// butterflies while the launch has at most kParts workgroups.
constexpr long kParts = 256;
int inv_parts(const dbec_ctx *c, int nb, bool split) {
    const int q = (int)c->Ny / 8;
    int best = split ? 2 : 1;
    for (int p = best + 1; p <= q; p++)
        if (q % p == 0 && c->Nx * nb * p <= kParts) best = p;
    return best;
}

template <typename P, typename R, bool PHI, bool SPLIT, int MAXT>
hipError_t inv_t(const dbec_ctx *c, const Solves &v, int parts) {
    static std::atomic<unsigned long> done{0};
    const long nb = PHI ? 1 : v.nb, own = c->Nx * parts * nb;
    const int extra = own + parts * nb <= kParts || own > kParts;
    const PlaneDims g = dims(c, parts, extra);
    const int bd = plane_threads(g.Ny, g.Nz);
    const size_t lds = inv_lds<P, R>(g.Ny, g.Nz);
    auto *kernel = &k_plane_inv<P, R, PHI, SPLIT, MAXT>;
    hipError_t e = allow_lds(kernel, lds, done);
    if (e != hipSuccess) return e;
    void *const *tw = std::is_same<R, float>::value ? c->b.twf : c->b.tw;
    kernel<<<dim3(xcd_blocks((g.Nx + (long)extra) * parts), (unsigned)nb), bd, lds, c->stream>>>(
        v, g, c->b.sq, nu_const(c), static_cast<R *>(c->b.phi), static_cast<const cpx<R> *>(tw[1]),
        static_cast<const cpx<R> *>(tw[2]));
    return hipGetLastError();
}
template <typename P, typename R, bool PHI, int MAXT>
hipError_t inv_m(const dbec_ctx *c, const Solves &v) {
    const int parts = inv_parts(c, PHI ? 1 : v.nb, MAXT == 1024 && sizeof(R) == 8);
    if constexpr (MAXT < 1024 || sizeof(R) == 4)  // FP64 at 1024 threads: always split, 128 registers
        if (parts == 1) return inv_t<P, R, PHI, false, MAXT>(c, v, parts);
    return inv_t<P, R, PHI, true, MAXT>(c, v, parts);
}
template <typename P, typename R, bool PHI>
hipError_t inv_p(const dbec_ctx *c, const Solves &v) {
    if constexpr (max_threads<P>() > 512) {
        if (block_class<P>(c) == 640) return inv_m<P, R, PHI, 640>(c, v);
        if (block_class<P>(c) == 1024) return inv_m<P, R, PHI, 1024>(c, v);
    }
    return inv_m<P, R, PHI, 512>(c, v);
}
template <typename P, typename R>
hipError_t inv(const dbec_ctx *c, const Solves &v, bool phi) {
    return phi ? inv_p<P, R, true>(c, v) : inv_p<P, R, false>(c, v);
}

}  // namespace

// Where the planes win, by size alone (the two forms round differently, so the
// choice must not depend on a tuned or batched launch).  Step times, one pass
// per kernel against planes, us (FP64 imaginary, mixed imaginary, FP64 real,
// mixed real; - where the plane does not fit LDS):
//   16x32x32    31  30  33  31   25  24  26  24
//   64x64x64    38  34  44  35   33  29  36  30
//   128x96x80   74  55  82  61   57  43  66  48
//   96x96x96    72  53  83  60   55  40   -  48
//   128x128x128 98  72 104  83   82  62   -  69
//   256x128x128 116 93 163  98  116  83   -  84
//   48x128x128  64  48  74  53   60  42   -  49
//   16x128x128  43  37  47  38   51  38   -  43
//   384x96x96   121 94 161 102  132  93   - 110
//   512x64x64   101 73 105  82   80  60  80  68
// So large planes need 48 of them or more (one workgroup each: fewer leave
// most of the chip idle during long launches), and past 256 planes, where the
// launches run in several rounds and bandwidth counts, only small grids gain.
// The same holds for batched launches that share the device with other buckets
// (the request loop): of its stream's first 200 requests it serves 28.2 a second
// without planes, 28.6 with planes up to 64x64, 26.9 up to 96x96, 25.9 with all.
bool plane_ok(const dbec_ctx *c, bool shared) {
    if (!plane_len(c->Ny) || !plane_len(c->Nz)) return false;
    if (shared && c->Ny * c->Nz > 64 * 64) return false;
    if (c->Ny * c->Nz > 96 * 96 && c->Nx < 48) return false;
    if (c->Nx > 256 && c->N > 512 * 64 * 64) return false;
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) return f32 ? fits<float, float>(c->Ny, c->Nz) : fits<double, double>(c->Ny, c->Nz);
    return f32 ? fits<cpx<float>, float>(c->Ny, c->Nz) : fits<cpx<double>, double>(c->Ny, c->Nz);
}

hipError_t launch_plane_fwd(const dbec_ctx *c, const Solves &v, bool sweeps, bool fft) {
    if (!c->planes || !(sweeps || fft)) return hipErrorInvalidValue;
    // complex lines: the sweeps use A = i a, mA = -A, A0r = 1 + i b
    for (int a = 1; c->mode == DBEC_REAL && a < 3; a++)
        if (c->A[a][0] != 0.0 || c->A0r[a][0] != 1.0 || c->mA[a][0] != 0.0 || c->mA[a][1] != -c->A[a][1])
            return hipErrorInvalidValue;
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) return f32 ? fwd<float, float>(c, v, sweeps, fft) : fwd<double, double>(c, v, sweeps, fft);
    return f32 ? fwd<cpx<float>, float>(c, v, sweeps, fft) : fwd<cpx<double>, double>(c, v, sweeps, fft);
}

hipError_t launch_plane_inv(const dbec_ctx *c, const Solves &v, bool phi) {
    if (!c->planes) return hipErrorInvalidValue;
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) return f32 ? inv<float, float>(c, v, phi) : inv<double, double>(c, v, phi);
    return f32 ? inv<cpx<float>, float>(c, v, phi) : inv<cpx<double>, double>(c, v, phi);
}

}  // namespace dbec
