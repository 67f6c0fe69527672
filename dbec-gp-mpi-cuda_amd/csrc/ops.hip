// ops.hip - pointwise kernels, sweeps and the norm of the split step.
//
// Reference aliases: imag3d.cu = src/imag3d-mpicuda/imag3d-mpicuda.cu,
// real3d.cu = src/real3d-mpicuda/real3d-mpicuda.cu, diffint.cu =
// src/utils/diffint.cu.
#include <cstdlib>
#include <type_traits>

#include "norm_device.hpp"
#include "ops.hpp"
#include "sweep_device.hpp"

namespace dbec {

// ---------------------------------------------------------------------------
// calcnu (calcnu_kernel imag3d.cu:1759-1783; real3d.cu:1856-1883), with psi
// read as psi * scale when a renormalisation is pending (imaginary time).  The
// trap is recomputed from the grid (nu_device.hpp).
template <typename P, typename R>
__global__ void __launch_bounds__(256)
k_calcnu(P *__restrict__ psi, const R *__restrict__ phi, const double *__restrict__ scale,
         const double *__restrict__ sq, TrapConst tc, NuConst nc, int Nx, int Ny, int Nz) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= Nz) return;
    const long row = blockIdx.y;  // x * Ny + y
    const int i = (int)(row / Ny), j = (int)(row % Ny);
    const long n = row * Nz + k;
    const double s = scale ? *scale : 1.0;
    const double pot = trap(tc, sq[i], sq[Nx + j], sq[Nx + Ny + k]);
    psi[n] = nu_apply(psi[n], s, phi[n], pot, nc);
}

TrapConst trap_const(const dbec_ctx *c) {
    TrapConst tc;
    tc.half_par = 0.5 * c->p.par;
    tc.g2 = c->p.vgamma * c->p.vgamma;
    tc.n2 = c->p.vnu * c->p.vnu;
    tc.l2 = c->p.vlambda * c->p.vlambda;
    return tc;
}

NuConst nu_const(const dbec_ctx *c) {
    NuConst nc;
    nc.dt = c->p.dt;
    nc.g = c->g;
    nc.gd = c->gd;
    const long nd = c->Nx * c->Ny * c->Nz;
    nc.nd = (double)nd;
    nd_split(nc, nd);
    nc.shift = 0.0;
    nc.cap = 0;
    nc.capped = nullptr;
    nu_prepare(nc);
    return nc;
}

hipError_t launch_calcnu(hipStream_t s, const dbec_ctx *c, const double *scale) {
    const auto &b = c->b;
    const TrapConst tc = trap_const(c);
    const NuConst nc = nu_const(c);
    dim3 block(256), grid((unsigned)((c->Nz + 255) / 256), (unsigned)(c->Nx * c->Ny));
    const int Nx = (int)c->Nx, Ny = (int)c->Ny, Nz = (int)c->Nz;
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) {
        if (!f32)
            k_calcnu<double, double><<<grid, block, 0, s>>>(static_cast<double *>(b.psi), static_cast<const double *>(b.phi),
                                                            scale, b.sq, tc, nc, Nx, Ny, Nz);
        else
            k_calcnu<float, float><<<grid, block, 0, s>>>(static_cast<float *>(b.psi), static_cast<const float *>(b.phi),
                                                          scale, b.sq, tc, nc, Nx, Ny, Nz);
    } else {
        if (!f32)
            k_calcnu<cpx<double>, double><<<grid, block, 0, s>>>(static_cast<cpx<double> *>(b.psi),
                                                                 static_cast<const double *>(b.phi), nullptr, b.sq, tc,
                                                                 nc, Nx, Ny, Nz);
        else
            k_calcnu<cpx<float>, float><<<grid, block, 0, s>>>(static_cast<cpx<float> *>(b.psi),
                                                               static_cast<const float *>(b.phi), nullptr, b.sq, tc, nc,
                                                               Nx, Ny, Nz);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// psi *= scale (the renormalisation of calcnorm_kernel, imag3d.cu:1220-1233).
template <typename P>
__global__ void k_scale(P *__restrict__ psi, const double *__restrict__ scale, long n) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double s = *scale;
    psi[t] = (P)((double)psi[t] * s);
}

hipError_t launch_scale(hipStream_t s, const dbec_ctx *c, const double *scale) {
    dim3 block(256);
    if (c->mode == DBEC_IMAG) {
        dim3 grid((unsigned)((c->N + 255) / 256));
        if (c->prec == DBEC_MIXED) k_scale<float><<<grid, block, 0, s>>>(static_cast<float *>(c->b.psi), scale, c->N);
        else k_scale<double><<<grid, block, 0, s>>>(static_cast<double *>(c->b.psi), scale, c->N);
    } else {
        dim3 grid((unsigned)((2 * c->N + 255) / 256));
        if (c->prec == DBEC_MIXED) k_scale<float><<<grid, block, 0, s>>>(static_cast<float *>(c->b.psi), scale, 2 * c->N);
        else k_scale<double><<<grid, block, 0, s>>>(static_cast<double *>(c->b.psi), scale, 2 * c->N);
    }
    return hipGetLastError();
}

__global__ void k_set_scalar(double *p, double v) { *p = v; }

hipError_t launch_set_scalar(hipStream_t s, double *p, double v) {
    k_set_scalar<<<1, 1, 0, s>>>(p, v);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// x and y sweeps: a workgroup covers L consecutive z (lanes; one 256-byte row
// per load) of the lines of one y (x sweep) or x (y sweep) plane; thread
// (l, s) loads its segment straight from HBM into registers.
template <typename S, int AXIS, int L, int M, bool PEEL>
__global__ void __launch_bounds__(512)
k_sweep_xy(Solves sv, int Nx, int Ny, int Nz, SweepTab<typename Arith<S>::T> tab,
           SweepConst<typename Arith<S>::T> k) {
    using A = typename Arith<S>::T;
    extern __shared__ char smem_raw[];
    S *__restrict__ psi = reinterpret_cast<S *>(solve_at(sv).psi);
    const int n = AXIS == 0 ? Nx : Ny;
    const int P = n / M;
    const int nt = L * P;
    SweepShared<A, M> sh(smem_raw, n, nt, L);
    const int tid = threadIdx.x;
    const int l = tid % L, s = tid / L;
    const int zt = (Nz + L - 1) / L;
    const int pl = blockIdx.x / zt, z0 = (blockIdx.x % zt) * L;
    const int nl = min(L, Nz - z0);
    const bool act = l < nl;
    const long base = (AXIS == 0 ? (long)pl * Nz : (long)pl * Ny * Nz) + z0 + l;
    const long es = AXIS == 0 ? (long)Ny * Nz : (long)Nz;
    const int e0 = s * M;
    const A zero = m_zero(k.A);
    const CoefPre<A> cp = coef_pre(tab, n, tid);
    // The segment's elements at 32-bit byte offsets j * es from its first one
    // (at most 16 * 512^2 * 16 bytes): one 64-bit address per thread, then a
    // 32-bit step per element instead of a 64-bit multiply-add.
    char *const seg = reinterpret_cast<char *>(psi + base + (long)e0 * es);
    const unsigned bes = (unsigned)(es * (long)sizeof(S));
    auto at = [&](int j) -> S & { return *reinterpret_cast<S *>(seg + (unsigned)j * bes); };
    // Predicated loads converted in place: fewer registers (higher occupancy)
    // than issuing them into a separate array, which measured faster here.
    A v[M];
#pragma unroll
    for (int j = 0; j < M; ++j) v[j] = act ? to_a(at(j)) : zero;
    const A hl = (act && e0 > 0) ? to_a(*reinterpret_cast<const S *>(seg - bes)) : zero;
    const A hr = (act && e0 + M < n) ? to_a(at(M)) : zero;
    coef_put(sh, cp, tab, n, tid, nt);
    __syncthreads();
    seg_solve<A, M, false, PEEL>(v, hl, hr, e0, n, s, l, L, P, sh, k, nullptr);
    if (act) {
#pragma unroll
        for (int j = 0; j < M; ++j) at(j) = from_a<S>(v[j]);
    }
}

// Row and column of packet tid + q * nt (VE elements each) of a run of rows
// of n elements, for q = 0, 1, ...: one division per thread, then a step and
// a wrap per packet (n is a run-time value: a division per packet costs
// tens of instructions).
struct RunPos {
    int row, e, dr, de;
    __device__ RunPos(int tid, int nt, int VE, int n)
        : row(tid * VE / n), e(tid * VE % n), dr(nt * VE / n), de(nt * VE % n) {}
    __device__ void next(int n) {
        row += dr;
        e += de;
        if (e >= n) {
            e -= n;
            ++row;
        }
    }
};

// z sweep: lines are contiguous rows.  A workgroup covers L rows of one x
// plane.  Staged (DIRECT false): the rows go through an LDS tile in the
// storage type (row-major, rows padded by one 16-byte packet: coalesced row
// loads and stores, and 16-byte LDS accesses without bank conflicts both for
// the row copies and for the segments), and each thread moves its segment
// between the tile and its registers.  Direct (DIRECT true): each thread
// loads its segment, M contiguous and 16-byte aligned values of its row,
// straight into registers as packets and stores it back the same way; the
// lanes of a wavefront read whole 64-128-byte runs of different rows, which
// the caches merge.  With COLS (imaginary time) the Simpson z integrals of
// the new psi^2 are summed per row and the rows of the tile with the y
// weights: colpart[tile][x] (calcnorm, imag3d.cu:1194-1209).
template <typename S, int L, int M, bool COLS, bool DIRECT>
__global__ void __launch_bounds__(512)
k_sweep_z(Solves sv, int Nx, int Ny, int Nz, SweepTab<typename Arith<S>::T> tab,
          SweepConst<typename Arith<S>::T> k, const double *__restrict__ wz, const double *__restrict__ wy) {
    using A = typename Arith<S>::T;
    extern __shared__ char smem_raw[];
    const SolveAt sr = solve_at(sv);
    S *__restrict__ psi = reinterpret_cast<S *>(sr.psi);
    double *__restrict__ colpart = sr.rows;
    const int n = Nz;
    constexpr int VE = Pk<S>::n, KV = M / VE;
    static_assert(M % VE == 0, "z sweep packets");
    // row stride of the tile: n + VE elements keeps every row 16-byte aligned
    // and consecutive rows 4 banks apart, so the packet accesses are
    // conflict-free
    const int RS = n + VE;
    const int P = n / M;
    const int nt = L * P;
    SweepShared<A, M> sh(smem_raw, n, nt, L);
    S *tile = reinterpret_cast<S *>(smem_raw + ((SweepShared<A, M>::bytes(n, nt, L, COLS) + 15) & ~size_t(15)));
    const int tid = threadIdx.x;
    const int l = tid % L, s = tid / L;
    const int yt = (Ny + L - 1) / L;
    const int xrow = blockIdx.x / yt, tno = blockIdx.x % yt, y0 = tno * L;
    const int nl = min(L, Ny - y0);
    const long base = ((long)xrow * Ny + y0) * Nz;
    const A zero = m_zero(k.A);
    const int npk = nl * n / VE;
    const int e0 = s * M;
    const bool act = l < nl;
    const CoefPre<A> cp = coef_pre(tab, n, tid);
    A v[M], hl, hr;
    if constexpr (DIRECT) {
        // rows past the tile's last read that row (clamped) and are not stored
        const S *src = psi + base + (long)min(l, nl - 1) * n + e0;
        typename Pk<S>::type r[KV];
#pragma unroll
        for (int q = 0; q < KV; ++q) r[q] = ld_pk(src + q * VE);
        const S sl = src[e0 > 0 ? -1 : 0], sr_ = src[e0 + M < n ? M : M - 1];
        coef_put(sh, cp, tab, n, tid, nt);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < KV; ++q)
#pragma unroll
            for (int j = 0; j < VE; ++j) v[q * VE + j] = act ? to_a(r[q].e[j]) : zero;
        hl = (act && e0 > 0) ? to_a(sl) : zero;
        hr = (act && e0 + M < n) ? to_a(sr_) : zero;
    } else {
        // The tile's nl rows are one contiguous run of nl * n elements; each
        // thread moves M / VE packets of it (all loads first).
        typename Pk<S>::type r[KV];
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const int iv = tid + q * nt;
            r[q] = ld_pk(psi + base + (unsigned)((iv < npk ? iv : 0) * VE));
        }
        coef_put(sh, cp, tab, n, tid, nt);
        RunPos rp(tid, nt, VE, n);
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            if (tid + q * nt < npk) st_pk(tile + rp.row * RS + rp.e, r[q]);
            rp.next(n);
        }
        __syncthreads();
        const S *row = tile + l * RS;
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const typename Pk<S>::type pk = ld_pk(row + e0 + q * VE);
#pragma unroll
            for (int j = 0; j < VE; ++j) v[q * VE + j] = act ? to_a(pk.e[j]) : zero;
        }
        hl = (act && e0 > 0) ? to_a(row[e0 - 1]) : zero;
        hr = (act && e0 + M < n) ? to_a(row[e0 + M]) : zero;
    }
    const double acc = seg_solve<A, M, COLS, true>(v, hl, hr, e0, n, s, l, L, P, sh, k, wz);
    // every thread read its segment before the first barrier inside seg_solve
    if constexpr (DIRECT) {
        if (act) {
            S *dst = psi + base + (long)l * n + e0;
#pragma unroll
            for (int q = 0; q < KV; ++q) {
                typename Pk<S>::type o;
#pragma unroll
                for (int j = 0; j < VE; ++j) o.e[j] = from_a<S>(v[q * VE + j]);
                st_pk(dst + q * VE, o);
            }
        }
    } else if (act) {
        S *orow = tile + l * RS;
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            typename Pk<S>::type o;
#pragma unroll
            for (int j = 0; j < VE; ++j) o.e[j] = from_a<S>(v[q * VE + j]);
            st_pk(orow + e0 + q * VE, o);
        }
    }
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
            if (tid == 0) colpart[(long)tno * Nx + xrow] = w;
        }
    } else if constexpr (!DIRECT) {
        __syncthreads();
    }
    if constexpr (!DIRECT) {
        RunPos rp(tid, nt, VE, n);
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const int iv = tid + q * nt;
            if (iv < npk) st_pk(psi + base + (unsigned)(iv * VE), ld_pk(tile + rp.row * RS + rp.e));
            rp.next(n);
        }
    }
}

// Segment length of the x / y sweeps for a line of n values of S: 32 for
// complex FP32 lines that split into at least 7 segments of 32 (measured at
// 96^3 to 256^3; at 192, 16-element segments are faster since the carry
// multipliers are tabulated: x 21.7 -> 20.9 us, y 21.8 -> 20.6 us at 192^3),
// for FP64 real lines of 512 or more (measured at 512^3: the
// x sweep 532 -> 407 us, the y sweep unchanged) and for lines whose
// 16-element segments would need more than 512 threads even with 128-byte
// rows; else 16.  It fixes the rounding of the partitioned solve, so it
// depends on the line only (never on a tuned choice).
template <typename S>
static int seg_len(long n) {
    using A = typename Arith<S>::T;
    if (!std::is_floating_point<A>::value && sizeof(A) == 8 && n % 32 == 0 && n / 32 >= 7) return 32;
    if (std::is_same<S, double>::value && n >= 512 && n % 32 == 0) return 32;
    if ((n / 16) * (long)(128 / sizeof(S)) > 512) return 32;
    return 16;
}

// z sweep: 16-element segments (more threads per tile row); rows per
// workgroup: a power of two >= 4 whose tile fits 64 KiB of LDS, with at most
// 256 threads (measured at 256^3 and 256x256x384).
static int z_seg_len(long) { return 16; }

static int env_int(const char *name, int dflt) {
    const char *e = getenv(name);
    return e ? atoi(e) : dflt;
}

// half: the tile holds half of the rows at a time.
template <typename S>
static int z_rows(long n, bool half = false) {
    static const int max_threads = env_int("DBEC_SWEEP_Z_THREADS", 256);
    static const long tile_max = 1024L * env_int("DBEC_SWEEP_Z_TILE_KB", 64);
    const int M = z_seg_len(n);
    const int P = (int)(n / M);
    const auto tile = [&](int L) { return (long)(n + Pk<S>::n) * (half ? L / 2 : L) * (long)sizeof(S); };
    int L = 64;
    while (L > 4 && ((long)L * P > max_threads || tile(L) > tile_max)) L /= 2;
    return L;
}

static size_t arith_elem(const dbec_ctx *c) { return c->mode == DBEC_REAL ? 16 : 8; }

int sweep_z_rows(const dbec_ctx *c) {
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) return f32 ? z_rows<float>(c->Nz) : z_rows<double>(c->Nz);
    return f32 ? z_rows<cpx<float>>(c->Nz) : z_rows<cpx<double>>(c->Nz);
}

// Rows per workgroup of the fused z kernel where its tile holds half of them
// at a time (complex lines), by the same bounds, which by default leave the most
// that give at most 256 threads (measured at 512 complex FP64: 8 rows 151, 4
// rows 200 us; at 128: 32 rows 41, 16 rows 46 us; twice the rows, so twice the
// threads at a barrier: 143 -> 159 us at 256^3, 229 -> 280 at 256x256x384).
// 0: no half tiles.  With whole tiles it takes the z sweep's rows.
int fused_z_rows_half(const dbec_ctx *c) {
    if (c->mode == DBEC_IMAG) return 0;
    if (c->prec == DBEC_MIXED) return fused_z_half<cpx<float>>(c->Nz) ? z_rows<cpx<float>>(c->Nz, true) : 0;
    return fused_z_half<cpx<double>>(c->Nz) ? z_rows<cpx<double>>(c->Nz, true) : 0;
}

AxisArgs sweep_axis_args(const dbec_ctx *c, int axis) {
    const CoefLayout lay(c->Nx, c->Ny, c->Nz);
    const bool cplx = c->mode == DBEC_REAL;
    const size_t el = sizeof(double) * (cplx ? 2 : 1);  // FP64 tables in every precision
    const char *base = reinterpret_cast<const char *>(c->b.coef);
    AxisArgs a;
    a.tab[0] = base + el * lay.ca(axis);
    a.tab[1] = base + el * lay.cg(axis);
    a.tab[2] = base + el * lay.gb(axis, 0);
    a.tab[3] = base + el * lay.fa(axis, 0);
    for (int q = 0; q < 2; q++) {
        a.k[0][q] = c->A0r[axis][q];
        a.k[1][q] = c->A[axis][q];
        a.k[2][q] = c->mA[axis][q];
    }
    return a;
}

void sweep_z_args(const dbec_ctx *c, FftArgs &a) {
    const AxisArgs z = sweep_axis_args(c, 2);
    for (int i = 0; i < 4; i++) a.ztab[i] = z.tab[i];
    for (int i = 0; i < 3; i++)
        for (int q = 0; q < 2; q++) a.zk[i][q] = z.k[i][q];
    a.wz = c->b.wgt + c->Nx + c->Ny;
    a.wy = c->b.wgt + c->Nx;
    a.zrows = sweep_z_rows(c);
    a.zrows_half = fused_z_rows_half(c);
}

long sweep_z_tiles(const dbec_ctx *c) {
    const bool f32 = c->prec == DBEC_MIXED;
    int L;
    if (c->mode == DBEC_IMAG) L = f32 ? z_rows<float>(c->Nz) : z_rows<double>(c->Nz);
    else L = f32 ? z_rows<cpx<float>>(c->Nz) : z_rows<cpx<double>>(c->Nz);
    return (c->Ny + L - 1) / L;
}

// Solves of one launch: the by-value `one` or nb entries of `many`.
struct Launch {
    hipStream_t s;
    Solves v;
};

// The tables of one axis for both segment lengths (16 and 32).
template <typename A>
struct SweepTabs {
    const typename TabOf<A>::T *ca, *cg, *gb[2], *fa[2];
    SweepTab<A> at(int M) const {
        const int m = M == 32 ? 1 : 0;
        return {ca, cg, gb[m], fa[m]};
    }
};

template <typename S, int AXIS, int L, bool PEEL>
static hipError_t sweep_xy_launch(const Launch &q, int Nx, int Ny, int Nz, const SweepTabs<typename Arith<S>::T> &t,
                                  const SweepConst<typename Arith<S>::T> &k, int M) {
    using A = typename Arith<S>::T;
    const int n = AXIS == 0 ? Nx : Ny;
    const int P = n / M;
    if (n % M != 0 || L * P > 512) return hipErrorInvalidValue;
    const long nblocks = (long)((Nz + L - 1) / L) * (AXIS == 0 ? Ny : Nx);
    dim3 grid((unsigned)nblocks, (unsigned)q.v.nb), block(L * P);
    const size_t lds =
        M == 32 ? SweepShared<A, 32>::bytes(n, L * P, L, false) : SweepShared<A, 16>::bytes(n, L * P, L, false);
    if constexpr (sizeof(A) <= 8) {
        if (M == 32) {
            k_sweep_xy<S, AXIS, L, 32, PEEL><<<grid, block, lds, q.s>>>(q.v, Nx, Ny, Nz, t.at(32), k);
            return hipGetLastError();
        }
    } else {
        if (M != 16) return hipErrorInvalidValue;
    }
    k_sweep_xy<S, AXIS, L, 16, PEEL><<<grid, block, lds, q.s>>>(q.v, Nx, Ny, Nz, t.at(16), k);
    return hipGetLastError();
}

// x / y sweeps: segments of seg_len elements; per axis the row width (bytes
// of z per load: 256, or 128 for FP32 real lines) and the boundary peeling
// (real lines) by rule, or as tuned for the context.  DBEC_SWEEP_XY_{ROWB,M}
// (FP64 and complex lines), DBEC_SWEEP_XY_{ROWB,M}32 (FP32 real lines) and
// DBEC_SWEEP_XY_PEEL (0 or 1) override (tuning runs).
template <typename S, int AXIS, bool PEEL>
static hipError_t sweep_xy_rows(const Launch &q, int Nx, int Ny, int Nz, const SweepTabs<typename Arith<S>::T> &t,
                                const SweepConst<typename Arith<S>::T> &k, int rowb, int M) {
    const int n = AXIS == 0 ? Nx : Ny;
    // 256-byte rows only where their workgroup stays within 512 threads
    if (rowb == 128 || (long)(256 / sizeof(S)) * (n / M) > 512)
        return sweep_xy_launch<S, AXIS, 128 / sizeof(S), PEEL>(q, Nx, Ny, Nz, t, k, M);
    return sweep_xy_launch<S, AXIS, 256 / sizeof(S), PEEL>(q, Nx, Ny, Nz, t, k, M);
}
template <typename S, int AXIS>
static hipError_t sweep_xy_dispatch(const Launch &q, int Nx, int Ny, int Nz, const SweepTabs<typename Arith<S>::T> &t,
                                    const SweepConst<typename Arith<S>::T> &k, const Tuning &tu) {
    using A = typename Arith<S>::T;
    static const int rowb_env = sizeof(S) == 4 ? env_int("DBEC_SWEEP_XY_ROWB32", 0) : env_int("DBEC_SWEEP_XY_ROWB", 0);
    static const int mset = sizeof(S) == 4 ? env_int("DBEC_SWEEP_XY_M32", 0) : env_int("DBEC_SWEEP_XY_M", 0);
    static const int peel_env = env_int("DBEC_SWEEP_XY_PEEL", -1);
    const int n = AXIS == 0 ? Nx : Ny;
    int M = (mset == 16 || mset == 32) ? mset : seg_len<S>(n);
    if (sizeof(A) > 8) M = 16;
    const int rowb = rowb_env ? rowb_env : (tu.xy_rowb[AXIS] ? tu.xy_rowb[AXIS] : (sizeof(S) == 4 ? 128 : 256));
    const int peel_t = peel_env >= 0 ? peel_env : tu.xy_peel[AXIS];
    const bool peel = peel_t >= 0 ? peel_t != 0 : std::is_floating_point<A>::value;
    if (peel) return sweep_xy_rows<S, AXIS, true>(q, Nx, Ny, Nz, t, k, rowb, M);
    return sweep_xy_rows<S, AXIS, false>(q, Nx, Ny, Nz, t, k, rowb, M);
}

template <typename S, int L, bool COLS, bool DIRECT>
static hipError_t sweep_z_launch(const Launch &q, int Nx, int Ny, int Nz, const SweepTab<typename Arith<S>::T> &t,
                                 const SweepConst<typename Arith<S>::T> &k, const double *wz, const double *wy) {
    using A = typename Arith<S>::T;
    const int P = Nz / 16;
    const long nblocks = (long)((Ny + L - 1) / L) * Nx;
    dim3 grid((unsigned)nblocks, (unsigned)q.v.nb), block(L * P);
    size_t lds = (SweepShared<A, 16>::bytes(Nz, L * P, L, COLS) + 15) & ~size_t(15);
    if (!DIRECT) lds += (size_t)(Nz + Pk<S>::n) * L * sizeof(S);
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_sweep_z<S, L, 16, COLS, DIRECT>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    k_sweep_z<S, L, 16, COLS, DIRECT><<<grid, block, lds, q.s>>>(q.v, Nx, Ny, Nz, t, k, wz, wy);
    return hipGetLastError();
}

template <typename S, bool COLS, bool DIRECT>
static hipError_t sweep_z_rows(const Launch &q, int Nx, int Ny, int Nz, const SweepTab<typename Arith<S>::T> &t,
                               const SweepConst<typename Arith<S>::T> &k, const double *wz, const double *wy) {
    switch (z_rows<S>(Nz)) {
    case 64: return sweep_z_launch<S, 64, COLS, DIRECT>(q, Nx, Ny, Nz, t, k, wz, wy);
    case 32: return sweep_z_launch<S, 32, COLS, DIRECT>(q, Nx, Ny, Nz, t, k, wz, wy);
    case 16: return sweep_z_launch<S, 16, COLS, DIRECT>(q, Nx, Ny, Nz, t, k, wz, wy);
    case 8: return sweep_z_launch<S, 8, COLS, DIRECT>(q, Nx, Ny, Nz, t, k, wz, wy);
    default: return sweep_z_launch<S, 4, COLS, DIRECT>(q, Nx, Ny, Nz, t, k, wz, wy);
    }
}

// The z sweep staged through LDS or direct (DBEC_SWEEP_Z_DIRECT, else the
// tuned choice, else staged).
template <typename S, bool COLS>
static hipError_t sweep_z_dispatch(const Launch &q, int Nx, int Ny, int Nz, const SweepTabs<typename Arith<S>::T> &ts,
                                   const SweepConst<typename Arith<S>::T> &k, const double *wz, const double *wy,
                                   const Tuning &tu) {
    if (Nz % 16 != 0) return hipErrorInvalidValue;
    static const int direct_env = env_int("DBEC_SWEEP_Z_DIRECT", -1);
    const int d = direct_env >= 0 ? direct_env : tu.z_direct;
    const SweepTab<typename Arith<S>::T> t = ts.at(16);
    if (d > 0) return sweep_z_rows<S, COLS, true>(q, Nx, Ny, Nz, t, k, wz, wy);
    return sweep_z_rows<S, COLS, false>(q, Nx, Ny, Nz, t, k, wz, wy);
}

template <typename S, typename A>
static hipError_t sweep_axis(const Launch &q, const dbec_ctx *c, int axis, const typename TabOf<A>::T *base,
                             const SweepConst<A> &k, bool cols) {
    const int Nx = (int)c->Nx, Ny = (int)c->Ny, Nz = (int)c->Nz;
    const CoefLayout lay(c->Nx, c->Ny, c->Nz);
    const SweepTabs<A> t{base + lay.ca(axis), base + lay.cg(axis),
                         {base + lay.gb(axis, 0), base + lay.gb(axis, 1)},
                         {base + lay.fa(axis, 0), base + lay.fa(axis, 1)}};
    const double *wy = c->b.wgt + c->Nx, *wz = c->b.wgt + c->Nx + c->Ny;
    if (axis == 0) return sweep_xy_dispatch<S, 0>(q, Nx, Ny, Nz, t, k, c->tune);
    if (axis == 1) return sweep_xy_dispatch<S, 1>(q, Nx, Ny, Nz, t, k, c->tune);
    if (cols) return sweep_z_dispatch<S, true>(q, Nx, Ny, Nz, t, k, wz, wy, c->tune);
    return sweep_z_dispatch<S, false>(q, Nx, Ny, Nz, t, k, wz, wy, c->tune);
}

hipError_t launch_sweep(hipStream_t s, const dbec_ctx *c, int axis, const Solves &v, bool cols) {
    const auto &b = c->b;
    const Launch q{s, v};
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) {
        if (f32) {
            SweepConst<float> k;
            k.A0r = (float)c->A0r[axis][0];
            k.A = (float)c->A[axis][0];
            k.mA = -k.A;
            return sweep_axis<float>(q, c, axis, b.coef, k, cols);
        }
        SweepConst<double> k;
        k.A0r = c->A0r[axis][0];
        k.A = c->A[axis][0];
        k.mA = -c->A[axis][0];
        return sweep_axis<double>(q, c, axis, b.coef, k, cols);
    }
    // complex lines: the sweep kernels use A = i a, mA = -A, A0r = 1 + i b
    if (c->A[axis][0] != 0.0 || c->A0r[axis][0] != 1.0 || c->mA[axis][0] != 0.0 || c->mA[axis][1] != -c->A[axis][1])
        return hipErrorInvalidValue;
    if (f32) {
        SweepConst<cpx<float>> k;
        k.A0r = {(float)c->A0r[axis][0], (float)c->A0r[axis][1]};
        k.A = {(float)c->A[axis][0], (float)c->A[axis][1]};
        k.mA = {(float)c->mA[axis][0], (float)c->mA[axis][1]};
        return sweep_axis<cpx<float>>(q, c, axis, reinterpret_cast<const cpx<double> *>(b.coef), k, cols);
    }
    SweepConst<cpx<double>> k;
    k.A0r = {c->A0r[axis][0], c->A0r[axis][1]};
    k.A = {c->A[axis][0], c->A[axis][1]};
    k.mA = {c->mA[axis][0], c->mA[axis][1]};
    return sweep_axis<cpx<double>>(q, c, axis, reinterpret_cast<const cpx<double> *>(b.coef), k, cols);
}

// norm^2 = sum_x wx[x] sum_t colpart[t][x]; scal[NORM] = norm, scal[SCALE] = 1/norm.
__global__ void __launch_bounds__(256)
k_norm_cols(Solves v, int tiles, const double *__restrict__ wx, int Nx) {
    __shared__ double sh[256];
    const SolveAt sr = solve_at(v);
    norm_from_cols<256>(sr.rows, tiles, wx, Nx, sr.scal, v.shift, sh);
}

hipError_t launch_norm_from_cols(hipStream_t s, const dbec_ctx *c, const Solves &v, int tiles) {
    k_norm_cols<<<dim3(1, (unsigned)v.nb), 256, 0, s>>>(v, tiles, c->b.wgt, (int)c->Nx);
    return hipGetLastError();
}

}  // namespace dbec
