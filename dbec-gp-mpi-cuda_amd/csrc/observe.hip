// observe.hip - the observables: Simpson norm, rms moments, mu and E
// (calcnorm, calcrms, calcmuen: imag3d.cu:1194-1291, 1639-1750;
// real3d.cu:1304-1383, 1733-1847).
//
// Every integral is the Simpson sum of the reference (diffint.cu:37-51),
// written as weights w[i] (h/3 times 1,4,2,...,4,1 plus the even-N end
// correction) so that integral = sum wx wy wz f.  A first launch leaves one
// partial sum per workgroup and integral, a second one of a single workgroup
// adds them; both in a fixed order, so results repeat bit for bit.  (Row sums
// added by one workgroup, a serial loop over y per x, took 65-86 us at 256^3;
// the partials take 4.)  The second launch also writes the scalars to the
// context's pinned host buffer, so a call that returns them waits for the
// stream and makes no copy (about 10 us a call).
#include <type_traits>

#include "ops.hpp"
#include "sweep_device.hpp"

namespace dbec {

namespace {

// |psi|^2 as x^2 + y^2 in one FMA, as calcnu forms it
__device__ __forceinline__ double obs_mod2(double v) { return v * v; }
__device__ __forceinline__ double obs_mod2(float v) { return (double)v * (double)v; }
__device__ __forceinline__ double obs_mod2(cpx<double> v) { return fma(v.x, v.x, v.y * v.y); }
__device__ __forceinline__ double obs_mod2(cpx<float> v) {
    return fma((double)v.x, (double)v.x, (double)v.y * (double)v.y);
}

// Sum of v over the workgroup's 4 wavefronts, valid in thread 0; sh: 4 doubles
// no other call uses.
__device__ __forceinline__ double block_sum(double v, double *sh) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Partials of I0 = sum w |psi|^2 and, with MOM, of the x^2, y^2, z^2 moments:
// part[q * B + b].  A stream over psi, bound by HBM; lanes take 16-byte
// packets of a row, a wavefront as many rows at once as fit (rpw rows of lpr
// lanes), rows strided over the launch.
template <typename P, bool MOM>
__global__ void __launch_bounds__(256)
k_obs_mod2(const P *__restrict__ psi, const double *__restrict__ wgt, const double *__restrict__ sq,
           double *__restrict__ part, int Nx, int Ny, int Nz, int lpr, int rpw) {
    constexpr int VE = Pk<P>::n;
    __shared__ double sh[4][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane / lpr, c0 = lane - sub * lpr, ppr = Nz / VE;
    const double *wz = wgt + Nx + Ny, *z2 = sq + Nx + Ny;
    double s0 = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    const int rows = Nx * Ny, step = (int)gridDim.x * 4 * rpw;
    if (sub < rpw) {
        for (int row = ((int)blockIdx.x * 4 + wave) * rpw + sub; row < rows; row += step) {
            const P *r = psi + (long)row * Nz;
            double a0 = 0.0, az = 0.0;
#pragma unroll 2
            for (int c = c0; c < ppr; c += lpr) {
                const typename Pk<P>::type v = ld_pk(r + c * VE);
#pragma unroll
                for (int j = 0; j < VE; ++j) {
                    const double m = wz[c * VE + j] * obs_mod2(v.e[j]);
                    a0 += m;
                    if (MOM) az = fma(m, z2[c * VE + j], az);
                }
            }
            const int x = row / Ny, y = row - x * Ny;
            const double w = wgt[x] * wgt[Nx + y];
            s0 = fma(w, a0, s0);
            if (MOM) {
                sx = fma(w * sq[x], a0, sx);
                sy = fma(w * sq[Nx + y], a0, sy);
                sz = fma(w, az, sz);
            }
        }
    }
    const int B = gridDim.x, b = blockIdx.x;
    const double t0 = block_sum(s0, sh[0]);
    if (threadIdx.x == 0) part[b] = t0;
    if (MOM) {
        const double tx = block_sum(sx, sh[1]), ty = block_sum(sy, sh[2]), tz = block_sum(sz, sh[3]);
        if (threadIdx.x == 0) {
            part[B + b] = tx;
            part[2 * B + b] = ty;
            part[3 * B + b] = tz;
        }
    }
}

struct MuenArgs {
    TrapConst tc;
    double i12[3], i2[3];   // 1 / (12 h), 1 / (2 h) per axis
    double ikin, g, gdn;    // 1 / (3 - par), g, gd / N
    int Nx, Ny, Nz, cx, ty, tz, blocks;
};

// What a derivative is taken of: |psi| (the reference's calcmuen), or with
// PHASE the real and imaginary parts.
template <bool PHASE, typename P>
struct MuenComp {
    static constexpr int n = 1;
    static __device__ __forceinline__ void of(P v, double *f) { f[0] = (double)v; }
};
template <typename R>
struct MuenComp<false, cpx<R>> {
    static constexpr int n = 1;
    static __device__ __forceinline__ void of(cpx<R> v, double *f) { f[0] = sqrt(obs_mod2(v)); }
};
template <typename R>
struct MuenComp<true, cpx<R>> {
    static constexpr int n = 2;
    static __device__ __forceinline__ void of(cpx<R> v, double *f) {
        f[0] = (double)v.x;
        f[1] = (double)v.y;
    }
};

// Five-point derivative with the boundary rule of calcmuen_kernel1x
// (imag3d.cu:1303-1332): 0 at both ends, centred 3-point at 1 and N-2.
__device__ __forceinline__ double deriv5(double m2, double m1, double p1, double p2, int i, int n, double i12, double i2) {
    const double d5 = (m2 - p2 + 8.0 * (p1 - m1)) * i12, d3 = (p1 - m1) * i2;
    return (i == 0 || i == n - 1) ? 0.0 : ((i == 1 || i == n - 2) ? d3 : d5);
}

// Partials of the chemical potential and energy integrals (calcmuen_kernel1x/
// 1y/1z and kernel2, imag3d.cu:1293-1450; real3d.cu:1382-1543): A = kinetic +
// trap terms, C = contact + dipolar terms, mu = A + C, E = A + C / 2.
// A workgroup takes a 16 x 16 tile of (y, z) and walks cx planes of x: the x
// derivative from a queue of five planes in registers, the y and z ones from
// the plane's tile and its halo of two in LDS (two buffers, one barrier per
// plane), the next plane's loads in flight meanwhile.  So each amplitude is
// formed 1.5 times and psi is read 1.5 times, mostly from L2; reading all 13
// points per point formed 13 square roots (149 us at 192^3 complex64 with
// the library hypot, 232 us at 256^3 FP64 with 7 divisions).  A run of
// neighbouring tiles stays on one XCD, which shares the halos' lines.
template <typename P, typename R, bool PHASE>
__global__ void __launch_bounds__(256)
k_obs_muen(const P *__restrict__ psi, const R *__restrict__ phi, const double *__restrict__ sq,
           const double *__restrict__ wgt, MuenArgs a, double *__restrict__ part) {
    using MC = MuenComp<PHASE, P>;
    constexpr int NC = MC::n, W = 21;
    __shared__ double tile[2][NC][20 * W];
    __shared__ double sh[2][4];
    const int tid = threadIdx.x;
    const int Nx = a.Nx, Ny = a.Ny, Nz = a.Nz;
    const int per = (a.blocks + 7) / 8, b = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (b >= a.blocks) return;
    const int tiles = a.ty * a.tz, chunk = b / tiles, t = b - chunk * tiles;
    const int y0 = t / a.tz * 16, z0 = (t % a.tz) * 16;
    const int x0 = chunk * a.cx, x1 = min(x0 + a.cx, Nx);
    const int ry = tid >> 4, rz = tid & 15, j = y0 + ry, k = z0 + rz;
    // halo point of threads 0..127: two rows above and below, two columns on
    // either side (clamped into the plane; the boundary rule does not use those)
    int hy, hz;
    if (tid < 64) {
        const int r = tid >> 4;
        hy = r < 2 ? r - 2 : 14 + r;
        hz = tid & 15;
    } else {
        const int c = tid & 3;
        hy = (tid >> 2) & 15;
        hz = c < 2 ? c - 2 : 14 + c;
    }
    const bool halo = tid < 128;
    const long NyNz = (long)Ny * Nz;
    const long own = (long)j * Nz + k;
    const long hal = (long)min(max(y0 + hy, 0), Ny - 1) * Nz + min(max(z0 + hz, 0), Nz - 1);
    const int own_at = (ry + 2) * W + rz + 2, hal_at = (hy + 2) * W + hz + 2;
    const double wyz = wgt[Nx + j] * wgt[Nx + Ny + k];
    const double y2 = sq[Nx + j], pz = trap_z(a.tc, sq[Nx + Ny + k]);
    double q[NC][5] = {};
    double sA = 0.0, sC = 0.0;
    const auto at = [&](int p) { return (long)min(max(p, 0), Nx - 1) * NyNz; };
    P nv = psi[at(x0 - 2) + own], nh = halo ? psi[at(x0 - 2) + hal] : P{};
    R nf = phi[at(x0 - 2) + own];
    for (int p = x0 - 2; p < x1 + 2; ++p) {
        const P v = nv, vh = nh;
        const R f = nf;
        nv = psi[at(p + 1) + own];
        if (halo) nh = psi[at(p + 1) + hal];
        nf = phi[at(p + 1) + own];
        double c[NC], ch[NC];
        MC::of(v, c);
#pragma unroll
        for (int n = 0; n < NC; ++n) {
#pragma unroll
            for (int u = 0; u < 4; ++u) q[n][u] = q[n][u + 1];
            q[n][4] = c[n];
        }
        if (p >= x0 && p < x1) {  // uniform
            double *tl = &tile[p & 1][0][0];
            if (halo) MC::of(vh, ch);
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                tl[n * 20 * W + own_at] = c[n];
                if (halo) tl[n * 20 * W + hal_at] = ch[n];
            }
            __syncthreads();
            double kin = 0.0;
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                const double *o = tl + n * 20 * W + own_at;
                const double dy = deriv5(o[-2 * W], o[-W], o[W], o[2 * W], j, Ny, a.i12[1], a.i2[1]);
                const double dz = deriv5(o[-2], o[-1], o[1], o[2], k, Nz, a.i12[2], a.i2[2]);
                kin = fma(dy, dy, fma(dz, dz, kin));
            }
            const double m = obs_mod2(v), w = wgt[p] * wyz;
            const double pot = trap_sum(a.tc, trap_xy(a.tc, sq[p], y2), pz);
            sA = fma(w, fma(pot, m, kin * a.ikin), sA);
            sC = fma(w, fma(a.g, m, (double)f * a.gdn) * m, sC);
        }
        const int i = p - 2;
        if (i >= x0 && i < x1) {  // uniform
            double kin = 0.0;
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                const double dx = deriv5(q[n][0], q[n][1], q[n][3], q[n][4], i, Nx, a.i12[0], a.i2[0]);
                kin = fma(dx, dx, kin);
            }
            sA = fma(wgt[i] * wyz, kin * a.ikin, sA);
        }
    }
    const double tA = block_sum(sA, sh[0]), tC = block_sum(sC, sh[1]);
    if (tid == 0) {
        part[b] = tA;
        part[a.blocks + b] = tC;
    }
}

// The integrals from the partials, one workgroup; the scalars in scal and,
// where there is one, in the pinned host copy.
//   FIN_NORM: NORM = sqrt(I0), SCALE = 1 / NORM
//   FIN_MOM:  NORM, RX / RY / RZ = sqrt(<x^2>, <y^2>, <z^2>), R0
//   FIN_EN:   MU, EN
enum { FIN_NORM, FIN_MOM, FIN_EN };
template <int MODE>
__global__ void __launch_bounds__(256)
k_obs_final(const double *__restrict__ part, int B, double *__restrict__ scal, double *host) {
    constexpr int Q = MODE == FIN_NORM ? 1 : (MODE == FIN_MOM ? 4 : 2);
    __shared__ double sh[Q][4];
    double s[Q] = {};
    for (int i = threadIdx.x; i < B; i += 256)
#pragma unroll
        for (int q = 0; q < Q; ++q) s[q] += part[q * B + i];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        s[q] = wave_sum(s[q]);
        if ((threadIdx.x & 63) == 0) sh[q][threadIdx.x >> 6] = s[q];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) s[q] = (sh[q][0] + sh[q][1]) + (sh[q][2] + sh[q][3]);
    const auto put = [&](int k, double v) {
        scal[k] = v;
        if (host) host[k] = v;
    };
    if constexpr (MODE == FIN_EN) {
        put(SC_MU, s[0] + s[1]);
        put(SC_EN, s[0] + 0.5 * s[1]);
    } else {
        const double norm = sqrt(s[0]);
        put(SC_NORM, norm);
        if constexpr (MODE == FIN_NORM) {
            put(SC_SCALE, 1.0 / norm);
        } else {
            const double rx = sqrt(s[1]), ry = sqrt(s[2]), rz = sqrt(s[3]);
            put(SC_RX, rx);
            put(SC_RY, ry);
            put(SC_RZ, rz);
            put(SC_R0, sqrt(rx * rx + ry * ry + rz * rz));
        }
    }
}

// scal[0, SC_COUNT) to the pinned host copy
__global__ void k_export_scalars(const double *__restrict__ scal, double *host) {
    if (threadIdx.x < SC_COUNT) host[threadIdx.x] = scal[threadIdx.x];
}
// psi[n] as {re, im} to the pinned host copy, entries SC_COUNT and SC_COUNT + 1
__device__ __forceinline__ void put_point(double *o, double v) { o[0] = v, o[1] = 0.0; }
__device__ __forceinline__ void put_point(double *o, float v) { o[0] = (double)v, o[1] = 0.0; }
__device__ __forceinline__ void put_point(double *o, cpx<double> v) { o[0] = v.x, o[1] = v.y; }
__device__ __forceinline__ void put_point(double *o, cpx<float> v) { o[0] = (double)v.x, o[1] = (double)v.y; }
template <typename P>
__global__ void k_export_point(const P *__restrict__ psi, long n, double *host) {
    put_point(host + SC_COUNT, psi[n]);
}

template <typename F>
hipError_t with_psi(const dbec_ctx *c, F &&f) {
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) {
        if (f32) f(static_cast<const float *>(c->b.psi), static_cast<const float *>(c->b.phi));
        else f(static_cast<const double *>(c->b.psi), static_cast<const double *>(c->b.phi));
    } else {
        if (f32) f(static_cast<const cpx<float> *>(c->b.psi), static_cast<const float *>(c->b.phi));
        else f(static_cast<const cpx<double> *>(c->b.psi), static_cast<const double *>(c->b.phi));
    }
    return hipGetLastError();
}

// Workgroups of the streaming sums: 8 per CU, at least a row per wavefront;
// 4 partials each fit the row buffer (2 Nx Ny doubles).
int mod2_blocks(long rows, int rpw) { return (int)std::max(1L, std::min(2048L, rows / (4 * rpw))); }

}  // namespace

hipError_t launch_obs_norm(hipStream_t s, const dbec_ctx *c, bool moments) {
    return with_psi(c, [&](auto *psi, auto *) {
        using P = typename std::remove_cv<typename std::remove_pointer<decltype(psi)>::type>::type;
        const int ppr = (int)(c->Nz / Pk<P>::n), lpr = std::min(64, ppr), rpw = 64 / lpr;
        const int B = mod2_blocks(c->Nx * c->Ny, rpw);
        const int Nx = (int)c->Nx, Ny = (int)c->Ny, Nz = (int)c->Nz;
        if (moments) {
            k_obs_mod2<P, true><<<B, 256, 0, s>>>(psi, c->b.wgt, c->b.sq, c->b.rows, Nx, Ny, Nz, lpr, rpw);
            k_obs_final<FIN_MOM><<<1, 256, 0, s>>>(c->b.rows, B, c->b.scal, c->h_scal);
        } else {
            k_obs_mod2<P, false><<<B, 256, 0, s>>>(psi, c->b.wgt, c->b.sq, c->b.rows, Nx, Ny, Nz, lpr, rpw);
            k_obs_final<FIN_NORM><<<1, 256, 0, s>>>(c->b.rows, B, c->b.scal, c->h_scal);
        }
    });
}

hipError_t launch_obs_muen(hipStream_t s, const dbec_ctx *c, bool phase) {
    MuenArgs a;
    a.tc = trap_const(c);
    const double h[3] = {c->p.dx, c->p.dy, c->p.dz};
    for (int i = 0; i < 3; i++) {
        a.i12[i] = 1.0 / (12.0 * h[i]);
        a.i2[i] = 1.0 / (2.0 * h[i]);
    }
    a.ikin = 1.0 / (3.0 - c->p.par);
    a.g = c->g;
    a.gdn = c->gd / (double)(c->Nx * c->Ny * c->Nz);
    a.Nx = (int)c->Nx;
    a.Ny = (int)c->Ny;
    a.Nz = (int)c->Nz;
    a.ty = a.Ny / 16;
    a.tz = a.Nz / 16;
    // planes per workgroup: 2048 workgroups (8 per CU), at least 4 planes
    // (each walk reads 4 more)
    a.cx = std::max(4, (int)((c->Nx * a.ty * a.tz + 2047) / 2048));
    a.blocks = a.ty * a.tz * ((a.Nx + a.cx - 1) / a.cx);
    const unsigned grid = (unsigned)((a.blocks + 7) / 8 * 8);
    return with_psi(c, [&](auto *psi, auto *phi) {
        using P = typename std::remove_cv<typename std::remove_pointer<decltype(psi)>::type>::type;
        using R = typename std::remove_cv<typename std::remove_pointer<decltype(phi)>::type>::type;
        if constexpr (!std::is_floating_point<P>::value) {
            if (phase) k_obs_muen<P, R, true><<<grid, 256, 0, s>>>(psi, phi, c->b.sq, c->b.wgt, a, c->b.rows);
        }
        if (std::is_floating_point<P>::value || !phase)
            k_obs_muen<P, R, false><<<grid, 256, 0, s>>>(psi, phi, c->b.sq, c->b.wgt, a, c->b.rows);
        k_obs_final<FIN_EN><<<1, 256, 0, s>>>(c->b.rows, a.blocks, c->b.scal, c->h_scal);
    });
}

hipError_t launch_export_scalars(hipStream_t s, const dbec_ctx *c) {
    k_export_scalars<<<1, 64, 0, s>>>(c->b.scal, c->h_scal);
    return hipGetLastError();
}

hipError_t launch_export_point(hipStream_t s, const dbec_ctx *c, long n) {
    return with_psi(c, [&](auto *psi, auto *) {
        using P = typename std::remove_cv<typename std::remove_pointer<decltype(psi)>::type>::type;
        k_export_point<P><<<1, 1, 0, s>>>(psi, n, c->h_scal);
    });
}

}  // namespace dbec
