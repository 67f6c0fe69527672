// density.hip - density extracts of the output writers (outden*, outpsi2*,
// imag3d.cu:1944-2399; real3d.cu:2042-2522): weighted sums of |psi|^2 over one
// or two axes, and sampled values.
//
// All of them stream psi once and are bound by HBM.  Sums over z give a
// wavefront per row (16-byte packets, lanes along z); sums over x or y give
// lanes along z and 8 wavefronts per workgroup that share the summed axis.
// One thread per output, which walked its row alone, took 55 us at 256^3
// FP64 for the 3-D sums and 55 us more for the 2-D ones.  Sums run in a fixed
// order, so results repeat bit for bit.  The sums form the sampled outputs
// only, packed (a launch of their own to pick those from all cost 1.5-2 us of
// the 27-30 that an extract takes at 16^3).
#include <type_traits>

#include "ops.hpp"
#include "sweep_device.hpp"

namespace dbec {

namespace {

// |psi|^2 as x^2 + y^2 in one FMA, as calcnu forms it
__device__ __forceinline__ double mod2_of(double v) { return v * v; }
__device__ __forceinline__ double mod2_of(float v) { return (double)v * (double)v; }
__device__ __forceinline__ double mod2_of(cpx<double> v) { return fma(v.x, v.x, v.y * v.y); }
__device__ __forceinline__ double mod2_of(cpx<float> v) {
    return fma((double)v.x, (double)v.x, (double)v.y * (double)v.y);
}

// out[a][b] = sum_z w[z] |psi|^2 at (a ox, b oy), a wavefront per row
template <typename P>
__global__ void __launch_bounds__(256)
k_sum_z(const P *__restrict__ psi, const double *__restrict__ w, double *__restrict__ out, int rows, int cb, int ox,
        int oy, int Ny, int Nz) {
    constexpr int VE = Pk<P>::n;
    const int lane = threadIdx.x & 63, row = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (row >= rows) return;  // uniform in the wavefront
    const int a = row / cb, b = row - a * cb;
    const P *r = psi + ((long)(a * ox) * Ny + b * oy) * Nz;
    double acc = 0.0;
    for (int c = lane; c < Nz / VE; c += 64) {
        const typename Pk<P>::type v = ld_pk(r + c * VE);
#pragma unroll
        for (int j = 0; j < VE; ++j) acc = fma(w[c * VE + j], mod2_of(v.e[j]), acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) out[row] = acc;
}

// out[o][k] = sum_a w[a] |psi|^2 at o * os + a * as + k oz (k < cz): lanes along
// z, the 8 wavefronts of a workgroup share the summed axis
template <typename P>
__global__ void __launch_bounds__(512)
k_sum_strided(const P *__restrict__ psi, const double *__restrict__ w, double *__restrict__ out, int na, long as,
              long os, int Nz, int oz, int cz) {
    __shared__ double sh[8][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int zt = (Nz + 63) / 64, o = (int)blockIdx.x / zt, z = ((int)blockIdx.x % zt) * 64 + lane;
    const P *p = psi + (long)o * os + (z < Nz ? z : 0);
    double acc = 0.0;
#pragma unroll 8
    for (int a = wave; a < na; a += 8) acc = fma(w[a], mod2_of(p[(long)a * as]), acc);
    sh[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && z < Nz && z % oz == 0) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += sh[q][lane];
        out[(long)o * cz + z / oz] = t;
    }
}

// 2-D sums: axis 1, out[a] = sum_b w[b] in[a][b], a wavefront per a; axis 0,
// out[b] = sum_a w[a] in[a][b], 64 outputs per workgroup of 8 wavefronts
__global__ void __launch_bounds__(256)
k_reduce2_rows(const double *__restrict__ in, int n0, int n1, const double *__restrict__ w, double *__restrict__ out) {
    const int lane = threadIdx.x & 63, row = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (row >= n0) return;
    double acc = 0.0;
    for (int b = lane; b < n1; b += 64) acc = fma(w[b], in[(long)row * n1 + b], acc);
    acc = wave_sum(acc);
    if (lane == 0) out[row] = acc;
}
__global__ void __launch_bounds__(512)
k_reduce2_cols(const double *__restrict__ in, int n0, int n1, const double *__restrict__ w, double *__restrict__ out) {
    __shared__ double sh[8][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, b = (int)blockIdx.x * 64 + lane;
    double acc = 0.0;
#pragma unroll 8
    for (int a = wave; a < n0; a += 8) acc = fma(w[a], in[(long)a * n1 + (b < n1 ? b : 0)], acc);
    sh[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && b < n1) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += sh[q][lane];
        out[b] = t;
    }
}

// dst[t] = |psi|^2 at (x0 + a ox, y0 + b oy, z0 + k oz), t = (a cy + b) cz + k
template <typename P>
__global__ void __launch_bounds__(256)
k_pick_mod2(const P *__restrict__ psi, int x0, int y0, int z0, int ox, int oy, int oz, unsigned cy, unsigned cz,
            unsigned n, double *__restrict__ dst, int Ny, int Nz) {
    const unsigned t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n) return;
    const unsigned row = t / cz, k = t - row * cz, a = row / cy, b = row - a * cy;
    dst[t] = mod2_of(psi[((long)(x0 + (int)a * ox) * Ny + y0 + (int)b * oy) * Nz + z0 + (int)k * oz]);
}

template <typename F>
hipError_t with_psi(const dbec_ctx *c, F &&f) {
    const bool f32 = c->prec == DBEC_MIXED;
    if (c->mode == DBEC_IMAG) {
        if (f32) f(static_cast<const float *>(c->b.psi));
        else f(static_cast<const double *>(c->b.psi));
    } else {
        if (f32) f(static_cast<const cpx<float> *>(c->b.psi));
        else f(static_cast<const cpx<double> *>(c->b.psi));
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_reduce3(hipStream_t s, const dbec_ctx *c, int axis, long o0, long o1, double *out) {
    const double *w = c->b.wgt + (axis == 0 ? 0 : (axis == 1 ? c->Nx : c->Nx + c->Ny));
    const long Nx = c->Nx, Ny = c->Ny, Nz = c->Nz, zt = (Nz + 63) / 64;
    const long n0 = axis == 0 ? Ny : Nx, n1 = axis == 2 ? Ny : Nz;
    o0 = std::min(o0, n0);  // (one sample either way)
    o1 = std::min(o1, n1);
    const long c0 = (n0 - 1) / o0 + 1, c1 = (n1 - 1) / o1 + 1;
    return with_psi(c, [&](auto *psi) {
        using P = typename std::remove_cv<typename std::remove_pointer<decltype(psi)>::type>::type;
        if (axis == 2)
            k_sum_z<P><<<(unsigned)((c0 * c1 + 3) / 4), 256, 0, s>>>(psi, w, out, (int)(c0 * c1), (int)c1, (int)o0, (int)o1,
                                                                     (int)Ny, (int)Nz);
        else if (axis == 1)  // out[x][z]
            k_sum_strided<P><<<(unsigned)(c0 * zt), 512, 0, s>>>(psi, w, out, (int)Ny, Nz, o0 * Ny * Nz, (int)Nz, (int)o1,
                                                                 (int)c1);
        else  // out[y][z]
            k_sum_strided<P><<<(unsigned)(c0 * zt), 512, 0, s>>>(psi, w, out, (int)Nx, Ny * Nz, o0 * Nz, (int)Nz, (int)o1,
                                                                 (int)c1);
    });
}

hipError_t launch_reduce2(hipStream_t s, const double *in, long n0, long n1, int axis, const double *w, double *out) {
    if (axis == 1) k_reduce2_rows<<<(unsigned)((n0 + 3) / 4), 256, 0, s>>>(in, (int)n0, (int)n1, w, out);
    else k_reduce2_cols<<<(unsigned)((n1 + 63) / 64), 512, 0, s>>>(in, (int)n0, (int)n1, w, out);
    return hipGetLastError();
}

hipError_t launch_pick_mod2(hipStream_t s, const dbec_ctx *c, const long start[3], const long step[3],
                            const long cnt[3], double *dst) {
    const long n = cnt[0] * cnt[1] * cnt[2];  // at most 512^3
    if (n <= 0) return hipSuccess;
    return with_psi(c, [&](auto *psi) {
        using P = typename std::remove_cv<typename std::remove_pointer<decltype(psi)>::type>::type;
        k_pick_mod2<P><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(psi, (int)start[0], (int)start[1], (int)start[2],
                                                                   (int)step[0], (int)step[1], (int)step[2],
                                                                   (unsigned)cnt[1], (unsigned)cnt[2], (unsigned)n, dst,
                                                                   (int)c->Ny, (int)c->Nz);
    });
}

}  // namespace dbec
