// ops.hpp - launch interfaces of the non-FFT kernels (ops.hip).
#pragma once

#include <algorithm>
#include <type_traits>

#include "internal.hpp"
#include "nu_device.hpp"

namespace dbec {

template <typename V>
struct SweepConst {
    V A0r, A, mA;  // diagonal of the explicit half, off-diagonal, and its negative
};

// Layout of the Crank-Nicolson coefficient buffer (b.coef, FP64 real or
// complex elements in both precisions): calpha and cgamma of the axes
// x, y, z back to back (n - 1 each), then the carry multipliers gb and fa of
// the partitioned sweeps (n each per axis) for segments of 16 and of 32:
//   [calpha | cgamma | gb16 | fa16 | gb32 | fa32]
struct CoefLayout {
    long tot, totn, off[3], offn[3];
    CoefLayout(long Nx, long Ny, long Nz)
        : tot(Nx + Ny + Nz - 3), totn(Nx + Ny + Nz), off{0, Nx - 1, Nx - 1 + Ny - 1}, offn{0, Nx, Nx + Ny} {}
    long ca(int a) const { return off[a]; }
    long cg(int a) const { return tot + off[a]; }
    long gb(int a, int m) const { return 2 * tot + 2 * m * totn + offn[a]; }  // m = 0: M = 16, 1: M = 32
    long fa(int a, int m) const { return 2 * tot + (2 * m + 1) * totn + offn[a]; }
    long size() const { return 2 * tot + 4 * totn; }
};

hipError_t launch_calcnu(hipStream_t s, const dbec_ctx *c, const double *scale);
hipError_t launch_scale(hipStream_t s, const dbec_ctx *c, const double *scale);
// *p = v on the stream (a one-thread kernel: also valid under graph capture)
hipError_t launch_set_scalar(hipStream_t s, double *p, double v);
// Sweep along `axis` of the solves v.
// The grid, coefficients and weights come from c.  The z sweep with cols also
// writes, per solve and (y tile t, x), rows[t][x] = sum over the tile's rows
// of wy[y] * (Simpson z integral of psi^2).
hipError_t launch_sweep(hipStream_t s, const dbec_ctx *c, int axis, const Solves &v, bool cols);
// number of y tiles of the z sweep (rows of the column partials)
long sweep_z_tiles(const dbec_ctx *c);
int sweep_z_rows(const dbec_ctx *c);
int fused_z_rows_half(const dbec_ctx *c);
// The z sweep's tables, constants, weights and rows per workgroup for the
// z sweep fused with the forward z pass.
void sweep_z_args(const dbec_ctx *c, FftArgs &a);
// One axis' sweep tables (calpha, cgamma, gb, fa for segments of 16; FP64 in
// every precision) and constants A0r, A, mA (re, im).
struct AxisArgs {
    const void *tab[4];
    double k[3][2];
};
AxisArgs sweep_axis_args(const dbec_ctx *c, int axis);
// The plane kernels (plane.hip): whether they are to carry the context's step
// (dbec_ctx::planes), the y and z sweeps and the next step's forward z and y passes (either or both),
// and the inverse y and z passes with calcnu (or writing phi).
// shared: the context's launches advance several solves and run beside other
// contexts' (the request loop).
bool plane_ok(const dbec_ctx *c, bool shared);
hipError_t launch_plane_fwd(const dbec_ctx *c, const Solves &v, bool sweeps, bool fft);
hipError_t launch_plane_inv(const dbec_ctx *c, const Solves &v, bool phi);
// norm of each solve from its column partials (`tiles` per x): scal[NORM], scal[SCALE]
hipError_t launch_norm_from_cols(hipStream_t s, const dbec_ctx *c, const Solves &v, int tiles);
TrapConst trap_const(const dbec_ctx *c);
NuConst nu_const(const dbec_ctx *c);
// Observables (observe.hip): scal[NORM], scal[SCALE], or with moments
// scal[NORM] and the rms values; scal[MU], scal[EN] from psi and phi (phase:
// complex psi's kinetic density |grad psi|^2 instead of (grad |psi|)^2).  The
// row buffer takes the partial sums; c->h_scal (may be null) the results too.
hipError_t launch_obs_norm(hipStream_t s, const dbec_ctx *c, bool moments);
hipError_t launch_obs_muen(hipStream_t s, const dbec_ctx *c, bool phase);
// device scalars, or psi[n] (entries SC_COUNT, SC_COUNT + 1), to c->h_scal
hipError_t launch_export_scalars(hipStream_t s, const dbec_ctx *c);
hipError_t launch_export_point(hipStream_t s, const dbec_ctx *c, long n);
// Density extracts (density.hip): out[a][b] = sum over `axis` of w |psi|^2 at
// every o0-th and o1-th of the other indices (in [x][y][z] order), out[a] =
// sum_b w[b] in[a][b] (axis 1) or out[b] = sum_a w[a] in[a][b] (axis 0).
hipError_t launch_reduce3(hipStream_t s, const dbec_ctx *c, int axis, long o0, long o1, double *out);
hipError_t launch_reduce2(hipStream_t s, const double *in, long n0, long n1, int axis, const double *w, double *out);
// dst[a][b][k] = |psi|^2 at (start + (a, b, k) * step), (a, b, k) < cnt
hipError_t launch_pick_mod2(hipStream_t s, const dbec_ctx *c, const long start[3], const long step[3],
                            const long cnt[3], double *dst);

}  // namespace dbec
