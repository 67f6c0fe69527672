// plane_device.hpp - transforms of run-time length over lines held in LDS,
// for the plane kernels (plane.hip).
//
// Lengths n = 8 q with q in {2, 4, 6, 8, 10, 12, 16}: two in-place passes,
// radix 8 and radix q, so one compiled kernel serves every such length and a
// line needs two passes where the compile-time plans take two or three.  The
// result of the forward transform is left in digit order: X[c + 8 d] in slot
// q c + d (fft_slot); the inverse starts from that order and ends in natural
// order.  Element e of line l sits at buf[e * st + l]: lanes run along the
// lines, so every access of a pass is a contiguous run and conflict-free
// whatever the length.
#pragma once

#include "fft_device.hpp"

namespace dbec {

// Index arithmetic in 24-bit multiplies: the 32-bit integer multiply (low or
// high half) issues at a quarter of the rate, and the planes' run-time strides
// need several per element.  Every factor here is below 2^24, every product
// below 2^31.
__device__ __forceinline__ int m24(int a, int b) { return (int)__umul24((unsigned)a, (unsigned)b); }

// i / d for 0 <= i <= 2^14 and 0 < d <= 2^9 as (i m) >> s with s = 14 +
// ceil(log2 d) and m = ceil(2^s / d): the excess i (m d - 2^s) <= i d <= 2^s
// stays below one unit (equal only for m d - 2^s = d, which no m has), and i m
// < 2^14 (2^15 + 1).
struct FastDiv {
    unsigned m, d, s;
    __host__ __device__ static FastDiv of(unsigned d) {
        FastDiv f;
        f.d = d;
        f.s = 14;
        while ((1u << (f.s - 14)) < d) ++f.s;
        f.m = ((1u << f.s) + d - 1) / d;
        return f;
    }
    __device__ __forceinline__ int div(int i) const { return (int)(__umul24((unsigned)i, m) >> s); }
    __device__ __forceinline__ void divmod(int i, int &q, int &r) const {
        q = div(i);
        r = i - m24(q, (int)d);
    }
};

// v, unknown to the compiler: an index formed from it is computed where it is
// used instead of being kept in registers since an earlier use.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

inline bool plane_len(long n) {
    switch (n) {
    case 16: case 32: case 48: case 64: case 80: case 96: case 128: return true;
    default: return false;
    }
}

// slot of frequency k in the digit order of a length 8 q
__device__ __forceinline__ int fft_slot(int k, int q) { return m24(k & 7, q) + (k >> 3); }

// Radix-8 pass: butterfly j of a line takes slots j + q r.  Forward: first
// pass, followed by the twiddles w^(j c); inverse: last pass, none.
template <int DIR, typename R>
__device__ __forceinline__ void pass8(cpx<R> *buf, int st, const FastDiv &nl, int q, const cpx<R> *tw, int tid, int nt) {
    const int items = m24(q, (int)nl.d), s = m24(q, st);
    for (int i = tid; i < items; i += nt) {
        int j, l;
        nl.divmod(i, j, l);
        cpx<R> *p = buf + m24(j, st) + l;
        cpx<R> v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = p[r * s];
        dft8<DIR>(v);
        if constexpr (DIR < 0) {
#pragma unroll
            for (int c = 1; c < 8; ++c) v[c] = cmul(v[c], tw[m24(j, c)]);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) p[r * s] = v[r];
    }
}

// Radix-q pass: butterfly c takes the q consecutive slots q c + j.  Forward:
// last pass; inverse: first pass, followed by the conjugate twiddles.
template <int Q, int DIR, typename R>
__device__ __forceinline__ void passq_t(cpx<R> *buf, int st, const FastDiv &nl, const cpx<R> *tw, int tid, int nt) {
    for (int i = tid; i < 8 * (int)nl.d; i += nt) {
        int c, l;
        nl.divmod(i, c, l);
        cpx<R> *p = buf + m24(Q * c, st) + l;
        cpx<R> v[Q];
#pragma unroll
        for (int r = 0; r < Q; ++r) v[r] = p[r * st];
        dft<Q, DIR>(v);
        if constexpr (DIR > 0) {
#pragma unroll
            for (int j = 1; j < Q; ++j) v[j] = cmulc(v[j], tw[m24(j, c)]);
        }
#pragma unroll
        for (int r = 0; r < Q; ++r) p[r * st] = v[r];
    }
}
template <int DIR, typename R>
__device__ __forceinline__ void passq(cpx<R> *buf, int st, const FastDiv &nl, int q, const cpx<R> *tw, int tid, int nt) {
    switch (q) {  // uniform
    case 2: passq_t<2, DIR>(buf, st, nl, tw, tid, nt); break;
    case 4: passq_t<4, DIR>(buf, st, nl, tw, tid, nt); break;
    case 6: passq_t<6, DIR>(buf, st, nl, tw, tid, nt); break;
    case 8: passq_t<8, DIR>(buf, st, nl, tw, tid, nt); break;
    case 10: passq_t<10, DIR>(buf, st, nl, tw, tid, nt); break;
    case 12: passq_t<12, DIR>(buf, st, nl, tw, tid, nt); break;
    default: passq_t<16, DIR>(buf, st, nl, tw, tid, nt); break;
    }
}

// The lines' transform; every thread of the workgroup calls it, with the
// lines complete in LDS (the caller's barrier); on return they are again.
template <int DIR, typename R>
__device__ __forceinline__ void fft_lines(cpx<R> *buf, int st, const FastDiv &nl, int q, const cpx<R> *tw, int tid, int nt) {
    if constexpr (DIR < 0) {
        pass8<DIR>(buf, st, nl, q, tw, tid, nt);
        __syncthreads();
        passq<DIR>(buf, st, nl, q, tw, tid, nt);
    } else {
        passq<DIR>(buf, st, nl, q, tw, tid, nt);
        __syncthreads();
        pass8<DIR>(buf, st, nl, q, tw, tid, nt);
    }
    __syncthreads();
}

}  // namespace dbec
