// transfer.hpp - fields between device memory and the caller's host arrays of
// doubles.
#pragma once

#include <cstddef>

#include "internal.hpp"

namespace dbec {

// n values at src (double, or float with f32) into dst; waits for the stream.
hipError_t fetch_field(const dbec_ctx *c, double *dst, const void *src, size_t n, bool f32);
// The same for doubles in one copy, without an allocation of any kind.
hipError_t fetch_plain(const dbec_ctx *c, double *dst, const double *src, size_t n);
// n doubles at src into dst (double, or rounded to float with f32); waits for
// the stream.
hipError_t store_field(const dbec_ctx *c, void *dst, const double *src, size_t n, bool f32);
// A context came into being or ended: the last one gives the staging buffers back.
void staging_user(int change);

}  // namespace dbec
