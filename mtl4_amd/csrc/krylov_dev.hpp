// krylov_dev.hpp -- the loop head of the recurrences on the device: what MTL4
// decides on the host between iterations, run by the lane that finishes a
// reduction.
#pragma once

#include <cmath>

#include "krylov.hpp"

namespace mtl4g {

enum { PCM_NONE = 0, PCM_DIAG = 1, PCM_GENERAL = 2 };

// basic_iteration::finished(Real) (basic_iteration.hpp:60-65,85-93,43-48)
// followed by ++iter when the loop goes on.  NaN/Inf residuals stop the
// solve with MTL4G_ERR_NONFINITE instead of running to max_iter.
// finished() alone (no ++iter): sets done when the loop must stop
__device__ __forceinline__ void iter_check(Ctl* c, double resid, double* hist) {
    if (c->hist_n < c->hist_cap) hist[c->hist_n] = resid;
    c->hist_n++;
    c->resid = resid;
    const bool conv = c->norm_r0 == 0 ? (resid <= c->atol)
                                      : (resid <= c->rtol * c->norm_r0 || resid <= c->atol);
    if (conv) { c->done = 1; return; }
    if (c->i >= c->max_iter) { c->error = 1; c->done = 1; return; }
    if (!isfinite(resid)) { c->status = MTL4G_ERR_NONFINITE; c->done = 1; return; }
}

__device__ __forceinline__ void iter_finished(Ctl* c, double resid, double* hist) {
    iter_check(c, resid, hist);
    if (c->done) return;
    c->i++;
    c->first = c->i <= 1;
}

__device__ __forceinline__ bool conv_test(const Ctl* c, double resid) {
    return c->norm_r0 == 0 ? (resid <= c->atol) : (resid <= c->rtol * c->norm_r0 || resid <= c->atol);
}

// A recurrence residual this far above the last FP64 residual is refreshed
// at once instead of iterating on.
constexpr double kGrowth = 10.0;
// Mixed-precision BiCGSTAB refreshes when its residual fell by this factor.
constexpr double kBicgDelta = 1e-5;

// Mixed precision, loop head on the recurrence residual: it only estimates
// convergence, so an estimated stop (or the iteration limit) pauses the
// recurrence and asks for an FP64 refresh, which decides.  A non-finite
// residual also pauses it and discards the low-precision correction; a
// residual that has grown by kGrowth since the last refresh is refreshed
// before the recurrence goes on.
__device__ __forceinline__ void mixed_check(Ctl* c, double resid32) {
    if (!isfinite(resid32)) { c->want_ru = 1; c->pause = 1; c->drop = 1; return; }
    if (conv_test(c, resid32)) { c->want_ru = 1; c->pause = 1; return; }
    if (c->i >= c->max_iter) { c->want_ru = 1; c->pause = 1; c->limit = 1; return; }
    if (resid32 > kGrowth * c->rmax) { c->want_ru = 1; c->pause = 1; return; }
    c->i++;
    c->first = c->i <= 1;
    if (resid32 <= c->delta * c->rmax) c->want_ru = 1;
}

}  // namespace mtl4g
