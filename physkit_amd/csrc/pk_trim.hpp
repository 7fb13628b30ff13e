// The Morton grid's range (k_broad.hip): the bounds of the bulk of the leaves on each axis,
// from a sample of them, so that a few bodies far away (fallen off the ground, flung off by
// an unstable contact) do not squeeze all others into a handful of cells, which leaves the
// hierarchy without spatial order and lets every query walk most of a world.
#pragma once
#include "pk_math.hpp"

namespace pk
{

constexpr uint32_t kTrimSample = 1024;

// Sample t of n > kTrimSample bodies: one from each of 1,024 stretches of the ids, at a
// hashed place. A fixed place would pick the same body of every world of a batch of 1,024
// (or any multiple) worlds of one size, for one their ground, whose one centroid then left
// the grid no extent (1,024 worlds of 256 bodies: pair query 0.65 ms a step, 0.38 so).
PK_HD uint32_t trim_sample(uint32_t t, uint32_t n)
{
    const uint64_t lo = static_cast<uint64_t>(t) * n / kTrimSample, hi = (static_cast<uint64_t>(t) + 1) * n / kTrimSample;
    return static_cast<uint32_t>(lo + mix32(t) % (hi - lo));
}

// The bulk on one axis from `finite` > 0 sorted centroids: without a 64th at either end,
// widened by half its extent each way, and then as far as leaves out a 256th of the leaves (or
// one sample) at either end at most: leaves outside share the border cells.
PK_HD void trim_axis(const double *v, int finite, double &lo, double &hi)
{
    const int few = finite < 256 ? (finite >= 64 ? 1 : 0) : finite / 256;
    const double a = v[finite / 64], b = v[finite - 1 - finite / 64], half = (b - a) * 0.5;
    lo = fmin(a - half, v[few]);
    hi = fmax(b + half, v[finite - 1 - few]);
}

// The grid's range on an axis from its exact bounds and its bulk, `widest` the longest bulk of
// the three axes: cells stay no flatter than cubes where the exact bounds are as wide. A layer of
// bodies at rest would otherwise be ordered by the differences of their heights, which
// mean nothing, before their places in it.
PK_HD void trim_range(double exact_lo, double exact_hi, double bulk_lo, double bulk_hi, double widest, double &lo,
                      double &hi)
{
    lo = exact_lo;
    hi = exact_hi;
    if (!(widest > 0.0)) return;
    const double grow = (widest - (bulk_hi - bulk_lo)) * 0.5;
    lo = fmax(exact_lo, grow > 0.0 ? bulk_lo - grow : bulk_lo);
    hi = fmin(exact_hi, grow > 0.0 ? fmax(bulk_hi + grow, lo + widest) : bulk_hi);
    if (grow > 0.0) lo = fmax(exact_lo, fmin(lo, hi - widest));
}

} // namespace pk
