// Shared by the kernels that march 64-cell columns of the flattened (y, z) plane over x (the half steps and
// the adjoint): accesses at a uniform base plus a 32-bit lane offset, CPML rows of a lane, and the launch
// shape.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"

namespace {

// The three components of one cell, read as one 12-byte (24-byte) access through a global pointer.
template <typename real>
struct Cell {
    real v[3];
};

template <typename real>
__device__ __forceinline__ Cell<real> cell_at(const real* base, long long i) {
    const auto p = global(base + 3 * i);
    return Cell<real>{{p[0], p[1], p[2]}};
}

template <typename real>
struct PlaneAxis {          // CPML rows of one axis, shared by its two terms: low side, then high side
    int lo[2], hi[2];       // empty: lo == hi == 0
    unsigned psi[2];        // byte offset of each term's low-side memory in the family's buffer
    unsigned high[2];       // what to add for the high side
    unsigned coef, coef_high;   // byte offset of b | c | inv_k of the low side, and what to add for the high side
};

// A value at a uniform base plus a 32-bit byte offset of the lane.
template <typename real>
__device__ __forceinline__ real at_byte(const real* base, unsigned off) {
    return *global(reinterpret_cast<const real*>(reinterpret_cast<const char*>(base) + off));
}

template <typename real>
__device__ __forceinline__ void put_byte(real* base, unsigned off, real v) {
    *global(reinterpret_cast<real*>(reinterpret_cast<char*>(base) + off)) = v;
}

template <typename real>
__device__ __forceinline__ Cell<real> cell_at_byte(const real* base, unsigned off) {
    const auto p = global(reinterpret_cast<const real*>(reinterpret_cast<const char*>(base) + off));
    return Cell<real>{{p[0], p[1], p[2]}};
}

// The CPML row of the y or z axis a lane lies in: the memory of its two terms and their coefficients.
template <typename real>
struct PlaneHit {
    bool on;
    unsigned at[2];     // byte offsets of the two terms' memory in the current plane
    unsigned stride;    // bytes per x plane
    real b, c, ik;
};

// The row k of an axis: w is its slab's width; `on` false leaves the rest unused.
template <typename real>
struct AxisRow {
    bool on;
    int q, w;
    unsigned psi[2], coef;
};

template <typename real>
__device__ __forceinline__ AxisRow<real> axis_row(const PlaneAxis<real>& p, int k, bool inside) {
    const int k0 = k - p.lo[0], k1 = k - p.lo[1], w0 = p.hi[0] - p.lo[0], w1 = p.hi[1] - p.lo[1];
    const bool low = (unsigned)k0 < (unsigned)w0, high = (unsigned)k1 < (unsigned)w1;
    AxisRow<real> r;
    r.on = inside & (low | high);
    r.q = low ? k0 : k1;
    r.w = low ? w0 : w1;
    for (int t = 0; t < 2; ++t) r.psi[t] = p.psi[t] + (low ? 0u : p.high[t]);
    r.coef = p.coef + (low ? 0u : p.coef_high);
    return r;
}

// The wavefront's number among those of its grid, as a scalar.
__device__ __forceinline__ unsigned wave_item(unsigned block) {
    return block * 4u + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// t % modulus, in 32 bits where both fit.
__device__ __forceinline__ long long slot_of(long long t, long long modulus) {
    if (((t | modulus) >> 31) == 0) return (long long)((unsigned)t % (unsigned)modulus);
    return t % modulus;
}

constexpr unsigned kXcdRun = 128;

// A launch holds fewer than 2^32 threads: wavefronts of a march, patches of 1024 threads.
constexpr long long kLaunchItems = 0x3ffffffLL & ~3LL, kLaunchPatches = 0x3fffffLL;

// Planes per march: two share the lane's set-up and the plane between them.  us a step with 1 / 2 / 4 planes: 160x120x40
// cells (12,000 column-planes) 17.6 / 16.8 / 17.6, 200x160x60 33.3 / 31.9 / 33.3, 192^3 102 / 95.6 / 95.3, 256^3 286 / 283 /
// 292, FP64 97x83x61 (7,760) 19.2 / 19.1 / 20.3.  A grid of few wavefronts keeps one, as it needs them all to fill the
// chip: 6.0 us against 7.2 on 160x120x1, 320 column-planes.
constexpr long long kSpanItems = 4096;

// Workgroups that one XCD takes in a row: neighbouring rows and planes are then read through one L2.
// Runs of 1 / 32 / 128 / 384 take 37.5 / 34.0 / 31.9 / 32.0 us on 200x160x60 cells, 108 / 96.7 / 95.6 / 92.6 us on 192^3
// and 290 / 303 / 283 / 298 us on 256^3; grids of few workgroups take shorter runs (FP64 97x83x61, 970 workgroups:
// 19.1 us, 20.4 with 128) so that every XCD has its share.
inline unsigned xcd_run(long long blocks) { return (unsigned)std::min<long long>(std::max<long long>(blocks / 32, 1), kXcdRun); }

}  // namespace
