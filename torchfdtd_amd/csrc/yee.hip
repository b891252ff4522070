// Yee/CPML half steps, point traces and plane DFTs for gfx950, behind the C ABI of
// include/tfdtd.h.
//
// Arithmetic follows the reference update (torchfdtd/boundaries.py:363-438) term by
// term: every product and sum is rounded to the field precision in the same order,
// and the library is built with -ffp-contract=off and denormals kept, so a step is
// reproducible bit for bit against the NumPy/Torch path of the same precision.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../include/tfdtd.h"
#include "common.h"
#include "plane_march.h"

namespace {

using ::tfdtd_fail;

int fail(int code, const char* msg) { return tfdtd_fail(code, "%s", msg); }

template <typename... A>
int fail(int code, const char* fmt, A... args) { return tfdtd_fail(code, fmt, args...); }

int check_launch(const char* what) { return tfdtd_check_launch(what); }

template <typename real>
struct Slab {          // one CPML segment in its fixed slot 2*term+side
    int lo, hi;        // empty slot: lo == hi == 0
    real* psi;
    const real* b;
    const real* c;
    const real* inv_k;
};

template <typename real>
struct Source {
    int comp;
    int lo[3], hi[3];
    const real* values;
};

template <typename real>
struct HalfStep {
    int nx, ny, nz;
    const real* src;
    real* dst;
    const real* inverse;
    int inverse_stride;
    real courant;
    int periodic_mask, pec_mask;
    real pec_factor[3];
    Slab<real> slab[12];
    int nsrc;
    int box_lo[3], box_hi[3];   // union of the source boxes
    Source<real> srcs[TFDTD_MAX_SOURCES];
    long long source_samples;
    const long long* counter;
};

// One cell.  forward=false: E update from backward differences of H;
// forward=true: H update from forward differences of E.  The cell and its three neighbours
// (x, y, z, one row back or ahead) are read whole; the terms then follow CURL_TERMS order.
template <typename real, bool forward>
__device__ __forceinline__ void half_step_cell(const HalfStep<real>& a, const long long i) {
    const int nyz = a.ny * a.nz;
    const int x = (int)(i / nyz);
    const int r = (int)(i - (long long)x * nyz);
    const int y = r / a.nz;
    const int z = r - y * a.nz;
    const int coord[3] = {x, y, z};
    const int dims[3] = {a.nx, a.ny, a.nz};
    const long long stride[3] = {(long long)nyz, (long long)a.nz, 1};
    const Cell<real> c = cell_at(a.src, i);
    Cell<real> nb[3];
    bool inside[3];
#pragma unroll
    for (int axis = 0; axis < 3; ++axis) {
        const int n = dims[axis], k = coord[axis];
        const long long s = stride[axis];
        inside[axis] = n > 1 && (forward ? (k < n - 1) : (k > 0));
        nb[axis] = Cell<real>{{real(0), real(0), real(0)}};
        if (inside[axis]) nb[axis] = cell_at(a.src, forward ? i + s : i - s);
        else if (n > 1 && ((a.periodic_mask >> axis) & 1)) {
            const long long span = (long long)(n - 1) * s;
            nb[axis] = cell_at(a.src, forward ? i - span : i + span);
        }
    }
    // CPML memory.  The two slabs of a term never overlap (tfdtd_assign_slot), so a cell meets at most
    // one slab per term.  Every memory value and coefficient the cell needs is read here and the new
    // memory is stored after the last load: a load placed after a store would wait for it (the
    // compiler cannot tell the arrays apart), one round trip per term.
    bool hit[6];
    real* at[6];
    real old_psi[6], cb[6], cc[6], cik[6], memory[6];
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int axis = term_axis(t);
        hit[t] = false;
        at[t] = nullptr;
        old_psi[t] = cb[t] = cc[t] = cik[t] = memory[t] = real(0);
        if (dims[axis] == 1 || !inside[axis]) continue;
        const int k = coord[axis];
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const Slab<real>& g = a.slab[2 * t + side];
            if (k >= g.lo && k < g.hi) {
                const int q = k - g.lo;
                const int w = g.hi - g.lo;
                long long p;
                if (axis == 0) p = ((long long)q * a.ny + y) * a.nz + z;
                else if (axis == 1) p = ((long long)x * w + q) * a.nz + z;
                else p = ((long long)x * a.ny + y) * w + q;
                hit[t] = true;
                at[t] = g.psi + p;
                old_psi[t] = *global(at[t]);
                cb[t] = global(g.b)[q];
                cc[t] = global(g.c)[q];
                cik[t] = global(g.inv_k)[q];
            }
        }
    }
    real curl[3] = {real(0), real(0), real(0)};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int axis = term_axis(t), ic = term_in(t), oc = term_out(t);
        const int n = dims[axis];
        if (n == 1) continue;
        real d = real(0);
        if (inside[axis]) {
            d = forward ? (nb[axis].v[ic] - c.v[ic]) : (c.v[ic] - nb[axis].v[ic]);
            if (hit[t]) {
                memory[t] = old_psi[t] * cb[t] + cc[t] * d;
                d = d * cik[t] + memory[t];
            }
        } else if ((a.periodic_mask >> axis) & 1) {
            d = forward ? (nb[axis].v[ic] - c.v[ic]) : (c.v[ic] - nb[axis].v[ic]);
        } else if (forward && ((a.pec_mask >> axis) & 1)) {
            d = -a.pec_factor[axis] * c.v[ic];
        }
        curl[oc] = term_sign(t) > 0 ? curl[oc] + d : curl[oc] - d;
    }
    const Cell<real> old = cell_at(a.dst, i);
    Cell<real> inv;
    if (a.inverse_stride == 3) inv = cell_at(a.inverse, i);
    else {
        const real v = global(a.inverse)[a.inverse_stride == 1 ? i : 0];
        inv = Cell<real>{{v, v, v}};
    }
    real out[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const real coefficient = a.courant * inv.v[m];
        out[m] = forward ? old.v[m] - coefficient * curl[m] : old.v[m] + coefficient * curl[m];
    }
    if (a.nsrc > 0 && x >= a.box_lo[0] && x < a.box_hi[0] && y >= a.box_lo[1] && y < a.box_hi[1] &&
        z >= a.box_lo[2] && z < a.box_hi[2]) {
        const long long n = *global(a.counter);
        for (int k = 0; k < a.nsrc && n < a.source_samples; ++k) {
            const Source<real>& box = a.srcs[k];
            if (x >= box.lo[0] && x < box.hi[0] && y >= box.lo[1] && y < box.hi[1] && z >= box.lo[2] &&
                z < box.hi[2]) {
                const real v = global(box.values)[n];
                if (box.comp == 0) out[0] = out[0] + v;
                else if (box.comp == 1) out[1] = out[1] + v;
                else out[2] = out[2] + v;
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 6; ++t)
        if (hit[t]) *global(at[t]) = memory[t];
    const auto cell = global(a.dst + 3 * i);
    cell[0] = out[0];
    cell[1] = out[1];
    cell[2] = out[2];
}

template <typename real, bool forward>
__global__ __launch_bounds__(256) void yee_half_step_kernel(const HalfStep<real> a) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)a.nx * a.ny * a.nz) return;
    half_step_cell<real, forward>(a, i);
}

// ---------------------------------------------------------------- half step marched over x planes
//
// A wavefront takes 64 consecutive cells of the flattened (y, z) plane and marches them over `span` x
// planes.  What depends on y and z alone -- the coordinates, the neighbours' offsets, the slab rows and
// their coefficients -- is computed once per march, x is uniform (its slab, its coefficients and the plane
// addresses are scalar), and every field access is a uniform base plus a 32-bit lane offset, so a cell
// costs little more than its own arithmetic.  One thread per cell of the whole grid (half_step_cell) was
// bound by its 64-bit divisions, per-term slab tests and dependent descriptor loads: a step of both
// families plus its trace took 26.5 us on 160x120x40 cells, 49.1 us on 200x160x60, 121 us on 192^3, 317 us
// on 256^3 (FP32), 30.4 us on 97x83x61 (FP64); the march takes 16.7, 32.0, 95.6, 283 and 19.1 us.  A cell of a
// wavefront without slab rows executes about 45 vector instructions (with the lanes' 64-bit address sums and
// the slabs' arithmetic left to every wavefront: 110).  What bounds it now is the traffic: past the 256 MB cache
// 5.3 TB/s where a float4 copy reaches 6.15, inside it 6.4 of 8.4.
constexpr int kPlaneTraces = TFDTD_FOLDED_TRACES;

struct PlaneTrace {         // a point trace: its cell and value, and its column among the run's traces
    int x, cell, component, magnetic;
};

template <typename real>
struct PlaneStep {
    int nx, ny, nz, nyz;
    int span, columns;      // planes per march, 64-cell columns of a plane
    Divider by_nz, by_columns;
    int xcd, chunks;        // workgroups an XCD takes in a row, marches along x
    const real* src;
    real* dst;
    const real* inverse;
    real* psi;
    const real* coef;
    PlaneAxis<real> axis[3];
    int box_lo[3], box_hi[3];
    int nsrc;
    int periodic_mask, pec_mask;
    real courant;
    real pec_factor[3];
    Source<real> srcs[TFDTD_MAX_SOURCES];
    long long source_samples;
    const long long* counter;
    // The step's observation folded in: E copies the counter to `shadow`, H (which then reads the copy) steps the
    // counter on and records the traces of its cells.
    long long* counter_to;
    int counter_add;
    int ntraces, trace_lo, trace_hi;    // traces, and the x planes [lo, hi) they lie in
    PlaneTrace trace[kPlaneTraces];
    real* traces;
    long long trace_steps;
};

// The step counter carried on while other workgroups of the launch still read `from`.
__device__ __forceinline__ void carry_counter(const long long* from, long long* to, int add) {
    if (to && blockIdx.x == 0 && threadIdx.x == 0) *global(to) = *global(from) + add;
}

// The adjoint's record folded into the E step: the curl that the update of a box cell adds, in slot
// counter % modulus.
template <typename real>
struct CurlBox {
    int lo[3], hi[3];
    long long modulus;
    real* record;
};

struct NoBox {};

template <typename real, bool forward, int INV, bool FLAT, typename Box>
__device__ __forceinline__ void march_half_step(const PlaneStep<real>& a, const unsigned item, const Box& box) {
    constexpr bool recorded = !std::is_same<Box, NoBox>::value;
    constexpr unsigned W = sizeof(real);
    const int nx = a.nx, ny = a.ny, nz = FLAT ? 1 : a.nz, nyz = a.nyz;
    // Spare lanes of the last column and spare wavefronts of the last workgroup repeat a cell and store nothing.
    const unsigned xchunk = min(divide(item, a.by_columns), (unsigned)a.chunks - 1u);
    const unsigned cell = (item - xchunk * a.columns) * 64u + (threadIdx.x & 63u);
    const bool owned = cell < (unsigned)nyz;
    const unsigned r = min(cell, (unsigned)nyz - 1u);
    const int xa = (int)xchunk * a.span, xb = min(nx, xa + a.span);
    const int y = FLAT ? (int)r : (int)divide(r, a.by_nz), z = FLAT ? 0 : (int)(r - (unsigned)y * nz);
    unsigned off = r * (3 * W), line = r * W;
    const bool iny = forward ? y < ny - 1 : y > 0, inz = !FLAT && (forward ? z < nz - 1 : z > 0);
    const bool wrapx = a.periodic_mask & 1, wrapy = a.periodic_mask & 2, wrapz = !FLAT && (a.periodic_mask & 4);
    const unsigned rowb = (unsigned)nz * (3 * W), lasty = (unsigned)(ny - 1) * rowb, lastz = (unsigned)(nz - 1) * (3 * W);
    // The neighbour across y or z: the wrapped cell of a periodic axis, else the cell itself at its end.
    const unsigned endy = wrapy ? (forward ? 0u - lasty : lasty) : 0u, endz = wrapz ? (forward ? 0u - lastz : lastz) : 0u;
    unsigned offy = off + (iny ? (forward ? rowb : 0u - rowb) : endy);
    unsigned offz = off + (inz ? (forward ? 3 * W : 0u - 3 * W) : endz);
    const long long plane = 3LL * nyz;
    const real* src = a.src + xa * plane;
    real* dst = a.dst + xa * plane;
    real one = real(0);
    if (INV == 0) one = global(a.inverse)[0];
    // Backward differences carry the plane just left as x - 1, forward ones the plane fetched as x + 1.
    Cell<real> here = cell_at_byte(src, off);
    Cell<real> side = cell_at_byte(forward ? src : xa > 0 ? src - plane : wrapx ? a.src + (nx - 1) * plane : src, off);
    const AxisRow<real> ry = axis_row(a.axis[1], y, iny);
    PlaneHit<real> hy{ry.on, {0u, 0u}, 0u, real(0), real(0), real(0)};
    if (ry.on) {
        const unsigned e = ((unsigned)ry.q * nz + z) * W, wide = (unsigned)ry.w * W, k = ry.coef + (unsigned)ry.q * W;
        hy.stride = wide * nz;
        hy.at[0] = ry.psi[0] + e + xa * hy.stride;
        hy.at[1] = ry.psi[1] + e + xa * hy.stride;
        hy.b = at_byte(a.coef, k);
        hy.c = at_byte(a.coef, k + wide);
        hy.ik = at_byte(a.coef, k + 2 * wide);
    }
    PlaneHit<real> hz{false, {0u, 0u}, 0u, real(0), real(0), real(0)};
    if (!FLAT) {
        const AxisRow<real> rz = axis_row(a.axis[2], z, inz);
        hz.on = rz.on;
        if (rz.on) {
            const unsigned wide = (unsigned)rz.w * W, e = y * wide + (unsigned)rz.q * W, k = rz.coef + (unsigned)rz.q * W;
            hz.stride = wide * ny;
            hz.at[0] = rz.psi[0] + e + xa * hz.stride;
            hz.at[1] = rz.psi[1] + e + xa * hz.stride;
            hz.b = at_byte(a.coef, k);
            hz.c = at_byte(a.coef, k + wide);
            hz.ik = at_byte(a.coef, k + 2 * wide);
        }
    }
    const bool source = owned && a.nsrc > 0 && y >= a.box_lo[1] && y < a.box_hi[1] && z >= a.box_lo[2] && z < a.box_hi[2];
    const bool sources = __builtin_amdgcn_ballot_w64(source) != 0;
    real courant = a.courant;
    asm volatile("" : "+s"(courant));   // read once, before the loop
    // A wavefront without slab rows of an axis skips that axis's memory.
    const bool anyy = __builtin_amdgcn_ballot_w64(hy.on) != 0, anyz = !FLAT && __builtin_amdgcn_ballot_w64(hz.on) != 0;
    real* const psi = a.psi;
    bool boxed = false;
    real* record = nullptr;     // the box's plane of this x, and the lane's byte offset in it
    unsigned record_at = 0u;
    long long record_plane = 0;
    if constexpr (recorded) {
        const int by = box.hi[1] - box.lo[1], bz = box.hi[2] - box.lo[2];
        boxed = owned & (y >= box.lo[1]) & (y < box.hi[1]) & (z >= box.lo[2]) & (z < box.hi[2]);
        record_at = (unsigned)((y - box.lo[1]) * bz + z - box.lo[2]) * (3 * W);
        record_plane = 3LL * by * bz;
        record = box.record + (slot_of(*global(a.counter), box.modulus) * (box.hi[0] - box.lo[0]) + xa - box.lo[0]) * record_plane;
    }
    for (int x = xa; x < xb; ++x) {
        // The lane offsets stay 32-bit values of the loop: widened once before it, every access would add them
        // to its base in 64-bit vector arithmetic.
        asm volatile("" : "+v"(off), "+v"(offy), "+v"(offz), "+v"(line));
        const bool inx = forward ? x < nx - 1 : x > 0;
        if (forward) side = cell_at_byte(inx ? src + plane : wrapx ? a.src : src, off);
        const Cell<real> old = cell_at_byte(dst, off);
        Cell<real> inv;
        if (INV == 3) inv = cell_at_byte(a.inverse + x * plane, off);
        else {
            const real v = INV == 1 ? at_byte(a.inverse + (long long)x * nyz, line) : one;
            inv = Cell<real>{{v, v, v}};
        }
        const Cell<real> nby = cell_at_byte(src, offy);
        Cell<real> nbz{{real(0), real(0), real(0)}};
        if (!FLAT) nbz = cell_at_byte(src, offz);
        Cell<real> ahead = here;      // backward: the next plane, read with this one's neighbours
        if (!forward && x + 1 < xb) ahead = cell_at_byte(src + plane, off);
        // Every CPML memory value is read before the first store (a load behind a store would wait for it).
        real mx[2], my[2], mz[2];
        const AxisRow<real> rx = axis_row(a.axis[0], x, inx);
        real bx = real(0), cx = real(0), ikx = real(0);
        real* psix[2] = {psi, psi};
        if (rx.on) {
            const unsigned wide = (unsigned)rx.w * W, k = rx.coef + (unsigned)rx.q * W, e = (unsigned)rx.q * (unsigned)nyz * W;
            bx = at_byte(a.coef, k);
            cx = at_byte(a.coef, k + wide);
            ikx = at_byte(a.coef, k + 2 * wide);
            for (int t = 0; t < 2; ++t) {
                psix[t] = reinterpret_cast<real*>(reinterpret_cast<char*>(psi) + rx.psi[t] + e);
                mx[t] = at_byte(psix[t], line);
            }
        }
        if (hy.on)
            for (int t = 0; t < 2; ++t) my[t] = at_byte(psi, hy.at[t]);
        if (hz.on)
            for (int t = 0; t < 2; ++t) mz[t] = at_byte(psi, hz.at[t]);
        real curl[3] = {real(0), real(0), real(0)};
        // The two terms of one axis: difference, CPML row (`any`: the wavefront has one), sum into the curl in
        // term order.
        auto axis_terms = [&](auto axis_tag, bool in, bool wrap, const Cell<real>& nb, bool any, bool hit, real b, real c, real ik, real* m) {
            constexpr int axis = decltype(axis_tag)::value;
            const bool pecs = forward && ((a.pec_mask >> axis) & 1);
            const real pec = pecs ? -a.pec_factor[axis] : real(0);
            real d[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int ic = term_in(2 * axis + k);
                d[k] = forward ? nb.v[ic] - here.v[ic] : here.v[ic] - nb.v[ic];
            }
            if (any) {
                asm volatile("");       // a branch: the rows' arithmetic is not run for every wavefront
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    m[k] = m[k] * b + c * d[k];
                    const real stretched = d[k] * ik + m[k];
                    d[k] = hit ? stretched : d[k];
                }
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int t = 2 * axis + k, ic = term_in(t), oc = term_out(t);
                if (!in && !wrap) d[k] = pecs ? pec * here.v[ic] : real(0);
                curl[oc] = term_sign(t) > 0 ? curl[oc] + d[k] : curl[oc] - d[k];
            }
        };
        axis_terms(std::integral_constant<int, 0>{}, inx, wrapx, side, rx.on, rx.on, bx, cx, ikx, mx);
        axis_terms(std::integral_constant<int, 1>{}, iny, wrapy, nby, anyy, hy.on, hy.b, hy.c, hy.ik, my);
        if (!FLAT) axis_terms(std::integral_constant<int, 2>{}, inz, wrapz, nbz, anyz, hz.on, hz.b, hz.c, hz.ik, mz);
        real out[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const real coefficient = courant * inv.v[m];
            out[m] = forward ? old.v[m] - coefficient * curl[m] : old.v[m] + coefficient * curl[m];
        }
        if (sources && x >= a.box_lo[0] && x < a.box_hi[0]) {
            const long long n = *global(a.counter);
            for (int k = 0; k < a.nsrc && n < a.source_samples; ++k) {
                const Source<real>& box = a.srcs[k];
                if (x < box.lo[0] || x >= box.hi[0]) continue;
                const bool in = owned & (y >= box.lo[1]) & (y < box.hi[1]) & (z >= box.lo[2]) & (z < box.hi[2]);
                const real v = global(box.values)[n];
#pragma unroll
                for (int m = 0; m < 3; ++m)
                    if (box.comp == m && in) out[m] = out[m] + v;
            }
        }
        if constexpr (recorded) {
            if (boxed && x >= box.lo[0] && x < box.hi[0]) {
                const auto to = global(reinterpret_cast<real*>(reinterpret_cast<char*>(record) + record_at));
                to[0] = curl[0];
                to[1] = curl[1];
                to[2] = curl[2];
            }
            record += record_plane;
        }
        if (owned) {
            if (rx.on)
                for (int t = 0; t < 2; ++t) put_byte(psix[t], line, mx[t]);
            if (hy.on)
                for (int t = 0; t < 2; ++t) put_byte(psi, hy.at[t], my[t]);
            if (hz.on)
                for (int t = 0; t < 2; ++t) put_byte(psi, hz.at[t], mz[t]);
            const auto to = global(reinterpret_cast<real*>(reinterpret_cast<char*>(dst) + off));
            to[0] = out[0];
            to[1] = out[1];
            to[2] = out[2];
        }
        if (forward && x >= a.trace_lo && x < a.trace_hi)
            for (int k = 0; k < a.ntraces; ++k) {
                const PlaneTrace& t = a.trace[k];
                if (x != t.x || cell != (unsigned)t.cell) continue;
                const long long n = *global(a.counter);
                if (n < a.trace_steps) {
                    const real e = t.component == 0 ? here.v[0] : t.component == 1 ? here.v[1] : here.v[2];
                    const real h = t.component == 0 ? out[0] : t.component == 1 ? out[1] : out[2];
                    global(a.traces)[n * a.ntraces + k] = t.magnetic ? h : e;
                }
            }
        if (!forward) { side = here; here = ahead; }
        else here = side;
        if (anyy)
            for (int t = 0; t < 2; ++t) hy.at[t] += hy.stride;
        if (anyz)
            for (int t = 0; t < 2; ++t) hz.at[t] += hz.stride;
        src += plane;
        dst += plane;
    }
}

template <typename real, bool forward, int INV, bool FLAT>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 4 : 8) void plane_half_step_kernel(const PlaneStep<real> a) {
    march_half_step<real, forward, INV, FLAT>(a, wave_item(xcd_block(blockIdx.x, gridDim.x, a.xcd)), NoBox{});
    carry_counter(a.counter, a.counter_to, a.counter_add);
}

// The E step with the adjoint's record.  A launch of its own for the record read H and the CPML memory again and
// took 4.7-4.9 us on a 50x50x6 box or a 71x66x37 grid, and its gap.
template <typename real, int INV, bool FLAT>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 4 : 8) void recorded_half_step_kernel(const PlaneStep<real> a, const CurlBox<real> box) {
    march_half_step<real, false, INV, FLAT>(a, wave_item(xcd_block(blockIdx.x, gridDim.x, a.xcd)), box);
    carry_counter(a.counter, a.counter_to, a.counter_add);
}

// ---------------------------------------------------------------- several steps of a flat grid in one launch
//
// A grid of one z plane with few cells is bound by its launches: two of 3 us a step, whatever its cells.  A workgroup here
// loads a 32 x 32 patch of cells, a lane each, with their CPML memory and coefficients, takes `steps` steps with the fields exchanged through LDS, and stores the cells that are right:
// a step spoils one more row on each side, so the patch owns its inner (32 - 2 steps)^2 cells and its
// neighbours compute the rest again.  Fields and memory go from one buffer set to the other (neighbours still read
// the old state).  Every cell's arithmetic is the half steps' in their order, so results are equal bit for bit.
//
// us per step in a graph, half steps and patches: 160x120 6.2 -> 1.34 (FP64 6.3 -> 1.82), 256x256 5.6 -> 1.4, 400x400
// 6.8 -> 2.4, 800x800 11.4 -> 5.5 (FP64 17.5 -> 10.2), 1500x1500 27.6 -> 14, 3000x3000 85 -> 48 (FP64 257 -> 109).  A small
// grid is bound by one patch's chain (two barriers and two rounds through LDS a step, its load and store), a large
// one by the cells computed twice.
constexpr int kFlatTile = 32, kFlatSteps = 8;

// Steps per launch.  More steps share the load, the store and the launch, but own fewer cells of the patch (66% at
// 3, 56% at 4, 39% at 6, 25% at 8).  8 while all patches run at once, two to a CU (256x256: 1.41 us a step, 1.63 with
// 6); 6 up to four such rounds (400x400: 2.43, 2.69 with 8 and 2.74 with 4; 800x800: 5.5, 6.4 and 5.9); 4 beyond (1500x1500:
// 14.0, 14.8 with 6 and 19.0 with 2; 3000x3000: 48, 55 and 69).  The times are FP32's; FP64, whose patches run one to a CU
// (its registers), takes the same line: 257 to 512 of its patches run in two rounds of 8 steps.
inline long long flat_tiles(int nx, int ny, int steps) {
    const int own = kFlatTile - 2 * steps;
    return (long long)((nx + own - 1) / own) * ((ny + own - 1) / own);
}

inline int flat_depth(int nx, int ny) { return flat_tiles(nx, ny, kFlatSteps) <= 512 ? kFlatSteps : flat_tiles(nx, ny, 6) <= 2048 ? 6 : 4; }

// Whether the patches are the faster way.  A grid narrower than a patch leaves its lanes idle, which costs nothing while the
// patches run in four rounds; beyond, a quarter of their lanes has to own a cell.  us per step, half steps / patches: FP32
// 5x40000 7.9 / 5.9, 8x60000 8.5 / 8.7, 5x100000 10.6 / 13.5, 8x1000000 88 / 121, 12x1000000 149 / 122; FP64 8x60000
// 12.3 / 15.8, 5x1000000 123 / 237, 12x100000 32 / 26.
inline bool flat_pays(int nx, int ny) {
    const int depth = flat_depth(nx, ny);
    return depth > 4 || 4LL * nx * ny >= flat_tiles(nx, ny, depth) * (kFlatTile * kFlatTile);
}

// Whether `n` steps are worth two launches of patches: two steps of patches load and store the state as often as two half
// step pairs do, with a rim of each patch twice, and pay while the patches run at once (FP64: one to a CU).  us per step,
// half steps / patches.  Two steps: FP32 300x300 9.4 / 8.4, 500x500 10.7 / 10.9, 800x800 13.9 / 16.9, 3000x3000 88 / 127;
// FP64 300x300 9.9 / 10.0, 500x500 11.7 / 16.4, 1500x1500 51 / 60, 3000x3000 (past the cache) 259 / 247.  Three: FP32
// 500x500 9.6 / 8.5, 3000x3000 88 / 89; FP64 500x500 10.8 / 12.7, 800x800 18.9 / 19.1, 1500x1500 50 / 44.  Four: FP32
// 3000x3000 87 / 71, FP64 500x500 10.2 / 9.3.
inline bool flat_block_pays(int nx, int ny, int n, bool wide) {
    const long long tiles = flat_tiles(nx, ny, 2);
    if (n >= 4 || tiles <= 256) return true;
    if (n == 3) return !wide || tiles > 768;
    return wide && 48LL * nx * ny > 256LL << 20;
}

template <typename real>
struct FlatSet {            // one buffer set: fields and each family's CPML memory
    real *e, *h, *psi_e, *psi_h;
};

template <typename real>
struct FlatPass {
    PlaneStep<real> e, h;
    FlatSet<real> in, out;
    int steps, tiles_y;
    const long long* counter;
    long long* counter_to;  // takes the counter after the steps
};

// A cell's CPML rows of one family: the memory of the two terms of the x and the y axis and their coefficients.
template <typename real>
struct FlatRows {
    bool on[2];
    unsigned at[2][2];
    real b[2], c[2], ik[2], m[2][2];
};

template <typename real, bool forward>
__device__ __forceinline__ FlatRows<real> flat_rows(const PlaneStep<real>& a, const real* psi, int x, int y, bool live) {
    constexpr unsigned W = sizeof(real);
    FlatRows<real> out;
#pragma unroll
    for (int ax = 0; ax < 2; ++ax) {
        const int k = ax ? y : x, n = ax ? a.ny : a.nx;
        const AxisRow<real> r = axis_row(a.axis[ax], k, live && (forward ? k < n - 1 : k > 0));
        out.on[ax] = r.on;
        out.b[ax] = out.c[ax] = out.ik[ax] = out.m[ax][0] = out.m[ax][1] = real(0);
        out.at[ax][0] = out.at[ax][1] = 0u;
        if (!r.on) continue;
        const unsigned wide = (unsigned)r.w * W, coef = r.coef + (unsigned)r.q * W;
        const unsigned cell = ax ? (unsigned)x * wide + (unsigned)r.q * W : ((unsigned)r.q * a.ny + y) * W;
        out.b[ax] = at_byte(a.coef, coef);
        out.c[ax] = at_byte(a.coef, coef + wide);
        out.ik[ax] = at_byte(a.coef, coef + 2 * wide);
        for (int t = 0; t < 2; ++t) {
            out.at[ax][t] = r.psi[t] + cell;
            out.m[ax][t] = at_byte(psi, out.at[ax][t]);
        }
    }
    return out;
}

template <typename real, bool forward>
__device__ __forceinline__ void flat_half(const PlaneStep<real>& a, const real (*from)[kFlatTile * kFlatTile], const int next[2],
                                          const Cell<real>& here, Cell<real>& field, const Cell<real>& coefficient,
                                          FlatRows<real>& rows, const bool any[2], int x, int y, bool source, bool sources, long long n) {
    real curl[3] = {real(0), real(0), real(0)};
#pragma unroll
    for (int ax = 0; ax < 2; ++ax) {
        const int k = ax ? y : x, last = (ax ? a.ny : a.nx) - 1;
        const bool in = forward ? k < last : k > 0, wrap = (a.periodic_mask >> ax) & 1;
        const bool pecs = forward && ((a.pec_mask >> ax) & 1);
        const real pec = pecs ? -a.pec_factor[ax] : real(0);
        real d[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ic = term_in(2 * ax + j);
            const real nb = from[ic][next[ax]];
            d[j] = forward ? nb - here.v[ic] : here.v[ic] - nb;
        }
        if (any[ax]) {
            asm volatile("");       // a branch, as in march_half_step
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const real m = rows.m[ax][j] * rows.b[ax] + rows.c[ax] * d[j];
                const real stretched = d[j] * rows.ik[ax] + m;
                rows.m[ax][j] = m;
                d[j] = rows.on[ax] ? stretched : d[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = 2 * ax + j, ic = term_in(t), oc = term_out(t);
            if (!in && !wrap) d[j] = pecs ? pec * here.v[ic] : real(0);
            curl[oc] = term_sign(t) > 0 ? curl[oc] + d[j] : curl[oc] - d[j];
        }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const real change = coefficient.v[m] * curl[m];
        field.v[m] = forward ? field.v[m] - change : field.v[m] + change;
    }
    if (sources)
        for (int k = 0; k < a.nsrc && n < a.source_samples; ++k) {
            const Source<real>& box = a.srcs[k];
            const bool hit = source & (x >= box.lo[0]) & (x < box.hi[0]) & (y >= box.lo[1]) & (y < box.hi[1]);
            const real v = global(box.values)[n];
#pragma unroll
            for (int m = 0; m < 3; ++m)
                if (box.comp == m && hit) field.v[m] = field.v[m] + v;
        }
}

template <typename real, int INV>
__global__ __launch_bounds__(kFlatTile * kFlatTile, sizeof(real) == 8 ? 4 : 8) void flat_steps_kernel(const FlatPass<real> a) {
    constexpr int T = kFlatTile;
    __shared__ real se[3][T * T], sh[3][T * T];
    const int nx = a.e.nx, ny = a.e.ny, tid = threadIdx.x, ly = tid & (T - 1), lx = tid / T;
    const int own = T - 2 * a.steps, bx = blockIdx.x / a.tiles_y, by = blockIdx.x - bx * a.tiles_y;
    int x = bx * own - a.steps + lx, y = by * own - a.steps + ly;
    const bool owned = lx >= a.steps && lx < T - a.steps && ly >= a.steps && ly < T - a.steps && x < nx && y < ny;
    // A periodic axis continues with its other end's cells; elsewhere lanes beyond the grid hold zeros that no cell reads.
    if (a.e.periodic_mask & 1) { x %= nx; x += x < 0 ? nx : 0; }
    if (a.e.periodic_mask & 2) { y %= ny; y += y < 0 ? ny : 0; }
    const bool live = x >= 0 && x < nx && y >= 0 && y < ny;
    const long long cell = live ? (long long)x * ny + y : 0;
    Cell<real> e{{real(0), real(0), real(0)}}, h = e, ce = e, ch = e;
    if (live) {
        e = cell_at(a.in.e, cell);
        h = cell_at(a.in.h, cell);
        if (INV == 3) ce = cell_at(a.e.inverse, cell);
        else ce.v[0] = ce.v[1] = ce.v[2] = global(a.e.inverse)[cell];
    }
    const real one = global(a.h.inverse)[0];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        ce.v[m] = a.e.courant * ce.v[m];
        ch.v[m] = a.h.courant * one;
    }
    FlatRows<real> re = flat_rows<real, false>(a.e, a.in.psi_e, x, y, live);
    FlatRows<real> rh = flat_rows<real, true>(a.h, a.in.psi_h, x, y, live);
    const long long n0 = *global(a.counter);
    auto any = [](bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; };
    const bool rows_e[2] = {any(re.on[0]), any(re.on[1])}, rows_h[2] = {any(rh.on[0]), any(rh.on[1])};
    const bool srcs_e = any(live && a.e.nsrc > 0 && x >= a.e.box_lo[0] && x < a.e.box_hi[0] && y >= a.e.box_lo[1] && y < a.e.box_hi[1]);
    const bool srcs_h = any(live && a.h.nsrc > 0 && x >= a.h.box_lo[0] && x < a.h.box_hi[0] && y >= a.h.box_lo[1] && y < a.h.box_hi[1]);
    bool trace = false;
    for (int k = 0; k < a.h.ntraces; ++k) trace |= owned && a.h.trace[k].x == x && a.h.trace[k].cell == y;
    const bool traces = any(trace);
    // Neighbours of lanes at the patch's edge lie outside it: those lanes read themselves, and their cells are spoilt.
    const int low[2] = {lx > 0 ? tid - T : tid, ly > 0 ? tid - 1 : tid};
    const int high[2] = {lx < T - 1 ? tid + T : tid, ly < T - 1 ? tid + 1 : tid};
#pragma unroll
    for (int m = 0; m < 3; ++m) sh[m][tid] = h.v[m];
    __syncthreads();
    for (int s = 0; s < a.steps; ++s) {
        flat_half<real, false>(a.e, sh, low, h, e, ce, re, rows_e, x, y, live, srcs_e, n0 + s);
#pragma unroll
        for (int m = 0; m < 3; ++m) se[m][tid] = e.v[m];
        __syncthreads();
        flat_half<real, true>(a.h, se, high, e, h, ch, rh, rows_h, x, y, live, srcs_h, n0 + s);
#pragma unroll
        for (int m = 0; m < 3; ++m) sh[m][tid] = h.v[m];
        if (traces && trace && n0 + s < a.h.trace_steps)
            for (int k = 0; k < a.h.ntraces; ++k) {
                const PlaneTrace& t = a.h.trace[k];
                if (t.x != x || t.cell != y) continue;
                const real fe = t.component == 0 ? e.v[0] : t.component == 1 ? e.v[1] : e.v[2];
                const real fh = t.component == 0 ? h.v[0] : t.component == 1 ? h.v[1] : h.v[2];
                global(a.h.traces)[(n0 + s) * a.h.ntraces + k] = t.magnetic ? fh : fe;
            }
        __syncthreads();
    }
    if (owned) {
        const auto to_e = global(a.out.e + 3 * cell), to_h = global(a.out.h + 3 * cell);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            to_e[m] = e.v[m];
            to_h[m] = h.v[m];
        }
#pragma unroll
        for (int ax = 0; ax < 2; ++ax)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (re.on[ax]) put_byte(a.out.psi_e, re.at[ax][t], re.m[ax][t]);
                if (rh.on[ax]) put_byte(a.out.psi_h, rh.at[ax][t], rh.m[ax][t]);
            }
    }
    if (blockIdx.x == 0 && tid == 0) *global(a.counter_to) = n0 + a.steps;
}

// One grid of a batched half step: its plane march where `march` is set, else the general step.
template <typename real>
struct BatchStep {
    HalfStep<real> general;
    PlaneStep<real> plane;
    int march, inverse_stride;
};

// Cells per thread of the general batched half step: a workgroup covers 256 * kBatchSpan cells of one
// grid, so the search for its grid and the descriptor loads are shared by more cells.
constexpr int kBatchSpan = 2;

// Many grids in one launch: block b belongs to the last grid g with prefix[g] <= b; the grids'
// descriptors are a table in device memory, read with wave-uniform loads.
template <typename real, bool forward>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 4 : 8) void batch_half_step_kernel(const BatchStep<real>* __restrict__ table,
                                                              const int* __restrict__ prefix, int grids,
                                                              const long long* counter, long long* counter_to, int counter_add) {
    carry_counter(counter, counter_to, counter_add);
    const int b = (int)xcd_block(blockIdx.x, gridDim.x, kXcdRun);
    int lo = 0, hi = grids;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= b) lo = mid;
        else hi = mid;
    }
    const BatchStep<real>& t = table[lo];
    if (t.march) {
        const unsigned item = wave_item((unsigned)(b - prefix[lo]));
        const bool flat = t.plane.nz == 1;
        if (forward) {
            if (flat) march_half_step<real, true, 0, true>(t.plane, item, NoBox{});
            else march_half_step<real, true, 0, false>(t.plane, item, NoBox{});
        } else if (t.inverse_stride == 1) {
            if (flat) march_half_step<real, false, 1, true>(t.plane, item, NoBox{});
            else march_half_step<real, false, 1, false>(t.plane, item, NoBox{});
        } else {
            if (flat) march_half_step<real, false, 3, true>(t.plane, item, NoBox{});
            else march_half_step<real, false, 3, false>(t.plane, item, NoBox{});
        }
        return;
    }
    const HalfStep<real>& a = t.general;
    const long long cells = (long long)a.nx * a.ny * a.nz;
    const long long base = (long long)(b - prefix[lo]) * (256 * kBatchSpan) + threadIdx.x;
#pragma unroll
    for (int j = 0; j < kBatchSpan; ++j) {
        const long long i = base + 256 * j;
        if (i < cells) half_step_cell<real, forward>(a, i);
    }
}

template <typename real>
struct Observe {
    int count;
    const long long* table;
    real* traces;
    long long steps;
    long long* counter;
};

// Single block: record the traces of this step, then advance the counter.
template <typename real>
__global__ __launch_bounds__(256) void observe_kernel(const Observe<real> a) {
    const long long n = *a.counter;
    __syncthreads();
    if (n < a.steps) {
        for (int k = threadIdx.x; k < a.count; k += blockDim.x) {
            const auto field = global(reinterpret_cast<const real*>(a.table[2 * k]));
            a.traces[n * a.count + k] = field[a.table[2 * k + 1]];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) a.counter[0] = n + 1;
}

// Many traces: one trace per thread over the grid (the counter advances in a launch of its own).
template <typename real>
__global__ __launch_bounds__(256) void observe_wide_kernel(const Observe<real> a) {
    const long long n = *a.counter;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.steps || k >= a.count) return;
    const auto field = global(reinterpret_cast<const real*>(a.table[2 * k]));
    a.traces[n * a.count + k] = field[a.table[2 * k + 1]];
}

__global__ void advance_counter_kernel(long long* counter) { counter[0] = counter[0] + 1; }

template <typename real, typename spec>
struct Plane {
    long long points;
    int nf, nc, ne, corners, downsample;
    const real* E;
    const real* H;
    const long long* indices[6];
    const real* weights[6];
    const real* window_e;
    const real* window_h;
    const double* omega;
    const spec* half;   // interleaved re, im
    spec* value;        // interleaved re, im
    long long samples;
    const long long* counter;
    int block;          // > 1: samples of `block` steps are staged and accumulated together
    real* stage;        // [block][points * nc]
    const long long* flushed;
};

// exp(i omega (step+1)) for E and the same times exp(i pi f dt) for H, from the absolute step in
// FP64 (cuda_monitors.py:68-84): p[0..1] E (re, im), p[2..3] H.
template <typename real, typename spec>
__device__ __forceinline__ void phases(const Plane<real, spec>& a, long long step, int f, spec* p) {
    double si, co;
    sincos(global(a.omega)[f] * (double)(step + 1), &si, &co);
    const spec er = (spec)co, ei = (spec)si;
    const spec hr = global(a.half)[2 * f], hi = global(a.half)[2 * f + 1];
    p[0] = er;
    p[1] = ei;
    p[2] = er * hr - ei * hi;
    p[3] = er * hi + ei * hr;
}

// n % d of a step number, in 32 bits where it fits (a 64-bit remainder takes some 150 instructions).
__device__ __forceinline__ int step_mod(long long n, int d) {
    return (n >> 31) == 0 ? (int)((unsigned)n % (unsigned)d) : (int)(n % d);
}

// Interpolated sample of (point p, component c) at step n, times the window.
template <typename real, typename spec>
__device__ __forceinline__ real plane_sample(const Plane<real, spec>& a, long long p, int c, long long n) {
    const bool electric = c < a.ne;
    const auto field = global(electric ? a.E : a.H);
    const auto idx = global(a.indices[c]);
    const auto w = global(a.weights[c]);
    real v = real(0);
    if (a.corners == 8 || a.corners == 4) {
        // Every corner's index and weight first, then every corner's field value, then the sum in
        // corner order: the loads overlap instead of forming one round trip per corner.
        long long at[8];
        real wt[8], f[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < a.corners) {
                at[j] = idx[j * a.points + p];
                wt[j] = w[j * a.points + p];
            }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < a.corners) f[j] = field[at[j]];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < a.corners) v = v + f[j] * wt[j];
    } else {
        for (int j = 0; j < a.corners; ++j) v = v + field[idx[j * a.points + p]] * w[j * a.points + p];
    }
    return v * global(electric ? a.window_e : a.window_h)[n];
}

// Accumulate the staged samples of steps [lo, hi) (one block at most): the phases of those steps go
// to LDS, each thread sums its sample's products in FP64 and adds the sum to its accumulators.  The
// staged values are read once per kFlushGroup frequencies and the remainders of the step numbers formed
// once (a pair of 64-bit remainders per step and frequency made the flush of 29,376 samples x 8
// frequencies x 32 steps take 90 us, twice a step's half steps).
constexpr int kFlushGroup = 4;

template <typename real, typename spec>
__device__ __forceinline__ void flush_range(const Plane<real, spec>& a, long long i, int c, long long lo, long long hi) {
    extern __shared__ unsigned char lds_raw[];
    spec* phase = reinterpret_cast<spec*>(lds_raw);
    const int count = (int)(hi - lo);
    for (int e = threadIdx.x; e < count * a.nf; e += blockDim.x) phases(a, lo + e / a.nf, e % a.nf, phase + 4 * e);
    __syncthreads();
    const long long samples = a.points * a.nc;
    if (i >= samples) return;
    const int o = c < a.ne ? 0 : 2;
    const int slot = step_mod(lo, a.block), skip = step_mod(lo, a.downsample);
    for (int f = 0; f < a.nf; f += kFlushGroup) {
        double sr[kFlushGroup], si[kFlushGroup];
#pragma unroll
        for (int g = 0; g < kFlushGroup; ++g) sr[g] = si[g] = 0.;
        int s = slot, m = skip;
        for (int j = 0; j < count; ++j) {
            if (m == 0) {
                const spec v = (spec)global(a.stage)[s * samples + i];
#pragma unroll
                for (int g = 0; g < kFlushGroup; ++g) {
                    const spec* p = phase + 4 * (j * a.nf + min(f + g, a.nf - 1)) + o;
                    sr[g] += (double)(p[0] * v);
                    si[g] += (double)(p[1] * v);
                }
            }
            if (++s == a.block) s = 0;
            if (++m == a.downsample) m = 0;
        }
#pragma unroll
        for (int g = 0; g < kFlushGroup; ++g)
            if (f + g < a.nf) {
                const auto out = global(a.value + 2 * ((long long)(f + g) * samples + i));
                out[0] = out[0] + (spec)sr[g];
                out[1] = out[1] + (spec)si[g];
            }
    }
}

// The component of sample i, and its point.
template <typename real, typename spec>
__device__ __forceinline__ int sample_component(const Plane<real, spec>& a, long long i, long long* point) {
    if (a.points * a.nc < 0x7fffffffLL) {
        const unsigned p = (unsigned)i / (unsigned)a.nc;
        *point = p;
        return (int)((unsigned)i - p * (unsigned)a.nc);
    }
    *point = i / a.nc;
    return (int)(i - *point * a.nc);
}

// One thread per (point, component) sample.  Per-step accumulation (block <= 1): the block first
// evaluates the nf phases of this step into LDS.  Blocked accumulation: the sample is staged and
// the block's last step (or the window's last sample) accumulates the staged block.
template <typename real, typename spec>
__device__ __forceinline__ void dft_plane_block(const Plane<real, spec>& a, long long block) {
    extern __shared__ unsigned char lds_raw[];
    spec* phase = reinterpret_cast<spec*>(lds_raw);
    const long long n = *global(a.counter);
    if (n >= a.samples) return;
    const long long samples = a.points * a.nc;
    const long long i = block * blockDim.x + threadIdx.x;
    long long point;
    const int c = sample_component(a, i, &point);
    const bool taken = a.downsample == 1 || step_mod(n, a.downsample) == 0;
    if (a.block > 1) {
        const int slot = step_mod(n, a.block);
        if (taken && i < samples) global(a.stage)[slot * samples + i] = plane_sample(a, point, c, n);
        if (slot + 1 == a.block || n + 1 == a.samples) {
            const long long first = n - slot;
            const long long flushed = *global(a.flushed);
            flush_range(a, i, c, first > flushed ? first : flushed, n + 1);
        }
        return;
    }
    if (!taken) return;
    for (int f = threadIdx.x; f < a.nf; f += blockDim.x) phases(a, n, f, phase + 4 * f);
    __syncthreads();
    if (i >= samples) return;
    const spec sv = (spec)plane_sample(a, point, c, n);
    const int o = c < a.ne ? 0 : 2;
    for (int f = 0; f < a.nf; ++f) {
        const auto out = global(a.value + 2 * ((long long)f * samples + i));
        out[0] = out[0] + phase[4 * f + o] * sv;
        out[1] = out[1] + phase[4 * f + o + 1] * sv;
    }
}

// Accumulate the staged steps of the unfinished block: [max(flushed, first of block), counter).
template <typename real, typename spec>
__global__ __launch_bounds__(256) void dft_flush_kernel(const Plane<real, spec> a) {
    const long long n = *a.counter < a.samples ? *a.counter : a.samples;
    if (a.block <= 1 || n == a.samples) return;     // a finished window was accumulated by its last step
    const long long first = n - step_mod(n, a.block);
    const long long lo = first > *a.flushed ? first : *a.flushed;
    if (lo >= n) return;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long point;
    const int c = sample_component(a, i, &point);
    flush_range(a, i, c, lo, n);
}

__global__ void set_flushed_kernel(const long long* counter, long long samples, long long* flushed) {
    flushed[0] = counter[0] < samples ? counter[0] : samples;
}

// 8 waves per SIMD (at most 64 VGPRs): the sampling is latency-bound, and the 64-grid batch and the
// observed 512^3 cube ran 0.3-0.4% faster than at the 75 VGPRs the flush path asks for otherwise.
template <typename real, typename spec>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void dft_plane_kernel(const Plane<real, spec> a) {
    dft_plane_block(a, blockIdx.x);
}

// Many planes in one launch: blockIdx.y selects the plane of a device table.
template <typename real, typename spec>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void batch_dft_kernel(const Plane<real, spec>* __restrict__ table) {
    const Plane<real, spec>& a = table[blockIdx.y];
    if ((long long)blockIdx.x * blockDim.x >= a.points * a.nc) return;
    dft_plane_block(a, blockIdx.x);
}

// ---------------------------------------------------------------- host side

template <typename real>
int make_half_step(const tfdtd_half_step* d, HalfStep<real>* a) {
    if (d->nx < 1 || d->ny < 1 || d->nz < 1) return fail(TFDTD_EINVAL, "grid dimensions must be positive");
    if (!d->src || !d->dst || !d->inverse) return fail(TFDTD_EINVAL, "field and coefficient pointers are required");
    if (d->inverse_stride != 0 && d->inverse_stride != 1 && d->inverse_stride != 3)
        return fail(TFDTD_EINVAL, "inverse_stride must be 0, 1 or 3");
    if (d->nseg < 0 || d->nseg > TFDTD_MAX_SEGMENTS) return fail(TFDTD_EINVAL, "too many CPML segments");
    if (d->nsrc < 0 || d->nsrc > TFDTD_MAX_SOURCES) return fail(TFDTD_EINVAL, "too many sources");
    std::memset(a, 0, sizeof *a);
    a->nx = d->nx; a->ny = d->ny; a->nz = d->nz;
    a->src = static_cast<const real*>(d->src);
    a->dst = static_cast<real*>(d->dst);
    a->inverse = static_cast<const real*>(d->inverse);
    a->inverse_stride = d->inverse_stride;
    a->courant = (real)d->courant;
    a->periodic_mask = d->periodic_mask & 7;
    a->pec_mask = d->pec_upper_mask & 7;
    for (int k = 0; k < 3; ++k) a->pec_factor[k] = (real)d->pec_upper_factor[k];
    const int dims[3] = {d->nx, d->ny, d->nz};
    int slot_lo[12] = {0}, slot_hi[12] = {0};
    for (int k = 0; k < d->nseg; ++k) {
        const tfdtd_cpml_segment& s = d->seg[k];
        const int slot = tfdtd_assign_slot(s.axis, s.comp, s.lo, s.hi, dims, k, slot_lo, slot_hi);
        if (slot < 0) return TFDTD_EINVAL;
        if (!s.psi || !s.b || !s.c || !s.inv_k) return fail(TFDTD_EINVAL, "segment %d: null pointer", k);
        a->slab[slot] = Slab<real>{s.lo, s.hi, static_cast<real*>(s.psi), static_cast<const real*>(s.b),
                                   static_cast<const real*>(s.c), static_cast<const real*>(s.inv_k)};
    }
    a->nsrc = d->nsrc;
    for (int k = 0; k < 3; ++k) { a->box_lo[k] = dims[k]; a->box_hi[k] = 0; }
    for (int k = 0; k < d->nsrc; ++k) {
        const tfdtd_source& s = d->srcs[k];
        if (s.comp < 0 || s.comp > 2 || !s.values) return fail(TFDTD_EINVAL, "source %d: bad component or values", k);
        Source<real>& o = a->srcs[k];
        o.comp = s.comp;
        o.values = static_cast<const real*>(s.values);
        for (int ax = 0; ax < 3; ++ax) {
            if (s.lo[ax] < 0 || s.hi[ax] <= s.lo[ax] || s.hi[ax] > dims[ax]) return fail(TFDTD_EINVAL, "source %d: box outside the grid", k);
            o.lo[ax] = s.lo[ax]; o.hi[ax] = s.hi[ax];
            if (s.lo[ax] < a->box_lo[ax]) a->box_lo[ax] = s.lo[ax];
            if (s.hi[ax] > a->box_hi[ax]) a->box_hi[ax] = s.hi[ax];
        }
    }
    if (d->nsrc > 0 && (!d->counter || d->source_samples < 0))
        return fail(TFDTD_EINVAL, "sources need the device step counter and their sample count");
    a->source_samples = d->source_samples;
    a->counter = reinterpret_cast<const long long*>(d->counter);
    return TFDTD_OK;
}

template <typename real>
long long plane_blocks(const PlaneStep<real>& a) {
    return ((long long)a.columns * a.chunks + 3) / 4;
}

// The plane march of a half step: true when the grid's layout allows it.  The two terms of an axis must
// share their slab rows and one coefficient block b | c | inv_k on each side, the family's memory, its
// coefficients and a plane's fields must each span less than 4 GiB (32-bit byte offsets), x and y need
// two cells or more, and the coefficient is per cell or component for E, one value for H.  Everything
// else keeps the general step.
template <typename real>
bool make_plane_step(const HalfStep<real>& h, bool forward, PlaneStep<real>* out) {
    PlaneStep<real>& a = *out;
    std::memset(&a, 0, sizeof a);
    constexpr long long limit = 0xffffffffLL;
    const long long nyz = (long long)h.ny * h.nz;
    if (forward ? h.inverse_stride != 0 : h.inverse_stride == 0) return false;
    if (h.nx < 2 || h.ny < 2 || nyz * 3 * (long long)sizeof(real) > limit) return false;
    auto address = [](const void* p) { return reinterpret_cast<const char*>(p); };
    const char* psi = nullptr;
    const char* coef = nullptr;
    for (const Slab<real>& s : h.slab)
        if (s.hi > s.lo) {
            if (!psi || address(s.psi) < psi) psi = address(s.psi);
            if (!coef || address(s.b) < coef) coef = address(s.b);
        }
    const int dims[3] = {h.nx, h.ny, h.nz};
    for (int ax = 0; ax < 3; ++ax) {
        unsigned at[2][2] = {{0u, 0u}, {0u, 0u}}, block[2] = {0u, 0u};
        for (int side = 0; side < 2; ++side) {
            const Slab<real>& p = h.slab[4 * ax + side];
            const Slab<real>& q = h.slab[4 * ax + 2 + side];
            const int w = p.hi - p.lo;
            if (p.lo != q.lo || p.hi != q.hi) return false;
            if (w == 0) continue;
            if (p.b != q.b || p.c != q.c || p.inv_k != q.inv_k || p.c != p.b + w || p.inv_k != p.b + 2 * w) return false;
            const long long bytes = w * ((long long)h.nx * nyz / dims[ax]) * (long long)sizeof(real);
            const long long offset[3] = {address(p.psi) - psi, address(q.psi) - psi, address(p.b) - coef};
            if (offset[0] + bytes > limit || offset[1] + bytes > limit || offset[2] + 3LL * w * (long long)sizeof(real) > limit) return false;
            at[side][0] = (unsigned)offset[0];
            at[side][1] = (unsigned)offset[1];
            block[side] = (unsigned)offset[2];
            a.axis[ax].lo[side] = p.lo;
            a.axis[ax].hi[side] = p.hi;
        }
        for (int t = 0; t < 2; ++t) {
            a.axis[ax].psi[t] = at[0][t];
            a.axis[ax].high[t] = at[1][t] - at[0][t];
        }
        a.axis[ax].coef = block[0];
        a.axis[ax].coef_high = block[1] - block[0];
    }
    a.psi = reinterpret_cast<real*>(const_cast<char*>(psi));
    a.coef = reinterpret_cast<const real*>(coef);
    a.nx = h.nx; a.ny = h.ny; a.nz = h.nz; a.nyz = (int)nyz;
    a.columns = (int)((nyz + 63) / 64);
    a.span = (long long)a.columns * h.nx < kSpanItems ? 1 : 2;
    a.by_nz = make_divider((unsigned)h.nz);
    a.by_columns = make_divider((unsigned)a.columns);
    a.chunks = (h.nx + a.span - 1) / a.span;
    const long long items = (long long)a.columns * a.chunks;
    if (items > kLaunchItems) return false;
    a.xcd = (int)xcd_run(plane_blocks(a));
    a.src = h.src; a.dst = h.dst; a.inverse = h.inverse;
    a.courant = h.courant;
    a.periodic_mask = h.periodic_mask; a.pec_mask = h.pec_mask;
    for (int k = 0; k < 3; ++k) {
        a.pec_factor[k] = h.pec_factor[k];
        a.box_lo[k] = h.box_lo[k]; a.box_hi[k] = h.box_hi[k];
    }
    a.nsrc = h.nsrc;
    std::memcpy(a.srcs, h.srcs, sizeof a.srcs);
    a.source_samples = h.source_samples;
    a.counter = h.counter;
    return true;
}

// Lanes that a march leaves idle: those past the last cell of a plane's last column.
template <typename real>
long long idle_lanes(const PlaneStep<real>& a) {
    return (64LL * a.columns - a.nyz) * a.chunks;
}

// Whether a plane fills less than `sixteenths` of the lanes of its columns.
template <typename real>
bool thin_plane(const PlaneStep<real>& a, int sixteenths) {
    return 16LL * a.nyz < 64LL * a.columns * sixteenths;
}

// Whether the march is the faster step of a grid that it can take.  A plane of few cells leaves lanes idle, which
// costs nothing until they are more than the chip holds at once (256 CUs of 2048 lanes).  us a step, march / general:
//   FP32 8000x5x1 7.4 / 9.1, 80000x5x1 36 / 12.5, 1000000x5x1 381 / 69, 375000x16x1 148 / 81, 60000x5x5 34 / 33,
//   187500x32x1 78 / 81; past the 256 MB cache 400000x65x1 386 / 364, 400000x7x5 234 / 229, 200000x9x8 231 / 235;
//   FP64 80000x5x1 46 / 17, 93750x16x1 54 / 41, 62500x24x1 40 / 41, 60000x5x5 43 / 47.
// FP64 fields past the cache are bound by HBM, where the march saves the neighbours' address arithmetic for nothing
// unless there is memory along z: without it 1500x90x90 388 / 351, 400x180x170 394 / 365, 182^3 198 / 189, 171^3
// (240 MB) 151 / 159; with it 464 / 517, 436 / 455, 222 / 235.
constexpr long long kIdleLanes = 256 * 2048;

template <typename real>
bool march_pays(const PlaneStep<real>& a) {
    constexpr bool wide = sizeof(real) == 8;
    const bool past_cache = 6LL * (long long)sizeof(real) * a.nx * a.nyz > 256LL << 20;
    if (wide && past_cache && a.axis[2].hi[0] == a.axis[2].lo[0] && a.axis[2].hi[1] == a.axis[2].lo[1]) return false;
    return !thin_plane(a, wide ? 6 : past_cache ? 9 : 8) || idle_lanes(a) <= kIdleLanes;
}

// The same for a grid of a batch, whose workgroups look their grid up: a plane has to fill more of its lanes, and the
// idle lanes are those of all such grids.  us a step, march / general: FP32 400 grids of 2000x5x1 746 / 77 (30: 54 / 17),
// 272 of 300x7x7 95 / 87, 400 of 100x10x10 96 / 88, 178 of 400x56x1 79 / 83, 30 of 400x5x5 18 / 19; FP64 307 of
// 100x13x10 140 / 128, 208 of 400x48x1 160 / 165.
template <typename real>
constexpr int kBatchThin = sizeof(real) == 8 ? 11 : 13;

template <typename real>
void launch_plane_step(const PlaneStep<real>& a, bool forward, int inverse_stride, hipStream_t stream) {
    const dim3 grid((unsigned)plane_blocks(a)), block(256);
    const bool flat = a.nz == 1;
    if (forward) {
        if (flat) hipLaunchKernelGGL((plane_half_step_kernel<real, true, 0, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((plane_half_step_kernel<real, true, 0, false>), grid, block, 0, stream, a);
    } else if (inverse_stride == 1) {
        if (flat) hipLaunchKernelGGL((plane_half_step_kernel<real, false, 1, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((plane_half_step_kernel<real, false, 1, false>), grid, block, 0, stream, a);
    } else {
        if (flat) hipLaunchKernelGGL((plane_half_step_kernel<real, false, 3, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((plane_half_step_kernel<real, false, 3, false>), grid, block, 0, stream, a);
    }
}

template <typename real>
int launch_half_step(const tfdtd_half_step* d, hipStream_t stream) {
    HalfStep<real> a;
    int status = make_half_step(d, &a);
    if (status) return status;
    const bool forward = d->family == TFDTD_FAMILY_H;
    PlaneStep<real> p;
    if (make_plane_step(a, forward, &p) && march_pays(p)) {
        launch_plane_step(p, forward, d->inverse_stride, stream);
        return check_launch("yee_half_step");
    }
    const long long count = (long long)d->nx * d->ny * d->nz;
    const long long blocks = (count + 255) / 256;
    if (blocks > 0x7fffffffLL) return fail(TFDTD_EINVAL, "grid too large for one launch");
    if (d->family == TFDTD_FAMILY_E)
        hipLaunchKernelGGL((yee_half_step_kernel<real, false>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL((yee_half_step_kernel<real, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
    return check_launch("yee_half_step");
}

template <typename real>
int launch_observe(const tfdtd_observe* d, hipStream_t stream) {
    if (!d->counter) return fail(TFDTD_EINVAL, "observe needs the device step counter");
    if (d->count < 0 || (d->count > 0 && (!d->table || !d->traces)))
        return fail(TFDTD_EINVAL, "observe: trace table and traces are required");
    Observe<real> a{d->count, reinterpret_cast<const long long*>(d->table), static_cast<real*>(d->traces),
                    (long long)d->steps, reinterpret_cast<long long*>(d->counter)};
    constexpr int kOneBlock = 4096;
    if (d->count <= kOneBlock) {
        hipLaunchKernelGGL((observe_kernel<real>), dim3(1), dim3(256), 0, stream, a);
        return check_launch("observe");
    }
    hipLaunchKernelGGL((observe_wide_kernel<real>), dim3((unsigned)((d->count + 255) / 256)), dim3(256), 0, stream, a);
    const int status = check_launch("observe");
    if (status) return status;
    hipLaunchKernelGGL(advance_counter_kernel, dim3(1), dim3(1), 0, stream, a.counter);
    return check_launch("observe counter");
}

template <typename real, typename spec>
int make_plane(const tfdtd_plane* d, Plane<real, spec>* out);

// LDS of one plane launch: the phases of one step, or of every step of a block.
template <typename spec>
size_t plane_lds(const tfdtd_plane* d) {
    return 4 * sizeof(spec) * (size_t)d->frequencies * (size_t)(d->block > 1 ? d->block : 1);
}

template <typename real, typename spec>
int launch_plane(const tfdtd_plane* d, hipStream_t stream, const long long* counter) {
    Plane<real, spec> a;
    int status = make_plane(d, &a);
    if (status) return status;
    if (counter) a.counter = counter;
    const size_t lds = plane_lds<spec>(d);
    const long long blocks = (d->points * d->components + 255) / 256;
    hipLaunchKernelGGL((dft_plane_kernel<real, spec>), dim3((unsigned)blocks), dim3(256), lds, stream, a);
    return check_launch("dft_plane");
}

template <typename real, typename spec>
int launch_flush(const tfdtd_plane* d, hipStream_t stream) {
    Plane<real, spec> a;
    int status = make_plane(d, &a);
    if (status) return status;
    const long long blocks = (d->points * d->components + 255) / 256;
    hipLaunchKernelGGL((dft_flush_kernel<real, spec>), dim3((unsigned)blocks), dim3(256), plane_lds<spec>(d), stream, a);
    status = check_launch("dft_flush");
    if (status) return status;
    hipLaunchKernelGGL(set_flushed_kernel, dim3(1), dim3(1), 0, stream, a.counter, a.samples, const_cast<long long*>(a.flushed));
    return check_launch("dft_flush counter");
}

template <typename real, typename spec>
int make_plane(const tfdtd_plane* d, Plane<real, spec>* out) {
    Plane<real, spec>& a = *out;
    if (d->points < 1 || d->frequencies < 1 || d->components < 1 || d->components > 6 || d->electric < 0 ||
        d->electric > d->components || d->corners < 1 || d->corners > 8 || d->time_downsample < 1)
        return fail(TFDTD_EINVAL, "plane: bad sizes");
    if (!d->E || !d->H || !d->window_e || !d->window_h || !d->omega || !d->half || !d->value || !d->counter)
        return fail(TFDTD_EINVAL, "plane: null pointer");
    if (d->block < 0) return fail(TFDTD_EINVAL, "plane: negative block");
    if (plane_lds<spec>(d) > 64 * 1024)
        return fail(TFDTD_EINVAL, "plane: %d frequencies x block %d exceed one launch", d->frequencies, d->block);
    if (d->block > 1 && (!d->stage || !d->flushed)) return fail(TFDTD_EINVAL, "plane: a block needs stage and flushed buffers");
    std::memset(&a, 0, sizeof a);
    a.points = d->points; a.nf = d->frequencies; a.nc = d->components; a.ne = d->electric;
    a.corners = d->corners; a.downsample = d->time_downsample;
    a.E = static_cast<const real*>(d->E); a.H = static_cast<const real*>(d->H);
    for (int c = 0; c < d->components; ++c) {
        if (!d->indices[c] || !d->weights[c]) return fail(TFDTD_EINVAL, "plane: component %d map missing", c);
        a.indices[c] = reinterpret_cast<const long long*>(d->indices[c]);
        a.weights[c] = static_cast<const real*>(d->weights[c]);
    }
    a.window_e = static_cast<const real*>(d->window_e); a.window_h = static_cast<const real*>(d->window_h);
    a.omega = d->omega; a.half = static_cast<const spec*>(d->half); a.value = static_cast<spec*>(d->value);
    a.counter = reinterpret_cast<const long long*>(d->counter);
    if (d->samples < 0) return fail(TFDTD_EINVAL, "plane: negative window length");
    a.samples = d->samples;
    a.block = d->block > 1 ? d->block : 1;
    a.stage = static_cast<real*>(d->stage);
    a.flushed = reinterpret_cast<const long long*>(d->flushed);
    if ((d->points * d->components + 255) / 256 > 0x7fffffffLL) return fail(TFDTD_EINVAL, "plane: too many samples");
    return TFDTD_OK;
}

// The source boxes of a half step alone: field[cell][comp] += values[counter] in source order, over
// the union box of the sources (the step's own update is not applied).
template <typename real>
__global__ __launch_bounds__(256) void inject_kernel(const HalfStep<real> a) {
    const int bx = a.box_hi[0] - a.box_lo[0], by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
    const long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= (long long)bx * by * bz) return;
    const int z = a.box_lo[2] + (int)(j % bz), y = a.box_lo[1] + (int)((j / bz) % by), x = a.box_lo[0] + (int)(j / ((long long)by * bz));
    const long long n = *global(a.counter);
    if (n >= a.source_samples) return;
    const long long i = ((long long)x * a.ny + y) * a.nz + z;
    real out[3] = {a.dst[3 * i], a.dst[3 * i + 1], a.dst[3 * i + 2]};
    bool hit = false;
    for (int k = 0; k < a.nsrc; ++k) {
        const Source<real>& box = a.srcs[k];
        if (x >= box.lo[0] && x < box.hi[0] && y >= box.lo[1] && y < box.hi[1] && z >= box.lo[2] && z < box.hi[2]) {
            const real v = global(box.values)[n];
            out[box.comp] = out[box.comp] + v;
            hit = true;
        }
    }
    if (hit) {
        a.dst[3 * i] = out[0];
        a.dst[3 * i + 1] = out[1];
        a.dst[3 * i + 2] = out[2];
    }
}

template <typename real>
int launch_inject(const tfdtd_half_step* d, hipStream_t stream) {
    HalfStep<real> a;
    int status = make_half_step(d, &a);
    if (status) return status;
    if (a.nsrc == 0) return TFDTD_OK;
    const long long count = (long long)(a.box_hi[0] - a.box_lo[0]) * (a.box_hi[1] - a.box_lo[1]) * (a.box_hi[2] - a.box_lo[2]);
    hipLaunchKernelGGL(inject_kernel<real>, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, a);
    return check_launch("inject");
}

int half_step(const tfdtd_half_step* d, hipStream_t stream) {
    if (!d) return fail(TFDTD_EINVAL, "null half-step descriptor");
    if (d->family != TFDTD_FAMILY_E && d->family != TFDTD_FAMILY_H) return fail(TFDTD_EINVAL, "family must be E or H");
    if (d->dtype == TFDTD_F32) return launch_half_step<float>(d, stream);
    if (d->dtype == TFDTD_F64) return launch_half_step<double>(d, stream);
    return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
}

int planes(const tfdtd_plane* p, int count, hipStream_t stream, const long long* counter = nullptr) {
    if (count < 0 || (count > 0 && !p)) return fail(TFDTD_EINVAL, "bad plane table");
    for (int k = 0; k < count; ++k) {
        int status;
        const tfdtd_plane* d = p + k;
        if (d->dtype == TFDTD_F32 && d->spectral == 0) status = launch_plane<float, float>(d, stream, counter);
        else if (d->dtype == TFDTD_F32 && d->spectral == 1) status = launch_plane<float, double>(d, stream, counter);
        else if (d->dtype == TFDTD_F64 && d->spectral == 1) status = launch_plane<double, double>(d, stream, counter);
        else status = fail(TFDTD_EINVAL, "plane %d: unsupported dtype/spectral pair", k);
        if (status) return status;
    }
    return TFDTD_OK;
}

template <typename real>
int launch_traces(const tfdtd_observe* d, const long long* counter, hipStream_t stream) {
    if (d->count == 0) return TFDTD_OK;
    if (d->count < 0 || !d->table || !d->traces) return fail(TFDTD_EINVAL, "observe: trace table and traces are required");
    const Observe<real> a{d->count, reinterpret_cast<const long long*>(d->table), static_cast<real*>(d->traces), (long long)d->steps,
                          const_cast<long long*>(counter)};
    hipLaunchKernelGGL((observe_wide_kernel<real>), dim3((unsigned)((d->count + 255) / 256)), dim3(256), 0, stream, a);
    return check_launch("observe");
}

// The traces at step *counter, without advancing it.
int record_traces(const tfdtd_observe* d, const long long* counter, hipStream_t stream) {
    if (d->dtype == TFDTD_F32) return launch_traces<float>(d, counter, stream);
    if (d->dtype == TFDTD_F64) return launch_traces<double>(d, counter, stream);
    return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
}

int observe(const tfdtd_observe* d, hipStream_t stream) {
    if (!d) return fail(TFDTD_EINVAL, "null observe descriptor");
    if (d->dtype == TFDTD_F32) return launch_observe<float>(d, stream);
    if (d->dtype == TFDTD_F64) return launch_observe<double>(d, stream);
    return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
}

template <typename real>
int pack_half_steps(const tfdtd_half_step* steps, int count, void* host_table, size_t bytes, int32_t* prefix) {
    if (count < 1 || !steps || !prefix) return fail(TFDTD_EINVAL, "batch: at least one descriptor and a prefix array");
    if (!host_table || bytes < sizeof(BatchStep<real>) * (size_t)count) return fail(TFDTD_EINVAL, "batch: table buffer too small");
    BatchStep<real>* table = static_cast<BatchStep<real>*>(host_table);
    long long total = 0, idle = 0;
    for (int k = 0; k < count; ++k) {
        if (steps[k].family != steps[0].family || steps[k].dtype != steps[0].dtype)
            return fail(TFDTD_EINVAL, "batch: descriptor %d differs in family or dtype", k);
        BatchStep<real>& t = table[k];
        const int status = make_half_step(steps + k, &t.general);
        if (status) return status;
        t.march = make_plane_step(t.general, steps[k].family == TFDTD_FAMILY_H, &t.plane) ? 1 : 0;
        t.inverse_stride = t.general.inverse_stride;
        if (t.march && thin_plane(t.plane, kBatchThin<real>)) idle += idle_lanes(t.plane);
    }
    for (int k = 0; k < count; ++k) {
        BatchStep<real>& t = table[k];
        if (t.march && idle > kIdleLanes && thin_plane(t.plane, kBatchThin<real>)) t.march = 0;
        prefix[k] = (int32_t)total;
        total += t.march ? plane_blocks(t.plane)
                         : ((long long)steps[k].nx * steps[k].ny * steps[k].nz + 256 * kBatchSpan - 1) / (256 * kBatchSpan);
        if (total > 0x7fffffffLL) return fail(TFDTD_EINVAL, "batch: too many cells for one launch");
    }
    prefix[count] = (int32_t)total;
    return TFDTD_OK;
}

template <typename real, typename spec>
int pack_planes(const tfdtd_plane* planes, int count, void* host_table, size_t bytes, int32_t* max_blocks, int32_t* max_phases) {
    if (count < 1 || !planes || !max_blocks || !max_phases) return fail(TFDTD_EINVAL, "batch planes: bad arguments");
    if (!host_table || bytes < sizeof(Plane<real, spec>) * (size_t)count) return fail(TFDTD_EINVAL, "batch planes: table buffer too small");
    Plane<real, spec>* table = static_cast<Plane<real, spec>*>(host_table);
    *max_blocks = 0;
    *max_phases = 0;
    for (int k = 0; k < count; ++k) {
        const int status = make_plane(planes + k, table + k);
        if (status) return status;
        *max_blocks = std::max<int32_t>(*max_blocks, (int32_t)((planes[k].points * planes[k].components + 255) / 256));
        *max_phases = std::max(*max_phases, planes[k].frequencies * std::max(planes[k].block, 1));
    }
    return TFDTD_OK;
}

int batch_half_step(const void* device_table, const int32_t* device_prefix, int count, int total_blocks, int dtype, int family,
                    const long long* counter, long long* counter_to, int counter_add, void* stream) {
    if (!device_table || !device_prefix || count < 1 || total_blocks < 0) return fail(TFDTD_EINVAL, "batch: bad launch arguments");
    if (total_blocks == 0) return TFDTD_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int* prefix = reinterpret_cast<const int*>(device_prefix);
    const dim3 grid(total_blocks), block(256);
    if (dtype == TFDTD_F32) {
        const BatchStep<float>* t = static_cast<const BatchStep<float>*>(device_table);
        if (family == TFDTD_FAMILY_E)
            hipLaunchKernelGGL((batch_half_step_kernel<float, false>), grid, block, 0, s, t, prefix, count, counter, counter_to, counter_add);
        else
            hipLaunchKernelGGL((batch_half_step_kernel<float, true>), grid, block, 0, s, t, prefix, count, counter, counter_to, counter_add);
    } else if (dtype == TFDTD_F64) {
        const BatchStep<double>* t = static_cast<const BatchStep<double>*>(device_table);
        if (family == TFDTD_FAMILY_E)
            hipLaunchKernelGGL((batch_half_step_kernel<double, false>), grid, block, 0, s, t, prefix, count, counter, counter_to, counter_add);
        else
            hipLaunchKernelGGL((batch_half_step_kernel<double, true>), grid, block, 0, s, t, prefix, count, counter, counter_to, counter_add);
    } else {
        return fail(TFDTD_EINVAL, "batch: dtype must be float32 or float64");
    }
    return check_launch("batch_half_step");
}

// The record of an E step as part of it: true where it reads what the step reads (the step's own H, memory and
// counter, every slab applied).
template <typename real>
bool make_curl_box(const tfdtd_curl_record& d, const tfdtd_half_step& e, const tfdtd_observe& obs, const PlaneStep<real>& step, CurlBox<real>* box) {
    if (d.dtype != e.dtype || d.nx != e.nx || d.ny != e.ny || d.nz != e.nz || d.H != e.src || d.counter != obs.counter ||
        (d.periodic_mask & 7) != step.periodic_mask || !d.record || d.modulus < 1)
        return false;
    if (step.psi && d.e.psi_in != step.psi) return false;
    const int n[3] = {d.nx, d.ny, d.nz};
    for (int k = 0; k < 3; ++k) {
        if (d.box_lo[k] < 0 || d.box_hi[k] <= d.box_lo[k] || d.box_hi[k] > n[k]) return false;
        box->lo[k] = d.box_lo[k];
        box->hi[k] = d.box_hi[k];
    }
    box->modulus = d.modulus;
    box->record = static_cast<real*>(d.record);
    return true;
}

template <typename real>
void launch_recorded_step(const PlaneStep<real>& a, const CurlBox<real>& box, int inverse_stride, hipStream_t stream) {
    const dim3 grid((unsigned)plane_blocks(a)), block(256);
    const bool flat = a.nz == 1;
    if (inverse_stride == 1) {
        if (flat) hipLaunchKernelGGL((recorded_half_step_kernel<real, 1, true>), grid, block, 0, stream, a, box);
        else hipLaunchKernelGGL((recorded_half_step_kernel<real, 1, false>), grid, block, 0, stream, a, box);
    } else {
        if (flat) hipLaunchKernelGGL((recorded_half_step_kernel<real, 3, true>), grid, block, 0, stream, a, box);
        else hipLaunchKernelGGL((recorded_half_step_kernel<real, 3, false>), grid, block, 0, stream, a, box);
    }
}

// The traces of a step at the cells its H launch updates, where they are few enough.
template <typename real>
int fold_traces(const tfdtd_observe* obs, const tfdtd_trace_cell* cells, PlaneStep<real>* h, bool* folded) {
    *folded = cells && obs->count > 0 && obs->count <= kPlaneTraces;
    if (!*folded) return TFDTD_OK;
    h->ntraces = obs->count;
    h->traces = static_cast<real*>(obs->traces);
    h->trace_steps = (long long)obs->steps;
    h->trace_lo = h->nx;
    const long long values = 3LL * h->nx * h->nyz;
    for (int k = 0; k < obs->count; ++k) {
        if (cells[k].element < 0 || cells[k].element >= values) return fail(TFDTD_EINVAL, "trace %d lies outside the grid", k);
        const long long cell = cells[k].element / 3;
        h->trace[k] = PlaneTrace{(int)(cell / h->nyz), (int)(cell % h->nyz), (int)(cells[k].element % 3), cells[k].magnetic};
        h->trace_lo = std::min(h->trace_lo, h->trace[k].x);
        h->trace_hi = std::max(h->trace_hi, h->trace[k].x + 1);
    }
    return TFDTD_OK;
}

// One step of a grid whose half steps both march: E (copying the counter to `shadow`), H (stepping the counter on and
// recording up to TFDTD_FOLDED_TRACES traces), planes and further traces, which read the copy.  A launch of its own
// for the traces and the counter cost 0.9 us a step on 160x120x40 cells (930 -> 884 us for 50 steps), 1.1 us
// on 160x120x1.
template <typename real>
int observed_step(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_plane* p, int plane_count,
                  const tfdtd_observe* obs, const tfdtd_trace_cell* cells, long long* shadow, const tfdtd_curl_record* record,
                  hipStream_t stream, bool* done) {
    *done = false;
    HalfStep<real> e, h;
    int status = make_half_step(e_step, &e);
    if (!status) status = make_half_step(h_step, &h);
    if (status) return status;
    PlaneStep<real> pe, ph;
    if (!make_plane_step(e, false, &pe) || !make_plane_step(h, true, &ph) || !march_pays(pe) || !march_pays(ph)) return TFDTD_OK;
    CurlBox<real> box;
    if (record && !make_curl_box(*record, *e_step, *obs, pe, &box)) return TFDTD_OK;
    *done = true;
    long long* const counter = reinterpret_cast<long long*>(obs->counter);
    pe.counter = counter;
    pe.counter_to = shadow;
    ph.counter = shadow;
    ph.counter_to = counter;
    ph.counter_add = 1;
    bool folded = false;
    status = fold_traces(obs, cells, &ph, &folded);
    if (status) return status;
    if (record) launch_recorded_step(pe, box, e_step->inverse_stride, stream);
    else launch_plane_step(pe, false, e_step->inverse_stride, stream);
    status = check_launch("yee_half_step");
    if (status) return status;
    launch_plane_step(ph, true, h_step->inverse_stride, stream);
    status = check_launch("yee_half_step");
    if (!status) status = planes(p, plane_count, stream, shadow);
    if (!status && obs->count > 0 && !folded) status = record_traces(obs, shadow, stream);
    return status;
}

// Passes of a flat run of `n` steps: an even number, so the state returns to its buffers, of nearly equal steps.
template <typename real>
int flat_steps(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_observe* obs, const tfdtd_trace_cell* cells,
               const FlatSet<real>& second, long long* shadow, int n, hipStream_t stream) {
    HalfStep<real> e, h;
    int status = make_half_step(e_step, &e);
    if (!status) status = make_half_step(h_step, &h);
    if (status) return status;
    FlatPass<real> a;
    if (e.nz != 1 || e.nx != h.nx || e.ny != h.ny || e.nz != h.nz || e.src != h.dst || e.dst != h.src ||
        e.periodic_mask != h.periodic_mask || !make_plane_step(e, false, &a.e) || !make_plane_step(h, true, &a.h))
        return fail(TFDTD_EUNSUPPORTED, "flat_steps needs one grid of one z plane that the plane march takes");
    if (flat_tiles(e.nx, e.ny, flat_depth(e.nx, e.ny)) > kLaunchPatches)
        return fail(TFDTD_EUNSUPPORTED, "flat_steps: the grid is too large for one launch of patches");
    if (!flat_pays(e.nx, e.ny)) return fail(TFDTD_EUNSUPPORTED, "flat_steps: the grid is too narrow for its patches");
    bool folded = false;
    status = fold_traces(obs, cells, &a.h, &folded);
    if (status) return status;
    if (obs->count > 0 && !folded) return fail(TFDTD_EUNSUPPORTED, "flat_steps records at most %d traces", kPlaneTraces);
    if (n == 0) return TFDTD_OK;
    if (!flat_block_pays(e.nx, e.ny, n, sizeof(real) == 8)) {
        for (int k = 0; k < n && !status; ++k)
            status = tfdtd_step_observed(e_step, h_step, nullptr, 0, obs, cells, reinterpret_cast<int64_t*>(shadow), stream);
        return status;
    }
    long long* const counter = reinterpret_cast<long long*>(obs->counter);
    const FlatSet<real> own{a.e.dst, a.h.dst, a.e.psi, a.h.psi};
    const int depth = flat_depth(a.e.nx, a.e.ny), passes = (n + 2 * depth - 1) / (2 * depth) * 2;
    for (int k = 0; k < passes; ++k) {
        const bool back = k & 1;
        a.in = back ? second : own;
        a.out = back ? own : second;
        a.counter = back ? shadow : counter;
        a.counter_to = back ? counter : shadow;
        a.steps = n / passes + (k < n % passes);
        const int width = kFlatTile - 2 * a.steps;
        a.tiles_y = (a.e.ny + width - 1) / width;
        const dim3 grid((unsigned)flat_tiles(a.e.nx, a.e.ny, a.steps)), block(kFlatTile * kFlatTile);
        if (e_step->inverse_stride == 1) hipLaunchKernelGGL((flat_steps_kernel<real, 1>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((flat_steps_kernel<real, 3>), grid, block, 0, stream, a);
        status = check_launch("flat_steps");
        if (status) return status;
    }
    return TFDTD_OK;
}

}  // namespace

extern "C" {

size_t tfdtd_batch_table_bytes(int32_t count, int32_t dtype) {
    if (count < 0) return 0;
    return (size_t)count * (dtype == TFDTD_F64 ? sizeof(BatchStep<double>) : sizeof(BatchStep<float>));
}

int tfdtd_batch_pack(const tfdtd_half_step* steps, int32_t count, void* host_table, size_t bytes, int32_t* block_prefix) {
    if (count < 1 || !steps) return fail(TFDTD_EINVAL, "batch: at least one descriptor");
    if (steps[0].dtype == TFDTD_F32) return pack_half_steps<float>(steps, count, host_table, bytes, block_prefix);
    if (steps[0].dtype == TFDTD_F64) return pack_half_steps<double>(steps, count, host_table, bytes, block_prefix);
    return fail(TFDTD_EINVAL, "batch: dtype must be float32 or float64");
}

int tfdtd_batch_half_step(const void* device_table, const int32_t* device_prefix, int32_t count, int32_t total_blocks,
                          int32_t dtype, int32_t family, void* stream) {
    return batch_half_step(device_table, device_prefix, count, total_blocks, dtype, family, nullptr, nullptr, 0, stream);
}

int tfdtd_batch_step(const void* e_table, const int32_t* e_prefix, int32_t e_blocks, const void* h_table, const int32_t* h_prefix,
                     int32_t h_blocks, int32_t count, int32_t dtype, int64_t* counter, int64_t* shadow, void* stream) {
    if (!counter || !shadow || e_blocks < 1 || h_blocks < 1) return fail(TFDTD_EINVAL, "batch step: counter, shadow and workgroups are required");
    long long* const n = reinterpret_cast<long long*>(counter);
    long long* const copy = reinterpret_cast<long long*>(shadow);
    const int status = batch_half_step(e_table, e_prefix, count, e_blocks, dtype, TFDTD_FAMILY_E, n, copy, 0, stream);
    if (status) return status;
    return batch_half_step(h_table, h_prefix, count, h_blocks, dtype, TFDTD_FAMILY_H, copy, n, 1, stream);
}

size_t tfdtd_batch_planes_bytes(int32_t count, int32_t dtype, int32_t spectral) {
    if (count < 0) return 0;
    if (dtype == TFDTD_F32 && spectral == 0) return (size_t)count * sizeof(Plane<float, float>);
    if (dtype == TFDTD_F32 && spectral == 1) return (size_t)count * sizeof(Plane<float, double>);
    return (size_t)count * sizeof(Plane<double, double>);
}

int tfdtd_batch_planes_pack(const tfdtd_plane* p, int32_t count, void* host_table, size_t bytes, int32_t* max_blocks,
                            int32_t* max_phases) {
    if (count < 1 || !p) return fail(TFDTD_EINVAL, "batch planes: at least one plane");
    for (int k = 1; k < count; ++k)
        if (p[k].dtype != p[0].dtype || p[k].spectral != p[0].spectral) return fail(TFDTD_EINVAL, "batch planes: mixed precision");
    if (p[0].dtype == TFDTD_F32 && p[0].spectral == 0) return pack_planes<float, float>(p, count, host_table, bytes, max_blocks, max_phases);
    if (p[0].dtype == TFDTD_F32 && p[0].spectral == 1) return pack_planes<float, double>(p, count, host_table, bytes, max_blocks, max_phases);
    if (p[0].dtype == TFDTD_F64 && p[0].spectral == 1) return pack_planes<double, double>(p, count, host_table, bytes, max_blocks, max_phases);
    return fail(TFDTD_EINVAL, "batch planes: unsupported dtype/spectral pair");
}

int tfdtd_batch_dft_update(const void* device_table, int32_t count, int32_t max_blocks, int32_t max_phases,
                           int32_t dtype, int32_t spectral, void* stream) {
    if (!device_table || count < 1 || max_blocks < 1 || max_phases < 1) return fail(TFDTD_EINVAL, "batch planes: bad launch arguments");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)max_blocks, (unsigned)count);
    if (dtype == TFDTD_F32 && spectral == 0) {
        const size_t lds = 4 * sizeof(float) * (size_t)max_phases;
        hipLaunchKernelGGL((batch_dft_kernel<float, float>), grid, dim3(256), lds, s, static_cast<const Plane<float, float>*>(device_table));
    } else if (dtype == TFDTD_F32 && spectral == 1) {
        const size_t lds = 4 * sizeof(double) * (size_t)max_phases;
        hipLaunchKernelGGL((batch_dft_kernel<float, double>), grid, dim3(256), lds, s, static_cast<const Plane<float, double>*>(device_table));
    } else if (dtype == TFDTD_F64 && spectral == 1) {
        const size_t lds = 4 * sizeof(double) * (size_t)max_phases;
        hipLaunchKernelGGL((batch_dft_kernel<double, double>), grid, dim3(256), lds, s, static_cast<const Plane<double, double>*>(device_table));
    } else {
        return fail(TFDTD_EINVAL, "batch planes: unsupported dtype/spectral pair");
    }
    return check_launch("batch_dft");
}


int tfdtd_abi_version(void) { return TFDTD_ABI_VERSION; }

#ifndef TFDTD_SOURCE_DIGEST
#define TFDTD_SOURCE_DIGEST "unknown"
#endif
const char* tfdtd_source_digest(void) { return TFDTD_SOURCE_DIGEST; }

size_t tfdtd_last_error(char* buffer, size_t size) {
    const std::string& message = tfdtd_detail::last_error;
    if (buffer && size) {
        std::strncpy(buffer, message.c_str(), size - 1);
        buffer[size - 1] = 0;
    }
    return message.size();
}

int tfdtd_yee_half_step(const tfdtd_half_step* step, void* stream) {
    return half_step(step, static_cast<hipStream_t>(stream));
}

int tfdtd_inject(const tfdtd_half_step* step, void* stream) {
    if (!step) return fail(TFDTD_EINVAL, "null half-step descriptor");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (step->dtype == TFDTD_F32) return launch_inject<float>(step, s);
    if (step->dtype == TFDTD_F64) return launch_inject<double>(step, s);
    return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
}

int tfdtd_dft_update(const tfdtd_plane* p, int32_t count, void* stream) {
    return planes(p, count, static_cast<hipStream_t>(stream));
}

int tfdtd_observe_step(const tfdtd_observe* d, void* stream) { return observe(d, static_cast<hipStream_t>(stream)); }

int tfdtd_dft_flush(const tfdtd_plane* p, int32_t count, void* stream) {
    if (count < 0 || (count > 0 && !p)) return fail(TFDTD_EINVAL, "bad plane table");
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int k = 0; k < count; ++k) {
        const tfdtd_plane* d = p + k;
        if (d->block <= 1) continue;
        int status;
        if (d->dtype == TFDTD_F32 && d->spectral == 0) status = launch_flush<float, float>(d, s);
        else if (d->dtype == TFDTD_F32 && d->spectral == 1) status = launch_flush<float, double>(d, s);
        else if (d->dtype == TFDTD_F64 && d->spectral == 1) status = launch_flush<double, double>(d, s);
        else status = fail(TFDTD_EINVAL, "plane %d: unsupported dtype/spectral pair", k);
        if (status) return status;
    }
    return TFDTD_OK;
}

int tfdtd_step_fused(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_plane* p,
                     int32_t plane_count, const tfdtd_observe* obs, int32_t n_steps, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n_steps < 0) return fail(TFDTD_EINVAL, "n_steps must be non-negative");
    if (!e_step || !h_step || e_step->family != TFDTD_FAMILY_E || h_step->family != TFDTD_FAMILY_H)
        return fail(TFDTD_EINVAL, "step_fused needs an E and an H descriptor");
    if (!obs) return fail(TFDTD_EINVAL, "step_fused needs the observe descriptor (it advances the counter)");
    for (int k = 0; k < n_steps; ++k) {
        int status = half_step(e_step, s);
        if (!status) status = half_step(h_step, s);
        if (!status) status = planes(p, plane_count, s);
        if (!status) status = observe(obs, s);
        if (status) return status;
    }
    return TFDTD_OK;
}

int tfdtd_step_observed(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_plane* p, int32_t plane_count,
                        const tfdtd_observe* obs, const tfdtd_trace_cell* cells, int64_t* shadow, void* stream) {
    return tfdtd_step_recorded(e_step, h_step, p, plane_count, obs, cells, shadow, nullptr, stream);
}

int tfdtd_step_recorded(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_plane* p, int32_t plane_count,
                        const tfdtd_observe* obs, const tfdtd_trace_cell* cells, int64_t* shadow, const tfdtd_curl_record* record,
                        void* stream) {
    if (!e_step || !h_step || e_step->family != TFDTD_FAMILY_E || h_step->family != TFDTD_FAMILY_H)
        return fail(TFDTD_EINVAL, "step_observed needs an E and an H descriptor");
    if (!obs || !obs->counter || !shadow) return fail(TFDTD_EINVAL, "step_observed needs the observe descriptor, its counter and the shadow");
    if (obs->count < 0 || (obs->count > 0 && (!obs->table || !obs->traces)))
        return fail(TFDTD_EINVAL, "observe: trace table and traces are required");
    if (e_step->dtype != h_step->dtype) return fail(TFDTD_EINVAL, "step_observed: E and H differ in dtype");
    hipStream_t s = static_cast<hipStream_t>(stream);
    long long* const copy = reinterpret_cast<long long*>(shadow);
    bool done = false;
    int status;
    if (e_step->dtype == TFDTD_F32) status = observed_step<float>(e_step, h_step, p, plane_count, obs, cells, copy, record, s, &done);
    else if (e_step->dtype == TFDTD_F64) status = observed_step<double>(e_step, h_step, p, plane_count, obs, cells, copy, record, s, &done);
    else return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
    if (status || done) return status;
    if (record && (status = tfdtd_record_curl(record, stream))) return status;
    return tfdtd_step_fused(e_step, h_step, p, plane_count, obs, 1, stream);
}

int tfdtd_flat_steps(const tfdtd_half_step* e_step, const tfdtd_half_step* h_step, const tfdtd_observe* obs,
                     const tfdtd_trace_cell* cells, const tfdtd_flat_buffers* second, int64_t* shadow, int32_t n_steps, void* stream) {
    if (!e_step || !h_step || e_step->family != TFDTD_FAMILY_E || h_step->family != TFDTD_FAMILY_H || e_step->dtype != h_step->dtype)
        return fail(TFDTD_EINVAL, "flat_steps needs an E and an H descriptor of one dtype");
    if (!obs || !obs->counter) return fail(TFDTD_EINVAL, "flat_steps needs the observe descriptor and its counter");
    if (obs->count < 0 || (obs->count > 0 && (!obs->table || !obs->traces)))
        return fail(TFDTD_EINVAL, "observe: trace table and traces are required");
    if (n_steps < 0 || n_steps == 1) return fail(TFDTD_EINVAL, "flat_steps takes two steps or more (0: asks whether it takes the grid)");
    if (n_steps > 0 && (!shadow || !second || !second->e || !second->h || !second->psi_e || !second->psi_h))
        return fail(TFDTD_EINVAL, "flat_steps needs a second buffer set and the shadow");
    const tfdtd_flat_buffers b = second ? *second : tfdtd_flat_buffers{};
    long long* const copy = reinterpret_cast<long long*>(shadow);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (e_step->dtype == TFDTD_F32)
        return flat_steps<float>(e_step, h_step, obs, cells, {(float*)b.e, (float*)b.h, (float*)b.psi_e, (float*)b.psi_h}, copy, n_steps, s);
    if (e_step->dtype == TFDTD_F64)
        return flat_steps<double>(e_step, h_step, obs, cells, {(double*)b.e, (double*)b.h, (double*)b.psi_e, (double*)b.psi_h}, copy, n_steps, s);
    return fail(TFDTD_EINVAL, "dtype must be float32 or float64");
}

int tfdtd_record_traces(const tfdtd_observe* d, void* stream) {
    if (!d || !d->counter) return fail(TFDTD_EINVAL, "traces need the observe descriptor and a step counter");
    return record_traces(d, reinterpret_cast<const long long*>(d->counter), static_cast<hipStream_t>(stream));
}

}  // extern "C"
