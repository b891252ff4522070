// Discrete adjoint of the Yee/CPML step for gfx950, and the forward record it needs.
//
// The exact transpose of one step (torchfdtd/differentiable.py:395-447 and 496-519; the
// reference's fused form is torchfdtd/cuda_adjoint.py:16-234) runs backwards in three
// launches per step, each thread owning one cell and writing only that cell (gather form,
// no atomics):
//   seeds:        e_bar/h_bar += the observation adjoints of step t (CSR over targets);
//   h_transpose:  e_bar += curl_T(forward)(-(S*inv_mu) h_bar), the H-family memory adjoint
//                 psi_bar_prev = b*(psi_bar + d) from one buffer into the other, and the
//                 permittivity gradient -S * e_bar . curl_H(t) * inv_eps^2 on the design box;
//   e_transpose:  h_bar += curl_T(backward)((S*inv_eps) e_bar), with the E-family memory
//                 adjoint likewise; block 0 then steps the counter back.
// The curl of H that step t's E update used is recorded during the forward run on the
// design box (record_curl) in slot t % modulus, so the backward sweep needs no forward
// state at all -- only the recorded box.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/tfdtd.h"
#include "common.h"
#include "cpml_faces.h"
#include "plane_march.h"

namespace {

template <typename real>
struct Adjoint {
    int n[3];
    real* e_bar;
    real* h_bar;
    const real* inv_eps;
    int eps_stride;
    const real* inv_mu;           // one value
    real S;                       // courant, rounded as the forward step rounds it
    int periodic, pec;
    real pec_factor[3];
    Family<real> ef, hf;          // psi_in: adjoint of the memory after the step, psi_out: before it
    int nseed;
    const long long* seed_targets;
    const int* seed_offsets;
    const int* seed_columns;
    const real* seeds;
    int seed_width;
    long long seed_rows;
    int box_lo[3], box_hi[3];
    const real* record;
    long long modulus;
    double* gradient;
    int gradient_stride;
    long long* counter;
};

__device__ __forceinline__ long long cell_index(const int n[3], int x, int y, int z) {
    return ((long long)x * n[1] + y) * n[2] + z;
}

// Offset of cell (x, y, z) inside a slab memory array of `axis` (extent w, slab row q).
__device__ __forceinline__ unsigned slab_offset(const int n[3], int axis, int q, int w, int x, int y, int z) {
    int c[3] = {x, y, z}, d[3] = {n[0], n[1], n[2]};
    c[axis] = q;
    d[axis] = w;
    return (unsigned)(((long long)c[0] * d[1] + c[1]) * d[2] + c[2]);
}

// d_D of one term at one row: d*inv_k + c*(psi_bar + d); the owner also stores b*(psi_bar + d).
template <typename real>
__device__ __forceinline__ real transpose_row(real d, const Family<real>& F, int axis, int which, int row,
                                              const int n[3], int x, int y, int z, bool owner) {
    const Hit h = find_hit(F, axis, row);
    if (h.face < 0) return d;
    const unsigned o = (which ? h.psi1 : h.psi0) + slab_offset(n, axis, h.q, h.w, x, y, z);
    const real b = F.coef[h.coef + h.q];
    const real c = F.coef[h.coef + h.w + h.q];
    const real ik = F.coef[h.coef + 2 * h.w + h.q];
    const real m = F.psi_in[o] + d;
    if (owner) F.psi_out[o] = b * m;
    return d * ik + c * m;
}

// The cell of this thread in the transpose launches: lanes along z, the block's four wavefronts
// along y, blocks over (z tile of 64, y tile of 4, x) -- the block's coordinates come from uniform
// 32-bit arithmetic, so no lane divides 64-bit indices.
constexpr int kTileZ = 64, kTileY = 4;

struct Cell3 {
    int x, y, z;
    long long j;
    bool inside;
};

__device__ __forceinline__ Cell3 locate(const int n[3]) {
    const int zt = (n[2] + kTileZ - 1) / kTileZ, yt = (n[1] + kTileY - 1) / kTileY;
    const int b = blockIdx.x;
    const int r = b / zt;
    Cell3 c;
    c.z = (b - r * zt) * kTileZ + (int)(threadIdx.x & (kTileZ - 1));
    c.x = r / yt;
    c.y = (r - c.x * yt) * kTileY + (int)(threadIdx.x / kTileZ);
    c.inside = c.x < n[0] && c.y < n[1] && c.z < n[2];
    c.j = ((long long)c.x * n[1] + c.y) * n[2] + c.z;
    return c;
}

inline unsigned transpose_blocks(const int n[3]) {
    return (unsigned)n[0] * (unsigned)((n[1] + kTileY - 1) / kTileY) * (unsigned)((n[2] + kTileZ - 1) / kTileZ);
}

template <typename real>
__global__ __launch_bounds__(256) void seed_kernel(const Adjoint<real> a) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nseed) return;
    const long long t = *a.counter;
    if (t < 0 || t >= a.seed_rows) return;
    real sum = real(0);
    for (int j = a.seed_offsets[k]; j < a.seed_offsets[k + 1]; ++j) sum = sum + a.seeds[t * a.seed_width + a.seed_columns[j]];
    real* field = a.seed_targets[2 * k] ? a.h_bar : a.e_bar;
    field[a.seed_targets[2 * k + 1]] += sum;
}

// Both transposes read every field value they need (the cell and its neighbour along each axis)
// into registers before the first memory-array store: stores through psi_out would otherwise keep
// the compiler from reusing or hoisting later field loads.
template <typename real>
__global__ __launch_bounds__(256) void h_transpose_kernel(const Adjoint<real> a) {
    const Cell3 cell = locate(a.n);
    if (!cell.inside) return;
    const int x = cell.x, y = cell.y, z = cell.z;
    const long long j = cell.j;
    const int p[3] = {x, y, z};
    const real hcoef = a.S * a.inv_mu[0];
    real ob[3], down[3][3], eb[3];
    for (int o = 0; o < 3; ++o) ob[o] = -hcoef * a.h_bar[3 * j + o];
    for (int c = 0; c < 3; ++c) eb[c] = a.e_bar[3 * j + c];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        // Row i-1 of the axis, or row n-1 across the periodic wrap at i = 0.
        const int na = a.n[ax], i = p[ax];
        const long long stride = ax == 0 ? (long long)a.n[1] * a.n[2] : ax == 1 ? a.n[2] : 1;
        const bool has = na > 1 && (i >= 1 || (a.periodic >> ax & 1));
        const long long nb = i >= 1 ? j - stride : j + (long long)(na - 1) * stride;
        for (int o = 0; o < 3; ++o) down[ax][o] = has ? -hcoef * a.h_bar[3 * nb + o] : real(0);
    }
    real acc[3] = {real(0), real(0), real(0)};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int ax = term_axis(t), c = term_in(t), o = term_out(t), s = term_sign(t);
        const int na = a.n[ax], i = p[ax];
        if (na == 1) continue;
        // Forward differences: rows 0 .. n-2 carry a derivative; E_c[i+1] += d_D[i], E_c[i] -= d_D[i].
        if (i <= na - 2) {
            const real d = transpose_row(real(s) * ob[o], a.hf, ax, t & 1, i, a.n, x, y, z, true);
            acc[c] = acc[c] - d;
        }
        if (i >= 1) {
            int q[3] = {x, y, z};
            q[ax] = i - 1;
            const real d = transpose_row(real(s) * down[ax][o], a.hf, ax, t & 1, i - 1, a.n, q[0], q[1], q[2], false);
            acc[c] = acc[c] + d;
        }
        if (a.periodic >> ax & 1) {
            // Wrap term at row n-1: E_c[0] += s*ob[n-1], E_c[n-1] -= s*ob[n-1].
            if (i == 0) acc[c] = acc[c] + real(s) * down[ax][o];
            if (i == na - 1) acc[c] = acc[c] - real(s) * ob[o];
        } else if ((a.pec >> ax & 1) && i == na - 1) {
            acc[c] = acc[c] - real(s) * a.pec_factor[ax] * ob[o];
        }
    }
    real e[3];
    for (int c = 0; c < 3; ++c) {
        e[c] = eb[c] + acc[c];
        a.e_bar[3 * j + c] = e[c];
    }
    const long long t = *a.counter;
    if (t >= 0 && x >= a.box_lo[0] && x < a.box_hi[0] && y >= a.box_lo[1] && y < a.box_hi[1] && z >= a.box_lo[2] && z < a.box_hi[2]) {
        const int bx = a.box_hi[0] - a.box_lo[0], by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
        const long long b = ((long long)(x - a.box_lo[0]) * by + (y - a.box_lo[1])) * bz + (z - a.box_lo[2]);
        const real* curl = a.record + ((t % a.modulus) * ((long long)bx * by * bz) + b) * 3;
        double sum = 0.;
        for (int c = 0; c < 3; ++c) {
            const real inv = a.inv_eps[a.eps_stride == 3 ? 3 * j + c : j];
            const real g = -a.S * e[c] * curl[c] * (inv * inv);
            if (a.gradient_stride == 3) a.gradient[3 * b + c] += (double)g;
            else sum += (double)g;
        }
        if (a.gradient_stride == 1) a.gradient[b] += sum;
    }
}

template <typename real>
__global__ __launch_bounds__(256) void e_transpose_kernel(const Adjoint<real> a) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.counter = *a.counter - 1;
    const Cell3 cell = locate(a.n);
    if (!cell.inside) return;
    const int x = cell.x, y = cell.y, z = cell.z;
    const long long j = cell.j;
    const int p[3] = {x, y, z};
    auto obar = [&](long long at, int o) {
        const real inv = a.inv_eps[a.eps_stride == 3 ? 3 * at + o : at];
        return (a.S * inv) * a.e_bar[3 * at + o];
    };
    real own[3], up[3][3], hb[3];
    for (int o = 0; o < 3; ++o) own[o] = obar(j, o);
    for (int c = 0; c < 3; ++c) hb[c] = a.h_bar[3 * j + c];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        // Row i+1 of the axis, or row 0 across the periodic wrap at i = n-1.
        const int na = a.n[ax], i = p[ax];
        const long long stride = ax == 0 ? (long long)a.n[1] * a.n[2] : ax == 1 ? a.n[2] : 1;
        const bool has = na > 1 && (i + 1 <= na - 1 || (a.periodic >> ax & 1));
        const long long nb = i + 1 <= na - 1 ? j + stride : j - (long long)(na - 1) * stride;
        for (int o = 0; o < 3; ++o) up[ax][o] = has ? obar(nb, o) : real(0);
    }
    real acc[3] = {real(0), real(0), real(0)};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int ax = term_axis(t), c = term_in(t), o = term_out(t), s = term_sign(t);
        const int na = a.n[ax], i = p[ax];
        if (na == 1) continue;
        // Backward differences: rows 1 .. n-1 carry a derivative; H_c[i] += d_D[i], H_c[i-1] -= d_D[i].
        if (i >= 1) {
            const real d = transpose_row(real(s) * own[o], a.ef, ax, t & 1, i, a.n, x, y, z, true);
            acc[c] = acc[c] + d;
        }
        if (i + 1 <= na - 1) {
            int q[3] = {x, y, z};
            q[ax] = i + 1;
            const real d = transpose_row(real(s) * up[ax][o], a.ef, ax, t & 1, i + 1, a.n, q[0], q[1], q[2], false);
            acc[c] = acc[c] - d;
        }
        if (a.periodic >> ax & 1) {
            // Wrap term at row 0: H_c[0] += s*ob[0], H_c[n-1] -= s*ob[0].
            if (i == 0) acc[c] = acc[c] + real(s) * own[o];
            if (i == na - 1) acc[c] = acc[c] - real(s) * up[ax][o];
        }
    }
    for (int c = 0; c < 3; ++c) a.h_bar[3 * j + c] = hb[c] + acc[c];
}

// ---------------------------------------------------------------- transposes marched over x planes
//
// The half steps' march (64 cells of the flattened (y, z) plane a wavefront, two x planes) for the two
// transposes.  What a cell needs of the x row before (H) or after (E) it is what the plane before computed or
// the plane after will: that row's value is carried, so its memory is read once; the neighbour rows along y
// and z are read with the cell's own.  The arithmetic and its order are those of the kernels above, which
// keep the grids that the march does not take.  200x160x60 cells in FP32: 40.0 + 39.2 -> 20.3 + 19.5 us (5.6 TB/s of
// the 76 bytes a cell and the memory); 71x66x37 in FP64: 15.5 + 14.6 -> 9.0 + 7.6 us.
template <typename real>
struct AdjointMarch {
    int nx, ny, nz, nyz;
    int span, columns;
    Divider by_nz, by_columns;
    int xcd;
    real* e_bar;
    real* h_bar;
    const real* inv_eps;
    const real* inv_mu;
    const real* psi_in;         // the memory of the launch's family
    real* psi_out;
    const real* coef;
    PlaneAxis<real> axis[3];
    real S;
    int periodic, pec;
    real pec_factor[3];
    int box_lo[3], box_hi[3];
    const real* record;
    long long modulus;
    double* gradient;
    int gradient_stride;
    long long* counter;
};

// The cells of a wavefront: lane position in the plane and its planes.  Spare lanes and wavefronts repeat a
// cell and store nothing.
struct MarchCell {
    bool owned;
    unsigned r;
    int xa, xb, y, z;
};

template <bool FLAT, typename A>
__device__ __forceinline__ MarchCell march_cell(const A& a) {
    const unsigned item = wave_item(xcd_block(blockIdx.x, gridDim.x, a.xcd));
    const unsigned chunks = (unsigned)(a.nx + a.span - 1) / (unsigned)a.span;
    const unsigned xchunk = min(divide(item, a.by_columns), chunks - 1u);
    const unsigned cell = (item - xchunk * a.columns) * 64u + (threadIdx.x & 63u);
    MarchCell c;
    c.owned = cell < (unsigned)a.nyz;
    c.r = min(cell, (unsigned)a.nyz - 1u);
    c.xa = (int)xchunk * a.span;
    c.xb = min(a.nx, c.xa + a.span);
    c.y = FLAT ? (int)c.r : (int)divide(c.r, a.by_nz);
    c.z = FLAT ? 0 : (int)(c.r - (unsigned)c.y * a.nz);
    return c;
}

// A row of an axis at a lane: the memory of its two terms and their coefficients.
template <typename real>
struct MarchRow {
    bool on;
    unsigned at[2], stride;     // byte offsets at x = 0 (x axis: of this row), bytes per x plane
    real b, c, ik;
    // d_D of a term; m: the memory before, then memory + d, of which b is the new memory.
    __device__ __forceinline__ real value(real d, real& m) const {
        if (!on) return d;
        m = m + d;
        return d * ik + c * m;
    }
};

template <typename real, int Axis, typename A>
__device__ __forceinline__ MarchRow<real> march_row(const A& a, int k, bool inside, const MarchCell& p) {
    constexpr unsigned W = sizeof(real);
    const AxisRow<real> r = axis_row(a.axis[Axis], k, inside);
    MarchRow<real> m{r.on, {0u, 0u}, 0u, real(0), real(0), real(0)};
    if (r.on) {
        const unsigned wide = (unsigned)r.w * W, q = (unsigned)r.q * W, at = r.coef + q;
        const unsigned e = Axis == 0 ? q * a.nyz + p.r * W : Axis == 1 ? q * a.nz + p.z * W : p.y * wide + q;
        m.stride = Axis == 0 ? 0u : wide * (unsigned)(Axis == 1 ? a.nz : a.ny);
        for (int t = 0; t < 2; ++t) m.at[t] = r.psi[t] + e;
        m.b = at_byte(a.coef, at);
        m.c = at_byte(a.coef, at + wide);
        m.ik = at_byte(a.coef, at + 2 * wide);
    }
    return m;
}

template <typename real>
__device__ __forceinline__ void read_memory(const real* psi, const MarchRow<real>& row, int x, real m[2]) {
    m[0] = m[1] = real(0);
    if (row.on)
        for (int k = 0; k < 2; ++k) m[k] = at_byte(psi, row.at[k] + x * row.stride);
}

template <typename real>
__device__ __forceinline__ void write_memory(real* psi, const MarchRow<real>& row, int x, const real m[2]) {
    if (row.on)
        for (int k = 0; k < 2; ++k) put_byte(psi, row.at[k] + x * row.stride, row.b * m[k]);
}

template <typename real, int INV, bool FLAT>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 3 : 5) void h_transpose_march_kernel(const AdjointMarch<real> a) {
    constexpr unsigned W = sizeof(real);
    const MarchCell p = march_cell<FLAT>(a);
    const int nx = a.nx, ny = a.ny, nz = FLAT ? 1 : a.nz, y = p.y, z = p.z;
    const bool wrapx = a.periodic & 1, wrapy = a.periodic & 2, wrapz = !FLAT && (a.periodic & 4);
    const unsigned off = p.r * (3 * W), rowb = (unsigned)nz * (3 * W);
    const unsigned offy = y >= 1 ? off - rowb : wrapy ? off + (unsigned)(ny - 1) * rowb : off;
    const unsigned offz = FLAT ? off : z >= 1 ? off - 3 * W : wrapz ? off + (unsigned)(nz - 1) * (3 * W) : off;
    const long long plane = 3LL * a.nyz;
    const real* h = a.h_bar + p.xa * plane;
    real* e = a.e_bar + p.xa * plane;
    const real hcoef = a.S * global(a.inv_mu)[0];
    auto scaled = [&](const Cell<real>& c) { return Cell<real>{{-hcoef * c.v[0], -hcoef * c.v[1], -hcoef * c.v[2]}}; };
    Cell<real> here = cell_at_byte(h, off);
    // Row x - 1; at x = 0 of a periodic axis row nx - 1.
    const Cell<real> below = scaled(cell_at_byte(p.xa > 0 ? h - plane : wrapx ? a.h_bar + (nx - 1) * plane : h, off));
    const MarchRow<real> oy = march_row<real, 1>(a, y, y <= ny - 2, p), dy = march_row<real, 1>(a, y - 1, y >= 1, p);
    MarchRow<real> oz{false, {0u, 0u}, 0u, real(0), real(0), real(0)}, dz = oz;
    if (!FLAT) {
        oz = march_row<real, 2>(a, z, z <= nz - 2, p);
        dz = march_row<real, 2>(a, z - 1, z >= 1, p);
    }
    real carried[2] = {real(0), real(0)};       // row x - 1's values of the two x terms
    if (p.xa > 0) {
        const MarchRow<real> row = march_row<real, 0>(a, p.xa - 1, true, p);
        real m[2];
        read_memory(a.psi_in, row, 0, m);
        for (int k = 0; k < 2; ++k) carried[k] = row.value(real(term_sign(k)) * below.v[term_out(k)], m[k]);
    }
    const bool in_box = p.owned && y >= a.box_lo[1] && y < a.box_hi[1] && z >= a.box_lo[2] && z < a.box_hi[2];
    for (int x = p.xa; x < p.xb; ++x, h += plane, e += plane) {
        const Cell<real> ob = scaled(here), eb = cell_at_byte(e, off), ylow = scaled(cell_at_byte(h, offy));
        Cell<real> zlow = ob, ahead = here;
        if (!FLAT) zlow = scaled(cell_at_byte(h, offz));
        if (x + 1 < p.xb) ahead = cell_at_byte(h + plane, off);
        // Every memory value is read before the first store.
        const MarchRow<real> ox = march_row<real, 0>(a, x, x <= nx - 2, p);
        real mx[2], my[2], mz[2], my_low[2], mz_low[2];
        read_memory(a.psi_in, ox, 0, mx);
        read_memory(a.psi_in, oy, x, my);
        read_memory(a.psi_in, dy, x, my_low);
        read_memory(a.psi_in, oz, x, mz);
        read_memory(a.psi_in, dz, x, mz_low);
        real acc[3] = {real(0), real(0), real(0)};
        // Term k of an axis at row i of n.  Forward differences: rows 0 .. n-2 carry a derivative;
        // E_c[i+1] += d_D[i], E_c[i] -= d_D[i]; the wrap term at row n-1: E_c[0] += s ob[n-1], E_c[n-1] -= s ob[n-1].
        auto term = [&](auto axis_tag, int k, int i, int n, bool wrap, real own, real lower, real low) {
            constexpr int axis = decltype(axis_tag)::value;
            const int t = 2 * axis + k, c = term_in(t), o = term_out(t);
            const real sg = real(term_sign(t));
            if (i <= n - 2) acc[c] = acc[c] - own;
            if (i >= 1) acc[c] = acc[c] + lower;
            if (wrap) {
                if (i == 0) acc[c] = acc[c] + sg * low;
                if (i == n - 1) acc[c] = acc[c] - sg * ob.v[o];
            } else if ((a.pec >> axis & 1) && i == n - 1) {
                acc[c] = acc[c] - sg * a.pec_factor[axis] * ob.v[o];
            }
        };
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int o = term_out(k);
            const real d = ox.value(real(term_sign(k)) * ob.v[o], mx[k]);
            term(std::integral_constant<int, 0>{}, k, x, nx, wrapx, d, carried[k], below.v[o]);
            carried[k] = d;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int o = term_out(2 + k);
            const real sg = real(term_sign(2 + k));
            term(std::integral_constant<int, 1>{}, k, y, ny, wrapy, oy.value(sg * ob.v[o], my[k]), dy.value(sg * ylow.v[o], my_low[k]), ylow.v[o]);
        }
        if (!FLAT)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int o = term_out(4 + k);
                const real sg = real(term_sign(4 + k));
                term(std::integral_constant<int, 2>{}, k, z, nz, wrapz, oz.value(sg * ob.v[o], mz[k]), dz.value(sg * zlow.v[o], mz_low[k]), zlow.v[o]);
            }
        if (p.owned) {
            write_memory(a.psi_out, ox, 0, mx);
            write_memory(a.psi_out, oy, x, my);
            write_memory(a.psi_out, oz, x, mz);
        }
        real value[3];
        for (int c = 0; c < 3; ++c) value[c] = eb.v[c] + acc[c];
        if (p.owned) {
            const auto to = global(reinterpret_cast<real*>(reinterpret_cast<char*>(e) + off));
            for (int c = 0; c < 3; ++c) to[c] = value[c];
        }
        here = ahead;
        if (!in_box || x < a.box_lo[0] || x >= a.box_hi[0]) continue;
        const long long t = *global(a.counter);
        if (t < 0) continue;
        const int bx = a.box_hi[0] - a.box_lo[0], by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
        const long long b = ((long long)(x - a.box_lo[0]) * by + (y - a.box_lo[1])) * bz + (z - a.box_lo[2]);
        const Cell<real> curl = cell_at(a.record, slot_of(t, a.modulus) * ((long long)bx * by * bz) + b);
        const long long j = (long long)x * a.nyz + p.r;
        double sum = 0.;
        for (int c = 0; c < 3; ++c) {
            const real inv = global(a.inv_eps)[INV == 3 ? 3 * j + c : j];
            const real g = -a.S * value[c] * curl.v[c] * (inv * inv);
            if (a.gradient_stride == 3) global(a.gradient)[3 * b + c] += (double)g;
            else sum += (double)g;
        }
        if (a.gradient_stride == 1) global(a.gradient)[b] += sum;
    }
}

template <typename real, int INV, bool FLAT>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 3 : 5) void e_transpose_march_kernel(const AdjointMarch<real> a) {
    constexpr unsigned W = sizeof(real);
    if (blockIdx.x == 0 && threadIdx.x == 0) *global(a.counter) = *global(a.counter) - 1;
    const MarchCell p = march_cell<FLAT>(a);
    const int nx = a.nx, ny = a.ny, nz = FLAT ? 1 : a.nz, y = p.y, z = p.z;
    const bool wrapx = a.periodic & 1, wrapy = a.periodic & 2, wrapz = !FLAT && (a.periodic & 4);
    const unsigned off = p.r * (3 * W), rowb = (unsigned)nz * (3 * W);
    const bool hasy = y + 1 <= ny - 1, hasz = !FLAT && z + 1 <= nz - 1;
    const unsigned offy = hasy ? off + rowb : wrapy ? off - (unsigned)(ny - 1) * rowb : off;
    const unsigned offz = FLAT ? off : hasz ? off + 3 * W : wrapz ? off - (unsigned)(nz - 1) * (3 * W) : off;
    const long long plane = 3LL * a.nyz;
    const real* e = a.e_bar + p.xa * plane;
    real* h = a.h_bar + p.xa * plane;
    // (S inv_eps) e_bar of the lane at byte offset `at` of a plane.
    auto obar = [&](const real* ep, int x, unsigned at) {
        const Cell<real> c = cell_at_byte(ep, at);
        Cell<real> i;
        if (INV == 3) i = cell_at_byte(a.inv_eps + x * plane, at);
        else {
            const real v = at_byte(a.inv_eps + (long long)x * a.nyz, at / 3);
            i = Cell<real>{{v, v, v}};
        }
        return Cell<real>{{(a.S * i.v[0]) * c.v[0], (a.S * i.v[1]) * c.v[1], (a.S * i.v[2]) * c.v[2]}};
    };
    Cell<real> own = obar(e, p.xa, off);
    const MarchRow<real> oy = march_row<real, 1>(a, y, y >= 1, p), uy = march_row<real, 1>(a, y + 1, hasy, p);
    MarchRow<real> oz{false, {0u, 0u}, 0u, real(0), real(0), real(0)}, uz = oz;
    if (!FLAT) {
        oz = march_row<real, 2>(a, z, z >= 1, p);
        uz = march_row<real, 2>(a, z + 1, hasz, p);
    }
    // Row x of the x axis: its values and memory, computed as the row after by the plane before.
    MarchRow<real> row = march_row<real, 0>(a, p.xa, p.xa >= 1, p);
    real mx[2], carried[2];
    read_memory(a.psi_in, row, 0, mx);
    for (int k = 0; k < 2; ++k) carried[k] = row.value(real(term_sign(k)) * own.v[term_out(k)], mx[k]);
    for (int x = p.xa; x < p.xb; ++x, h += plane, e += plane) {
        const bool hasx = x + 1 <= nx - 1;
        const Cell<real> hb = cell_at_byte(h, off), yup = obar(e, x, offy);
        Cell<real> zup = own;
        if (!FLAT) zup = obar(e, x, offz);
        const Cell<real> xup = hasx ? obar(e + plane, x + 1, off) : wrapx ? obar(a.e_bar, 0, off) : own;
        const MarchRow<real> next = march_row<real, 0>(a, x + 1, hasx, p);
        real mn[2], my[2], mz[2], my_up[2], mz_up[2];
        read_memory(a.psi_in, next, 0, mn);
        read_memory(a.psi_in, oy, x, my);
        read_memory(a.psi_in, uy, x, my_up);
        read_memory(a.psi_in, oz, x, mz);
        read_memory(a.psi_in, uz, x, mz_up);
        real acc[3] = {real(0), real(0), real(0)};
        // Backward differences: rows 1 .. n-1 carry a derivative; H_c[i] += d_D[i], H_c[i-1] -= d_D[i]; the wrap
        // term at row 0: H_c[0] += s ob[0], H_c[n-1] -= s ob[0].
        auto term = [&](auto axis_tag, int k, int i, int n, bool wrap, real mine, real upper, real up) {
            constexpr int axis = decltype(axis_tag)::value;
            const int t = 2 * axis + k, c = term_in(t), o = term_out(t);
            const real sg = real(term_sign(t));
            if (i >= 1) acc[c] = acc[c] + mine;
            if (i + 1 <= n - 1) acc[c] = acc[c] - upper;
            if (wrap) {
                if (i == 0) acc[c] = acc[c] + sg * own.v[o];
                if (i == n - 1) acc[c] = acc[c] - sg * up;
            }
        };
        real following[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int o = term_out(k);
            following[k] = next.value(real(term_sign(k)) * xup.v[o], mn[k]);
            term(std::integral_constant<int, 0>{}, k, x, nx, wrapx, carried[k], following[k], xup.v[o]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int o = term_out(2 + k);
            const real sg = real(term_sign(2 + k));
            term(std::integral_constant<int, 1>{}, k, y, ny, wrapy, oy.value(sg * own.v[o], my[k]), uy.value(sg * yup.v[o], my_up[k]), yup.v[o]);
        }
        if (!FLAT)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int o = term_out(4 + k);
                const real sg = real(term_sign(4 + k));
                term(std::integral_constant<int, 2>{}, k, z, nz, wrapz, oz.value(sg * own.v[o], mz[k]), uz.value(sg * zup.v[o], mz_up[k]), zup.v[o]);
            }
        if (p.owned) {
            write_memory(a.psi_out, row, 0, mx);
            write_memory(a.psi_out, oy, x, my);
            write_memory(a.psi_out, oz, x, mz);
            const auto to = global(reinterpret_cast<real*>(reinterpret_cast<char*>(h) + off));
            for (int c = 0; c < 3; ++c) to[c] = hb.v[c] + acc[c];
        }
        own = xup;
        row = next;
        for (int k = 0; k < 2; ++k) { mx[k] = mn[k]; carried[k] = following[k]; }
    }
}

template <typename real>
struct Record {
    int n[3];
    const real* H;
    int periodic;
    int box_lo[3], box_hi[3];
    real* record;
    long long modulus;
    const long long* counter;
    int cpml;                     // 1: apply the E-family slabs of ef (psi_in = memory before the step)
    Family<real> ef;
};

// curl_H of the E update (backward differences, terms in curl order) on the design box; in an
// E-family slab row a term is d inv_k + (b psi + c d), the value the update adds there.
template <typename real>
__global__ __launch_bounds__(256) void record_kernel(const Record<real> a) {
    const int bx = a.box_hi[0] - a.box_lo[0], by = a.box_hi[1] - a.box_lo[1], bz = a.box_hi[2] - a.box_lo[2];
    const long long count = (long long)bx * by * bz;
    const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= count) return;
    const int z = a.box_lo[2] + (int)(b % bz), y = a.box_lo[1] + (int)((b / bz) % by), x = a.box_lo[0] + (int)(b / ((long long)by * bz));
    const int p[3] = {x, y, z};
    const long long j = cell_index(a.n, x, y, z);
    real curl[3] = {real(0), real(0), real(0)};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const int ax = term_axis(t), c = term_in(t), o = term_out(t), s = term_sign(t);
        const int na = a.n[ax];
        if (na == 1) continue;
        const long long stride = ax == 0 ? (long long)a.n[1] * a.n[2] : ax == 1 ? a.n[2] : 1;
        real d;
        if (p[ax] >= 1) d = a.H[3 * j + c] - a.H[3 * (j - stride) + c];
        else if (a.periodic >> ax & 1) d = a.H[3 * j + c] - a.H[3 * (j + (long long)(na - 1) * stride) + c];
        else continue;
        if (a.cpml) {
            const Hit h = find_hit(a.ef, ax, p[ax]);
            if (h.face >= 0) {
                const unsigned m = ((t & 1) ? h.psi1 : h.psi0) + slab_offset(a.n, ax, h.q, h.w, x, y, z);
                const real b = a.ef.coef[h.coef + h.q];
                const real cc = a.ef.coef[h.coef + h.w + h.q];
                const real ik = a.ef.coef[h.coef + 2 * h.w + h.q];
                const real psi = b * a.ef.psi_in[m] + cc * d;
                d = d * ik + psi;
            }
        }
        curl[o] = curl[o] + real(s) * d;
    }
    real* out = a.record + ((*a.counter % a.modulus) * count + b) * 3;
    for (int o = 0; o < 3; ++o) out[o] = curl[o];
}

// The same march over the design box for the record: `box` is the box as a plane march (its planes, its (y, z)
// plane), `grid` the field's planes and E-family memory.
struct MarchBox {
    int nx, nyz, nz, span, columns;
    Divider by_nz, by_columns;
    int xcd;
};

template <typename real>
struct MarchGrid {
    int ny, nz, nyz;
    const real* coef;
    PlaneAxis<real> axis[3];
};

template <typename real>
struct RecordMarch {
    MarchBox box;
    MarchGrid<real> grid;
    int nx, lo[3];
    const real* H;
    const real* psi;
    int periodic;
    real* record;
    long long modulus;
    const long long* counter;
};

template <typename real>
__global__ __launch_bounds__(256, sizeof(real) == 8 ? 4 : 8) void record_march_kernel(const RecordMarch<real> a) {
    constexpr unsigned W = sizeof(real);
    const MarchCell in = march_cell<false>(a.box);
    const int ny = a.grid.ny, nz = a.grid.nz;
    MarchCell p = in;
    p.y = in.y + a.lo[1];
    p.z = in.z + a.lo[2];
    p.r = (unsigned)(p.y * nz + p.z);
    const bool iny = p.y >= 1, inz = p.z >= 1, wrapx = a.periodic & 1, wrapy = a.periodic & 2, wrapz = a.periodic & 4;
    const unsigned off = p.r * (3 * W), rowb = (unsigned)nz * (3 * W);
    const unsigned offy = iny ? off - rowb : wrapy ? off + (unsigned)(ny - 1) * rowb : off;
    const unsigned offz = inz ? off - 3 * W : wrapz ? off + (unsigned)(nz - 1) * (3 * W) : off;
    const long long plane = 3LL * a.grid.nyz;
    const real* h = a.H + (in.xa + a.lo[0]) * plane;
    Cell<real> below = cell_at_byte(in.xa + a.lo[0] > 0 ? h - plane : wrapx ? a.H + (a.nx - 1) * plane : h, off);
    const MarchRow<real> ry = march_row<real, 1>(a.grid, p.y, iny, p);
    const MarchRow<real> rz = march_row<real, 2>(a.grid, p.z, inz && nz > 1, p);
    real* out = a.record + (slot_of(*global(a.counter), a.modulus) * ((long long)a.box.nx * a.box.nyz) + (long long)in.xa * a.box.nyz + in.r) * 3;
    for (int i = in.xa; i < in.xb; ++i, h += plane, out += 3LL * a.box.nyz) {
        const int x = i + a.lo[0];
        const Cell<real> here = cell_at_byte(h, off), ylow = cell_at_byte(h, offy), zlow = cell_at_byte(h, offz);
        const MarchRow<real> rx = march_row<real, 0>(a.grid, x, x >= 1 && a.nx > 1, p);
        real mx[2], my[2], mz[2], curl[3] = {real(0), real(0), real(0)};
        read_memory(a.psi, rx, 0, mx);
        read_memory(a.psi, ry, x, my);
        read_memory(a.psi, rz, x, mz);
        auto terms = [&](auto axis_tag, bool derivative, const Cell<real>& low, const MarchRow<real>& row, const real* m) {
            constexpr int axis = decltype(axis_tag)::value;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int t = 2 * axis + k, c = term_in(t), o = term_out(t);
                real d = here.v[c] - low.v[c];
                if (row.on) {
                    const real psi = row.b * m[k] + row.c * d;
                    d = d * row.ik + psi;
                }
                if (derivative) curl[o] = curl[o] + real(term_sign(t)) * d;
            }
        };
        terms(std::integral_constant<int, 0>{}, a.nx > 1 && (x >= 1 || wrapx), below, rx, mx);
        terms(std::integral_constant<int, 1>{}, ny > 1 && (iny || wrapy), ylow, ry, my);
        terms(std::integral_constant<int, 2>{}, nz > 1 && (inz || wrapz), zlow, rz, mz);
        if (in.owned)
            for (int o = 0; o < 3; ++o) global(out)[o] = curl[o];
        below = here;
    }
}

// The slabs of a family as the marches read them; false beyond 32-bit byte offsets.
template <typename real>
bool march_axes(const Family<real>& f, const int n[3], PlaneAxis<real> axis[3]) {
    constexpr long long limit = 0xffffffffLL, W = sizeof(real);
    const long long cells = (long long)n[0] * n[1] * n[2];
    for (int ax = 0; ax < 3; ++ax) {
        unsigned at[2][2] = {{0u, 0u}, {0u, 0u}}, block[2] = {0u, 0u};
        for (int side = 0; side < 2; ++side) {
            const Face& face = f.face[ax][side];
            const long long w = face.hi - face.lo, values = w * (cells / n[ax]);
            if (w == 0) continue;
            if ((face.psi[0] + values) * W > limit || (face.psi[1] + values) * W > limit || (face.coef + 3 * w) * W > limit) return false;
            for (int t = 0; t < 2; ++t) at[side][t] = face.psi[t] * (unsigned)W;
            block[side] = face.coef * (unsigned)W;
            axis[ax].lo[side] = face.lo;
            axis[ax].hi[side] = face.hi;
        }
        for (int t = 0; t < 2; ++t) {
            axis[ax].psi[t] = at[0][t];
            axis[ax].high[t] = at[1][t] - at[0][t];
        }
        axis[ax].coef = block[0];
        axis[ax].coef_high = block[1] - block[0];
    }
    return true;
}

template <typename real>
bool make_record_march(const Record<real>& d, RecordMarch<real>* out) {
    RecordMarch<real>& a = *out;
    std::memset(&a, 0, sizeof a);
    const long long nyz = (long long)d.n[1] * d.n[2];
    if (nyz * 3 * (long long)sizeof(real) > 0xffffffffLL) return false;
    if (d.cpml && !march_axes(d.ef, d.n, a.grid.axis)) return false;
    a.grid.ny = d.n[1]; a.grid.nz = d.n[2]; a.grid.nyz = (int)nyz;
    a.grid.coef = d.ef.coef;
    const int by = d.box_hi[1] - d.box_lo[1], bz = d.box_hi[2] - d.box_lo[2];
    a.box.nx = d.box_hi[0] - d.box_lo[0];
    a.box.nz = bz;
    a.box.nyz = by * bz;
    a.box.columns = (a.box.nyz + 63) / 64;
    a.box.span = (long long)a.box.columns * a.box.nx < kSpanItems ? 1 : 2;
    a.box.by_nz = make_divider((unsigned)bz);
    a.box.by_columns = make_divider((unsigned)a.box.columns);
    const long long items = (long long)a.box.columns * ((a.box.nx + a.box.span - 1) / a.box.span);
    if (items > kLaunchItems) return false;
    a.box.xcd = (int)xcd_run((items + 3) / 4);
    a.nx = d.n[0];
    for (int k = 0; k < 3; ++k) a.lo[k] = d.box_lo[k];
    a.H = d.H; a.psi = d.ef.psi_in;
    a.periodic = d.periodic;
    a.record = d.record; a.modulus = d.modulus;
    a.counter = d.counter;
    return true;
}

template <typename real>
void launch_record(const Record<real>& a, unsigned blocks, hipStream_t s) {
    RecordMarch<real> m;
    if (make_record_march(a, &m)) {
        const long long items = (long long)m.box.columns * ((m.box.nx + m.box.span - 1) / m.box.span);
        hipLaunchKernelGGL(record_march_kernel<real>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s, m);
    } else {
        hipLaunchKernelGGL(record_kernel<real>, dim3(blocks), dim3(256), 0, s, a);
    }
}

// The x march of one family: true when the grid allows it (two cells or more along x and y, the family's memory,
// its coefficients and a plane's fields each below 4 GiB).
template <typename real>
bool make_march(const Adjoint<real>& d, const Family<real>& f, AdjointMarch<real>* out) {
    AdjointMarch<real>& a = *out;
    std::memset(&a, 0, sizeof a);
    const long long nyz = (long long)d.n[1] * d.n[2];
    if (d.n[0] < 2 || d.n[1] < 2 || nyz * 3 * (long long)sizeof(real) > 0xffffffffLL) return false;
    if (!march_axes(f, d.n, a.axis)) return false;
    a.nx = d.n[0]; a.ny = d.n[1]; a.nz = d.n[2]; a.nyz = (int)nyz;
    a.columns = (int)((nyz + 63) / 64);
    a.span = (long long)a.columns * a.nx < kSpanItems ? 1 : 2;
    a.by_nz = make_divider((unsigned)a.nz);
    a.by_columns = make_divider((unsigned)a.columns);
    const long long items = (long long)a.columns * ((a.nx + a.span - 1) / a.span);
    if (items > kLaunchItems) return false;
    a.xcd = (int)xcd_run((items + 3) / 4);
    a.e_bar = d.e_bar; a.h_bar = d.h_bar; a.inv_eps = d.inv_eps; a.inv_mu = d.inv_mu;
    a.psi_in = f.psi_in; a.psi_out = f.psi_out; a.coef = f.coef;
    a.S = d.S;
    a.periodic = d.periodic; a.pec = d.pec;
    for (int k = 0; k < 3; ++k) {
        a.pec_factor[k] = d.pec_factor[k];
        a.box_lo[k] = d.box_lo[k];
        a.box_hi[k] = d.box_hi[k];
    }
    a.record = d.record; a.modulus = d.modulus;
    a.gradient = d.gradient; a.gradient_stride = d.gradient_stride;
    a.counter = d.counter;
    return true;
}

template <typename real, int INV, bool FLAT>
void launch_march(const AdjointMarch<real>& h, const AdjointMarch<real>& e, hipStream_t s) {
    const dim3 grid((unsigned)(((long long)h.columns * ((h.nx + h.span - 1) / h.span) + 3) / 4)), block(256);
    hipLaunchKernelGGL((h_transpose_march_kernel<real, INV, FLAT>), grid, block, 0, s, h);
    hipLaunchKernelGGL((e_transpose_march_kernel<real, INV, FLAT>), grid, block, 0, s, e);
}

int check_box(const int32_t lo[3], const int32_t hi[3], const int n[3]) {
    for (int ax = 0; ax < 3; ++ax)
        if (lo[ax] < 0 || hi[ax] <= lo[ax] || hi[ax] > n[ax]) return tfdtd_fail(TFDTD_EINVAL, "adjoint: design box outside the grid");
    return TFDTD_OK;
}

template <typename real>
int make_adjoint(const tfdtd_adjoint* d, Adjoint<real>* a) {
    std::memset(a, 0, sizeof *a);
    const int n[3] = {d->nx, d->ny, d->nz};
    if (n[0] < 1 || n[1] < 1 || n[2] < 1) return tfdtd_fail(TFDTD_EINVAL, "adjoint: grid dimensions must be positive");
    if (!d->e_bar || !d->h_bar || !d->inverse_permittivity || !d->inverse_permeability || !d->counter)
        return tfdtd_fail(TFDTD_EINVAL, "adjoint: null field, material or counter pointer");
    if (d->eps_stride != 1 && d->eps_stride != 3) return tfdtd_fail(TFDTD_EINVAL, "adjoint: eps_stride must be 1 or 3");
    for (int ax = 0; ax < 3; ++ax) a->n[ax] = n[ax];
    a->e_bar = static_cast<real*>(d->e_bar);
    a->h_bar = static_cast<real*>(d->h_bar);
    a->inv_eps = static_cast<const real*>(d->inverse_permittivity);
    a->eps_stride = d->eps_stride;
    return TFDTD_OK;
}

}  // namespace

extern "C" int tfdtd_record_curl(const tfdtd_curl_record* d, void* stream) {
    if (!d || !d->H || !d->record || !d->counter || d->modulus < 1) return tfdtd_fail(TFDTD_EINVAL, "record: null pointer or modulus < 1");
    const int n[3] = {d->nx, d->ny, d->nz};
    if (n[0] < 1 || n[1] < 1 || n[2] < 1) return tfdtd_fail(TFDTD_EINVAL, "record: grid dimensions must be positive");
    int status = check_box(d->box_lo, d->box_hi, n);
    if (status) return status;
    const long long count = (long long)(d->box_hi[0] - d->box_lo[0]) * (d->box_hi[1] - d->box_lo[1]) * (d->box_hi[2] - d->box_lo[2]);
    const unsigned blocks = (unsigned)((count + 255) / 256);
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto fill = [&](auto* a) -> int {
        using real = std::remove_pointer_t<decltype(a->record)>;
        for (int ax = 0; ax < 3; ++ax) { a->n[ax] = n[ax]; a->box_lo[ax] = d->box_lo[ax]; a->box_hi[ax] = d->box_hi[ax]; }
        a->H = static_cast<const real*>(d->H);
        a->periodic = d->periodic_mask & 7;
        a->record = static_cast<real*>(d->record);
        a->modulus = d->modulus;
        a->counter = reinterpret_cast<const long long*>(d->counter);
        a->cpml = d->e.psi_in != nullptr;
        if (!a->cpml) {
            std::memset(&a->ef, 0, sizeof a->ef);
            return TFDTD_OK;
        }
        // The record reads psi_in only: in-place (split step) and double-buffered layouts both serve.
        return make_family(d->e, d->e.psi_in != d->e.psi_out, n, &a->ef);
    };
    if (d->dtype == TFDTD_F32) {
        Record<float> a;
        if ((status = fill(&a))) return status;
        launch_record(a, blocks, s);
    } else if (d->dtype == TFDTD_F64) {
        Record<double> a;
        if ((status = fill(&a))) return status;
        launch_record(a, blocks, s);
    } else {
        return tfdtd_fail(TFDTD_EINVAL, "record: dtype must be float32 or float64");
    }
    return tfdtd_check_launch("record_curl");
}

template <typename real>
static int launch_adjoint(const tfdtd_adjoint* d, hipStream_t s) {
    Adjoint<real> a;
    int status = make_adjoint(d, &a);
    if (status) return status;
    const int dims[3] = {d->nx, d->ny, d->nz};
    status = make_family(d->e, true, dims, &a.ef);
    if (!status) status = make_family(d->h, true, dims, &a.hf);
    if (status) return status;
    a.inv_mu = static_cast<const real*>(d->inverse_permeability);
    a.S = (real)d->courant;
    a.periodic = d->periodic_mask & 7;
    a.pec = d->pec_upper_mask & 7 & ~a.periodic;
    for (int ax = 0; ax < 3; ++ax) a.pec_factor[ax] = (real)d->pec_upper_factor[ax];
    a.nseed = d->nseed;
    if (d->nseed < 0 || (d->nseed > 0 && (!d->seed_targets || !d->seed_offsets || !d->seed_columns || !d->seeds || d->seed_width < 1)))
        return tfdtd_fail(TFDTD_EINVAL, "adjoint: malformed seed table");
    a.seed_targets = reinterpret_cast<const long long*>(d->seed_targets);
    a.seed_offsets = d->seed_offsets;
    a.seed_columns = d->seed_columns;
    a.seeds = static_cast<const real*>(d->seeds);
    a.seed_width = d->seed_width;
    a.seed_rows = d->seed_rows;
    if (d->record) {
        status = check_box(d->box_lo, d->box_hi, dims);
        if (status) return status;
        if (!d->gradient || d->record_modulus < 1 || (d->gradient_stride != 1 && d->gradient_stride != 3))
            return tfdtd_fail(TFDTD_EINVAL, "adjoint: a record needs a gradient buffer, a modulus >= 1 and gradient_stride 1 or 3");
        // A plain difference record serves only boxes that stay out of the E-family slabs.
        for (int ax = 0; ax < 3 && !d->record_cpml; ++ax)
            for (int f = 0; f < 2; ++f) {
                const Face& face = a.ef.face[ax][f];
                if (face.hi > face.lo && face.lo < d->box_hi[ax] && d->box_lo[ax] < face.hi)
                    return tfdtd_fail(TFDTD_EINVAL, "adjoint: the design box meets the CPML slab of axis %d and the "
                                                    "record has no CPML terms", ax);
            }
        for (int ax = 0; ax < 3; ++ax) { a.box_lo[ax] = d->box_lo[ax]; a.box_hi[ax] = d->box_hi[ax]; }
        a.record = static_cast<const real*>(d->record);
        a.modulus = d->record_modulus;
        a.gradient = d->gradient;
        a.gradient_stride = d->gradient_stride;
    } else {
        for (int ax = 0; ax < 3; ++ax) { a.box_lo[ax] = 0; a.box_hi[ax] = 0; }   // no gradient cells
        a.modulus = 1;
    }
    a.counter = reinterpret_cast<long long*>(d->counter);
    const unsigned long long tiles = (unsigned long long)dims[0] * ((dims[1] + kTileY - 1) / kTileY) *
                                     ((dims[2] + kTileZ - 1) / kTileZ);
    if (tiles > 0x7fffffffULL) return tfdtd_fail(TFDTD_EINVAL, "adjoint: grid too large for one launch");
    const unsigned blocks = transpose_blocks(dims);
    if (a.nseed > 0) {
        hipLaunchKernelGGL(seed_kernel<real>, dim3((unsigned)((a.nseed + 255) / 256)), dim3(256), 0, s, a);
        status = tfdtd_check_launch("adjoint seeds");
        if (status) return status;
    }
    AdjointMarch<real> mh, me;
    if (make_march(a, a.hf, &mh) && make_march(a, a.ef, &me)) {
        if (a.n[2] == 1) {
            if (a.eps_stride == 3) launch_march<real, 3, true>(mh, me, s);
            else launch_march<real, 1, true>(mh, me, s);
        } else {
            if (a.eps_stride == 3) launch_march<real, 3, false>(mh, me, s);
            else launch_march<real, 1, false>(mh, me, s);
        }
        return tfdtd_check_launch("adjoint transposes");
    }
    hipLaunchKernelGGL(h_transpose_kernel<real>, dim3(blocks), dim3(256), 0, s, a);
    status = tfdtd_check_launch("adjoint h_transpose");
    if (status) return status;
    hipLaunchKernelGGL(e_transpose_kernel<real>, dim3(blocks), dim3(256), 0, s, a);
    return tfdtd_check_launch("adjoint e_transpose");
}

extern "C" int tfdtd_adjoint_step(const tfdtd_adjoint* d, void* stream) {
    if (!d) return tfdtd_fail(TFDTD_EINVAL, "null adjoint descriptor");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (d->dtype == TFDTD_F32) return launch_adjoint<float>(d, s);
    if (d->dtype == TFDTD_F64) return launch_adjoint<double>(d, s);
    return tfdtd_fail(TFDTD_EINVAL, "adjoint: dtype must be float32 or float64");
}
