// BF16 implicit-GEMM 3D convolution for gfx950 MFMA, FP32 accumulation: forward with fused
// bias + GELU, input gradient (dgrad) and weight gradient (wgrad).  No reference
// counterpart: the reference has no neural surrogate (its design loops are
// torchfdtd/design.py and torchfdtd/design_problem.py); these kernels serve the learned
// screening model of the inverse-design loop.
//
// Layouts: activations channels-last [n][d][h][w][c] (bf16); forward weights [co][kp]
// with k = tap*ci + c, tap = (kd*ks + kh)*ks + kw, zero-padded to kp (a multiple of 32);
// dgrad weights [ci][ks^3*co] (k = tap*co + c); wgrad reads dY transposed [co][m].
//
// Layers whose channels are multiples of 8 (and one-channel inputs) take gather_gemm_kernel,
// narrow_forward_kernel and weight_grad_kernel, further down.  Every other layer takes gemm_kernel: one
// workgroup (4 waves) computes a 64 x 64 tile of C = A B over K in steps of 32: the A tile (64
// rows x 32 k) and B tile (64 columns x 32 k) are gathered from global memory (the implicit
// im2col) into LDS with k fastest, and each wave multiplies its 32 x 32 quarter with 2 x 2
// v_mfma_f32_16x16x32_bf16.  blockIdx.z splits K for the weight gradient, whose reduction
// runs over every output position.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/tfdtd.h"
#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f4;
typedef unsigned short bf16_bits;
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));

constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;   // LDS rows padded by 16 bytes

// Round to nearest even, infinities and NaN kept, as torch's float -> bfloat16 conversion: one instruction on
// gfx950 (two values at a time where the caller converts neighbours).
__device__ __forceinline__ bf16_bits float_to_bf16(float f) { return __builtin_bit_cast(bf16_bits, (__bf16)f); }

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

struct Conv {
    int n, di, hi, wi, ci;      // input
    int dout, hout, wout, co;   // output
    int ks, stride, pad;
    int kp;                     // forward K (ks^3 * ci) padded to a multiple of 32
};

struct Gemm {
    int op;                     // 0 forward, 1 dgrad, 2 wgrad
    Conv c;
    int M, N, K;                // C is M x N, reduction K (padded)
    int k_per_split;
    const bf16_bits* a;         // forward: x; dgrad: dY [m_out][co]; wgrad: dY^T [co][m_out]
    const bf16_bits* b;         // forward: W [co][kp]; dgrad: Wd [ci][ks^3 co]; wgrad: x
    const float* bias;          // forward only (may be null)
    int activation;             // forward: 1 GELU, 0 identity
    float* out;                 // forward: pre-activation [M][N]; dgrad: dX [M][N]; wgrad: partial [split][M][N]
    bf16_bits* act;             // forward: bf16 activation [M][N]
};

// Input position of output position m and tap (kd, kh, kw); false when it lies in the padding.
__device__ __forceinline__ bool input_of(const Conv& c, long long m, int tap, long long* cell) {
    const int wo = (int)(m % c.wout);
    const int ho = (int)((m / c.wout) % c.hout);
    const int dd = (int)((m / ((long long)c.wout * c.hout)) % c.dout);
    const long long nb = m / ((long long)c.wout * c.hout * c.dout);
    const int kw = tap % c.ks, kh = (tap / c.ks) % c.ks, kd = tap / (c.ks * c.ks);
    const int z = dd * c.stride - c.pad + kd, y = ho * c.stride - c.pad + kh, x = wo * c.stride - c.pad + kw;
    if (z < 0 || z >= c.di || y < 0 || y >= c.hi || x < 0 || x >= c.wi) return false;
    *cell = ((nb * c.di + z) * c.hi + y) * c.wi + x;
    return true;
}

// Output position that input position m_in reaches through tap; false when none.
__device__ __forceinline__ bool output_of(const Conv& c, long long m, int tap, long long* cell) {
    const int x = (int)(m % c.wi);
    const int y = (int)((m / c.wi) % c.hi);
    const int z = (int)((m / ((long long)c.wi * c.hi)) % c.di);
    const long long nb = m / ((long long)c.wi * c.hi * c.di);
    const int kw = tap % c.ks, kh = (tap / c.ks) % c.ks, kd = tap / (c.ks * c.ks);
    const int tz = z + c.pad - kd, ty = y + c.pad - kh, tx = x + c.pad - kw;
    if (tz < 0 || ty < 0 || tx < 0 || tz % c.stride || ty % c.stride || tx % c.stride) return false;
    const int dd = tz / c.stride, ho = ty / c.stride, wo = tx / c.stride;
    if (dd >= c.dout || ho >= c.hout || wo >= c.wout) return false;
    *cell = ((nb * c.dout + dd) * c.hout + ho) * c.wout + wo;
    return true;
}

__device__ __forceinline__ void load8(bf16_bits* dst, const bf16_bits* src) {
    *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
}

__device__ __forceinline__ void zero8(bf16_bits* dst) { *reinterpret_cast<uint4*>(dst) = make_uint4(0, 0, 0, 0); }

// Element (m, k) of the forward im2col matrix of the input x.
__device__ __forceinline__ bf16_bits im2col(const Conv& c, const bf16_bits* x, long long m, int k) {
    if (k >= c.ks * c.ks * c.ks * c.ci) return 0;
    long long cell;
    if (!input_of(c, m, k / c.ci, &cell)) return 0;
    return x[cell * c.ci + k % c.ci];
}

// A tile: sA[row][k] for rows row0.., k0..k0+31.  Thread t fills row t/4, k chunk (t%4)*8.
__device__ __forceinline__ void fill_a(const Gemm& g, bf16_bits* sA, long long row0, int k0) {
    const int t = threadIdx.x, r = t >> 2, q = (t & 3) * 8;
    bf16_bits* dst = sA + r * LDK + q;
    const long long row = row0 + r;
    const int k = k0 + q;
    const Conv& c = g.c;
    if (row >= g.M || k >= g.K) { zero8(dst); return; }
    if (g.op == 0) {
        if (c.ci % 8 == 0) {
            long long cell;
            if (k < c.ks * c.ks * c.ks * c.ci && input_of(c, row, k / c.ci, &cell)) load8(dst, g.a + cell * c.ci + k % c.ci);
            else zero8(dst);
        } else {
            for (int j = 0; j < 8; ++j) dst[j] = im2col(c, g.a, row, k + j);
        }
    } else if (g.op == 1) {
        // dY gathered at the output position this input position reaches by tap k / co.
        long long cell;
        if (output_of(c, row, k / c.co, &cell)) load8(dst, g.a + cell * c.co + k % c.co);
        else zero8(dst);
    } else {
        // dY^T [co][m]: 8 consecutive output positions of channel `row`.
        const long long m_total = (long long)c.n * c.dout * c.hout * c.wout;
        if (k + 8 <= m_total && (m_total % 8) == 0) load8(dst, g.a + row * m_total + k);
        else for (int j = 0; j < 8; ++j) dst[j] = k + j < m_total ? g.a[row * m_total + k + j] : 0;
    }
}

// B tile: sB[col][k] for columns col0.., k0..k0+31.
__device__ __forceinline__ void fill_b(const Gemm& g, bf16_bits* sB, int col0, int k0) {
    const int t = threadIdx.x;
    const Conv& c = g.c;
    if (g.op != 2) {
        const int r = t >> 2, q = (t & 3) * 8;
        bf16_bits* dst = sB + r * LDK + q;
        const int col = col0 + r, k = k0 + q;
        if (col >= g.N || k >= g.K) { zero8(dst); return; }
        load8(dst, g.b + (long long)col * g.K + k);          // weights padded to K columns
    } else {
        // Weight gradient: B(m, k) = im2col(m, k) for 32 reductions m and 64 columns k.  Thread t
        // takes reduction row t/8 and columns (t%8)*8 .. +7, loading along k and storing transposed.
        const int mr = t >> 3, q = (t & 7) * 8;
        const long long m = (long long)k0 + mr;
        const long long m_total = (long long)c.n * c.dout * c.hout * c.wout;
        const int kk = col0 + q;
        const int kmax = c.ks * c.ks * c.ks * c.ci;
        bf16_bits v[8];
        if (m >= m_total) {
            for (int j = 0; j < 8; ++j) v[j] = 0;
        } else if (c.ci % 8 == 0 && kk + 8 <= kmax) {
            long long cell;
            if (input_of(c, m, kk / c.ci, &cell)) *reinterpret_cast<uint4*>(v) = *reinterpret_cast<const uint4*>(g.b + cell * c.ci + kk % c.ci);
            else for (int j = 0; j < 8; ++j) v[j] = 0;
        } else {
            for (int j = 0; j < 8; ++j) v[j] = im2col(c, g.b, m, kk + j);
        }
        for (int j = 0; j < 8; ++j) sB[(q + j) * LDK + mr] = v[j];
    }
}

__global__ __launch_bounds__(256) void gemm_kernel(const Gemm g) {
    __shared__ __attribute__((aligned(16))) bf16_bits sA[BM * LDK];
    __shared__ __attribute__((aligned(16))) bf16_bits sB[BN * LDK];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long row0 = (long long)blockIdx.x * BM;
    const int col0 = blockIdx.y * BN;
    const int kb = blockIdx.z * g.k_per_split, ke = min(g.K, kb + g.k_per_split);
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    f4 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = kb; k0 < ke; k0 += BK) {
        __syncthreads();
        fill_a(g, sA, row0, k0);
        fill_b(g, sB, col0, k0);
        __syncthreads();
        // Lane l supplies row (l % 16) and k (l / 16) * 8 .. +7 of each 16 x 32 operand.
        const int r = lane & 15, kq = (lane >> 4) * 8;
        bf16x8 a[2], b[2];
        for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(sA + (wr + 16 * i + r) * LDK + kq);
        for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const bf16x8*>(sB + (wc + 16 * j + r) * LDK + kq);
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    // D layout: lane l holds rows (l / 16) * 4 + e, column l % 16 of each 16 x 16 tile.
    const int cn = lane & 15, rq = (lane >> 4) * 4;
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int e = 0; e < 4; ++e) {
                const long long row = row0 + wr + 16 * i + rq + e;
                const int col = col0 + wc + 16 * j + cn;
                if (row >= g.M || col >= g.N) continue;
                float v = acc[i][j][e];
                if (g.op == 2) {
                    g.out[((long long)blockIdx.z * g.M + row) * g.N + col] = v;
                } else if (g.op == 0) {
                    if (g.bias) v += g.bias[col];
                    g.out[row * g.N + col] = v;
                    g.act[row * g.N + col] = float_to_bf16(g.activation ? gelu(v) : v);
                } else {
                    g.out[row * g.N + col] = v;
                }
            }
}

// Sum of the K splits of the weight gradient: a workgroup takes 64 values, each of its four wavefronts every
// fourth split.
__global__ __launch_bounds__(256) void split_sum_kernel(const float* partial, int splits, long long count, float* out) {
    __shared__ float sums[3][64];
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
    for (long long first = (long long)blockIdx.x * 64; first < count; first += 64LL * gridDim.x) {
        const long long i = first + lane;
        float s = 0.f;
        if (i < count)
#pragma unroll 4
            for (int z = part; z < splits; z += 4) s += partial[z * count + i];
        if (part) sums[part - 1][lane] = s;
        __syncthreads();
        if (part == 0 && i < count) out[i] = s + sums[0][lane] + sums[1][lane] + sums[2][lane];
        __syncthreads();
    }
}

// A launch holds fewer than 2^32 threads: more values than 2^29 are summed in several turns.
unsigned split_sum_blocks(long long count) { return (unsigned)std::min<long long>((count + 63) / 64, 1 << 23); }

// dPre = dY * GELU'(pre) (or dY), written in FP32 and BF16.
__global__ __launch_bounds__(256) void gelu_backward_kernel(const float* dy, const float* pre, long long count, int activation,
                                                           float* dpre, bf16_bits* dpre16) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const float v = activation ? dy[i] * gelu_grad(pre[i]) : dy[i];
    dpre[i] = v;
    dpre16[i] = float_to_bf16(v);
}

// ---------------------------------------------------------------- gathered GEMM
//
// The forward convolution and the input gradient are one contraction: C[row][col] is the sum over taps and
// source channels of source(row's position under the tap)[c] * weight[col][tap * channels + c].  Rows are
// output positions (forward) or, for the input gradient, the input positions of one parity class of a
// strided layer: rows of one class see the same taps, so no tap is multiplied that the stride rules out.
//
// A workgroup (4 waves, 8 at 128 x 128) computes BM rows x BN columns over K in stages of 64: source rows and weight rows
// go from global memory straight into LDS (16 bytes a lane, no registers), `Depth` - 1 stages ahead of the
// stage being multiplied.  A lane keeps its rows' addresses and a bit per tap (inside or padding) for the
// whole loop, so a stage costs it one offset and a select; padding reads a chunk of zeros.  A row's 16-byte
// chunks lie in LDS at chunk ^ ((row >> 1) & 7), which spreads the 16 rows of one operand read over all
// banks.  Every product enters its accumulator in the order of gemm_kernel (the same MFMA over ascending K),
// so results are equal bit for bit; a tap that is padding for every row of the workgroup is skipped when the
// weights are finite (it would add zeros).
//
// 64x32x32x16 positions, 64 -> 128 channels, 3x3x3 (0.46 TFLOP): forward 2.72 -> 0.88 ms (530 TFLOP/s), input
// gradient 3.5 -> 0.76 ms (610).  gemm_kernel gathered through registers with a division chain per chunk and
// two barriers per 32 of K.  The forward layer's matrix instructions take a quarter of its cycles and its epilogue
// (GELU, two FP32 outputs) a fifth; the rest is the latency of the stages, which is why eight waves per tile
// beat four (0.95 ms with the same stages) and why fewer, larger stages do not help (256 x 128 tiles, two or three
// stages deep: 0.99 ms; 128 x 128 three deep, one workgroup per CU: 1.5 ms).
typedef __attribute__((address_space(3))) void lds_void;

__device__ const uint4 kZeroChunk = {0u, 0u, 0u, 0u};

// 16 bytes of global memory per lane into LDS at `to` + 16 * lane.
__device__ __forceinline__ void chunk_to_lds(const void* from, bf16_bits* to) {
    __builtin_amdgcn_global_load_lds(global(const_cast<void*>(from)), (lds_void*)to, 16, 0, 0);
}

struct GatherGemm {
    Conv c;
    int dgrad;                  // 0 forward, 1 input gradient
    int wide;                   // 1: the source is FP32, rounded to bf16 as it is read (narrow forward)
    int rows_max;               // rows of the largest class
    unsigned run;               // row tiles an XCD takes in a row
    int N, channels, ldw;       // columns, source channels, weight row length
    const bf16_bits* source;    // forward: x; input gradient: dY
    const bf16_bits* weight;    // [N][ldw]
    const int* nonfinite;       // per part of the weights: 1 where a value is not finite (null: no tap is skipped)
    int parts;
    const float* bias;
    int activation;
    float* pre;                 // forward: pre-activation (may be null); input gradient: dX
    float* y;                   // forward: FP32 value of the activation (may be null)
    bf16_bits* act;             // forward: activation (may be null)
};

// The bias of four consecutive columns, read once per workgroup tile: behind the outputs' stores each row would
// wait for it again.
__device__ __forceinline__ f4 column_bias(const GatherGemm& g, int col) {
    f4 b = f4{0.f, 0.f, 0.f, 0.f};
    if (!g.dgrad && g.bias)
        for (int e = 0; e < 4; ++e)
            if (col + e < g.N) b[e] = g.bias[col + e];
    return b;
}

// Four consecutive columns of a row to the outputs: bias, pre-activation, activation; the input gradient as it is.
__device__ __forceinline__ void finish_columns(const GatherGemm& g, long long cell, int col, f4 v, f4 bias) {
    if (col + 3 < g.N && g.N % 4 == 0) {
        const long long o = cell * g.N + col;
        if (g.dgrad) {
            *reinterpret_cast<f4*>(g.pre + o) = v;
            return;
        }
        if (g.bias)
            for (int e = 0; e < 4; ++e) v[e] += bias[e];
        if (g.pre) *reinterpret_cast<f4*>(g.pre + o) = v;
        bf16_bits b[4];
        for (int e = 0; e < 4; ++e) b[e] = float_to_bf16(g.activation ? gelu(v[e]) : v[e]);
        if (g.act) *reinterpret_cast<uint2*>(g.act + o) = make_uint2(b[0] | (unsigned)b[1] << 16, b[2] | (unsigned)b[3] << 16);
        if (g.y) {
            f4 f;
            for (int e = 0; e < 4; ++e) f[e] = __uint_as_float((unsigned)b[e] << 16);
            *reinterpret_cast<f4*>(g.y + o) = f;
        }
        return;
    }
    for (int e = 0; e < 4; ++e) {
        if (col + e >= g.N) continue;
        const long long o = cell * g.N + col + e;
        float f = v[e];
        if (!g.dgrad && g.bias) f += bias[e];
        if (g.pre) g.pre[o] = f;
        if (g.dgrad) continue;
        const bf16_bits b = float_to_bf16(g.activation ? gelu(f) : f);
        if (g.act) g.act[o] = b;
        if (g.y) g.y[o] = __uint_as_float((unsigned)b << 16);
    }
}

// One axis of the rows: its length, where tap k of row q lies (q * mul + at(k)), and where row q itself lies.
struct RowAxis {
    int rows, source, mul, first, shift, sign, out_mul;
    __device__ __forceinline__ int at(int k) const { return (first + sign * k) >> shift; }
    __device__ __forceinline__ bool meets(int k) const { return ((first + sign * k) & ((1 << shift) - 1)) == 0; }
};

__device__ __forceinline__ RowAxis row_axis(const GatherGemm& g, int in, int out, int parity, int* begin) {
    RowAxis a;
    if (!g.dgrad) {
        *begin = 0;
        a = RowAxis{out, in, g.c.stride, -g.c.pad, 0, 1, 1};
    } else if (g.c.stride == 1) {
        *begin = 0;
        a = RowAxis{in, out, 1, g.c.pad, 0, -1, 1};
    } else {
        *begin = (parity + g.c.pad) & 1;      // first position z with (z + pad) % 2 == parity
        a = RowAxis{(in - *begin + 1) >> 1, out, 1, *begin + g.c.pad, 1, -1, 2};
    }
    return a;
}

// K in pieces of 32: (tap, channel) of each, taps in ascending order from a mask.
struct Pieces {
    unsigned left;
    int tap, c;
    bool more;
    __device__ __forceinline__ void start(unsigned mask) {
        more = mask != 0;
        tap = more ? __builtin_ctz(mask) : 0;
        left = mask & (mask - 1u);
        c = 0;
    }
    __device__ __forceinline__ void next(int channels) {
        c += 32;
        if (c < channels) return;
        c = 0;
        more = left != 0;
        if (more) {
            tap = __builtin_ctz(left);
            left &= left - 1u;
        }
    }
};

// `Whole`: the channels are a multiple of 32, so a piece of 32 has one tap; otherwise (a multiple of 8) each
// 16-byte chunk finds its own.
template <int BM, int BN, int WM, int WN, int Depth, bool Whole>
__global__ __launch_bounds__(BM / WM * (BN / WN) * 64) void gather_gemm_kernel(const GatherGemm g) {
    constexpr int Waves = BM / WM * (BN / WN);
    constexpr int XI = BM / (8 * Waves), WI = BN / (8 * Waves);         // staging instructions per wave
    static_assert(XI * 8 * Waves == BM && WI * 8 * Waves == BN, "whole staging instructions");
    constexpr int RT = WM / 16, CT = WN / 16;          // 16-row and 16-column tiles per wave
    constexpr int Stage = (BM + BN) * 64;
    __shared__ __attribute__((aligned(16))) bf16_bits s0[Stage];
    __shared__ __attribute__((aligned(16))) bf16_bits s1[Stage];
    __shared__ __attribute__((aligned(16))) bf16_bits s2[Depth > 2 ? Stage : 8];
    __shared__ unsigned s_mask, s_bad;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Conv& c = g.c;
    const int ks = c.ks, taps = ks * ks * ks, C = g.channels;
    const int cls = blockIdx.z;
    int begin[3];
    const RowAxis ax[3] = {row_axis(g, c.di, c.dout, cls & 1, &begin[0]), row_axis(g, c.hi, c.hout, (cls >> 1) & 1, &begin[1]),
                           row_axis(g, c.wi, c.wout, cls >> 2, &begin[2])};
    const int rows = c.n * ax[0].rows * ax[1].rows * ax[2].rows;
    const int row0 = (int)xcd_block(blockIdx.x, gridDim.x, g.run) * BM, col0 = blockIdx.y * BN;
    if (row0 >= rows) return;                          // a smaller class: the whole workgroup leaves
    if (tid == 0) { s_mask = 0u; s_bad = 0u; }
    __syncthreads();
    // Rows of this lane: position under tap offset 0 and a bit per tap that lies inside the source.
    const bf16_bits* row_at[XI];
    unsigned row_taps[XI], any = 0u;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int row = row0 + (wave * XI + i) * 8 + (lane >> 3);
        unsigned mask = 0u;
        long long cell = 0;
        if (row < rows) {
            int q[3], t = row / ax[2].rows;
            q[2] = row - t * ax[2].rows;
            const int u = t / ax[1].rows;
            q[1] = t - u * ax[1].rows;
            const int nb = u / ax[0].rows;
            q[0] = u - nb * ax[0].rows;
            unsigned in[3];
            for (int a = 0; a < 3; ++a) {
                in[a] = 0u;
                for (int k = 0; k < ks; ++k) {
                    const int p = q[a] * ax[a].mul + ax[a].at(k);
                    if (ax[a].meets(k) && p >= 0 && p < ax[a].source) in[a] |= 1u << k;
                }
            }
            for (int kd = 0; kd < ks; ++kd)
                for (int kh = 0; kh < ks; ++kh)
                    if ((in[0] >> kd & 1u) && (in[1] >> kh & 1u)) mask |= in[2] << ((kd * ks + kh) * ks);
            cell = (((long long)nb * ax[0].source + q[0] * ax[0].mul) * ax[1].source + q[1] * ax[1].mul) * ax[2].source + q[2] * ax[2].mul;
        }
        row_at[i] = g.source + cell * C;
        row_taps[i] = mask;
        any |= mask;
    }
    unsigned todo = taps == 32 ? ~0u : (1u << taps) - 1u;
    if (Whole && g.nonfinite) {
        int bad = 0;
        for (int i = tid; i < g.parts; i += 64 * Waves) bad |= g.nonfinite[i];
        atomicOr(&s_mask, any);
        if (bad) s_bad = 1u;
        __syncthreads();
        if (!s_bad) todo = s_mask;
        todo = (unsigned)__builtin_amdgcn_readfirstlane((int)todo);
    }
    // Elements from a row's position under tap offset 0 to its position under a tap (one sample is below 2^31).
    auto tap_offset = [&](int tap) -> int {
        const int kd = tap * 57 >> 9, r = tap - 9 * kd, kh = r * 11 >> 5, kw = r - 3 * kh;     // tap / 9, / 3, % 3 (one tap: 0)
        return ((ax[0].at(kd) * ax[1].source + ax[1].at(kh)) * ax[2].source + ax[2].at(kw)) * C;
    };
    const int pieces = Whole ? __popc(todo) * (C / 32) : (taps * C + 31) / 32;
    const int stages = (pieces + 1) / 2;
    // A lane's two kinds of chunk (even and odd i): position (lane & 7) of its row holds chunk (lane & 7) ^ swizzle.
    const int odd = wave * XI & 1;
    const int chunk_of[2] = {(lane & 7) ^ (((lane >> 4) + 4 * odd) & 7), (lane & 7) ^ (((lane >> 4) + 4 * (odd ^ 1)) & 7)};
    Pieces at;
    at.start(todo);
    int own_tap[2] = {0, 0}, own_c[2] = {0, 0};        // !Whole: the chunk's own tap and channel
    if (!Whole)
        for (int v = 0; v < 2; ++v) {
            own_tap[v] = chunk_of[v] * 8 / C;
            own_c[v] = chunk_of[v] * 8 % C;
        }
    int staged = 0;
    const bf16_bits* const zero = reinterpret_cast<const bf16_bits*>(&kZeroChunk);
    // Whole: a lane's chunk places of its rows and weight rows are fixed, so a stage adds one offset per half to
    // pointers formed here.  Weight rows past the last repeat it and K past the last piece repeats the first:
    // neither is used.
    const bf16_bits* weight_at[WI];
    if (Whole) {
#pragma unroll
        for (int i = 0; i < XI; ++i) row_at[i] += (chunk_of[i & 1] & 3) * 8;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int r = (wave * WI + i) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
            weight_at[i] = g.weight + (long long)min(col0 + r, g.N - 1) * g.ldw + (chunk & 3) * 8;
        }
    }
    const int odd_weights = wave * WI & 1;
    const bool upper[2] = {(chunk_of[0] >> 2) != 0, (chunk_of[1] >> 2) != 0};       // which half of a stage, by parity
    const bool upper_weights[2] = {(((lane & 7) ^ (((lane >> 4) + 4 * odd_weights) & 7)) >> 2) != 0,
                                   (((lane & 7) ^ (((lane >> 4) + 4 * (odd_weights ^ 1)) & 7)) >> 2) != 0};
    auto stage = [&](bf16_bits* into) {
        bf16_bits* const weights = into + BM * 64;
        if (Whole) {
            int offset[2], k[2];
            unsigned bit[2];
            for (int h = 0; h < 2; ++h) {
                offset[h] = at.more ? tap_offset(at.tap) + at.c : 0;
                bit[h] = at.more ? 1u << at.tap : 0u;
                k[h] = at.more ? at.tap * C + at.c : 0;
                at.next(C);
            }
            int mine[2], ours[2];
            unsigned need[2];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                mine[v] = upper[v] ? offset[1] : offset[0];
                need[v] = upper[v] ? bit[1] : bit[0];
                ours[v] = upper_weights[v] ? k[1] : k[0];
            }
#pragma unroll
            for (int i = 0; i < XI; ++i)
                chunk_to_lds(row_taps[i] & need[i & 1] ? row_at[i] + mine[i & 1] : zero, into + (wave * XI + i) * 512);
#pragma unroll
            for (int i = 0; i < WI; ++i) chunk_to_lds(weight_at[i] + ours[i & 1], weights + (wave * WI + i) * 512);
            ++staged;
            return;
        }
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const bf16_bits* from = zero;
            if (own_tap[i & 1] < taps && (row_taps[i] >> own_tap[i & 1] & 1u))
                from = row_at[i] + tap_offset(own_tap[i & 1]) + own_c[i & 1];
            chunk_to_lds(from, into + (wave * XI + i) * 512);
        }
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int r = (wave * WI + i) * 8 + (lane >> 3);
            const int chunk = (lane & 7) ^ ((r >> 1) & 7), kk = staged * 64 + chunk * 8;
            const bf16_bits* from = zero;
            if (col0 + r < g.N && kk < g.ldw) from = g.weight + (long long)(col0 + r) * g.ldw + kk;
            chunk_to_lds(from, weights + (wave * WI + i) * 512);
        }
        ++staged;
        if (!Whole)
            for (int v = 0; v < 2; ++v) {
                own_c[v] += 64;
                while (own_c[v] >= C) { own_c[v] -= C; ++own_tap[v]; }
            }
    };
    const int wm = wave / (BN / WN) * WM, wn = wave % (BN / WN) * WN;
    f4 acc[CT][RT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, fc = lane >> 4, fs = (fr >> 1) & 7;   // operand row, chunk and swizzle of a lane
    auto multiply = [&](const bf16_bits* from, int number) {
        const bf16_bits* const weights = from + BM * 64;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 1 && 2 * number + 1 >= pieces) break;
            const int place = ((4 * h + fc) ^ fs) * 8;
            bf16x8 x[RT], w[CT];
#pragma unroll
            for (int j = 0; j < RT; ++j) x[j] = *reinterpret_cast<const bf16x8*>(from + (wm + 16 * j + fr) * 64 + place);
#pragma unroll
            for (int i = 0; i < CT; ++i) w[i] = *reinterpret_cast<const bf16x8*>(weights + (wn + 16 * i + fr) * 64 + place);
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int j = 0; j < RT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[j], acc[i][j], 0, 0, 0);
        }
    };
    // The barrier after a stage's loads have landed (all but those of later stages) also ends the reads of the
    // buffer that the next loads overwrite: both are waited for, as a raw barrier orders neither.
    constexpr int PerStage = XI + WI;
    static_assert(PerStage <= 15, "vmcnt of one stage in the low bits of the wait");
    auto arrive = [&](bool later) {
        asm volatile("" ::: "memory");
        if (Depth > 2 && later) __builtin_amdgcn_s_waitcnt(0x0070 | PerStage);      // vmcnt(PerStage) lgkmcnt(0)
        else __builtin_amdgcn_s_waitcnt(0x0070);                                    // vmcnt(0) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (stages > 0) stage(s0);
    if (Depth > 2 && stages > 1) stage(s1);
    for (int s = 0; s < stages;) {
        arrive(Depth > 2 && s + 1 < stages);
        if (Depth == 2) { if (s + 1 < stages) stage(s1); }
        else if (s + 2 < stages) stage(s2);
        multiply(s0, s);
        if (++s >= stages) break;
        arrive(Depth > 2 && s + 1 < stages);
        if (Depth == 2) { if (s + 1 < stages) stage(s0); }
        else if (s + 2 < stages) stage(s0);
        multiply(s1, s);
        if (++s >= stages) break;
        if (Depth > 2) {
            arrive(s + 1 < stages);
            if (s + 2 < stages) stage(s1);
            multiply(s2, s);
            ++s;
        }
    }
    // A lane holds four consecutive columns of one row per tile.
    f4 bias[CT];
#pragma unroll
    for (int i = 0; i < CT; ++i) bias[i] = column_bias(g, col0 + wn + 16 * i + fc * 4);
#pragma unroll
    for (int j = 0; j < RT; ++j) {
        const int row = row0 + wm + 16 * j + fr;
        if (row >= rows) continue;
        long long cell = row;
        if (g.dgrad) {
            int t = row / ax[2].rows;
            const int qx = row - t * ax[2].rows, u = t / ax[1].rows;
            const int qy = t - u * ax[1].rows, nb = u / ax[0].rows, qz = u - nb * ax[0].rows;
            cell = (((long long)nb * c.di + qz * ax[0].out_mul + begin[0]) * c.hi + qy * ax[1].out_mul + begin[1]) * c.wi +
                   qx * ax[2].out_mul + begin[2];
        }
#pragma unroll
        for (int i = 0; i < CT; ++i) {
            const int col = col0 + wn + 16 * i + fc * 4;
            finish_columns(g, cell, col, acc[i][j], bias[i]);
        }
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Row tiles that one XCD takes in a row, so that the taps' overlapping rows are read through one L2.
constexpr unsigned kRowRun = 64;

template <int BM, int BN, int WM, int WN, int Depth>
void launch_gather(GatherGemm g, int classes, hipStream_t stream) {
    g.run = kRowRun;
    // A single tap is never padding, so its flags are not read: 262,144 of them on 16384 x 16384, where every workgroup's
    // look-up was 360 of a linear layer's 496 us (8 rows).
    if (g.c.ks == 1) g.nonfinite = nullptr;
    const dim3 grid((g.rows_max + BM - 1) / BM, (g.N + BN - 1) / BN, classes), block(BM / WM * (BN / WN) * 64);
    if (g.channels % 32 == 0) hipLaunchKernelGGL((gather_gemm_kernel<BM, BN, WM, WN, Depth, true>), grid, block, 0, stream, g);
    else hipLaunchKernelGGL((gather_gemm_kernel<BM, BN, WM, WN, Depth, false>), grid, block, 0, stream, g);
}

// FP32 weights [co][taps][ci] of several layers to the bf16 operands of the forward convolution, [co][kp],
// and of the input gradient, [ci][taps * co] (transposed through LDS), and per tap and 32 x 32 channels
// whether a value is not finite.  One launch for a network's layers: each alone takes the time of a launch.
struct WeightsJob {
    const float* weight;
    bf16_bits* w16;
    bf16_bits* transposed;      // null: not wanted
    int* nonfinite;
    int co, ci, taps, kp, first;    // first: the job's first workgroup
};

struct WeightsJobs {
    int count;
    WeightsJob job[TFDTD_CONV_WEIGHT_JOBS];
};

__global__ __launch_bounds__(256) void weights_kernel(const WeightsJobs jobs) {
    __shared__ bf16_bits tile[32][33];
    __shared__ int bad;
    int which = 0;
    for (int k = 1; k < jobs.count; ++k)
        if ((int)blockIdx.x >= jobs.job[k].first) which = k;
    const WeightsJob& j = jobs.job[which];
    const int co = j.co, ci = j.ci, taps = j.taps, kp = j.kp, part = (int)blockIdx.x - j.first, across = (ci + 31) / 32;
    const int tap = part % taps, c0 = part / taps % across * 32, o0 = part / (taps * across) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    bool mine = false;
    for (int r = ty; r < 32; r += 8) {
        const int o = o0 + r, c = c0 + tx;
        if (o < co && c < ci) {
            const bf16_bits b = float_to_bf16(j.weight[((long long)o * taps + tap) * ci + c]);
            mine |= (b & 0x7f80u) == 0x7f80u;      // infinite or NaN, also a finite value that rounds to infinity
            j.w16[(long long)o * kp + tap * ci + c] = b;
            tile[r][tx] = b;
        }
        if (tap == taps - 1 && o < co && c0 + 32 >= ci)
            for (int k = taps * ci + tx; k < kp; k += 32) j.w16[(long long)o * kp + k] = 0;
    }
    __syncthreads();
    if (j.transposed)
        for (int r = ty; r < 32; r += 8) {
            const int c = c0 + r, o = o0 + tx;
            if (c < ci && o < co) j.transposed[((long long)c * taps + tap) * co + o] = tile[tx][r];
        }
    if (mine) bad = 1;
    __syncthreads();
    if (threadIdx.x == 0) j.nonfinite[part] = bad;
}

// Forward convolution with at most 32 values of K (a one-channel input): no staging pays, a wavefront takes
// 64 rows, gathers each row's K values into the MFMA operand and keeps the weights of its columns in
// registers.  Bound by its vector instructions, of which the activation is nearly half, and its scattered 2- or
// 4-byte loads: 524,288 rows x 32 columns to FP32 and bf16 take 39 us (107 in gemm_kernel and its conversion pass; 41
// with the taps' mask formed tap by tap instead of axis by axis), 2,097,152 rows to bf16 from bf16 108 us (128 with a
// division and three comparisons per value, the bias read again behind every row's stores and the rounding in
// integer instructions).  An FP32 source (`Wide`) is rounded as it is read: 113 us, where the conversion pass before it
// took 20.
// n / d for n, d <= 32: (n * small_reciprocal(d)) >> 10 (the excess n * (d - 1) stays below 1024).
__host__ __device__ constexpr int small_reciprocal(int d) { return (1023 + d) / d; }

struct NarrowSplit {
    Divider by_w, by_h, by_d;
    int per_ci, per_ks, per_ks2;    // small_reciprocal of ci, ks and ks * ks
};

template <int CT, bool Wide>
__global__ __launch_bounds__(256) void narrow_forward_kernel(const GatherGemm g, int rows, const NarrowSplit split) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Conv& c = g.c;
    const int col0 = blockIdx.y * CT * 16, fr = lane & 15, fc = lane >> 4;
    bf16x8 w[CT];
    f4 bias[CT];
#pragma unroll
    for (int i = 0; i < CT; ++i) {
        bias[i] = column_bias(g, col0 + 16 * i + fc * 4);
        s8 v = {0, 0, 0, 0, 0, 0, 0, 0};
        const int col = col0 + 16 * i + fr;
        if (col < g.N) v = *reinterpret_cast<const s8*>(g.weight + (long long)col * 32 + fc * 8);
        w[i] = __builtin_bit_cast(bf16x8, v);
    }
    // A lane's 8 values of K: the tap of each (31: none, the padding of K), and its elements from the row's position.
    const int ks = c.ks, kmax = ks * ks * ks * c.ci;
    int tap[8], at[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int k = fc * 8 + t, own = k * split.per_ci >> 10, z = own * split.per_ks2 >> 10, line = own * split.per_ks >> 10;
        const int y = line - z * ks, x = own - line * ks;
        tap[t] = k < kmax ? own : 31;
        at[t] = (((z - c.pad) * c.hi + y - c.pad) * c.wi + x - c.pad) * c.ci + (k - own * c.ci);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = (blockIdx.x * 4 + wave) * 64 + 16 * j + fr;
        const unsigned u = divide((unsigned)row, split.by_w), v = divide(u, split.by_h), nb = divide(v, split.by_d);
        const int x = (row - (int)u * c.wout) * c.stride, y = (int)(u - v * c.hout) * c.stride, z = (int)(v - nb * c.dout) * c.stride;
        const int from = ((((int)nb * c.di + z) * c.hi + y) * c.wi + x) * c.ci;
        // A bit per tap that lies inside the input, from a bit per axis and offset.
        auto axis_bits = [&](int at, int n) {
            unsigned bits = 0u;
            for (int k = 0; k < ks; ++k) bits |= (unsigned)(at + k - c.pad) < (unsigned)n ? 1u << k : 0u;
            return bits;
        };
        const unsigned bx = axis_bits(x, c.wi), by = axis_bits(y, c.hi), bz = axis_bits(z, c.di);
        unsigned line = 0u, inside = 0u;
        for (int k = 0; k < ks; ++k) line |= by >> k & 1u ? bx << k * ks : 0u;
        for (int k = 0; k < ks; ++k) inside |= bz >> k & 1u ? line << k * ks * ks : 0u;
        if (row >= rows) inside = 0u;
        s8 taken;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            taken[t] = 0;
            if (inside >> tap[t] & 1u) {
                const unsigned element = (unsigned)(from + at[t]);
                if (Wide) taken[t] = (short)float_to_bf16(*global(reinterpret_cast<const float*>(reinterpret_cast<const char*>(g.source) + element * 4u)));
                else taken[t] = *global(reinterpret_cast<const short*>(reinterpret_cast<const char*>(g.source) + element * 2u));
            }
        }
#pragma unroll
        for (int i = 0; i < CT; ++i) {
            const f4 sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], __builtin_bit_cast(bf16x8, taken), f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            if (row < rows) finish_columns(g, row, col0 + 16 * i + fc * 4, sum, bias[i]);
        }
    }
}

// Runs the gathered GEMM when source and weights allow 16-byte chunks; false leaves it to gemm_kernel.
bool gather_gemm(GatherGemm g, hipStream_t stream) {
    const long long inside = (long long)g.c.di * g.c.hi * g.c.wi, outside = (long long)g.c.dout * g.c.hout * g.c.wout;
    // Rows are counted in 32 bits, the last workgroup's past the end among them.
    if (g.c.n * inside > 0x7fffffffLL - 256 || g.c.n * outside > 0x7fffffffLL - 256) return false;
    if (inside * g.channels > 0x7fffffffLL || outside * g.channels > 0x7fffffffLL) return false;
    if (g.N % 4 == 0 && (!aligned16(g.pre) || !aligned16(g.y) || (reinterpret_cast<uintptr_t>(g.act) & 7u))) return false;
    if (!g.dgrad && g.ldw == 32 && aligned16(g.weight) && g.c.n * inside * g.c.ci <= (g.wide ? 0x3fffffffLL : 0x7fffffffLL)) {     // 32-bit byte offsets
        const int rows = g.c.n * g.c.dout * g.c.hout * g.c.wout, columns = g.N <= 32 ? 2 : 4;
        const dim3 grid((rows + 255) / 256, (g.N + columns * 16 - 1) / (columns * 16)), block(256);
        const NarrowSplit split{make_divider((unsigned)g.c.wout), make_divider((unsigned)g.c.hout), make_divider((unsigned)g.c.dout),
                                small_reciprocal(g.c.ci), small_reciprocal(g.c.ks), small_reciprocal(g.c.ks * g.c.ks)};
        if (columns == 2) {
            if (g.wide) hipLaunchKernelGGL((narrow_forward_kernel<2, true>), grid, block, 0, stream, g, rows, split);
            else hipLaunchKernelGGL((narrow_forward_kernel<2, false>), grid, block, 0, stream, g, rows, split);
        } else {
            if (g.wide) hipLaunchKernelGGL((narrow_forward_kernel<4, true>), grid, block, 0, stream, g, rows, split);
            else hipLaunchKernelGGL((narrow_forward_kernel<4, false>), grid, block, 0, stream, g, rows, split);
        }
        return true;
    }
    if (g.wide) return false;
    if (g.channels % 8 || !aligned16(g.source) || !aligned16(g.weight) || g.ldw % 8) return false;
    int classes = 1;
    if (g.dgrad && g.c.stride == 2) {
        classes = 8;
        g.rows_max = g.c.n * ((g.c.di + 1) / 2) * ((g.c.hi + 1) / 2) * ((g.c.wi + 1) / 2);
    } else {
        g.rows_max = g.dgrad ? g.c.n * g.c.di * g.c.hi * g.c.wi : g.c.n * g.c.dout * g.c.hout * g.c.wout;
    }
    // The largest tile that still gives each CU two workgroups: its operands are staged least often.  Layers
    // of few rows take small tiles three stages deep, bound by the latency of their K loop: 2048 rows of 256
    // columns (8x8x1 x 128 channels in, stride 2) make 32 tiles of 128 x 128 and 256 of 32 x 64.
    auto blocks = [&](int bm, int bn) { return (long long)((g.rows_max + bm - 1) / bm) * ((g.N + bn - 1) / bn) * classes; };
    if (g.N <= 32) {
        if (blocks(128, 32) >= 512) launch_gather<128, 32, 32, 32, 2>(g, classes, stream);
        else launch_gather<32, 32, 16, 16, 3>(g, classes, stream);
    } else if (g.N > 64 && blocks(128, 128) >= 512) {
        launch_gather<128, 128, 64, 32, 2>(g, classes, stream);     // 64 columns: four waves 0.76 ms, eight 0.83
    } else if (blocks(128, 64) >= 512) {
        launch_gather<128, 64, 64, 32, 2>(g, classes, stream);
    } else if (blocks(64, 64) >= 512) {
        launch_gather<64, 64, 32, 32, 3>(g, classes, stream);
    } else {
        launch_gather<32, 64, 16, 32, 3>(g, classes, stream);
    }
    return true;
}

// ---------------------------------------------------------------- weight gradient
//
// dW[co][k] is the sum over output positions m of dY[m][co] * im2col(m)[k].  Both operands lie with the
// reduction m slowest, so stages of 64 positions go into LDS as they are (rows of dY, gathered 16-byte
// chunks of x) and each MFMA operand is read transposed (ds_read_b64_tr_b16: 4 positions x 16 columns a
// group of 16 lanes) -- no transposed copy of dY in memory.  Chunks lie at chunk ^ swizzle(row), which spreads
// the 16 rows of a transposed read over the banks.  The positions are split over blockIdx.z; each split
// writes its partial sums, which split_sum_kernel adds.  64x32x32x16 positions, 64 -> 128 channels: 0.75 ms
// (620 TFLOP/s), against 3.1 ms and 1.2 ms for the transposed copy of dY; 0.99 ms while each chunk's position
// was found by division in every stage, 0.78 ms with four wavefronts a tile.  The next stage's loads are issued before
// a stage is multiplied, but do not run beside it: the compiler cannot tell the transposed reads from the buffer being
// loaded and waits for the loads before the first of them, so a stage takes its loads' latency and its products in turn.

struct WeightGrad {
    Conv c;
    const bf16_bits* dy;        // [m][co]
    const bf16_bits* x;
    float* partial;             // [split][co][kp]
    int m_total, per_split;
    Divider by_w, by_h, by_d;
    // 64 output positions on, without carries: input cells along x, y and z, and chunks of 8 channels in all; a
    // carry of an axis moves `carry` chunks more.
    int step[3];
    unsigned on, carry[3];
};

template <int Chunks>
__device__ __forceinline__ int row_swizzle(int row) {
    if (Chunks == 16) return 2 * ((row & 3) | (row >> 3 & 1) << 2);
    if (Chunks == 8) return 2 * ((row >> 1 & 1) | (row >> 3 & 1) << 1);
    return 2 * (row >> 3 & 1);
}

// Operand of 16 columns from column `col` (a multiple of 16) and 32 rows from `row` of a [64][Columns] stage.
template <int Columns>
__device__ __forceinline__ bf16x8 transposed(const bf16_bits* stage, int row, int col, int lane) {
    constexpr int Chunks = Columns / 8;
    const int r = row + (lane >> 4) * 8 + ((lane & 15) >> 2);
    const int chunk = (col / 8 + ((lane & 3) >> 1)) ^ row_swizzle<Chunks>(r);
    const bf16_bits* at = stage + r * Columns + chunk * 8 + (lane & 1) * 4;
    typedef __attribute__((address_space(3))) s4 lds_s4;
    const s4 low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)at);
    const s4 high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + 4 * Columns));
    const s8 both = __builtin_shufflevector(low, high, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, both);
}

template <int BC, int BK, int Waves>
__global__ __launch_bounds__(64 * Waves, Waves / 2) void weight_grad_kernel(const WeightGrad g) {
    constexpr int DC = BC / 8, XC = BK / 8;                     // 16-byte chunks of a row
    constexpr int DI = DC / Waves, XI = XC / Waves;             // staging instructions per wave
    constexpr int WC = BC / 2, WK = BK / (Waves / 2), CT = WC / 16, KT = WK / 16;
    static_assert(DI * Waves == DC && XI * Waves == XC, "whole staging instructions");
    constexpr int Stage = 64 * (BC + BK);
    __shared__ __attribute__((aligned(16))) bf16_bits s0[Stage];
    __shared__ __attribute__((aligned(16))) bf16_bits s1[Stage];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Conv& c = g.c;
    const int co0 = blockIdx.x * BC, k0 = blockIdx.y * BK;
    const int begin = blockIdx.z * g.per_split, end = min(g.m_total, begin + g.per_split);
    const bf16_bits* const zero = reinterpret_cast<const bf16_bits*>(&kZeroChunk);
    // The x chunk of each staging instruction: its tap and channel stay for the whole loop, its input cell moves on
    // by 64 output positions a stage, axis by axis with carries -- finding it anew took three divisions and
    // 64-bit products per chunk, more than the matrix instructions.  `at` counts chunks of 8 channels.
    int tx[XI], ty[XI], tz[XI], end_x[XI], end_y[XI], end_z[XI], row_of[XI];
    unsigned at[XI];
    const int ks = c.ks, kmax = ks * ks * ks * c.ci, wide = c.wout * c.stride, high = c.hout * c.stride, deep = c.dout * c.stride;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int row = (wave * XI + i) * (64 / XC) + lane / XC;
        const int k = k0 + ((lane % XC) ^ row_swizzle<XC>(row)) * 8;
        const int tap = k / c.ci, kx = tap % ks - c.pad, ky = tap / ks % ks - c.pad, kz = tap / (ks * ks) - c.pad;
        row_of[i] = k < kmax ? row : 0x7fffffff;
        const unsigned m = (unsigned)(begin + row), u = divide(m, g.by_w), v = divide(u, g.by_h), nb = divide(v, g.by_d);
        tx[i] = (int)(m - u * c.wout) * c.stride + kx;
        ty[i] = (int)(u - v * c.hout) * c.stride + ky;
        tz[i] = (int)(v - nb * c.dout) * c.stride + kz;
        end_x[i] = wide + kx;
        end_y[i] = high + ky;
        end_z[i] = deep + kz;
        at[i] = (unsigned)((((((long long)nb * c.di + tz[i]) * c.hi + ty[i]) * c.wi + tx[i]) * c.ci + (k - tap * c.ci)) >> 3);
    }
    const bf16_bits* dy_at[DI];
#pragma unroll
    for (int i = 0; i < DI; ++i) {
        const int row = (wave * DI + i) * (64 / DC) + lane / DC;
        dy_at[i] = g.dy + (long long)(begin + row) * c.co + co0 + ((lane % DC) ^ row_swizzle<DC>(row)) * 8;
    }
    const long long dy_on = 64LL * c.co;
    auto stage = [&](bf16_bits* into, int m0) {
        const int left = end - m0;
#pragma unroll
        for (int i = 0; i < DI; ++i) {
            const int row = (wave * DI + i) * (64 / DC) + lane / DC, col = co0 + ((lane % DC) ^ row_swizzle<DC>(row)) * 8;
            chunk_to_lds(row < left && col < c.co ? dy_at[i] : zero, into + (wave * DI + i) * 512);
            dy_at[i] += dy_on;
        }
        bf16_bits* const xs = into + 64 * BC;
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const bool inside = (row_of[i] < left) & ((unsigned)tx[i] < (unsigned)c.wi) & ((unsigned)ty[i] < (unsigned)c.hi) &
                                ((unsigned)tz[i] < (unsigned)c.di);
            chunk_to_lds(inside ? g.x + (long long)at[i] * 8 : zero, xs + (wave * XI + i) * 512);
            at[i] += g.on;
            tx[i] += g.step[0];
            const bool cx = tx[i] >= end_x[i];
            tx[i] -= cx ? wide : 0;
            at[i] += cx ? g.carry[0] : 0u;
            ty[i] += cx ? g.step[1] + c.stride : g.step[1];
            const bool cy = ty[i] >= end_y[i];
            ty[i] -= cy ? high : 0;
            at[i] += cy ? g.carry[1] : 0u;
            tz[i] += cy ? g.step[2] + c.stride : g.step[2];
            const bool cz = tz[i] >= end_z[i];
            tz[i] -= cz ? deep : 0;
            at[i] += cz ? g.carry[2] : 0u;
        }
    };
    const int wc = (wave & 1) * WC, wk = (wave >> 1) * WK;
    f4 acc[KT][CT];
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const bf16_bits* from) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 d[CT], x[KT];
#pragma unroll
            for (int j = 0; j < CT; ++j) d[j] = transposed<BC>(from, 32 * h, wc + 16 * j, lane);
#pragma unroll
            for (int i = 0; i < KT; ++i) x[i] = transposed<BK>(from + 64 * BC, 32 * h, wk + 16 * i, lane);
#pragma unroll
            for (int i = 0; i < KT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i], d[j], acc[i][j], 0, 0, 0);
        }
    };
    auto arrive = [&] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070);       // vmcnt(0) lgkmcnt(0): this wave's stage has landed, its reads are done
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (begin < end) stage(s0, begin);
    for (int m = begin; m < end; m += 128) {
        arrive();
        if (m + 64 < end) stage(s1, m + 64);
        multiply(s0);
        if (m + 64 >= end) break;
        arrive();
        if (m + 128 < end) stage(s0, m + 128);
        multiply(s1);
    }
    float* const out = g.partial + (long long)blockIdx.z * c.co * c.kp;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int co = co0 + wc + 16 * j + (lane & 15);
        if (co >= c.co) continue;
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            const int k = k0 + wk + 16 * i + (lane >> 4) * 4;
            if (k < c.kp) *reinterpret_cast<f4*>(out + (long long)co * c.kp + k) = acc[i][j];
        }
    }
}

// The same for at most 32 values of k (a one-channel input): a wavefront gathers its operands from global
// memory element by element -- 32 positions of dY rows and of the 27 shifted inputs -- and the four
// wavefronts of a workgroup add their sums in LDS.  524,288 positions, 1 -> 32 channels: 71 us against
// 2.2 ms (64 workgroups of gemm_kernel, each gathering 8,192 positions one value at a time).
constexpr int kNarrowColumns = 32;

__global__ __launch_bounds__(256) void weight_grad_narrow_kernel(const WeightGrad g) {
    __shared__ float sums[4][kNarrowColumns][33];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Conv& c = g.c;
    const int co0 = blockIdx.x * kNarrowColumns;
    const int begin = blockIdx.z * g.per_split, end = min(g.m_total, begin + g.per_split);
    const int ks = c.ks, kmax = ks * ks * ks * c.ci;
    int tz[2], ty[2], tx[2], ch[2];
    for (int i = 0; i < 2; ++i) {
        const int k = 16 * i + (lane & 15), tap = k / c.ci;
        ch[i] = k < kmax ? k - tap * c.ci : -1;
        tx[i] = tap % ks - c.pad;
        ty[i] = tap / ks % ks - c.pad;
        tz[i] = tap / (ks * ks) - c.pad;
    }
    f4 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    for (int m0 = begin + wave * 32; m0 < end; m0 += 128) {
        s8 x[2], d[2];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int m = m0 + (lane >> 4) * 8 + t;
            const unsigned u = divide((unsigned)m, g.by_w), v = divide(u, g.by_h), nb = divide(v, g.by_d);
            const int px = (m - (int)u * c.wout) * c.stride, py = (int)(u - v * c.hout) * c.stride, pz = (int)(v - nb * c.dout) * c.stride;
            for (int i = 0; i < 2; ++i) {
                const int xx = px + tx[i], yy = py + ty[i], zz = pz + tz[i];
                x[i][t] = 0;
                if (m < end && ch[i] >= 0 && (unsigned)xx < (unsigned)c.wi && (unsigned)yy < (unsigned)c.hi && (unsigned)zz < (unsigned)c.di)
                    x[i][t] = (short)g.x[((((long long)nb * c.di + zz) * c.hi + yy) * c.wi + xx) * c.ci + ch[i]];
            }
            for (int j = 0; j < 2; ++j) {
                const int co = co0 + 16 * j + (lane & 15);
                d[j][t] = 0;
                if (m < end && co < c.co) d[j][t] = (short)g.dy[(long long)m * c.co + co];
            }
        }
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[i]), __builtin_bit_cast(bf16x8, d[j]),
                                                                    acc[i][j], 0, 0, 0);
    }
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int e = 0; e < 4; ++e) sums[wave][16 * j + (lane & 15)][16 * i + (lane >> 4) * 4 + e] = acc[i][j][e];
    __syncthreads();
    for (int e = tid; e < kNarrowColumns * 32; e += 256) {
        const int co = e >> 5, k = e & 31;
        if (co0 + co < c.co)
            g.partial[((long long)blockIdx.z * c.co + co0 + co) * c.kp + k] =
                sums[0][co][k] + sums[1][co][k] + sums[2][co][k] + sums[3][co][k];
    }
}

// Column tiles and K tiles of the weight gradient; 0 where it is left to gemm_kernel.
struct WeightGradShape {
    int bc, bk, splits;
};

WeightGradShape weight_grad_shape(const tfdtd_conv& d, const Conv& c) {
    const long long m = (long long)d.n * c.dout * c.hout * c.wout;
    if (m > 0x7fffffffLL - 256) return {0, 0, 0};
    long long tiles, least;          // workgroups per split, positions a split takes at least
    WeightGradShape s{0, 0, 0};
    if (d.kp == 32) {
        s.bc = kNarrowColumns; s.bk = 32;
        tiles = (d.co + s.bc - 1) / s.bc;
        least = 256;
    } else if (d.ci % 8 == 0 && d.co % 8 == 0 && (long long)d.n * d.di * d.hi * d.wi <= 0xffffffffLL / (d.ci / 8)) {
        s.bc = d.co <= 32 ? 32 : d.co <= 64 ? 64 : 128;
        s.bk = 128;
        tiles = (long long)((d.co + s.bc - 1) / s.bc) * ((d.kp + s.bk - 1) / s.bk);
        least = 256;
    } else {
        return s;
    }
    // Enough workgroups to fill the chip, and up to 6.3 M positions (512 splits, which bound the partial sums' memory) no
    // FP32 sum longer than 12,288 positions (4,096 up to 64 splits); beyond, sums of a 512th of the positions.
    const long long fill = std::min<long long>(768 / tiles, (m + least - 1) / least);
    const long long precise = std::max<long long>((m + 12287) / 12288, std::min<long long>(64, m / 4096));
    s.splits = (int)std::max<long long>(1, std::min<long long>(std::max(fill, precise), 512));
    return s;
}

// dPre = dY * GELU'(pre) (or dY) in bf16, and its sum over the rows before the rounding: each thread keeps
// four channels and adds its rows in FP64, the workgroup adds its threads, bias_sum_kernel adds the workgroups.
// Memory-bound (8 bytes read, 2 written a value): 1.34 GB in 315 us (4.3 TB/s) on 1 M rows of 128; the FP32 copy
// of dPre and its separate sum took 430 + 168 us.
constexpr int kBiasBlocks = TFDTD_BIAS_BLOCKS;

typedef __attribute__((ext_vector_type(4))) double d4;

__global__ __launch_bounds__(256) void gelu_backward_rows_kernel(const float* dy, const float* pre, long long rows, int channels,
                                                                int activation, bf16_bits* dpre16, double* partial) {
    __shared__ d4 sums[256];
    const int quads = channels / 4, per = 256 / quads, q = threadIdx.x % quads, r = threadIdx.x / quads;
    d4 sum = d4{0., 0., 0., 0.};
    if (r < per)
        for (long long row = (long long)blockIdx.x * per + r; row < rows; row += (long long)gridDim.x * per) {
            const long long o = row * channels + 4 * q;
            const f4 d = *reinterpret_cast<const f4*>(dy + o);
            f4 v = d;
            if (activation) {
                const f4 p = *reinterpret_cast<const f4*>(pre + o);
                for (int e = 0; e < 4; ++e) v[e] = d[e] * gelu_grad(p[e]);
            }
            for (int e = 0; e < 4; ++e) sum[e] += (double)v[e];
            *reinterpret_cast<uint2*>(dpre16 + o) = make_uint2(float_to_bf16(v[0]) | (unsigned)float_to_bf16(v[1]) << 16,
                                                              float_to_bf16(v[2]) | (unsigned)float_to_bf16(v[3]) << 16);
        }
    sums[threadIdx.x] = sum;
    __syncthreads();
    if (r == 0) {
        for (int k = 1; k < per; ++k) sum += sums[k * quads + q];
        *reinterpret_cast<d4*>(partial + (long long)blockIdx.x * channels + 4 * q) = sum;
    }
}

__global__ __launch_bounds__(1024) void bias_sum_kernel(const double* partial, int blocks, int channels, float* out) {
    __shared__ double sums[32][32];
    const int c = blockIdx.x * 32 + (threadIdx.x & 31), part = threadIdx.x >> 5;
    double s = 0.;
    if (c < channels)
#pragma unroll 4
        for (int b = part; b < blocks; b += 32) s += partial[(long long)b * channels + c];
    sums[part][threadIdx.x & 31] = s;
    __syncthreads();
    if (part == 0 && c < channels) {
        for (int k = 1; k < 32; ++k) s += sums[k][threadIdx.x];
        out[c] = (float)s;
    }
}

int check_conv(const tfdtd_conv& d) {
    if (d.n < 1 || d.di < 1 || d.hi < 1 || d.wi < 1 || d.ci < 1 || d.co < 1)
        return tfdtd_fail(TFDTD_EINVAL, "conv: sizes must be positive");
    if ((d.ks != 1 && d.ks != 3) || d.stride < 1 || d.stride > 2 || d.pad < 0 || d.pad >= d.ks)
        return tfdtd_fail(TFDTD_EINVAL, "conv: kernel 1 or 3, stride 1 or 2, 0 <= pad < kernel");
    const int k = d.ks * d.ks * d.ks * d.ci;
    if (d.kp < k || d.kp % 32) return tfdtd_fail(TFDTD_EINVAL, "conv: kp must be ks^3*ci rounded up to a multiple of 32");
    return TFDTD_OK;
}

Conv make_conv(const tfdtd_conv& d) {
    Conv c;
    c.n = d.n; c.di = d.di; c.hi = d.hi; c.wi = d.wi; c.ci = d.ci; c.co = d.co;
    c.ks = d.ks; c.stride = d.stride; c.pad = d.pad; c.kp = d.kp;
    c.dout = (d.di + 2 * d.pad - d.ks) / d.stride + 1;
    c.hout = (d.hi + 2 * d.pad - d.ks) / d.stride + 1;
    c.wout = (d.wi + 2 * d.pad - d.ks) / d.stride + 1;
    return c;
}

}  // namespace

extern "C" {

int tfdtd_conv_output(const tfdtd_conv* d, int32_t* dout, int32_t* hout, int32_t* wout) {
    if (!d) return tfdtd_fail(TFDTD_EINVAL, "conv: null descriptor");
    const int status = check_conv(*d);
    if (status) return status;
    const Conv c = make_conv(*d);
    if (c.dout < 1 || c.hout < 1 || c.wout < 1) return tfdtd_fail(TFDTD_EINVAL, "conv: empty output");
    *dout = c.dout; *hout = c.hout; *wout = c.wout;
    return TFDTD_OK;
}

int tfdtd_conv_forward(const tfdtd_conv* d, const void* x, const void* weight, const float* bias, int32_t activation,
                       float* pre, void* act, void* stream) {
    if (!d || !x || !weight || !pre || !act) return tfdtd_fail(TFDTD_EINVAL, "conv forward: null pointer");
    int status = check_conv(*d);
    if (status) return status;
    Gemm g{};
    g.op = 0;
    g.c = make_conv(*d);
    g.M = (int)((long long)d->n * g.c.dout * g.c.hout * g.c.wout);
    g.N = d->co;
    g.K = d->kp;
    g.k_per_split = g.K;
    g.a = static_cast<const bf16_bits*>(x);
    g.b = static_cast<const bf16_bits*>(weight);
    g.bias = bias;
    g.activation = activation;
    g.out = pre;
    g.act = static_cast<bf16_bits*>(act);
    if ((long long)d->n * g.c.dout * g.c.hout * g.c.wout > 0x7fffffffLL) return tfdtd_fail(TFDTD_EINVAL, "conv: too many positions");
    GatherGemm h{};
    h.c = g.c;
    h.N = d->co; h.channels = d->ci; h.ldw = d->kp;
    h.source = g.a; h.weight = g.b;
    h.bias = bias; h.activation = activation;
    h.pre = pre; h.act = g.act;
    if (gather_gemm(h, static_cast<hipStream_t>(stream))) return tfdtd_check_launch("conv forward");
    hipLaunchKernelGGL(gemm_kernel, dim3((g.M + BM - 1) / BM, (g.N + BN - 1) / BN, 1), dim3(256), 0,
                       static_cast<hipStream_t>(stream), g);
    return tfdtd_check_launch("conv forward");
}

int tfdtd_conv_dgrad(const tfdtd_conv* d, const void* dy, const void* weight_t, float* dx, void* stream) {
    if (!d || !dy || !weight_t || !dx) return tfdtd_fail(TFDTD_EINVAL, "conv dgrad: null pointer");
    int status = check_conv(*d);
    if (status) return status;
    if (d->co % 8) return tfdtd_fail(TFDTD_EINVAL, "conv dgrad: output channels must be a multiple of 8");
    Gemm g{};
    g.op = 1;
    g.c = make_conv(*d);
    g.M = (int)((long long)d->n * d->di * d->hi * d->wi);
    g.N = d->ci;
    g.K = d->ks * d->ks * d->ks * d->co;
    g.k_per_split = g.K;
    g.a = static_cast<const bf16_bits*>(dy);
    g.b = static_cast<const bf16_bits*>(weight_t);
    g.out = dx;
    GatherGemm h{};
    h.c = g.c;
    h.dgrad = 1;
    h.N = d->ci; h.channels = d->co; h.ldw = g.K;
    h.source = g.a; h.weight = g.b;
    h.pre = dx;
    if (gather_gemm(h, static_cast<hipStream_t>(stream))) return tfdtd_check_launch("conv dgrad");
    hipLaunchKernelGGL(gemm_kernel, dim3((g.M + BM - 1) / BM, (g.N + BN - 1) / BN, 1), dim3(256), 0,
                       static_cast<hipStream_t>(stream), g);
    return tfdtd_check_launch("conv dgrad");
}

int tfdtd_conv_wgrad(const tfdtd_conv* d, const void* dy_t, const void* x, int32_t splits, float* partial, float* dw,
                     void* stream) {
    if (!d || !dy_t || !x || !partial || !dw || splits < 1) return tfdtd_fail(TFDTD_EINVAL, "conv wgrad: bad arguments");
    int status = check_conv(*d);
    if (status) return status;
    Gemm g{};
    g.op = 2;
    g.c = make_conv(*d);
    const long long m_total = (long long)d->n * g.c.dout * g.c.hout * g.c.wout;
    g.M = d->co;
    g.N = d->kp;
    g.K = (int)((m_total + BK - 1) / BK * BK);
    g.k_per_split = (int)((g.K / BK + splits - 1) / splits * BK);
    g.a = static_cast<const bf16_bits*>(dy_t);
    g.b = static_cast<const bf16_bits*>(x);
    g.out = partial;
    const int used = (g.K + g.k_per_split - 1) / g.k_per_split;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(gemm_kernel, dim3((g.M + BM - 1) / BM, (g.N + BN - 1) / BN, used), dim3(256), 0, s, g);
    status = tfdtd_check_launch("conv wgrad");
    if (status) return status;
    const long long count = (long long)g.M * g.N;
    hipLaunchKernelGGL(split_sum_kernel, dim3(split_sum_blocks(count)), dim3(256), 0, s, partial, used, count, dw);
    return tfdtd_check_launch("conv wgrad sum");
}

int tfdtd_conv_weight_parts(const tfdtd_conv* d) {
    if (!d || check_conv(*d)) return 0;
    return d->ks * d->ks * d->ks * ((d->ci + 31) / 32) * ((d->co + 31) / 32);
}

int tfdtd_conv_weights(const tfdtd_conv* convs, int32_t count, const float* const* weights, void* const* w16,
                       void* const* weights_t, int32_t* const* nonfinite, void* stream) {
    if (!convs || !weights || !w16 || !nonfinite || count < 1 || count > TFDTD_CONV_WEIGHT_JOBS)
        return tfdtd_fail(TFDTD_EINVAL, "conv weights: null pointer, or not 1 to %d layers", TFDTD_CONV_WEIGHT_JOBS);
    WeightsJobs jobs{};
    jobs.count = count;
    long long blocks = 0;
    for (int k = 0; k < count; ++k) {
        const tfdtd_conv& d = convs[k];
        const int status = check_conv(d);
        if (status) return status;
        if (!weights[k] || !w16[k] || !nonfinite[k]) return tfdtd_fail(TFDTD_EINVAL, "conv weights: layer %d: null pointer", k);
        jobs.job[k] = WeightsJob{weights[k], static_cast<bf16_bits*>(w16[k]), weights_t ? static_cast<bf16_bits*>(weights_t[k]) : nullptr,
                                 nonfinite[k], d.co, d.ci, d.ks * d.ks * d.ks, d.kp, (int)blocks};
        blocks += tfdtd_conv_weight_parts(&d);
        if (blocks > 0x7fffffffLL) return tfdtd_fail(TFDTD_EINVAL, "conv weights: too many weights for one launch");
    }
    hipLaunchKernelGGL(weights_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), jobs);
    return tfdtd_check_launch("conv weights");
}

int tfdtd_conv_forward_rows(const tfdtd_conv* d, const void* x, int32_t x_dtype, const void* weight, const int32_t* nonfinite,
                            const float* bias, int32_t activation, float* pre, float* y, void* act, void* stream) {
    if (x_dtype != TFDTD_CONV_BF16 && x_dtype != TFDTD_F32) return tfdtd_fail(TFDTD_EINVAL, "conv forward: x is bf16 or float32");
    if (!d || !x || !weight || (!pre && !y && !act)) return tfdtd_fail(TFDTD_EINVAL, "conv forward: null pointer");
    int status = check_conv(*d);
    if (status) return status;
    GatherGemm g{};
    g.c = make_conv(*d);
    if ((long long)d->n * g.c.dout * g.c.hout * g.c.wout > 0x7fffffffLL) return tfdtd_fail(TFDTD_EINVAL, "conv: too many positions");
    g.N = d->co; g.channels = d->ci; g.ldw = d->kp;
    g.wide = x_dtype == TFDTD_F32;
    g.source = static_cast<const bf16_bits*>(x);
    g.weight = static_cast<const bf16_bits*>(weight);
    g.nonfinite = nonfinite;
    g.parts = tfdtd_conv_weight_parts(d);
    g.bias = bias;
    g.activation = activation;
    g.pre = pre; g.y = y; g.act = static_cast<bf16_bits*>(act);
    if (!gather_gemm(g, static_cast<hipStream_t>(stream)))
        return tfdtd_fail(TFDTD_EUNSUPPORTED, "conv forward: channels or alignment are left to tfdtd_conv_forward");
    return tfdtd_check_launch("conv forward");
}

int tfdtd_conv_dgrad_rows(const tfdtd_conv* d, const void* dy, const void* weight_t, const int32_t* nonfinite, float* dx,
                          void* stream) {
    if (!d || !dy || !weight_t || !dx) return tfdtd_fail(TFDTD_EINVAL, "conv dgrad: null pointer");
    int status = check_conv(*d);
    if (status) return status;
    GatherGemm g{};
    g.c = make_conv(*d);
    g.dgrad = 1;
    g.N = d->ci; g.channels = d->co; g.ldw = d->ks * d->ks * d->ks * d->co;
    g.source = static_cast<const bf16_bits*>(dy);
    g.weight = static_cast<const bf16_bits*>(weight_t);
    g.nonfinite = nonfinite;
    g.parts = tfdtd_conv_weight_parts(d);
    g.pre = dx;
    if (!gather_gemm(g, static_cast<hipStream_t>(stream)))
        return tfdtd_fail(TFDTD_EUNSUPPORTED, "conv dgrad: channels or alignment are left to tfdtd_conv_dgrad");
    return tfdtd_check_launch("conv dgrad");
}

int tfdtd_conv_wgrad_splits(const tfdtd_conv* d) {
    if (!d || check_conv(*d)) return 0;
    return weight_grad_shape(*d, make_conv(*d)).splits;
}

int tfdtd_conv_wgrad_rows(const tfdtd_conv* d, const void* dy, const void* x, float* partial, float* dw, void* stream) {
    if (!d || !dy || !x || !partial || !dw) return tfdtd_fail(TFDTD_EINVAL, "conv wgrad: bad arguments");
    int status = check_conv(*d);
    if (status) return status;
    WeightGrad g{};
    g.c = make_conv(*d);
    const WeightGradShape shape = weight_grad_shape(*d, g.c);
    if (shape.splits == 0) return tfdtd_fail(TFDTD_EINVAL, "conv wgrad: channels must be multiples of 8, or at most 32 kernel values");
    if (d->kp != 32 && (!aligned16(dy) || !aligned16(x) || !aligned16(partial)))
        return tfdtd_fail(TFDTD_EINVAL, "conv wgrad: operands must be 16-byte aligned");
    g.dy = static_cast<const bf16_bits*>(dy);
    g.x = static_cast<const bf16_bits*>(x);
    g.partial = partial;
    g.m_total = d->n * g.c.dout * g.c.hout * g.c.wout;
    g.per_split = (int)(((long long)g.m_total + 64LL * shape.splits - 1) / (64LL * shape.splits) * 64);
    g.by_w = make_divider((unsigned)g.c.wout);
    g.by_h = make_divider((unsigned)g.c.hout);
    g.by_d = make_divider((unsigned)g.c.dout);
    const int x64 = 64 % g.c.wout, u64 = 64 / g.c.wout, y64 = u64 % g.c.hout, v64 = u64 / g.c.hout, z64 = v64 % g.c.dout;
    const long long chunk = d->ci / 8, line = chunk * d->wi, page = line * d->hi;
    g.step[0] = x64 * d->stride; g.step[1] = y64 * d->stride; g.step[2] = z64 * d->stride;
    g.on = (unsigned)(g.step[0] * chunk + g.step[1] * line + g.step[2] * page + v64 / g.c.dout * (page * d->di));
    g.carry[0] = (unsigned)(d->stride * (line - g.c.wout * chunk));
    g.carry[1] = (unsigned)(d->stride * (page - g.c.hout * line));
    g.carry[2] = (unsigned)(page * d->di - (long long)d->stride * g.c.dout * page);
    const int used = (g.m_total + g.per_split - 1) / g.per_split;
    const dim3 grid((d->co + shape.bc - 1) / shape.bc, (d->kp + shape.bk - 1) / shape.bk, used), block(256), wide(512);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (d->kp == 32) hipLaunchKernelGGL(weight_grad_narrow_kernel, grid, block, 0, s, g);
    else if (shape.bc == 32) hipLaunchKernelGGL((weight_grad_kernel<32, 128, 4>), grid, block, 0, s, g);
    else if (shape.bc == 64) hipLaunchKernelGGL((weight_grad_kernel<64, 128, 8>), grid, wide, 0, s, g);
    else hipLaunchKernelGGL((weight_grad_kernel<128, 128, 8>), grid, wide, 0, s, g);
    status = tfdtd_check_launch("conv wgrad");
    if (status) return status;
    const long long count = (long long)d->co * d->kp;
    hipLaunchKernelGGL(split_sum_kernel, dim3(split_sum_blocks(count)), dim3(256), 0, s, partial, used, count, dw);
    return tfdtd_check_launch("conv wgrad sum");
}

int tfdtd_gelu_backward_rows(const float* dy, const float* pre, int64_t rows, int32_t channels, int32_t activation, void* dpre16,
                             double* partial, float* bias_grad, void* stream) {
    if (!dy || (activation && !pre) || !dpre16 || !partial || !bias_grad || rows < 1 || channels < 4 || channels > 1024 || channels % 4)
        return tfdtd_fail(TFDTD_EINVAL, "gelu backward rows: bad arguments (channels: a multiple of 4, at most 1024)");
    if (!aligned16(dy) || !aligned16(pre) || !aligned16(partial) || (reinterpret_cast<uintptr_t>(dpre16) & 7u))
        return tfdtd_fail(TFDTD_EINVAL, "gelu backward rows: operands must be 16-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int per = 256 / (channels / 4);
    const int blocks = (int)std::min<int64_t>(kBiasBlocks, (rows + 4LL * per - 1) / (4 * per));
    hipLaunchKernelGGL(gelu_backward_rows_kernel, dim3(blocks), dim3(256), 0, s, dy, pre, (long long)rows, channels, activation,
                       static_cast<bf16_bits*>(dpre16), partial);
    int status = tfdtd_check_launch("gelu backward rows");
    if (status) return status;
    hipLaunchKernelGGL(bias_sum_kernel, dim3((channels + 31) / 32), dim3(1024), 0, s, partial, blocks, channels, bias_grad);
    return tfdtd_check_launch("bias gradient");
}

int tfdtd_gelu_backward(const float* dy, const float* pre, int64_t count, int32_t activation, float* dpre, void* dpre16,
                        void* stream) {
    if (!dy || (activation && !pre) || !dpre || !dpre16 || count < 0) return tfdtd_fail(TFDTD_EINVAL, "gelu backward: bad arguments");
    if (count == 0) return TFDTD_OK;
    hipLaunchKernelGGL(gelu_backward_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       dy, pre, (long long)count, activation, dpre, static_cast<bf16_bits*>(dpre16));
    return tfdtd_check_launch("gelu backward");
}

}  // extern "C"
