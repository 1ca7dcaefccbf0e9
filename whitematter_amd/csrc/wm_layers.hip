// Normalisation and attention-softmax kernels (reference core/layer.cpp).
//
// LayerNorm (core/layer.cpp:395-504).  One row (instance) per workgroup,
// held in registers (RowTile): the forward is the reference's two passes
// (mean, then the sum of squared deviations) over registers, so the row is
// read once and written once.  The backward computes both row sums of the
// closure with one barrier, writes dx, and keeps the dgamma / dbeta column
// partials of the rows it visits in registers (a thread owns the same
// columns in every row), so the parameter gradients cost one
// [workgroups, n] partial write and a fixed-order column pass instead of a
// second read of g and x.  Rows longer than 8192 elements stream through
// global memory instead and take the parameter gradients in a separate
// column pass.
//
// BatchNorm2d (core/layer.cpp:202-374).  x is [batch, channels, spatial];
// a channel's elements are `batch` planes of `spatial` contiguous floats.
// A channel of up to 16384 floats (8192 where its units are single floats:
// planes that are not a multiple of 4, or unaligned) is held in one
// workgroup's registers: one launch reads it once, reduces it and writes the
// result.  Larger channels take two passes of (channel, chunk) workgroups that
// walk the channel's units across plane ends.  Either way the channel's
// constants are loaded once per workgroup.  The statistics accumulate sum(x)
// and sum(x^2) (forward) and sum(g), sum(g (x - mean)), sum(x - mean)
// (backward) in double per thread and per chunk, combined in a fixed order:
// one pass over the data, no cancellation problem at fp32 data magnitudes,
// deterministic.
//
// MultiHeadAttention's softmax (core/layer.cpp:1198-1237, backward
// :1343-1360): one row of scores per workgroup with the mask row added in
// registers, the reference's max-from--FLT_MAX, and its plain backward
// attn * (d_attn - sum(attn * d_attn)).  The reference divides each
// exponential by the row sum; here they are multiplied by one reciprocal per
// row (within an ulp of the quotient, inside the softmax tolerance, and an
// IEEE division per element would cost more than the row's memory traffic).
#include "wm_rows.hpp"

#include <algorithm>
#include <cfloat>

#include "../../include/wm_layers.h"

namespace wm {
namespace {

// Two sums across the workgroup with one barrier.  `lds` must not be
// written again until every thread has read it: callers alternate between
// two arrays per row (see ln_bwd_kernel).
template <int NT>
__device__ __forceinline__ float2 block_sum2_1(float a, float b, float2* lds) {
    constexpr int NW = NT / 64;
    a = wave_sum(a);
    b = wave_sum(b);
    if (NW == 1) return make_float2(a, b);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = make_float2(a, b);
    __syncthreads();
    float2 t = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        t.x += lds[i].x;
        t.y += lds[i].y;
    }
    return t;
}

// Sum of a double over a 256-thread workgroup into thread 0 (fixed order).
__device__ __forceinline__ double block_sum_d256(double v, double* lds) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0) t = (lds[0] + lds[1]) + (lds[2] + lds[3]);
    __syncthreads();
    return t;
}

// ---------------------------------------------------------------------------
// LayerNorm
// ---------------------------------------------------------------------------

template <int NT, int ITEMS, bool VEC>
__global__ void __launch_bounds__(NT) ln_fwd_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                     const float* __restrict__ beta, int64_t rows, int64_t n,
                                                     float eps, float* __restrict__ y, float* __restrict__ mean_out,
                                                     float* __restrict__ inv_out) {
    using Tile = RowTile<NT, ITEMS, VEC>;
    __shared__ float lds_a[NT / 64], lds_b[NT / 64];
    Tile gt, bt;  // this thread's columns of gamma / beta, the same in every row
    gt.template load<true>(gamma, n, 0.f);
    bt.template load<true>(beta, n, 0.f);
    const float nf = (float)n;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        Tile t;
        t.load(x + r * n, n, 0.f);
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) s += t.v[i][e];
        const float mean = block_sum_1<NT>(s, lds_a) / nf;
        float q = 0.f;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (Tile::col(i, e) < n) {
                    const float d = t.v[i][e] - mean;
                    q += d * d;
                }
        const float var = block_sum_1<NT>(q, lds_b) / nf;
        const float inv = 1.0f / sqrtf(var + eps);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) t.v[i][e] = gt.v[i][e] * ((t.v[i][e] - mean) * inv) + bt.v[i][e];
        t.store(y + r * n, n);
        if (threadIdx.x == 0) {
            mean_out[r] = mean;
            inv_out[r] = inv;
        }
    }
}

// pgamma / pbeta: [gridDim.x, n] partials of this workgroup's rows (NULL
// when that gradient is not wanted).
//
// The second __launch_bounds__ argument is HIP's minimum waves per SIMD: a
// 1024-thread workgroup puts 4 waves on each SIMD, so 8 keeps the kernel
// within 64 VGPRs and two workgroups resident per CU (one float4 per
// thread and row; the compiler's own choice, 66, left one: 67 -> 71 % of
// the HBM peak at [32768, 4096]).  Two float4s per thread need more than
// 64 without spilling.
template <int NT, int ITEMS>
constexpr int ln_bwd_min_waves() { return NT == 1024 && ITEMS == 1 ? 8 : 1; }

template <int NT, int ITEMS, bool VEC>
__global__ void __launch_bounds__(NT, (ln_bwd_min_waves<NT, ITEMS>())) ln_bwd_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                     const float* __restrict__ gamma, const float* __restrict__ mean,
                                                     const float* __restrict__ inv_std, int64_t rows, int64_t n,
                                                     float* __restrict__ gx, int acc, float* __restrict__ pgamma,
                                                     float* __restrict__ pbeta) {
    using Tile = RowTile<NT, ITEMS, VEC>;
    __shared__ float2 lds2[2][NT / 64];
    Tile gt;
    gt.template load<true>(gamma, n, 0.f);
    float pg[ITEMS][4], pb[ITEMS][4];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) pg[i][e] = pb[i][e] = 0.f;
    const float nf = (float)n;
    int k = 0;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x, ++k) {
        Tile dy, xv;
        dy.load(g + r * n, n, 0.f);
        xv.load(x + r * n, n, 0.f);
        const float m = mean[r], iv = inv_std[r];
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float xn = (xv.v[i][e] - m) * iv;
                xv.v[i][e] = xn;
                const float dg = dy.v[i][e] * gt.v[i][e];
                s1 += dg;
                s2 += dg * xn;
                pg[i][e] += dy.v[i][e] * xn;  // padding: dy = 0
                pb[i][e] += dy.v[i][e];
            }
        const float2 S = block_sum2_1<NT>(s1, s2, lds2[k & 1]);
        if (gx) {
            const float mdg = S.x / nf, mdgx = S.y / nf;
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    dy.v[i][e] = iv * (dy.v[i][e] * gt.v[i][e] - mdg - xv.v[i][e] * mdgx);
            if (acc) {
                Tile old;
                old.load(gx + r * n, n, 0.f);
#pragma unroll
                for (int i = 0; i < ITEMS; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dy.v[i][e] = old.v[i][e] + dy.v[i][e];
            }
            dy.store(gx + r * n, n);
        }
    }
    float* pgr = pgamma ? pgamma + (int64_t)blockIdx.x * n : nullptr;
    float* pbr = pbeta ? pbeta + (int64_t)blockIdx.x * n : nullptr;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t c = Tile::col(i, e);
            if (c < n) {
                if (pgr) pgr[c] = pg[i][e];
                if (pbr) pbr[c] = pb[i][e];
            }
        }
}

// Rows of up to 1024 elements: a wave per row (no barrier inside a row), four
// rows of a workgroup at a time.  The four waves' parameter partials are added
// through LDS at the end, so a workgroup leaves one partial row for four
// waves' worth of rows in flight.  [8192, 768]: 17 us against 36.6
// for a 256-thread workgroup per row (32 rows each; 17.9 with 8 rows each, and
// 10 more for the sums over its four times as many partial rows).
template <int ITEMS, bool VEC>
__global__ void __launch_bounds__(256) ln_bwd_wave_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                           const float* __restrict__ gamma,
                                                           const float* __restrict__ mean,
                                                           const float* __restrict__ inv_std, int64_t rows, int64_t n,
                                                           float* __restrict__ gx, int acc, float* __restrict__ pgamma,
                                                           float* __restrict__ pbeta) {
    using Tile = RowTile<64, ITEMS, VEC>;
    __shared__ float lds[4][ITEMS * 256];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    Tile gt;
    gt.template load<true>(gamma, n, 0.f);
    float pg[ITEMS][4], pb[ITEMS][4];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) pg[i][e] = pb[i][e] = 0.f;
    const float nf = (float)n;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        Tile dy, xv;
        dy.load(g + r * n, n, 0.f);
        xv.load(x + r * n, n, 0.f);
        const float m = mean[r], iv = inv_std[r];
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float xn = (xv.v[i][e] - m) * iv;
                xv.v[i][e] = xn;
                const float dg = dy.v[i][e] * gt.v[i][e];
                s1 += dg;
                s2 += dg * xn;
                pg[i][e] += dy.v[i][e] * xn;  // padding: dy = 0
                pb[i][e] += dy.v[i][e];
            }
        if (gx) {
            const float mdg = wave_sum(s1) / nf, mdgx = wave_sum(s2) / nf;
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    dy.v[i][e] = iv * (dy.v[i][e] * gt.v[i][e] - mdg - xv.v[i][e] * mdgx);
            if (acc) {
                Tile old;
                old.load(gx + r * n, n, 0.f);
#pragma unroll
                for (int i = 0; i < ITEMS; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dy.v[i][e] = old.v[i][e] + dy.v[i][e];
            }
            dy.store(gx + r * n, n);
        }
    }
    auto fold = [&](const float (&p)[ITEMS][4], float* part) {
        if (!part) return;  // uniform
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) lds[wave][Tile::col(i, e)] = p[i][e];
        __syncthreads();
        for (int c = (int)threadIdx.x; c < n; c += 256)
            part[(int64_t)blockIdx.x * n + c] = (lds[0][c] + lds[1][c]) + (lds[2][c] + lds[3][c]);
    };
    fold(pg, pgamma);
    fold(pb, pbeta);
}

// Column sums of [parts, n] partials: out[c] (+)= sum_p part[p][c].  A
// workgroup owns S adjacent columns; its NT / S row lanes take every
// (NT / S)-th partial row in 8 interleaved accumulators and are added in a
// tree through LDS.  blockIdx.z picks one of two independent sums (the weight and
// bias gradients share the launch).
template <int S, int NT>
__global__ void __launch_bounds__(NT) colsum_parts_kernel(const float* __restrict__ part0,
                                                            const float* __restrict__ part1, int64_t parts, int64_t n,
                                                            float* __restrict__ out0, float* __restrict__ out1,
                                                            int acc0, int acc1) {
    constexpr int G = NT / S;
    __shared__ float lds[G][S];
    const float* part = blockIdx.z ? part1 : part0;
    float* out = blockIdx.z ? out1 : out0;
    const int acc = blockIdx.z ? acc1 : acc0;
    const int cl = threadIdx.x % S, g = threadIdx.x / S;
    const int64_t c = (int64_t)blockIdx.x * S + cl;
    lds[g][cl] = c < n ? strided_sum<G>(part + c, n, g, parts) : 0.f;
#pragma unroll
    for (int h = G / 2; h > 0; h /= 2) {
        __syncthreads();
        if (g < h) lds[g][cl] += lds[g + h][cl];
    }
    if (g == 0 && c < n) out[c] = acc ? out[c] + lds[0][cl] : lds[0][cl];
}

// Column sums of [parts, n] partial rows into out_g and out_b (+= when
// acc_*; a null partial array skips its sum), in one launch.  Few columns per
// workgroup, or many row lanes, where there are few columns, so that they still
// spread over the chip (as colsum_finalize_kernel; a stage of 64-row sums in front
// cost a second dispatch: 8.5 -> 4.5 us at [256, 768] partials).
int colsum_parts(const float* part_g, float* out_g, int acc_g, const float* part_b, float* out_b, int acc_b,
                 int64_t parts, int64_t n, const char* what) {
    hipStream_t st = stream();
    if (!part_g) {  // the bias sum alone: slot 0
        part_g = part_b; out_g = out_b; acc_g = acc_b;
        part_b = nullptr;
    }
    if (!part_g) return WM_OK;
    const unsigned jobs = part_b ? 2u : 1u;
    const int64_t cols = n * jobs, want = num_cus();
#define WM_CP(S, NT)                                                                                          \
    launch_kernel((colsum_parts_kernel<S, NT>), dim3((unsigned)((n + S - 1) / S), 1u, jobs), dim3(NT), 0, st, \
                  part_g, part_b, parts, n, out_g, out_b, acc_g, acc_b)
    if (cols >= 64 * want) WM_CP(64, 256);
    else if (cols >= 8 * want) WM_CP(64, 1024);
    else WM_CP(4, 256);
#undef WM_CP
    return check_launch(what);
}

// Rows longer than the register tile: three streaming passes per row.
__global__ void __launch_bounds__(1024) ln_fwd_long_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                            const float* __restrict__ beta, int64_t rows, int64_t n,
                                                            float eps, float* __restrict__ y,
                                                            float* __restrict__ mean_out, float* __restrict__ inv_out) {
    __shared__ float lds_a[16], lds_b[16];
    const float nf = (float)n;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float* xr = x + r * n;
        float s = 0.f;
        for (int64_t c = threadIdx.x; c < n; c += 1024) s += xr[c];
        const float mean = block_sum_1<1024>(s, lds_a) / nf;
        float q = 0.f;
        for (int64_t c = threadIdx.x; c < n; c += 1024) {
            const float d = xr[c] - mean;
            q += d * d;
        }
        const float inv = 1.0f / sqrtf(block_sum_1<1024>(q, lds_b) / nf + eps);
        for (int64_t c = threadIdx.x; c < n; c += 1024) y[r * n + c] = gamma[c] * ((xr[c] - mean) * inv) + beta[c];
        if (threadIdx.x == 0) {
            mean_out[r] = mean;
            inv_out[r] = inv;
        }
    }
}

__global__ void __launch_bounds__(1024) ln_bwd_long_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                            const float* __restrict__ gamma,
                                                            const float* __restrict__ mean,
                                                            const float* __restrict__ inv_std, int64_t rows, int64_t n,
                                                            float* __restrict__ gx, int acc) {
    __shared__ float2 lds2[2][16];
    const float nf = (float)n;
    int k = 0;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x, ++k) {
        const float* gr = g + r * n;
        const float* xr = x + r * n;
        const float m = mean[r], iv = inv_std[r];
        float s1 = 0.f, s2 = 0.f;
        for (int64_t c = threadIdx.x; c < n; c += 1024) {
            const float dg = gr[c] * gamma[c];
            s1 += dg;
            s2 += dg * ((xr[c] - m) * iv);
        }
        const float2 S = block_sum2_1<1024>(s1, s2, lds2[k & 1]);
        const float mdg = S.x / nf, mdgx = S.y / nf;
        for (int64_t c = threadIdx.x; c < n; c += 1024) {
            const float d = iv * (gr[c] * gamma[c] - mdg - ((xr[c] - m) * iv) * mdgx);
            gx[r * n + c] = acc ? gx[r * n + c] + d : d;
        }
    }
}

// dgamma / dbeta partials for the long-row path: [chunks, n], each thread a
// column, each workgroup a chunk of rows.
__global__ void __launch_bounds__(256) ln_param_parts_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                              const float* __restrict__ mean,
                                                              const float* __restrict__ inv_std, int64_t rows,
                                                              int64_t n, int64_t rows_per_chunk,
                                                              float* __restrict__ pgamma, float* __restrict__ pbeta) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_chunk;
    const int64_t r1 = r0 + rows_per_chunk < rows ? r0 + rows_per_chunk : rows;
    if (c >= n) return;
    float sg = 0.f, sb = 0.f;
    for (int64_t r = r0; r < r1; ++r) {
        const float dy = g[r * n + c];
        sg += dy * ((x[r * n + c] - mean[r]) * inv_std[r]);
        sb += dy;
    }
    if (pgamma) pgamma[(int64_t)blockIdx.y * n + c] = sg;
    if (pbeta) pbeta[(int64_t)blockIdx.y * n + c] = sb;
}

// ---------------------------------------------------------------------------
// BatchNorm2d
// ---------------------------------------------------------------------------

// A channel's units: a unit is a float4 (VEC: spatial % 4 == 0 and aligned
// bases) or a float, `units` of them per plane, B * units per channel, numbered
// plane after plane.  Threads take consecutive units whatever the plane size
// (a 14 x 14 plane is 49 float4s: one plane per 256-thread step left 4 of 5
// lanes idle), and advance by a constant number of planes and units, without
// dividing.
constexpr int64_t kBnStep = 4 * 256;  // units of a workgroup's step in the two-pass kernels

struct BnGeom {
    int64_t C, S, units;   // units per plane
    int64_t total;         // units per channel
    int64_t per, chunks;   // units per chunk, chunks per channel (gridDim.x)
};

struct BnWalk {
    int64_t plane, unit, step_plane, step_unit, units, stride, at;
    // The walk of channel c from its unit u in steps of `step` units.
    __device__ __forceinline__ BnWalk(const BnGeom& gm, int64_t c, int64_t u, int step)
        : units(gm.units), stride(gm.C * gm.S), at(c * gm.S) {
        if ((gm.total + gm.per) >> 31) {  // uniform
            plane = u / units;
            step_plane = step / units;
        } else {
            plane = (uint32_t)u / (uint32_t)units;
            step_plane = (uint32_t)step / (uint32_t)units;
        }
        unit = u - plane * units;
        step_unit = step - step_plane * units;
    }
    template <int W>
    __device__ __forceinline__ int64_t offset() const { return plane * stride + at + unit * W; }
    __device__ __forceinline__ void next() {
        plane += step_plane;
        unit += step_unit;
        if (unit >= units) { unit -= units; ++plane; }
    }
};

// Visit every unit of this workgroup's chunk (blockIdx.x) of its channel
// (blockIdx.y): f(offsets in floats, which of them are in the chunk), four
// units per thread per step.
template <bool VEC, class F>
__device__ __forceinline__ void bn_for_chunk(const BnGeom& gm, F&& f) {
    const int64_t u0 = (int64_t)blockIdx.x * gm.per, u1 = u0 + gm.per < gm.total ? u0 + gm.per : gm.total;
    int64_t u = u0 + threadIdx.x;
    BnWalk w(gm, blockIdx.y, u, 256);
    for (; u < u1; u += 4 * 256) {
        int64_t off[4];
        bool in[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            off[k] = w.offset<VEC ? 4 : 1>();
            in[k] = u + k * 256 < u1;
            w.next();
        }
        f(off, in);
    }
}

// Sums of N doubles over a workgroup of NT threads, in every thread (fixed
// order).  `lds`: N * NT / 64 doubles.
template <int NT, int N>
__device__ __forceinline__ void block_sums_all(double (&v)[N], double* lds) {
    constexpr int NW = NT / 64;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] += __shfl_xor(v[i], off, 64);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int i = 0; i < N; ++i) lds[i * NW + (threadIdx.x >> 6)] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = lds[i * NW];
#pragma unroll
        for (int w = 1; w < NW; ++w) v[i] += lds[i * NW + w];
    }
}

// Cached loads: the apply pass reads x again right after, and for a tensor
// of a few tens of MiB part of that re-read then comes from the caches
// (measured: a re-read of 64 MiB 2-15 % faster, of 192 MiB no faster).
template <bool VEC>
__global__ void __launch_bounds__(256) bn_stats_kernel(const float* __restrict__ x, BnGeom gm,
                                                        double* __restrict__ part) {
    __shared__ double lds[4];
    double s = 0.0, q = 0.0;
    bn_for_chunk<VEC>(gm, [&](const int64_t(&off)[4], const bool(&in)[4]) {
        if (VEC) {
            float4 v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[k] = in[k] ? *reinterpret_cast<const float4*>(x + off[k]) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double a = v[k].x, b = v[k].y, cc = v[k].z, d = v[k].w;
                s += (a + b) + (cc + d);
                q += (a * a + b * b) + (cc * cc + d * d);
            }
        } else {
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = in[k] ? x[off[k]] : 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double a = v[k];
                s += a;
                q += a * a;
            }
        }
    });
    s = block_sum_d256(s, lds);
    q = block_sum_d256(q, lds);
    if (threadIdx.x == 0) {
        double* o = part + ((int64_t)blockIdx.y * gm.chunks + blockIdx.x) * 2;
        o[0] = s;
        o[1] = q;
    }
}

// Channel c's statistics: the chunk partials combined in order, then the
// reference's float arithmetic for the running statistics and 1/std.  With
// `update`, the running statistics and the saved mean / 1/std are written.
struct BnStats {
    const double* part;
    int64_t chunks;
    int64_t n;
    float eps, momentum;
    int training;
    float* running_mean;
    float* running_var;
    float* mean_out;
    float* inv_out;
};

// From a channel's sums (s = sum(x), q = sum(x^2)); `update` in one thread.
__device__ __forceinline__ float2 bn_stats_of(const BnStats& a, int64_t c, double s, double q, bool update) {
#pragma clang fp contract(off)
    float mean, var;
    if (a.training) {
        const double md = s / (double)a.n;
        const double m2 = q - s * md;
        mean = (float)md;
        var = (float)((m2 > 0.0 ? m2 : 0.0) / (double)a.n);
        if (update) {
            a.running_mean[c] = (1.0f - a.momentum) * a.running_mean[c] + a.momentum * mean;
            a.running_var[c] = (1.0f - a.momentum) * a.running_var[c] + a.momentum * var;
        }
    } else {
        mean = a.running_mean[c];
        var = a.running_var[c];
    }
    const float inv = 1.0f / sqrtf(var + a.eps);
    if (update) {
        a.mean_out[c] = mean;
        a.inv_out[c] = inv;
    }
    return make_float2(mean, inv);
}

// Sum of N doubles per chunk over a channel's chunks, by a whole wave (every
// lane gets the totals): lane l takes chunks l, l + 64, ..., then the lanes
// combine in a fixed order.
template <int N>
__device__ __forceinline__ void bn_wave_sums(const double* part, int64_t c, int64_t chunks, double (&t)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = 0.0;
    for (int64_t k = threadIdx.x & 63; k < chunks; k += 64)
#pragma unroll
        for (int i = 0; i < N; ++i) t[i] += part[(c * chunks + k) * N + i];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int i = 0; i < N; ++i) t[i] += __shfl_xor(t[i], off, 64);
}

// Called by every lane of one wave; lane 0 updates.
__device__ __forceinline__ float2 bn_channel_stats(const BnStats& a, int64_t c, bool update) {
    double t[2] = {0.0, 0.0};
    if (a.training) bn_wave_sums(a.part, c, a.chunks, t);
    return bn_stats_of(a, c, t[0], t[1], update && (threadIdx.x & 63) == 0);
}

// One wave per channel (the statistics alone, when no output is wanted).
__global__ void __launch_bounds__(64) bn_stats_finalize_kernel(BnStats a) {
    (void)bn_channel_stats(a, blockIdx.x, true);
}

// Each workgroup combines its channel's partials itself (chunk 0's also
// writes the running and saved statistics): no finalize launch between the
// two passes.
template <bool VEC>
__global__ void __launch_bounds__(256) bn_apply_kernel(const float* __restrict__ x, const float* __restrict__ gamma,
                                                        const float* __restrict__ beta, BnStats sa, BnGeom gm,
                                                        float* __restrict__ y) {
    const int64_t c = blockIdx.y;
    __shared__ float2 s_mi;
    if (threadIdx.x < 64) {
        const float2 mi = bn_channel_stats(sa, c, blockIdx.x == 0);
        if (threadIdx.x == 0) s_mi = mi;
    }
    __syncthreads();
    const float gc = gamma[c], bc = beta[c], mc = s_mi.x, ic = s_mi.y;
    auto nrm = [&](float v) { return gc * ((v - mc) * ic) + bc; };
    bn_for_chunk<VEC>(gm, [&](const int64_t(&off)[4], const bool(&in)[4]) {
        if (VEC) {
            float4 v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) v[k] = ld_stream(x + off[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k])
                    st_stream(y + off[k], make_float4(nrm(v[k].x), nrm(v[k].y), nrm(v[k].z), nrm(v[k].w)));
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) st_stream1(y + off[k], nrm(ld_stream1(x + off[k])));
            }
        }
    });
}

// Backward sums per chunk: sum(g), sum(g (x - mean)), sum(x - mean), with
// x - mean in float as the closure computes it (cached loads, as in
// bn_stats_kernel: the dx pass re-reads g and x).
template <bool VEC>
__global__ void __launch_bounds__(256) bn_bwd_sums_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                           const float* __restrict__ mean, BnGeom gm,
                                                           double* __restrict__ part) {
    __shared__ double lds[4];
    const float mc = mean[blockIdx.y];
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
    bn_for_chunk<VEC>(gm, [&](const int64_t(&off)[4], const bool(&in)[4]) {
        if (VEC) {
            float4 gv[4], xv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                gv[k] = in[k] ? *reinterpret_cast<const float4*>(g + off[k]) : make_float4(0.f, 0.f, 0.f, 0.f);
                xv[k] = in[k] ? *reinterpret_cast<const float4*>(x + off[k]) : make_float4(mc, mc, mc, mc);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float d0 = xv[k].x - mc, d1 = xv[k].y - mc, d2 = xv[k].z - mc, d3 = xv[k].w - mc;
                s1 += ((double)gv[k].x + (double)gv[k].y) + ((double)gv[k].z + (double)gv[k].w);
                s2 += ((double)gv[k].x * d0 + (double)gv[k].y * d1) + ((double)gv[k].z * d2 + (double)gv[k].w * d3);
                s3 += ((double)d0 + (double)d1) + ((double)d2 + (double)d3);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) {
                    const float gv = g[off[k]], d = x[off[k]] - mc;
                    s1 += gv;
                    s2 += (double)gv * d;
                    s3 += d;
                }
            }
        }
    });
    s1 = block_sum_d256(s1, lds);
    s2 = block_sum_d256(s2, lds);
    s3 = block_sum_d256(s3, lds);
    if (threadIdx.x == 0) {
        double* o = part + ((int64_t)blockIdx.y * gm.chunks + blockIdx.x) * 3;
        o[0] = s1;
        o[1] = s2;
        o[2] = s3;
    }
}

// Channel c's backward coefficients from the chunk sums: the closure's
// dvar, dmean; with `update`, dgamma and dbeta (accumulated as requested).
struct BnBwdCoef {
    const double* part;
    int64_t chunks;
    int64_t n;
    const float* gamma;
    const float* inv_std;
    float* dgamma;
    int acc_gamma;
    float* dbeta;
    int acc_beta;
};

// From a channel's sums s1 = sum(g), s2 = sum(g (x - mean)), s3 = sum(x - mean).
__device__ __forceinline__ float2 bn_coef_of(const BnBwdCoef& a, int64_t c, double s1, double s2, double s3,
                                             bool update) {
    const double iv = a.inv_std[c], gm = a.gamma[c];
    if (update && a.dgamma) {
        const float dg = (float)(s2 * iv);
        a.dgamma[c] = a.acc_gamma ? a.dgamma[c] + dg : dg;
    }
    if (update && a.dbeta) {
        const float db = (float)s1;
        a.dbeta[c] = a.acc_beta ? a.dbeta[c] + db : db;
    }
    const float dvar = (float)(gm * s2 * -0.5 * iv * iv * iv);
    const float dmean = (float)(-gm * iv * s1 + (double)dvar * (-2.0 * s3) / (double)a.n);
    return make_float2(dvar, dmean);
}

// Called by every lane of one wave; lane 0 updates.
__device__ __forceinline__ float2 bn_channel_coef(const BnBwdCoef& a, int64_t c, bool update) {
    double t[3];
    bn_wave_sums(a.part, c, a.chunks, t);
    return bn_coef_of(a, c, t[0], t[1], t[2], update && (threadIdx.x & 63) == 0);
}

// One wave per channel: dgamma, dbeta when no input gradient is wanted.
__global__ void __launch_bounds__(64) bn_bwd_finalize_kernel(BnBwdCoef a) {
    (void)bn_channel_coef(a, blockIdx.x, true);
}

// Each workgroup combines its channel's sums itself (chunk 0's also writes
// dgamma / dbeta): no finalize launch between the two passes.
template <bool VEC>
__global__ void __launch_bounds__(256) bn_bwd_apply_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                            const float* __restrict__ gamma,
                                                            const float* __restrict__ mean,
                                                            const float* __restrict__ inv_std, BnBwdCoef ca,
                                                            BnGeom gm, float nf, float* __restrict__ gx, int acc) {
    const int64_t c = blockIdx.y;
    __shared__ float2 s_cf;
    if (threadIdx.x < 64) {
        const float2 cf = bn_channel_coef(ca, c, blockIdx.x == 0);
        if (threadIdx.x == 0) s_cf = cf;
    }
    __syncthreads();
    const float gc = gamma[c], mc = mean[c], ic = inv_std[c];
    const float2 cf = s_cf;
    const float dm = cf.y / nf;
    auto dx = [&](float gv, float xv) { return gv * gc * ic + cf.x * 2.0f * (xv - mc) / nf + dm; };
    bn_for_chunk<VEC>(gm, [&](const int64_t(&off)[4], const bool(&in)[4]) {
        if (VEC) {
            float4 gv[4], xv[4], ov[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) {
                    gv[k] = ld_stream(g + off[k]);
                    xv[k] = ld_stream(x + off[k]);
                    if (acc) ov[k] = ld_stream(gx + off[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) {
                    float4 d = make_float4(dx(gv[k].x, xv[k].x), dx(gv[k].y, xv[k].y), dx(gv[k].z, xv[k].z),
                                           dx(gv[k].w, xv[k].w));
                    if (acc) d = make_float4(ov[k].x + d.x, ov[k].y + d.y, ov[k].z + d.z, ov[k].w + d.w);
                    st_stream(gx + off[k], d);
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (in[k]) {
                    float d = dx(ld_stream1(g + off[k]), ld_stream1(x + off[k]));
                    if (acc) d = ld_stream1(gx + off[k]) + d;
                    st_stream1(gx + off[k], d);
                }
            }
        }
    });
}

// ---- a channel in one workgroup's registers -----------------------------------
//
// NU units per thread.  One read of each input and one launch, where the two
// passes read them twice: [64, 256, 14, 14] forward and backward 72 us before
// (two passes, one plane per step), 29.5 with the walk above alone, 20.3 so.
// Bound by HBM (or the caches) and, at small channels, by the latency of one load,
// two barriers and one store.
template <int NT, int NU, bool VEC>
__global__ void __launch_bounds__(NT) bn_fwd_channel_kernel(const float* __restrict__ x,
                                                             const float* __restrict__ gamma,
                                                             const float* __restrict__ beta, BnStats sa, BnGeom gm,
                                                             float* __restrict__ y) {
    constexpr int W = VEC ? 4 : 1;
    __shared__ double lds[2 * NT / 64];
    const int64_t c = blockIdx.x;
    float v[NU][W];
    BnWalk w(gm, c, threadIdx.x, NT);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const bool in = (int64_t)k * NT + threadIdx.x < gm.total;
        const int64_t off = w.offset<W>();
        if constexpr (VEC) {
            const float4 q = in ? ld_stream(x + off) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[k][0] = q.x; v[k][1] = q.y; v[k][2] = q.z; v[k][3] = q.w;
        } else {
            v[k][0] = in ? ld_stream1(x + off) : 0.f;
        }
        w.next();
    }
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NU; ++k)
#pragma unroll
        for (int e = 0; e < W; ++e) {
            const double a = v[k][e];
            s[0] += a;
            s[1] += a * a;
        }
    block_sums_all<NT>(s, lds);
    const float2 mi = bn_stats_of(sa, c, s[0], s[1], threadIdx.x == 0);
    const float gc = gamma[c], bc = beta[c], mc = mi.x, ic = mi.y;
    BnWalk o(gm, c, threadIdx.x, NT);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const bool in = (int64_t)k * NT + threadIdx.x < gm.total;
        const int64_t off = o.offset<W>();
        float r[W];
#pragma unroll
        for (int e = 0; e < W; ++e) r[e] = gc * ((v[k][e] - mc) * ic) + bc;
        if constexpr (VEC) { if (in) st_stream(y + off, make_float4(r[0], r[1], r[2], r[3])); }
        else { if (in) st_stream1(y + off, r[0]); }
        o.next();
    }
}

template <int NT, int NU, bool VEC>
__global__ void __launch_bounds__(NT) bn_bwd_channel_kernel(const float* __restrict__ g, const float* __restrict__ x,
                                                             const float* __restrict__ mean, BnBwdCoef ca, BnGeom gm,
                                                             float nf, float* __restrict__ gx, int acc) {
    constexpr int W = VEC ? 4 : 1;
    __shared__ double lds[3 * NT / 64];
    const int64_t c = blockIdx.x;
    const float mc = mean[c];
    float gv[NU][W], d[NU][W];  // g, x - mean
    BnWalk w(gm, c, threadIdx.x, NT);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const bool in = (int64_t)k * NT + threadIdx.x < gm.total;
        const int64_t off = w.offset<W>();
        if constexpr (VEC) {
            const float4 a = in ? ld_stream(g + off) : make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 b = in ? ld_stream(x + off) : make_float4(mc, mc, mc, mc);
            gv[k][0] = a.x; gv[k][1] = a.y; gv[k][2] = a.z; gv[k][3] = a.w;
            d[k][0] = b.x; d[k][1] = b.y; d[k][2] = b.z; d[k][3] = b.w;
        } else {
            gv[k][0] = in ? ld_stream1(g + off) : 0.f;
            d[k][0] = in ? ld_stream1(x + off) : mc;
        }
        w.next();
    }
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NU; ++k)
#pragma unroll
        for (int e = 0; e < W; ++e) {
            d[k][e] -= mc;
            s[0] += (double)gv[k][e];
            s[1] += (double)gv[k][e] * d[k][e];
            s[2] += (double)d[k][e];
        }
    block_sums_all<NT>(s, lds);
    const float2 cf = bn_coef_of(ca, c, s[0], s[1], s[2], threadIdx.x == 0);
    if (!gx) return;
    const float gc = ca.gamma[c], ic = ca.inv_std[c], dm = cf.y / nf;
    BnWalk o(gm, c, threadIdx.x, NT);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const bool in = (int64_t)k * NT + threadIdx.x < gm.total;
        const int64_t off = o.offset<W>();
        float r[W];
#pragma unroll
        for (int e = 0; e < W; ++e) r[e] = gv[k][e] * gc * ic + cf.x * 2.0f * d[k][e] / nf + dm;
        if (in) {
            if constexpr (VEC) {
                if (acc) {
                    const float4 p = ld_stream(gx + off);
                    r[0] = p.x + r[0]; r[1] = p.y + r[1]; r[2] = p.z + r[2]; r[3] = p.w + r[3];
                }
                st_stream(gx + off, make_float4(r[0], r[1], r[2], r[3]));
            } else {
                if (acc) r[0] = ld_stream1(gx + off) + r[0];
                st_stream1(gx + off, r[0]);
            }
        }
        o.next();
    }
}

// The register tile for a channel of `total` units: 256 threads up to 4 units
// each, else 1024; 0 units when it does not fit (more than 4 float4s or 8
// floats per thread: with twice as many the backward spills, and takes 37 us
// against 11 for the two passes at [40, 64, 28, 28]).
struct BnTile {
    int nt = 0, nu = 0;
};

BnTile bn_tile(int64_t total, bool vec) {
    for (int nu : {1, 2, 4})
        if (total <= 256 * nu) return {256, nu};
    for (int nu : {2, 4, 8})
        if (total <= 1024 * nu && (!vec || nu <= 4)) return {1024, nu};
    return {};
}

#define WM_BN_TILES(CASE)                                                                       \
    CASE(256, 1, true) CASE(256, 2, true) CASE(256, 4, true) CASE(1024, 2, true)                 \
    CASE(1024, 4, true) CASE(256, 1, false) CASE(256, 2, false) CASE(256, 4, false)              \
    CASE(1024, 2, false) CASE(1024, 4, false) CASE(1024, 8, false)

// ---------------------------------------------------------------------------
// Attention softmax
// ---------------------------------------------------------------------------

template <int NT, int ITEMS, bool VEC>
__global__ void __launch_bounds__(NT) attn_softmax_fwd_kernel(const float* __restrict__ scores,
                                                               const float* __restrict__ mask, int64_t mask_bstride,
                                                               int64_t heads_tq, int64_t tq, int64_t rows, int64_t tk,
                                                               float* __restrict__ attn) {
    using Tile = RowTile<NT, ITEMS, VEC>;
    __shared__ float lds_m[NT / 64], lds_s[NT / 64];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        Tile t;
        t.load(scores + r * tk, tk, -INFINITY);
        if (mask) {
            const int64_t b = r / heads_tq, i = r % tq;
            Tile mt;
            mt.template load<true>(mask + b * mask_bstride + i * tk, tk, 0.f);
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) t.v[k][e] = t.v[k][e] + mt.v[k][e];
        }
        float mx = -INFINITY;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) mx = fmaxf(mx, t.v[k][e]);
        // max_val starts at -FLT_MAX (core/layer.cpp:1215); std::max skips NaN like fmaxf
        const float m = fmaxf(block_max_1<NT>(mx, lds_m), -FLT_MAX);
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                t.v[k][e] = exp_rr(t.v[k][e] - m);  // padding: exp(-inf) = 0
                s += t.v[k][e];
            }
        const float rs = 1.0f / block_sum_1<NT>(s, lds_s);
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) t.v[k][e] = t.v[k][e] * rs;
        t.store(attn + r * tk, tk);
    }
}

template <int NT, int ITEMS, bool VEC>
__global__ void __launch_bounds__(NT) attn_softmax_bwd_kernel(const float* __restrict__ attn,
                                                               const float* __restrict__ da, int64_t rows, int64_t tk,
                                                               float* __restrict__ ds) {
    using Tile = RowTile<NT, ITEMS, VEC>;
    __shared__ float lds[2][NT / 64];
    int k2 = 0;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x, ++k2) {
        Tile a, d;
        a.load(attn + r * tk, tk, 0.f);
        d.load(da + r * tk, tk, 0.f);
        float dot = 0.f;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) dot += a.v[k][e] * d.v[k][e];
        dot = block_sum_1<NT>(dot, lds[k2 & 1]);
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) d.v[k][e] = a.v[k][e] * (d.v[k][e] - dot);
        d.store(ds + r * tk, tk);
    }
}

// Rows longer than the register tile.
__global__ void __launch_bounds__(1024) attn_softmax_fwd_long_kernel(const float* __restrict__ scores,
                                                                      const float* __restrict__ mask,
                                                                      int64_t mask_bstride, int64_t heads_tq,
                                                                      int64_t tq, int64_t rows, int64_t tk,
                                                                      float* __restrict__ attn) {
    __shared__ float lds_m[16], lds_s[16];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float* sr = scores + r * tk;
        const float* mr = mask ? mask + (r / heads_tq) * mask_bstride + (r % tq) * tk : nullptr;
        float* ar = attn + r * tk;
        float mx = -INFINITY;
        for (int64_t c = threadIdx.x; c < tk; c += 1024) mx = fmaxf(mx, mr ? sr[c] + mr[c] : sr[c]);
        const float m = fmaxf(block_max_1<1024>(mx, lds_m), -FLT_MAX);
        float s = 0.f;
        for (int64_t c = threadIdx.x; c < tk; c += 1024) {
            const float e = exp_rr((mr ? sr[c] + mr[c] : sr[c]) - m);
            ar[c] = e;
            s += e;
        }
        const float rs = 1.0f / block_sum_1<1024>(s, lds_s);
        for (int64_t c = threadIdx.x; c < tk; c += 1024) ar[c] = ar[c] * rs;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(1024) attn_softmax_bwd_long_kernel(const float* __restrict__ attn,
                                                                      const float* __restrict__ da, int64_t rows,
                                                                      int64_t tk, float* __restrict__ ds) {
    __shared__ float lds[2][16];
    int k2 = 0;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x, ++k2) {
        const float* ar = attn + r * tk;
        const float* dr = da + r * tk;
        float dot = 0.f;
        for (int64_t c = threadIdx.x; c < tk; c += 1024) dot += ar[c] * dr[c];
        dot = block_sum_1<1024>(dot, lds[k2 & 1]);
        for (int64_t c = threadIdx.x; c < tk; c += 1024) ds[r * tk + c] = ar[c] * (dr[c] - dot);
    }
}

// ---------------------------------------------------------------------------
// Dropout mask
// ---------------------------------------------------------------------------

// splitmix64 (Vigna): one 64-bit state step, a bijective mix of the counter.
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void __launch_bounds__(256) dropout_mask_kernel(float* __restrict__ mask, int64_t n, float p, float scale,
                                                            uint64_t seed) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float u = (float)(uint32_t)(splitmix64(seed + (uint64_t)i) >> 40) * 0x1p-24f;
        mask[i] = u > p ? scale : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------

// LayerNorm register tiles: a wave with up to 4 float4s per lane (1024
// columns), else 256 or 1024 threads with up to 2; rows over 8192 elements
// take the streaming path (nt == 0).
TileChoice ln_tile(int64_t n) {
    TileChoice t;
    const int nts[3] = {64, 256, 1024};
    for (int nt : nts)
        for (int items = 1; items <= (nt == 64 ? 4 : 2); ++items)
            if (n <= (int64_t)nt * 4 * items) {
                t.nt = nt;
                t.items = items;
                return t;
            }
    return t;
}

int ln_waves(int nt) { return nt == 64 ? 16 : nt == 256 ? 4 : 2; }  // workgroups per CU in the grid

int launch_ln_fwd(const float* x, const float* gamma, const float* beta, int64_t rows, int64_t n, float eps,
                  float* y, float* mean, float* inv) {
    hipStream_t st = stream();
    const TileChoice tc = ln_tile(n);
    const bool vec = n % 4 == 0 && aligned16(x) && aligned16(y) && aligned16(gamma) && aligned16(beta);
    if (tc.nt == 0) {
        dim3 grid((unsigned)std::min<int64_t>(rows, (int64_t)num_cus() * 2));
        launch_kernel(ln_fwd_long_kernel, grid, dim3(1024), 0, st, x, gamma, beta, rows, n, eps, y, mean, inv);
        return check_launch("wm_layernorm_fwd(long)");
    }
    dim3 grid((unsigned)std::min<int64_t>(rows, (int64_t)num_cus() * ln_waves(tc.nt) * 2));
#define WM_LNF(NTv, IT)                                                                                         \
    if (tc.nt == NTv && tc.items == IT) {                                                                       \
        if (vec)                                                                                                \
            launch_kernel((ln_fwd_kernel<NTv, IT, true>), grid, dim3(NTv), 0, st, x, gamma, beta, rows, n, \
                               eps, y, mean, inv);                                                              \
        else                                                                                                    \
            launch_kernel((ln_fwd_kernel<NTv, IT, false>), grid, dim3(NTv), 0, st, x, gamma, beta, rows,   \
                               n, eps, y, mean, inv);                                                           \
        return check_launch("wm_layernorm_fwd");                                                                \
    }
    WM_LNF(64, 1) WM_LNF(64, 2) WM_LNF(64, 3) WM_LNF(64, 4) WM_LNF(256, 2) WM_LNF(1024, 1) WM_LNF(1024, 2)
#undef WM_LNF
    return set_error(WM_ERR_INVALID, "wm_layernorm_fwd: no tile");
}

int launch_ln_bwd(const float* g, const float* x, const float* gamma, const float* mean, const float* inv,
                  int64_t rows, int64_t n, float* gx, int acc_x, float* dgamma, int acc_g, float* dbeta, int acc_b) {
    hipStream_t st = stream();
    const TileChoice tc = ln_tile(n);
    const bool want_p = dgamma || dbeta;
    if (tc.nt == 0) {
        if (gx) {
            dim3 grid((unsigned)std::min<int64_t>(rows, (int64_t)num_cus() * 2));
            launch_kernel(ln_bwd_long_kernel, grid, dim3(1024), 0, st, g, x, gamma, mean, inv, rows, n, gx,
                               acc_x);
            WM_TRY(check_launch("wm_layernorm_bwd(long)"));
        }
        if (!want_p) return WM_OK;
        const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(rows / 64, 256));
        const int64_t rpc = (rows + chunks - 1) / chunks;
        Workspace wg(dgamma ? (size_t)(chunks * n) * sizeof(float) : 0);
        Workspace wb(dbeta ? (size_t)(chunks * n) * sizeof(float) : 0);
        if ((dgamma && !wg.p) || (dbeta && !wb.p)) return set_error(WM_ERR_NOMEM, "wm_layernorm_bwd: workspace");
        launch_kernel(ln_param_parts_kernel, dim3((unsigned)((n + 255) / 256), (unsigned)chunks), dim3(256), 0,
                           st, g, x, mean, inv, rows, n, rpc, wg.as<float>(), wb.as<float>());
        WM_TRY(check_launch("wm_layernorm_bwd(params)"));
        return colsum_parts(dgamma ? wg.as<float>() : nullptr, dgamma, acc_g, dbeta ? wb.as<float>() : nullptr,
                            dbeta, acc_b, chunks, n, "wm_layernorm_bwd(colsum)");
    }
    // Fused path: G workgroups, each leaving one [n] partial per parameter
    // gradient.  With parameter gradients a wave-per-row workgroup takes at
    // least 8 rows (two per wave) and the grid stops at one workgroup per CU
    // (four for rows of one float4 per lane, which keep fewer bytes in
    // flight): [8192, 768] 17.3 + 4.5 us for the two dispatches, against 16.7 + 6.2
    // at two per CU and 17.2 + 9.8 at four; [32768, 128] 12.9 + 4.4 at four
    // against 27.9 + 4.5 at one.  Wider rows: at least 8 rows per workgroup, or 4
    // when there are few (32 rows each: [768, 8192] 83 us against 28), on at most
    // two workgroups per CU, one for rows of two float4s per thread of 1024 (more
    // leave more partials to write and read than they hide: [16384, 2048] 89.5
    // us at 8 per CU, 71.4 at two; [8192, 4096] 84.1 at four, 76.9; [8192, 8192]
    // 169 at four, 152 at two, 145 at one).
    const bool wave = tc.nt == 64;
    const int per_cu = !want_p ? (wave ? 4 : ln_waves(tc.nt) * 2)
                       : wave  ? (tc.items > 1 ? 1 : 4)
                               : (tc.nt == 1024 && tc.items > 1 ? 1 : 2);
    int64_t G = std::min<int64_t>(wave ? (rows + 3) / 4 : rows, (int64_t)num_cus() * per_cu);
    const int64_t least = wave || rows >= 1024 ? 8 : 4;
    if (want_p) G = std::max<int64_t>(1, std::min<int64_t>(G, (rows + least - 1) / least));
    Workspace wg(dgamma ? (size_t)(G * n) * sizeof(float) : 0);
    Workspace wb(dbeta ? (size_t)(G * n) * sizeof(float) : 0);
    if ((dgamma && !wg.p) || (dbeta && !wb.p)) return set_error(WM_ERR_NOMEM, "wm_layernorm_bwd: workspace");
    const bool vec = n % 4 == 0 && aligned16(g) && aligned16(x) && aligned16(gamma) && (!gx || aligned16(gx));
    dim3 grid((unsigned)G);
    bool launched = false;
#define WM_LNB(NTv, IT)                                                                                         \
    if (!launched && tc.nt == NTv && tc.items == IT) {                                                          \
        if (vec)                                                                                                \
            launch_kernel((ln_bwd_kernel<NTv, IT, true>), grid, dim3(NTv), 0, st, g, x, gamma, mean, inv,  \
                               rows, n, gx, acc_x, wg.as<float>(), wb.as<float>());                             \
        else                                                                                                    \
            launch_kernel((ln_bwd_kernel<NTv, IT, false>), grid, dim3(NTv), 0, st, g, x, gamma, mean, inv, \
                               rows, n, gx, acc_x, wg.as<float>(), wb.as<float>());                             \
        launched = true;                                                                                        \
    }
    WM_LNB(256, 2) WM_LNB(1024, 1) WM_LNB(1024, 2)
#undef WM_LNB
#define WM_LNW(IT)                                                                                                  \
    if (!launched && wave && tc.items == IT) {                                                                      \
        if (vec)                                                                                                    \
            launch_kernel((ln_bwd_wave_kernel<IT, true>), grid, dim3(256), 0, st, g, x, gamma, mean, inv, rows, n,  \
                          gx, acc_x, wg.as<float>(), wb.as<float>());                                               \
        else                                                                                                        \
            launch_kernel((ln_bwd_wave_kernel<IT, false>), grid, dim3(256), 0, st, g, x, gamma, mean, inv, rows, n, \
                          gx, acc_x, wg.as<float>(), wb.as<float>());                                               \
        launched = true;                                                                                            \
    }
    WM_LNW(1) WM_LNW(2) WM_LNW(3) WM_LNW(4)
#undef WM_LNW
    if (!launched) return set_error(WM_ERR_INVALID, "wm_layernorm_bwd: no tile");
    WM_TRY(check_launch("wm_layernorm_bwd"));
    return colsum_parts(dgamma ? wg.as<float>() : nullptr, dgamma, acc_g, dbeta ? wb.as<float>() : nullptr, dbeta,
                        acc_b, G, n, "wm_layernorm_bwd(colsum)");
}

// Workgroups per CU for a pass of two kernels: as many as both keep
// resident, at most 8, so the grid runs in one round (the backward's
// kernels hold 7 per CU: a grid of 8 per CU ran as 7 plus a one-per-CU
// tail, 178.7 against 164.2 us at [64, 256, 56, 56]).
template <class K1, class K2>
int bn_per_cu(K1 k1, K2 k2) {
    int a = 0, b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, k1, 256, 0) != hipSuccess || a < 1) a = 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k2, 256, 0) != hipSuccess || b < 1) b = 1;
    return std::min(8, std::min(a, b));
}

// per_cu: workgroups per CU the grid aims at.
BnGeom bn_geom(int64_t B, int64_t C, int64_t S, bool vec, int per_cu) {
    BnGeom gm;
    gm.C = C;
    gm.S = S;
    gm.units = std::max<int64_t>(1, vec ? S / 4 : S);
    gm.total = B * (vec ? S / 4 : S);
    const int64_t want = std::max<int64_t>(1, ((int64_t)num_cus() * per_cu + C - 1) / C);
    gm.per = std::max<int64_t>(kBnStep, ((gm.total + want - 1) / want + 63) / 64 * 64);
    gm.chunks = std::max<int64_t>(1, (gm.total + gm.per - 1) / gm.per);
    return gm;
}

int check_bn(int64_t B, int64_t C, int64_t S, const char* what) {
    if (B < 0 || C < 0 || S < 0) return set_error(WM_ERR_INVALID, std::string(what) + ": negative extent");
    if (C > 65535) return set_error(WM_ERR_UNSUPPORTED, std::string(what) + ": more than 65535 channels");
    return WM_OK;
}

}  // namespace
}  // namespace wm

using namespace wm;

extern "C" {

int wm_layernorm_fwd(const float* x, const float* gamma, const float* beta, int64_t rows, int64_t n, float eps,
                     float* y, float* mean, float* inv_std) {
    if (rows < 0 || n < 0) return set_error(WM_ERR_INVALID, "wm_layernorm_fwd: negative extent");
    if (rows == 0 || n == 0) return WM_OK;
    if (!x || !gamma || !beta || !y || !mean || !inv_std)
        return set_error(WM_ERR_INVALID, "wm_layernorm_fwd: null pointer");
    WM_CHECK_INIT();
    return launch_ln_fwd(x, gamma, beta, rows, n, eps, y, mean, inv_std);
}

int wm_layernorm_bwd(const float* g, const float* x, const float* gamma, const float* mean, const float* inv_std,
                     int64_t rows, int64_t n, float* gx, int acc_x, float* dgamma, int acc_gamma, float* dbeta,
                     int acc_beta) {
    if (rows < 0 || n < 0) return set_error(WM_ERR_INVALID, "wm_layernorm_bwd: negative extent");
    if (n == 0 || (!gx && !dgamma && !dbeta)) return WM_OK;
    if (rows == 0) {
        // no instances: the parameter gradients receive zero contributions
        WM_CHECK_INIT();
        if (dgamma && !acc_gamma) WM_TRY(wm_fill(dgamma, 0.0f, n));
        if (dbeta && !acc_beta) WM_TRY(wm_fill(dbeta, 0.0f, n));
        return WM_OK;
    }
    if (!g || !x || !gamma || !mean || !inv_std) return set_error(WM_ERR_INVALID, "wm_layernorm_bwd: null pointer");
    WM_CHECK_INIT();
    return launch_ln_bwd(g, x, gamma, mean, inv_std, rows, n, gx, acc_x, dgamma, acc_gamma, dbeta, acc_beta);
}

int wm_batchnorm2d_fwd(const float* x, const float* gamma, const float* beta, float* running_mean,
                       float* running_var, int64_t batch, int64_t channels, int64_t spatial, float eps,
                       float momentum, int training, float* y, float* mean, float* inv_std) {
    WM_TRY(check_bn(batch, channels, spatial, "wm_batchnorm2d_fwd"));
    if (channels == 0) return WM_OK;
    if (!gamma || !beta || !running_mean || !running_var || !mean || !inv_std)
        return set_error(WM_ERR_INVALID, "wm_batchnorm2d_fwd: null pointer");
    const int64_t n = batch * spatial;
    if (n > 0 && (!x || !y)) return set_error(WM_ERR_INVALID, "wm_batchnorm2d_fwd: null pointer");
    WM_CHECK_INIT();
    hipStream_t st = stream();
    const bool vec = spatial % 4 == 0 && aligned16(x) && aligned16(y);
    if (const BnTile tile = bn_tile(batch * (vec ? spatial / 4 : spatial), vec); training && n > 0 && tile.nu) {
        const BnGeom gm = bn_geom(batch, channels, spatial, vec, 1);
        const BnStats sa{nullptr, 0, n, eps, momentum, training, running_mean, running_var, mean, inv_std};
#define WM_BN_FWD(NT, NU, V)                                                                                     \
    if (tile.nt == NT && tile.nu == NU && vec == V)                                                              \
        launch_kernel((bn_fwd_channel_kernel<NT, NU, V>), dim3((unsigned)channels), dim3(NT), 0, st, x, gamma, beta, \
                      sa, gm, y);
        WM_BN_TILES(WM_BN_FWD)
#undef WM_BN_FWD
        return check_launch("wm_batchnorm2d_fwd(channel)");
    }
    const BnGeom gm = bn_geom(batch, channels, spatial, vec,
                              vec ? bn_per_cu(bn_stats_kernel<true>, bn_apply_kernel<true>)
                                  : bn_per_cu(bn_stats_kernel<false>, bn_apply_kernel<false>));
    Workspace part(training ? (size_t)(channels * gm.chunks) * 2 * sizeof(double) : 0);
    if (training && !part.p) return set_error(WM_ERR_NOMEM, "wm_batchnorm2d_fwd: workspace");
    const BnStats sa{part.as<double>(), gm.chunks, n, eps, momentum, training, running_mean, running_var, mean,
                     inv_std};
    if (n == 0) {  // no elements: the statistics of empty sums (the reference's 0 / 0)
        if (training) {
            launch_kernel(bn_stats_kernel<false>, dim3((unsigned)gm.chunks, (unsigned)channels), dim3(256), 0, st, x,
                          gm, part.as<double>());
            WM_TRY(check_launch("wm_batchnorm2d_fwd(stats)"));
        }
        launch_kernel(bn_stats_finalize_kernel, dim3((unsigned)channels), dim3(64), 0, st, sa);
        return check_launch("wm_batchnorm2d_fwd(finalize)");
    }
    const dim3 grid((unsigned)gm.chunks, (unsigned)channels);
    if (training) {
        if (vec) launch_kernel(bn_stats_kernel<true>, grid, dim3(256), 0, st, x, gm, part.as<double>());
        else launch_kernel(bn_stats_kernel<false>, grid, dim3(256), 0, st, x, gm, part.as<double>());
        WM_TRY(check_launch("wm_batchnorm2d_fwd(stats)"));
    }
    if (vec) launch_kernel(bn_apply_kernel<true>, grid, dim3(256), 0, st, x, gamma, beta, sa, gm, y);
    else launch_kernel(bn_apply_kernel<false>, grid, dim3(256), 0, st, x, gamma, beta, sa, gm, y);
    return check_launch("wm_batchnorm2d_fwd(apply)");
}

int wm_batchnorm2d_bwd(const float* g, const float* x, const float* gamma, const float* mean, const float* inv_std,
                       int64_t batch, int64_t channels, int64_t spatial, float* gx, int acc_x, float* dgamma,
                       int acc_gamma, float* dbeta, int acc_beta) {
    WM_TRY(check_bn(batch, channels, spatial, "wm_batchnorm2d_bwd"));
    if (channels == 0 || (!gx && !dgamma && !dbeta)) return WM_OK;
    if (!gamma || !mean || !inv_std) return set_error(WM_ERR_INVALID, "wm_batchnorm2d_bwd: null pointer");
    const int64_t n = batch * spatial;
    if (n > 0 && (!g || !x)) return set_error(WM_ERR_INVALID, "wm_batchnorm2d_bwd: null pointer");
    WM_CHECK_INIT();
    hipStream_t st = stream();
    const bool vec = spatial % 4 == 0 && aligned16(g) && aligned16(x) && (!gx || aligned16(gx));
    const float nf = (float)n;
    if (const BnTile tile = bn_tile(batch * (vec ? spatial / 4 : spatial), vec); n > 0 && tile.nu) {
        const BnGeom gm = bn_geom(batch, channels, spatial, vec, 1);
        const BnBwdCoef ca{nullptr, 0, n, gamma, inv_std, dgamma, acc_gamma, dbeta, acc_beta};
#define WM_BN_BWD(NT, NU, V)                                                                                    \
    if (tile.nt == NT && tile.nu == NU && vec == V)                                                             \
        launch_kernel((bn_bwd_channel_kernel<NT, NU, V>), dim3((unsigned)channels), dim3(NT), 0, st, g, x, mean, ca, \
                      gm, nf, gx, acc_x);
        WM_BN_TILES(WM_BN_BWD)
#undef WM_BN_BWD
        return check_launch("wm_batchnorm2d_bwd(channel)");
    }
    const BnGeom gm = bn_geom(batch, channels, spatial, vec,
                              vec ? bn_per_cu(bn_bwd_sums_kernel<true>, bn_bwd_apply_kernel<true>)
                                  : bn_per_cu(bn_bwd_sums_kernel<false>, bn_bwd_apply_kernel<false>));
    Workspace part((size_t)(channels * gm.chunks) * 3 * sizeof(double));
    if (!part.p) return set_error(WM_ERR_NOMEM, "wm_batchnorm2d_bwd: workspace");
    const BnBwdCoef ca{part.as<double>(), gm.chunks, n, gamma, inv_std, dgamma, acc_gamma, dbeta, acc_beta};
    const dim3 grid((unsigned)gm.chunks, (unsigned)channels);
    if (vec) launch_kernel(bn_bwd_sums_kernel<true>, grid, dim3(256), 0, st, g, x, mean, gm, part.as<double>());
    else launch_kernel(bn_bwd_sums_kernel<false>, grid, dim3(256), 0, st, g, x, mean, gm, part.as<double>());
    WM_TRY(check_launch("wm_batchnorm2d_bwd(sums)"));
    if (!gx || n == 0) {  // the parameter gradients alone
        launch_kernel(bn_bwd_finalize_kernel, dim3((unsigned)channels), dim3(64), 0, st, ca);
        return check_launch("wm_batchnorm2d_bwd(finalize)");
    }
    if (vec)
        launch_kernel(bn_bwd_apply_kernel<true>, grid, dim3(256), 0, st, g, x, gamma, mean, inv_std, ca, gm, nf, gx,
                      acc_x);
    else
        launch_kernel(bn_bwd_apply_kernel<false>, grid, dim3(256), 0, st, g, x, gamma, mean, inv_std, ca, gm, nf, gx,
                      acc_x);
    return check_launch("wm_batchnorm2d_bwd(apply)");
}

int wm_attention_softmax_fwd(const float* scores, const float* mask, int64_t mask_batches, int64_t batch,
                             int64_t heads, int64_t tq, int64_t tk, float* attn) {
    if (batch < 0 || heads < 0 || tq < 0 || tk < 0)
        return set_error(WM_ERR_INVALID, "wm_attention_softmax_fwd: negative extent");
    if (mask && mask_batches != 1 && mask_batches != batch)
        return set_error(WM_ERR_INVALID, "wm_attention_softmax_fwd: mask batch must be 1 or the batch size");
    const int64_t rows = batch * heads * tq;
    if (rows == 0 || tk == 0) return WM_OK;
    if (!scores || !attn) return set_error(WM_ERR_INVALID, "wm_attention_softmax_fwd: null pointer");
    WM_CHECK_INIT();
    hipStream_t st = stream();
    const int64_t mstride = mask_batches == 1 ? 0 : tq * tk;
    const TileChoice tc = choose_tile(tk);
    const bool vec = tk % 4 == 0 && aligned16(scores) && aligned16(attn) && (!mask || aligned16(mask));
    // One row per workgroup on a grid that covers every row: 68.4 -> 75.7 %
    // of the HBM peak at [8, 16, 1024, 1024] (backward 66.5 -> 79.6 %)
    // against 32 one-wave workgroups per CU looping over rows.
    dim3 grid((unsigned)std::min<int64_t>(rows, (int64_t)num_cus() * (1 << 12)));
    if (tc.nt == 0) {
        launch_kernel(attn_softmax_fwd_long_kernel, grid, dim3(1024), 0, st, scores, mask, mstride, heads * tq,
                           tq, rows, tk, attn);
        return check_launch("wm_attention_softmax_fwd(long)");
    }
#define WM_ASF(NTv, IT)                                                                                          \
    if (tc.nt == NTv && tc.items == IT) {                                                                        \
        if (vec)                                                                                                 \
            launch_kernel((attn_softmax_fwd_kernel<NTv, IT, true>), grid, dim3(NTv), 0, st, scores, mask,   \
                               mstride, heads * tq, tq, rows, tk, attn);                                         \
        else                                                                                                     \
            launch_kernel((attn_softmax_fwd_kernel<NTv, IT, false>), grid, dim3(NTv), 0, st, scores, mask,  \
                               mstride, heads * tq, tq, rows, tk, attn);                                         \
        return check_launch("wm_attention_softmax_fwd");                                                         \
    }
    WM_ASF(64, 1) WM_ASF(64, 2) WM_ASF(64, 4) WM_ASF(64, 8)
    WM_ASF(1024, 1) WM_ASF(1024, 2) WM_ASF(1024, 4) WM_ASF(1024, 8)
#undef WM_ASF
    return set_error(WM_ERR_INVALID, "wm_attention_softmax_fwd: no tile");
}

int wm_attention_softmax_bwd(const float* attn, const float* d_attn, int64_t rows, int64_t tk, float* d_scores) {
    if (rows < 0 || tk < 0) return set_error(WM_ERR_INVALID, "wm_attention_softmax_bwd: negative extent");
    if (rows == 0 || tk == 0) return WM_OK;
    if (!attn || !d_attn || !d_scores) return set_error(WM_ERR_INVALID, "wm_attention_softmax_bwd: null pointer");
    WM_CHECK_INIT();
    hipStream_t st = stream();
    const TileChoice tc = choose_tile(tk);
    const bool vec = tk % 4 == 0 && aligned16(attn) && aligned16(d_attn) && aligned16(d_scores);
    dim3 grid((unsigned)std::min<int64_t>(rows, (int64_t)num_cus() * (1 << 12)));  // as in the forward
    if (tc.nt == 0) {
        launch_kernel(attn_softmax_bwd_long_kernel, grid, dim3(1024), 0, st, attn, d_attn, rows, tk, d_scores);
        return check_launch("wm_attention_softmax_bwd(long)");
    }
#define WM_ASB(NTv, IT)                                                                                         \
    if (tc.nt == NTv && tc.items == IT) {                                                                       \
        if (vec)                                                                                                \
            launch_kernel((attn_softmax_bwd_kernel<NTv, IT, true>), grid, dim3(NTv), 0, st, attn, d_attn,  \
                               rows, tk, d_scores);                                                             \
        else                                                                                                    \
            launch_kernel((attn_softmax_bwd_kernel<NTv, IT, false>), grid, dim3(NTv), 0, st, attn, d_attn, \
                               rows, tk, d_scores);                                                             \
        return check_launch("wm_attention_softmax_bwd");                                                        \
    }
    WM_ASB(64, 1) WM_ASB(64, 2) WM_ASB(64, 4) WM_ASB(64, 8)
    WM_ASB(1024, 1) WM_ASB(1024, 2) WM_ASB(1024, 4) WM_ASB(1024, 8)
#undef WM_ASB
    return set_error(WM_ERR_INVALID, "wm_attention_softmax_bwd: no tile");
}

int wm_dropout_mask(float* mask, int64_t n, float p, uint64_t seed) {
    if (n < 0) return set_error(WM_ERR_INVALID, "wm_dropout_mask: negative size");
    if (n == 0) return WM_OK;
    if (!mask) return set_error(WM_ERR_INVALID, "wm_dropout_mask: null pointer");
    WM_CHECK_INIT();
    const float scale = 1.0f / (1.0f - p);  // core/layer.cpp:55
    launch_kernel(dropout_mask_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream(), mask, n, p, scale, seed);
    return check_launch("wm_dropout_mask");
}

}  // extern "C"
