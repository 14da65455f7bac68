// Multiresolution hash-grid encoder (drop-in for source/gridencoder/src/gridencoder.cu,
// bound in source/gridencoder/grid.py:54,84,194).
//
// Layout: one lane per (point, level) with the level fastest, so a wavefront
// writes a contiguous span of the [B, L*C] output (the reference writes
// [L, B, C] and permutes in Python, grid.py:57).  Table gathers read C
// contiguous features per corner (float2 / half2 for C = 2).  fp16 tables are
// interpolated in fp32 and rounded once on store; the adjoint accumulates into
// an fp32 gradient table (the reference accumulates fp16 with __half2 atomics).
// Index math is uint32 with wrap-around exactly as gridencoder.cu:50-84.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "n3ds_capi.h"
#include "n3ds_math.h"

namespace n3ds {

__device__ __forceinline__ uint32_t grid_hash(const uint32_t* pg, int D) {
    const uint32_t primes[7] = {1u, 2654435761u, 805459861u, 3674653429u, 2097192037u, 1434869437u, 2165219737u};
    uint32_t r = 0;
    for (int i = 0; i < D; i++) r ^= pg[i] * primes[i];
    return r;
}

template <int D>
__device__ __forceinline__ uint32_t grid_index(int gridtype, bool align, uint32_t hs, uint32_t res, const uint32_t* pg) {
    uint32_t stride = 1, index = 0;
#pragma unroll
    for (int d = 0; d < D; d++) {
        if (stride <= hs) {
            index += pg[d] * stride;
            stride *= align ? res : (res + 1);
        }
    }
    if (gridtype == 0 && stride > hs) {
        const uint32_t primes[7] = {1u, 2654435761u, 805459861u, 3674653429u, 2097192037u, 1434869437u, 2165219737u};
        index = 0;
#pragma unroll
        for (int d = 0; d < D; d++) index ^= pg[d] * primes[d];
    }
    return index % hs;
}

template <typename T>
__device__ __forceinline__ float to_f(T v);
template <>
__device__ __forceinline__ float to_f<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_f<__half>(__half v) { return __half2float(v); }
template <typename T>
__device__ __forceinline__ T from_f(float v);
template <>
__device__ __forceinline__ float from_f<float>(float v) { return v; }
template <>
__device__ __forceinline__ __half from_f<__half>(float v) { return __float2half(v); }

// keeps a float32 result from being folded with its conversion to half into one rounding
// (v_fma_mixlo_f16): results stay those of a float32 interpolation rounded once on store
__device__ __forceinline__ float rounded(float v) {
    asm volatile("" : "+v"(v));
    return v;
}

struct LevelCoord {
    uint32_t hs, res;
    float scale;
    bool oob;
};

constexpr int MAX_LEVELS = 64;
// Per-level grid scale exp2(level*S)*H - 1 (gridencoder.cu:138), evaluated once
// on the host with float32 operands and a correctly rounded exp2, so integer
// powers of two are exact.
struct LevelTab {
    float scale[MAX_LEVELS];
};

static LevelTab make_level_tab(int L, float S, int H) {
    LevelTab t;
    for (int l = 0; l < MAX_LEVELS; l++) {
        float ls = (float)l * S;
        float e = (float)exp2((double)ls);
        t.scale[l] = l < L ? (e * (float)H) - 1.0f : 0.f;
    }
    return t;
}

template <int D>
__device__ __forceinline__ LevelCoord level_coords(const float* in, int level, const int* offsets, const LevelTab& lt,
                                                   bool align, int interp, float* pos, float* deriv, uint32_t* pg) {
    LevelCoord lc;
    lc.oob = false;
#pragma unroll
    for (int d = 0; d < D; d++)
        if (in[d] < 0.f || in[d] > 1.f) lc.oob = true;
    lc.hs = (uint32_t)(offsets[level + 1] - offsets[level]);
    if (lc.hs == 0) lc.oob = true;  // empty level: nothing to gather (avoids a modulo by zero)
    lc.scale = lt.scale[level];
    lc.res = (uint32_t)ceilf(lc.scale) + 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
        // one rounding, as nvcc contracts the reference's x * scale + 0.5 (at the
        // finest levels the float32 ulp of pos is 1/16, so double rounding matters)
        float p = fmaf(in[d], lc.scale, align ? 0.0f : 0.5f);
        float f = floorf(p);
        pg[d] = (uint32_t)f;
        p -= f;
        if (interp == 1) {
            deriv[d] = 6.f * p * (1.f - p);
            p = p * p * (3.f - 2.f * p);
        } else {
            deriv[d] = 1.f;
        }
        pos[d] = p;
    }
    return lc;
}

template <typename T, int D, int C>
__global__ __launch_bounds__(256) void grid_fwd_kernel(const float* __restrict__ inputs, const T* __restrict__ grid,
                                                       const int* __restrict__ offsets, T* __restrict__ outputs,
                                                       int64_t B, int L, LevelTab lt, T* __restrict__ dy_dx,
                                                       int gridtype, int align, int interp) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= B * L) return;
    const int64_t b = tid / L;
    const int level = (int)(tid - b * L);
    const float* in = inputs + b * D;
    float pos[D], deriv[D];
    uint32_t pg[D];
    LevelCoord lc = level_coords<D>(in, level, offsets, lt, align != 0, interp, pos, deriv, pg);
    T* out = outputs + tid * C;
    if (lc.oob) {
#pragma unroll
        for (int c = 0; c < C; c++) out[c] = from_f<T>(0.f);
        if (dy_dx) {
            T* dd = dy_dx + b * (int64_t)L * D * C + (int64_t)level * D * C;
            for (int i = 0; i < D * C; i++) dd[i] = from_f<T>(0.f);
        }
        return;
    }
    const T* g = grid + (int64_t)offsets[level] * C;
    // every corner is gathered once: the slopes are differences of the same values (gathering
    // them again for each axis, 24 more for D = 3, took 630 of the 943 us of a forward and
    // adjoint with input gradients at 200003 points x 16 levels)
    float acc[C], val[1 << D][C];
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.f;
#pragma unroll
    for (int corner = 0; corner < (1 << D); corner++) {
        float w = 1.f;
        uint32_t loc[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (corner & (1 << d)) { w *= pos[d]; loc[d] = pg[d] + 1; }
            else { w *= 1.f - pos[d]; loc[d] = pg[d]; }
        }
        uint32_t idx = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc) * C;
#pragma unroll
        for (int c = 0; c < C; c++) {
            val[corner][c] = to_f<T>(g[idx + c]);
            acc[c] += w * val[corner][c];
        }
    }
#pragma unroll
    for (int c = 0; c < C; c++) out[c] = from_f<T>(rounded(acc[c]));
    if (dy_dx) {
        T* dd = dy_dx + b * (int64_t)L * D * C + (int64_t)level * D * C;
#pragma unroll
        for (int gd = 0; gd < D; gd++) {
            float rg[C];
#pragma unroll
            for (int c = 0; c < C; c++) rg[c] = 0.f;
#pragma unroll
            for (int corner = 0; corner < (1 << (D - 1)); corner++) {
                float w = lc.scale;
                int left = 0;  // the corner with the axis's bit clear
#pragma unroll
                for (int nd = 0; nd < D - 1; nd++) {
                    const int d = nd >= gd ? nd + 1 : nd;
                    if (corner & (1 << nd)) { w *= pos[d]; left |= 1 << d; }
                    else { w *= 1.f - pos[d]; }
                }
#pragma unroll
                for (int c = 0; c < C; c++) rg[c] += w * (val[left | (1 << gd)][c] - val[left][c]) * deriv[gd];
            }
#pragma unroll
            for (int c = 0; c < C; c++) dd[gd * C + c] = from_f<T>(rounded(rg[c]));
        }
    }
}

template <typename T, int D, int C>
__global__ __launch_bounds__(256) void grid_bwd_kernel(const T* __restrict__ grad, const float* __restrict__ inputs,
                                                       const int* __restrict__ offsets, float* __restrict__ ggrid,
                                                       int64_t B, int L, LevelTab lt, int gridtype, int align,
                                                       int interp) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= B * L) return;
    const int64_t b = tid / L;
    const int level = (int)(tid - b * L);
    const float* in = inputs + b * D;
    float pos[D], deriv[D];
    uint32_t pg[D];
    LevelCoord lc = level_coords<D>(in, level, offsets, lt, align != 0, interp, pos, deriv, pg);
    if (lc.oob) return;
    float gcur[C];
#pragma unroll
    for (int c = 0; c < C; c++) gcur[c] = to_f<T>(grad[tid * C + c]);
    float* gg = ggrid + (int64_t)offsets[level] * C;
#pragma unroll
    for (int corner = 0; corner < (1 << D); corner++) {
        float w = 1.f;
        uint32_t loc[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (corner & (1 << d)) { w *= pos[d]; loc[d] = pg[d] + 1; }
            else { w *= 1.f - pos[d]; loc[d] = pg[d]; }
        }
        uint32_t idx = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc) * C;
#pragma unroll
        for (int c = 0; c < C; c++) atomicAdd(gg + idx + c, w * gcur[c]);
    }
}

// ---------------------------------------------------------------------------
// Level-ordered forward / atomic adjoint: a block owns GT consecutive points,
// one lane per point, and walks the levels in order, so the blocks resident at
// one time gather from one or two level tables (an XCD's 4 MB L2 holds one fine
// level in fp32) instead of all of them.  The [GT, L*C] slab of the output (or
// of the upstream gradient) passes through LDS so that global memory sees
// whole rows; LDS rows are padded to L*C + 1 floats against bank conflicts.
// ---------------------------------------------------------------------------
constexpr int GT = 256;
constexpr int GT_MAX_LC = 63;  // LDS slab of GT * (63 + 1) floats = 64 KB

// Forward: the block's [GT, L*C] slab of outputs is assembled in LDS and written
// as whole rows.  The LDS slab (33 KB at 16 levels x 2 features) also keeps the
// number of resident blocks, and with it the number of levels gathered from at
// one time, low: measured faster than keeping 64-byte runs of the row in
// registers at twice the occupancy (0.73 vs 0.82 ms at 2^20 points, fp32).
template <typename T, int D, int C>
__device__ __forceinline__ void grid_level_acc(const float* in, int level, const int* __restrict__ offsets,
                                               const LevelTab& lt, const T* __restrict__ grid, int gridtype,
                                               int align, int interp, float* acc) {
    float pos[D], deriv[D];
    uint32_t pg[D];
    const LevelCoord lc = level_coords<D>(in, level, offsets, lt, align != 0, interp, pos, deriv, pg);
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.f;
    if (lc.oob) return;
    const T* g = grid + (int64_t)offsets[level] * C;
#pragma unroll
    for (int corner = 0; corner < (1 << D); corner++) {
        float w = 1.f;
        uint32_t loc[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (corner & (1 << d)) { w *= pos[d]; loc[d] = pg[d] + 1; }
            else { w *= 1.f - pos[d]; loc[d] = pg[d]; }
        }
        const uint32_t idx = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc) * C;
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] += w * to_f<T>(g[idx + c]);
    }
}

template <typename T, int D, int C>
__global__ __launch_bounds__(GT) void grid_fwd_tile_kernel(const float* __restrict__ inputs, const T* __restrict__ grid,
                                                           const int* __restrict__ offsets, T* __restrict__ outputs,
                                                           int64_t B, int L, LevelTab lt, int gridtype, int align,
                                                           int interp) {
    extern __shared__ float slab[];
    const int LC = L * C, row = LC + 1;
    const int64_t b0 = (int64_t)blockIdx.x * GT;
    const int nb = (int)min((int64_t)GT, B - b0);
    const int t = threadIdx.x;
    if (t < nb) {
        float in[D];
#pragma unroll
        for (int d = 0; d < D; d++) in[d] = inputs[(b0 + t) * D + d];
        // two levels per iteration: 2 x 2^D independent gathers in flight
#pragma unroll 1
        for (int level = 0; level < L; level += 2) {
            float a0[C], a1[C];
            grid_level_acc<T, D, C>(in, level, offsets, lt, grid, gridtype, align, interp, a0);
            if (level + 1 < L) grid_level_acc<T, D, C>(in, level + 1, offsets, lt, grid, gridtype, align, interp, a1);
#pragma unroll
            for (int c = 0; c < C; c++) slab[t * row + level * C + c] = a0[c];
            if (level + 1 < L) {
#pragma unroll
                for (int c = 0; c < C; c++) slab[t * row + (level + 1) * C + c] = a1[c];
            }
        }
    }
    __syncthreads();
    T* out = outputs + b0 * LC;
    for (int i = t; i < nb * LC; i += GT) {
        const int p = i / LC;
        out[i] = from_f<T>(slab[p * row + (i - p * LC)]);
    }
}

template <typename T, int D, int C>
__global__ __launch_bounds__(GT) void grid_bwd_tile_kernel(const T* __restrict__ grad, const float* __restrict__ inputs,
                                                           const int* __restrict__ offsets, float* __restrict__ ggrid,
                                                           int64_t B, int L, LevelTab lt, int gridtype, int align,
                                                           int interp) {
    extern __shared__ float slab[];
    const int LC = L * C, row = LC + 1;
    const int64_t b0 = (int64_t)blockIdx.x * GT;
    const int nb = (int)min((int64_t)GT, B - b0);
    const int t = threadIdx.x;
    const T* gsrc = grad + b0 * LC;
    for (int i = t; i < nb * LC; i += GT) {
        const int p = i / LC;
        slab[p * row + (i - p * LC)] = to_f<T>(gsrc[i]);
    }
    float in[D];
    if (t < nb) {
#pragma unroll
        for (int d = 0; d < D; d++) in[d] = inputs[(b0 + t) * D + d];
    }
    __syncthreads();
    if (t >= nb) return;
#pragma unroll 1
    for (int level = 0; level < L; level++) {
        float pos[D], deriv[D];
        uint32_t pg[D];
        const LevelCoord lc = level_coords<D>(in, level, offsets, lt, align != 0, interp, pos, deriv, pg);
        if (lc.oob) continue;
        float gcur[C];
#pragma unroll
        for (int c = 0; c < C; c++) gcur[c] = slab[t * row + level * C + c];
        float* gg = ggrid + (int64_t)offsets[level] * C;
#pragma unroll
        for (int corner = 0; corner < (1 << D); corner++) {
            float w = 1.f;
            uint32_t loc[D];
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (corner & (1 << d)) { w *= pos[d]; loc[d] = pg[d] + 1; }
                else { w *= 1.f - pos[d]; loc[d] = pg[d]; }
            }
            const uint32_t idx = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc) * C;
#pragma unroll
            for (int c = 0; c < C; c++) atomicAdd(gg + idx + c, w * gcur[c]);
        }
    }
}

// dL/dx[b, d] = sum_{l, c} grad[b, l, c] * dy_dx[b, l, d, c]   (gridencoder.cu:343-369)
template <typename T, int D, int C>
__global__ void grid_input_bwd_kernel(const T* __restrict__ grad, const T* __restrict__ dy_dx, T* __restrict__ gin,
                                      int64_t B, int L) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= B * D) return;
    const int64_t b = t / D;
    const int d = (int)(t - b * D);
    float r = 0.f;
    for (int l = 0; l < L; l++)
#pragma unroll
        for (int c = 0; c < C; c++)
            r += to_f<T>(grad[(b * L + l) * C + c]) * to_f<T>(dy_dx[b * (int64_t)L * D * C + (int64_t)l * D * C + d * C + c]);
    gin[t] = from_f<T>(r);
}

__global__ void grid_fill_int_kernel(int* __restrict__ p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <typename T>
__global__ void f32_to_kernel(const float* __restrict__ src, T* __restrict__ dst, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = from_f<T>(src[i]);
}

// total-variation gradient added into grad (gridencoder.cu:506-610)
template <typename T, int D, int C>
__global__ void grid_tv_kernel(const float* __restrict__ inputs, const T* __restrict__ grid, float* __restrict__ grad,
                               const int* __restrict__ offsets, float weight, int64_t B, int L, LevelTab lt,
                               int gridtype, int align) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= B * L) return;
    const int64_t b = tid / L;
    const int level = (int)(tid - b * L);
    const float* in = inputs + b * D;
    float pos[D], deriv[D];
    uint32_t pg[D];
    LevelCoord lc = level_coords<D>(in, level, offsets, lt, align != 0, 0, pos, deriv, pg);
    if (lc.oob) return;
    const T* g = grid + (int64_t)offsets[level] * C;
    float* gr = grad + (int64_t)offsets[level] * C;
    uint32_t idx = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, pg) * C;
    float res[C], idel[C];
#pragma unroll
    for (int c = 0; c < C; c++) { res[c] = 0.f; idel[c] = 0.f; }
    const float w = weight / (2 * D);
#pragma unroll
    for (int d = 0; d < D; d++) {
        uint32_t cur = pg[d];
        if (cur < lc.res) {
            pg[d] = cur + 1;
            uint32_t ir = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, pg) * C;
#pragma unroll
            for (int c = 0; c < C; c++) {
                float v = to_f<T>(g[idx + c]) - to_f<T>(g[ir + c]);
                res[c] += v;
                idel[c] += v * v;
            }
        }
        if (cur > 0) {
            pg[d] = cur - 1;
            uint32_t il = grid_index<D>(gridtype, align != 0, lc.hs, lc.res, pg) * C;
#pragma unroll
            for (int c = 0; c < C; c++) {
                float v = to_f<T>(g[idx + c]) - to_f<T>(g[il + c]);
                res[c] += v;
                idel[c] += v * v;
            }
        }
        pg[d] = cur;
    }
#pragma unroll
    for (int c = 0; c < C; c++) atomicAdd(gr + idx + c, w * res[c] * rsqrtf(idel[c] + 1e-9f));
}

// ---------------------------------------------------------------------------
// Bucketed gradient scatter (no float atomics to global memory on the hot path).
// Device-scope float atomics run at a fraction of HBM speed, so the adjoint
// groups its (row, value) contributions by bucket of RB consecutive table rows
// and sums each bucket in LDS:
//   1. count:   per (level, point tile) block, an LDS histogram of the buckets
//               its contributions fall into, added to the global bucket counts;
//   2. scan:    bucket starts and, per bucket, the number of SEG-record segments;
//   3. scatter: the same contributions again, written as (row, C values) records
//               into per-bucket ranges reserved with one atomic per (block, bucket);
//   4. reduce:  one block per bucket segment accumulates its records into an
//               LDS copy of the bucket's rows and adds it to the gradient table
//               (plain read-modify-write when the bucket has one segment).
// ---------------------------------------------------------------------------
constexpr int GB_THREADS = 256;
constexpr int GB_PPT = 8;           // points per thread in the count / scatter passes
constexpr int GB_HBINS = 4096;      // LDS histogram bins per block (buckets one level spans)
constexpr int64_t GB_SEG = 262144;  // records per reduce block

__host__ __device__ constexpr int gb_rows(int C) { return 16384 / C; }  // RB: 64 KB of fp32 rows in LDS

struct GridBucketWs {
    int* count;      // [NB]
    int* start;      // [NB + 1]
    int* cursor;     // [NB]
    int* segstart;   // [NB + 1]
    uint32_t* rows;  // [records]
    float* vals;     // [records * C]
};

static int64_t gb_num_buckets(int64_t n_rows, int C) { return (n_rows + gb_rows(C) - 1) / gb_rows(C); }

static int64_t gb_workspace_bytes(int64_t B, int D, int C, int L, int64_t n_rows) {
    const int64_t NB = gb_num_buckets(n_rows, C);
    const int64_t records = B * L * (1ll << D);
    int64_t head = (4 * NB + 2) * 4;
    head = (head + 255) / 256 * 256;
    return head + records * 4 + records * C * 4;
}

static GridBucketWs gb_carve(void* ws, int64_t B, int D, int C, int L, int64_t n_rows) {
    const int64_t NB = gb_num_buckets(n_rows, C);
    const int64_t records = B * L * (1ll << D);
    GridBucketWs w;
    int* ip = (int*)ws;
    w.count = ip;
    w.start = ip + NB;
    w.cursor = ip + 2 * NB + 1;
    w.segstart = ip + 3 * NB + 1;
    int64_t head = (4 * NB + 2) * 4;
    head = (head + 255) / 256 * 256;
    w.rows = (uint32_t*)((char*)ws + head);
    w.vals = (float*)((char*)ws + head + records * 4);
    return w;
}

// PASS 0: count, PASS 1: scatter.  blockIdx.y = level, blockIdx.x = tile of GB_THREADS * GB_PPT points.
template <typename T, int D, int C, int PASS>
__global__ __launch_bounds__(GB_THREADS) void grid_bucket_kernel(const T* __restrict__ grad,
                                                                 const float* __restrict__ inputs,
                                                                 const int* __restrict__ offsets, int64_t B, int L,
                                                                 LevelTab lt, int gridtype, int align, int interp,
                                                                 GridBucketWs ws) {
    constexpr int RB = gb_rows(C);
    __shared__ int hist[GB_HBINS];
    __shared__ int base[GB_HBINS];
    const int level = blockIdx.y;
    const int row0 = offsets[level], row1 = offsets[level + 1];
    const int b_lo = row0 / RB;
    const int nbins = row1 > row0 ? (row1 - 1) / RB - b_lo + 1 : 0;
    const bool local = nbins <= GB_HBINS;
    for (int i = threadIdx.x; i < GB_HBINS; i += GB_THREADS) hist[i] = 0;
    __syncthreads();
    const int64_t p_begin = (int64_t)blockIdx.x * GB_THREADS * GB_PPT;
    // pass 1 needs the histogram before it can place records: count first (both passes)
#pragma unroll 1
    for (int it = 0; it < GB_PPT; it++) {
        const int64_t b = p_begin + (int64_t)it * GB_THREADS + threadIdx.x;
        if (b >= B) break;
        float pos[D], deriv[D];
        uint32_t pg[D];
        LevelCoord lc = level_coords<D>(inputs + b * D, level, offsets, lt, align != 0, interp, pos, deriv, pg);
        if (lc.oob) continue;
#pragma unroll
        for (int corner = 0; corner < (1 << D); corner++) {
            uint32_t loc[D];
#pragma unroll
            for (int d = 0; d < D; d++) loc[d] = (corner & (1 << d)) ? pg[d] + 1 : pg[d];
            const int row = row0 + (int)grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc);
            const int bk = row / RB;
            if (local) atomicAdd(&hist[bk - b_lo], 1);
            else if (PASS == 0) atomicAdd(&ws.count[bk], 1);
        }
    }
    __syncthreads();
    if (PASS == 0) {
        if (local)
            for (int i = threadIdx.x; i < nbins; i += GB_THREADS)
                if (hist[i]) atomicAdd(&ws.count[b_lo + i], hist[i]);
        return;
    }
    // pass 1: reserve this block's range in each bucket, then write the records
    if (local) {
        for (int i = threadIdx.x; i < nbins; i += GB_THREADS) {
            base[i] = hist[i] ? atomicAdd(&ws.cursor[b_lo + i], hist[i]) : 0;
            hist[i] = 0;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int it = 0; it < GB_PPT; it++) {
        const int64_t b = p_begin + (int64_t)it * GB_THREADS + threadIdx.x;
        if (b >= B) break;
        float pos[D], deriv[D];
        uint32_t pg[D];
        LevelCoord lc = level_coords<D>(inputs + b * D, level, offsets, lt, align != 0, interp, pos, deriv, pg);
        if (lc.oob) continue;
        float gcur[C];
#pragma unroll
        for (int c = 0; c < C; c++) gcur[c] = to_f<T>(grad[(b * L + level) * C + c]);
#pragma unroll
        for (int corner = 0; corner < (1 << D); corner++) {
            float wgt = 1.f;
            uint32_t loc[D];
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (corner & (1 << d)) { wgt *= pos[d]; loc[d] = pg[d] + 1; }
                else { wgt *= 1.f - pos[d]; loc[d] = pg[d]; }
            }
            const int row = row0 + (int)grid_index<D>(gridtype, align != 0, lc.hs, lc.res, loc);
            const int bk = row / RB;
            const int64_t slot = local ? (int64_t)base[bk - b_lo] + atomicAdd(&hist[bk - b_lo], 1)
                                       : (int64_t)atomicAdd(&ws.cursor[bk], 1);
            ws.rows[slot] = (uint32_t)row;
#pragma unroll
            for (int c = 0; c < C; c++) ws.vals[slot * C + c] = wgt * gcur[c];
        }
    }
}

// bucket starts, reservation cursors and per-bucket segment offsets (one block)
__global__ __launch_bounds__(1024) void grid_bucket_scan_kernel(GridBucketWs ws, int64_t NB) {
    __shared__ int sa[1024], sb[1024];
    __shared__ int carry_a, carry_b;
    if (threadIdx.x == 0) { carry_a = 0; carry_b = 0; }
    __syncthreads();
    for (int64_t t0 = 0; t0 < NB; t0 += 1024) {
        const int64_t i = t0 + threadIdx.x;
        const int cnt = i < NB ? ws.count[i] : 0;
        const int nseg = (int)((cnt + GB_SEG - 1) / GB_SEG);
        sa[threadIdx.x] = cnt;
        sb[threadIdx.x] = nseg;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            int va = threadIdx.x >= off ? sa[threadIdx.x - off] : 0;
            int vb = threadIdx.x >= off ? sb[threadIdx.x - off] : 0;
            __syncthreads();
            sa[threadIdx.x] += va;
            sb[threadIdx.x] += vb;
            __syncthreads();
        }
        if (i < NB) {
            const int ea = carry_a + sa[threadIdx.x] - cnt;
            ws.start[i] = ea;
            ws.cursor[i] = ea;
            ws.segstart[i] = carry_b + sb[threadIdx.x] - nseg;
        }
        __syncthreads();
        if (threadIdx.x == 1023) {
            carry_a += sa[1023];
            carry_b += sb[1023];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ws.start[NB] = carry_a;
        ws.segstart[NB] = carry_b;
    }
}

template <int C>
__global__ __launch_bounds__(GB_THREADS) void grid_bucket_reduce_kernel(GridBucketWs ws, int64_t NB, int64_t n_rows,
                                                                        float* __restrict__ ggrid) {
    constexpr int RB = gb_rows(C);
    __shared__ float acc[RB * C];
    const int64_t j = blockIdx.x;
    if (j >= ws.segstart[NB]) return;
    // bucket of segment j: last bucket with segstart <= j
    int64_t lo = 0, hi = NB - 1;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (ws.segstart[mid] <= j) lo = mid;
        else hi = mid - 1;
    }
    const int64_t bk = lo;
    const int nseg = ws.segstart[bk + 1] - ws.segstart[bk];
    const int64_t r0 = ws.start[bk] + (j - ws.segstart[bk]) * GB_SEG;
    const int64_t r1 = min(r0 + GB_SEG, (int64_t)ws.start[bk + 1]);
    for (int i = threadIdx.x; i < RB * C; i += GB_THREADS) acc[i] = 0.f;
    __syncthreads();
    const int row_base = (int)(bk * RB);
    for (int64_t r = r0 + threadIdx.x; r < r1; r += GB_THREADS) {
        const int lr = (int)ws.rows[r] - row_base;
#pragma unroll
        for (int c = 0; c < C; c++) atomicAdd(&acc[lr * C + c], ws.vals[r * C + c]);
    }
    __syncthreads();
    const int64_t nr = min((int64_t)RB, n_rows - row_base);
    float* g = ggrid + (int64_t)row_base * C;
    for (int64_t i = threadIdx.x; i < nr * C; i += GB_THREADS) {
        const float v = acc[i];
        if (v == 0.f) continue;
        if (nseg == 1) g[i] += v;
        else atomicAdd(&g[i], v);
    }
}

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Table-gradient scatter by sorted tiles (hash grids in 3 dimensions).  The bucketed
// scatter above lists 8 records of 4 + 4 C bytes per (point, level), placed one by one,
// and adds them with LDS float atomics, which this card runs at one lane per three
// clocks per CU (measured; 64-bit float atomics: 2.1 lanes per clock, whatever the
// addresses).  Here
//   1. sort: a block per (tile of 1024 points, level) sorts the tile's hits by bucket in
//      LDS and writes them in that order, coalesced: a hit is one of the 4 (y, z) corner
//      pairs of a point, whose two x corners always share a bucket (the hash multiplies
//      x by 1, so x moves only the row's low bits; a dense level's buckets are whole
//      lines of x), 8 + 4 C bytes: both rows within the bucket, the fraction in x and
//      the upstream gradient times the pair's weight;
//   2. add:  a block per bucket, whose rows it keeps in LDS as doubles (128 KB, one
//      block per CU), streams its segment of every tile and adds both corners;
//   3. sum:  the parts' copies of a level added into the gradient table (a level taken
//      in one part adds to the table itself).
// Gathering each hit's point and gradient in the add pass instead of writing them out
// was slower: one lane per clock and CU (2^20 points x 16 levels x 2 features: 0.67 ms
// of gathers in place of 16 bytes per hit written and read).  A level that fits neither
// form (a hashed level of a size that is no power of two, say) adds with float atomics
// to the table.
// ---------------------------------------------------------------------------
constexpr int GS_THREADS = 1024;
constexpr int GS_WAVES = GS_THREADS / 64;
constexpr int GS_TILE = 1024;             // points per sorted tile
constexpr int GS_HITS = 4 * GS_TILE;      // hits per tile at most
constexpr int GS_SORT_THREADS = 512;
constexpr int GS_MAX_NB = 512;            // buckets per level
constexpr int GS_XCD = 8;
// Hits of one row in a wavefront that are summed before the add: additions to one address take 13
// times as long as to different ones (2^18 points in one cell, 4 dense levels x 2 features: 2664 us
// without, 745 with; 16 of a row are still the faster one by one).
constexpr int GS_SAME = 24;

__host__ __device__ constexpr int gs_rows(int C) { return 16384 / C; }  // rows of a bucket: 128 KB of doubles

enum { GS_NONE = 0, GS_HASH = 1, GS_DENSE = 2, GS_DIRECT = 3 };

struct GsLevel {
    int row0, hs, mode, nb;  // first row, rows, form, buckets
    int rows;                // rows that corners can reach (a dense level's table is padded)
    int lines;               // GS_DENSE: lines of x per bucket
    uint32_t R;              // lattice points per axis
};

__device__ __forceinline__ GsLevel gs_level(const int* __restrict__ offsets, float scale, int level, int RB) {
    GsLevel v;
    v.row0 = offsets[level];
    v.hs = offsets[level + 1] - v.row0;
    v.R = (uint32_t)ceilf(scale) + 2u;
    v.rows = v.hs;
    v.lines = 0;
    v.nb = 1;
    if (v.hs <= 0) {
        v.mode = GS_NONE;
        v.nb = 0;
        return v;
    }
    v.mode = GS_DIRECT;
    if (v.R > (uint32_t)RB) return v;
    const uint64_t R2 = (uint64_t)v.R * v.R, hs = (uint64_t)v.hs;
    uint32_t stride = 1;  // grid_index's strides, wrapping like it
    for (int d = 0; d < 3; d++)
        if (stride <= (uint32_t)v.hs) stride *= v.R;
    if (R2 * v.R <= hs) {
        v.lines = RB / (int)v.R;
        const int nb = ((int)R2 + v.lines - 1) / v.lines;
        if (nb <= GS_MAX_NB) {
            v.mode = GS_DENSE;
            v.nb = nb;
            v.rows = (int)(R2 * v.R);
        }
    } else if (stride > (uint32_t)v.hs && (hs & (hs - 1)) == 0 && v.hs / RB <= GS_MAX_NB) {
        v.mode = GS_HASH;
        v.nb = v.hs > RB ? v.hs / RB : 1;
    }
    return v;
}

// Parts the points are taken in: one for a level of 64 buckets or more (a part more costs a
// copy of the level's rows written and read: 72 us for 2 parts of 16 levels at 2^20 points),
// else about 128 blocks per level, whose short items fill in behind the long ones, with at
// least 16384 hits each.
__host__ __device__ inline int gs_parts(int64_t B, int nb) {
    if (nb >= 64) return 1;
    int64_t p = (128 + nb - 1) / nb;
    const int64_t most = B / ((int64_t)4096 * nb);
    if (p > most) p = most;
    return p < 1 ? 1 : (int)p;
}

struct GsWs {
    uint32_t* hits;  // [L, 2 + C, tiles * GS_HITS]: rows (first | second << 16), x fraction, values
    uint32_t* segs;  // [L, GS_MAX_NB, tiles] first hit << 16 | hits
    int* next;       // items of the add pass handed out
    float* copies;   // parts of the levels taken in several, level after level
    int tiles;
};

static int64_t gs_tiles(int64_t B) { return (B + GS_TILE - 1) / GS_TILE; }

// bound on the copies' rows: a level taken in parts has at most 63 buckets
static int64_t gs_copy_rows(int64_t B, int C, int L) {
    const int64_t most = B / 4096;
    return most > 1 ? (int64_t)L * gs_rows(C) * (most < 191 ? most : 191) : 0;
}

static int64_t gs_workspace_bytes(int64_t B, int C, int L) {
    return gs_tiles(B) * L * (GS_HITS * 4 * (2 + C) + GS_MAX_NB * 4) + 256 + gs_copy_rows(B, C, L) * C * 4;
}

static GsWs gs_carve(void* ws, int64_t B, int C, int L) {
    GsWs w;
    w.tiles = (int)gs_tiles(B);
    w.hits = (uint32_t*)ws;
    w.segs = w.hits + (int64_t)w.tiles * L * GS_HITS * (2 + C);
    w.next = (int*)(w.segs + (int64_t)w.tiles * L * GS_MAX_NB);
    w.copies = (float*)(w.next + 64);
    return w;
}

// Lattices wider than a bucket do not fit (their x moves the row out of it), and past 256
// buckets per level the tiles' segments get much shorter than a wavefront.  Few points do not
// fill the tiles of a block per CU (16 levels of up to 2^19 rows, sorted against bucketed in us:
// 1 feature 256 points 35 / 38, 16 28 / 27; 2 features 1024 points 61 / 76, 256 43 / 38; 4 features
// 4096 points 110 / 231, 1024 93 / 88).
static bool gs_applies(int64_t B, int D, int C, int L, int64_t n_rows, int gridtype, int align, const LevelTab& lt) {
    if (D != 3 || gridtype != 0 || align || B >= (1ll << 28) || n_rows > (int64_t)256 * L * gs_rows(C)) return false;
    if (B < (C < 4 ? 512 * C : 2048)) return false;
    for (int l = 0; l < L; l++)
        if (!(lt.scale[l] + 3.f < (float)gs_rows(C))) return false;
    return true;
}

// points are padded by one per 32 in LDS (a wavefront reads them 32 apart)
constexpr int GS_PAD_TILE = GS_TILE + GS_TILE / 32;
__host__ __device__ constexpr int gs_sort_lds(int C) { return GS_PAD_TILE * 4 * (3 + C) + GS_HITS * 4; }

template <typename T, int C>
__global__ __launch_bounds__(GS_SORT_THREADS) void gs_sort_kernel(const T* __restrict__ grad,
                                                                  const float* __restrict__ inputs,
                                                                  const int* __restrict__ offsets, int64_t B, int L,
                                                                  LevelTab lt, int interp, GsWs ws,
                                                                  float* __restrict__ ggrid) {
    constexpr int RB = gs_rows(C), PT = GS_TILE / GS_SORT_THREADS;
    extern __shared__ float sm[];
    float* sx = sm;                           // [3, GS_PAD_TILE] points, then their cell fractions
    float* sg = sm + 3 * GS_PAD_TILE;         // [C, GS_PAD_TILE]
    uint32_t* sorted = (uint32_t*)(sg + C * GS_PAD_TILE);  // [GS_HITS] point | pair << 10 | row << 12 | span << 26
    static_assert(GS_TILE == 1 << 10 && gs_rows(1) <= 1 << 14, "a sorted hit is one word");
    __shared__ int count[GS_MAX_NB];
    __shared__ int wsum[GS_MAX_NB / 64];
    static_assert(GS_MAX_NB == GS_SORT_THREADS, "one bucket per thread in the scan");
    const int t = threadIdx.x, lane = t & 63;
    if (blockIdx.x == 0 && t == 0) *ws.next = 0;
    // a tile's levels run next to each other on one XCD (blocks go to XCDs round robin), so
    // that its L2 serves the rows of the upstream gradient, which hold every level
    const int64_t group = blockIdx.x / (GS_XCD * L);
    const int rest = (int)(blockIdx.x - group * (GS_XCD * L));
    const int64_t tile = group * GS_XCD + rest % GS_XCD;
    const int level = rest / GS_XCD;
    if (tile >= ws.tiles) return;
    const GsLevel v = gs_level(offsets, lt.scale[level], level, RB);
    if (v.mode == GS_NONE) return;
    const int64_t b0 = tile * GS_TILE;
    const int LC = L * C;
    if (v.mode == GS_DIRECT) {
        float* gg = ggrid + (int64_t)v.row0 * C;
        for (int64_t b = b0 + t; b < min(B, b0 + GS_TILE); b += GS_SORT_THREADS) {
            float pos[3], deriv[3];
            uint32_t pg[3];
            const LevelCoord lc = level_coords<3>(inputs + b * 3, level, offsets, lt, false, interp, pos, deriv, pg);
            if (lc.oob) continue;
            for (int corner = 0; corner < 8; corner++) {
                float w = 1.f;
                uint32_t loc[3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    if (corner & (1 << d)) { w *= pos[d]; loc[d] = pg[d] + 1; }
                    else { w *= 1.f - pos[d]; loc[d] = pg[d]; }
                }
                const int64_t r = grid_index<3>(0, false, lc.hs, lc.res, loc);
#pragma unroll
                for (int c = 0; c < C; c++) atomicAdd(&gg[r * C + c], w * to_f<T>(grad[b * LC + level * C + c]));
            }
        }
        return;
    }
    const float inv_lines = v.mode == GS_DENSE ? 1.f / (float)v.lines : 0.f;
    // bucket of a line of x and the line's place in it (lines < 2^24: exact after one step)
    auto line_bucket = [&](uint32_t ln, uint32_t& in_bucket) {
        uint32_t q = (uint32_t)((float)ln * inv_lines);
        if (q * (uint32_t)v.lines > ln) q--;
        else if ((q + 1u) * (uint32_t)v.lines <= ln) q++;
        in_bucket = ln - q * (uint32_t)v.lines;
        return q;
    };
    const uint32_t mask = (uint32_t)min(v.hs, RB) - 1u;  // GS_HASH: row within the bucket
    count[t] = 0;
    const int np = (int)min((int64_t)GS_TILE, B - b0);
    for (int i = t; i < 3 * np; i += GS_SORT_THREADS) {
        const int p = i / 3;
        sx[(i - 3 * p) * GS_PAD_TILE + p + (p >> 5)] = inputs[b0 * 3 + i];
    }
    for (int p = t; p < np; p += GS_SORT_THREADS)
#pragma unroll
        for (int c = 0; c < C; c++)
            sg[c * GS_PAD_TILE + p + (p >> 5)] = to_f<T>(grad[(b0 + p) * LC + level * C + c]);
    __syncthreads();
    // the lanes of a wavefront take points 32 apart, so that neighbours in a bucket's order
    // lie in different cells when the points are samples along rays (equal LDS addresses
    // are added one by one)
    uint32_t at[PT][4], row[PT][4];  // bucket << 16 | rank within the bucket; row within it | span << 14
#pragma unroll
    for (int i = 0; i < PT; i++) {
        const int p = lane * (GS_TILE / 64) + (t >> 6) * PT + i, pp = p + (p >> 5);
        bool on = p < np;
        float in[3] = {-1.f, -1.f, -1.f}, pos[3], deriv[3];
        uint32_t pg[3];
        if (on) {
#pragma unroll
            for (int d = 0; d < 3; d++) in[d] = sx[d * GS_PAD_TILE + pp];
        }
        const LevelCoord lc = level_coords<3>(in, level, offsets, lt, false, interp, pos, deriv, pg);
        on = on && !lc.oob;
        if (on) {
#pragma unroll
            for (int d = 0; d < 3; d++) sx[d * GS_PAD_TILE + pp] = pos[d];
        }
        // the rows of x and x + 1 differ by the bits up to x's lowest zero bit
        const uint32_t span = (uint32_t)min(__builtin_ctz(~pg[0]), 13);
        const uint32_t hy = pg[1] * 2654435761u, hz = pg[2] * 805459861u;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            at[i][c] = ~0u;
            row[i][c] = 0;
            if (on) {
                uint32_t id;
                if (v.mode == GS_HASH) {
                    const uint32_t h = pg[0] ^ ((c & 1) ? hy + 2654435761u : hy) ^ ((c >> 1) ? hz + 805459861u : hz);
                    id = (h & ((uint32_t)v.hs - 1u)) / (uint32_t)RB;
                    row[i][c] = (h & mask) | (span << 14);
                } else {
                    uint32_t in_bucket;
                    id = line_bucket(pg[1] + (c & 1) + (pg[2] + (c >> 1)) * v.R, in_bucket);
                    row[i][c] = pg[0] + in_bucket * v.R;
                }
                at[i][c] = (id << 16) | (uint32_t)atomicAdd(&count[id], 1);
            }
        }
    }
    __syncthreads();
    // exclusive prefix of the bucket counts
    const int own = count[t];
    int incl = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(incl, off, 64);
        if (lane >= off) incl += u;
    }
    if (lane == 63) wsum[t >> 6] = incl;
    __syncthreads();
    int start = incl - own, total = 0;
#pragma unroll
    for (int q = 0; q < GS_MAX_NB / 64; q++) {
        if (q < (t >> 6)) start += wsum[q];
        total += wsum[q];
    }
    count[t] = start;
    if (t < v.nb)
        ws.segs[((int64_t)level * GS_MAX_NB + t) * ws.tiles + tile] = ((uint32_t)start << 16) | (uint32_t)own;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; i++)
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (at[i][c] != ~0u)
                sorted[count[at[i][c] >> 16] + (at[i][c] & 0xffffu)] =
                    (uint32_t)(lane * (GS_TILE / 64) + (t >> 6) * PT + i) | (c << 10) | (row[i][c] << 12);
    __syncthreads();
    const int64_t plane = (int64_t)ws.tiles * GS_HITS;
    uint32_t* dst = ws.hits + (int64_t)level * (2 + C) * plane + tile * GS_HITS;
    for (int i = t; i < total; i += GS_SORT_THREADS) {
        const uint32_t e = sorted[i], p = e & (GS_TILE - 1), pp = p + (p >> 5);
        const uint32_t r0 = (e >> 12) & 0x3fffu;
        const uint32_t r1 = v.mode == GS_HASH ? r0 ^ (((2u << (e >> 26)) - 1u) & mask) : r0 + 1u;
        const float wy = sx[GS_PAD_TILE + pp], wz = sx[2 * GS_PAD_TILE + pp];
        const float w = ((e & (1u << 10)) ? wy : 1.f - wy) * ((e & (1u << 11)) ? wz : 1.f - wz);
        dst[i] = r0 | (r1 << 16);
        dst[plane + i] = __float_as_uint(sx[pp]);
#pragma unroll
        for (int c = 0; c < C; c++) dst[(2 + c) * plane + i] = __float_as_uint(w * sg[c * GS_PAD_TILE + pp]);
    }
}

// the sum over the wavefront, all lanes active, inside the vector registers (as wave_sum)
__device__ __forceinline__ double wave_sum_double(double v) {
    auto step = [&](auto k) {
        constexpr int K = decltype(k)::value;
        v += __hiloint2double(lane_before<K>(0, __double2hiint(v)), lane_before<K>(0, __double2loint(v)));
    };
    step(std::integral_constant<int, 0>());
    step(std::integral_constant<int, 1>());
    step(std::integral_constant<int, 2>());
    step(std::integral_constant<int, 3>());
    step(std::integral_constant<int, 4>());
    step(std::integral_constant<int, 5>());
    return __hiloint2double(lane_i(__double2hiint(v), 63), lane_i(__double2loint(v), 63));
}

// One bucket of one level over one part of the tiles; copy: the first row of the level's
// copies (-1: the only part, which adds to the table itself).
template <int C>
__device__ __forceinline__ void gs_add_item(const int* __restrict__ offsets, int64_t B, const LevelTab& lt,
                                            const GsWs& ws, float* __restrict__ ggrid, int level, int part, int bucket,
                                            int64_t copy, double* acc, int t, int lane, int wave) {
    constexpr int RB = gs_rows(C), U = 4;
    const GsLevel v = gs_level(offsets, lt.scale[level], level, RB);
    const int parts = gs_parts(B, v.nb);
    const int per = (ws.tiles + parts - 1) / parts;
    const int t0 = min(ws.tiles, per * part), t1 = min(ws.tiles, t0 + per);
    const int first_row = v.mode == GS_DENSE ? bucket * v.lines * (int)v.R : bucket * RB;
    const int nrow = min(v.rows - first_row, v.mode == GS_DENSE ? v.lines * (int)v.R : RB);
    for (int i = t; i < RB * C; i += GS_THREADS) acc[i] = 0.0;
    __syncthreads();
    // a wavefront takes every GS_WAVES-th tile, 64 of them at a time: lane l holds the l-th
    // one's segment, and the segments are walked end to end in full wavefronts
    const uint32_t* segs = ws.segs + ((int64_t)level * GS_MAX_NB + bucket) * ws.tiles;
    const int64_t plane = (int64_t)ws.tiles * GS_HITS;
    const uint32_t* hits = ws.hits + (int64_t)level * (2 + C) * plane;
    for (int base = t0 + wave; base < t1; base += 64 * GS_WAVES) {
        const int tile = base + lane * GS_WAVES;
        const uint32_t sg = tile < t1 ? segs[tile] : 0u;
        const int n = (int)(sg & 0xffffu);
        int end = n;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(end, off, 64);
            if (lane >= off) end += u;
        }
        const int total = __builtin_amdgcn_readlane(end, 63);
        const int shift = tile * GS_HITS + (int)(sg >> 16) - (end - n);  // hit of position p: shift + p
        int j = 0, ej = __builtin_amdgcn_readlane(end, 0), oj = __builtin_amdgcn_readlane(shift, 0);
        for (int i0 = 0; i0 < total; i0 += 64 * U) {
            int at[U];
#pragma unroll
            for (int q = 0; q < U; q++) {
                const int p = i0 + 64 * q + lane;
                at[q] = oj;
                while (j < 63 && ej <= i0 + 64 * q + 63) {  // the segment ends within this wavefront's 64
                    j++;
                    oj = __builtin_amdgcn_readlane(shift, j);
                    if (p >= ej) at[q] = oj;
                    ej = __builtin_amdgcn_readlane(end, j);
                }
                at[q] = p < total ? at[q] + p : -1;
            }
            uint32_t rr[U] = {};
            float fx[U] = {}, val[U][C] = {};
#pragma unroll
            for (int q = 0; q < U; q++)
                if (at[q] >= 0) {
                    const uint32_t* h = hits + at[q];
                    rr[q] = h[0];
                    fx[q] = __uint_as_float(h[plane]);
#pragma unroll
                    for (int c = 0; c < C; c++) val[q][c] = __uint_as_float(h[(2 + c) * plane]);
                }
#pragma unroll
            for (int q = 0; q < U; q++) {
                unsigned long long left = __ballot(at[q] >= 0);
                while (left != 0ull) {  // hits of one row (points in one cell) are summed first
                    const int lead = __builtin_ctzll(left);
                    const uint32_t row = __builtin_amdgcn_readlane(rr[q], lead);
                    const unsigned long long same = __ballot(rr[q] == row) & left;
                    if (__popcll(same) < GS_SAME) break;
                    const bool in = (same >> lane) & 1ull;
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        const double a = wave_sum_double(in ? (double)((1.f - fx[q]) * val[q][c]) : 0.0);
                        const double b = wave_sum_double(in ? (double)(fx[q] * val[q][c]) : 0.0);
                        if (lane == 0) {
                            atomicAdd(&acc[c * RB + (row & 0xffffu)], a);
                            atomicAdd(&acc[c * RB + (row >> 16)], b);
                        }
                    }
                    left &= ~same;
                }
                if ((left >> lane) & 1ull) {
#pragma unroll
                    for (int c = 0; c < C; c++) {
                        atomicAdd(&acc[c * RB + (rr[q] & 0xffffu)], (double)((1.f - fx[q]) * val[q][c]));
                        atomicAdd(&acc[c * RB + (rr[q] >> 16)], (double)(fx[q] * val[q][c]));
                    }
                }
            }
        }
    }
    __syncthreads();
    if (copy < 0) {  // the only part: the bucket's rows belong to this block
        float* dst = ggrid + ((int64_t)v.row0 + first_row) * C;
        for (int i = t; i < nrow * C; i += GS_THREADS) {
            const float a = (float)acc[(i % C) * RB + i / C];
            if (a != 0.f) dst[i] += a;
        }
    } else {
        float* dst = ws.copies + (copy + (int64_t)part * v.rows + first_row) * C;
        for (int i = t; i < nrow * C; i += GS_THREADS) dst[i] = (float)acc[(i % C) * RB + i / C];
    }
}

template <int C>
__global__ __launch_bounds__(GS_THREADS) void gs_add_kernel(const int* __restrict__ offsets, int64_t B, int L,
                                                            LevelTab lt, GsWs ws, float* __restrict__ ggrid) {
    extern __shared__ double acc[];  // [C, RB]
    __shared__ int pick[3];
    __shared__ int64_t pick_copy;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // items (level, part, bucket), the finest level first: its few long items start early and
    // the coarse levels' many short ones fill in behind; lane l holds the l-th one's place
    const int mine = L - 1 - lane;
    GsLevel v;
    v.nb = 0;
    v.rows = 0;
    v.mode = GS_NONE;
    int parts = 0;
    if (lane < L) {
        v = gs_level(offsets, lt.scale[mine], mine, gs_rows(C));
        if (v.nb > 0 && v.mode != GS_DIRECT) parts = gs_parts(B, v.nb);
    }
    int64_t cincl = parts > 1 ? (int64_t)parts * v.rows : 0;
    const int64_t cown = cincl;
    int iincl = parts * v.nb;
    const int iown = iincl;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(iincl, off, 64);
        const int64_t cu = __shfl_up(cincl, off, 64);
        if (lane >= off) {
            iincl += u;
            cincl += cu;
        }
    }
    for (bool first = true;; first = false) {
        if (wave == 0) {
            // the next item, taken as the blocks get done
            int s = blockIdx.x;
            if (!first) {
                if (lane == 0) s = (int)gridDim.x + atomicAdd(ws.next, 1);
                s = __builtin_amdgcn_readfirstlane(s);
            }
            const int at = s - (iincl - iown);
            if (lane == 0) pick[0] = -1;
            wave_fence();
            if (at >= 0 && at < iown) {
                pick[0] = mine;
                pick[1] = at / v.nb;
                pick[2] = at % v.nb;
                pick_copy = parts > 1 ? cincl - cown : -1;
            }
        }
        __syncthreads();
        const int level = __builtin_amdgcn_readfirstlane(pick[0]);
        if (level < 0) return;  // past the last item
        const int part = __builtin_amdgcn_readfirstlane(pick[1]), bucket = __builtin_amdgcn_readfirstlane(pick[2]);
        gs_add_item<C>(offsets, B, lt, ws, ggrid, level, part, bucket, pick_copy, acc, t, lane, wave);
        __syncthreads();
    }
}

// ggrid += the parts' copies.  blockIdx.y = level.
template <int C>
__global__ __launch_bounds__(256) void gs_sum_kernel(const int* __restrict__ offsets, int64_t B, int L, LevelTab lt,
                                                     GsWs ws, float* __restrict__ ggrid) {
    constexpr int RB = gs_rows(C);
    const int level = blockIdx.y;
    const GsLevel v = gs_level(offsets, lt.scale[level], level, RB);
    if (v.nb == 0 || v.mode == GS_DIRECT) return;
    const int parts = gs_parts(B, v.nb);
    if (parts == 1) return;
    int64_t copy = 0;  // rows of the finer levels, whose copies come first
    for (int l = L - 1; l > level; l--) {
        const GsLevel u = gs_level(offsets, lt.scale[l], l, RB);
        const int p = u.nb > 0 && u.mode != GS_DIRECT ? gs_parts(B, u.nb) : 0;
        if (p > 1) copy += (int64_t)p * u.rows;
    }
    const int64_t n = (int64_t)v.rows * C;
    const float* src = ws.copies + copy * C;
    float* dst = ggrid + (int64_t)v.row0 * C;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float a = 0.f;
#pragma unroll 8
        for (int p = 0; p < parts; p++) a += src[p * n + i];
        if (a != 0.f) dst[i] += a;
    }
}

static int g_pf_cu = 0;

static int prop_blocks(int64_t work, int threads, int per_cu, int64_t* out) {
    if (g_pf_cu == 0) {
        int dev;
        N3DS_HIP_CHECK(hipGetDevice(&dev));
        N3DS_HIP_CHECK(hipDeviceGetAttribute(&g_pf_cu, hipDeviceAttributeMultiprocessorCount, dev));
    }
    int64_t nb = (work + threads - 1) / threads;
    const int64_t cap = (int64_t)g_pf_cu * per_cu;
    *out = nb < 1 ? 1 : (nb > cap ? cap : nb);
    return N3DS_OK;
}

template <typename T, int C>
static int gs_launch(const T* grad, const float* inputs, const int* offsets, int64_t B, int L, const LevelTab& lt,
                     int interp, void* workspace, float* ggrid, hipStream_t s) {
    const GsWs ws = gs_carve(workspace, B, C, L);
    const size_t lds = (size_t)gs_rows(C) * C * 8;
    N3DS_HIP_CHECK(hipFuncSetAttribute((const void*)gs_add_kernel<C>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds));
    N3DS_HIP_CHECK(hipFuncSetAttribute((const void*)gs_sort_kernel<T, C>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       gs_sort_lds(C)));
    int64_t nb;
    const int st = prop_blocks((int64_t)1 << 40, 1, 1, &nb);  // one persistent block per CU
    if (st) return st;
    const int64_t groups = (ws.tiles + GS_XCD - 1) / GS_XCD;
    hipLaunchKernelGGL((gs_sort_kernel<T, C>), dim3((unsigned)(groups * GS_XCD * L)), dim3(GS_SORT_THREADS),
                       gs_sort_lds(C), s, grad, inputs, offsets, B, L, lt, interp, ws, ggrid);
    hipLaunchKernelGGL((gs_add_kernel<C>), dim3((unsigned)nb), dim3(GS_THREADS), lds, s, offsets, B, L, lt, ws, ggrid);
    hipLaunchKernelGGL((gs_sum_kernel<C>), dim3(128, (unsigned)L), dim3(256), 0, s, offsets, B, L, lt, ws, ggrid);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

// ---------------------------------------------------------------------------
// Fused proposal density field: the reference's PropMLP forward
// (source/models.py:286-523 with disable_rgb: _warp_coords, GridEncoder with
// bound 1, density_layer = Linear(F, 64) -> ReLU -> Linear(64, 1), then
// softplus(raw + density_bias)), F = L * C grid features, in one kernel; the
// adjoint recomputes features and hidden units per point instead of storing
// the [N, 64] activations, writes dL/dfeatures for the grid scatter and
// reduces the weight gradients in LDS.
// ---------------------------------------------------------------------------
constexpr int PF_HID = 64;
constexpr int PF_MAXF = 32;
constexpr int PF_FWD_THREADS = 256;
// Adjoint: persistent blocks, as many as a CU holds at once.  Up to 12 features one block of 12
// wavefronts (522 us at 4.2 M points and 10 features; without the density's products, each with
// one float32 chain a wavefront, 450 of 512, and 606 with three blocks of four), beyond them blocks
// of 4: two up to 20 features, one above, where a wavefront needs more than 256 registers.  (Three
// blocks launched where two or one fit: 897 instead of 750 us at 16 features, 1500 instead of
// 921 at 20, 1930 instead of 1880 at 28, with the torch calls around them.)
constexpr int pf_bwd_threads(int fm) { return fm <= 12 ? 768 : 256; }
constexpr int pf_bwd_blocks(int fm) { return fm > 12 && fm <= 20 ? 2 : 1; }
// Tiles of 64 points whose weight gradients a wavefront sums in float32 before they go to the
// block's doubles.  With all of its points in one chain, dW1 of 2^24 equal points was off by
// 5.0e-5 of its largest entry, now 2.7e-6, in no more time at 10 features (570 us at 4.2 M
// points with the torch calls around it) and 3 % more at 28.
constexpr int PF_HELD = 4;

struct PropArgs {
    const float* coords;  // [N, 3] sample positions
    int64_t N;
    int warp;             // 0: none (coords in [-1, 1]), 1: contract then / 2, 2: divide by half the box side
    float inv_half_box;
    const void* emb;
    const int* offsets;
    int L;
    LevelTab lt;
    int gridtype, align, interp;
    const float* W1;  // [64, F]
    const float* b1;  // [64]
    const float* W2;  // [1, 64]
    const float* b2;  // [1]
    float dbias;
};

// models.py:19-33 and coord.contract (utils/coord.py:5-11), then grid.py:158
// (inputs + bound) / (2 bound) with bound 1
__device__ __forceinline__ void prop_warp(const PropArgs& P, int64_t b, float* cw, float* x01) {
    float x[3] = {P.coords[b * 3], P.coords[b * 3 + 1], P.coords[b * 3 + 2]};
    if (P.warp == 1) {
        const float eps = 1.1920929e-07f;
        const float m2 = fmaxf(x[0] * x[0] + x[1] * x[1] + x[2] * x[2], eps);
        const float k = m2 <= 1.f ? 1.f : (2.f * sqrtf(m2) - 1.f) / m2;
#pragma unroll
        for (int d = 0; d < 3; d++) x[d] = (m2 <= 1.f ? x[d] : k * x[d]) / 2.f;
    } else if (P.warp == 2) {
#pragma unroll
        for (int d = 0; d < 3; d++) x[d] = x[d] * P.inv_half_box;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        cw[d] = x[d];
        x01[d] = (x[d] + 1.f) / 2.f;
    }
}

template <typename T, int C, int FM>
__device__ __forceinline__ void prop_features(const PropArgs& P, const float* x01, float* f) {
#pragma unroll
    for (int l = 0; l < FM / C; l++) {
        float a[C];
#pragma unroll
        for (int c = 0; c < C; c++) a[c] = 0.f;
        if (l < P.L) grid_level_acc<T, 3, C>(x01, l, P.offsets, P.lt, (const T*)P.emb, P.gridtype, P.align, P.interp, a);
#pragma unroll
        for (int c = 0; c < C; c++) f[l * C + c] = a[c];
    }
}

// Features of many points with the levels in step over the whole chip, for tables larger than
// an XCD's L2.  One resident block per CU owns a run of points, kept in LDS, and all blocks
// walk the levels at the same pace, a hashed level's table in parts of at most an L2: what is
// gathered from at one time stays in every L2.  Blocks at any level of their own hold several
// levels' tables at once, and most gathers go to memory, which answers 55 G scattered lines a
// second here (4.2 M points, 10 levels of up to 8 MB: 1843 us, 108 M lines).  Gathers that hit
// the L2 are then bound by the vector cache, 2 to 3 clocks a line: a load of 16 bytes serves
// both corners of most x edges.  The rows of a point's corners wait in registers until the last
// part, so that they are summed in the one kernel's order, to the bit (a hidden unit at its
// kink passes on or not by the last bit of its features); two features a row do not fit the
// registers that way and take a level whole.  Features are written level by level, [L, n, C]; with
// the head after it 1435 us (1538 + 140 with whole levels of 8 MB, 1149 + 140 with sums kept from
// part to part).
constexpr int LS_THREADS = 1024;
constexpr int LS_POINTS = 8;                // per thread and round at most
constexpr int64_t LS_PART_BYTES = 4 << 20;  // of a level's table gathered from at one time

// A table row of 2 or 4 bytes as it is held until the sum
template <typename T, int C>
union GridRow {
    uint32_t bits;
    T v[C];
};

struct LevelPoint {
    float f[3];
    uint32_t pg[3];
    bool oob;
};

// as level_coords
__device__ __forceinline__ LevelPoint level_point(const float* x, float scale, int align, int interp) {
    LevelPoint p;
    p.oob = false;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float xd = x[d * LS_THREADS];
        if (xd < 0.f || xd > 1.f) p.oob = true;
        float t = fmaf(xd, scale, align ? 0.0f : 0.5f);
        const float fl = floorf(t);
        p.pg[d] = (uint32_t)fl;
        t -= fl;
        if (interp == 1) t = t * t * (3.f - 2.f * t);
        p.f[d] = t;
    }
    return p;
}

template <typename T, int C>
__device__ __forceinline__ void level_sum(const LevelPoint& p, const GridRow<T, C> (&row)[8], float (&acc)[C]) {
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        float w = 1.f;
#pragma unroll
        for (int d = 0; d < 3; d++) w *= k & (1 << d) ? p.f[d] : 1.f - p.f[d];
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] += w * to_f<T>(row[k].v[c]);
    }
    if (p.oob)
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] = 0.f;
}

// row r mod QR of the QR rows in 16 bytes (a row of 2 bytes in the low half)
template <int QR>
__device__ __forceinline__ uint32_t quad_row(uint4 e, uint32_t r) {
    const uint32_t i = QR == 8 ? r >> 1 : r;
    const uint32_t lo = i & 1 ? e.y : e.x, hi = i & 1 ? e.w : e.z;
    const uint32_t w = i & 2 ? hi : lo;
    return QR == 8 && (r & 1) ? w >> 16 : w;
}

// The corners of a level hashed into hs = 2^k rows that lie in [lo, lo + width), a multiple of
// 16 rows; the others' rows stay as they are.
template <typename T, int C>
__device__ __forceinline__ void level_hashed(const LevelPoint& p, const T* __restrict__ g, uint32_t hs, uint32_t lo,
                                             uint32_t width, GridRow<T, C> (&row)[8]) {
    constexpr int QR = 16 / (C * (int)sizeof(T));  // rows of 16 bytes
    static_assert(QR == 4 || QR == 8, "rows of 2 or 4 bytes");
    const uint32_t y0 = p.pg[1] * 2654435761u, y1 = y0 + 2654435761u;
    const uint32_t z0 = p.pg[2] * 805459861u, z1 = z0 + 805459861u;
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
        // the two corners of an x edge: x and x + 1 mostly differ in the low bits only
        const uint32_t yz = (k & 2 ? y1 : y0) ^ (k & 4 ? z1 : z0);
        const uint32_t a = (p.pg[0] ^ yz) & (hs - 1), b = ((p.pg[0] + 1) ^ yz) & (hs - 1);
        const bool ina = !p.oob && a - lo < width, inb = !p.oob && b - lo < width;
        union {
            uint4 q;
            T v[QR * C];
        } e;  // not used unless loaded
        if (ina) e.q = *(const uint4*)(g + (a & ~(uint32_t)(QR - 1)) * C);
        if constexpr (sizeof(T) == 4) {
            T va = e.v[0], vb = e.v[0];
#pragma unroll
            for (int i = 1; i < 4; i++) {
                va = (a & 3) == i ? e.v[i] : va;
                vb = (b & 3) == i ? e.v[i] : vb;
            }
            row[k].v[0] = ina ? va : row[k].v[0];
            row[k + 1].v[0] = ina && (a ^ b) < QR ? vb : row[k + 1].v[0];
        } else {
            const uint32_t va = quad_row<QR>(e.q, a), vb = quad_row<QR>(e.q, b);
            row[k].bits = ina ? va : row[k].bits;
            row[k + 1].bits = ina && (a ^ b) < QR ? vb : row[k + 1].bits;
        }
        if (inb && (a ^ b) >= QR) {
#pragma unroll
            for (int c = 0; c < C; c++) row[k + 1].v[c] = g[b * C + c];
        }
    }
}

// any other level; r1 > 0: a lattice of r1^3 <= hs rows (no remainder to take)
template <typename T, int C>
__device__ __forceinline__ void level_direct(const LevelPoint& p, const T* __restrict__ g, uint32_t hs, uint32_t res,
                                             uint32_t r1, int gridtype, int align, GridRow<T, C> (&row)[8]) {
    if (p.oob) return;
    const uint32_t r0 = p.pg[0] + r1 * (p.pg[1] + r1 * p.pg[2]);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        uint32_t at = r0 + (k & 1) + (k & 2 ? r1 : 0) + (k & 4 ? r1 * r1 : 0);
        if (r1 == 0) {
            const uint32_t loc[3] = {p.pg[0] + (k & 1), p.pg[1] + ((k >> 1) & 1), p.pg[2] + (k >> 2)};
            at = grid_index<3>(gridtype, align != 0, hs, res, loc);
        }
#pragma unroll
        for (int c = 0; c < C; c++) row[k].v[c] = g[at * C + c];
    }
}

template <typename T, int C>
__device__ __forceinline__ void level_store(float* __restrict__ stage, int64_t n, int level, int64_t b,
                                            const float (&acc)[C]) {
    if (b < n) {
#pragma unroll
        for (int c = 0; c < C; c++) stage[((int64_t)level * n + b) * C + c] = acc[c];
    }
}

template <typename T, int C>
__global__ __launch_bounds__(LS_THREADS) void prop_level_kernel(PropArgs P, int64_t b0, int64_t n,
                                                                float* __restrict__ stage, int ppt) {
    extern __shared__ float ls[];  // [ppt][3][LS_THREADS]: the points' coordinates
    const int t = threadIdx.x;
    for (int64_t p0 = (int64_t)blockIdx.x * LS_THREADS * ppt; p0 < n; p0 += (int64_t)gridDim.x * LS_THREADS * ppt) {
        for (int q = 0; q < ppt; q++) {
            float cw[3], x01[3];
            prop_warp(P, b0 + min(p0 + q * LS_THREADS + t, n - 1), cw, x01);
#pragma unroll
            for (int d = 0; d < 3; d++) ls[(q * 3 + d) * LS_THREADS + t] = x01[d];
        }
        for (int level = 0; level < P.L; level++) {
            const uint32_t hs = (uint32_t)(P.offsets[level + 1] - P.offsets[level]);
            const float scale = P.lt.scale[level];
            const uint32_t res = (uint32_t)ceilf(scale) + 1, r1 = res + 1;
            const T* g = (const T*)P.emb + (int64_t)P.offsets[level] * C;
            // r1 below 1626: its cube fits 32 bits; below 65536: its square does
            const bool lattice = !P.align && r1 < 1626u && r1 * r1 * r1 <= hs;
            const bool hashed = !P.align && P.gridtype == 0 && r1 < 65536u && !lattice && (hs & (hs - 1)) == 0 &&
                                !(r1 >= 1626u && r1 * r1 <= hs) && hs >= 16 && ((uintptr_t)g & 15) == 0;
            const uint32_t part = (uint32_t)(LS_PART_BYTES / (C * (int)sizeof(T)));
            if (C == 1 && hashed && hs > part) {
                GridRow<T, C> row[LS_POINTS][8];
#pragma unroll
                for (int q = 0; q < LS_POINTS; q++)
#pragma unroll
                    for (int k = 0; k < 8; k++) row[q][k].bits = 0;
                for (uint32_t lo = 0; lo < hs; lo += part) {
#pragma unroll
                    for (int q = 0; q < LS_POINTS; q++) {
                        if (q < ppt)
                            level_hashed<T, C>(level_point(ls + q * 3 * LS_THREADS + t, scale, 0, 0), g, hs, lo, part,
                                               row[q]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (int q = 0; q < LS_POINTS; q++) {
                    if (q < ppt) {
                        float acc[C];
                        level_sum<T, C>(level_point(ls + q * 3 * LS_THREADS + t, scale, 0, P.interp), row[q], acc);
                        level_store<T, C>(stage, n, level, p0 + q * LS_THREADS + t, acc);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll 2
                for (int q = 0; q < ppt; q++) {
                    LevelPoint p = level_point(ls + q * 3 * LS_THREADS + t, scale, P.align, P.interp);
                    if (hs == 0) p.oob = true;  // an empty level
                    GridRow<T, C> row[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) row[k].bits = 0;
                    if (hashed) level_hashed<T, C>(p, g, hs, 0, hs, row);
                    else level_direct<T, C>(p, g, hs, res, lattice ? r1 : 0, P.gridtype, P.align, row);
                    float acc[C];
                    level_sum<T, C>(p, row, acc);
                    level_store<T, C>(stage, n, level, p0 + q * LS_THREADS + t, acc);
                }
            }
        }
    }
}

// torch.nn.functional.softplus (beta 1, threshold 20) and its derivative
__device__ __forceinline__ float softplus20(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float dsoftplus20(float x) { return x > 20.f ? 1.f : 1.f / (1.f + expf(-x)); }

template <int FM>
__device__ __forceinline__ float prop_raw(const float* sW1, const float* sb1, const float* sW2, float b2, int F,
                                          const float* f) {
    float raw = b2;
#pragma unroll 4
    for (int j = 0; j < PF_HID; j++) {
        float a = sb1[j];
#pragma unroll
        for (int i = 0; i < FM; i++)
            if (i < F) a += sW1[j * F + i] * f[i];
        raw += sW2[j] * fmaxf(a, 0.f);
    }
    return raw;
}

// FM: per-lane feature capacity (16 or 32 >= F)
// FX > 0: the feature count is FX (= FM) at compile time
// STAGED: points [b0, b0 + n) with their features from prop_level_kernel's [L, n, C]
template <typename T, int C, int FM, int FX = 0, bool STAGED = false>
__global__ __launch_bounds__(PF_FWD_THREADS) void prop_fwd_kernel(PropArgs P, const float* __restrict__ stage,
                                                                  int64_t b0, int64_t n, float* __restrict__ density,
                                                                  float* __restrict__ coord_out,
                                                                  float* __restrict__ feat_out,
                                                                  float* __restrict__ x01_out) {
    __shared__ float sW1[PF_HID * PF_MAXF], sb1[PF_HID], sW2[PF_HID];
    const int F = FX > 0 ? FX : P.L * C;
    for (int i = threadIdx.x; i < PF_HID * F; i += PF_FWD_THREADS) sW1[i] = P.W1[i];
    for (int i = threadIdx.x; i < PF_HID; i += PF_FWD_THREADS) {
        sb1[i] = P.b1[i];
        sW2[i] = P.W2[i];
    }
    __syncthreads();
    const float b2 = P.b2[0];
    for (int64_t i = (int64_t)blockIdx.x * PF_FWD_THREADS + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * PF_FWD_THREADS) {
        const int64_t b = STAGED ? b0 + i : i;  // (b0 is 0 without the stage)
        float cw[3], x01[3], f[FM];
        prop_warp(P, b, cw, x01);
        if constexpr (STAGED) {
#pragma unroll
            for (int l = 0; l < FM / C; l++)
#pragma unroll
                for (int c = 0; c < C; c++) f[l * C + c] = l < P.L ? stage[((int64_t)l * n + i) * C + c] : 0.f;
        } else {
            prop_features<T, C, FM>(P, x01, f);
        }
        const float raw = prop_raw<FM>(sW1, sb1, sW2, b2, F, f);
        density[b] = softplus20(raw + P.dbias);
        if (coord_out) {
#pragma unroll
            for (int d = 0; d < 3; d++) coord_out[b * 3 + d] = cw[d];
        }
        if (feat_out) {  // kept for the adjoint, which then gathers nothing
#pragma unroll
            for (int i = 0; i < FM; i++)
                if (i < F) feat_out[b * F + i] = f[i];
#pragma unroll
            for (int d = 0; d < 3; d++) x01_out[b * 3 + d] = x01[d];
        }
    }
}

typedef float f4 __attribute__((ext_vector_type(4)));

// D = A B + C in float32 on the matrix cores: A 16 x 4 (lane l: row l % 16, column l / 16),
// B 4 x 16 (lane l: column l % 16, row l / 16), C and D 16 x 16 (lane l: column l % 16, rows
// 4 (l / 16) + 0..3).
__device__ __forceinline__ f4 mfma16(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Adjoint of the head.  Its contractions (hidden units from features, the density from the
// hidden units, feature gradients from hidden gradients, weight gradients over the points) run
// on the matrix cores in float32, 16 points at a time:
//   H [hidden x point] = W1 F: the operands' lanes hold W1 and the features; a lane then has
//     4 hidden units of one point per 16 x 16 tile, at once the right operand of
//   raw = W2 relu(H), the units in their order, as one lane sums them in the forward (summed
//     by lanes first, the density's last bits differ: where the bias's gradient cancels over
//     the points, its error against 64 bits grew from below 1e-6 to above); dH in H's place is
//     the right operand of
//   dF [feature x point] = W1^T dH (step r takes the units 4 r + l / 16);
//   H' [point x hidden] = the first product with its operands exchanged: dH' of it is the
//     right operand of dW1 [feature x hidden] += F^T dH', summed over PF_HELD tiles of a
//     wavefront's points in the accumulator registers.
// 72 matrix instructions per 16 points and 10 features.  The vector version went through
// LDS for every product (7 LDS reads per point and hidden unit): 1560 us at 4.2 M points.
template <typename T, int C, int FM, int FX = 0>
__global__ __launch_bounds__(pf_bwd_threads(FM), pf_bwd_blocks(FM)) void prop_bwd_kernel(PropArgs P, const float* __restrict__ gdens,
                                                                  const float* __restrict__ feat_in,
                                                                  float* __restrict__ gfeat, float* __restrict__ x01_out,
                                                                  float* __restrict__ gW1, float* __restrict__ gb1,
                                                                  float* __restrict__ gW2, float* __restrict__ gb2,
                                                                  double* __restrict__ gsum) {
    constexpr int NT = pf_bwd_threads(FM), NW = NT / 64, KS = (FM + 3) / 4, FT = (FM + 15) / 16, HT = PF_HID / 16;
    constexpr int FP = 16 * FT + 1;  // row of a point's features in LDS
    __shared__ float sf[NW][64][FP];  // a wavefront's 64 points: features, then their gradients
    __shared__ double sum[PF_HID * (FM + 2) + 1];  // dW1 [hidden, feature], db1, dW2, db2 of the block
    const int F = FX > 0 ? FX : P.L * C;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int lc = lane & 15, lr = lane >> 4;
    for (int i = threadIdx.x; i < PF_HID * (FM + 2) + 1; i += NT) sum[i] = 0.0;
    // A tile's row 4 a + b is hidden unit 16 t + 4 b + a, so that a lane's r-th unit of H is the
    // k-th of the r-th step of a product over the units in their order: jl is lc's unit.
    const int jl = 4 * (lc & 3) + (lc >> 2);
    // constant operands: w1[t][k] = W1[16 t + jl][4 k + lr], w1t[q][t][r] = W1[16 t + 4 r + lr][16 q + lc]
    float w1[HT][KS], w1t[FT][HT][4], b1q[HT], w2q[HT];
    f4 b1p[HT], w2p[HT];
#pragma unroll
    for (int t = 0; t < HT; t++) {
#pragma unroll
        for (int k = 0; k < KS; k++) w1[t][k] = 4 * k + lr < F ? P.W1[(16 * t + jl) * F + 4 * k + lr] : 0.f;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 16 * t + 4 * r + lr;
#pragma unroll
            for (int q = 0; q < FT; q++) w1t[q][t][r] = 16 * q + lc < F ? P.W1[j * F + 16 * q + lc] : 0.f;
            b1p[t][r] = P.b1[j];
            w2p[t][r] = P.W2[j];
        }
        b1q[t] = P.b1[16 * t + jl];
        w2q[t] = P.W2[16 * t + jl];
    }
    const float b2 = P.b2[0];
    f4 aw1[FT][HT];
    float ab1[HT], aw2[HT];
    double ab2 = 0.0;  // 16 lanes take all of the wavefront's points: in float32 less exact than a lane per point
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < HT; t++) {
            ab1[t] = aw2[t] = 0.f;
#pragma unroll
            for (int q = 0; q < FT; q++) aw1[q][t] = (f4){0.f, 0.f, 0.f, 0.f};
        }
    };
    // the wavefronts' sums meet in LDS, one global atomic per weight and block at the end
    auto drain = [&]() {
#pragma unroll
        for (int t = 0; t < HT; t++) {
            const int j = 16 * t + jl;
#pragma unroll
            for (int q = 0; q < FT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = 16 * q + 4 * lr + r;
                    if (i < F) atomicAdd(&sum[j * FM + i], (double)aw1[q][t][r]);
                }
            atomicAdd(&sum[PF_HID * FM + j], (double)ab1[t]);
            atomicAdd(&sum[PF_HID * (FM + 1) + j], (double)aw2[t]);
        }
    };
    clear();
    int held = 0;
    __syncthreads();
    const int64_t ntile = (P.N + 63) / 64;
    for (int64_t tile = (int64_t)blockIdx.x * NW + wave; tile < ntile; tile += (int64_t)gridDim.x * NW) {
        const int64_t b0 = tile * 64;
        const int np = (int)min((int64_t)64, P.N - b0);
        float(*pt)[FP] = sf[wave];
        if (feat_in) {
            for (int i = lane; i < 64 * 16 * FT; i += 64) {
                const int p = i / (16 * FT), c = i - p * (16 * FT);
                if (c >= F || p >= np) pt[p][c] = 0.f;
            }
            for (int i = lane; i < np * F; i += 64) {
                const int p = i / F;
                pt[p][i - p * F] = feat_in[b0 * F + i];
            }
        } else {
            float f[FM], cw[3], x01[3];
#pragma unroll
            for (int i = 0; i < FM; i++) f[i] = 0.f;
            if (lane < np) {
                prop_warp(P, b0 + lane, cw, x01);
                prop_features<T, C, FM>(P, x01, f);
#pragma unroll
                for (int d = 0; d < 3; d++) x01_out[(b0 + lane) * 3 + d] = x01[d];
            }
#pragma unroll
            for (int i = 0; i < 16 * FT; i++) pt[lane][i] = i < FM && i < F ? f[i < FM ? i : 0] : 0.f;
        }
        const float gown = lane < np ? gdens[b0 + lane] : 0.f;
        wave_fence();
#pragma unroll 1
        for (int s = 0; s < 4; s++) {  // 16 points
            float f[KS], ft[FT][4];
#pragma unroll
            for (int k = 0; k < KS; k++) f[k] = pt[16 * s + lc][4 * k + lr];
#pragma unroll
            for (int q = 0; q < FT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) ft[q][r] = pt[16 * s + 4 * lr + r][16 * q + lc];
            wave_fence();  // every lane has read the rows that the gradients go to below
            f4 h[HT];
#pragma unroll
            for (int t = 0; t < HT; t++) {
                h[t] = b1p[t];
#pragma unroll
                for (int k = 0; k < KS; k++) h[t] = mfma16(w1[t][k], f[k], h[t]);
            }
            // without a point in the last tile no unit is on and the gradient is 0, whatever the
            // weights are (0 times an infinite one is NaN)
            const bool on = 16 * s + lc < np;
            // every row of the product is the density's pre-activation, its 64 terms in order
            f4 raw = (f4){b2, b2, b2, b2};
#pragma unroll
            for (int t = 0; t < HT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) raw = mfma16(w2p[t][r], fmaxf(h[t][r], 0.f), raw);
            const float gp = __shfl(gown, 16 * s + lc, 64) * dsoftplus20(raw[0] + P.dbias), g = on ? gp : 0.f;
            if (lr == 0) ab2 += (double)g;
            f4 df[FT];
#pragma unroll
            for (int q = 0; q < FT; q++) df[q] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < HT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float dh = h[t][r] > 0.f && on ? g * w2p[t][r] : 0.f;
#pragma unroll
                    for (int q = 0; q < FT; q++) df[q] = mfma16(w1t[q][t][r], dh, df[q]);
                }
            float gq[4];
#pragma unroll
            for (int r = 0; r < 4; r++) gq[r] = __shfl(g, 4 * lr + r, 64);
#pragma unroll
            for (int t = 0; t < HT; t++) {
                f4 hq = (f4){b1q[t], b1q[t], b1q[t], b1q[t]};
#pragma unroll
                for (int k = 0; k < KS; k++) hq = mfma16(f[k], w1[t][k], hq);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float dh = hq[r] > 0.f && 16 * s + 4 * lr + r < np ? gq[r] * w2q[t] : 0.f;
                    ab1[t] += dh;
                    aw2[t] += gq[r] * fmaxf(hq[r], 0.f);
#pragma unroll
                    for (int q = 0; q < FT; q++) aw1[q][t] = mfma16(ft[q][r], dh, aw1[q][t]);
                }
            }
            // the points' features are done with: their gradients take the place
#pragma unroll
            for (int q = 0; q < FT; q++)
#pragma unroll
                for (int r = 0; r < 4; r++) pt[16 * s + lc][16 * q + 4 * lr + r] = df[q][r];
        }
        wave_fence();
        for (int i = lane; i < np * F; i += 64) {
            const int p = i / F;
            gfeat[b0 * F + i] = pt[p][i - p * F];
        }
        wave_fence();
        if (++held == PF_HELD) {
            drain();
            clear();
            held = 0;
        }
    }
    drain();
    if (lr == 0) atomicAdd(&sum[PF_HID * (FM + 2)], ab2);
    __syncthreads();
    if (gsum) {  // [W1 | b1 | W2 | b2] in doubles: what the order of the blocks rounds is far below a float's last bit
        for (int i = threadIdx.x; i < PF_HID * (F + 2) + 1; i += NT)
            atomicAdd(&gsum[i], i < PF_HID * F ? sum[(i / F) * FM + i % F] : sum[PF_HID * FM + i - PF_HID * F]);
        return;
    }
    for (int i = threadIdx.x; i < PF_HID * F; i += NT)
        atomicAdd(&gW1[i], (float)sum[(i / F) * FM + i % F]);
    for (int i = threadIdx.x; i < PF_HID; i += NT) {
        atomicAdd(&gb1[i], (float)sum[PF_HID * FM + i]);
        atomicAdd(&gW2[i], (float)sum[PF_HID * (FM + 1) + i]);
    }
    if (threadIdx.x == 0) atomicAdd(&gb2[0], (float)sum[PF_HID * (FM + 2)]);
}

#define N3DS_GRID_DISPATCH(KERNEL_LAUNCH)                                                           \
    switch (D * 16 + C) {                                                                          \
        case 2 * 16 + 1: KERNEL_LAUNCH(2, 1); break;                                               \
        case 2 * 16 + 2: KERNEL_LAUNCH(2, 2); break;                                               \
        case 2 * 16 + 4: KERNEL_LAUNCH(2, 4); break;                                               \
        case 2 * 16 + 8: KERNEL_LAUNCH(2, 8); break;                                               \
        case 3 * 16 + 1: KERNEL_LAUNCH(3, 1); break;                                               \
        case 3 * 16 + 2: KERNEL_LAUNCH(3, 2); break;                                               \
        case 3 * 16 + 4: KERNEL_LAUNCH(3, 4); break;                                               \
        case 3 * 16 + 8: KERNEL_LAUNCH(3, 8); break;                                               \
        case 4 * 16 + 2: KERNEL_LAUNCH(4, 2); break;                                               \
        case 5 * 16 + 2: KERNEL_LAUNCH(5, 2); break;                                               \
        default: N3DS_REQUIRE(false, "unsupported input_dim %d / level_dim %d", D, C);             \
    }

static int grid_check(int64_t B, int D, int C, int L, int dtype) {
    N3DS_REQUIRE(B >= 0 && L > 0 && L <= MAX_LEVELS, "bad sizes B=%lld L=%d", (long long)B, L);
    N3DS_REQUIRE(D >= 2 && D <= 5, "input_dim must be in [2, 5] (got %d)", D);
    N3DS_REQUIRE(C == 1 || C == 2 || C == 4 || C == 8, "level_dim must be 1, 2, 4 or 8 (got %d)", C);
    N3DS_REQUIRE(dtype == 0 || dtype == 1, "dtype must be 0 (float32) or 1 (float16)");
    return N3DS_OK;
}

}  // namespace n3ds

using namespace n3ds;

N3DS_EXPORT int n3ds_grid_encode_forward(const float* inputs, const void* embeddings, const int32_t* offsets,
                                         void* outputs, int64_t B, int D, int C, int L, float S, int H, void* dy_dx,
                                         int gridtype, int align_corners, int interp, int dtype, void* stream) {
    int st = grid_check(B, D, C, L, dtype);
    const LevelTab lt = make_level_tab(L, S, H);
    if (st) return st;
    if (B == 0) return N3DS_OK;
    dim3 grid((unsigned)((B * L + 255) / 256));
    hipStream_t s = (hipStream_t)stream;
    const bool tiled = dy_dx == nullptr && L * C <= GT_MAX_LC;
    const dim3 tgrid((unsigned)((B + GT - 1) / GT));
    const size_t tlds = (size_t)GT * (L * C + 1) * sizeof(float);
#define LAUNCH_F(DD, CC)                                                                                         \
    if (tiled && dtype == 0)                                                                                     \
        hipLaunchKernelGGL((grid_fwd_tile_kernel<float, DD, CC>), tgrid, dim3(GT), tlds, s, inputs,              \
                           (const float*)embeddings, offsets, (float*)outputs, B, L, lt, gridtype, align_corners, \
                           interp);                                                                              \
    else if (tiled)                                                                                              \
        hipLaunchKernelGGL((grid_fwd_tile_kernel<__half, DD, CC>), tgrid, dim3(GT), tlds, s, inputs,             \
                           (const __half*)embeddings, offsets, (__half*)outputs, B, L, lt, gridtype,             \
                           align_corners, interp);                                                               \
    else if (dtype == 0)                                                                                         \
        hipLaunchKernelGGL((grid_fwd_kernel<float, DD, CC>), grid, dim3(256), 0, s, inputs, (const float*)embeddings, \
                           offsets, (float*)outputs, B, L, lt, (float*)dy_dx, gridtype, align_corners, interp); \
    else                                                                                                         \
        hipLaunchKernelGGL((grid_fwd_kernel<__half, DD, CC>), grid, dim3(256), 0, s, inputs,                     \
                           (const __half*)embeddings, offsets, (__half*)outputs, B, L, lt,            \
                           (__half*)dy_dx, gridtype, align_corners, interp);
    N3DS_GRID_DISPATCH(LAUNCH_F)
#undef LAUNCH_F
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

N3DS_EXPORT int64_t n3ds_grid_encode_backward_workspace_bytes(int64_t B, int D, int C, int L, int64_t n_rows) {
    if (B < 0 || D < 1 || D > 5 || C < 1 || C > 8 || L < 1 || n_rows < 0) return -1;
    // either scatter (the grid type, alignment and scales are not known here)
    const int64_t gb = gb_workspace_bytes(B, D, C, L, n_rows);
    const int64_t gs = D == 3 ? gs_workspace_bytes(B, C, L) : 0;
    return gb > gs ? gb : gs;
}

// grad_embeddings_f32: fp32 accumulation table (zero-initialised by the caller);
// grad_embeddings_out: optional table of the embedding dtype that receives the
// rounded result (may alias grad_embeddings_f32 when dtype == float32).
// workspace (workspace_bytes >= n3ds_grid_encode_backward_workspace_bytes):
// bucketed scatter; NULL: one float atomic per contribution.
N3DS_EXPORT int n3ds_grid_encode_backward(const void* grad, const float* inputs, const int32_t* offsets,
                                          float* grad_embeddings_f32, void* grad_embeddings_out, int64_t n_rows,
                                          int64_t B, int D, int C, int L, float S, int H, const void* dy_dx,
                                          void* grad_inputs, int gridtype, int align_corners, int interp, int dtype,
                                          void* workspace, int64_t workspace_bytes, void* stream) {
    int st = grid_check(B, D, C, L, dtype);
    const LevelTab lt = make_level_tab(L, S, H);
    if (st) return st;
    hipStream_t s = (hipStream_t)stream;
    const bool bucketed = workspace != nullptr;
    if (bucketed)
        N3DS_REQUIRE(workspace_bytes >= gb_workspace_bytes(B, D, C, L, n_rows), "grid workspace too small");
    const bool sorted = bucketed && gs_applies(B, D, C, L, n_rows, gridtype, align_corners, lt) &&
                        workspace_bytes >= gs_workspace_bytes(B, C, L);
    if (B > 0 && sorted && n_rows > 0) {
#define LAUNCH_S(CC)                                                                                             \
    st = dtype == 0 ? gs_launch<float, CC>((const float*)grad, inputs, offsets, B, L, lt, interp, workspace,     \
                                           grad_embeddings_f32, s)                                               \
                    : gs_launch<__half, CC>((const __half*)grad, inputs, offsets, B, L, lt, interp, workspace,   \
                                            grad_embeddings_f32, s)
        switch (C) {
            case 1: LAUNCH_S(1); break;
            case 2: LAUNCH_S(2); break;
            case 4: LAUNCH_S(4); break;
            default: LAUNCH_S(8); break;
        }
#undef LAUNCH_S
        if (st) return st;
    } else if (B > 0 && bucketed && n_rows > 0) {
        const GridBucketWs ws = gb_carve(workspace, B, D, C, L, n_rows);
        const int64_t NB = gb_num_buckets(n_rows, C);
        hipLaunchKernelGGL(grid_fill_int_kernel, dim3((unsigned)((NB + 255) / 256)), dim3(256), 0, s, ws.count, NB);
        N3DS_LAUNCH_CHECK();
        dim3 gpass((unsigned)((B + GB_THREADS * GB_PPT - 1) / (GB_THREADS * GB_PPT)), (unsigned)L);
        const int64_t max_segs = (B * L * (1ll << D) + GB_SEG - 1) / GB_SEG + NB;
#define LAUNCH_G(DD, CC)                                                                                          \
    if (dtype == 0) {                                                                                             \
        hipLaunchKernelGGL((grid_bucket_kernel<float, DD, CC, 0>), gpass, dim3(GB_THREADS), 0, s,                 \
                           (const float*)grad, inputs, offsets, B, L, lt, gridtype, align_corners, interp, ws);   \
        hipLaunchKernelGGL(grid_bucket_scan_kernel, dim3(1), dim3(1024), 0, s, ws, NB);                           \
        hipLaunchKernelGGL((grid_bucket_kernel<float, DD, CC, 1>), gpass, dim3(GB_THREADS), 0, s,                 \
                           (const float*)grad, inputs, offsets, B, L, lt, gridtype, align_corners, interp, ws);   \
    } else {                                                                                                      \
        hipLaunchKernelGGL((grid_bucket_kernel<__half, DD, CC, 0>), gpass, dim3(GB_THREADS), 0, s,                \
                           (const __half*)grad, inputs, offsets, B, L, lt, gridtype, align_corners, interp, ws);  \
        hipLaunchKernelGGL(grid_bucket_scan_kernel, dim3(1), dim3(1024), 0, s, ws, NB);                           \
        hipLaunchKernelGGL((grid_bucket_kernel<__half, DD, CC, 1>), gpass, dim3(GB_THREADS), 0, s,                \
                           (const __half*)grad, inputs, offsets, B, L, lt, gridtype, align_corners, interp, ws);  \
    }                                                                                                             \
    hipLaunchKernelGGL((grid_bucket_reduce_kernel<CC>), dim3((unsigned)max_segs), dim3(GB_THREADS), 0, s, ws, NB, \
                       n_rows, grad_embeddings_f32);
        N3DS_GRID_DISPATCH(LAUNCH_G)
#undef LAUNCH_G
        N3DS_LAUNCH_CHECK();
    }
    if (B > 0) {
        dim3 grid((unsigned)((B * L + 255) / 256));
        const bool tiled = L * C <= GT_MAX_LC;
        const dim3 tgrid((unsigned)((B + GT - 1) / GT));
        const size_t tlds = (size_t)GT * (L * C + 1) * sizeof(float);
#define LAUNCH_B(DD, CC)                                                                                          \
    if (!bucketed && tiled && dtype == 0)                                                                         \
        hipLaunchKernelGGL((grid_bwd_tile_kernel<float, DD, CC>), tgrid, dim3(GT), tlds, s, (const float*)grad,   \
                           inputs, offsets, grad_embeddings_f32, B, L, lt, gridtype, align_corners, interp);      \
    else if (!bucketed && tiled)                                                                                  \
        hipLaunchKernelGGL((grid_bwd_tile_kernel<__half, DD, CC>), tgrid, dim3(GT), tlds, s, (const __half*)grad, \
                           inputs, offsets, grad_embeddings_f32, B, L, lt, gridtype, align_corners, interp);      \
    else if (!bucketed && dtype == 0)                                                                             \
        hipLaunchKernelGGL((grid_bwd_kernel<float, DD, CC>), grid, dim3(256), 0, s, (const float*)grad, inputs,   \
                           offsets, grad_embeddings_f32, B, L, lt, gridtype, align_corners, interp);   \
    else if (!bucketed)                                                                                           \
        hipLaunchKernelGGL((grid_bwd_kernel<__half, DD, CC>), grid, dim3(256), 0, s, (const __half*)grad, inputs, \
                           offsets, grad_embeddings_f32, B, L, lt, gridtype, align_corners, interp);   \
    if (dy_dx && grad_inputs) {                                                                                   \
        dim3 g2((unsigned)((B * DD + 255) / 256));                                                                \
        if (dtype == 0)                                                                                           \
            hipLaunchKernelGGL((grid_input_bwd_kernel<float, DD, CC>), g2, dim3(256), 0, s, (const float*)grad,   \
                               (const float*)dy_dx, (float*)grad_inputs, B, L);                                   \
        else                                                                                                      \
            hipLaunchKernelGGL((grid_input_bwd_kernel<__half, DD, CC>), g2, dim3(256), 0, s, (const __half*)grad, \
                               (const __half*)dy_dx, (__half*)grad_inputs, B, L);                                 \
    }
        N3DS_GRID_DISPATCH(LAUNCH_B)
#undef LAUNCH_B
        N3DS_LAUNCH_CHECK();
    }
    if (grad_embeddings_out && dtype == 1 && n_rows > 0) {
        int64_t n = n_rows * C;
        hipLaunchKernelGGL(f32_to_kernel<__half>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                           grad_embeddings_f32, (__half*)grad_embeddings_out, n);
        N3DS_LAUNCH_CHECK();
    }
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_grid_grad_tv(const float* inputs, const void* embeddings, float* grad_f32, const int32_t* offsets,
                                  float weight, int64_t B, int D, int C, int L, float S, int H, int gridtype,
                                  int align_corners, int dtype, void* stream) {
    int st = grid_check(B, D, C, L, dtype);
    const LevelTab lt = make_level_tab(L, S, H);
    if (st) return st;
    if (B == 0) return N3DS_OK;
    dim3 grid((unsigned)((B * L + 255) / 256));
    hipStream_t s = (hipStream_t)stream;
#define LAUNCH_T(DD, CC)                                                                                         \
    if (dtype == 0)                                                                                              \
        hipLaunchKernelGGL((grid_tv_kernel<float, DD, CC>), grid, dim3(256), 0, s, inputs, (const float*)embeddings, \
                           grad_f32, offsets, weight, B, L, lt, gridtype, align_corners);             \
    else                                                                                                         \
        hipLaunchKernelGGL((grid_tv_kernel<__half, DD, CC>), grid, dim3(256), 0, s, inputs,                      \
                           (const __half*)embeddings, grad_f32, offsets, weight, B, L, lt, gridtype,  \
                           align_corners);
    N3DS_GRID_DISPATCH(LAUNCH_T)
#undef LAUNCH_T
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

// ---------------------------------------------------------------------------
// fused proposal density field entry points
// ---------------------------------------------------------------------------
static int prop_check(int64_t N, int C, int L, int dtype, int warp) {
    N3DS_REQUIRE(N >= 0, "bad point count");
    N3DS_REQUIRE(C == 1 || C == 2 || C == 4, "level_dim must be 1, 2 or 4 (got %d)", C);
    N3DS_REQUIRE(L >= 1 && L * C <= PF_MAXF, "num_levels * level_dim must be in [1, %d] (got %d x %d)", PF_MAXF, L, C);
    N3DS_REQUIRE(dtype == 0 || dtype == 1, "dtype must be 0 (float32) or 1 (float16)");
    N3DS_REQUIRE(warp >= 0 && warp <= 2, "warp must be 0 (none), 1 (contract) or 2 (box)");
    return N3DS_OK;
}

static PropArgs prop_args(const float* coords, int64_t N, int warp, float box_size, const void* emb,
                          const int32_t* offsets, int L, float S, int H, int gridtype, int align, int interp,
                          const float* W1, const float* b1, const float* W2, const float* b2, float dbias) {
    PropArgs P;
    P.coords = coords; P.N = N; P.warp = warp; P.inv_half_box = box_size > 0.f ? 2.f / box_size : 1.f;
    P.emb = emb; P.offsets = offsets; P.L = L; P.lt = make_level_tab(L, S, H);
    P.gridtype = gridtype; P.align = align; P.interp = interp;
    P.W1 = W1; P.b1 = b1; P.W2 = W2; P.b2 = b2; P.dbias = dbias;
    return P;
}

// The staged features pay where the tables do not fit an L2, 16 bytes hold four rows or more,
// and there are enough points to fetch every table into every L2 for.  Forward with kept
// features, staged against fused (us), 10 levels:
//   rows of 4 bytes, tables of 57 MB: 2^17 points 75 / 65, 2^18 97 / 122, 2^22 1435 / 1848;
//   15 MB: 2^17 65 / 47, 2^18 72 / 88, 2^22 970 / 1420; 4.2 MB: 2^18 62 / 63, 2^21 385 / 437;
//   two half features, levels of 2 MB: 2^17 73 / 50, 2^18 89 / 93, 2^22 1130 / 1478; four of
//   ten of 8 MB (42 MB; the whole call): 2^20 640 / 610, 2^22 1863 / 1870 (in parts, spilling the
//   rows kept: 750, 2185);
//   rows of 8 bytes, 30 MB: 2^18 117 / 110, 2^21 917 / 862; of 16 bytes: 2^21 1412 / 1119.
// The head of ten levels is compiled for its 10 or 20 features; any other count's loops to 16 or
// 32, which the one kernel does in the shadow of its gathers, so there levels must stay in an L2
// (2 MB at most) for more points (the whole call, 2^20 and 2^22 points):
//   7 levels to 2 MB: 394 / 383, 1201 / 1185; 8: 438 / 443, 1386 / 1427; 16: 866 / 942, 2934 / 3412;
//   8 levels to 4 MB: 520 / 489, 1690 / 1583; 16: 1121 / 1016, 3400 / 3400; to 8 MB: 551 / 539,
//   1763 / 1726; 1154 / 1109, 3685 / 3876; two half features, 12 levels to 4 MB: 1026 / 900,
//   3304 / 3001.
constexpr int64_t PF_STAGE_TABLE = 4 << 20;  // bytes of all tables
constexpr int64_t PF_STAGE_ROW = 4;          // bytes of a row at most
constexpr int64_t PF_STAGE_POINTS = 1 << 18;
constexpr int64_t PF_STAGE_CHUNK = 1 << 22;  // points whose features are staged at one time
constexpr int PF_STAGE_LEVELS = 8;               // not ten of them: levels,
constexpr int64_t PF_STAGE_LEVEL = 7 << 18;      // bytes of one on average at most,
constexpr int64_t PF_STAGE_MORE = 1 << 20;       // and points

N3DS_EXPORT int64_t n3ds_prop_field_workspace_bytes(int64_t n_points, int num_levels, int level_dim, int64_t n_rows,
                                                    int dtype) {
    if (n_points < PF_STAGE_POINTS || num_levels < 1 || level_dim < 1 || n_rows < 0) return 0;
    const int64_t row = level_dim * (dtype == 1 ? 2 : 4);
    if (row > PF_STAGE_ROW || n_rows * row <= PF_STAGE_TABLE) return 0;
    if (num_levels != 10 && (level_dim != 1 || num_levels < PF_STAGE_LEVELS || n_points < PF_STAGE_MORE ||
                             n_rows * row > num_levels * PF_STAGE_LEVEL))
        return 0;
    // two half features take a level whole: past an L2 a level on average the gathers leave it
    if (level_dim == 2 && n_rows * row > num_levels * LS_PART_BYTES) return 0;
    return std::min(n_points, PF_STAGE_CHUNK) * num_levels * level_dim * 4;
}

// n3ds_prop_field_forward with device scratch of n3ds_prop_field_workspace_bytes (n_rows: rows of
// the whole table); with NULL or fewer bytes, or where that is 0, one kernel as without it.
N3DS_EXPORT int n3ds_prop_field_forward_ws(const float* coords, int64_t n_points, int warp, float box_size,
                                           const void* embeddings, const int32_t* offsets, int num_levels,
                                           int level_dim, float S, int H, int gridtype, int align_corners, int interp,
                                           int dtype, const float* w1, const float* b1, const float* w2,
                                           const float* b2, float density_bias, float* density_out,
                                           float* coord_out, float* features_out, float* grid_inputs_out,
                                           int64_t n_rows, void* workspace, int64_t workspace_bytes, void* stream) {
    N3DS_REQUIRE((features_out == nullptr) == (grid_inputs_out == nullptr),
                 "features_out and grid_inputs_out are kept together");
    int st = prop_check(n_points, level_dim, num_levels, dtype, warp);
    if (st) return st;
    if (n_points == 0) return N3DS_OK;
    const PropArgs P = prop_args(coords, n_points, warp, box_size, embeddings, offsets, num_levels, S, H, gridtype,
                                 align_corners, interp, w1, b1, w2, b2, density_bias);
    hipStream_t s = (hipStream_t)stream;
    const int64_t need = n3ds_prop_field_workspace_bytes(n_points, num_levels, level_dim, n_rows, dtype);
    const bool staged = need > 0 && workspace != nullptr && workspace_bytes >= need;
    float* stage = (float*)workspace;
    const int64_t step = staged ? PF_STAGE_CHUNK : n_points;
    for (int64_t at = 0; at < n_points; at += step) {
        const int64_t n = std::min(step, n_points - at);
        int64_t nb;
        if (staged) {
            // one block per CU; its points in as few equal rounds as the registers allow
            const int cap = LS_POINTS;
            st = prop_blocks(n, LS_THREADS, 1, &nb);
            if (st) return st;
            const int64_t per = (n + nb * LS_THREADS - 1) / (nb * LS_THREADS), rounds = (per + cap - 1) / cap;
            const int ppt = (int)((per + rounds - 1) / rounds);
            const size_t lds = (size_t)ppt * 3 * LS_THREADS * 4;
#define LAUNCH_PL(T, CC)                                                                                         \
    {                                                                                                            \
        N3DS_HIP_CHECK(hipFuncSetAttribute((const void*)prop_level_kernel<T, CC>,                                \
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LS_POINTS * 3 * LS_THREADS * 4)); \
        hipLaunchKernelGGL((prop_level_kernel<T, CC>), dim3((unsigned)nb), dim3(LS_THREADS), lds, s, P, at, n,   \
                           stage, ppt);                                                                          \
    }
            if (dtype == 0) LAUNCH_PL(float, 1)
            else if (level_dim == 1) LAUNCH_PL(__half, 1)
            else LAUNCH_PL(__half, 2)
#undef LAUNCH_PL
            N3DS_LAUNCH_CHECK();
        }
        st = prop_blocks(n, PF_FWD_THREADS, 8, &nb);
        if (st) return st;
#define LAUNCH_PF(CC, FM, FX)                                                                                    \
    if (CC <= 2 && staged)                                                                                       \
        hipLaunchKernelGGL((prop_fwd_kernel<float, CC <= 2 ? CC : 1, FM, FX, true>), dim3((unsigned)nb),         \
                           dim3(PF_FWD_THREADS), 0, s, P, stage, at, n, density_out, coord_out, features_out,    \
                           grid_inputs_out);                                                                     \
    else if (dtype == 0)                                                                                         \
        hipLaunchKernelGGL((prop_fwd_kernel<float, CC, FM, FX>), dim3((unsigned)nb), dim3(PF_FWD_THREADS), 0, s, \
                           P, stage, at, n, density_out, coord_out, features_out, grid_inputs_out);              \
    else                                                                                                         \
        hipLaunchKernelGGL((prop_fwd_kernel<__half, CC, FM, FX>), dim3((unsigned)nb), dim3(PF_FWD_THREADS), 0,   \
                           s, P, stage, at, n, density_out, coord_out, features_out, grid_inputs_out);
        const bool small = num_levels * level_dim <= 16;
        if (level_dim == 1 && num_levels == 10) {
            LAUNCH_PF(1, 10, 10)
        } else if (level_dim == 2 && num_levels == 10) {
            LAUNCH_PF(2, 20, 20)
        } else if (level_dim == 1) {
            if (small) { LAUNCH_PF(1, 16, 0) } else { LAUNCH_PF(1, 32, 0) }
        } else if (level_dim == 2) {
            if (small) { LAUNCH_PF(2, 16, 0) } else { LAUNCH_PF(2, 32, 0) }
        } else {
            if (small) { LAUNCH_PF(4, 16, 0) } else { LAUNCH_PF(4, 32, 0) }
        }
#undef LAUNCH_PF
        N3DS_LAUNCH_CHECK();
    }
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_prop_field_forward(const float* coords, int64_t n_points, int warp, float box_size,
                                        const void* embeddings, const int32_t* offsets, int num_levels,
                                        int level_dim, float S, int H, int gridtype, int align_corners, int interp,
                                        int dtype, const float* w1, const float* b1, const float* w2,
                                        const float* b2, float density_bias, float* density_out,
                                        float* coord_out, float* features_out, float* grid_inputs_out,
                                        void* stream) {
    return n3ds_prop_field_forward_ws(coords, n_points, warp, box_size, embeddings, offsets, num_levels, level_dim, S,
                                      H, gridtype, align_corners, interp, dtype, w1, b1, w2, b2, density_bias,
                                      density_out, coord_out, features_out, grid_inputs_out, 0, nullptr, 0, stream);
}

static int prop_field_backward(double* gsum, const float* coords, int64_t n_points, int warp, float box_size,
                                         const void* embeddings, const int32_t* offsets, int num_levels,
                                         int level_dim, float S, int H, int gridtype, int align_corners, int interp,
                                         int dtype, const float* w1, const float* b1, const float* w2,
                                         const float* b2, float density_bias, const float* grad_density,
                                         const float* features, float* grad_features, float* grid_inputs,
                                         float* grad_w1, float* grad_b1, float* grad_w2, float* grad_b2,
                                         void* stream) {
    int st = prop_check(n_points, level_dim, num_levels, dtype, warp);
    if (st) return st;
    if (n_points == 0) return N3DS_OK;
    const PropArgs P = prop_args(coords, n_points, warp, box_size, embeddings, offsets, num_levels, S, H, gridtype,
                                 align_corners, interp, w1, b1, w2, b2, density_bias);
    int64_t nb;
    hipStream_t s = (hipStream_t)stream;
#define LAUNCH_PB(CC, FM, FX)                                                                                    \
    st = prop_blocks(n_points, pf_bwd_threads(FM), pf_bwd_blocks(FM), &nb);                                      \
    if (st) return st;                                                                                          \
    if (dtype == 0)                                                                                              \
        hipLaunchKernelGGL((prop_bwd_kernel<float, CC, FM, FX>), dim3((unsigned)nb), dim3(pf_bwd_threads(FM)), 0, s, \
                           P, grad_density, features, grad_features, grid_inputs, grad_w1, grad_b1, grad_w2,     \
                           grad_b2, gsum);                                                                             \
    else                                                                                                         \
        hipLaunchKernelGGL((prop_bwd_kernel<__half, CC, FM, FX>), dim3((unsigned)nb), dim3(pf_bwd_threads(FM)), 0,   \
                           s, P, grad_density, features, grad_features, grid_inputs, grad_w1, grad_b1, grad_w2,  \
                           grad_b2, gsum);
    const bool small = num_levels * level_dim <= 16;
    if (level_dim == 1 && num_levels == 10) {
        LAUNCH_PB(1, 12, 10)
    } else if (level_dim == 2 && num_levels == 10) {
        LAUNCH_PB(2, 20, 20)
    } else if (level_dim == 1) {
        if (small) { LAUNCH_PB(1, 16, 0) } else { LAUNCH_PB(1, 32, 0) }
    } else if (level_dim == 2) {
        if (small) { LAUNCH_PB(2, 16, 0) } else { LAUNCH_PB(2, 32, 0) }
    } else {
        if (small) { LAUNCH_PB(4, 16, 0) } else { LAUNCH_PB(4, 32, 0) }
    }
#undef LAUNCH_PB
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_prop_field_backward(const float* coords, int64_t n_points, int warp, float box_size,
                                         const void* embeddings, const int32_t* offsets, int num_levels,
                                         int level_dim, float S, int H, int gridtype, int align_corners, int interp,
                                         int dtype, const float* w1, const float* b1, const float* w2,
                                         const float* b2, float density_bias, const float* grad_density,
                                         const float* features, float* grad_features, float* grid_inputs,
                                         float* grad_w1, float* grad_b1, float* grad_w2, float* grad_b2,
                                         void* stream) {
    return prop_field_backward(nullptr, coords, n_points, warp, box_size, embeddings, offsets, num_levels,
                               level_dim, S, H, gridtype, align_corners, interp, dtype, w1, b1, w2, b2,
                               density_bias, grad_density, features, grad_features, grid_inputs, grad_w1,
                               grad_b1, grad_w2, grad_b2, stream);
}

// n3ds_prop_field_backward with the weight gradients added into grad_sums [64 F | 64 | 64 | 1] doubles
N3DS_EXPORT int n3ds_prop_field_backward_sums(const float* coords, int64_t n_points, int warp, float box_size,
                                              const void* embeddings, const int32_t* offsets, int num_levels,
                                              int level_dim, float S, int H, int gridtype, int align_corners, int interp,
                                              int dtype, const float* w1, const float* b1, const float* w2,
                                              const float* b2, float density_bias, const float* grad_density,
                                              const float* features, float* grad_features, float* grid_inputs,
                                              double* grad_sums, void* stream) {
    return prop_field_backward(grad_sums, coords, n_points, warp, box_size, embeddings, offsets, num_levels,
                               level_dim, S, H, gridtype, align_corners, interp, dtype, w1, b1, w2, b2,
                               density_bias, grad_density, features, grad_features, grid_inputs, nullptr,
                               nullptr, nullptr, nullptr, stream);
}
