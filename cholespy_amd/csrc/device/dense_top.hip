// The dense top of a solve: z_T = S^{-1} r_T with the explicit inverse of the
// Schur complement of the top rows, between the forward and the backward
// pass; or, for a small system, the whole solve x = A^{-1} b in one launch.
//
// Why: near the root of the elimination tree few blocks are left and each of
// their levels costs three hand-offs between workgroups in the forward pass
// and two in the backward one (7 us a level and pass, whatever its size),
// while the inverse of the rows above a cut streams at memory bandwidth. A
// small system is one product. Measured, block passes alone and with this:
// k = 3, icosphere(3), n = 642, FP32 41.9 -> 6.9 us; icosphere(5), FP32, a top
// of 2,640 rows 66 -> 39 us; a vector, 61 x 47 grid, FP64 50.7 -> 13.4 us (its
// 66 MB inverse at 5 TB/s); k = 128, icosphere(6), FP32, 3,488 rows 342 -> 225
// us; k = 32, 48^3 grid, FP32, 6,256 rows 460 -> 382 us; k = 3, icosphere(7),
// FP64, 2,896 rows 163 -> 160 us.
// choose_dense_top (block_plan.cpp) weighs the two.
//
// Rounding: an inverse rounded to FP32 keeps the block passes' accuracy only
// if its long dot products do not round in FP32 as well (one running FP32 sum
// lost a factor of 3 to 4): products are summed a few at a time, and those
// sums in FP64. FP32 solves are then 1.1 to 3 times closer to the exact
// solution than the block passes' were, FP64 ones within 20 % of them.
//
// Layout: S^{-1} (symmetric) in panels of 16 output rows, each contiguous:
// the entry of output c and input rho is element
//   (rho / G) * 64 V + ((rho % 4) * 16 + c % 16) * V + (rho % G) / 4
// of panel c / 16, V = 16 bytes / element size, G = 4 V, inputs padded with
// zeros to a multiple of 16. One 16-byte load per lane is then the A operand
// of V successive 16x16x4 MFMA steps, and a panel is one contiguous stream
// whatever n is.
#include <algorithm>

#include "block_plan.hpp"
#include "common.hpp"
#include "launchers.hpp"

namespace cholespy_amd {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename F> struct Pack;
template <> struct Pack<float> {
    using Vec = f32x4;
    using Acc = f32x4;
    static constexpr int V = 4;
    static __device__ __forceinline__ Acc step(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }
};
template <> struct Pack<double> {
    using Vec = f64x2;
    using Acc = f64x4;
    static constexpr int V = 2;
    static __device__ __forceinline__ Acc step(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return q + 4 * v; }
};

// The panel a workgroup starts at, and its system's top.
struct Top {
    int row0, n, npad, panel, k;
    long long vbase;
    int64_t off;
};
// Consecutive workgroups go to different XCDs (round robin over 8): give each
// XCD a run of consecutive panels, so that what neighbours share stays in one L2.
__device__ __forceinline__ Top top_of(const DenseTopArgs &a) {
    const int count = gridDim.x, per = count / 8, extra = count % 8, x = blockIdx.x % 8;
    const int g = x * per + min(x, extra) + blockIdx.x / 8;
    Top r;
    if (!a.tiles) {   // one system: no record to load
        r.row0 = a.row0;
        r.n = a.n;
        r.panel = g;
        r.k = a.k;
        r.vbase = 0;
        r.off = 0;
    } else {
        const DenseTopTile t = a.tiles[g];
        r.row0 = t.row0;
        r.n = t.n;
        r.panel = t.panel;
        r.k = a.sys_k[t.sys];
        r.vbase = a.sys_vbase[t.sys];
        r.off = t.off;
    }
    r.npad = (r.n + 15) / 16 * 16;
    r.off += (int64_t)r.panel * r.npad * 16;
    return r;
}

// Output row c, column col: z (read by the backward pass) and row xrow of the solution.
template <typename F>
__device__ __forceinline__ void put(const DenseTopArgs &a, const Top &top, int c, int col, int xrow, F v) {
    if (a.z) static_cast<F *>(a.z)[top.vbase + (long long)(top.row0 + c) * top.k + col] = v;
    const long long o = top.vbase + (long long)xrow * top.k + col;
    if (a.xmode == 0) {
        static_cast<F *>(a.x)[o] = v;
    } else {
        double *x64 = static_cast<double *>(a.x);
        x64[o] = (a.xmode == 2 ? x64[o] : 0.0) + (double)v;
    }
}

// Bounds-checked loads: a buffer of `bytes` bytes at p (uniform over the
// wavefront), whose loads past the end return zero without touching memory.
// Loads under a condition instead split the unrolled loops into blocks, and
// the compiler then spilled the inputs it had read ahead (165 registers).
struct Buffer {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ Buffer(const void *p, unsigned bytes)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000)) {}
    template <typename T>
    __device__ __forceinline__ T at(unsigned offset) const {
        if constexpr (sizeof(T) == 4)
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc, offset, 0, 0));
        else if constexpr (sizeof(T) == 8)
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, 0, 0));
        else
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0));
    }
};

// Up to KT right-hand sides: one workgroup per panel, its 16 wavefronts take
// the panel's groups of G inputs in turn. A chunk is kFly groups of every
// wavefront: all its loads are in flight at once, and each register is loaded
// for the next chunk as soon as it is used, while the next chunk's inputs go
// to the other LDS buffer. Bound by streaming the panel; the launch's fixed
// cost is about 4.5 us.
constexpr int kNarrowThreads = 1024;
constexpr int kNarrowWaves = kNarrowThreads / kWave;
constexpr int kFly = 6;
template <typename F, int KT>
__global__ __launch_bounds__(kNarrowThreads) __attribute__((amdgpu_waves_per_eu(8))) void dense_narrow(DenseTopArgs a) {
    using P = Pack<F>;
    using Vec = typename P::Vec;
    constexpr int V = P::V, G = 4 * V;
    constexpr int kGroups = kFly * kNarrowWaves, kChunk = kGroups * G;
    constexpr int kIn = kChunk * KT / kNarrowThreads;   // inputs a thread stages per chunk
    __shared__ __align__(16) F in[2][kChunk * KT];
    __shared__ double red[kNarrowWaves * 16 * KT];
    const Top top = top_of(a);
    const int k = top.k;
    if (k <= 0) return;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int ng = top.npad / G;
    constexpr unsigned kVec = sizeof(Vec);
    const Buffer M(static_cast<const F *>(a.M) + top.off, (unsigned)top.npad * 16 * sizeof(F));
    const Buffer src(static_cast<const F *>(a.in) + top.vbase + (long long)top.row0 * k,
                     (unsigned)top.n * (unsigned)k * (unsigned)sizeof(F));
    const unsigned m0 = (unsigned)tid * kVec;   // this lane's vector of group `wave`
    Vec mv[kFly];
#pragma unroll
    for (int u = 0; u < kFly; ++u) mv[u] = M.at<Vec>(m0 + u * kNarrowWaves * kWave * kVec);
    F st[kIn];
    auto load_in = [&](int c0) {
#pragma unroll
        for (int q = 0; q < kIn; ++q) {
            const int i = tid + q * kNarrowThreads, r = c0 + i / KT, t = i % KT;
            st[q] = src.at<F>(t < k ? (unsigned)(r * k + t) * (unsigned)sizeof(F) : ~0u);
        }
    };
    load_in(0);
    // The solution row of this thread's output, needed last.
    const int oc = top.panel * 16 + tid / KT, ot = tid % KT;
    const bool out = tid < 16 * KT && oc < top.n && ot < k;
    const int xrow = out && a.perm ? a.perm[top.row0 + oc] : top.row0 + oc;
    double acc[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = 0.0;
    for (int g0 = 0, buf = 0; g0 < ng; g0 += kGroups, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < kIn; ++q) in[buf][tid + q * kNarrowThreads] = st[q];
        __syncthreads();
        if (g0 + kGroups < ng) load_in((g0 + kGroups) * G);
#pragma unroll
        for (int u = 0; u < kFly; ++u) {
            const F *v = &in[buf][(size_t)((wave + u * kNarrowWaves) * G + lane / 16) * KT];
            F part[KT];   // V products, then a sum in FP64
#pragma unroll
            for (int t = 0; t < KT; ++t) part[t] = mv[u][0] * v[t];
#pragma unroll
            for (int j = 1; j < V; ++j)
#pragma unroll
                for (int t = 0; t < KT; ++t) part[t] = fma(mv[u][j], v[4 * j * KT + t], part[t]);
#pragma unroll
            for (int t = 0; t < KT; ++t) acc[t] += (double)part[t];
            mv[u] = M.at<Vec>(m0 + (unsigned)((g0 + kGroups + u * kNarrowWaves) * kWave) * kVec);
        }
    }
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        acc[t] += __shfl_xor(acc[t], 16, kWave);
        acc[t] += __shfl_xor(acc[t], 32, kWave);
    }
    if (lane < 16)
#pragma unroll
        for (int t = 0; t < KT; ++t) red[(wave * 16 + lane) * KT + t] = acc[t];
    __syncthreads();
    if (out) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kNarrowWaves; ++w) s += red[w * 16 * KT + tid];
        put(a, top, oc, ot, xrow, (F)s);
    }
}

// More right-hand sides: a workgroup takes a panel and NT tiles of 16
// right-hand sides, its 8 wavefronts split the inputs and add their partial
// tiles through LDS. A streams from the panel, B from the input rows (out of
// the L2: an XCD's workgroups read the same rows), D groups of inputs in
// flight per wavefront. Bound by the latency of those streams, not by the
// matrix cores. Two panels a workgroup with one group in flight and B loaded a
// value at a time, against this: icosphere(6), k = 128, FP32 (top 3,488) 65 ->
// 50 us, 511 x 389 grid, k = 17, FP64 (top 2,048) 39 -> 18 us, 48^3 grid,
// k = 32, FP32 (top 6,256) 62 -> 56 us, a batch of 64 systems, k = 1 to 128,
// FP32 159 -> 111 us; 33^3 grid, k = 5, FP64 (top 4,512) 63 -> 51 us. 16
// wavefronts a workgroup measured the same.
constexpr int kWideThreads = 512;
constexpr int kWideWaves = kWideThreads / kWave;
constexpr int kOneTileFly = 5;   // D of one tile
template <typename F, int NT, int D>
__device__ __forceinline__ void wide_tiles(const DenseTopArgs &a, const Top &top, int t0, double (*red)[kWave * 4]) {
    using P = Pack<F>;
    using Vec = typename P::Vec;
    using Acc = typename P::Acc;
    constexpr int V = P::V, G = 4 * V, kHalf = kWideWaves / 2;
    const int k = top.k;
    const int lane = threadIdx.x % kWave, q = lane / 16, l = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const Buffer M(static_cast<const F *>(a.M) + top.off, (unsigned)top.npad * 16 * (unsigned)sizeof(F));
    const Buffer src(static_cast<const F *>(a.in) + top.vbase + (long long)top.row0 * k,
                     (unsigned)top.n * (unsigned)k * (unsigned)sizeof(F));
    const int ng = top.npad / G;
    Vec m[D];
    // B of tile n, lane column l: right-hand side col0 + n, so that a lane's
    // tiles are one load of NT consecutive values. Lanes past the row's end
    // compute its last NT columns again and store only those from their own
    // first column on: a column stored twice, by lanes that reach it with
    // different n, would take a refinement's += twice. (NT > 1: k > 16.)
    const int col0 = NT == 1 ? t0 + l : min(t0 + NT * l, k - NT);
    const unsigned b0 = NT > 1 || col0 < k ? (unsigned)(q * k + col0) * (unsigned)sizeof(F) : 1u << 31;
    F b[D][V][NT];
    constexpr int kPer = NT * (int)sizeof(F) <= 16 ? NT : 16 / (int)sizeof(F);   // values per load
    typedef F BVec __attribute__((ext_vector_type(kPer)));
    auto load = [&](int d, int g) {
        // (Groups past the end are past the end of both buffers: zero.)
        m[d] = M.at<Vec>((unsigned)(g * kWave + lane) * (unsigned)sizeof(Vec));
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const unsigned at = b0 + (unsigned)((g * G + 4 * j) * k) * (unsigned)sizeof(F);
#pragma unroll
            for (int n = 0; n < NT; n += kPer) {
                if constexpr (kPer == 1) {
                    b[d][j][n] = src.at<F>(at);
                } else {
                    const BVec v = src.at<BVec>(at + n * (unsigned)sizeof(F));
#pragma unroll
                    for (int e = 0; e < kPer; ++e) b[d][j][n + e] = v[e];
                }
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
        load(d, wave + d * kWideWaves);
        __builtin_amdgcn_sched_barrier(0);
    }
    double sum[NT][4] = {};
    for (int g0 = wave; g0 < ng; g0 += D * kWideWaves) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            // Two steps (8 products an entry) at a time, summed in FP64.
#pragma unroll
            for (int j = 0; j < V; j += 2)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const Acc acc = P::step(m[d][j + 1], b[d][j + 1][n], P::step(m[d][j], b[d][j][n], Acc{}));
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[n][v] += (double)acc[v];
                }
            // (The scheduler would gather the D loads at the loop's end, and
            // its head would wait for all of them.)
            __builtin_amdgcn_sched_barrier(0);
            load(d, g0 + (D + d) * kWideWaves);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The upper half of the wavefronts hands its sums to the lower half, which
    // then shares out the tiles.
    for (int half = 1; half >= 0; --half) {
        if (wave / kHalf == half)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[wave % kHalf * NT + n][v * kWave + lane] = sum[n][v];
        __syncthreads();
        if (half == 1) {
            if (wave < kHalf)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[n][v] += red[wave * NT + n][v * kWave + lane];
            __syncthreads();
        }
    }
    for (int i = wave; i < 4 * NT; i += kWideWaves) {
        const int n = i / 4, v = i % 4, col = col0 + n, e = v * kWave + lane, c = top.panel * 16 + P::row(q, v);
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kHalf; ++w) s += red[w * NT + n][e];
        if (c < top.n && col < k && col >= t0 + NT * l) put(a, top, c, col, a.perm ? a.perm[top.row0 + c] : top.row0 + c, (F)s);
    }
}

template <typename F, int NT, int D>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(4))) void dense_wide(DenseTopArgs a) {
    __shared__ double red[kWideWaves / 2 * NT][kWave * 4];
    const Top top = top_of(a);
    const int t0 = blockIdx.y * NT * 16;
    if (t0 >= top.k) return;
    // A rest of one tile: a batch's systems differ in their right-hand sides.
    if (NT > 1 && top.k - t0 <= 16)
        wide_tiles<F, 1, kOneTileFly>(a, top, t0, red);
    else
        wide_tiles<F, NT, D>(a, top, t0, red);
}

__global__ void copy_words(uint32_t *dst, const uint32_t *src, size_t count) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

}  // namespace

hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t stream) {
    const size_t count = bytes / 4;
    if (count == 0) return hipSuccess;
    copy_words<<<dim3((unsigned)std::min<size_t>((count + 255) / 256, 4096)), 256, 0, stream>>>(
        static_cast<uint32_t *>(dst), static_cast<const uint32_t *>(src), count);
    return hipGetLastError();
}

hipError_t launch_dense_top(int float_bytes, const DenseTopArgs &args, int tiles, int max_k,
                            hipStream_t stream) {
    DenseTopArgs a = args;
    void *p[] = {&a};
    const void *kern;
    if (max_k <= kNarrowTile) {
        kern = float_bytes == 4 ? reinterpret_cast<const void *>(&dense_narrow<float, kNarrowTile>)
                                : reinterpret_cast<const void *>(&dense_narrow<double, kNarrowTile>);
        return hipLaunchKernel(kern, dim3(tiles), dim3(kNarrowThreads), p, 0, stream);
    }
    const int nt = max_k <= 16 ? 1 : (max_k <= 32 ? 2 : 4);
#define CHOLESPY_DENSE(F)                                                    \
    (nt == 1   ? reinterpret_cast<const void *>(&dense_wide<F, 1, kOneTileFly>) \
     : nt == 2 ? reinterpret_cast<const void *>(&dense_wide<F, 2, 3>)        \
               : reinterpret_cast<const void *>(&dense_wide<F, 4, 2>))
    kern = float_bytes == 4 ? CHOLESPY_DENSE(float) : CHOLESPY_DENSE(double);
#undef CHOLESPY_DENSE
    return hipLaunchKernel(kern, dim3(tiles, (max_k + 16 * nt - 1) / (16 * nt)), dim3(kWideThreads), p, 0, stream);
}

}  // namespace cholespy_amd
