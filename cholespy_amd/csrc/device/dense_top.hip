// The dense top of a solve: z_T = S^{-1} r_T with the explicit inverse of the
// Schur complement of the top rows, between the forward and the backward
// pass; or, for a small system, the whole solve x = A^{-1} b in one launch.
//
// Why: near the root of the elimination tree few blocks are left and each of
// their levels costs three hand-offs between workgroups in the forward pass
// and two in the backward one (7 us a level and pass, whatever its size),
// while the inverse of the rows above a cut streams at memory bandwidth. A
// small system is one product. Measured, block passes alone and with this
// (k = 3): icosphere(3), n = 642, FP32 52.9 -> 6.5 us; a 61 x 47 grid, FP64
// 60.4 -> 13.4 us (its 66 MB inverse at 5 TB/s); icosphere(5), FP32, a top of
// 2,640 rows 91.9 -> 45.6 us; icosphere(6), k = 128, FP32, a top of 3,488 rows
// 371 -> 259 us. choose_dense_top (block_plan.cpp) weighs the two.
//
// Rounding: an inverse rounded to FP32 keeps the block passes' accuracy only
// if its long dot products do not round in FP32 as well (one running FP32 sum
// lost a factor of 3 to 4): products are summed a few at a time, and those
// sums in FP64. FP32 solves are then 1.1 to 3 times closer to the exact
// solution than the block passes' were, FP64 ones within 15 % of them.
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
__device__ __forceinline__ Top top_of(const DenseTopArgs &a, int panels_per_group) {
    const int count = gridDim.x, per = count / 8, extra = count % 8, x = blockIdx.x % 8;
    const int g = x * per + min(x, extra) + blockIdx.x / 8;
    Top r;
    if (!a.tiles) {   // one system: no record to load
        r.row0 = a.row0;
        r.n = a.n;
        r.panel = g * panels_per_group;
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
    const Top top = top_of(a, 1);
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

// More right-hand sides: a workgroup takes two panels and NT tiles of 16
// right-hand sides, its 8 wavefronts split the inputs and add their partial
// tiles through LDS. A streams from the panels, B from the input rows (each
// loaded once for both panels). Two wavefronts per SIMD cover the loads of
// one group of inputs with the MFMAs of the other.
constexpr int kWideThreads = 512;
constexpr int kWideWaves = kWideThreads / kWave;
template <typename F, int NT>
__global__ __launch_bounds__(kWideThreads) void dense_wide(DenseTopArgs a) {
    using P = Pack<F>;
    using Vec = typename P::Vec;
    using Acc = typename P::Acc;
    constexpr int V = P::V, G = 4 * V, kPanels = 2, kTiles = kPanels * NT, kHalf = kWideWaves / 2;
    __shared__ double red[kHalf][kTiles][kWave * 4];
    const Top top = top_of(a, kPanels);
    const int k = top.k, t0 = blockIdx.y * NT * 16;
    if (t0 >= k) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, q = lane / 16, l = lane % 16;
    const bool two = (top.panel + 1) * 16 < top.npad;
    const Vec *M0 = reinterpret_cast<const Vec *>(static_cast<const F *>(a.M) + top.off) + lane;
    const Vec *M1 = two ? M0 + (size_t)top.npad * 16 / V : M0;
    const F *src = static_cast<const F *>(a.in) + top.vbase + (long long)top.row0 * k + t0 + l;
    double sum[kPanels][NT][4] = {};
    const int ng = top.npad / G;
    Vec m0 = {}, m1 = {};
    F b[V][NT];
    auto load = [&](int g) {
        if (g < ng) {
            m0 = M0[(size_t)g * kWave];
            m1 = M1[(size_t)g * kWave];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int r = g * G + 4 * j + q;
#pragma unroll
            for (int n = 0; n < NT; ++n)
                b[j][n] = r < top.n && t0 + 16 * n + l < k ? src[(long long)r * k + 16 * n] : F(0);
        }
    };
    load(wave);
    for (int g = wave; g < ng; g += kWideWaves) {
        const Vec a0 = m0, a1 = m1;
        F bb[V][NT];
#pragma unroll
        for (int j = 0; j < V; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n) bb[j][n] = b[j][n];
        load(g + kWideWaves);
        // Two steps (8 products an entry) at a time, summed in FP64.
#pragma unroll
        for (int j = 0; j < V; j += 2)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int p = 0; p < kPanels; ++p) {
                    const Vec ap = p == 0 ? a0 : a1;
                    const Acc acc = P::step(ap[j + 1], bb[j + 1][n], P::step(ap[j], bb[j][n], Acc{}));
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[p][n][v] += (double)acc[v];
                }
    }
    // The upper half of the wavefronts hands its sums to the lower half, which
    // then shares out the tiles.
    for (int half = 1; half >= 0; --half) {
        if (wave / kHalf == half)
#pragma unroll
            for (int i = 0; i < kTiles; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[wave % kHalf][i][v * kWave + lane] = sum[i / NT][i % NT][v];
        __syncthreads();
        if (half == 1) {
            if (wave < kHalf)
#pragma unroll
                for (int i = 0; i < kTiles; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[i / NT][i % NT][v] += red[wave][i][v * kWave + lane];
            __syncthreads();
        }
    }
    for (int i = wave; i < kTiles; i += kWideWaves) {
        const int p = i / NT, col = t0 + 16 * (i % NT) + l;
        if (p == 1 && !two) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int e = v * kWave + lane, c = (top.panel + p) * 16 + P::row(q, v);
            const F s = (F)(red[0][i][e] + red[1][i][e] + red[2][i][e] + red[3][i][e]);
            if (c < top.n && col < k) put(a, top, c, col, a.perm ? a.perm[top.row0 + c] : top.row0 + c, s);
        }
    }
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

hipError_t launch_dense_top(int float_bytes, const DenseTopArgs &args, int narrow_tiles, const DenseTopTile *wide_list,
                            int wide_tiles, int max_k, hipStream_t stream) {
    DenseTopArgs a = args;
    void *p[] = {&a};
    if (max_k <= kNarrowTile) {
        const void *kern = float_bytes == 4 ? reinterpret_cast<const void *>(&dense_narrow<float, kNarrowTile>)
                                            : reinterpret_cast<const void *>(&dense_narrow<double, kNarrowTile>);
        return hipLaunchKernel(kern, dim3(narrow_tiles), dim3(kNarrowThreads), p, 0, stream);
    }
    if (a.tiles) a.tiles = wide_list;
    const int nt = max_k <= 16 ? 1 : (max_k <= 32 ? 2 : 4);
    const void *kern;
#define CHOLESPY_DENSE(F)                                                                \
    (nt == 1 ? reinterpret_cast<const void *>(&dense_wide<F, 1>)                         \
             : nt == 2 ? reinterpret_cast<const void *>(&dense_wide<F, 2>)               \
                       : reinterpret_cast<const void *>(&dense_wide<F, 4>))
    kern = float_bytes == 4 ? CHOLESPY_DENSE(float) : CHOLESPY_DENSE(double);
#undef CHOLESPY_DENSE
    return hipLaunchKernel(kern, dim3(wide_tiles, (max_k + 16 * nt - 1) / (16 * nt)), dim3(kWideThreads), p, 0, stream);
}

}  // namespace cholespy_amd
