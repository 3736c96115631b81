// The dense top of a solve: z_T = X' (X r_T) with X = L_TT^{-1}, the explicit
// inverse of L's top rows, as one product after the block tasks of the forward
// pass (y_T = X r_T) and one before those of the backward pass (z_T = X' y_T);
// or, where every row is a top row, the whole solve in these two launches.
//
// Why: near the root of the elimination tree few blocks are left and each of
// their levels costs three hand-offs between workgroups in the forward pass
// and two in the backward one (7 us a level and pass, whatever its size),
// while a product with X streams at memory bandwidth. choose_dense_top
// (block_plan.cpp) weighs the two.
//
// Why two triangular products and not one with S^{-1} = X' X: that one square
// is not backward stable, its residual grows with the condition number; the
// two triangular ones keep the residual of the block passes. ||b - A x|| /
// ||b||, k = 3, block passes / S^{-1} / X'(X r): 61 x 47 grid, shift 1e-4,
// FP64 2.9e-16 / 3.6e-15 / 3.4e-16, FP32 1.4e-7 / 7.8e-7 / 9.7e-8; 16^3 grid,
// kappa 1e6, FP64 3.4e-16 / 1.5e-12 / 1.0e-15. X is sparse where S^{-1} is
// full (dense_top_plan.hpp), so that the two read less, and are formed in less
// time: refactorize + solve of a 100 x 60 grid, FP32, 2.37 ms with the values
// formed on the host and no top, 7.1 with S^{-1}, 1.9 with X; 61 x 47 1.13 /
// 2.36 / 0.92 ms. The price is a launch: icosphere(3), k = 3, FP32 53 us by
// the block passes, 6.4 with S^{-1}, 10.4; icosphere(5) 65 / 40 / 43; but
// icosphere(6), k = 128, FP32 342 / 225 / 189.
//
// Rounding: products are summed a few at a time, and those sums in FP64 (one
// running FP32 sum lost a factor of 3 to 4).
//
// Layout, per direction: panels of 16 output rows, each contiguous; in a
// panel, per 16 inputs (a unit), the entry of output c and input rho is element
//   (rho / G) * 64 V + ((rho % 4) * 16 + c % 16) * V + (rho % G) / 4,
// V = 16 bytes / element size, G = 4 V, zeros outside X. One 16-byte load per
// lane is then the A operand of V successive 16x16x4 MFMA steps, and a panel
// is one contiguous stream whatever its inputs are.
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

// The panel of a workgroup and its system's vectors.
struct Top {
    int row0, n, panel, first, count, seg, nseg, slot, k;
    long long vbase;
    int64_t off;
};
__device__ __forceinline__ Top top_of(const DenseTopArgs &a) {
    const DenseTopPanel t = a.panels[blockIdx.x];
    Top r{t.row0, t.n, t.panel, t.first, t.count, t.seg, t.nseg, t.slot, a.k, 0, t.off};
    if (a.sys_k) {
        r.k = a.sys_k[t.sys];
        r.vbase = a.sys_vbase[t.sys];
    }
    return r;
}

// Output row c, column col: the work vector (y or z) and row xrow of the solution.
template <typename F>
__device__ __forceinline__ void put(const DenseTopArgs &a, const Top &top, int c, int col, int xrow, F v) {
    if (a.out) static_cast<F *>(a.out)[top.vbase + (long long)(top.row0 + c) * top.k + col] = v;
    if (!a.x) return;
    const long long o = top.vbase + (long long)xrow * top.k + col;
    if (a.xmode == 0) {
        static_cast<F *>(a.x)[o] = v;
    } else {
        double *x64 = static_cast<double *>(a.x);
        x64[o] = (a.xmode == 2 ? x64[o] : 0.0) + (double)v;
    }
}

// Segment sums (panels of more than kTopSegment units): a segment publishes
// its sums (put_sum), and the one that arrives last, whichever that is, finds
// all of them complete and adds them in segment order (sum_of). Nobody waits
// for another workgroup. The stores and loads are agent-scope ones, each
// store complete before its workgroup's arrival is counted.
__device__ __forceinline__ double *sum_at(const DenseTopArgs &a, const Top &top, int seg, int row, int col) {
    return a.sums + ((size_t)(top.slot + seg) * kTopUnit + row) * kMaxRhs + col;
}
__device__ __forceinline__ void put_sum(const DenseTopArgs &a, const Top &top, int row, int col, double s) {
    publish(sum_at(a, top, top.seg, row, col), s);
}
__device__ __forceinline__ bool arrives_last(const DenseTopArgs &a, const Top &top, int tile, int *last) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned *n = a.arrived + (size_t)top.slot * kTopArrivals + tile;
        *last = __hip_atomic_fetch_add(n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)top.nseg - 1;
        if (*last) __hip_atomic_store(n, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return *last != 0;
}
__device__ __forceinline__ double sum_of(const DenseTopArgs &a, const Top &top, int row, int col) {
    double s = 0.0;
    for (int seg = 0; seg < top.nseg; ++seg) s += from_bits<double>(load_bits(sum_at(a, top, seg, row, col)));
    return s;
}

// Where a product's inputs are: rows of the top in order from unit `first` on
// (kRange), the units listed (kList), or, for a whole system's first product,
// rows of b in the caller's order (kPerm).
constexpr int kRange = 0, kList = 1, kPerm = 2;

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
// the panel's (or the segment's) groups of G inputs in turn. A chunk is kFly groups of every
// wavefront: all its loads are in flight at once, and each register is loaded
// for the next chunk as soon as it is used, while the next chunk's inputs go
// to the other LDS buffer. Bound by streaming the panel and, for the many
// short panels, by the launch and a chain of four memory latencies.
constexpr int kNarrowThreads = 1024;
constexpr int kNarrowWaves = kNarrowThreads / kWave;
constexpr int kFly = 6;
template <typename F, int KT, int kIn>
__global__ __launch_bounds__(kNarrowThreads) __attribute__((amdgpu_waves_per_eu(8))) void dense_narrow(DenseTopArgs a) {
    using P = Pack<F>;
    using Vec = typename P::Vec;
    constexpr int V = P::V, G = 4 * V;
    constexpr int kGroups = kFly * kNarrowWaves, kChunk = kGroups * G;
    constexpr int kStage = kChunk * KT / kNarrowThreads;   // inputs a thread stages per chunk
    static_assert(kTopUnit * KT == kWave, "a wavefront stages one unit at a time");
    __shared__ __align__(16) F in[2][kChunk * KT];
    __shared__ double red[kNarrowWaves * 16 * KT];
    __shared__ int last;
    const Top top = top_of(a);
    const int k = top.k;
    if (k <= 0) return;
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int ng = top.count * kTopUnit / G;
    constexpr unsigned kVec = sizeof(Vec);
    const Buffer M(static_cast<const F *>(a.M) + top.off, (unsigned)top.count * kTopUnitEntries * (unsigned)sizeof(F));
    // Rows of the range that exist, and the inputs up to their end.
    const int in0 = kIn == kList ? 0 : top.first * kTopUnit;
    const int end = kIn == kList ? top.n : min(top.n, in0 + top.count * kTopUnit);
    const Buffer src(static_cast<const F *>(a.in) + (kIn == kPerm ? 0 : top.vbase + (long long)top.row0 * k),
                     (unsigned)(kIn == kPerm ? a.b_rows : end) * (unsigned)k * (unsigned)sizeof(F));
    const Buffer rows(kIn == kPerm ? a.rows + top.row0 : nullptr, kIn == kPerm ? (unsigned)end * 4u : 0u);
    const unsigned m0 = (unsigned)tid * kVec;   // this lane's vector of group `wave`
    Vec mv[kFly];
#pragma unroll
    for (int u = 0; u < kFly; ++u) mv[u] = M.at<Vec>(m0 + u * kNarrowWaves * kWave * kVec);
    F st[kStage];
    const int si = lane / KT, stt = lane % KT;   // row and right-hand side in a unit
    const unsigned s0 = stt < k ? (unsigned)(si * k + stt) * (unsigned)sizeof(F) : 1u << 31;
    auto load_in = [&](int c0) {
#pragma unroll
        for (int q = 0; q < kStage; ++q) {
            const int unit = c0 / kTopUnit + wave + q * kNarrowWaves;
            if (kIn == kPerm) {
                const int r = in0 + unit * kTopUnit + si;
                const int row = rows.at<int>((unsigned)r * 4u);
                st[q] = src.at<F>(stt < k && r < end ? (unsigned)(row * k + stt) * (unsigned)sizeof(F) : 1u << 31);
            } else {
                // (Units past the end: rows past the end of src.)
                int r = in0 + unit * kTopUnit;
                if (kIn == kList) r = unit < top.count ? a.units[top.first + unit] * kTopUnit : end;
                st[q] = src.at<F>(s0 + (unsigned)(r * k) * (unsigned)sizeof(F));
            }
        }
    };
    load_in(0);
    // The solution row of this thread's output, needed last.
    const int oc = top.panel * 16 + tid / KT, ot = tid % KT;
    const bool out = tid < 16 * KT && oc < top.n && ot < k;
    const int xrow = out && a.x ? a.perm[top.row0 + oc] : 0;
    double acc[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = 0.0;
    for (int g0 = 0, buf = 0; g0 < ng; g0 += kGroups, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < kStage; ++q) in[buf][tid + q * kNarrowThreads] = st[q];
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
    double s = 0.0;
    if (out)
#pragma unroll
        for (int w = 0; w < kNarrowWaves; ++w) s += red[w * 16 * KT + tid];
    if (top.nseg > 1) {
        if (out) put_sum(a, top, tid / KT, ot, s);
        if (!arrives_last(a, top, 0, &last)) return;
        if (out) s = sum_of(a, top, tid / KT, ot);
    }
    if (out) put(a, top, oc, ot, xrow, (F)s);
}

// More right-hand sides: a workgroup takes a panel and NT tiles of 16
// right-hand sides, its 8 wavefronts split the inputs and add their partial
// tiles through LDS. A streams from the panel, B from the input rows (out of
// the L2), D groups of inputs in flight per wavefront. Bound by the latency of
// those streams, not by the matrix cores.
constexpr int kWideThreads = 512;
constexpr int kWideWaves = kWideThreads / kWave;
constexpr int kOneTileFly = 5;   // D of one tile
// (A wavefront's groups, with those asked for ahead, fit two registers a lane.)
static_assert(kTopMaxRows / (Pack<double>::V * 4 * kWideWaves) + 2 * kOneTileFly - 2 < 2 * kWave, "kTopMaxRows");
template <typename F, int NT, int D, int kIn>
__device__ __forceinline__ void wide_tiles(const DenseTopArgs &a, const Top &top, int t0, double (*red)[kWave * 4], int *last) {
    using P = Pack<F>;
    using Vec = typename P::Vec;
    using Acc = typename P::Acc;
    constexpr int V = P::V, G = 4 * V, kHalf = kWideWaves / 2;
    const int k = top.k;
    const int lane = threadIdx.x % kWave, q = lane / 16, l = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const Buffer M(static_cast<const F *>(a.M) + top.off, (unsigned)top.count * kTopUnitEntries * (unsigned)sizeof(F));
    const int in0 = kIn == kList ? 0 : top.first * kTopUnit;
    const int end = kIn == kList ? top.n : min(top.n, in0 + top.count * kTopUnit);
    const Buffer src(static_cast<const F *>(a.in) + top.vbase + (long long)top.row0 * k,
                     (unsigned)end * (unsigned)k * (unsigned)sizeof(F));
    const int ng = top.count * kTopUnit / G;
    // First input row of this wavefront's i-th group (wave + 8 i): from the
    // unit list held one entry a lane, or counted on. Past the last group: past
    // the end of src.
    int li[2];
    if (kIn == kList)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = (wave + (lane + h * kWave) * kWideWaves) * G, unit = r / kTopUnit;
            li[h] = unit < top.count ? a.units[top.first + unit] * kTopUnit + r % kTopUnit : top.n;
        }
    auto first_row = [&](int i) {
        if (kIn == kRange) return in0 + (wave + i * kWideWaves) * G;
        const int r0 = __builtin_amdgcn_readlane(li[0], i % kWave), r1 = __builtin_amdgcn_readlane(li[1], i % kWave);
        return i < kWave ? r0 : r1;
    };
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
    auto load = [&](int d, int i) {
        // (Groups past the end are past the end of both buffers: zero.)
        m[d] = M.at<Vec>((unsigned)((wave + i * kWideWaves) * kWave + lane) * (unsigned)sizeof(Vec));
        const int row = first_row(i);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const unsigned at = b0 + (unsigned)((row + 4 * j) * k) * (unsigned)sizeof(F);
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
        load(d, d);
        __builtin_amdgcn_sched_barrier(0);
    }
    double sum[NT][4] = {};
    for (int i = 0; wave + i * kWideWaves < ng; i += D) {
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
            load(d, i + D + d);
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
        if (c >= top.n || col >= k || col < t0 + NT * l) continue;
        if (top.nseg > 1) put_sum(a, top, c - top.panel * 16, col, s);
        else put(a, top, c, col, a.x ? a.perm[top.row0 + c] : 0, (F)s);
    }
    if (top.nseg == 1 || !arrives_last(a, top, t0 / 16, last)) return;
    const int width = min(16 * NT, k - t0);
    for (int e = threadIdx.x; e < kTopUnit * width; e += kWideThreads) {
        const int row = e / width, col = t0 + e % width, c = top.panel * 16 + row;
        if (c < top.n) put(a, top, c, col, a.x ? a.perm[top.row0 + c] : 0, (F)sum_of(a, top, row, col));
    }
}

template <typename F, int NT, int D, int kIn>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(4))) void dense_wide(DenseTopArgs a) {
    __shared__ double red[kWideWaves / 2 * NT][kWave * 4];
    __shared__ int last;
    const Top top = top_of(a);
    const int t0 = blockIdx.y * NT * 16;
    if (t0 >= top.k) return;
    // A rest of one tile: a batch's systems differ in their right-hand sides.
    if (NT > 1 && top.k - t0 <= 16)
        wide_tiles<F, 1, kOneTileFly, kIn>(a, top, t0, red, &last);
    else
        wide_tiles<F, NT, D, kIn>(a, top, t0, red, &last);
}

// dst row i = src row rows[i], k columns.
template <typename F>
__global__ void gather_rows_of(F *dst, const F *src, const int *rows, int n, int k) {
    const size_t total = (size_t)n * k;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x)
        dst[e] = src[(size_t)rows[e / k] * k + e % k];
}

}  // namespace

hipError_t launch_gather_rows(int float_bytes, void *dst, const void *src, const int *rows, int n, int k, hipStream_t stream) {
    const size_t total = (size_t)n * k;
    if (total == 0) return hipSuccess;
    const dim3 grid((unsigned)std::min<size_t>((total + 255) / 256, 4096));
    if (float_bytes == 4)
        gather_rows_of<float><<<grid, 256, 0, stream>>>(static_cast<float *>(dst), static_cast<const float *>(src), rows, n, k);
    else
        gather_rows_of<double><<<grid, 256, 0, stream>>>(static_cast<double *>(dst), static_cast<const double *>(src), rows, n, k);
    return hipGetLastError();
}

template <typename F>
static const void *dense_kernel(const DenseTopArgs &a, int max_k) {
    if (max_k <= kNarrowTile)
        return a.units  ? reinterpret_cast<const void *>(&dense_narrow<F, kNarrowTile, kList>)
               : a.rows ? reinterpret_cast<const void *>(&dense_narrow<F, kNarrowTile, kPerm>)
                        : reinterpret_cast<const void *>(&dense_narrow<F, kNarrowTile, kRange>);
#define CHOLESPY_DENSE(NT, D)                                                 \
    (a.units ? reinterpret_cast<const void *>(&dense_wide<F, NT, D, kList>)   \
             : reinterpret_cast<const void *>(&dense_wide<F, NT, D, kRange>))
    return max_k <= 16 ? CHOLESPY_DENSE(1, kOneTileFly) : max_k <= 32 ? CHOLESPY_DENSE(2, 3) : CHOLESPY_DENSE(4, 2);
#undef CHOLESPY_DENSE
}

hipError_t launch_dense_top(int float_bytes, const DenseTopArgs &args, int panels, int max_k, hipStream_t stream) {
    DenseTopArgs a = args;
    void *p[] = {&a};
    const void *kern = float_bytes == 4 ? dense_kernel<float>(a, max_k) : dense_kernel<double>(a, max_k);
    const int nt = max_k <= 16 ? 1 : (max_k <= 32 ? 2 : 4);
    constexpr int kMost = 1 << 21;   // (a launch takes fewer than 2^32 threads)
    for (int lo = 0; lo < panels; lo += kMost, a.panels += kMost) {
        const unsigned grid = (unsigned)std::min(kMost, panels - lo);
        const hipError_t e = max_k <= kNarrowTile
                                 ? hipLaunchKernel(kern, dim3(grid), dim3(kNarrowThreads), p, 0, stream)
                                 : hipLaunchKernel(kern, dim3(grid, (max_k + 16 * nt - 1) / (16 * nt)), dim3(kWideThreads), p, 0, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace cholespy_amd
