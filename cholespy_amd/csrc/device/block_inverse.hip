// Dense values of the block plan (block_plan.hpp), formed on the GPU in FP64
// from the factor L and rounded once to the solver's precision:
//   M_B = [ L_BB^{-1} ; -L_RB L_BB^{-1} ]   per block, in both packed layouts;
//   X = L_TT^{-1}                           for a dense top block, in the panels of dense_top.hip.
//
// Blocks of up to 64 rows (nearly all of them) take one workgroup each, all
// in LDS: scatter L_BB, invert it column per thread, then multiply L_RB by
// the inverse 64 rows at a time. Larger blocks go through dense work arrays:
// the 64 x 64 diagonal inverses first, then inverses of doubled size,
//   X_21 = -X_22 (L_21 X_11),
// two tile products per doubling for all blocks at once (gemm_tiles, FP64
// MFMA, zero parts of triangular operands skipped), then -L_RB X, and a pack
// kernel that writes both layouts through LDS. Top blocks take the same steps
// on the tiles that X has (dense_top_plan.hpp), in place.
//
// Why on the GPU: the host fill is a few GFLOP of FP64 products and the
// writing, conversion and upload of two copies of M; here only L is uploaded
// (FP64, half to a fifth of M's bytes). refactorize + solve of icosphere(6)
// in FP32: 89 ms with the host fill, 49 ms with this one (what is left is the
// host's numeric factorisation); building a solver for icosphere(7) 1.1 s,
// now 0.45 s.
#include "block_inverse.hpp"

#include <algorithm>
#include <cstdlib>
#include <limits>
#include <vector>

#include "common.hpp"

namespace cholespy_amd {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kSmall = 64;        // rows of a block that is inverted in LDS
constexpr int kLd = kSmall + 1;   // LDS leading dimension
constexpr int kTile = 64;         // output tile of gemm_tiles
constexpr int kKStep = 16;
constexpr int kThreads = 256;

// Packed offsets of M_B entries (block_plan.cpp).
__device__ __forceinline__ int64_t fwd_at(int64_t rows, int64_t c, int64_t rho) {
    return c * rows - c * (c - 1) / 2 + (rho - c);
}
__device__ __forceinline__ int64_t bwd_at(int64_t m, int64_t rho, int64_t c) {
    return rho < m ? rho * (rho + 1) / 2 + c : m * (m + 1) / 2 + (rho - m) * m + c;
}

// Position of row i in the sorted list r[0..n).
__device__ __forceinline__ int find_row(const int *r, int n, int i) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (r[mid] < i) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// X := L^{-1} for the m x m lower triangle L in LDS (row-major, m <= kSmall);
// thread c of the first wavefront solves for column c. The other threads
// wait at the caller's barrier.
__device__ __forceinline__ void invert_lower(const double *L, double *X, int m) {
    const int c = threadIdx.x;
    if (c >= m) return;
    for (int i = 0; i < m; ++i) {
        double s = i == c ? 1.0 : 0.0;
#pragma unroll 8
        for (int j = 0; j < i; ++j) s = fma(-L[i * kLd + j], X[j * kLd + c], s);
        X[i * kLd + c] = s / L[i * kLd + i];
    }
}

template <typename F>
__global__ __launch_bounds__(kThreads) void small_blocks(InverseArgs a, const int *blocks, F *mfwd, F *mbwd) {
    __shared__ double L[kSmall * kLd], X[kSmall * kLd];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b = blocks[blockIdx.x];
    const int a0 = a.start[b], m = a.start[b + 1] - a0, r0 = a.rptr[b], R = a.rptr[b + 1] - r0, rows = m + R;
    F *fw = mfwd + a.moff[b], *bw = mbwd + a.moff[b];
    // Entries of the block's columns: those of L_BB (part 0), or of rows
    // [q0, q0 + kSmall) of L_RB, into L.
    auto scatter = [&](bool diag, int q0) {
        for (int i = tid; i < kSmall * kLd; i += kThreads) L[i] = 0.0;
        __syncthreads();
        for (int c = wave; c < m; c += kThreads / 64) {
            const int j = a.src[a0 + c];
            for (int64_t p = a.colptr[j] + lane; p < a.colptr[j + 1]; p += 64) {
                const int i = a.rank[a.rowidx[p]];
                if ((i < a0 + m) != diag) continue;
                const int q = diag ? i - a0 : find_row(a.rlist + r0, R, i) - q0;
                if (q >= 0 && q < kSmall) L[q * kLd + c] = a.val[p];
            }
        }
        __syncthreads();
    };
    scatter(true, 0);
    if (wave == 0) invert_lower(L, X, m);
    __syncthreads();
    for (int i = tid; i < m * m; i += kThreads) {
        const int r = i % m, c = i / m;
        if (r >= c) fw[fwd_at(rows, c, r)] = (F)X[r * kLd + c];
        const int rr = i / m, cc = i % m;
        if (rr >= cc) bw[bwd_at(m, rr, cc)] = (F)X[rr * kLd + cc];
    }
    for (int q0 = 0; q0 < R; q0 += kSmall) {
        const int nq = min(kSmall, R - q0);
        scatter(false, q0);
        // Lane = row of L_RB, each wavefront 16 columns, four at a time.
        double out[kSmall / 4];
#pragma unroll
        for (int u = 0; u < kSmall / 4; ++u) out[u] = 0.0;
        const int cw = wave * (kSmall / 4);
        for (int j = cw; j < m; ++j) {
            const double l = L[lane * kLd + j];
#pragma unroll
            for (int u = 0; u < kSmall / 4; ++u)
                if (cw + u <= j) out[u] = fma(-l, X[j * kLd + cw + u], out[u]);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kSmall / 4; ++u) {
            const int c = cw + u;
            if (c < m && lane < nq) {
                fw[fwd_at(rows, c, m + q0 + lane)] = (F)out[u];
                L[lane * kLd + c] = out[u];
            }
        }
        __syncthreads();
        for (int i = tid; i < nq * m; i += kThreads) {
            const int q = i / m, c = i % m;
            bw[bwd_at(m, m + q0 + q, c)] = (F)L[q * kLd + c];
        }
        __syncthreads();
    }
}

// Dense copy of the columns of large blocks: one wavefront per column,
// rows [0, m) of L_BB then the R rows of L_RB (D zeroed by the caller).
__global__ __launch_bounds__(64) void scatter_columns(InverseArgs a, const InverseColumn *cols) {
    const InverseColumn col = cols[blockIdx.x];
    const int a0 = a.start[col.block], m = a.start[col.block + 1] - a0, r0 = a.rptr[col.block];
    const int R = a.rptr[col.block + 1] - r0;
    const int j = a.src[a0 + col.c];
    for (int64_t p = a.colptr[j] + threadIdx.x; p < a.colptr[j + 1]; p += 64) {
        const int i = a.rank[a.rowidx[p]];
        const int q = i < a0 + m ? i - a0 : m + find_row(a.rlist + r0, R, i);
        col.dst[q] = a.val[p];
    }
}

// total += A B of one step of kKStep in LDS, for the wavefront's 32 x 32
// quarter at (wi, wj). Sums of kKStep products, then a sum of those: long dot
// products round twice as badly in one running sum.
template <int LD>
__device__ __forceinline__ void step_products(const double (&As)[kKStep][LD], const double (&Bs)[kKStep][LD], int lane, int wi,
                                              int wj, f64x4 (&total)[2][2]) {
    f64x4 acc[2][2] = {};
#pragma unroll
    for (int kk = 0; kk < kKStep; kk += 4) {
        const int k = kk + (lane >> 4);
        const double a0 = As[k][wi + (lane & 15)], a1 = As[k][wi + 16 + (lane & 15)];
        const double b0 = Bs[k][wj + (lane & 15)], b1 = Bs[k][wj + 16 + (lane & 15)];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) total[x][y] += acc[x][y];
}

// C (ldc) := inverse of the m x m lower triangle A (lda), m <= kSmall, by one
// workgroup; C may be A.
__device__ __forceinline__ void invert_tile(const double *A, int64_t lda, double *C, int64_t ldc, int m) {
    __shared__ double L[kSmall * kLd], X[kSmall * kLd];
    for (int i = threadIdx.x; i < m * kSmall; i += kThreads) {
        const int r = i % kSmall, c = i / kSmall;
        if (r < m) L[r * kLd + c] = r >= c ? A[r + c * lda] : 0.0;
    }
    __syncthreads();
    if (threadIdx.x < 64) invert_lower(L, X, m);
    __syncthreads();
    for (int i = threadIdx.x; i < m * kSmall; i += kThreads) {
        const int r = i % kSmall, c = i / kSmall;
        if (r < m && r >= c) C[r + c * ldc] = X[r * kLd + c];
    }
}

// 64 x 64 diagonal inverses: job.C (ldc) := inverse of the M x M lower triangle job.A (lda).
__global__ __launch_bounds__(kThreads) void diagonal_inverses(const InverseJob *jobs) {
    const InverseJob job = jobs[blockIdx.x];
    invert_tile(job.A, job.lda, job.C, job.ldc, job.M);
}

// Top blocks (dense_top_plan.hpp): L into their tiles (zeroed by the caller),
// one wavefront per column; the diagonal tiles inverted in place; a stage of
// tile products; both layouts from the finished tiles.
__global__ __launch_bounds__(64) void top_scatter(InverseArgs a, const TopLists::Column *columns, const int *map, double *D) {
    const TopLists::Column col = columns[blockIdx.x];
    const int nt = map[col.map], j = a.src[col.row0 + col.c];
    const int *tile = map + col.map + 1;
    for (int64_t p = a.colptr[j] + threadIdx.x; p < a.colptr[j + 1]; p += 64) {
        const int i = a.rank[a.rowidx[p]] - col.row0;
        const int t = tile[i / kTopTile * nt + col.c / kTopTile];
        D[(int64_t)t * kTopTileEntries + i % kTopTile + col.c % kTopTile * kTopTile] = a.val[p];
    }
}

__global__ __launch_bounds__(kThreads) void top_diagonals(const TopLists::Diagonal *diagonals, double *D) {
    const TopLists::Diagonal d = diagonals[blockIdx.x];
    double *t = D + (int64_t)d.tile * kTopTileEntries;
    invert_tile(t, kTopTile, t, kTopTile, d.rows);
}

// Out tile := alpha times the sum of the job's tile products A B, as gemm_tiles.
__global__ __launch_bounds__(kThreads) void top_products(const TopLists::Job *jobs, const TopLists::Pair *pairs,
                                                         const double *A, const double *B, double *C, double alpha) {
    constexpr int kLdA = kTopTile + 2, kSteps = kTopTile / kKStep;
    __shared__ double As[kKStep][kLdA], Bs[kKStep][kLdA];
    const TopLists::Job job = jobs[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, total_steps = job.count * kSteps;
    double ra[4], rb[4];
    auto load = [&](int s) {
        const TopLists::Pair pr = pairs[job.first + s / kSteps];
        const double *ta = A + (int64_t)pr.a * kTopTileEntries + s % kSteps * kKStep * kTopTile;
        const double *tb = B + (int64_t)pr.b * kTopTileEntries + s % kSteps * kKStep;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            ra[q] = ta[lane + (wave + 4 * q) * kTopTile];
            rb[q] = tb[tid % 16 + (tid / 16 + 16 * q) * kTopTile];
        }
    };
    f64x4 total[2][2] = {};
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    if (total_steps > 0) load(0);
    for (int s = 0; s < total_steps; ++s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            As[wave + 4 * q][lane] = ra[q];
            Bs[tid % 16][tid / 16 + 16 * q] = rb[q];
        }
        __syncthreads();
        if (s + 1 < total_steps) load(s + 1);
        step_products(As, Bs, lane, wi, wj, total);
        __syncthreads();
    }
    double *out = C + (int64_t)job.out * kTopTileEntries;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                out[wi + 16 * x + (lane >> 4) + 4 * v + (wj + 16 * y + (lane & 15)) * kTopTile] = alpha * total[x][y][v];
}

// One unit a workgroup, of X (fwd) or X'.
template <typename F>
__global__ __launch_bounds__(kTopUnitEntries) void top_pack(const int *pack, const double *D, F *dst, bool fwd) {
    constexpr int V = 16 / (int)sizeof(F), G = 4 * V;
    const int code = pack[blockIdx.x], tid = threadIdx.x;
    const int lane = tid % (64 * V) / V, c = lane % 16, rho = tid / (64 * V) * G + tid % V * 4 + lane / 16;
    double v = 0.0;
    if (code >= 0) {
        const int i0 = code / 4 % 4 * kTopUnit, j0 = code % 4 * kTopUnit;
        v = D[(int64_t)(code / 16) * kTopTileEntries + i0 + (fwd ? c : rho) + (j0 + (fwd ? rho : c)) * kTopTile];
    }
    dst[(int64_t)blockIdx.x * kTopUnitEntries + tid] = (F)v;
}

// C := alpha A B on 64 x 64 tiles (column-major), one workgroup per tile:
// 4 wavefronts of 2 x 2 MFMA 16x16x4 tiles, K in steps of 16 through LDS,
// the next step's entries loaded while the current one is multiplied.
__global__ __launch_bounds__(kThreads) void gemm_tiles(const InverseJob *jobs, const InverseTile *tiles) {
    constexpr int kLdA = kTile + 2;
    __shared__ double As[kKStep][kLdA], Bs[kKStep][kLdA];
    const InverseTile tile = tiles[blockIdx.x];
    const InverseJob job = jobs[tile.job];
    const int i0 = tile.i0, j0 = tile.j0;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int kb = 0, ke = job.K;
    if (job.flags & kBLower) kb = j0;
    if (job.flags & kALower) ke = min(ke, i0 + kTile);
    double ra[4], rb[4];
    auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ak = k0 + wave + 4 * q;
            ra[q] = i0 + lane < job.M && ak < ke ? job.A[i0 + lane + (int64_t)ak * job.lda] : 0.0;
            const int bj = tid / 16 + 16 * q, bk = k0 + tid % 16;
            rb[q] = j0 + bj < job.N && bk < ke ? job.B[bk + (int64_t)(j0 + bj) * job.ldb] : 0.0;
        }
    };
    f64x4 total[2][2] = {};
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
    if (kb < ke) load(kb);
    for (int k0 = kb; k0 < ke; k0 += kKStep) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            As[wave + 4 * q][lane] = ra[q];
            Bs[tid % 16][tid / 16 + 16 * q] = rb[q];
        }
        __syncthreads();
        if (k0 + kKStep < ke) load(k0 + kKStep);
        step_products(As, Bs, lane, wi, wj, total);
        __syncthreads();
    }
    // Accumulator element v of lane l: row l / 16 + 4 v, column l % 16.
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wi + 16 * x + (lane >> 4) + 4 * v, j = j0 + wj + 16 * y + (lane & 15);
                if (i < job.M && j < job.N) job.C[i + (int64_t)j * job.ldc] = job.alpha * total[x][y][v];
            }
}

// Both packed layouts of a large block's 32 x 32 tile (rows i0.., columns
// j0.. of [X ; Q]).
template <typename F>
__global__ __launch_bounds__(kThreads) void pack_tiles(const InversePack *packs, const InverseTile *tiles, F *mfwd,
                                                       F *mbwd) {
    __shared__ double t[32][33];
    const InverseTile tile = tiles[blockIdx.x];
    const InversePack pk = packs[tile.job];
    const int m = pk.m, rows = pk.m + pk.R, lx = threadIdx.x % 32, ly = threadIdx.x / 32;
    for (int q = ly; q < 32; q += kThreads / 32) {
        const int r = tile.i0 + lx, c = tile.j0 + q;
        double v = 0.0;
        if (r < rows && c < m && r >= c) {
            v = r < m ? pk.X[r + (int64_t)c * m] : pk.Q[r - m + (int64_t)c * pk.R];
            mfwd[pk.off + fwd_at(rows, c, r)] = (F)v;
        }
        t[q][lx] = v;   // [column][row]
    }
    __syncthreads();
    for (int q = ly; q < 32; q += kThreads / 32) {
        const int r = tile.i0 + q, c = tile.j0 + lx;
        if (r < rows && c < m && r >= c) mbwd[pk.off + bwd_at(m, r, c)] = (F)t[lx][q];
    }
}

template <typename F>
__global__ void cast_factor(int64_t nnz, const double *val, const int *csr_src, F *lvals, F *uvals) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < nnz; p += (int64_t)gridDim.x * blockDim.x) {
        uvals[p] = (F)val[p];
        lvals[p] = (F)val[csr_src[p]];
    }
}

// Work memory of one group of a fill, within CHOLESPY_FILL_MIB if that is set.
struct Arena {
    std::vector<void *> held;
    int64_t left = std::getenv("CHOLESPY_FILL_MIB") ? fill_work_bytes() : std::numeric_limits<int64_t>::max();
    ~Arena() {
        for (void *p : held) (void)hipFree(p);
    }
    template <typename T>
    hipError_t get(T **p, size_t count) {
        void *q = nullptr;
        *p = nullptr;
        if ((int64_t)(count * sizeof(T)) > left) return hipErrorOutOfMemory;
        left -= (int64_t)(count * sizeof(T));
        const hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
        if (e == hipSuccess) held.push_back(q);
        else (void)hipGetLastError();   // (not for the next launch to report)
        *p = static_cast<T *>(q);
        return e;
    }
    template <typename T>
    hipError_t put(T **p, const std::vector<T> &v) {
        hipError_t e = get(p, v.size());
        if (e == hipSuccess && !v.empty()) e = hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
        return e;
    }
};

#define INV_TRY(expr)                      \
    do {                                   \
        const hipError_t e_ = (expr);      \
        if (e_ != hipSuccess) return e_;   \
    } while (0)

// launch(first, grid) over [lo, hi) in grids that a launch takes (fewer than
// 2^32 threads).
template <typename Launch>
hipError_t in_grids(int64_t lo, int64_t hi, Launch launch) {
    constexpr int64_t kMost = int64_t(1) << 22;
    for (; lo < hi; lo += kMost) {
        launch(lo, (unsigned)std::min(kMost, hi - lo));
        INV_TRY(hipGetLastError());
    }
    return hipSuccess;
}

// The blocks `large` of P through dense work arrays.
template <typename F>
hipError_t fill_large(const BlockPlan &P, const InverseArgs &args, const std::vector<int> &large, F *mfwd, F *mbwd) {
    Arena arena;
    // Work arrays: D = [L_BB ; L_RB] (rows x m), X and T (m x m), Q (R x m).
    size_t dn = 0, xn = 0, qn = 0;
    for (int b : large) {
        const size_t m = P.start[b + 1] - P.start[b], R = P.rptr[b + 1] - P.rptr[b];
        dn += (m + R) * m;
        xn += m * m;
        qn += R * m;
    }
    double *D = nullptr, *X = nullptr, *T = nullptr, *Q = nullptr;
    INV_TRY(arena.get(&D, dn));
    INV_TRY(arena.get(&X, xn));
    INV_TRY(arena.get(&T, xn));
    INV_TRY(arena.get(&Q, qn));
    INV_TRY(hipMemsetAsync(D, 0, dn * sizeof(double), nullptr));
    INV_TRY(hipMemsetAsync(X, 0, xn * sizeof(double), nullptr));
    std::vector<InverseColumn> cols;
    std::vector<InverseJob> diag, jobs;
    std::vector<InverseTile> tiles, ptiles;
    std::vector<InversePack> packs;
    std::vector<size_t> stage{0};   // tile ranges that may run together
    int max_m = 0;
    struct Place {
        double *D, *X, *T, *Q;
        int m, R;
    };
    std::vector<Place> at;
    {
        double *d = D, *x = X, *t = T, *q = Q;
        for (int b : large) {
            const int m = P.start[b + 1] - P.start[b], R = P.rptr[b + 1] - P.rptr[b], rows = m + R;
            at.push_back({d, x, t, q, m, R});
            for (int c = 0; c < m; ++c) cols.push_back({b, c, d + (size_t)c * rows});
            for (int i = 0; i < m; i += kSmall) {
                const int w = std::min(kSmall, m - i);
                diag.push_back({d + i + (size_t)i * rows, nullptr, x + i + (size_t)i * m, rows, 0, m, w, w, w, 0, 1.0});
            }
            packs.push_back({x, q, P.moff[b], m, R});
            for (int i = 0; i < rows; i += 32)
                for (int j = 0; j < m && j <= i; j += 32) ptiles.push_back({(int)packs.size() - 1, i, j});
            max_m = std::max(max_m, m);
            d += (size_t)rows * m;
            x += (size_t)m * m;
            t += (size_t)m * m;
            q += (size_t)R * m;
        }
    }
    auto add = [&](const InverseJob &j) {
        jobs.push_back(j);
        for (int i = 0; i < j.M; i += kTile)
            for (int c = 0; c < j.N; c += kTile) tiles.push_back({(int)jobs.size() - 1, i, c});
    };
    for (int s = kSmall; s < max_m; s *= 2) {
        for (int half = 0; half < 2; ++half) {
            for (const Place &p : at)
                for (int i = 0; i + s < p.m; i += 2 * s) {
                    const int n2 = std::min(s, p.m - i - s), rows = p.m + p.R;
                    const size_t o11 = i + (size_t)i * p.m, o21 = i + s + (size_t)i * p.m,
                                 o22 = i + s + (size_t)(i + s) * p.m;
                    if (half == 0)
                        add({p.D + i + s + (size_t)i * rows, p.X + o11, p.T + o21, rows, p.m, p.m, n2, s, s, kBLower, 1.0});
                    else
                        add({p.X + o22, p.T + o21, p.X + o21, p.m, p.m, p.m, n2, s, n2, kALower, -1.0});
                }
            stage.push_back(tiles.size());
        }
    }
    for (const Place &p : at)
        if (p.R > 0) add({p.D + p.m, p.X, p.Q, p.m + p.R, p.m, p.R, p.R, p.m, p.m, kBLower, -1.0});
    stage.push_back(tiles.size());
    InverseColumn *dcols = nullptr;
    InverseJob *ddiag = nullptr, *djobs = nullptr;
    InverseTile *dtiles = nullptr, *dptiles = nullptr;
    InversePack *dpacks = nullptr;
    INV_TRY(arena.put(&dcols, cols));
    INV_TRY(arena.put(&ddiag, diag));
    INV_TRY(arena.put(&djobs, jobs));
    INV_TRY(arena.put(&dtiles, tiles));
    INV_TRY(arena.put(&dptiles, ptiles));
    INV_TRY(arena.put(&dpacks, packs));
    scatter_columns<<<dim3((unsigned)cols.size()), 64>>>(args, dcols);
    INV_TRY(hipGetLastError());
    diagonal_inverses<<<dim3((unsigned)diag.size()), kThreads>>>(ddiag);
    INV_TRY(hipGetLastError());
    for (size_t q = 0; q + 1 < stage.size(); ++q) {
        const size_t count = stage[q + 1] - stage[q];
        if (count == 0) continue;
        gemm_tiles<<<dim3((unsigned)count), kThreads>>>(djobs, dtiles + stage[q]);
        INV_TRY(hipGetLastError());
    }
    pack_tiles<F><<<dim3((unsigned)ptiles.size()), kThreads>>>(dpacks, dptiles, mfwd, mbwd);
    INV_TRY(hipGetLastError());
    return hipDeviceSynchronize();   // the work arrays are freed on return
}

// The top blocks' X and X', group by group.
template <typename F>
hipError_t fill_tops(const InverseArgs &args, const DeviceTopLists &t, F *mtop) {
    for (const TopLists::Group &g : t.groups) {
        Arena arena;
        double *D = nullptr, *T = nullptr;
        INV_TRY(arena.get(&D, (size_t)g.tiles * kTopTileEntries));
        INV_TRY(arena.get(&T, (size_t)g.temps * kTopTileEntries));
        INV_TRY(hipMemsetAsync(D, 0, (size_t)g.tiles * kTopTileEntries * sizeof(double), nullptr));
        INV_TRY(in_grids(g.columns[0], g.columns[1], [&](int64_t lo, unsigned grid) {
            top_scatter<<<dim3(grid), 64>>>(args, t.columns + lo, t.map, D);
        }));
        INV_TRY(in_grids(g.diagonals[0], g.diagonals[1], [&](int64_t lo, unsigned grid) {
            top_diagonals<<<dim3(grid), kThreads>>>(t.diagonals + lo, D);
        }));
        for (size_t s = 0; s + 1 < g.stages.size(); ++s) {
            const bool even = s % 2 == 0;
            INV_TRY(in_grids(g.stages[s], g.stages[s + 1], [&](int64_t lo, unsigned grid) {
                top_products<<<dim3(grid), kThreads>>>(t.jobs + lo, t.pairs, D, even ? D : T, even ? T : D, even ? 1.0 : -1.0);
            }));
        }
        const int64_t units = t.entries / kTopUnitEntries;
        INV_TRY(in_grids(g.fwd_units[0], g.fwd_units[1], [&](int64_t lo, unsigned grid) {
            top_pack<F><<<dim3(grid), kTopUnitEntries>>>(t.pack + lo, D, mtop + lo * kTopUnitEntries, true);
        }));
        INV_TRY(in_grids(units + g.bwd_units[0], units + g.bwd_units[1], [&](int64_t lo, unsigned grid) {
            top_pack<F><<<dim3(grid), kTopUnitEntries>>>(t.pack + lo, D, mtop + lo * kTopUnitEntries, false);
        }));
        INV_TRY(hipDeviceSynchronize());   // the work arrays are freed
    }
    return hipSuccess;
}

template <typename F>
hipError_t fill(const BlockPlan &P, const InverseArgs &args, const int *small, int n_small, const DeviceTopLists &tops,
                F *mfwd, F *mbwd, F *mtop) {
    std::vector<int> large;
    for (int b = 0; b < P.nblocks; ++b)
        if (!P.is_top(b) && P.start[b + 1] - P.start[b] > kSmall) large.push_back(b);
    INV_TRY(in_grids(0, n_small, [&](int64_t lo, unsigned grid) {
        small_blocks<F><<<dim3(grid), kThreads>>>(args, small + lo, mfwd, mbwd);
    }));
    const size_t most = (size_t)fill_work_bytes() / sizeof(double);
    for (size_t lo = 0; lo < large.size();) {
        size_t hi = lo, words = 0;
        std::vector<int> group;
        for (; hi < large.size(); ++hi) {
            const size_t m = P.start[large[hi] + 1] - P.start[large[hi]], R = P.rptr[large[hi] + 1] - P.rptr[large[hi]];
            words += 3 * m * m + 2 * R * m;
            if (hi > lo && words > most) break;
            group.push_back(large[hi]);
        }
        INV_TRY(fill_large<F>(P, args, group, mfwd, mbwd));
        lo = hi;
    }
    INV_TRY(fill_tops<F>(args, tops, mtop));
    return hipDeviceSynchronize();
}

template <typename T>
hipError_t put(T **dst, const std::vector<T> &v) {
    *dst = nullptr;
    if (v.empty()) return hipSuccess;
    const hipError_t e = hipMalloc(reinterpret_cast<void **>(dst), v.size() * sizeof(T));
    return e != hipSuccess ? e : hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
}

}  // namespace

void DeviceTopLists::release() {
    for (void *p : {(void *)columns, (void *)map, (void *)pack, (void *)diagonals, (void *)jobs, (void *)pairs})
        if (p) (void)hipFree(p);
    *this = DeviceTopLists();
}

hipError_t DeviceTopLists::upload(const TopLists &l) {
    release();
    INV_TRY(put(&columns, l.columns));
    INV_TRY(put(&map, l.map));
    INV_TRY(put(&pack, l.pack));
    INV_TRY(put(&diagonals, l.diagonals));
    INV_TRY(put(&jobs, l.jobs));
    INV_TRY(put(&pairs, l.pairs));
    entries = l.entries;
    groups = l.groups;
    return hipSuccess;
}

int64_t fill_work_bytes() {
    const char *e = std::getenv("CHOLESPY_FILL_MIB");
    return e ? std::min<int64_t>(kTopWorkBytes, (int64_t)std::max(0, std::atoi(e)) << 20) : kTopWorkBytes;
}

std::vector<int> small_block_list(const BlockPlan &P) {
    std::vector<int> small;
    for (int b = 0; b < P.nblocks; ++b)
        if (!P.is_top(b) && P.start[b + 1] - P.start[b] <= kSmall) small.push_back(b);
    return small;
}

hipError_t fill_block_plan_on_device(const BlockPlan &P, const InverseArgs &args, const int *small, int n_small,
                                     const DeviceTopLists &tops, int float_bytes, void *mfwd, void *mbwd, void *mtop) {
    if (P.n == 0) return hipSuccess;
    if (float_bytes == 4)
        return fill<float>(P, args, small, n_small, tops, static_cast<float *>(mfwd), static_cast<float *>(mbwd),
                           static_cast<float *>(mtop));
    return fill<double>(P, args, small, n_small, tops, static_cast<double *>(mfwd), static_cast<double *>(mbwd),
                        static_cast<double *>(mtop));
}

hipError_t launch_cast_factor(int float_bytes, int64_t nnz, const double *val, const int *csr_src, void *lvals,
                              void *uvals) {
    if (nnz == 0) return hipSuccess;
    const unsigned grid = (unsigned)std::min<int64_t>((nnz + 255) / 256, 8192);
    if (float_bytes == 4)
        cast_factor<float><<<grid, 256>>>(nnz, val, csr_src, static_cast<float *>(lvals), static_cast<float *>(uvals));
    else
        cast_factor<double><<<grid, 256>>>(nnz, val, csr_src, static_cast<double *>(lvals), static_cast<double *>(uvals));
    return hipGetLastError();
}

}  // namespace cholespy_amd
