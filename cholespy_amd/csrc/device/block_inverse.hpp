// Dense values of a block plan on the GPU (block_inverse.hip).
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>

#include "block_plan.hpp"

namespace cholespy_amd {

// Device arrays the fill reads: the factor in compressed columns (FP64), the
// plan's structure, and the plan's row numbering: plan row r is factor row
// src[r], factor row i is plan row rank[i].
struct InverseArgs {
    const int64_t *colptr;
    const int *rowidx;
    const double *val;
    const int *src, *rank;
    const int *start, *rptr, *rlist;
    const int64_t *moff;
};

// One product C := alpha op(A) B (column-major, M x N, reduction K).
constexpr int kBLower = 1;   // B is lower triangular: columns from j0 start at k = j0
constexpr int kALower = 2;   // A is lower triangular: rows up to i0 + 63 end at k = i0 + 63
constexpr int kGram = 4;     // op(A) = A', A = B lower triangular; only the lower half of C
struct InverseJob {
    const double *A, *B;
    double *C;
    int64_t lda, ldb, ldc;
    int M, N, K, flags;
    double alpha;
};
struct InverseTile {
    int job, i0, j0;
};
struct InverseColumn {
    int block, c;
    double *dst;
};
struct InversePack {
    const double *X, *Q;
    int64_t off;
    int m, R;
};

// Fills mfwd and mbwd (offsets P.moff) and, for dense top blocks, mtop
// (offsets P.top_off). order (device, null if no top block is a whole system):
// for a whole system, caller row i of it (plan row start + i) is row
// order[start + i] of its factor.
hipError_t fill_block_plan_on_device(const BlockPlan &P, const InverseArgs &args, const int *order, int float_bytes,
                                     void *mfwd, void *mbwd, void *mtop);

// The factor's values in the solver's precision: uvals[p] = val[p] (column
// form), lvals[p] = val[csr_src[p]] (row form).
hipError_t launch_cast_factor(int float_bytes, int64_t nnz, const double *val, const int *csr_src, void *lvals,
                              void *uvals);

}  // namespace cholespy_amd
