// Dense values of a block plan on the GPU (block_inverse.hip).
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>

#include "block_plan.hpp"
#include "dense_top_plan.hpp"

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

// One product C := alpha A B (column-major, M x N, reduction K).
constexpr int kBLower = 1;   // B is lower triangular: columns from j0 start at k = j0
constexpr int kALower = 2;   // A is lower triangular: rows up to i0 + 63 end at k = i0 + 63
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

// Device copies of the lists that form the top blocks' inverses
// (dense_top_plan.hpp), the groups on the host.
struct DeviceTopLists {
    TopLists::Column *columns = nullptr;
    int *map = nullptr, *pack = nullptr;
    TopLists::Diagonal *diagonals = nullptr;
    TopLists::Job *jobs = nullptr;
    TopLists::Pair *pairs = nullptr;
    int64_t entries = 0;           // elements of one direction's array
    std::vector<TopLists::Group> groups;
    void release();
    hipError_t upload(const TopLists &lists);
};

// Fills mfwd and mbwd (offsets P.moff) and the top blocks' mtop (X, then X',
// tops.entries elements each). small: device list of the n_small blocks of up
// to 64 rows that are not top blocks. Work memory that cannot be had, or more
// of it at a time than CHOLESPY_FILL_MIB allows, ends in
// hipErrorOutOfMemory, by then with some values overwritten.
hipError_t fill_block_plan_on_device(const BlockPlan &P, const InverseArgs &args, const int *small, int n_small,
                                     const DeviceTopLists &tops, int float_bytes, void *mfwd, void *mbwd, void *mtop);
// The work memory a fill takes at a time where one block does not need more:
// 4 GiB, or what CHOLESPY_FILL_MIB allows.
int64_t fill_work_bytes();
// The blocks of P that `small` lists.
std::vector<int> small_block_list(const BlockPlan &P);

// The factor's values in the solver's precision: uvals[p] = val[p] (column
// form), lvals[p] = val[csr_src[p]] (row form).
hipError_t launch_cast_factor(int float_bytes, int64_t nnz, const double *val, const int *csr_src, void *lvals,
                              void *uvals);

}  // namespace cholespy_amd
