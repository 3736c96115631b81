// Block plan for the supernodal partitioned-inverse solve (host side).
//
// The postordered elimination tree of L is cut into contiguous index ranges
// ("blocks") B = [a, a + m). For each block the plan stores the dense matrix
//     M_B = [ L_BB^{-1} ; -L_RB L_BB^{-1} ]          ((m + |R_B|) x m)
// where R_B is the sorted set of rows below the block touched by its columns.
// With it both triangular passes become one dense product per block:
//   forward   r_B = (P b)_B + sum of the partials other blocks wrote for B's rows
//             [y_B ; part_B] = M_B r_B      (part_B: partials for the rows R_B)
//   backward  z_B = M_B' [y_B ; z_{R_B}]
// This is the partitioned-inverse idea (Alvarado & Schreiber 1993; Pothen &
// Alvarado 1992) applied to one dense diagonal block at a time: inside a
// block there is no sequential dependency left, so the only hand-offs between
// workgroups are between blocks, whose tree is far shallower than the
// elimination tree.
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

namespace cholespy_amd {

constexpr int kTaskInts = 8;   // ints per task record (CHOLESPY_TASK_INTS of the C ABI)
constexpr int kGatherSlots = 16;   // contribution slots per row in BlockPlan::gslot
// Leaf blocks: blocks without child blocks (forward level 0) of at most
// kLeafMaxM rows and kLeafMaxRows rows of M_B. They take nothing from other
// blocks in the forward pass and give nothing to other blocks in the
// backward pass, so their tasks can run in a launch of their own before the
// forward pass and after the backward pass (one wavefront per task).
constexpr int kLeafMaxM = 64;
constexpr int kLeafMaxRows = 160;
// Split index and split count of a split task, in one int.
constexpr int split_code(int s, int nsplit) { return nsplit | (s << 8); }
constexpr int split_count(int code) { return code & 255; }
constexpr int split_index(int code) { return code >> 8; }

struct BlockPlanOptions {
    // Rows per block of a chain (the dense inverse is m x m). 0 = automatic:
    // the largest power of two <= the elimination tree's longest chain,
    // within [1024, 4096]. Large 3D separators then take fewer block levels
    // (the 64^3 Laplacian's 4096-row chains: k = 32 refined 7.22 -> 6.29 ms
    // with 4096 against 1024), while icosphere(7), whose longest chain has
    // ~2,000 rows, keeps 1024 (2048 costs it 5 %).
    int max_block = 0;
    int leaf_max = 64;      // whole subtrees up to this size become one block
    int fwd_rows = 64;      // rows of M_B per forward task
    int bwd_cols = 32;      // columns of M_B per backward task
    int split_gather = 65;  // blocks with m >= this gather r_B in separate tasks
    // Blocks with m >= split_gather are few and sit at the top of the block
    // tree, where few tasks run at once: their product tasks are narrower so
    // more workgroups stream each block's M_B concurrently.
    int fwd_rows_big = 32;  // rows per forward product task of such blocks
    int bwd_cols_big = 32;  // columns per backward task of such blocks
    // A product task of such a block that covers more than split_entries
    // entries of M_B is split along its reduction (columns forward, rows
    // backward) into up to max_split tasks of about split_entries entries
    // whose partial results the group's last split adds (0 = no splitting).
    // 8 rather than 16: the icosphere(6) k = 128 FP32 solve 536 -> 517 us,
    // icosphere(7) k = 3 FP64 190 -> 188 us.
    int split_entries = 4096;
    int max_split = 8;
    // Levels whose large blocks hold fewer than level_tasks * split_entries
    // entries split them finer, down to min_split_entries per task, so the
    // level still has about level_tasks tasks (0 = fixed split_entries).
    int level_tasks = 0;
    int min_split_entries = 512;
    // The task list for wide right-hand sides (the MFMA panel kernels, whose
    // tasks carry k times more work per entry): on levels that would give
    // fewer than wide_level_tasks tasks with the narrow shape, narrower
    // gathers and small blocks, more blocks with gather tasks, narrower
    // backward tasks and finer splits; other levels keep the narrow shape.
    int wide_fwd_rows = 16;
    // Rows per forward product task of large blocks on the wide list's
    // sparse levels: 16 (one 16-row MFMA group, the tile columns spread over
    // the 4 wavefronts); busy levels keep fwd_rows_big.
    int wide_fwd_rows_big = 16;
    int wide_split_gather = 33;
    int wide_level_tasks = 512;
    int wide_min_split_entries = 512;
    int wide_fine_bwd_cols_big = 16;   // columns per backward task of large blocks on sparse levels
    // false: the wide list is a copy of the narrow one (batches, whose many
    // systems already give each level enough tasks).
    bool wide_list = true;
    // Order of the blocks inside a level: true = the blocks with the longest
    // chain of levels still ahead of them first (forward: most block
    // ancestors; backward: most block levels below), so the tasks on the
    // pass's critical path take the early tickets; false = block index.
    // Blocks of one level are independent, so either order is a valid
    // schedule.
    bool critical_order = true;
    // Rows of the dense top: the last top_rows rows of the factor (an
    // ancestor-closed set: see choose_dense_top), one block per tree of the
    // elimination forest among them, solved with the explicit inverse X of
    // L's part between the two passes. 0 = none. The host fill does not form
    // its values.
    int top_rows = 0;
    // What choose_dense_top weighs, in microseconds and GB/s: the two passes'
    // launches and leaf tasks, a level of a pass (its hand-offs, and its M_B
    // at the rate the block tasks reach), and the products with X and X' (two
    // launches and X's entries at the rate they reach). Fitted to solves of
    // k = 3 over all cuts of eight systems, in us without a top and with what
    // the rule takes: icosphere(5) FP32 65.3 -> 43.0 (2,640 rows), (6) FP32
    // 93.2 -> 66.2 (5,274), (6) FP64 99.3 -> 72.8, (7) FP32 144.1 -> 142.1
    // (5,109; k = 17 258 -> 221), (7) FP64 none (163.6; 165.6 with 2,886 rows,
    // k = 17 291 and 272), 511 x 389 grid FP64 162.1 -> 151.6 (3,479; 153.1
    // with 6,114), 200 x 150 grid FP64 78.2 -> 51.6 (5,455), 33^3 grid FP64
    // 154.8 -> 123.2 (4,507), 48^3 grid FP32 243.7 -> 230.9 (6,241);
    // k = 32, 64^3 grid (5,514) FP32 1035 -> 996, FP64 1412 -> 1375. More right-
    // hand sides gain more from the same cuts. Of tops of more rows than
    // top_max_rows only 33^3 was measured (6,565: FP32 101.8 -> 95.6, FP64
    // 123.2 -> 122.1): their inverse costs a refactorisation more.
    double pass_us = 25.0, level_us = 3.0, level_gbs = 4000.0, top_us = 10.5, top_gbs = 4000.0;
    int64_t top_max_rows = 6400;
    bool top_forced = false;   // a top wherever a cut fits top_max_rows, estimate or not
    // Host threads for the dense block inverses (0 = hardware count, at most
    // 16). Batches already build one plan per thread and pass 1.
    int threads = 0;
};

struct BlockPlan {
    int n = 0;
    int nblocks = 0;
    // Per block b: rows [start[b], start[b+1]); R rows at rlist[rptr[b]..rptr[b+1]).
    std::vector<int> start, rptr, rlist;
    // Partial-sum slots: block b owns slots [rptr[b], rptr[b+1]) (one per R row).
    // contrib_ptr / contrib_slot: for each row i, the slots whose partial sums
    // belong to row i (CSR over rows).
    std::vector<int> contrib_ptr, contrib_slot;
    // The first kGatherSlots entries of each row's contribution list at a
    // fixed stride (row i at gslot[i * kGatherSlots], -1 padded): a gather
    // loads them without first loading contrib_ptr[i].
    std::vector<int> gslot;
    // Values of M_B in two layouts (one per pass), offsets per block.
    //   forward : column-major packed  (column c holds rows c .. m+|R|-1)
    //   backward: row-major packed     (row rho holds columns 0 .. min(rho, m-1))
    std::vector<int64_t> moff;            // same size for both layouts
    std::vector<double> mfwd, mbwd;
    // Block level in the block tree: forward level (height) and backward level (depth).
    std::vector<int> level_fwd, level_bwd;
    // Tasks in schedule order, kTaskInts ints each:
    //   (block, first, last, kind, lo, hi, sbase, split).
    // Forward kinds: 0 = gather r_B and multiply rows [first, last) of M_B;
    // 1 = gather rows [first, last) of r_B only (published for kinds 2, 3);
    // 4 = the same for a dense top block, into z (read after the pass);
    // 2 = multiply rows [first, last) of M_B by the published r_B;
    // 3 = split s of nsplit (split = split_code(s, nsplit)): as 2 over
    //     columns [lo, hi) only, result published to the split rows
    //     sbase + s * (last - first) + (rho - first) (an array of its own,
    //     k values a row); split nsplit - 1 (the group's last ticket)
    //     waits for the others, adds all nsplit results in split order
    //     and finishes the rows as kind 2 would.
    // Backward kinds: 0 = columns [first, last) of M_B; 1 = split s of
    // nsplit over rows [lo, hi), combined the same way and finished as 0.
    std::vector<int> fwd_task, bwd_task;
    // The leaf blocks' tasks are the first n_leaf_fwd forward tasks and the
    // last n_leaf_bwd backward tasks (the order stays valid for one launch
    // over all tasks).
    int n_leaf_fwd = 0, n_leaf_bwd = 0;
    // The same two passes as tasks for wide right-hand sides (same records,
    // BlockPlanOptions' wide_* shape), leaf tasks first and last as well.
    std::vector<int> fwd_task_wide, bwd_task_wide;
    int n_leaf_fwd_wide = 0, n_leaf_bwd_wide = 0;
    // Dense top blocks (none, or one per tree of a system's top). They have no
    // entries in mfwd / mbwd, no R rows and no backward tasks; their forward
    // tasks are gathers (kind 4) that leave r_B in z, for the products of
    // dense_top.hip. parent: the elimination tree among the block's rows
    // (counted from its first, -1 at the root).
    struct TopBlock {
        int block;
        std::vector<int> parent;
    };
    std::vector<TopBlock> tops;
    std::vector<char> top_flag;            // per block (empty: no top block)
    bool is_top(int b) const { return !top_flag.empty() && top_flag[(std::size_t)b] != 0; }
    int nsplit_rows = 0;                   // rows of the split-result array (either list)
    int max_m = 0, max_rows = 0;           // largest m and m + |R|
    int64_t nnz_l = 0;
};

// Builds the plan, with its values, from L in compressed-column form (rows
// ascending, diagonal first), postordered so that parent(j) > j. The CPU checks
// of the schedule run on it; a solver forms the values on the GPU
// (block_inverse.hip).
BlockPlan build_block_plan(int n, const int *colptr, const int *rowidx, const double *val,
                           const BlockPlanOptions &opt);

// The two halves of build_block_plan. The structure (blocks, R rows, slots,
// levels, tasks) depends only on the pattern of L and is kept over numeric
// refactorisations; fill_block_plan_values computes mfwd / mbwd, but for top
// blocks, on up to `threads` host threads (0 = hardware count, at most 16).
BlockPlan build_block_plan_structure(int n, const int *colptr, const int *rowidx, const BlockPlanOptions &opt);
void fill_block_plan_values(BlockPlan &P, const int *colptr, const int *rowidx, const double *val, int threads);

// The most rows of a dense top (dense_top.hip keeps a wavefront's input units
// in two registers of a row).
constexpr int kTopMaxRows = 7168;
// The most trees a dense top may hold: each is a block with panels of its own.
constexpr int kTopMaxTrees = 64;

// The rows that are worth solving by an explicit inverse, and a numbering
// that puts them last. src[r] = factor row at plan row r (the other rows keep
// their order, then the top rows tree by tree, each in order: a topological
// order of the elimination forest, so L keeps its pattern under it); empty
// src: no top block. Blocks at forward level >= cut (in the partition that
// `opt` gives) are the top rows; the cut minimises the estimated time of the
// levels below it and of the products with the inverse.
struct DenseTop {
    int rows = 0;
    int max_block = 0;   // chain cap of the whole factor's partition
    std::vector<int> src;
};
DenseTop choose_dense_top(int n, const int *colptr, const int *rowidx, const BlockPlanOptions &opt, int float_bytes);

// The pattern of L in the numbering src (columns and rows renumbered, rows ascending).
void renumber_pattern(int n, const int *colptr, const int *rowidx, const std::vector<int> &src,
                      std::vector<int> &new_colptr, std::vector<int> &new_rowidx);

}  // namespace cholespy_amd
