// CPU emulation of plans with a dense top (cholespy_amd/csrc/device/
// block_plan.cpp, dense_top_plan.cpp), used by tests/test_dense_top_plan.py.
//
// Forms X = L_TT^{-1} with the tile lists, runs the forward tasks of one list,
// y_T = X r_T by panels, z_T = X' y_T by panels and the backward tasks, one at
// a time in ticket order, every published value NaN until it is written, and
// compares with a sequential solve. Fails as well when
//   - the numbering is no topological order, a panel, unit or tile lies outside
//     its block or array, or the panels do not cover the top's rows once;
//   - the leaf tasks (of either list) do not fit the leaf kernels, do not come
//     first (forward) and last (backward), or receive partial sums;
//   - a top block has a backward task or a forward task that is no gather;
//   - a NaN in the right-hand side of one tree of the elimination forest
//     reaches the solution of another.
//
// Usage: dense_top_emulator FILE narrow|wide ROWS SHUFFLE MIB
// FILE as in plan_emulator.cpp; ROWS: the most rows of the top, whose levels
// are then always worth it; SHUFFLE != 0: the factor renumbered first by a
// random topological order (no postorder); MIB: the work
// arrays' bound, in groups.
#include "block_plan.hpp"
#include "dense_top_plan.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <queue>
#include <random>
#include <set>
#include <string>
#include <vector>

using namespace cholespy_amd;

namespace {

struct Failure {
    std::string what;
};
void check(bool ok, const char *what) {
    if (!ok) throw Failure{what};
}

struct Factor {
    int n = 0;
    std::vector<int> cp, ri;
    std::vector<double> v;
};

Factor renumbered(const Factor &f, const std::vector<int> &src) {
    Factor g;
    g.n = f.n;
    std::vector<int> rank((size_t)f.n, -1);
    for (int r = 0; r < f.n; ++r) rank[src[r]] = r;
    for (int r : rank) check(r >= 0, "the numbering is no permutation");
    g.cp.push_back(0);
    for (int r = 0; r < f.n; ++r) {
        std::vector<std::pair<int, double>> col;
        for (int p = f.cp[src[r]]; p < f.cp[src[r] + 1]; ++p) col.push_back({rank[f.ri[p]], f.v[p]});
        std::sort(col.begin(), col.end());
        check(col[0].first == r, "the numbering is no topological order");
        for (auto &e : col) {
            g.ri.push_back(e.first);
            g.v.push_back(e.second);
        }
        g.cp.push_back((int)g.ri.size());
    }
    return g;
}

std::vector<int> random_topological(const Factor &f) {
    std::vector<int> children((size_t)f.n, 0), src;
    auto parent = [&](int j) { return f.cp[j + 1] - f.cp[j] > 1 ? f.ri[f.cp[j] + 1] : -1; };
    for (int j = 0; j < f.n; ++j)
        if (parent(j) >= 0) ++children[parent(j)];
    std::mt19937 gen(3);
    std::priority_queue<std::pair<unsigned, int>> ready;
    for (int j = 0; j < f.n; ++j)
        if (children[j] == 0) ready.push({gen(), j});
    while (!ready.empty()) {
        const int j = ready.top().second;
        ready.pop();
        src.push_back(j);
        const int p = parent(j);
        if (p >= 0 && --children[p] == 0) ready.push({gen(), p});
    }
    return src;
}

// X in both packed arrays, unit by unit: element [unit][output][input].
void form_inverse(const Factor &f, const TopLists &L, std::vector<double> &xf, std::vector<double> &xb) {
    const size_t units = (size_t)(L.entries / kTopUnitEntries);
    check(L.pack.size() == 2 * units, "one pack code a unit");
    xf.assign(units * kTopUnitEntries, NAN);
    xb.assign(units * kTopUnitEntries, NAN);
    int columns = 0, diagonals = 0, jobs = 0;
    int64_t fwd = 0, bwd = 0;
    for (const TopLists::Group &g : L.groups) {
        check(g.columns[0] == columns && g.diagonals[0] == diagonals && g.stages.front() == jobs && g.fwd_units[0] == fwd &&
                  g.bwd_units[0] == bwd,
              "groups follow one another");
        columns = g.columns[1], diagonals = g.diagonals[1], jobs = g.stages.back(), fwd = g.fwd_units[1], bwd = g.bwd_units[1];
        std::vector<double> D((size_t)g.tiles * kTopTileEntries, 0.0), T((size_t)g.temps * kTopTileEntries, NAN);
        auto at = [](std::vector<double> &v, int tile, int i, int j) -> double & {
            return v[(size_t)tile * kTopTileEntries + i + (size_t)j * kTopTile];
        };
        for (int q = g.columns[0]; q < g.columns[1]; ++q) {
            const auto &c = L.columns[q];
            for (int p = f.cp[c.row0 + c.c]; p < f.cp[c.row0 + c.c + 1]; ++p) {
                const int i = f.ri[p] - c.row0, nt = L.map[c.map];
                check(i / kTopTile < nt, "an entry of a top column lies below its block");
                const int tile = L.map[c.map + 1 + i / kTopTile * nt + c.c / kTopTile];
                check(tile >= 0 && tile < g.tiles, "an entry of L has no tile");
                at(D, tile, i % kTopTile, c.c % kTopTile) = f.v[p];
            }
        }
        for (int q = g.diagonals[0]; q < g.diagonals[1]; ++q) {
            const auto &d = L.diagonals[q];
            std::vector<double> X((size_t)kTopTileEntries, 0.0);
            for (int c = 0; c < d.rows; ++c)
                for (int i = c; i < d.rows; ++i) {
                    double s = i == c ? 1.0 : 0.0;
                    for (int j = c; j < i; ++j) s -= at(D, d.tile, i, j) * X[(size_t)j + (size_t)c * kTopTile];
                    X[(size_t)i + (size_t)c * kTopTile] = s / at(D, d.tile, i, i);
                }
            std::copy(X.begin(), X.end(), D.begin() + (size_t)d.tile * kTopTileEntries);
        }
        for (size_t s = 0; s + 1 < g.stages.size(); ++s) {
            const bool even = s % 2 == 0;
            std::vector<double> &B = even ? D : T, &C = even ? T : D;
            std::vector<std::pair<int, std::vector<double>>> results;   // a stage's jobs are independent
            for (int q = g.stages[s]; q < g.stages[s + 1]; ++q) {
                const auto &job = L.jobs[q];
                check(job.out >= 0 && job.out < (even ? g.temps : g.tiles), "a job's result has no place");
                std::vector<double> out((size_t)kTopTileEntries, 0.0);
                for (int p = job.first; p < job.first + job.count; ++p) {
                    const auto &pr = L.pairs[p];
                    check(pr.a >= 0 && pr.a < g.tiles && pr.b >= 0 && pr.b < (even ? g.tiles : g.temps), "a pair's tile");
                    for (int j = 0; j < kTopTile; ++j)
                        for (int k = 0; k < kTopTile; ++k) {
                            const double b = at(B, pr.b, k, j);
                            if (b != 0.0)
                                for (int i = 0; i < kTopTile; ++i) out[(size_t)i + (size_t)j * kTopTile] += at(D, pr.a, i, k) * b;
                        }
                }
                if (!even)
                    for (double &v : out) v = -v;
                results.push_back({job.out, out});
            }
            for (auto &r : results) std::copy(r.second.begin(), r.second.end(), C.begin() + (size_t)r.first * kTopTileEntries);
        }
        for (int dir = 0; dir < 2; ++dir)
            for (int64_t u = (dir ? g.bwd_units : g.fwd_units)[0]; u < (dir ? g.bwd_units : g.fwd_units)[1]; ++u) {
                const int code = L.pack[(size_t)u + dir * units];
                check(code < 16 * g.tiles, "a unit's tile");
                for (int o = 0; o < kTopUnit; ++o)
                    for (int i = 0; i < kTopUnit; ++i) {
                        const int r0 = code / 4 % 4 * kTopUnit, c0 = code % 4 * kTopUnit;
                        (dir ? xb : xf)[((size_t)u * kTopUnit + o) * kTopUnit + i] =
                            code < 0 ? 0.0 : dir ? at(D, code / 16, r0 + i, c0 + o) : at(D, code / 16, r0 + o, c0 + i);
                    }
            }
    }
    check(columns == (int)L.columns.size() && diagonals == (int)L.diagonals.size() && jobs == (int)L.jobs.size(),
          "groups cover the lists");
}

// The product of one direction: out = X in or X' in on the top rows.
void product(const TopLists &L, bool forward, const std::vector<double> &x, const std::vector<double> &in,
             std::vector<double> &out) {
    std::set<int> rows, slots;
    std::set<std::pair<int, int>> segments;
    for (const auto &c : L.columns) out[(size_t)c.row0 + c.c] = 0.0;
    int longest = 1 << 30;
    for (const DenseTopPanel &p : forward ? L.fwd : L.bwd) {
        check(p.count > 0 && p.count <= kTopSegment && p.count <= longest, "panels longest first");
        check(p.seg >= 0 && p.seg < p.nseg && segments.insert({p.row0 + p.panel * kTopUnit, p.seg}).second, "a segment twice");
        if (p.nseg > 1) check(p.slot >= 0 && p.slot + p.nseg <= L.slots && slots.insert(p.slot + p.seg).second, "a slot twice");
        longest = p.count;
        check(p.off >= 0 && p.off + (int64_t)p.count * kTopUnitEntries <= L.entries, "a panel outside its array");
        for (int o = 0; o < kTopUnit; ++o) {
            const int c = p.panel * kTopUnit + o;
            if (c >= p.n) continue;
            if (p.seg == 0) check(rows.insert(p.row0 + c).second, "a top row in two panels");
            double s = 0.0;
            for (int u = 0; u < p.count; ++u) {
                const int unit = forward ? p.first + u : L.units[(size_t)p.first + u];
                check(unit >= 0 && unit * kTopUnit < p.n, "a unit outside its block");
                for (int i = 0; i < kTopUnit; ++i)
                    if (unit * kTopUnit + i < p.n)
                        s += x[(size_t)p.off + (size_t)(u * kTopUnit + o) * kTopUnit + i] * in[(size_t)p.row0 + unit * kTopUnit + i];
            }
            out[(size_t)p.row0 + c] += s;
        }
    }
    for (const DenseTopPanel &p : forward ? L.fwd : L.bwd)
        for (int q = 0; q < p.nseg; ++q) check(segments.count({p.row0 + p.panel * kTopUnit, q}) == 1, "a segment is missing");
    size_t n = 0;
    for (const auto &c : L.columns) n += (size_t)(c.c >= 0);
    check(rows.size() == n, "panels cover the top rows");
}

void check_leaves(const BlockPlan &P, const std::vector<int> &fwd, const std::vector<int> &bwd, int nlf, int nlb) {
    std::set<int> leaf, leaf_bwd;
    const size_t nf = fwd.size() / kTaskInts, nb = bwd.size() / kTaskInts;
    check((size_t)nlf <= nf && (size_t)nlb <= nb, "leaf counts exceed the lists");
    for (int t = 0; t < nlf; ++t) {
        const int *T = &fwd[(size_t)t * kTaskInts];
        const int b = T[0], m = P.start[b + 1] - P.start[b], R = P.rptr[b + 1] - P.rptr[b];
        check(T[3] == 0 && P.level_fwd[b] == 0 && m <= kLeafMaxM && m + R <= kLeafMaxRows && T[2] - T[1] <= 64 && !P.is_top(b),
              "a leaf forward task does not fit the leaf kernels");
        for (int i = P.start[b]; i < P.start[b + 1]; ++i)
            check(P.contrib_ptr[i + 1] == P.contrib_ptr[i], "a leaf block's row receives partial sums");
        leaf.insert(b);
    }
    for (size_t t = nb - (size_t)nlb; t < nb; ++t) {
        const int *T = &bwd[t * kTaskInts];
        check(T[3] == 0 && T[2] - T[1] <= 32, "a leaf backward task does not fit the leaf kernels");
        leaf_bwd.insert(T[0]);
    }
    check(leaf == leaf_bwd, "forward and backward leaf tasks cover different blocks");
    for (size_t t = (size_t)nlf; t < nf; ++t) check(!leaf.count(fwd[t * kTaskInts]), "a leaf block's task among the others");
}

std::vector<double> solve(const BlockPlan &P, const TopLists &L, const std::vector<double> &xf, const std::vector<double> &xb,
                          bool wide, const std::vector<double> &b, bool nans) {
    const std::vector<int> &ft = wide ? P.fwd_task_wide : P.fwd_task, &bt = wide ? P.bwd_task_wide : P.bwd_task;
    std::vector<double> y((size_t)P.n, NAN), z((size_t)P.n, NAN), rbuf((size_t)P.n, NAN), part(P.rlist.size(), NAN),
        split((size_t)std::max(1, P.nsplit_rows), NAN);
    std::vector<char> written(P.rlist.size(), 0), zset((size_t)P.n, 0);
    for (size_t t = 0; t < ft.size() / kTaskInts; ++t) {
        const int *T = &ft[t * kTaskInts];
        const int blk = T[0], first = T[1], last = T[2], kind = T[3], sbase = T[6];
        const int nsp = split_count(T[7]), sidx = split_index(T[7]);
        const int a0 = P.start[blk], m = P.start[blk + 1] - a0, r0 = P.rptr[blk], rows = m + P.rptr[blk + 1] - r0;
        check(P.is_top(blk) == (kind == 4), "a top block's forward tasks are its gathers");
        const double *M = P.mfwd.data() + P.moff[blk];
        auto gather = [&](int i) {
            double s = b[(size_t)a0 + i];
            for (int p = P.contrib_ptr[a0 + i]; p < P.contrib_ptr[a0 + i + 1]; ++p) {
                check(written[P.contrib_slot[p]], "an unwritten partial sum is read");
                s += part[P.contrib_slot[p]];
            }
            return s;
        };
        if (kind == 1 || kind == 4) {
            for (int i = first; i < last; ++i) (kind == 4 ? z : rbuf)[(size_t)a0 + i] = gather(i);
            continue;
        }
        auto put = [&](int rho, double v) {
            if (rho < m) y[(size_t)a0 + rho] = v;
            else {
                part[(size_t)r0 + rho - m] = v;
                written[(size_t)r0 + rho - m] = 1;
            }
        };
        const int lo = kind == 3 ? T[4] : 0, hi = kind == 3 ? T[5] : m;
        for (int rho = first; rho < last; ++rho) {
            double s = 0.0;
            for (int c = lo; c < std::min(rho < m ? rho + 1 : m, hi); ++c)
                s += M[(int64_t)c * rows - (int64_t)c * (c - 1) / 2 + rho - c] * (kind == 0 ? gather(c) : rbuf[(size_t)a0 + c]);
            if (kind == 3) split[(size_t)sbase + sidx * (last - first) + rho - first] = s;
            else put(rho, s);
        }
        if (kind == 3 && sidx == nsp - 1)
            for (int i = 0; i < last - first; ++i) {
                double s = 0.0;
                for (int q = 0; q < nsp; ++q) s += split[(size_t)sbase + q * (last - first) + i];
                put(first + i, s);
            }
    }
    product(L, true, xf, z, y);
    product(L, false, xb, y, z);
    for (const auto &c : L.columns) zset[(size_t)c.row0 + c.c] = 1;
    for (size_t t = 0; t < bt.size() / kTaskInts; ++t) {
        const int *T = &bt[t * kTaskInts];
        const int blk = T[0], first = T[1], last = T[2], kind = T[3], sbase = T[6];
        const int nsp = split_count(T[7]), sidx = split_index(T[7]);
        const int a0 = P.start[blk], m = P.start[blk + 1] - a0, r0 = P.rptr[blk], rows = m + P.rptr[blk + 1] - r0;
        check(!P.is_top(blk), "a top block has a backward task");
        const double *M = P.mbwd.data() + P.moff[blk];
        const int lo = kind == 1 ? T[4] : 0, hi = kind == 1 ? T[5] : rows;
        for (int c = first; c < last; ++c) {
            double s = 0.0;
            for (int rho = std::max(lo, c); rho < hi; ++rho) {
                if (rho >= m) check(zset[P.rlist[r0 + rho - m]], "an unwritten row of z is read");
                s += M[rho < m ? (int64_t)rho * (rho + 1) / 2 + c : (int64_t)m * (m + 1) / 2 + (int64_t)(rho - m) * m + c] *
                     (rho < m ? y[(size_t)a0 + rho] : z[P.rlist[r0 + rho - m]]);
            }
            if (kind == 1) split[(size_t)sbase + sidx * (last - first) + c - first] = s;
            else z[(size_t)a0 + c] = s, zset[(size_t)a0 + c] = 1;
        }
        if (kind == 1 && sidx == nsp - 1)
            for (int i = 0; i < last - first; ++i) {
                double s = 0.0;
                for (int q = 0; q < nsp; ++q) s += split[(size_t)sbase + q * (last - first) + i];
                z[(size_t)a0 + first + i] = s;
                zset[(size_t)a0 + first + i] = 1;
            }
    }
    for (int i = 0; i < P.n; ++i) check(zset[i] && (nans || !std::isnan(z[i])), "a row of the solution is missing");
    return z;
}

int run(const char *path, bool wide, int most, bool shuffle, int mib) {
    Factor f;
    FILE *fh = std::fopen(path, "rb");
    check(fh != nullptr, "cannot open the factor file");
    int64_t hdr[2];
    check(std::fread(hdr, 8, 2, fh) == 2, "short file");
    f.n = (int)hdr[0];
    f.cp.resize((size_t)f.n + 1);
    f.ri.resize((size_t)hdr[1]);
    f.v.resize((size_t)hdr[1]);
    check(std::fread(f.cp.data(), 4, f.cp.size(), fh) == f.cp.size() && std::fread(f.ri.data(), 4, f.ri.size(), fh) == f.ri.size() &&
              std::fread(f.v.data(), 8, f.v.size(), fh) == f.v.size(),
          "short file");
    std::fclose(fh);
    if (shuffle) f = renumbered(f, random_topological(f));

    BlockPlanOptions opt;
    opt.threads = 1;
    opt.top_max_rows = most;
    BlockPlanOptions choose = opt;
    choose.level_us = 1e6;   // every level above the cap is worth removing
    const DenseTop top = choose_dense_top(f.n, f.cp.data(), f.ri.data(), choose, 8);
    check(top.rows <= std::min(most, kTopMaxRows), "more top rows than asked for");
    if (top.rows > 0) {
        opt.top_rows = top.rows;
        opt.max_block = top.max_block;
        std::vector<int> cp, ri;
        renumber_pattern(f.n, f.cp.data(), f.ri.data(), top.src, cp, ri);
        f = renumbered(f, top.src);
        check(cp == f.cp && ri == f.ri, "renumber_pattern");
    }
    BlockPlan P = build_block_plan_structure(f.n, f.cp.data(), f.ri.data(), opt);
    fill_block_plan_values(P, f.cp.data(), f.ri.data(), f.v.data(), 1);
    const TopLists L = top_lists(P, nullptr, (int64_t)mib << 20);
    int tiles = 0, temps = 0;
    size_t stages = 0;
    for (const TopLists::Group &g : L.groups) {
        std::set<int> blocks;
        for (int q = g.columns[0]; q < g.columns[1]; ++q) blocks.insert(L.columns[q].row0);
        check(blocks.size() == 1 || (int64_t)(g.tiles + g.temps) * kTopTileEntries * 8 <= (int64_t)mib << 20, "a group's bound");
        tiles += g.tiles;
        temps = std::max(temps, g.temps);
        stages = std::max(stages, g.stages.size() - 1);
    }
    std::vector<double> xf, xb;
    form_inverse(f, L, xf, xb);
    check_leaves(P, P.fwd_task, P.bwd_task, P.n_leaf_fwd, P.n_leaf_bwd);
    check_leaves(P, P.fwd_task_wide, P.bwd_task_wide, P.n_leaf_fwd_wide, P.n_leaf_bwd_wide);

    std::mt19937 gen(7);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    std::vector<double> b((size_t)f.n);
    for (double &e : b) e = U(gen);
    std::vector<double> ref = b;
    for (int j = 0; j < f.n; ++j) {
        ref[j] /= f.v[f.cp[j]];
        for (int p = f.cp[j] + 1; p < f.cp[j + 1]; ++p) ref[f.ri[p]] -= f.v[p] * ref[j];
    }
    for (int j = f.n - 1; j >= 0; --j) {
        for (int p = f.cp[j] + 1; p < f.cp[j + 1]; ++p) ref[j] -= f.v[p] * ref[f.ri[p]];
        ref[j] /= f.v[f.cp[j]];
    }
    const std::vector<double> z = solve(P, L, xf, xb, wide, b, false);
    double err = 0.0, scale = 0.0;
    for (int i = 0; i < f.n; ++i) {
        err = std::max(err, std::fabs(z[i] - ref[i]));
        scale = std::max(scale, std::fabs(ref[i]));
    }
    check(err <= 1e-10 * scale, "the solution differs from the sequential solve");

    // One tree's right-hand side NaN: the other trees' solutions stay as they were.
    std::vector<int> root((size_t)f.n);
    std::set<int> trees;
    for (int j = f.n - 1; j >= 0; --j) {
        root[j] = f.cp[j + 1] - f.cp[j] > 1 ? root[f.ri[f.cp[j] + 1]] : j;
        trees.insert(root[j]);
    }
    std::vector<double> bn = b;
    for (int j = 0; j < f.n; ++j)
        if (root[j] == root[f.n - 1]) bn[j] = NAN;
    const std::vector<double> zn = solve(P, L, xf, xb, wide, bn, true);
    for (int j = 0; j < f.n; ++j)
        check(root[j] == root[f.n - 1] ? std::isnan(zn[j]) : zn[j] == z[j], "a NaN reaches another tree");
    std::printf("ok n %d top %d in %zu blocks of %d, trees %zu, panels %zu units %lld tiles %d temps %d stages %zu groups %zu err %.1e\n", f.n,
                top.rows, P.tops.size(), P.nblocks, trees.size(), L.fwd.size(), (long long)(L.entries / kTopUnitEntries), tiles,
                temps, stages, L.groups.size(), err / scale);
    return 0;
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 6) {
        std::fprintf(stderr, "usage: %s FILE narrow|wide ROWS SHUFFLE MIB\n", argv[0]);
        return 2;
    }
    try {
        return run(argv[1], std::strcmp(argv[2], "wide") == 0, std::atoi(argv[3]), std::atoi(argv[4]) != 0, std::atoi(argv[5]));
    } catch (const Failure &e) {
        std::printf("FAIL %s\n", e.what.c_str());
    } catch (const std::exception &e) {
        std::printf("FAIL %s\n", e.what());
    }
    return 1;
}
