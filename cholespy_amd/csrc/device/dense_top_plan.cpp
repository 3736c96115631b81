#include "dense_top_plan.hpp"

#include <algorithm>

namespace cholespy_amd {

TopLists top_lists(const BlockPlan &P, const std::vector<int> *blk_sys, int64_t work_bytes) {
    TopLists L;
    std::vector<int> pack_bwd;
    int64_t fwd_units = 0, bwd_units = 0;
    int slots[2] = {0, 0};
    // A panel's segments, as even as they go.
    auto push = [&](bool fwd, DenseTopPanel p) {
        const int count = p.count, first = p.first;
        const int64_t off = p.off;
        p.nseg = (count + kTopSegment - 1) / kTopSegment;
        p.slot = p.nseg > 1 ? slots[fwd] : 0;
        if (p.nseg > 1) slots[fwd] += p.nseg;
        for (p.seg = 0; p.seg < p.nseg; ++p.seg) {
            const int lo = (int)((int64_t)count * p.seg / p.nseg), hi = (int)((int64_t)count * (p.seg + 1) / p.nseg);
            p.first = first + lo;
            p.count = hi - lo;
            p.off = off + (int64_t)lo * kTopUnitEntries;
            (fwd ? L.fwd : L.bwd).push_back(p);
        }
    };
    // The jobs of the group's blocks, by stage.
    struct Pending {
        TopLists::Job job;
        int stage;
    };
    std::vector<Pending> pending;
    std::vector<int> temps_of_stage;
    TopLists::Group group;
    auto open = [&]() {
        group = TopLists::Group();
        group.columns[0] = (int)L.columns.size();
        group.diagonals[0] = (int)L.diagonals.size();
        group.fwd_units[0] = fwd_units;
        group.bwd_units[0] = bwd_units;
        pending.clear();
        temps_of_stage.clear();
    };
    auto close = [&]() {
        group.columns[1] = (int)L.columns.size();
        group.diagonals[1] = (int)L.diagonals.size();
        group.fwd_units[1] = fwd_units;
        group.bwd_units[1] = bwd_units;
        for (int t : temps_of_stage) group.temps = std::max(group.temps, t);
        std::stable_sort(pending.begin(), pending.end(), [](const Pending &a, const Pending &b) {
            return a.stage != b.stage ? a.stage < b.stage : a.job.count > b.job.count;
        });
        group.stages.assign(1, (int)L.jobs.size());
        for (const Pending &q : pending) {
            while ((int)group.stages.size() <= q.stage) group.stages.push_back((int)L.jobs.size());
            L.jobs.push_back(q.job);
        }
        group.stages.push_back((int)L.jobs.size());
        L.groups.push_back(group);
    };
    open();
    for (const BlockPlan::TopBlock &top : P.tops) {
        const int row0 = P.start[top.block], m = (int)top.parent.size(), sys = blk_sys ? (*blk_sys)[top.block] : 0;
        const int np = (m + kTopUnit - 1) / kTopUnit, nt = (m + kTopTile - 1) / kTopTile, per = kTopTile / kTopUnit;
        // has[p * np + q]: unit (p, q) of X holds a pair of an ancestor and its descendant.
        std::vector<char> has((size_t)np * np, 0);
        // (An ancestor among the same 16 columns marks the rest of the path.)
        for (int j = 0; j < m; ++j)
            for (int i = j; i >= 0; i = top.parent[i]) {
                has[(size_t)(i / kTopUnit) * np + j / kTopUnit] = 1;
                if (i > j && i / kTopUnit == j / kTopUnit) break;
            }
        std::vector<int> tile((size_t)nt * nt, -1);
        int count = 0;
        for (int p = 0; p < np; ++p)
            for (int q = 0; q <= p; ++q)
                if (has[(size_t)p * np + q] && tile[(size_t)(p / per) * nt + q / per] < 0)
                    tile[(size_t)(p / per) * nt + q / per] = count++;
        // (Temporaries: at most the tiles below the diagonal.)
        if (group.tiles > 0 && (int64_t)2 * (group.tiles + count) * kTopTileEntries * 8 > work_bytes) {
            close();
            open();
        }
        for (int &t : tile)
            if (t >= 0) t += group.tiles;
        group.tiles += count;
        const int map = (int)L.map.size();
        L.map.push_back(nt);
        L.map.insert(L.map.end(), tile.begin(), tile.end());
        for (int c = 0; c < m; ++c) L.columns.push_back({c, row0, map});
        auto code = [&](int p, int q) {
            const int t = tile[(size_t)(p / per) * nt + q / per];
            return t < 0 ? -1 : t * per * per + p % per * per + q % per;
        };
        // Panels. A row's descendants are consecutive under a postorder; any
        // other numbering keeps the whole range from the lowest one on.
        for (int p = 0; p < np; ++p) {
            int lo = 0;
            while (!has[(size_t)p * np + lo]) ++lo;
            push(true, {row0, m, p, sys, lo, p - lo + 1, 0, 1, 0, 0, fwd_units * kTopUnitEntries});
            for (int q = lo; q <= p; ++q) L.pack.push_back(code(p, q));
            fwd_units += p - lo + 1;
            const int first = (int)L.units.size();
            for (int r = p; r < np; ++r)
                if (has[(size_t)r * np + p]) {
                    L.units.push_back(r);
                    pack_bwd.push_back(code(r, p));
                }
            const int count = (int)L.units.size() - first;
            push(false, {row0, m, p, sys, first, count, 0, 1, 0, 0, bwd_units * kTopUnitEntries});
            bwd_units += count;
        }
        // Stages 2 s' (into temporaries) and 2 s' + 1 (back) of doubling s'.
        for (int i = 0; i < nt; ++i) L.diagonals.push_back({tile[(size_t)i * nt + i], std::min(kTopTile, m - i * kTopTile)});
        int stage = 0;
        for (int s = 1; s < nt; s *= 2, stage += 2) {
            if ((int)temps_of_stage.size() <= stage) temps_of_stage.resize((size_t)stage + 2, 0);
            std::vector<int> temp((size_t)nt * nt, -1);
            for (int half = 0; half < 2; ++half)
                for (int g = 0; g + s < nt; g += 2 * s)
                    for (int i = g + s; i < std::min(nt, g + 2 * s); ++i)
                        for (int j = g; j < g + s; ++j) {
                            const int out = tile[(size_t)i * nt + j];
                            if (out < 0) continue;
                            TopLists::Job job{out, (int)L.pairs.size(), 0};
                            if (half == 0) job.out = temp[(size_t)i * nt + j] = temps_of_stage[(size_t)stage]++;
                            const int k0 = half == 0 ? j : g + s, k1 = half == 0 ? g + s : i + 1;
                            for (int k = k0; k < k1; ++k) {
                                const int a = tile[(size_t)i * nt + k];
                                const int b = half == 0 ? tile[(size_t)k * nt + j] : temp[(size_t)k * nt + j];
                                if (a >= 0 && b >= 0) L.pairs.push_back({a, b});
                            }
                            job.count = (int)L.pairs.size() - job.first;
                            pending.push_back({job, stage + half});
                        }
        }
    }
    if (group.tiles > 0) close();
    L.slots = std::max(slots[0], slots[1]);
    L.entries = std::max(fwd_units, bwd_units) * kTopUnitEntries;
    L.pack.resize((size_t)std::max(fwd_units, bwd_units), -1);
    pack_bwd.resize(L.pack.size(), -1);
    L.pack.insert(L.pack.end(), pack_bwd.begin(), pack_bwd.end());
    auto longest = [](const DenseTopPanel &a, const DenseTopPanel &b) { return a.count > b.count; };
    std::stable_sort(L.fwd.begin(), L.fwd.end(), longest);
    std::stable_sort(L.bwd.begin(), L.bwd.end(), longest);
    return L;
}

}  // namespace cholespy_amd
