// ofx_sweep.h -- schedule of the pipelined LU-SGS sweeps (host code, no GPU).
//
// A numbering with many narrow dependency levels (a structured-like order)
// cannot fill the GPU one level at a time.  The pipelined sweep cuts the
// traversal order (ascending cell ids for the lower sweep, descending for the
// upper one) into ranges of consecutive cells, one workgroup each.  A cell
// depends on cells earlier in the traversal only, so range k depends on
// ranges before k only: the ranges form a pipeline, each lagging the one
// before it by the levels their cells share, and a workgroup needs no more
// than its own cells' increments and a halo of earlier ranges' in LDS.
//
// Range sizes follow the grid: a range grows while its cells keep to a few per
// level (its workgroup then works at the pace of the dependency chain), up to
// what LDS holds; where levels are wide (rings of triangles, say) ranges stay
// small, so that many workgroups share a level.
//
// Within a range the cells are stored by (dependency level, traversal order),
// the level being the one of the whole grid (the longest path to the cell),
// so that cells come in the order in which they can become ready.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace ofx {

constexpr int SW_MAXNE = 6;  // dependencies per cell the kernels are built for

// The static part of a stream cell's header (four ints after its values).
struct SweepMeta {
    int n;     // dependencies
    int cell;  // storage cell
    int xid;   // export slot (another range reads this cell's increment), or -1
    int pos2;  // the cell's position in the other direction's stream
};

struct SweepPlan {
    int C = 0, R = 0, W = 0;  // cells, most cells of a range, ranges
    int NE = 0;               // most dependencies of any cell
    int nX = 0;               // exported cells
    int maxHalo = 0;
    std::vector<SweepMeta> meta;   // by position
    std::vector<int> slot;         // [position][NE]: increment's index in the range's LDS array
                                   // (its cells by local position, then the halo at R + item)
    std::vector<int> posOf;        // storage cell -> position
    std::vector<int> rngOff;       // first position of each range (W + 1)
    std::vector<int> haloOff, haloX;   // per range: export slots of its halo, by first level needing them
    std::vector<int> levOff;           // per range: its levels in lev
    std::vector<uint32_t> lev;         // start within the range | halo items needed so far << 16
};

// The work of the compute waves: a level's cells in groups of `cpg`, dealt to
// `nw` waves in turn, as one list per range and wave (wave w of range r:
// [off[nw r + w], off[nw r + w + 1])).
struct SweepGroup {
    uint16_t pos, cnt;     // cells, within the range
    uint16_t start, need;  // cells before the level, halo items it needs
};
struct SweepGroups {
    std::vector<int> off;
    std::vector<SweepGroup> g;
    int max = 0;  // most groups of a range
};
inline SweepGroups sweep_groups(const SweepPlan& P, int cpg, int nw) {
    SweepGroups G;
    G.off.assign(1, 0);
    for (int r = 0; r < P.W; ++r) {
        const int n = P.rngOff[r + 1] - P.rngOff[r], first = (int)G.g.size();
        for (int w = 0; w < nw; ++w) {
            for (int L = P.levOff[r]; L < P.levOff[r + 1]; ++L) {
                const int s = (int)(P.lev[L] & 0xffffu), need = (int)(P.lev[L] >> 16);
                const int e = L + 1 < P.levOff[r + 1] ? (int)(P.lev[L + 1] & 0xffffu) : n;
                for (int p = s + cpg * w; p < e; p += cpg * nw)
                    G.g.push_back({(uint16_t)p, (uint16_t)std::min(cpg, e - p), (uint16_t)s, (uint16_t)need});
            }
            G.off.push_back((int)G.g.size());
        }
        G.max = std::max(G.max, (int)G.g.size() - first);
    }
    return G;
}

// Polls after which a wave's waits over a whole range give up, the guard against a
// fault of the schedule (its order by itself ends every wait).  A wait may
// rightly last as long as the sweep, at worst every range after the one before it:
// 1 us per group and 2 us per range (measured 0.3 to 1 and 2).  A poll is at least an
// LDS round trip of 64 cycles, 25 ns; ten times the polls that fit, and 4 million for
// kernels beside this one.  0: more than a counter holds (a chain of seconds).
inline int sweep_polls(const SweepPlan& P, const SweepGroups& G) {
    const double us = (double)G.g.size() + 2.0 * P.W, n = 10.0 * us / 0.025 + (1 << 22);
    return n < 2e9 ? (int)n : 0;
}

constexpr int SW_RMIN = 64;  // a range takes at least this many cells

// off / nb: faces of each storage cell (CSR) and the neighbour of each (>= C:
// ghost); id: storage cell -> grid id; level: dependency level by storage cell;
// R: most cells of a range; width: cells per level a range may hold.  Returns
// false when a cell has too many dependencies or a halo too many items.
inline bool build_sweep_plan(int C, const std::vector<int>& off, const std::vector<int>& nb, const std::vector<int>& id,
                             const std::vector<int>& level, bool upper, int R, int width, SweepPlan& P) {
    P = SweepPlan();
    P.C = C;
    auto trav = [&](int c) { return upper ? C - 1 - id[c] : id[c]; };
    std::vector<int> cellAt(C);  // traversal index -> storage cell
    for (int c = 0; c < C; ++c) cellAt[trav(c)] = c;
    for (int c = 0; c < C; ++c) {
        const int t = trav(c);
        int n = 0;
        for (int k = off[c]; k < off[c + 1]; ++k)
            if (nb[k] < C && trav(nb[k]) < t) ++n;
        P.NE = std::max(P.NE, n);
    }
    if (P.NE > SW_MAXNE) return false;
    P.NE = std::max(P.NE, 1);
    const int nlev = 1 + *std::max_element(level.begin(), level.end());
    std::vector<int> seen(C, -1), hidx(C, 0), lseen(nlev, -1), ord;
    {
        P.rngOff.assign(1, 0);
        for (int b = 0; b < C;) {
            const int w = (int)P.rngOff.size();
            int e = b, levels = 0;
            while (e < C && e - b < R) {
                if (e - b >= SW_RMIN && e - b >= width * levels) break;
                int& l = lseen[level[cellAt[e++]]];
                if (l != w) { l = w; ++levels; }
            }
            P.rngOff.push_back(b = e);
        }
        const int W = P.W = (int)P.rngOff.size() - 1;
        P.meta.assign(C, SweepMeta{0, 0, -1, 0});
        P.slot.assign((size_t)C * P.NE, 0);
        P.posOf.assign(C, 0);
        P.haloOff.assign(W + 1, 0);
        P.levOff.assign(W + 1, 0);
        ord = cellAt;
        for (int w = 0; w < W; ++w) {
            const int b = P.rngOff[w], e = P.rngOff[w + 1];
            P.R = std::max(P.R, e - b);
            std::sort(ord.begin() + b, ord.begin() + e, [&](int x, int y) {
                return level[x] != level[y] ? level[x] < level[y] : trav(x) < trav(y);
            });
            for (int p = b; p < e; ++p) P.posOf[ord[p]] = p;
        }
        std::vector<int> haloCell;  // storage cells, by halo item over all ranges
        for (int w = 0; w < W; ++w) {
            const int b = P.rngOff[w], e = P.rngOff[w + 1];
            const int h0 = (int)haloCell.size();
            for (int p = b; p < e;) {
                int q = p;  // the level's cells [p, q)
                while (q < e && level[ord[q]] == level[ord[p]]) ++q;
                for (int s = p; s < q; ++s) {
                    const int c = ord[s], t = trav(c);
                    int n = 0;
                    for (int k = off[c]; k < off[c + 1]; ++k) {
                        const int j = nb[k];
                        if (j >= C || trav(j) >= t) continue;
                        int sl;
                        if (trav(j) >= b) sl = P.posOf[j] - b;
                        else {
                            if (seen[j] != w) {
                                seen[j] = w;
                                hidx[j] = (int)haloCell.size() - h0;
                                haloCell.push_back(j);
                            }
                            sl = P.R + hidx[j];
                        }
                        P.slot[(size_t)s * P.NE + n++] = sl;
                    }
                    P.meta[s].n = n;
                    P.meta[s].cell = c;
                }
                const int need = (int)haloCell.size() - h0;
                if (need > 65000) return false;
                P.lev.push_back((uint32_t)(p - b) | (uint32_t)need << 16);
                p = q;
            }
            P.haloOff[w + 1] = (int)haloCell.size();
            P.levOff[w + 1] = (int)P.lev.size();
            P.maxHalo = std::max(P.maxHalo, (int)haloCell.size() - h0);
        }
        P.haloX.resize(haloCell.size());
        for (size_t h = 0; h < haloCell.size(); ++h) {
            SweepMeta& m = P.meta[P.posOf[haloCell[h]]];
            if (m.xid < 0) m.xid = P.nX++;
            P.haloX[h] = m.xid;
        }
    }
    return true;
}

}  // namespace ofx
