// Host check of the pipelined sweep schedule (ofx_sweep.h): on grids of
// several shapes and numberings, in both directions and for several range
// sizes, every cell's dependencies must be found where its slots point
// (its own range: an earlier level; the halo: an item received by its level,
// exported by an earlier range), in face order, and the groups dealt to the
// compute waves must cover each range once.  Then the division by a stored
// reciprocal (ofx_math.h) against the processor's: the same quotient wherever
// div_by_ok holds, dense, sparse and extreme significands, products of the
// divisor and their neighbours among the dividends.  Last the waits' guard:
// on rows numbered back and forth (as many levels as cells, the longest chain a
// grid can have) a wave may poll several times as long as the sweep takes.
// Prints "ok <plans>" or the first failure.
#include "../oneflow_amd/csrc/ofx_sweep.h"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <random>

#define OFX_HD inline
#include "../oneflow_amd/csrc/ofx_math.h"

using namespace ofx;

static int fail(const char* what, int a, int b) { std::printf("%s %d %d\n", what, a, b); return 1; }

int main() {
    std::mt19937 rng(3);
    long plans = 0;
    for (int trial = 0; trial < 160; ++trial) {
        // ni x nj quads (periodic in i for odd trials), some cut into two triangles' worth of extra cells
        const int ni = 2 + (int)(rng() % 90), nj = 1 + (int)(rng() % 60), C = ni * nj;
        std::vector<std::vector<int>> adj(C);
        auto link = [&](int a, int b) { if (a != b) { adj[a].push_back(b); adj[b].push_back(a); } };
        for (int j = 0; j < nj; ++j)
            for (int i = 0; i < ni; ++i) {
                if (i + 1 < ni) link(j * ni + i, j * ni + i + 1);
                else if (trial & 1 && ni > 2) link(j * ni + i, j * ni);
                if (j + 1 < nj && rng() % 50) link(j * ni + i, (j + 1) * ni + i);
            }
        for (auto& a : adj) {
            while (a.size() < 3) a.push_back(C + (int)(rng() % 5));  // ghosts
            std::shuffle(a.begin(), a.end(), rng);
        }
        std::vector<int> off(C + 1, 0), nb, id(C);
        for (int c = 0; c < C; ++c) {
            nb.insert(nb.end(), adj[c].begin(), adj[c].end());
            off[c + 1] = (int)nb.size();
        }
        std::iota(id.begin(), id.end(), 0);  // grid id of each storage cell
        if (trial % 3 == 1) std::shuffle(id.begin(), id.end(), rng);
        if (trial % 3 == 2)  // columns first
            for (int c = 0; c < C; ++c) id[c] = (c % ni) * nj + c / ni;
        std::vector<int> at(C);
        for (int c = 0; c < C; ++c) at[id[c]] = c;
        for (int up = 0; up < 2; ++up) {
            auto trav = [&](int c) { return up ? C - 1 - id[c] : id[c]; };
            std::vector<int> level(C, 0);
            for (int t = 0; t < C; ++t) {
                const int c = at[up ? C - 1 - t : t];
                for (int k = off[c]; k < off[c + 1]; ++k)
                    if (nb[k] < C && trav(nb[k]) < t) level[c] = std::max(level[c], level[nb[k]] + 1);
            }
            const int maxR[] = {64, 256, 2560}, width[] = {4, 16, 1000};
            SweepPlan P;
            const int R = maxR[rng() % 3];
            if (!build_sweep_plan(C, off, nb, id, level, up == 1, R, width[rng() % 3], P)) continue;
            ++plans;
            if (P.R > R || P.rngOff[0] != 0 || P.rngOff[P.W] != C) return fail("size", trial, P.R);
            // the groups of a range cover its cells once, in order within a wave, each inside its level
            const int cpg = 1 + (int)(rng() % 8), nw = 1 + (int)(rng() % 3);
            const SweepGroups G = sweep_groups(P, cpg, nw);
            if ((int)G.off.size() != P.W * nw + 1) return fail("group lists", trial, P.W);
            for (int w = 0; w < P.W; ++w) {
                std::vector<int> hit(P.rngOff[w + 1] - P.rngOff[w], 0);
                if (G.off[nw * w + nw] - G.off[nw * w] > G.max) return fail("group count", trial, w);
                for (int v = 0; v < nw; ++v)
                    for (int k = G.off[nw * w + v], last = -1; k < G.off[nw * w + v + 1]; ++k) {
                        const SweepGroup& x = G.g[k];
                        if (x.cnt < 1 || x.cnt > cpg || (int)x.pos <= last || x.start > x.pos) return fail("group", trial, k);
                        last = x.pos;
                        bool level = false;  // its level starts at `start` and needs `need` halo items
                        for (int L = P.levOff[w]; L < P.levOff[w + 1]; ++L) {
                            const int s = (int)(P.lev[L] & 0xffff);
                            const int e = L + 1 < P.levOff[w + 1] ? (int)(P.lev[L + 1] & 0xffff) : (int)hit.size();
                            level = level || (s == x.start && x.pos + x.cnt <= e && (int)(P.lev[L] >> 16) == x.need);
                        }
                        if (!level) return fail("group level", trial, k);
                        for (int p = x.pos; p < x.pos + x.cnt; ++p) ++hit[p];
                    }
                for (int h : hit)
                    if (h != 1) return fail("group cover", trial, w);
            }
            std::vector<int> cellOfX(P.nX, -1);
            for (int p = 0; p < C; ++p) {
                if (P.posOf[P.meta[p].cell] != p) return fail("position", trial, p);
                if (P.meta[p].xid >= P.nX) return fail("export", trial, p);
                if (P.meta[p].xid >= 0) cellOfX[P.meta[p].xid] = P.meta[p].cell;
            }
            for (int w = 0; w < P.W; ++w) {
                const int b = P.rngOff[w], n = P.rngOff[w + 1] - b;
                if (n < 1 || n > P.R) return fail("range size", trial, w);
                const int nl = P.levOff[w + 1] - P.levOff[w], nh = P.haloOff[w + 1] - P.haloOff[w];
                if (nh > P.maxHalo || nl < 1) return fail("counts", trial, w);
                for (int L = 0; L < nl; ++L) {
                    const uint32_t x = P.lev[P.levOff[w] + L];
                    const int s = (int)(x & 0xffff), need = (int)(x >> 16);
                    const int e = L + 1 < nl ? (int)(P.lev[P.levOff[w] + L + 1] & 0xffff) : n;
                    if ((L == 0 && s != 0) || e <= s || e > n || need > nh) return fail("level", trial, L);
                    for (int p = b + s; p < b + e; ++p) {
                        const int c = P.meta[p].cell, t = trav(c);
                        if (t < b || t >= b + n) return fail("range", trial, p);
                        int m = 0;
                        for (int k = off[c]; k < off[c + 1]; ++k) {
                            if (nb[k] >= C || trav(nb[k]) >= t) continue;
                            const int sl = P.slot[(size_t)p * P.NE + m++];
                            if (sl < P.R) {
                                if (sl >= s || P.meta[b + sl].cell != nb[k]) return fail("own slot", trial, p);
                            } else {
                                const int it = sl - P.R;
                                if (it >= need) return fail("halo need", trial, p);
                                const int y = cellOfX[P.haloX[P.haloOff[w] + it]];
                                if (y != nb[k] || trav(y) >= b) return fail("halo cell", trial, p);
                            }
                        }
                        if (m != P.meta[p].n || m > P.NE) return fail("dependencies", trial, p);
                    }
                }
            }
        }
    }
    std::mt19937_64 g(1);
    auto number = [&](int e) {
        uint64_t m = g();
        switch (g() % 4) {
            case 0: m = g() % 16; break;
            case 1: m = ~(g() % 16); break;
            case 2: m &= 0xffffffff00000000ull; break;
            default: break;
        }
        const uint64_t b = (m & 0xfffffffffffffull) | (uint64_t)(1023 + (int)(g() % (2 * e)) - e) << 52;
        double x;
        std::memcpy(&x, &b, 8);
        return x;
    };
    for (int k = 0; k < 2000000; ++k) {
        const double b = number(299), y = ofxm::div_reciprocal(b), c = number(200) * b;
        const double as[] = {number(599), -number(599), c, std::nextafter(c, 0.0), 0.0, -0.0, number(1000)};
        for (double a : as) {
            if (!ofxm::div_by_ok(a, y)) continue;
            const double q = ofxm::div_by(a, b, y);
            if (q != a / b || std::signbit(q) != std::signbit(a / b)) return fail("quotient", k, 0);
        }
    }
    if (ofxm::div_reciprocal(0.0) != 0.0 || ofxm::div_reciprocal(-1.0) != 0.0 || ofxm::div_reciprocal(1e300) != 0.0 ||
        ofxm::div_reciprocal(NAN) != 0.0 || ofxm::div_by_ok(INFINITY, 1.0) || ofxm::div_by_ok(NAN, 1.0) ||
        ofxm::div_by_ok(1e-200, 1.0) || ofxm::div_by_ok(1.0, 0.0))
        return fail("domain", 0, 0);
    for (int n : {30, 300, 1000, 1700}) {
        const int C = n * n;
        std::vector<int> off(C + 1, 0), nb, id(C), level[2] = {std::vector<int>(C), std::vector<int>(C)};
        for (int c = 0; c < C; ++c) {  // storage cell (i, j)
            const int i = c % n, j = c / n;
            id[c] = j * n + (j & 1 ? n - 1 - i : i);
            if (i > 0) nb.push_back(c - 1);
            if (i + 1 < n) nb.push_back(c + 1);
            if (j > 0) nb.push_back(c - n);
            if (j + 1 < n) nb.push_back(c + n);
            off[c + 1] = (int)nb.size();
            level[0][c] = id[c];
            level[1][c] = C - 1 - id[c];
        }
        for (int up = 0; up < 2; ++up) {
            SweepPlan P;
            if (!build_sweep_plan(C, off, nb, id, level[up], up == 1, 1024, 6, P)) return fail("long chain", n, up);
            for (int cpg : {4, 64}) {  // NS, SA
                const double chain_us = 0.46 * C + 2.0 * P.W;  // measured per level and per range
                const double poll_us = 0.025;                  // one LDS round trip, the least it can be
                const int polls = sweep_polls(P, sweep_groups(P, cpg, cpg == 4 ? 3 : 2));
                if (polls < 8 * chain_us / poll_us) return fail("polls", n, polls);
            }
        }
    }
    {  // more than a counter holds: not swept by the pipeline
        SweepPlan P;
        P.W = 6000000;
        if (sweep_polls(P, SweepGroups()) != 0) return fail("poll limit", 0, 0);
    }
    std::printf("ok %ld\n", plans);
    return 0;
}
