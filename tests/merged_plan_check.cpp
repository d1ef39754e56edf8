// Host-side check of the merged solves' plan (BuildMerged, DefaultSlices and
// BuildBlockTiles in psp_amd/csrc/symbolic.cpp) for the grid given on the
// command line:
//   merged_plan_check nx ny nz [precision cutoff minTiles maxSplit slice]
// For every panel class it fills F with numbers on the merged fronts' entries
// and runs the forward and backward passes twice: as the kernels do, from
// tiles, block lists and vector rows (every index checked against its array),
// and front by front from the fine elimination tree, keyed by unknown.  Both
// must agree, on a second pass over the same buffers too.  The fold's lists
// must write every entry of F exactly once and nothing else.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "symbolic.hpp"

using namespace psp_amd;

static int fails = 0;
static void need(bool ok, const char* what, long a = 0, long b = 0)
{
    if (ok) return;
    std::fprintf(stderr, "FAIL %s (%ld, %ld)\n", what, a, b);
    if (++fails > 20) std::exit(1);
}

static double value(int m, int row, int col)
{
    unsigned h = 2654435761u * (unsigned)(m * 1000003 + row * 8191 + col + 1);
    h ^= h >> 15;
    return ((h % 2001) / 1000.0 - 1.0) * 0.05;
}

static void check(const ClassPlan& C)
{
    const int nn = (int)C.nodes.size();
    const VecRows V(C);
    need(!C.bnodes.empty() && !C.groups.empty(), "merged fronts");
    int d = 0;
    for (const auto& g : C.groups) {
        need(g[0] == d && g[1] >= g[0], "groups cover the depths", g[0], g[1]);
        d = g[1] + 1;
    }
    need(d == C.maxDepth + 1, "groups end at the leaves");
    // entries of F by merged front: column of every fine pivot
    std::vector<std::vector<int>> members(C.bnodes.size());
    std::vector<int> mcol(nn, -1);
    for (int t = 0; t < nn; ++t)
        if (C.bnodeOf[t] >= 0) members[C.bnodeOf[t]].push_back(t);
    std::vector<double> F((size_t)C.nblocks * 256, 0.0);
    std::vector<int> writes(F.size(), 0), want(F.size(), 0);
    auto at = [&](int m, int row, int col) -> size_t {
        const BlockNode& b = C.bnodes[m];
        const int r = row >> 4, c = col >> 4;
        need(r >= 0 && r < b.sb + b.ub && c >= C.browLo[b.br0 + r] && c < std::min(b.sb, r + 1),
             "block not stored", row, col);
        return (size_t)(C.browBase[b.br0 + r] + c) * 256 + (col & 15) * 16 + (row & 15);
    };
    struct Entry {
        int row, col;
    };
    std::vector<std::vector<Entry>> entries(C.bnodes.size());
    for (size_t m = 0; m < C.bnodes.size(); ++m) {
        const BlockNode& b = C.bnodes[m];
        int s = 0;
        for (int t : members[m]) {
            mcol[t] = s;
            s += C.nodes[t].size;
        }
        need(s == b.s && b.u == C.nodes[b.top].usize, "front sizes", s, b.s);
        for (int t : members[m])
            for (int j = 0; j < C.nodes[t].size; ++j) {
                const int col = mcol[t] + j;
                for (int i = j; i < C.nodes[t].size; ++i) entries[m].push_back({mcol[t] + i, col});
                for (int a = t; a != b.top;) {
                    a = C.nodes[a].parent;
                    for (int i = 0; i < C.nodes[a].size; ++i) entries[m].push_back({mcol[a] + i, col});
                }
                for (int i = 0; i < b.u; ++i) entries[m].push_back({16 * b.sb + i, col});
            }
        for (const Entry& e : entries[m]) {
            const size_t p = at((int)m, e.row, e.col);
            F[p] = e.row == e.col ? 1.0 : value((int)m, e.row, e.col);
            ++want[p];
        }
    }
    // the fold writes exactly these
    std::map<int, int> frontAt;
    for (size_t m = 0; m < C.bnodes.size(); ++m) frontAt[C.bnodes[m].br0] = (int)m;
    for (const TransItem& it : C.packs) {
        const FoldNode& f = C.foldNodes[it.node];
        const int m = frontAt.at(f.br0);
        need(m == C.bnodeOf[it.node] && f.mcol == mcol[it.node] &&
                 f.x0 == C.bnodes[m].x0 + f.mcol,
             "fold node", it.node);
        for (int j = it.j0; j < std::min(it.j0 + 32, f.s); ++j)
            for (int i = it.i0; i < std::min(it.i0 + 32, it.i0 < f.s ? f.s : f.s + f.u); ++i) {
                if (it.i0 < f.s && i < j) continue;
                ++writes[at(m, i < f.s ? f.mcol + i : f.urow + i - f.s, f.mcol + j)];
            }
    }
    for (const GemmLaunch& gl : C.composeSteps)
        for (int i = gl.tileStart; i < gl.tileStart + gl.tileCount; ++i) {
            const GemmTile& tl = C.composeTiles[i];
            const ComposeDesc& g = C.compose[tl.desc];
            const int m = frontAt.at(g.br0);
            int keys = 0;
            for (int k = 0; k < g.piv; ++k)
                if (C.fsrc.at(g.src + k) >= 0) {
                    const ComposeKey& key = C.fkeys.at(g.kl + keys++);
                    need(key.pos == k && key.col == C.flist[g.list + k] && key.row == C.fsrc[g.src + k],
                         "compose key", i, k);
                }
            need(keys == g.k && tl.pad_ <= g.k, "compose keys", i, keys);
            need(g.list + g.rows <= (int)C.flist.size() && g.src + g.rows <= (int)C.fsrc.size(),
                 "compose lists", i);
            for (int k = 0; k < g.rows; ++k) {
                need(C.fsrc[g.src + k] < g.lde, "compose source row", i, k);
                const int row = C.flist[g.list + k];
                need((row < C.bnodes[m].s) == (k < g.piv), "pivots first", i, k);
                // every entry the product reads is stored
                for (int q = 0; q < g.k; ++q) {
                    const ComposeKey& key = C.fkeys.at(g.kl + q);
                    if (i == gl.tileStart || q == g.k - 1)
                        at(m, row, k >= key.pos ? key.col : row);
                    if (key.pos < std::min(tl.tm + 64, g.rows)) need(q < tl.pad_, "key range", i, q);
                }
            }
            for (int r = tl.tm; r < std::min(tl.tm + 64, g.rows); ++r)
                for (int c = tl.tn; c < std::min(tl.tn + 64, g.n); ++c)
                    ++writes[at(m, C.flist[g.list + r], g.ccol + c)];
        }
    for (size_t i = 0; i < want.size(); ++i) need(writes[i] == want[i], "fold writes", (long)i, writes[i]);

    // both passes, twice (the second over the rows the first left behind)
    std::vector<double> vec(V.total, 0.0), P((size_t)std::max(C.bslots, 1) * 64, 0.0);
    std::vector<double> dinv(C.xrows, 0.0);
    for (int r = 0; r < C.xrows; ++r)
        if (C.sv[r] >= 0) dinv[r] = 0.5 + (r % 7) / 10.0;
    auto row = [&](long r) -> double& {
        need(r >= 0 && r < V.total, "vector row", r);
        return vec[r];
    };
    auto finish = [&](int ph, const BlockTile& t, int r, double v) {
        if (ph == 1) {
            if (r < t.s) row(t.x0 + r) = v;
        } else if (r < t.s) {
            row(V.w + t.x0 + r) = v * dinv[t.x0 + r];
        } else if (r >= 16 * t.sb && r - 16 * t.sb < t.u) {
            const int dst = C.udst.at(t.u0 + r - 16 * t.sb);
            double g = t.leaf ? 0.0 : row(V.g0 + t.u0 + r - 16 * t.sb) + row(V.g1 + t.w0 + r);
            if (dst < C.xrows) g += row(dst);
            row(dst) = g + v;
        }
    };
    auto launch = [&](int g, int ph) {
        const ClassPlan::BlockLevel& L = C.blevels[g];
        std::vector<std::pair<const BlockTile*, std::vector<double>>> done;
        std::map<int, int> arrived, residue;
        std::set<int> slots;
        for (int i = L.start[ph]; i < L.start[ph] + L.count[ph]; ++i) {
            const BlockTile& t = C.btiles.at(i);
            if (t.nob <= 0) {
                need(L.rcount[ph] > 0 && t.slot < 0 && t.red < 0, "hole", i);
                continue;
            }
            need(t.nob <= 4 && t.nib >= 1, "tile shape", t.nob, t.nib);
            std::vector<double> out(64, 0.0);
            for (int q = 0; q < t.nob; ++q)
                for (int j = 0; j < t.nib; ++j) {
                    long blk;
                    if (ph == 0) {
                        const int c = t.ib0 + j;
                        if (c < t.lo[q] || c >= t.hi[q]) continue;
                        blk = (long)t.base[q] + c;
                    } else {
                        blk = C.blist.at(4 * (size_t)(t.lst + t.ib0 + j) + q);
                        if (blk == C.nblocks) continue;  // the block of zeros
                    }
                    need(blk >= 0 && blk < C.nblocks, "block index", blk);
                    for (int a = 0; a < 16; ++a)
                        for (int b = 0; b < 16; ++b) {
                            const double f = F[(size_t)blk * 256 + (ph == 0 ? b * 16 + a : a * 16 + b)];
                            double v;
                            if (ph == 0) {
                                const int col = 16 * (t.ib0 + j) + b;
                                v = row(t.x0 + col);
                                if (!t.leaf) v += row(V.g1 + t.w0 + col);
                            } else {
                                v = row(C.bsrc.at(16 * (size_t)(t.lst + t.ib0 + j) + b));
                            }
                            out[16 * q + a] += f * v;
                        }
                }
            if (t.slot >= 0) {
                need(t.slot < C.bslots && slots.insert(t.slot).second, "slot", t.slot);
                need(t.red >= L.rstart[ph] && t.red < L.rstart[ph] + L.rcount[ph], "reduce item", t.red);
                const BlockRed& rd = C.breds.at(t.red);
                need(rd.ob0 == t.ob0 && rd.nob == t.nob && rd.w0 == t.w0 && rd.x0 == t.x0 &&
                         rd.u0 == t.u0 && rd.s == t.s && rd.u == t.u && rd.sb == t.sb &&
                         rd.leaf == t.leaf && t.slot >= rd.slot0 && t.slot < rd.slot0 + rd.nslots,
                     "reduce record", t.red);
                const int res = (i - L.start[ph]) % 8;
                need(residue.emplace(t.red, res).first->second == res, "slices on two XCDs", t.red);
                for (int e = 0; e < 64; ++e) P[(size_t)t.slot * 64 + e] = out[e];
                if (++arrived[t.red] == rd.nslots) {
                    std::vector<double> sum(64, 0.0);
                    for (int j = 0; j < rd.nslots; ++j)
                        for (int e = 0; e < 64; ++e) sum[e] += P[(size_t)(rd.slot0 + j) * 64 + e];
                    done.push_back({&t, sum});
                }
            } else {
                done.push_back({&t, out});
            }
        }
        need((int)arrived.size() == L.rcount[ph], "split tiles", (long)arrived.size());
        for (const auto& dn : done)  // stores after every read of the launch
            for (int e = 0; e < 16 * dn.first->nob; ++e)
                finish(ph, *dn.first, 16 * dn.first->ob0 + e, dn.second[e]);
    };
    for (int pass = 0; pass < 2; ++pass) {
        std::vector<double> b(C.n), y(C.n), x(C.n);
        for (int q = 0; q < C.n; ++q) b[q] = std::sin(1.0 + 0.37 * q + pass);
        std::vector<int> xrow(C.n, -1);
        for (size_t m = 0; m < C.bnodes.size(); ++m)
            for (int t : members[m])
                for (int j = 0; j < C.nodes[t].size; ++j) {
                    const int q = C.nodes[t].off + j, r = C.bnodes[m].x0 + mcol[t] + j;
                    xrow[q] = r;
                    need(C.sv.at(r) == C.qv[q] && C.sxy.at(r) == C.qxy[q], "solve order", q);
                }
        int real = 0;
        for (int r = 0; r < C.xrows; ++r) real += C.sv[r] >= 0;
        need(real == C.n, "padding rows", real, C.n);
        for (int q = 0; q < C.n; ++q) row(xrow[q]) = b[q];
        const int ng = (int)C.groups.size();
        for (int g = ng - 1; g >= 0; --g) launch(g, 0);
        for (int g = 0; g < ng; ++g) launch(g, 1);
        // front by front
        std::vector<std::map<int, double>> up(C.bnodes.size());  // contributions by unknown
        for (int g = ng - 1; g >= 0; --g)
            for (size_t m = 0; m < C.bnodes.size(); ++m) {
                const BlockNode& bn = C.bnodes[m];
                if (bn.group != g) continue;
                const Node& t = C.nodes[bn.top];
                std::map<int, double> in;  // children's contributions
                for (size_t c = 0; c < C.bnodes.size(); ++c)
                    if (C.bnodes[c].parent == (int)m)
                        for (const auto& kv : up[c]) in[kv.first] += kv.second;
                std::vector<double> gt(bn.s), o(16 * (bn.sb + bn.ub), 0.0);
                std::vector<int> unk(bn.s);
                for (int f : members[m])
                    for (int j = 0; j < C.nodes[f].size; ++j) {
                        const int q = C.nodes[f].off + j;
                        unk[mcol[f] + j] = q;
                        gt[mcol[f] + j] = b[q] + (in.count(q) ? in[q] : 0.0);
                        in.erase(q);
                    }
                for (const Entry& e : entries[m]) o[e.row] += F[at((int)m, e.row, e.col)] * gt[e.col];
                for (int j = 0; j < bn.s; ++j) y[unk[j]] = o[j] * dinv[bn.x0 + j];
                for (int i = 0; i < bn.u; ++i) {
                    const int q = C.structs[t.ustart + i];
                    up[m][q] = o[16 * bn.sb + i] + (in.count(q) ? in[q] : 0.0);
                    in.erase(q);
                }
                need(in.empty(), "contribution without a row", (long)m);
            }
        for (int g = 0; g < ng; ++g)
            for (size_t m = 0; m < C.bnodes.size(); ++m) {
                const BlockNode& bn = C.bnodes[m];
                if (bn.group != g) continue;
                const Node& t = C.nodes[bn.top];
                std::vector<int> unk(bn.s);
                for (int f : members[m])
                    for (int j = 0; j < C.nodes[f].size; ++j) unk[mcol[f] + j] = C.nodes[f].off + j;
                std::vector<double> o(bn.s, 0.0);
                for (const Entry& e : entries[m])
                    o[e.col] += F[at((int)m, e.row, e.col)] *
                                (e.row < bn.s ? y[unk[e.row]] : x[C.structs[t.ustart + e.row - 16 * bn.sb]]);
                for (int j = 0; j < bn.s; ++j) x[unk[j]] = o[j];
            }
        double err = 0, nrm = 0;
        for (int q = 0; q < C.n; ++q) {
            err = std::max(err, std::fabs(x[q] - row(xrow[q])));
            nrm = std::max(nrm, std::fabs(x[q]));
        }
        // sums of at most a few thousand terms in another order
        need(err <= 1e-11 * nrm && nrm > 0, "passes differ", pass, (long)(err / nrm * 1e15));
    }
    std::printf("class %d: %zu groups, %zu merged fronts of %d nodes, %d blocks, %d slots\n", C.cls,
                C.groups.size(), C.bnodes.size(), nn, C.nblocks, C.bslots);
}

int main(int argc, char** argv)
{
    if (argc < 4) return 2;
    psp_hip_desc d{};
    d.nx = std::atoi(argv[1]);
    d.ny = std::atoi(argv[2]);
    d.nz = std::atoi(argv[3]);
    const double h = 1.0 / (std::max(d.nx, std::max(d.ny, d.nz)) + 1);
    d.wx = (d.nx + 1) * h;
    d.wy = (d.ny + 1) * h;
    d.wz = (d.nz + 1) * h;
    d.omega = 30.0;
    d.bx = d.by = d.bz = 5;
    d.sigmax = d.sigmay = d.sigmaz = 1.5;
    d.damping = 7.0;
    d.planesPerPanel = 4;
    d.precision = argc > 4 ? std::atoi(argv[4]) : 0;
    d.cutoff = argc > 5 ? std::atoi(argv[5]) : 12;
    Plan plan;
    if (argc > 6) plan.minTiles = std::atoi(argv[6]);
    if (argc > 7) plan.maxSplit = std::atoi(argv[7]);
    std::string msg;
    if (BuildPlan(d, plan, msg) != PSP_HIP_OK) {
        std::fprintf(stderr, "plan: %s\n", msg.c_str());
        return 2;
    }
    for (int c = 0; c < 3; ++c) {
        if (!plan.present[c]) continue;
        ClassPlan& C = plan.cls[c];
        if (argc > 8) {
            for (auto& s : C.slices) s = {std::atoi(argv[8]), std::atoi(argv[8])};
            BuildBlockTiles(C);
        }
        check(C);
    }
    return fails ? 1 : 0;
}
