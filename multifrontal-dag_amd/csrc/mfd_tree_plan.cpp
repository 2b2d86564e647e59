// Builds the bottom-of-the-tree launch; see mfd_tree_plan.h.
#include "mfd_tree_plan.h"

#include <algorithm>
#include <climits>
#include <cstdio>

namespace mfd {

namespace {
// Fronts of one height beyond kManyTasks are taken several to a ticket, at
// most kTicketMost (every ticket is an addition to one counter; 512 systems
// 9.13 ms, 9.15 with one each, 9.11 with 16).
constexpr int kManyTasks = 8192, kTicketMost = 4;

// Microseconds of a factorization (FP64) whose eligible fronts of order <=
// `order` are in the launch, the others in the level schedule, as far as the
// choice of `order` changes it.  In the launch a front takes 3 us per panel of
// 16 pivot columns and 0.06 us per row, 0.0625 per row and panel, and waits
// only for its children; a level takes 10 us and 0.1 per row for fronts of
// order <= 64, 12 us, 0.28 per column of a block and 17 per further block for
// larger ones, whatever their number, and 8 us for every child outside the
// launch that one of its fronts has beyond the first (a launch per rank);
// where fronts are many, one costs 0.012 us and its time over 800 in the
// launch, 0.02 us and 7.5e-6 n^2 outside it.  Fitted to forests of 1 to 1024
// chains of equal fronts of order 16 to 128 (errors up to 30%).
double predicted_us(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<char>& eligible, int order)
{
    const int m = (int)nodes.size();
    std::vector<char> in(m, 0);
    std::vector<int> depth(m, 0);
    std::vector<double> path(m, 0.0), small, large;
    std::vector<int> ranks;
    double longest = 0.0, many = 0.0;
    bool any = false;
    for (int s = 0; s < m; ++s) {  // children before parents
        const double n = nodes[s].n, panels = (nodes[s].c + 15) / 16, us = 0.06 * n + panels * (3.0 + 0.0625 * n);
        in[s] = eligible[s] && nodes[s].n <= order;
        for (int ch : S.children[s]) {
            in[s] = in[s] && in[ch - 1];
            path[s] = std::max(path[s], path[ch - 1]);
        }
        if (in[s]) {
            any = true;
            path[s] += us;
            longest = std::max(longest, path[s]);
        }
        many += in[s] ? 0.012 + us / 800.0 : 0.02 + 7.5e-6 * n * n;
    }
    for (int s = m - 1; s >= 0; --s) {  // parents before children
        const int pa = nodes[s].parent, n = nodes[s].n, c = nodes[s].c;
        if (pa >= 0) depth[s] = depth[pa] + 1;
        if (in[s]) continue;
        auto& level = n <= kTile ? small : large;
        if ((int)level.size() <= depth[s]) level.resize(depth[s] + 1, 0.0);
        const double us = n <= kTile ? 10.0 + 0.1 * n : 12.0 + 0.28 * std::min(c, kPanel) + 17.0 * ((c - 1) / kPanel);
        level[depth[s]] = std::max(level[depth[s]], us);
        int outside = 0;
        for (int ch : S.children[s]) outside += !in[ch - 1];
        if ((int)ranks.size() <= depth[s]) ranks.resize(depth[s] + 1, 1);
        ranks[depth[s]] = std::max(ranks[depth[s]], outside);
    }
    double t = (any ? 10.0 + longest : 0.0) + many;
    for (int r : ranks) t += 8.0 * (r - 1);
    for (double us : small) t += us;
    for (double us : large) t += us;
    return t;
}

// The largest order of the launch's fronts: kTreeFront, unless the launch is
// predicted to lose clearly by it.  It wins where the tree branches (512
// systems of a batch: 9.1 ms against 11.4 in either other way; a 100^2 grid
// 0.48 against 0.53 with fronts of order <= 64 only, 0.76 without it), and
// loses where a few fronts follow one another, of which it takes one at a time
// by one workgroup: 64 x 64 blocks in a chain of 12 took 699 us in it and 387
// in the level schedule, 60 x 60 blocks by themselves 55 and 34.  The bound of
// 0.85 keeps every tree that branches where it measured faster; a forest
// without branches, where the prediction is good to a few percent, needs less
// of a margin.
int largest_order(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<char>& eligible)
{
    bool branches = false;
    for (const auto& ch : S.children) branches = branches || ch.size() > 1;
    double best = predicted_us(S, nodes, eligible, kTreeFront) * (branches ? 0.85 : 0.9);
    int order = kTreeFront;
    for (int o : {kTile, 0}) {
        const double us = predicted_us(S, nodes, eligible, o);
        if (us < best) best = us, order = o;
    }
    return order;
}
}  // namespace

void build_tree_plan(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<char>& eligible,
                     TreePlan& P)
{
    P = TreePlan{};
    const int m = (int)nodes.size();
    if (S.snidx.size() > (size_t)INT_MAX) return;  // entry indices are 32-bit here
    std::vector<char> in(m, 0);
    std::vector<int> height(m, 0);
    int count = 0;
    const int order = largest_order(S, nodes, eligible);
    for (int s = 0; s < m; ++s) {  // children before parents
        in[s] = eligible[s] && nodes[s].n <= order;
        for (int ch : S.children[s]) {
            in[s] = in[s] && in[ch - 1];
            height[s] = std::max(height[s], height[ch - 1] + 1);
        }
        count += in[s];
    }
    if (count == 0) return;
    P.in = in;
    P.node.reserve(count);
    for (int s = 0; s < m; ++s)
        if (in[s]) P.node.push_back(s);
    // by height; the largest of a height first, so that the last to start are short
    std::stable_sort(P.node.begin(), P.node.end(), [&](int a, int b) {
        return height[a] != height[b] ? height[a] < height[b] : nodes[a].n > nodes[b].n;
    });
    std::vector<int> pos(m, -1);
    for (int i = 0; i < count; ++i) pos[P.node[i]] = i;
    P.tasks.resize(count);
    int64_t entries = 0, panels = 0;
    for (int s : P.node) {
        const int c0 = nodes[s].first, c1 = c0 + nodes[s].c;
        entries += S.a_colptr[c1] - S.a_colptr[c0];
        panels += (nodes[s].c + 15) / 16 + 1;
    }
    P.apos.reserve(entries);
    P.asrc.reserve(entries);
    P.arc.reserve(entries);
    P.aptr.reserve(panels);
    for (int s = 0; s < m; ++s) {  // (the lists in the order of the nodes, as the structure has them)
        if (!in[s]) continue;
        const int i = pos[s];
        const NodeDev& d = nodes[s];
        TreeTask t{};
        t.front = d.front;
        t.inv = d.inv;
        t.n = d.n;
        t.c = d.c;
        t.first = d.first;
        t.child = (int)P.children.size();
        t.nchild = (int)S.children[s].size();
        t.aptr = (int)P.aptr.size();
        t.flag = i;
        t.sig = d.parent >= 0 && in[d.parent] ? pos[d.parent] : -1;
        for (int ch : S.children[s]) {
            const NodeDev& k = nodes[ch - 1];
            P.children.push_back(TreeChild{k.front + k.c + (int64_t)k.c * k.n, k.n, k.w, (int)k.lidx, 0});
        }
        for (int q = 0; q < d.c; ++q) {
            if (q % 16 == 0) P.aptr.push_back((int)P.asrc.size());
            const int j = d.first + q;  // 0-based global column
            for (int64_t p = S.a_colptr[j]; p < S.a_colptr[j + 1]; ++p) {
                if (!assembled(S, p)) continue;
                const int r = S.snidx[p];
                const int grow = r <= d.c ? d.first + r - 1 : S.l_rows[S.l_ptr[s] + (r - d.c - 1)] - 1;
                P.apos.push_back((r - 1) | (q % 16) << 8);
                P.asrc.push_back((int)(S.ccs_perm[p] - 1));
                P.arc.push_back(TreePlan::RowCol{grow, j});
            }
        }
        P.aptr.push_back((int)P.asrc.size());
        P.tasks[i] = t;
    }
    P.entries = (int64_t)P.asrc.size();
    for (int i = 0; i < count;) {
        int e = i;
        while (e < count && height[P.node[e]] == height[P.node[i]]) ++e;
        const int per = e - i > kManyTasks ? std::min(kTicketMost, (e - i) / (kManyTasks / 2)) : 1;
        for (; i < e; ++i) P.tasks[i].per = per;
    }
}

int64_t check_tree_plan(const TreePlan& P, std::string& report)
{
    std::vector<int> now(P.tasks.size(), 0), total(P.tasks.size(), 0);
    for (const TreeTask& t : P.tasks)
        if (t.sig >= 0) total[t.sig]++;
    int64_t bad = 0;
    char line[128];
    for (size_t i = 0; i < P.tasks.size(); ++i) {
        const TreeTask& t = P.tasks[i];
        if (now[t.flag] != t.nchild || total[t.flag] != t.nchild || t.flag != (int)i)
            if (++bad <= 8) {
                snprintf(line, sizeof line, "tree task %zu: %d of %d children before it, %d in all\n", i, now[t.flag],
                         t.nchild, total[t.flag]);
                report += line;
            }
        if (t.sig >= 0) now[t.sig]++;
    }
    return bad;
}

}  // namespace mfd
