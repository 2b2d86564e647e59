// Builds the solves' task list; see mfd_solve_plan.h.
//
// Task order (the order of tickets): the forward sweep level by level from
// the leaves' level up, the backward sweep from the roots' level down.  Per
// level, forward: superblock by superblock the pivot rows of every front,
// then the update rows.  Backward: the partial sums over the update rows,
// then superblock by superblock, last first, the pivot columns.
#include "mfd_solve_plan.h"

#include <algorithm>
#include <climits>
#include <cstdio>

#include "mfdag.h"

namespace mfd {

namespace {

// A front of one superblock whose update rows its own workgroup takes as
// well (no hand-over to other workgroups): with at most kWholeRows of them,
// where a hand-over (about 3 us) costs more than the rows do; on a level of
// at least kManyFronts fronts, which fill the chip by themselves, at most
// kWholeMany.
constexpr int kWholeRows = 128, kWholeMany = 256;
constexpr int kManyFronts = 512;
// Rows per forward task: 16, four waves a quarter of the columns each, until
// a level has more than kManyRows tasks of them; then 64.
constexpr int kManyRows = 2048;
// A level's tasks of one phase beyond kManyTasks are taken several to a
// ticket, at most kTicketMost (every ticket is an addition to one counter).
constexpr int kManyTasks = 4096, kTicketMost = 8;
constexpr int kFlagLine = 32;  // super fronts keep their counters a cache line apart: many workgroups poll each

}  // namespace

int build_solve_plan(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<int>& level_ptr,
                     const std::vector<int>& level_nodes, int super_min, SolvePlan& P)
{
    P = SolvePlan{};
    const int m = (int)nodes.size(), levels = (int)level_ptr.size() - 1;
    auto super = [&](int s) { return super_min > 0 && nodes[s].c >= super_min; };
    auto nsup = [&](int s) { return (nodes[s].c + kSuper - 1) / kSuper; };
    auto width = [&](int s, int u) { return std::min(kSuper, nodes[s].c - kSuper * u); };
    auto chunks = [&](int s) { return (nodes[s].w + kSuper - 1) / kSuper; };

    // superblock matrices
    std::vector<int64_t> xoff(m, -1);
    for (int s = 0; s < m; ++s)
        if (super(s)) {
            xoff[s] = P.sinv_elems;
            P.sinv_elems += nsup(s) * kSuperMats;
        }
    for (int wv = 0; wv < 2; ++wv) {
        if (wv) P.nx = (int)P.xinv.size();
        for (int s = 0; s < m; ++s) {
            if (xoff[s] < 0) continue;
            const int c = nodes[s].c;
            for (int u = 0; u * kSuper < c; ++u) {
                const int64_t xo = xoff[s] + u * kSuperMats;
                if (!wv) {
                    for (int j = 0; j < kSuper / 16; ++j) P.xinv.push_back(SuperInvTask{s, u, 0, j, xo});
                    continue;
                }
                for (int i = 0; u > 0 && i < 4; ++i)
                    for (int j = 0; j < 4; ++j) P.xinv.push_back(SuperInvTask{s, u, i, 4 + j, xo});
                for (int i = 0; (u + 1) * kSuper < c && i < 4; ++i)
                    for (int j = 0; j < 4; ++j) P.xinv.push_back(SuperInvTask{s, u, i, 8 + j, xo});
            }
        }
    }

    // whole[s]: the front's update rows go with its pivot block
    std::vector<char> whole(m, 0);
    for (int L = 0; L < levels; ++L) {
        const bool many = level_ptr[L + 1] - level_ptr[L] >= kManyFronts;
        for (int k = level_ptr[L]; k < level_ptr[L + 1]; ++k) {
            const int s = level_nodes[k];
            whole[s] = !super(s) && nsup(s) == 1 && nodes[s].w > 0 && nodes[s].w <= (many ? kWholeMany : kWholeRows);
        }
    }

    // Planes: a front's update rows (with its pivot rows, where tasks pass
    // them on) in the forward sweep, its partial sums in the backward one.
    // The partial sums of a tree take the place of that tree's rows: its
    // backward sweep starts when its forward sweep has ended.
    std::vector<int> root(m);
    for (int s = m - 1; s >= 0; --s) root[s] = nodes[s].parent < 0 ? s : root[nodes[s].parent];
    std::vector<int64_t> rows(m, 0), slots(m, 0), base(m, 0);  // per root
    std::vector<int64_t> z(m), slot0(m);
    for (int s = 0; s < m; ++s) {
        const bool keep = nsup(s) > (super(s) ? 2 : 1);
        z[s] = rows[root[s]] - (keep ? 0 : nodes[s].c);
        rows[root[s]] += keep ? nodes[s].n : nodes[s].w;
        slot0[s] = slots[root[s]];
        if (!whole[s] && nodes[s].w > 0) slots[root[s]] += (int64_t)64 * ((nodes[s].c + 63) / 64) * chunks(s);
    }
    for (int s = 0; s < m; ++s)
        if (root[s] == s) {
            base[s] = P.plane;
            P.plane += std::max(rows[s], slots[s]);
        }
    int64_t glen = 0, grows = (int64_t)S.l_rows.size();
    for (int s = 0; s < m; ++s)
        if (!S.children[s].empty()) glen += nodes[s].n;
    // counters
    std::vector<int> flag(m), fstr(m);
    int64_t nflags = 0;
    for (int s = 0; s < m; ++s) {
        fstr[s] = super(s) ? kFlagLine : 1;
        flag[s] = (int)nflags;
        nflags += (int64_t)fstr[s] * (1 + 5 * nsup(s));
        if (nflags > INT_MAX / 2) return MFD_ERR_NOMEM;
    }
    if (P.plane > INT_MAX || glen > INT_MAX || grows > INT_MAX) return MFD_ERR_NOMEM;
    P.nflags = (int)nflags;
    P.grow.resize(grows);
    for (int64_t k = 0; k < grows; ++k) P.grow[k] = S.l_rows[k] - 1;
    // gather tables, children in child order
    std::vector<int> goff(m, -1);
    P.gat.reserve(glen);
    std::vector<int> more;
    for (int s = 0; s < m; ++s) {
        if (S.children[s].empty()) continue;
        goff[s] = (int)P.gat.size();
        const int n = nodes[s].n;
        P.gat.resize(P.gat.size() + n, SolvePlan::Gather{-1, -1});
        SolvePlan::Gather* g = P.gat.data() + goff[s];
        auto each = [&](auto&& f) {
            for (int ch : S.children[s]) {
                const NodeDev& d = nodes[ch - 1];
                for (int k = 0; k < d.w; ++k)
                    f(S.lidx[d.lidx + k] - 1, (int)(base[root[s]] + z[ch - 1] + d.c + k));
            }
        };
        more.assign(n, 0);
        int most = 0;
        each([&](int i, int at) {
            most = std::max(most, ++more[i]);
            (more[i] == 1 ? g[i].s0 : g[i].s1) = at;  // a third and later ones replace it below
        });
        if (most <= 2) continue;
        for (int i = 0; i < n; ++i)
            if (more[i] > 2) {
                g[i].s1 = -2 - (int)P.gsrc.size();
                P.gsrc.resize(P.gsrc.size() + more[i], 0);
            }
        more.assign(n, 0);
        each([&](int i, int at) {
            if (++more[i] >= 2 && g[i].s1 < -1) {
                int* list = &P.gsrc[-2 - g[i].s1];
                list[++list[0]] = at;
            }
        });
    }

    // counter of front s: kind q (0 z, 1 y, 2 p, 3 t, 4 x) of superblock u
    auto asm_flag = [&](int s) { return flag[s]; };
    auto counter = [&](int s, int q, int u) { return flag[s] + fstr[s] * (1 + q * nsup(s) + u); };
    auto yx_target = [&](int s, int u) { return super(s) ? (width(s, u) + 15) / 16 : 1; };
    std::vector<int> arrivals(m, 0);  // signals to each front's asm counter
    auto task = [&](int s, int kind, int u) {
        const NodeDev& d = nodes[s];
        SolveTask t{};
        t.front = d.front;
        t.n = d.n;
        t.c = d.c;
        t.first = d.first;
        t.z = (int)(base[root[s]] + z[s]);
        t.kind = kind;
        t.u = u;
        t.goff = goff[s];
        t.grow = (int)d.lidx;
        t.w0 = t.sig = -1;
        t.flag = flag[s];
        t.fstr = fstr[s];
        t.nsup = nsup(s);
        t.super = super(s) ? 1 : 0;
        t.aux = super(s) ? xoff[s] + (int64_t)u * kSuperMats : d.inv + (int64_t)u * (kSuper / 64) * 4096;
        t.slot = (int)(base[root[s]] + slot0[s]) + 64 * chunks(s) * (kSuper / 64) * u;
        return t;
    };
    auto wait = [](SolveTask& t, int f, int target) {
        t.w0 = target > 0 ? f : -1;
        t.w0t = target;
    };
    size_t seg = 0;
    auto close = [&]() {  // ends a phase of a level
        const int cnt = (int)(P.tasks.size() - seg);
        const int per = cnt > kManyTasks ? std::min(kTicketMost, cnt / (kManyTasks / 2)) : 1;
        for (; seg < P.tasks.size(); ++seg) P.tasks[seg].per = per;
    };

    for (int L = 0; L < levels; ++L) {
        const int b0 = level_ptr[L], b1 = level_ptr[L + 1];
        int steps = 0;
        int64_t nrows = 0;
        for (int k = b0; k < b1; ++k) {
            const int s = level_nodes[k];
            steps = std::max(steps, nsup(s));
            if (!whole[s]) nrows += nodes[s].w;
        }
        const int R = nrows > (int64_t)16 * kManyRows ? 64 : 16;
        // rows [r0, r1) of front s with superblocks v < nv applied
        auto add_rows = [&](int s, int r0, int r1, int nv, int u, int sig) {
            int cnt = 0;
            for (int r = r0; r < r1; r += R, ++cnt) {
                SolveTask t = task(s, R == 64 ? kFwdRows64 : kFwdRows, u);
                t.r0 = r;
                t.nr = std::min(R, r1 - r);
                t.nslot = nv;
                t.sig = sig;
                wait(t, asm_flag(s), arrivals[s]);
                P.tasks.push_back(t);
            }
            return cnt;
        };
        for (int u = 0; u < steps; ++u) {
            for (int k = b0; k < b1; ++k) {
                const int s = level_nodes[k];
                if (u >= nsup(s)) continue;
                const int w = width(s, u), first_kept = super(s) ? 2 : 1;
                int zt = 0;
                if (u >= first_kept)
                    zt = add_rows(s, kSuper * u, kSuper * u + w, super(s) ? u - 1 : u, u, counter(s, 0, u));
                for (int r = 0; r < (super(s) ? w : 1); r += 16) {
                    SolveTask t = task(s, super(s) ? kFwdTop : kFwdPiv, u);
                    t.r0 = r;
                    if (u >= first_kept)
                        wait(t, counter(s, 0, u), zt);
                    else
                        wait(t, asm_flag(s), arrivals[s]);
                    if (whole[s]) {
                        t.nr = nodes[s].w;
                        if (nodes[s].parent >= 0) {
                            t.sig = asm_flag(nodes[s].parent);
                            arrivals[nodes[s].parent]++;
                        }
                    }
                    P.tasks.push_back(t);
                }
            }
            close();
        }
        for (int k = b0; k < b1; ++k) {
            const int s = level_nodes[k], pa = nodes[s].parent;
            if (whole[s] || nodes[s].w == 0) continue;
            const int cnt = add_rows(s, nodes[s].c, nodes[s].n, nsup(s), 0, pa >= 0 ? asm_flag(pa) : -1);
            if (pa >= 0) arrivals[pa] += cnt;
        }
        close();
    }
    P.fwd_tasks = (int)P.tasks.size();
    for (int L = levels - 1; L >= 0; --L) {
        const int b0 = level_ptr[L], b1 = level_ptr[L + 1];
        int steps = 0;
        for (int k = b0; k < b1; ++k) {
            const int s = level_nodes[k], pa = nodes[s].parent;
            steps = std::max(steps, nsup(s));
            if (whole[s] || nodes[s].w == 0) continue;
            for (int c0 = 0; c0 < nodes[s].c; c0 += 32)
                for (int q = 0; q < chunks(s); ++q) {
                    SolveTask t = task(s, kBwdPart, c0 / kSuper);
                    t.r0 = nodes[s].c + kSuper * q;
                    t.nr = std::min(kSuper, nodes[s].n - t.r0);
                    t.slot = (int)(base[root[s]] + slot0[s]) + 64 * (c0 / 64 * chunks(s) + q) + c0 % 64;
                    t.nslot = c0;
                    t.sig = counter(s, 2, c0 / kSuper);
                    if (pa >= 0) wait(t, counter(pa, 4, 0), yx_target(pa, 0));
                    P.tasks.push_back(t);
                }
        }
        close();
        for (int u = steps - 1; u >= 0; --u) {
            for (int k = b0; k < b1; ++k) {
                const int s = level_nodes[k], pa = nodes[s].parent;
                if (u >= nsup(s)) continue;
                const int w = width(s, u), vlo = u + (super(s) ? 2 : 1);
                const int nslot = whole[s] ? 0 : chunks(s);  // 0 without update rows
                // what y_u waits for: the partial sums, or, with no update
                // rows, its own forward tasks
                auto wait_y = [&](SolveTask& t) {
                    if (nslot > 0)
                        wait(t, counter(s, 2, u), (w + 31) / 32 * nslot);
                    else
                        wait(t, counter(s, 1, u), yx_target(s, u));
                    t.nslot = nslot;
                };
                const bool cols = vlo < nsup(s);
                for (int r = 0; cols && r < w; r += 16) {
                    SolveTask t = task(s, kBwdCols, u);
                    t.r0 = r;
                    t.nr = std::min(16, w - r);
                    t.grow = vlo;
                    t.sig = counter(s, 3, u);
                    wait_y(t);
                    P.tasks.push_back(t);
                }
                for (int r = 0; r < (super(s) ? w : 1); r += 16) {
                    SolveTask t = task(s, super(s) ? kBwdTop : kBwdPiv, u);
                    t.r0 = r;
                    if (cols) {
                        wait(t, counter(s, 3, u), (w + 15) / 16);
                    } else if (whole[s] && pa >= 0) {
                        t.nr = nodes[s].w;
                        wait(t, counter(pa, 4, 0), yx_target(pa, 0));
                    } else {
                        wait_y(t);
                    }
                    P.tasks.push_back(t);
                }
            }
            close();
        }
    }
    if (P.tasks.size() > (size_t)INT_MAX) return MFD_ERR_NOMEM;
    return MFD_OK;
}

int64_t check_solve_plan(const SolvePlan& P, std::string& report)
{
    std::vector<int> now(P.nflags, 0), total(P.nflags, 0);
    auto counter = [](const SolveTask& t, int q, int u) { return t.flag + t.fstr * (1 + q * t.nsup + u); };
    auto target = [](const SolveTask& t, int u) { return t.super ? (std::min(kSuper, t.c - kSuper * u) + 15) / 16 : 1; };
    // the counters a task raises, as its kernel function does
    auto raise = [&](const SolveTask& t, std::vector<int>& f) {
        if (t.kind == kFwdTop || t.kind == kFwdPiv) f[counter(t, 1, t.u)]++;
        if (t.kind == kBwdTop || t.kind == kBwdPiv) f[counter(t, 4, t.u)]++;
        if (t.kind != kFwdTop && t.kind != kBwdTop && t.kind != kBwdPiv && t.sig >= 0) f[t.sig]++;
    };
    for (const SolveTask& t : P.tasks) raise(t, total);
    int64_t bad = 0;
    char line[160];
    for (size_t i = 0; i < P.tasks.size(); ++i) {
        const SolveTask& t = P.tasks[i];
        auto need = [&](int f, int want) {
            if (f < 0 || (now[f] >= want && total[f] == want)) return;
            if (++bad <= 8) {
                snprintf(line, sizeof line, "solve task %zu (kind %d, superblock %d): counter %d at %d of %d, wants %d\n", i,
                         t.kind, t.u, f, now[f], total[f], want);
                report += line;
            }
        };
        need(t.w0, t.w0t);
        if (t.kind == kFwdRows || t.kind == kFwdRows64)
            for (int v = 0; v < t.nslot; ++v) need(counter(t, 1, v), target(t, v));
        if (t.kind == kFwdTop && t.u > 0) need(counter(t, 1, t.u - 1), target(t, t.u - 1));
        if (t.kind == kBwdCols)
            for (int v = t.nsup - 1; v >= t.grow; --v) need(counter(t, 4, v), target(t, v));
        if (t.kind == kBwdTop && t.u + 1 < t.nsup) need(counter(t, 4, t.u + 1), target(t, t.u + 1));
        raise(t, now);
    }
    return bad;
}

}  // namespace mfd
