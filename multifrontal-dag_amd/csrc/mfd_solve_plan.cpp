// Builds the solves' task list; see mfd_solve_plan.h.
//
// Task order (the order of tickets): the forward sweep level by level from
// the leaves' level up, the backward sweep from the roots' level down.  Per
// level, forward: superblock by superblock the pivot rows of every front,
// then the update rows.  Backward: the partial sums over the update rows,
// then superblock by superblock, last first, the pivot columns.
#include "mfd_solve_plan.h"

#include <algorithm>
#include <array>
#include <climits>
#include <cstdio>

#include "mfdag.h"

namespace mfd {

namespace {

// A front of one superblock whose update rows its own workgroup takes as
// well (no hand-over to other workgroups): with at most kWholeRows of them,
// where a hand-over (about 3 us) costs more than the rows do (solves of a
// 37 x 29 x 23 grid, 33 right-hand sides, and of a 250^2 grid with fronts of
// its own columns only: 547 and 1619 us; with 64 rows 588 and 1619, with 256
// 542 and 1728); on a level of at least kManyFronts fronts, which fill the chip
// by themselves, at most kWholeMany (512 systems 3.82 ms, 3.85 with 128).
constexpr int kWholeRows = 128, kWholeMany = 256;
constexpr int kManyFronts = 512;
// Rows per forward task: 16, four waves a quarter of the columns each, until
// a level has more than kManyRows tasks of them; then 64 (48^3 solves 747 us
// from 2048 tasks on, 729 from 1024, 714 from 512, 729 from 256; 64^3 with four
// right-hand sides 1.570 ms, 1.556, 1.551, 1.550; with 16 rows throughout 800
// and 1.765).
constexpr int kManyRows = 512;
// A level's tasks of one phase beyond kManyTasks are taken several to a
// ticket, at most kTicketMost (every ticket is an addition to one counter):
// 512 systems 3.82 ms, 3.86 with one each.
constexpr int kManyTasks = 4096, kTicketMost = 8;
constexpr int kFlagLine = 32;  // super fronts keep their counters up to a cache line apart: many workgroups poll each

}  // namespace

int build_solve_plan(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<int>& level_ptr,
                     const std::vector<int>& level_nodes, int super_min, SolvePlan& P)
{
    P = SolvePlan{};
    const int m = (int)nodes.size(), levels = (int)level_ptr.size() - 1;
    auto super = [&](int s) { return super_min > 0 && nodes[s].c >= super_min; };
    auto nsup = [&](int s) { return (nodes[s].c + kSuper - 1) / kSuper; };
    auto width = [&](int s, int u) { return std::min(kSuper, nodes[s].c - kSuper * u); };
    std::vector<int> part_rows(m, kSuper);  // update rows of a kBwdPart task
    auto chunks = [&](int s) { return (nodes[s].w + part_rows[s] - 1) / part_rows[s]; };

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

    // Planes: a front's update rows (and the pivot rows that tasks pass on,
    // those of superblock first_kept and later ones) in the forward sweep, its
    // partial sums in the backward one.  The partial sums of a tree take the
    // place of that tree's rows: its backward sweep starts when its forward
    // sweep has ended.  Those of a front's children, written when the front's
    // x is complete, take the place of its own.
    std::vector<int> root(m);
    for (int s = m - 1; s >= 0; --s) root[s] = nodes[s].parent < 0 ? s : root[nodes[s].parent];
    std::vector<int64_t> rows(m, 0), base(m, 0), most(m, 0);  // per root
    std::vector<int64_t> z(m), slots(m), slot0(m, 0);
    auto first_kept = [&](int s) { return super(s) ? 2 : 1; };
    for (int s = 0; s < m; ++s) {
        const int from = std::min(kSuper * first_kept(s), nodes[s].c);  // the first row kept
        z[s] = rows[root[s]] - from;
        rows[root[s]] += nodes[s].n - from;
        most[root[s]] += nodes[s].w + nodes[s].c * 3LL / 4;
    }
    // A tree whose partial sums would take more than its rows do, and than its
    // update rows and three quarters of an entry per unknown (few, large
    // fronts), forms them over more rows at a time: with y, b and x a solve
    // then takes at most the update rows and four vectors, however the fronts
    // are shaped.
    for (bool again = true; again;) {
        again = false;
        std::vector<int64_t> below(m, 0);
        for (int s = 0; s < m; ++s) {  // of the subtree: its own, or its children's
            const int64_t own = !whole[s] && nodes[s].w > 0 ? (int64_t)64 * ((nodes[s].c + 63) / 64) * chunks(s) : 0;
            slots[s] = std::max(own, below[s]);
            if (nodes[s].parent >= 0) below[nodes[s].parent] += slots[s];
        }
        for (int s = m - 1; s >= 0; --s) {  // roots before their fronts
            const int r = root[s];
            if (slots[r] <= std::max(rows[r], most[r]) || part_rows[s] >= nodes[s].w) continue;
            part_rows[s] *= 2;
            again = true;
        }
    }
    for (int s = 0; s < m; ++s)
        if (root[s] == s) {
            base[s] = P.plane;
            P.plane += std::max(rows[s], slots[s]);
        }
    for (int s = m - 1; s >= 0; --s) {  // parents before children
        int64_t at = slot0[s];
        for (int ch : S.children[s]) {
            slot0[ch - 1] = at;
            at += slots[ch - 1];
        }
    }
    int64_t glen = 0, grows = (int64_t)S.l_rows.size();
    for (int s = 0; s < m; ++s)
        if (!S.children[s].empty()) glen += nodes[s].n;
    // counters: asm, and z, y, p, t and x of every superblock, or (fstr 0) one
    // for all of a front of one superblock that is no super front, whose
    // phases follow one another: asm, y, p, x.  Six words of memory each (two
    // and four for fronts of one and two columns, so that counters never take
    // more than an entry per unknown): a word each, 32 fronts polled and raised
    // in one cache line, makes a solve 2 to 4% slower.
    std::vector<int> flag(m), fstr(m);
    int64_t nflags = 0;
    for (int s = 0; s < m; ++s) {
        const int c = nodes[s].c;
        fstr[s] = super(s) ? std::max(1, std::min(kFlagLine, c / 3)) : nsup(s) == 1 ? 0 : 1;
        flag[s] = (int)nflags;
        nflags += fstr[s] == 0 ? std::min(6, 2 * c) : (int64_t)fstr[s] * (1 + 5 * nsup(s));
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
    std::vector<int> arrivals(m, 0);  // signals to each front's asm counter
    auto before_y = [&](int s) { return fstr[s] == 0 ? arrivals[s] : 0; };
    auto parts = [&](int s, int u) { return whole[s] || nodes[s].w == 0 ? 0 : (width(s, u) + 31) / 32 * chunks(s); };
    auto yx_count = [&](int s, int u) { return super(s) ? (width(s, u) + 15) / 16 : 1; };
    auto y_target = [&](int s, int u) { return before_y(s) + yx_count(s, u); };
    auto p_target = [&](int s, int u) { return (fstr[s] == 0 ? y_target(s, u) : 0) + parts(s, u); };
    auto x_target = [&](int s, int u) { return (fstr[s] == 0 ? p_target(s, u) : 0) + yx_count(s, u); };
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
                const int w = width(s, u);
                int zt = 0;
                if (u >= first_kept(s))
                    zt = add_rows(s, kSuper * u, kSuper * u + w, super(s) ? u - 1 : u, u, counter(s, 0, u));
                for (int r = 0; r < (super(s) ? w : 1); r += 16) {
                    SolveTask t = task(s, super(s) ? kFwdTop : kFwdPiv, u);
                    t.r0 = r;
                    if (u >= first_kept(s))
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
                    t.r0 = nodes[s].c + part_rows[s] * q;
                    t.nr = std::min(part_rows[s], nodes[s].n - t.r0);
                    t.slot = (int)(base[root[s]] + slot0[s]) + 64 * (c0 / 64 * chunks(s) + q) + c0 % 64;
                    t.nslot = c0;
                    t.sig = counter(s, 2, c0 / kSuper);
                    if (pa >= 0) wait(t, counter(pa, 4, 0), x_target(pa, 0));
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
                        wait(t, counter(s, 2, u), p_target(s, u));
                    else
                        wait(t, counter(s, 1, u), y_target(s, u));
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
                        wait(t, counter(pa, 4, 0), x_target(pa, 0));
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
    auto counter = [](const SolveTask& t, int q, int u) { return t.flag + t.fstr * (1 + q * t.nsup + u); };
    auto count = [](const SolveTask& t, int u) { return t.super ? (std::min(kSuper, t.c - kSuper * u) + 15) / 16 : 1; };
    // the counters a task raises, as its kernel function does; which of its
    // phases a shared counter (fstr 0) is in: 0 asm, 1 y, 2 p, 3 x
    auto raise = [&](const SolveTask& t, auto&& f) {
        if (t.kind == kFwdTop || t.kind == kFwdPiv) f(counter(t, 1, t.u), 1);
        if (t.kind == kBwdTop || t.kind == kBwdPiv) f(counter(t, 4, t.u), 3);
        if (t.kind != kFwdTop && t.kind != kBwdTop && t.kind != kBwdPiv && t.sig >= 0)
            f(t.sig, t.kind == kBwdPart ? 2 : 0);
    };
    int64_t bad = 0;
    char line[160];
    auto fault = [&](size_t i, const char* what, int f, int now, int want) {
        if (++bad > 8) return;
        snprintf(line, sizeof line, "solve task %zu (kind %d, superblock %d): %s, counter %d at %d, wants %d\n", i,
                 P.tasks[i].kind, P.tasks[i].u, what, f, now, want);
        report += line;
    };
    // signals of each counter up to the end of each phase (separate counters
    // have one phase, whatever its number)
    std::vector<int> now(P.nflags, 0);
    std::vector<std::array<int, 4>> upto(P.nflags, std::array<int, 4>{0, 0, 0, 0});
    std::vector<char> shared(P.nflags, 0);
    for (const SolveTask& t : P.tasks)
        if (t.fstr == 0) shared[t.flag] = 1;
    for (const SolveTask& t : P.tasks)
        raise(t, [&](int f, int ph) {
            for (int q = shared[f] ? ph : 0; q < 4; ++q) upto[f][q]++;
        });
    for (size_t i = 0; i < P.tasks.size(); ++i) {
        const SolveTask& t = P.tasks[i];
        auto need = [&](int f, int want) {
            if (f < 0) return;
            const auto& e = upto[f];
            if (now[f] < want)
                fault(i, "waits for later tasks", f, now[f], want);
            else if (std::find(e.begin(), e.end(), want) == e.end())
                fault(i, "waits for part of a phase", f, now[f], want);
        };
        need(t.w0, t.w0t);
        const int y0 = t.fstr == 0 ? t.w0t : 0;  // as fwd_rows and fwd_rows64 wait
        if (t.kind == kFwdRows || t.kind == kFwdRows64)
            for (int v = 0; v < t.nslot; ++v) need(counter(t, 1, v), y0 + count(t, v));
        if (t.kind == kFwdTop && t.u > 0) need(counter(t, 1, t.u - 1), count(t, t.u - 1));
        if (t.kind == kBwdCols)
            for (int v = t.nsup - 1; v >= t.grow; --v) need(counter(t, 4, v), count(t, v));
        if (t.kind == kBwdTop && t.u + 1 < t.nsup) need(counter(t, 4, t.u + 1), count(t, t.u + 1));
        raise(t, [&](int f, int ph) {
            // a shared counter's phase starts when the one before has ended: y
            // after a wait for asm; p, and x without partial sums, after one
            // for the parent's x, which follows this front's y; x after one
            // for p, or, in a root, for y
            if (shared[f] && ph > 0) {
                if (now[f] < upto[f][ph - 1]) fault(i, "raises a phase early", f, now[f], upto[f][ph - 1]);
                const int after = upto[f][ph - 1];
                const bool own = t.w0 == f && t.w0t == after, none = after == 0;
                const bool parent = t.w0 >= 0 && t.w0 != f && (ph == 2 || upto[f][2] == upto[f][1]);
                if (!own && !(ph == 1 && none) && !(ph >= 2 && parent)) fault(i, "raises a phase unordered", f, now[f], after);
            }
            now[f]++;
        });
    }
    return bad;
}

}  // namespace mfd
