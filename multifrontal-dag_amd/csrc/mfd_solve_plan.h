// The solves' task list (mfd_solve.hip): what each workgroup's turn does,
// what it waits for, and where the vectors passed between tasks lie.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

#include "mfd_analysis.h"
#include "mfd_plan.h"

namespace mfd {

struct SolvePlan {
    std::vector<SolveTask> tasks;
    int fwd_tasks = 0;          // those of the forward sweep (the first ones)
    // children's update rows that add into each front row: plane positions
    // of the first and the second (-1: none), or -2 - k: the second and the
    // others at gsrc[k] (their number, then their positions)
    struct Gather {
        int s0, s1;
    };
    std::vector<Gather> gat;
    std::vector<int> gsrc;
    std::vector<int> grow;  // global row (0-based) of every update row
    // the superblock matrices: X's columns (up to nx), then the blocks of W and V
    std::vector<SuperInvTask> xinv;
    int nx = 0;
    int64_t sinv_elems = 0;
    int64_t plane = 0;  // entries per right-hand side of the plane array
    int nflags = 0;     // counters per group of right-hand sides
};

// levels: node ids per level, lowest first (level_ptr / level_nodes);
// children always lie below their parents.  Fronts with at least super_min
// pivot columns (0: none) are super fronts.  Returns 0 or MFD_ERR_NOMEM (an
// index would not fit 32 bits).
int build_solve_plan(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<int>& level_ptr,
                     const std::vector<int>& level_nodes, int super_min, SolvePlan& P);

// Number of waits that the tasks before the waiting one would not satisfy
// (each would hang the launch), or whose count differs from the signals its
// counter gets in all (the wait would end early); report receives the first
// few.
int64_t check_solve_plan(const SolvePlan& P, std::string& report);

}  // namespace mfd
