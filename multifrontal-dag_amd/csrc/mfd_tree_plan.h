// The fronts that one launch assembles and factors at the bottom of the tree
// (mfd_tree.hip): which they are, in which order, and their entries of A.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

#include "mfd_analysis.h"
#include "mfd_plan.h"

namespace mfd {

struct TreePlan {
    std::vector<char> in;  // per node: 1 = in this plan (empty: none is)
    std::vector<int> node;  // node of each task
    std::vector<TreeTask> tasks;  // in ticket order
    std::vector<TreeChild> children;
    std::vector<int> apos, asrc, aptr;
    struct RowCol {
        int row, col;
    };
    std::vector<RowCol> arc;
    int64_t entries = 0;  // entries of A of these fronts
    bool has(int s) const { return !in.empty() && in[s]; }
};

// eligible: per node, whether the front may be in the plan; it is if all its
// children are and its order is at most kTreeFront, or less where the launch
// would lose by the larger ones (none: the plan is empty).
void build_tree_plan(const Structure& S, const std::vector<NodeDev>& nodes, const std::vector<char>& eligible,
                     TreePlan& P);

// Number of tasks whose children do not all come before them in ticket order
// or do not all raise their counter (their waits would hang the launch or
// end early); report receives the first few.
int64_t check_tree_plan(const TreePlan& P, std::string& report);

}  // namespace mfd
