// Device half of the dense-node solves (hdd_nodeplan.h).
#pragma once
#include <vector>
#include "hdd_nodeplan.h"
#include "hdd_runtime.h"

namespace hdd {

struct NodePlan {
    int n = 0;
    std::vector<NodePlanHost::Level> levels;
    DBuf<NodeItem> fwd, bwd;
    DBuf<int> inst_prob, orig, zidx, more;
    DBuf<NodePos> pos_y, pos_c;
    DBuf<float> tiles, scale;  // the blocks' operators, 256 floats per tile, and their D^-2
    DBuf<float> t, y, z, c;    // padded columns (b less the children's sums, D^-2 y, the result), boundary rows; a zero slot follows z and c
    // false when the batch is outside the form's limits
    bool build(const std::vector<const SupernodalFactor*>& F, const std::vector<int>& offsets, const std::vector<int>& prob_of);
    // x = (A + eps I)^{-1} b; supernodes of problems with active[p] == 0 are skipped (nullptr: none)
    void solve(const float* b, float* x, const int* active, hipStream_t s);
    size_t bytes() const;
};

}  // namespace hdd
