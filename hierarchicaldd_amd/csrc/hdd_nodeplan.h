// Dense-node form of the exact solves x = (A + eps I)^{-1} b of a batch of
// supernodal factors (SIGMA_SMOOTHER::Smooth and Compute_Residual,
// IFS/SIGMA_SMOOTHER.cpp:292-352, which the reference hands to PARDISO).
//
// The elimination trees have 5-16 heights of small supernodes, and a launch per
// height and pass leaves the GPU waiting on latency. Here the heights are cut
// into a few bands; every connected piece of a tree inside a band is one node,
// held as one dense block: with L the factor's columns of the node (its n
// columns' rows, then its nr boundary rows),
//   forward   [y; u] = [I + S; W] t,  S = D Linv - I, Linv = L11^{-1}, D = diag(L11), W = L21 Linv
//             t = b - sum of the children's u at the node's columns,
//             u += the children's u at the node's boundary rows
//   backward  z = [I + S^T | -W^T] [D^-2 y; z of the boundary rows]
// A closed node (no boundary rows: the root of a tree) holds its inverse, z = Linv^T Linv t, in
// place of the triangle and its transpose (the same number of elements in one launch instead of
// two; a launch of a few us is most of a small solve) and has no backward pass, unless the block
// is nearly singular (constant_share in hdd_nodeplan.cpp), when it keeps the two passes with a
// boundary tile of zeros. So a pass is one
// launch per band (level), less the last band's backward, and one more forward for the
// children's sums where there are any. Blocks are formed in double on the
// device at set-up and held in float, as the per-height plan holds its own. With
// D taken out, the triangle's diagonal is exactly one: it is not stored, and
// the largest term of a row is added once, after the sum of the others, so that
// neither loses to the other's rounding (emulated on the 96^3 level-0 interface:
// rms error of a solve 1.1e-7 with the diagonal inside the sums, 5.9e-8 outside).
//
// Nodes with bit-identical factor columns (subdomains of one shape, interface
// faces that are translates of each other) share a block; up to kRun of them
// are the columns of one matrix product, done with 16x16x4 FP32 MFMA tiles.
#pragma once
#include <vector>
#include "hdd_factor.h"

namespace hdd {

// One workgroup's work: row tiles [rt0, rt1) of a run of `cnt` nodes that share a block.
struct alignas(16) NodeItem {
    int tile;            // first tile of the block's operator for this pass (forward of a closed block: its inverse)
    int inst0;           // the run: instances [inst0, inst0 + cnt)
    int y0, c0;          // first column and boundary row of the first; the others follow, nk and nrk tiles each
    int cnt, split;      // split: waves that share a row tile
    int nk, nrk;         // column and boundary tiles of the block
    int rt0, rt1;
    int one;             // the block has runs of one node only: vector sums instead of matrix products
    int scale;           // first of the block's D^-2 (closed: of its inverse's diagonal)
};

struct NodePos {  // child contributions of one row: positions in c (the zero slot when there is none);
    int p0, p1;   // p1 < 0: ~p1 is the row's list in `more` (count, then positions beyond p0)
};

struct NodePlanHost {
    static constexpr int kTile = 16;         // rows and columns of an operator tile (1 KiB)
    static constexpr int kRun = 16;          // nodes per run at most (columns of an MFMA tile)
    static constexpr int kMaxLdsFloats = 36000;  // one node's operand vector (n + nr rows)
    static constexpr int kRunLdsFloats = 12288;  // operand vectors of a run of several nodes
    static constexpr size_t kSetupChunk = size_t(24) << 20;  // doubles of blocks set up together, unless one needs more
    struct Block {
        const SupernodalFactor* f = nullptr;
        std::vector<int> sns;                // its supernodes, ascending; the last is the node's root
        int n = 0, nr = 0, nk = 0, nrk = 0;
        int fwd = 0, bwd = 0;                // first tile of the forward and backward operator (closed: of its inverse)
        int scale = 0;                       // first of its 16 nk entries of D^-2 (closed: of its inverse's diagonal)
    };
    struct Level {
        int fwd0 = 0, fwd1 = 0, bwd0 = 0, bwd1 = 0;  // items
        int fwd_waves = 4, bwd_waves = 4;            // waves per workgroup
        int fwd_lds = 0, bwd_lds = 0;                // floats of the operand vectors
        int y0 = 0, y1 = 0, c0 = 0, c1 = 0;          // its padded columns and boundary rows
        bool children = false;
    };
    int n = 0;                    // rows of the batch
    int ysize = 0, csize = 0;     // padded columns and boundary rows of all nodes
    long long tiles = 0;
    int scales = 0;
    std::vector<Block> blocks;
    std::vector<Level> levels;
    std::vector<NodeItem> fwd, bwd;
    std::vector<int> inst_prob;   // problem of each instance
    std::vector<int> orig;        // padded column -> row of the batch (-1: padding)
    std::vector<int> zidx;        // padded boundary row -> padded column (ysize: the zero slot)
    std::vector<NodePos> pos_y, pos_c;  // child contributions of each padded column and boundary row
    std::vector<int> more;
};

// Plans the nodes of a batch of factors (offsets: first row of each; prob_of: problem of each, empty: all 0).
// False when the batch is outside the form's limits (a separator whose vectors exceed the LDS, index ranges).
bool build_nodeplan(const std::vector<const SupernodalFactor*>& F, const std::vector<int>& offsets, const std::vector<int>& prob_of,
                    NodePlanHost& P);

// Row of a block's padded columns (16 nk + 16 nrk of them: L11, then L21) that each sub-diagonal row of
// its supernodes falls on, supernode after supernode.
void node_block_rows(const NodePlanHost::Block& B, std::vector<int>& rows);

// Factor columns of a block, row-major, (16 nk + 16 nrk) x 16 nk doubles: L11 (padding: identity), then L21.
void node_block_columns(const NodePlanHost::Block& B, double* L);

// Device bytes of the plan that build_nodeplan makes of these factors (repeats included: subdomains of one
// shape): what it holds, and what its set-up needs beside it while it runs. Not planned: the batch is
// outside the form's limits.
struct PlanBytes { double held = 0, setup = 0; bool planned = false; };
PlanBytes nodeplan_bytes(const std::vector<const SupernodalFactor*>& F);

}  // namespace hdd
