// Launch shapes that depend on a whole batch, planned on the host without a device.
#pragma once
#include <vector>

#include "tasks.hpp"

namespace spand {

// Workgroups of NTHREADS threads that one launch may have: HIP takes fewer than 2^32 work items
// along x (and 65,536 workgroups along y and z, which a batch of pivots exceeds: the level-0
// scaling of a 128^3 grid has 77,949, of a 2048^2 grid 97,539).
constexpr long long launch_blocks_max(int nthreads) { return ((1ll << 32) - 1) / nthreads; }

// One launch of the LU panel kernels over tasks [first, first + count) of a batch sorted by size,
// largest first: blocks = count x per_task workgroups of `threads` threads along x.
struct GetrfLaunch {
    enum Kind { PANEL, TRAIL, SPLIT };
    int kind;
    int kb, nb;      // panel: first column, columns (PANEL, TRAIL)
    int first, count;
    int per_task;    // workgroups per task
    int threads;
};
// The launches that factor pivots of n[0] >= n[1] >= .. rows (n[0] <= GETRF_PANEL_MAX), in order.
std::vector<GetrfLaunch> plan_getrf(const std::vector<int>& n);

// Workgroups of the persistent RRQR launches of one dependency wave: whole clusters in chunks that
// the device holds at once (at most cap slabs), one launch each. Block b of a launch runs on XCD
// b % 8, so a cluster's slabs go to places of one residue, largest clusters first onto the emptiest
// XCD: its slabs then exchange their candidates through that XCD's L2 (the kernel checks where they
// run). A cluster that no XCD holds alone spreads over the device, in a chunk of its kind. No chunk
// at all if some cluster exceeds cap.
struct SlabChunk {
    int first, count;  // workgroups
    int steps;
    bool waits;        // some cluster has several slabs, which wait for each other
};
struct SlabPlan {
    std::vector<RrqrSlab> place;  // by workgroup; big = -1 for a place without a slab
    std::vector<SlabChunk> chunk;
    int spread = 0;               // chunks whose clusters spread over the XCDs
};
// nsub[c], steps[c]: slabs and pivot steps of cluster c
SlabPlan place_slabs(const std::vector<int>& nsub, const std::vector<int>& steps, int cap);

}  // namespace spand
