// Static device workspace of the allocation-free apply (scratch.cpp).
#pragma once
#include <cstddef>

namespace spand {

// Size of the static workspace: the apply's segments (Tree::apply_workspace_bytes) must fit,
// e.g. N = 262,144 (64^3, 12 levels, tol 1e-2: 3.45 N doubles a column) with 9 right-hand sides.
constexpr size_t SCRATCH_BYTES = (size_t)64 << 20;

// Device address of the workspace on the current device (looked up on first use per device).
double* scratch_device_ptr();

}  // namespace spand
