// How many workgroups of the chain-following kernels may be resident together
// (host arithmetic; rb_fused.hip).
#pragma once

#include <algorithm>

namespace rb {

// other live plans whose ordinary launches may run beside a cooperative one
constexpr int kSmallStreams = 3;

// the largest grid (waves) of a plan that is launched beside others
inline int small_grid(int ncu) { return std::max(1, ncu / 8); }

// Workgroups of which per_cu fit a compute unit that are resident together
// whatever of the others' grids is there already: every workgroup of theirs
// may hold a compute unit to itself (k_staged takes 97 of its 160 KB of LDS and
// leaves room for one k_fused of 33 KB instead of four).
inline int resident_slots(int per_cu, int ncu, int others) {
    return per_cu * std::max(1, ncu - others * small_grid(ncu));
}

}  // namespace rb
