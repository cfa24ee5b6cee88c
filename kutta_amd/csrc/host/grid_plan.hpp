// How the multi-workgroup V-cycle (KH_GRID_CYCLE) splits a hierarchy: which
// levels its workgroups share, which the first of them runs alone, and the
// tables they read. Host only.
#pragma once

#include <cstdint>
#include <vector>

#include "amg_setup.hpp"
#include "kutta_hip.h"

namespace kutta_amd {

// The padded layout of one shared level (see kh_grid_level).
struct GridLevelPlan {
  std::vector<std::uint16_t> place, local_col;
  std::vector<Index> slot;
};

struct GridPlan {
  int parts = 0, count = 0, grid = 0;  // workgroups, levels, shared levels
  int lds_words = 0;
  std::vector<GridLevelPlan> levels;
  std::vector<kh_grid_part> table;  // parts x count
};

// Plans levels patterns[0..] (the first is where the launch starts) over
// `parts` workgroups. The levels of at most KH_GRID_BOTTOM_ROWS rows at the
// end belong to the first workgroup. Returns false where the plan does not
// fit: a member's share of all its levels, the launch's widest window and the
// terms of its largest level that forms them must lie in KH_GRID_POOL_WORDS
// words of LDS, with the first member's bottom levels and their iterates.
bool plan_grid(const std::vector<const CsrHost*>& patterns, int parts, GridPlan& plan);

}  // namespace kutta_amd
