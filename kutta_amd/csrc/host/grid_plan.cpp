#include "grid_plan.hpp"

#include <algorithm>

namespace kutta_amd {
namespace {

constexpr Index kChunk = 4;      // rows are padded to whole chunks of this many slots
constexpr int kMaxLevels = 16;
// How a level's rows are summed (kh_grid_part::mode). Where a member's rows
// leave at least half of its 16 wavefronts idle, all lanes form the terms
// first: above that the rows fill the workgroup and the second pass over the
// entries costs more than the shorter serial part saves.
constexpr Index kTermsRows = 512;

Index share_begin(Index rows, int part, int parts) {
  return Index(std::int64_t(rows) * part / parts);
}

std::size_t round4(std::size_t words) { return (words + 3) / 4 * 4; }

}  // namespace

bool plan_grid(const std::vector<const CsrHost*>& patterns, int parts, GridPlan& plan) {
  plan = GridPlan();
  const int count = int(patterns.size());
  if (count < 1 || count > kMaxLevels || parts < 1 || parts > KH_GRID_MAX_PARTS) return false;
  int grid = count;
  while (grid > 1 && patterns[grid - 1]->n_rows <= KH_GRID_BOTTOM_ROWS) --grid;
  // The coarsest level's few-row form runs only in the first workgroup alone.
  if (grid == count && patterns.back()->n_rows <= 24) return false;
  plan.parts = parts;
  plan.count = count;
  plan.grid = grid;
  plan.levels.resize(std::size_t(count));
  plan.table.resize(std::size_t(count) * parts);
  std::size_t terms = 0, window = 0;
  for (int k = 0; k < count; ++k) {
    const CsrHost& a = *patterns[k];
    GridLevelPlan& l = plan.levels[k];
    l.place.resize(std::size_t(a.n_rows));
    const int owners = k < grid ? parts : 1;
    Index most = 0, most_rows = 0;
    for (int p = 0; p < parts; ++p) {
      kh_grid_part& g = plan.table[std::size_t(p) * count + k];
      g = kh_grid_part{};
      if (p >= owners) continue;
      const Index first = share_begin(a.n_rows, p, owners), last = share_begin(a.n_rows, p + 1, owners);
      g.first = first;
      g.rows = last - first;
      g.slot0 = Index(l.slot.size());
      if (g.rows == 0) continue;
      Index lo = first, hi = last;
      for (Index j = a.row_ptr[first]; j < a.row_ptr[last]; ++j) {
        lo = std::min(lo, a.col[j]);
        hi = std::max(hi, a.col[j] + 1);
      }
      if (hi - lo >= 0xffff) return false;
      g.window = lo;
      g.window_rows = hi - lo;
      if (k < grid) window = std::max(window, std::size_t(hi - lo));
      for (Index i = first; i < last; ++i) {
        const Index length = a.row_ptr[i + 1] - a.row_ptr[i], chunks = (length + kChunk - 1) / kChunk;
        const std::size_t base = l.slot.size();
        if (length < 1 || base - std::size_t(g.slot0) > 0xffff) return false;
        l.place[i] = std::uint16_t(base - std::size_t(g.slot0));
        l.slot.resize(base + std::size_t(KH_GRID_CHUNKS(chunks)) * kChunk, -1);
        l.local_col.resize(l.slot.size(), 0xffff);
        for (Index j = 0; j < length; ++j) {
          l.slot[base + j] = a.row_ptr[i] + j;
          l.local_col[base + j] = std::uint16_t(a.col[a.row_ptr[i] + j] - lo);
        }
      }
      g.slots = Index(l.slot.size()) - g.slot0;
      if (g.slots > KH_GRID_POOL_WORDS) return false;
      most = std::max(most, Index(g.slots));
      most_rows = std::max(most_rows, Index(g.rows));
    }
    const int mode = most_rows > kTermsRows ? 0 : 1;
    for (int p = 0; p < parts; ++p) plan.table[std::size_t(p) * count + k].mode = mode;
    terms = std::max(terms, std::size_t(2 * mode) * std::size_t(most));
  }
  window = round4(window);
  const std::size_t shared = round4(window + terms);
  std::size_t words = 0;
  for (int p = 0; p < parts; ++p) {
    std::size_t at = shared;
    for (int k = 0; k < count; ++k) {
      kh_grid_part& g = plan.table[std::size_t(p) * count + k];
      g.terms = std::int32_t(window);
      g.lds = std::int32_t(at);
      if (g.rows == 0) continue;
      // values, columns (16 bits), weights and right-hand sides, places and lengths (16 bits each)
      at += round4(std::size_t(g.slots) + std::size_t(g.slots) / 2 + 3 * std::size_t(g.rows));
    }
    // The levels of the first workgroup keep their two iterates each at the end.
    if (p == 0 && grid < count) {
      plan.table[std::size_t(grid)].iterates = std::int32_t(at);
      at += std::size_t(2 * KH_GRID_BOTTOM_ROWS) * std::size_t(count - grid);
    }
    words = std::max(words, at);
  }
  if (words > KH_GRID_POOL_WORDS) return false;
  plan.lds_words = int(std::max<std::size_t>(words, 1));
  return true;
}

}  // namespace kutta_amd
