// How the workgroups of a KH_GRID_CYCLE launch find out which of them work:
// the steps of one thread of each, on a control block `Ctl`. They are constexpr
// templates, which kernels and host code may both call: the host runs them on a
// model of the block, in every order the workgroups' steps can take
// (tests/grid_gather_model.cpp).
//
// Each access of `Ctl` has taken effect before it returns. With grid the number
// of workgroups in the launch:
//   arrive(v)  adds v to the arrivals, returns what they were: the number of
//              workgroups started (16 bits) and of ranks taken (16 bits)
//   arrivals() the same without adding
//   settle(to) state 0 -> to; returns the state before
//   state()    0 gathering, 1 all have started, 2 one works alone
//   leave()    adds one to the workgroups done, returns how many were before
//   clear()    all of it back to zero
//   wait(), expired()  starts the time limit, and whether it has passed
#pragma once

#include <cstdint>

namespace kh {

enum class GridRole { Leave, Member, Solo };
struct GridPlace {
  GridRole role;
  int rank;
};
constexpr unsigned kGridStarted = 1u, kGridRank = 1u << 16;

// A workgroup comes in; `here`: it is on the home XCD and takes a rank. Exactly
// `parts` workgroups of the launch end as members, or one works alone.
template <class Ctl>
constexpr GridPlace grid_enter(Ctl& c, unsigned grid, int parts, bool here) {
  const unsigned old = c.arrive(here ? kGridStarted + kGridRank : kGridStarted);
  const int rank = int(old >> 16);
  const bool last = (old & 0xffff) + 1 == grid;
  if (!here) {
    // The last to start speaks for all; if no workgroup is on the home XCD it
    // works alone.
    if (last) c.settle(rank == 0 ? 2 : 1);
    return {last && rank == 0 ? GridRole::Solo : GridRole::Leave, 0};
  }
  if (last) c.settle(1);
  c.wait();
  unsigned state = c.state();
  while (state == 0) {
    if (c.expired() && c.settle(2) == 0) return {GridRole::Solo, rank};
    state = c.state();
  }
  if (state == 1) {
    if (int(c.arrivals() >> 16) == parts) return {GridRole::Member, rank};
    if (rank == 0) return {GridRole::Solo, 0};
  }
  return {GridRole::Leave, 0};
}
// Every workgroup leaves, its part done; the last clears the block for the next
// launch. Until it has left no workgroup settles the state any more, so none
// can settle a cleared one.
template <class Ctl>
constexpr void grid_leave(Ctl& c, unsigned grid) {
  if (c.leave() + 1 == grid) c.clear();
}

}  // namespace kh
