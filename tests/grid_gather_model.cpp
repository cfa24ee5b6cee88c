// Runs the gathering of a KH_GRID_CYCLE launch (kh_grid_gather.hpp) on a model
// of its control block in every order its workgroups' accesses can take, and
// checks that exactly `parts` members work together or one workgroup alone,
// that no wait is without end, and that the block is clear for the next launch.
//   grid_gather_model PARTS HOME AWAY EXPIRES
// HOME and AWAY: workgroups on and off the home XCD. EXPIRES 0: the time limit
// never passes, so only the workgroups' own steps may end a wait.
#include <algorithm>
#include <array>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "kh_grid_gather.hpp"

namespace {

enum class Op { Arrive, Arrivals, Settle, State, Leave, Expired, Clear, BarrierAdd, BarrierWait, Done };
enum Word { Arrived, Left, Settled, Bar, kWords };
using Shared = std::array<unsigned, kWords>;

// A workgroup is the results of its accesses so far: replaying them leads to
// the next one, which is thrown.
struct Next {
  Op op;
  unsigned arg;
};
struct Replay {
  const std::vector<unsigned>& log;
  std::size_t at = 0;
  unsigned next(Op op, unsigned arg = 0) {
    if (at == log.size()) throw Next{op, arg};
    return log[at++];
  }
  unsigned arrive(unsigned v) { return next(Op::Arrive, v); }
  unsigned arrivals() { return next(Op::Arrivals); }
  unsigned settle(unsigned to) { return next(Op::Settle, to); }
  unsigned state() { return next(Op::State); }
  unsigned leave() { return next(Op::Leave); }
  void wait() {}
  bool expired() { return next(Op::Expired) != 0; }
  void clear() {
    for (unsigned w = 0; w < kWords; ++w) next(Op::Clear, w);
  }
};

struct Group {
  bool here;
  std::vector<unsigned> log;
  bool operator<(const Group& o) const { return here != o.here ? here < o.here : log < o.log; }
  bool operator==(const Group& o) const { return here == o.here && log == o.log; }
};
struct Model {
  int parts;
  unsigned grid;
  bool expires;
  std::set<std::pair<Shared, std::vector<Group>>> seen;
  long ends = 0, members = 0, alone = 0;

  Next step(const Group& g, kh::GridPlace* place) const {
    Replay c{g.log};
    try {
      const kh::GridPlace p = kh::grid_enter(c, grid, parts, g.here);
      if (place) *place = p;
      if (p.role == kh::GridRole::Member) {  // one barrier over the members
        c.next(Op::BarrierAdd);
        c.next(Op::BarrierWait);
      }
      kh::grid_leave(c, grid);
    } catch (const Next& n) {
      return n;
    }
    return {Op::Done, 0};
  }
  [[noreturn]] void fail(const char* what, const Shared& s) const {
    std::printf("%s: arrived %x left %u state %u bar %u\n", what, s[Arrived], s[Left], s[Settled], s[Bar]);
    std::exit(1);
  }
  void run(const Shared& s, const std::vector<Group>& groups) {
    auto key = groups;  // workgroups alike are interchangeable
    std::sort(key.begin(), key.end());
    if (!seen.insert({s, key}).second) return;
    bool moved = false, all = true;
    for (std::size_t k = 0; k < key.size(); ++k) {
      if (k > 0 && key[k] == key[k - 1]) continue;
      const Next n = step(key[k], nullptr);
      if (n.op == Op::Done) continue;
      all = false;
      Shared t = s;
      std::vector<unsigned> results;
      switch (n.op) {
        case Op::Arrive: results = {s[Arrived]}; t[Arrived] += n.arg; break;
        case Op::Arrivals: results = {s[Arrived]}; break;
        case Op::Settle: results = {s[Settled]}; if (s[Settled] == 0) t[Settled] = n.arg; break;
        case Op::State:
          // Still gathering and the limit not passed: the same wait again.
          if (s[Settled] != 0) results = {s[Settled]};
          else if (expires) results = {0, 1};
          else continue;
          break;
        case Op::Leave: results = {s[Left]}; t[Left] += 1; break;
        case Op::Clear: results = {0}; t[n.arg] = 0; break;
        case Op::BarrierAdd: results = {0}; t[Bar] += 1; break;
        case Op::BarrierWait:
          if (s[Bar] < unsigned(parts)) continue;
          results = {0};
          break;
        default: fail("a step out of place", s);
      }
      moved = true;
      auto next = key;
      next[k].log.insert(next[k].log.end(), results.begin(), results.end());
      run(t, next);
    }
    if (!all) {
      if (!moved) fail("a wait without end", s);
      return;
    }
    long together = 0, solo = 0;
    for (const Group& g : key) {
      kh::GridPlace p{};
      step(g, &p);
      together += p.role == kh::GridRole::Member;
      solo += p.role == kh::GridRole::Solo;
    }
    if (!(together == parts && solo == 0) && !(together == 0 && solo == 1)) fail("not one cycle", s);
    if (s != Shared{}) fail("not clear for the next launch", s);
    ++ends;
    members += together > 0;
    alone += solo;
  }
};

}  // namespace

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int parts = std::atoi(argv[1]), home = std::atoi(argv[2]), away = std::atoi(argv[3]);
  Model m{parts, unsigned(home + away), std::atoi(argv[4]) != 0, {}};
  std::vector<Group> groups;
  for (int k = 0; k < home + away; ++k) groups.push_back({k < home, {}});
  m.run(Shared{}, groups);
  std::printf("%zu states, %ld ends: %ld together, %ld alone\n", m.seen.size(), m.ends, m.members, m.alone);
  return 0;
}
