// Host orchestration of the device Krylov solvers and the aggregation-AMG
// V-cycle (linalg/solver.cpp:75-393, linalg/amg.cpp:176-342), expressed as
// kernel launches through the kutta_hip C ABI.
//
// The MI355X path fuses the reference's launch sequence where the fused kernel
// computes the identical floats: spmv+dot+alpha, step+dot+check, residual+
// restriction, prolongation+first post-sweep, and the last fine sweep with the
// r.z reduction and beta. set_fused(false) runs the reference sequence kernel
// by kernel instead; both give the same iterates.
#include "krylov.hpp"

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <functional>
#include <array>
#include <chrono>
#include <cmath>
#include <iomanip>
#include <sstream>

#include "grid_plan.hpp"
#include "learned.hpp"

namespace kutta_amd {

OwnedCsr::OwnedCsr(HipDevice& dev, const CsrHost& a)
    : n_rows(a.n_rows), nnz(a.nnz()), row_ptr(to_device(dev, a.row_ptr)),
      col(to_device(dev, a.col)), diag(to_device(dev, a.diag)), val(dev, a.val.size()) {
  std::vector<float> v(a.val.size());
  for (std::size_t j = 0; j < v.size(); ++j) v[j] = static_cast<float>(a.val[j]);
  val.upload(v);
}

namespace {

// Normalized (hi, lo) pair of a double (runtime/cpu/cpu_device.cpp:83-86).
std::array<float, 2> pair_of(double value) {
  const float hi = static_cast<float>(value);
  return {hi, std::isfinite(hi) ? static_cast<float>(value - double(hi)) : 0.0f};
}

struct Level {
  Index rows = 0, nnz = 0;
  Index max_row = 0;  // longest row (entries)
  OwnedCsr matrix;  // coarse levels only; level 0 uses the caller's operator
  CsrHost host;     // coarse levels: the operator as built (pattern and setup values)
  DeviceArray<std::uint16_t> val16;  // bfloat16 copy of the values (mixed path)
  DeviceArray<float> l1, x, b, r, projection;
  bool has_transfer = false;
  DeviceArray<Index> aggregate, member_offsets, members, entry_offsets, entries;
  Index coarse_rows = 0;
  // How the fused path restricts this level's residual (all bitwise equal,
  // picked by the autotuner): 0 one kernel, 64 coarse rows per workgroup;
  // 1 the same with 128; 2 a row-parallel residual then the member sums,
  // which reads the fine rows coalesced when aggregates are scattered; 3 the
  // same with the residual one wavefront per row (levels with long rows).
  int restrict_mode = 0;
  // How the fused path prolongs into this level (bitwise equal, picked by the
  // autotuner): 0 the prolongation folded into the first post-smoothing
  // sweep's gathers; 1 the in-place prolongation, then a plain sweep, which
  // keeps the sweep's gathers to one dependent load per entry; 2 the folded
  // form one wavefront per row (levels with long rows).
  int prolong_mode = 0;
  // The plain sweep's form (bitwise equal, picked by the autotuner for levels
  // with rows longer than KH_WIDE_ROW): 0 one thread per row, 1 one
  // wavefront per row.
  int sweep_mode = 0;
  // The coarsest level's row partition for KH_COARSE_SWEEPS_RESIDENT and its
  // register capacity (0: the level does not fit).
  DeviceArray<Index> resident;
  int resident_cap = 0;
  // K-cycle workspaces of a coarse level (linalg/amg.cpp:185-193): the inner
  // corrections' vectors, 12 pair scalars and 1-int status.
  DeviceArray<float> kp, kq, kz, kt, kscalars;
  DeviceArray<Index> kstatus;
};

Index longest_row(const CsrHost& a) {
  Index longest = 0;
  for (Index i = 0; i < a.n_rows; ++i) longest = std::max(longest, a.row_ptr[i + 1] - a.row_ptr[i]);
  return longest;
}

// What the caller wants fused into the last sweep of the fine level.
enum class Tail { None, DotBeta };

}  // namespace

struct KrylovSolver::Impl {
  HipDevice& dev;
  SolverKind kind;
  AmgOptions options;
  bool amg, nullspace, fused = true;
  Index n = 0, nnz = 0;
  double complexity = 0;
  std::vector<Level> levels;
  DeviceArray<float> jacobi_inverse, jacobi_invalid;
  DeviceArray<float> r, z, p, q, shadow, s, t, zs, best;
  DeviceArray<float> scalars;
  DeviceArray<Index> status;
  DeviceArray<float> projection;
  double best_residual = 0;
  int previous_iterations = 0;
  bool verified_current = false;
  int waits = 0;
  // Coarse-grid tail: levels [tail_first, end) run as one KH_FUSED_COARSE_TAIL
  // launch (0: off). tail_request < 0 picks the level automatically.
  int tail_request = -1;
  int tail_first = 0;
  DeviceArray<kh_tail_level> tail_table;
  // The multi-workgroup V-cycle: levels [grid_first, end) run as one
  // KH_GRID_CYCLE launch (0: off), in place of the tail, when the tail is
  // automatic. grid_request < 0 picks the level by the rule in pick_grid;
  // grid_off: the caller wants none, whatever is picked or timed.
  int grid_request = -1;
  bool grid_off = false;
  int grid_first = 0;
  int grid_limit_us = 2000;  // how long its workgroups wait for each other
  GridPlan grid_plan;
  struct GridLevelArrays {
    DeviceArray<Index> slot;
    DeviceArray<std::uint16_t> place, local_col;
  };
  std::vector<GridLevelArrays> grid_arrays;
  DeviceArray<kh_grid_level> grid_levels;
  DeviceArray<kh_grid_part> grid_table;
  DeviceArray<std::uint32_t> grid_ctl;
  int grid_polls = 1 << 21;  // what its barriers wait before they give up
  Index grid_given_up = 0;   // launches that did, as last seen
  // Launches in which one workgroup worked alone cost the wait and then some
  // milliseconds on one CU. Another stream's kernels on the card cause them, so
  // after kGridMisses in one solve a cycle that nobody asked for by level rests
  // for kGridRest solves, the tail or the levels' launches in its place.
  static constexpr int kGridMisses = 3, kGridRest = 256;
  bool grid_asked = false;
  Index grid_alone = 0;  // as last seen
  int grid_missed = 0;   // of this solve
  int grid_rest = 0;     // solves left without the cycle, this one among them
  bool grid_spread = false;  // launches go over the XCDs as the cycle needs
  // The level it is planned from (0: none; it has no bfloat16 form), and
  // whether cycles run it now.
  int grid_level() const { return coarse_bf16 ? 0 : grid_first; }
  bool grid_on() const { return grid_level() > 0 && grid_rest == 0; }

  Impl(HipDevice& d, SolverKind k, const CsrHost& a, const AmgOptions& o)
      : dev(d), kind(k), options(o),
        amg(k == SolverKind::AmgPcg || k == SolverKind::AmgBicgstab || k == SolverKind::AmgFgmres),
        nullspace(o.nullspace == NullSpace::Constant), n(a.n_rows), nnz(a.nnz()) {
    validate_host(a);
    // The solver's status, and what the multi-workgroup cycle counts: one
    // poll reads both.
    status = DeviceArray<Index>(dev, 3 + KH_GRID_REPORT_WORDS);
    dev.fill_int(status.data(), 0, status.size());
    if (amg) {
      KA_REQUIRE(options.pre_sweeps > 0 && options.post_sweeps > 0 && options.coarse_sweeps > 0 &&
                     options.coarse_rows >= 1 && options.max_levels >= 1 &&
                     options.aggregation_passes >= 1 && options.aggregation_passes <= 8 &&
                     std::isfinite(options.strength_threshold) && options.strength_threshold >= 0 &&
                     options.strength_threshold <= 1,
                 "AMG: invalid options");
      KA_REQUIRE(k != SolverKind::AmgPcg || options.pre_sweeps == options.post_sweeps,
                 "AMG-PCG requires equal pre/post sweeps");
      KA_REQUIRE(k != SolverKind::AmgFgmres || options.nullspace == NullSpace::None,
                 "FGMRES: constant-nullspace operators are not supported");
      if (options.structure == Structure::SymmetricMMatrix) check_m_matrix(a);
      build_hierarchy(a);
      plan_tail();
    } else {
      jacobi_inverse = to_device(dev, diagonal_values(a, false, false));
      jacobi_invalid = DeviceArray<float>(dev, n);
    }
    r = DeviceArray<float>(dev, n);
    z = DeviceArray<float>(dev, n);
    p = DeviceArray<float>(dev, n);
    q = DeviceArray<float>(dev, n);
    best = DeviceArray<float>(dev, n);
    if (bicg()) {
      shadow = DeviceArray<float>(dev, n);
      s = DeviceArray<float>(dev, n);
      t = DeviceArray<float>(dev, n);
      zs = DeviceArray<float>(dev, n);
    }
    scalars = DeviceArray<float>(dev, 24);
    projection = DeviceArray<float>(dev, 2);
    dev.fill(scalars.data(), 0.0f, 24);
  }
  bool bicg() const { return kind == SolverKind::BicgstabJacobi || kind == SolverKind::AmgBicgstab; }
  bool gmres() const { return kind == SolverKind::FgmresJacobi || kind == SolverKind::AmgFgmres; }

  // Flexible GMRES(m) (Saad 1993), right preconditioned by the V-cycle or the
  // Jacobi inverse: the cycle's Arnoldi steps, rotations and convergence test
  // run on the device (kh_gmres.hip); the host polls every
  // residual_check_interval steps and verifies the true residual after each
  // cycle, restarting from it.
  // Mixed-precision AMG (no reference counterpart): level `direct_level` is
  // solved by an FP64 dense inverse (blocked Gauss-Jordan on the FP64 MFMA
  // at refresh, one GEMV per V-cycle) instead of coarser levels and sweeps;
  // 0 is off.
  int direct_level = 0;
  bool direct_ready = false;
  // Mixed-precision AMG: coarse levels (1 and below) smoothed, restricted and
  // prolonged from bfloat16 copies of their values (FP32 arithmetic), made at
  // each refresh. The coarse tail and the dense direct level keep FP32.
  bool coarse_bf16 = false, bf16_ready = false;
  bool bf16_level(const Level& l) const {
    return coarse_bf16 && fused && &l != &levels[0] && !l.val16.empty();
  }
  void set_coarse_bf16(bool on) {
    drop_graphs();
    KA_REQUIRE(!on || amg, "AMG: bfloat16 coarse levels need an AMG solver");
    KA_REQUIRE(!on || !nullspace, "AMG: bfloat16 coarse levels are not supported with the nullspace projection");
    coarse_bf16 = on;
    bf16_ready = false;
    if (!on)
      for (auto& l : levels) l.val16 = DeviceArray<std::uint16_t>();
  }
  DeviceArray<double> dense_inverse;
  // Lazy dense refresh (no reference counterpart): with a tolerance > 0 a
  // refresh keeps the inverse while the level's values stay within that
  // relative l2 distance of the values it was computed from (`dense_basis`);
  // 0 recomputes it at every refresh.
  double dense_tolerance = 0.0, dense_staleness = 0.0;
  DeviceArray<float> dense_basis;
  long dense_inversions = 0, dense_skips = 0;
  int set_direct(Index rows) {
    drop_graphs();
    direct_level = 0;
    direct_ready = false;
    dense_basis = DeviceArray<float>();
    dense_inverse = DeviceArray<double>();
    if (rows <= 0) {
      plan_tail();
      return 0;
    }
    KA_REQUIRE(amg && options.structure == Structure::SymmetricMMatrix && !nullspace,
               "AMG: the dense coarse solve needs a symmetric M-matrix operator without nullspace");
    KA_REQUIRE(rows <= 8192, "AMG: the dense coarse solve takes at most 8192 rows");
    for (std::size_t i = 1; i < levels.size(); ++i)
      if (levels[i].rows <= rows) {
        direct_level = int(i);
        break;
      }
    KA_REQUIRE(direct_level > 0, "AMG: no coarse level has at most " + std::to_string(rows) + " rows");
    const std::size_t nc = std::size_t(levels[direct_level].rows);
    dense_inverse = DeviceArray<double>(dev, nc * nc);
    plan_tail();
    return direct_level;
  }
  int restart_length = 30;
  DeviceArray<float> basis_v, basis_z, gmres_w;
  DeviceArray<double> gmres_block, gmres_partials;
  std::size_t gmres_target_slot() const {
    const std::size_t m = std::size_t(restart_length);
    return (m + 1) * m + 5 * m + 2;
  }
  void gmres_buffers() {
    const std::size_t m = std::size_t(restart_length);
    if (basis_v.size() != (m + 1) * std::size_t(n)) {
      basis_v = DeviceArray<float>(dev, (m + 1) * std::size_t(n));
      basis_z = DeviceArray<float>(dev, m * std::size_t(n));
    }
    if (gmres_w.size() != std::size_t(n)) gmres_w = DeviceArray<float>(dev, n);
    if (gmres_block.size() != gmres_target_slot() + 1) gmres_block = DeviceArray<double>(dev, gmres_target_slot() + 1);
    const std::size_t blocks = (std::size_t(n) + 255) / 256;
    if (gmres_partials.size() != blocks * 64) gmres_partials = DeviceArray<double>(dev, std::max<std::size_t>(blocks * 64, 1));
  }
  // Learned coarse correction stage (no reference counterpart): in FGMRES,
  // after the V-cycle z = M v, the network maps the residual v - A z,
  // restricted to level `learned_level` through the composite aggregates, to
  // a correction that is prolonged back and added to z. Mode 1 harvests the
  // restricted residuals of plain V-cycle steps instead; their exact
  // corrections (learned_targets) are level solves by AMG-PCG. Plain AMG
  // stays the fallback twice over: a network whose last training epoch left
  // more than learned_max_relative of its targets' mean square unexplained
  // is not applied at all, and within a solve the stage is dropped for the
  // remaining steps when the FGMRES residual estimate falls by less than
  // learned_reduction per step on average since the cycle began (checked at
  // each poll).
  int learned_level = 0, learned_mode = 0;
  double learned_reduction = 0.5, learned_max_relative = 0.5;
  double learned_relative = -1;  // unexplained fraction after training; < 0: not trained here
  std::unique_ptr<LearnedNetwork> learned;
  std::unique_ptr<KrylovSolver> level_solver;
  DeviceArray<Index> learned_map, learned_offsets, learned_members;
  DeviceArray<float> learned_r, learned_e, learned_fine, harvest, targets;
  int learned_group = 1;  // lanes per coarse node in the restriction gather
  int harvest_capacity = 0, harvested = 0, targeted = 0;
  long learned_applications = 0, learned_fallbacks = 0, learned_solves = 0, learned_gated = 0;
  double learned_loss = 0;
  bool learned_active = false;

  void set_learned(int level, int layers, std::uint64_t seed, int capacity) {
    KA_REQUIRE(amg && gmres(), "learned stage: needs the AMG FGMRES solver kind");
    KA_REQUIRE(level >= 1 && std::size_t(level) < levels.size(),
               "learned stage: level must be a coarse level of the hierarchy");
    KA_REQUIRE(capacity >= 0, "learned stage: negative harvest capacity");
    const Level& target_level = levels[level];
    const Index rows = target_level.rows;
    // Composite aggregate of every fine row (-1: not aggregated).
    std::vector<Index> map(static_cast<std::size_t>(n));
    for (Index i = 0; i < n; ++i) map[i] = i;
    for (int k = 0; k < level; ++k) {
      const auto agg = levels[k].aggregate.download();
      for (auto& v : map) v = v >= 0 ? agg[std::size_t(v)] : -1;
    }
    std::vector<Index> offsets(std::size_t(rows) + 1, 0), members;
    for (Index v : map)
      if (v >= 0) ++offsets[std::size_t(v) + 1];
    for (Index a = 0; a < rows; ++a) offsets[a + 1] += offsets[a];
    members.resize(std::size_t(offsets.back()));
    std::vector<Index> cursor(offsets.begin(), offsets.end() - 1);
    for (Index i = 0; i < n; ++i)
      if (map[i] >= 0) members[std::size_t(cursor[map[i]]++)] = i;
    learned_level = level;
    learned_map = to_device(dev, map);
    learned_offsets = to_device(dev, offsets);
    learned_members = to_device(dev, members.empty() ? std::vector<Index>{0} : members);
    learned_r = DeviceArray<float>(dev, rows);
    learned_e = DeviceArray<float>(dev, rows);
    learned_fine = DeviceArray<float>(dev, n);
    learned_group = 1;
    while (learned_group < 64 && std::size_t(learned_group) * std::size_t(rows) < members.size()) learned_group *= 2;
    learned = std::make_unique<LearnedNetwork>(dev, layers, seed);
    learned->set_graph(target_level.matrix.view());
    AmgOptions sub;
    sub.structure = options.structure;
    level_solver = std::make_unique<KrylovSolver>(dev, SolverKind::AmgPcg, target_level.host, sub);
    harvest_capacity = capacity;
    harvest = capacity ? DeviceArray<float>(dev, std::size_t(capacity) * rows) : DeviceArray<float>();
    targets = capacity ? DeviceArray<float>(dev, std::size_t(capacity) * rows) : DeviceArray<float>();
    harvested = targeted = 0;
    learned_applications = learned_fallbacks = learned_solves = learned_gated = 0;
    learned_relative = -1;
    learned_mode = 0;
  }
  // Exact corrections of the harvested residuals: A_l e = r by AMG-PCG on the
  // level operator (current values) to `rel_tol`.
  int learned_targets(double rel_tol) {
    KA_REQUIRE(learned != nullptr, "learned stage: not configured");
    const DeviceCsr op = levels[learned_level].matrix.view();
    level_solver->refresh(op);
    const std::size_t rows = std::size_t(op.n_rows);
    SolveControl control{rel_tol, 1e-30, 500, 8};
    for (int k = targeted; k < harvested; ++k) {
      float* e = targets.data() + std::size_t(k) * rows;
      dev.fill(e, 0.0f, rows);
      level_solver->solve(op, e, harvest.data() + std::size_t(k) * rows, control);
    }
    targeted = harvested;
    return targeted;
  }
  TrainResult learned_train(int steps, float lr, int pairs) {
    KA_REQUIRE(learned != nullptr, "learned stage: not configured");
    KA_REQUIRE(targeted > 0, "learned stage: no harvested pairs with targets");
    KA_REQUIRE(pairs >= 0, "learned stage: negative training pair count");
    const int used = pairs > 0 ? std::min(pairs, targeted) : targeted;
    auto result = learned->train(harvest.data(), targets.data(), used, steps, lr);
    if (!result.loss.empty()) {
      learned_loss = result.loss.back();
      // The last epoch: one step per pair (or every step, if fewer).
      const std::size_t k = std::min<std::size_t>(std::size_t(used), result.relative.size());
      double sum = 0;
      for (std::size_t i = result.relative.size() - k; i < result.relative.size(); ++i) sum += result.relative[i];
      learned_relative = sum / double(k);
    }
    return result;
  }
  // The mean unexplained fraction of the network on harvested pairs
  // [first, first + count), without training on them (held-out pairs).
  double learned_evaluate(int first, int count) {
    KA_REQUIRE(learned != nullptr, "learned stage: not configured");
    KA_REQUIRE(first >= 0 && count >= 1 && first + count <= targeted, "learned stage: pairs out of range");
    const std::size_t rows = std::size_t(levels[learned_level].rows);
    double sum = 0;
    for (int k = first; k < first + count; ++k) {
      const double loss = learned->gradient(harvest.data() + std::size_t(k) * rows,
                                            targets.data() + std::size_t(k) * rows);
      const double energy = learned->target_energy();
      sum += energy > 0 ? loss / energy : 0.0;
    }
    return sum / count;
  }
  void learned_stage(const DeviceCsr& a, const float* v, float* zj) {
    const Index rows = levels[learned_level].rows;
    dev.launch(KH_LEARNED_RESTRICT, rows,
               {a.row_ptr, a.col, a.val, v, zj, learned_offsets, learned_members, learned_r, learned_fine,
                int(n), learned_group});
    learned->infer(learned_r.data(), learned_e.data());
    dev.launch(KH_LEARNED_PROLONG, n, {learned_map, learned_e, zj});
    ++learned_applications;
  }
  void learned_harvest(const DeviceCsr& a, const float* v, const float* zj) {
    const Index rows = levels[learned_level].rows;
    dev.launch(KH_LEARNED_RESTRICT, rows,
               {a.row_ptr, a.col, a.val, v, zj, learned_offsets, learned_members,
                harvest.data() + std::size_t(harvested) * rows, learned_fine, int(n), learned_group});
    ++harvested;
  }
  // Whether the residual estimate has fallen by at least learned_reduction
  // per step on average over the first `steps` steps of the cycle.
  bool learned_keeps_pace(int steps) {
    const std::size_t m = std::size_t(restart_length), g = (m + 1) * m;
    ++waits;
    const auto block = gmres_block.download();
    const double start = std::fabs(block[g]), now = std::fabs(block[g + std::size_t(steps)]);
    if (!(start > 0) || !std::isfinite(now)) return false;
    const double factor = std::pow(now / start, 1.0 / steps);
    return 1.0 - factor >= learned_reduction;
  }

  void fgmres(const DeviceCsr& a, float* x, const float* b, const SolveControl& c, double target,
              SolveStats& st) {
    const int m = restart_length;
    gmres_buffers();
    {
      std::vector<double> host(gmres_block.size(), 0.0);
      host[gmres_target_slot()] = target;
      gmres_block.upload(host);
    }
    learned_active = learned && learned_mode == 2;
    if (learned_active) {
      ++learned_solves;
      if (learned_relative > learned_max_relative) {
        learned_active = false;
        ++learned_gated;
      }
    }
    int restarts = 0;
    double last = st.initial_residual;
    while (st.iterations < c.max_iter) {
      reset(st.iterations);
      dev.launch(KH_GMRES_START, n, {r, basis_v, gmres_block, m, status, gmres_partials});
      const int steps = std::min(m, c.max_iter - st.iterations);
      const int harvest_start = harvested;
      verified_current = false;
      for (int j = 0; j < steps; ++j) {
        float* vj = basis_v.data() + std::size_t(j) * n;
        float* zj = basis_z.data() + std::size_t(j) * n;
        apply(a, vj, zj, Tail::None);
        if (learned_active) learned_stage(a, vj, zj);
        else if (learned && learned_mode == 1 && harvested < harvest_capacity) learned_harvest(a, vj, zj);
        dev.launch(KH_CSR_SPMV_GUARDED, n, {a.row_ptr, a.col, a.val, zj, gmres_w, status});
        dev.launch(KH_GMRES_ARNOLDI, n, {basis_v, gmres_w, gmres_block, m, j, status, gmres_partials});
        if ((j + 1) % c.residual_check_interval == 0 && j + 1 < steps) {
          if (poll()[0] != 0) break;
          if (learned_active && !learned_keeps_pace(j + 1)) {
            learned_active = false;
            ++learned_fallbacks;
          }
        }
      }
      dev.launch(KH_GMRES_UPDATE, n, {basis_z, x, gmres_block, m, status});
      const auto state = poll();
      st.iterations = state[1];
      // Only the steps whose columns were built hold meaningful residuals.
      harvested = std::min(harvested, harvest_start + int(state[2]));
      if (verified(a, x, b, target, st) || diverged(st)) break;
      restarts = st.final_residual >= 0.9 * last ? restarts + 1 : 0;
      last = st.final_residual;
      if (restarts >= 12) break;
    }
  }

  // linalg/amg.cpp:200-226
  void build_hierarchy(const CsrHost& a) {
    levels.emplace_back();
    levels.back().rows = a.n_rows;
    levels.back().nnz = a.nnz();
    levels.back().max_row = longest_row(a);
    levels.back().l1 = to_device(dev, diagonal_values(a, true, nullspace));
    levels.back().r = DeviceArray<float>(dev, a.n_rows);
    if (nullspace) levels.back().projection = DeviceArray<float>(dev, 2);
    const CsrHost* current = &a;
    CsrHost owned;
    std::size_t total = a.nnz();
    while (current->n_rows > options.coarse_rows && levels.size() < std::size_t(options.max_levels)) {
      Coarsening c = aggregate(*current, options);
      const auto active = c.members.size();
      if (active == 0 || c.matrix.n_rows >= 0.85 * double(active)) break;
      Level& fine = levels.back();
      fine.has_transfer = true;
      fine.coarse_rows = c.matrix.n_rows;
      fine.aggregate = to_device(dev, c.aggregate);
      fine.member_offsets = to_device(dev, c.member_offsets);
      fine.members = to_device(dev, c.members);
      fine.entry_offsets = to_device(dev, c.entry_offsets);
      fine.entries = to_device(dev, c.entries);
      total += c.matrix.nnz();
      Level coarse;
      coarse.rows = c.matrix.n_rows;
      coarse.nnz = c.matrix.nnz();
      coarse.max_row = longest_row(c.matrix);
      coarse.l1 = to_device(dev, diagonal_values(c.matrix, true, nullspace));
      coarse.x = DeviceArray<float>(dev, c.matrix.n_rows);
      coarse.b = DeviceArray<float>(dev, c.matrix.n_rows);
      coarse.r = DeviceArray<float>(dev, c.matrix.n_rows);
      if (nullspace) coarse.projection = DeviceArray<float>(dev, 2);
      if (options.cycle == AmgCycle::K) {
        for (auto* v : {&coarse.kp, &coarse.kq, &coarse.kz, &coarse.kt})
          *v = DeviceArray<float>(dev, c.matrix.n_rows);
        coarse.kscalars = DeviceArray<float>(dev, 12);
        coarse.kstatus = DeviceArray<Index>(dev, 1);
        dev.fill(coarse.kscalars.data(), 0.0f, 12);
        dev.fill_int(coarse.kstatus.data(), 0, 1);
      }
      coarse.matrix = OwnedCsr(dev, c.matrix);
      coarse.host = c.matrix;
      owned = std::move(c.matrix);
      levels.push_back(std::move(coarse));
      current = &owned;
    }
    complexity = a.nnz() ? double(total) / a.nnz() : 0;
    Level& last = levels.back();
    if (levels.size() > 1 && last.rows <= KH_RESIDENT_MAX_ROWS) {
      std::vector<Index> table(KH_RESIDENT_TABLE_INTS);
      int32_t cap = 0;
      if (kh_resident_partition(last.host.row_ptr.data(), last.host.col.data(), last.rows, table.data(), &cap) == 0) {
        last.resident = to_device(dev, table);
        last.resident_cap = cap;
      }
    }
  }

  // Whether levels [first, end) fit one KH_FUSED_COARSE_TAIL workgroup: all
  // iterates and right-hand sides, one sweep's new values and the largest
  // level's operator copy in LDS at once.
  bool tail_fits(std::size_t first) const {
    if (first < tail_floor() || first >= levels.size() || levels.size() - first > KH_TAIL_MAX_LEVELS) return false;
    std::size_t vectors = 0, widest = 0, largest = 0;
    for (std::size_t i = first; i < levels.size(); ++i) {
      const std::size_t rows = std::size_t(levels[i].rows), nnz = std::size_t(levels[i].nnz);
      if (rows > KH_TAIL_MAX_ROWS) return false;
      vectors += 2 * rows;
      widest = std::max(widest, rows);
      largest = std::max(largest, 3 * rows + 1 + 2 * nnz);
    }
    return vectors <= KH_TAIL_LDS_FLOATS && vectors + widest + largest <= KH_TAIL_POOL_WORDS;
  }

  // Picks the tail's first level: the requested one, or else the first level
  // of at most kTailAutoRows rows from which the rest of the hierarchy fits
  // one workgroup. Above that size one CU's compensated sweeps cost more than
  // a level's own launches, whose sweeps spread over the whole chip.
  static constexpr Index kTailAutoRows = 2048;
  void plan_tail() {
    drop_graphs();
    tail_first = 0;
    tail_table = DeviceArray<kh_tail_level>();
    drop_grid();
    if (!amg || tail_request == 0 || direct_level > 0) return;
    if (tail_request > 0) {
      KA_REQUIRE(tail_fits(std::size_t(tail_request)),
                 "AMG: coarse tail level " + std::to_string(tail_request) + " does not fit one workgroup");
      tail_first = tail_request;
    } else {
      for (std::size_t i = 1; i < levels.size(); ++i)
        if (levels[i].rows <= kTailAutoRows && tail_fits(i)) {
          tail_first = int(i);
          break;
        }
      pick_grid();
    }
    if (tail_first > 0) tail_table = to_device(dev, tail_levels(std::size_t(tail_first)));
  }
  std::vector<kh_tail_level> tail_levels(std::size_t first) const {
    std::vector<kh_tail_level> table;
    for (std::size_t i = first; i < levels.size(); ++i) {
      const Level& l = levels[i];
      const DeviceCsr m = l.matrix.view();
      kh_tail_level t{};
      t.row_ptr = m.row_ptr;
      t.col = m.col;
      t.val = m.val;
      t.inverse = l.l1.data();
      if (l.has_transfer) {
        t.member_offsets = l.member_offsets.data();
        t.members = l.members.data();
        t.aggregate = l.aggregate.data();
        t.coarse_rows = l.coarse_rows;
      }
      t.rows = l.rows;
      t.nnz = l.nnz;
      table.push_back(t);
    }
    return table;
  }

  // ---- the multi-workgroup V-cycle (KH_GRID_CYCLE)
  // By itself it takes over from the first level, at least two before the end,
  // whose plan fits the LDS of 16 workgroups. Solves of tetrahedral pressure
  // problems, V(5,5), ms (repeats differ by up to 2% at 10k and 78k cells, by 4%
  // at 1.0M; "tail": the best the automatic tail's rule allows):
  //     first level's rows           none   tail     8      16      32
  //     10k cells,   2,611           4.57   3.98   2.60    2.60    2.65
  //                    681                         2.87    2.92    2.94
  //     78k cells,  19,808           5.81   7.18     -       -     5.10
  //                  5,138                         5.00    4.94    5.26
  //                  1,397                         4.97    5.02    5.31
  //     1.0M cells, 17,004          18.29  23.70     -       -    17.06
  //                  5,023                           -    17.15   17.21
  //                  2,017                        17.40   17.40   17.45
  //                  1,067                        17.77   17.78   17.75
  // so 8 or 16 workgroups do alike, and 32, which hold more, within the noise of
  // the next level on 16 at 1.0M cells and worse at 78k: they are for the
  // autotuner and for callers that ask. A last level by itself (15,292 rows, 4
  // sweeps a visit under a K-cycle) took 19.25 against 18.81: only the autotuner
  // tries it.
  static constexpr Index kGridAutoRows = 24576;
  static constexpr int kGridParts = 16;
  bool grid_allowed(std::size_t first) const {
    return amg && !nullspace && !coarse_bf16 && direct_level == 0 && first >= tail_floor() && first < levels.size() &&
           levels[first].rows <= kGridAutoRows && levels[first].rows > KH_GRID_BOTTOM_ROWS;
  }
  bool plan_grid_at(std::size_t first, GridPlan& plan, bool automatic = false) const {
    if (!grid_allowed(first)) return false;
    std::vector<const CsrHost*> patterns;
    for (std::size_t i = first; i < levels.size(); ++i) patterns.push_back(&levels[i].host);
    return plan_grid(patterns, kGridParts, plan) || (!automatic && plan_grid(patterns, KH_GRID_MAX_PARTS, plan));
  }
  void drop_grid() {
    grid_first = 0;
    grid_arrays.clear();
    grid_levels = DeviceArray<kh_grid_level>();
    grid_table = DeviceArray<kh_grid_part>();
    grid_missed = grid_rest = 0;
  }
  // The control block, made on first use.
  void grid_block() {
    if (!grid_ctl.empty()) return;
    grid_ctl = DeviceArray<std::uint32_t>(dev, KH_GRID_CTL_WORDS);
    dev.launch(KH_GRID_INIT, 1, {grid_ctl});
    const Index* report = status.data() + 3;
    ok(kh_upload(dev.raw(), grid_ctl.data() + KH_GRID_CTL_REPORT, &report, sizeof report));
    set_grid_polls(grid_polls);
    grid_spread = grid_ctl.download()[KH_GRID_CTL_SPREAD] == KH_GRID_MAX_PARTS;
  }
  void pick_grid() {
    if (grid_request == 0 || grid_off) return;
    if (grid_request > 0) {
      if (plan_grid_at(std::size_t(grid_request), grid_plan)) use_grid(grid_request);
      return;
    }
    for (std::size_t i = 1; i + 1 < levels.size(); ++i)
      if (plan_grid_at(i, grid_plan, true)) {
        grid_block();
        if (grid_spread) use_grid(int(i));
        return;
      }
  }
  // Uploads grid_plan's tables for levels [first, end).
  void use_grid(int first) {
    std::vector<kh_grid_level> table;
    grid_arrays.clear();
    for (std::size_t i = std::size_t(first); i < levels.size(); ++i) {
      const Level& l = levels[i];
      const DeviceCsr m = l.matrix.view();
      kh_grid_level g{};
      g.row_ptr = m.row_ptr;
      g.col = m.col;
      g.val = m.val;
      g.inverse = l.l1.data();
      if (l.has_transfer) {
        g.member_offsets = l.member_offsets.data();
        g.members = l.members.data();
        g.aggregate = l.aggregate.data();
      }
      const GridLevelPlan& p = grid_plan.levels[i - std::size_t(first)];
      grid_arrays.push_back({to_device(dev, p.slot), to_device(dev, p.place), to_device(dev, p.local_col)});
      g.place = grid_arrays.back().place.data();
      g.slot = grid_arrays.back().slot.data();
      g.local_col = grid_arrays.back().local_col.data();
      g.x = l.x.data();
      g.w = l.r.data();
      g.b = l.b.data();
      g.rows = l.rows;
      table.push_back(g);
    }
    grid_levels = to_device(dev, table);
    grid_table = to_device(dev, grid_plan.table);
    grid_block();
    grid_first = first;
  }
  void set_grid_polls(int polls) {
    grid_polls = polls;
    if (!grid_ctl.empty()) dev.fill_int(grid_ctl.data() + KH_GRID_CTL_POLLS, polls, 1);
  }
  // What the launches since the last look counted (`report` as downloaded with
  // the status). After a barrier that gave up the iterate is wrong: the cycle
  // is left off from here on and the caller told.
  void look_at_grid(const Index* report) {
    const Index given_up = report[KH_GRID_REPORT_GIVEN_UP], alone = report[KH_GRID_REPORT_ALONE];
    grid_missed += alone - grid_alone;
    grid_alone = alone;
    if (grid_missed >= kGridMisses && !grid_asked && grid_on()) {
      drop_graphs();
      grid_rest = kGridRest + 1;
    }
    if (given_up == grid_given_up) return;
    grid_given_up = given_up;
    grid_request = 0;
    plan_tail();
    throw Error("AMG: a barrier of the multi-workgroup cycle gave up; the cycle is off now");
  }
  void grid_cycle(const float* b, float* x, const int* st) {
    dev.launch(KH_GRID_CYCLE, 1,
               {grid_levels, grid_table, grid_ctl, grid_plan.count, grid_plan.grid, options.pre_sweeps,
                options.post_sweeps, options.coarse_sweeps, grid_plan.parts, grid_plan.lds_words, grid_limit_us, b, x,
                st});
  }

  DeviceCsr level_operator(std::size_t i, const DeviceCsr& fine) const {
    return i == 0 ? fine : levels[i].matrix.view();
  }

  // linalg/amg.cpp:228-256
  void refresh_amg(const DeviceCsr& a) {
    std::vector<kh_reduction> checks;
    std::vector<double> allowed;
    for (std::size_t i = 0; i < levels.size(); ++i) {
      Level& l = levels[i];
      const DeviceCsr m = level_operator(i, a);
      dev.launch(KH_KRYLOV_DIAGONAL, m.n_rows, {m.row_ptr, m.diag, m.val, l.l1, l.r, 1});
      allowed.push_back(nullspace && m.n_rows == 1 ? 1 : 0);
      checks.push_back(HipDevice::max_abs(l.r.data(), m.n_rows));
      if (i + 1 < levels.size()) {
        const DeviceCsr c = levels[i + 1].matrix.view();
        dev.launch(KH_AMG_GALERKIN, c.nnz, {l.entry_offsets, l.entries, m.val, c.val});
        if (options.structure == Structure::SymmetricMMatrix)
          dev.launch(KH_AMG_M_MATRIX_DIAGONAL, c.n_rows,
                     {l.member_offsets, l.members, m.row_ptr, m.diag, m.val, c.row_ptr, c.diag, c.val});
      }
    }
    // The dense level's distance from the values its inverse was computed
    // from: |a|^2, |s|^2 and a.s in FP64, in the same host wait.
    const bool lazy = direct_level > 0 && direct_ready && dense_tolerance > 0 && !dense_basis.empty();
    if (lazy) {
      const DeviceCsr c = levels[direct_level].matrix.view();
      checks.push_back(HipDevice::dot(c.val, c.val, c.nnz));
      checks.push_back(HipDevice::dot(dense_basis.data(), dense_basis.data(), c.nnz));
      checks.push_back(HipDevice::dot(c.val, dense_basis.data(), c.nnz));
    }
    const auto invalid = dev.reduce_many(checks);
    ++waits;
    for (std::size_t i = 0; i < allowed.size(); ++i) {
      KA_REQUIRE(invalid[i] != 3, "AMG: requires positive diagonals");
      KA_REQUIRE(invalid[i] <= allowed[i], "AMG: invalid values or zero diagonal");
    }
    if (direct_level > 0) {
      const DeviceCsr c = levels[direct_level].matrix.view();
      bool invert = true;
      if (lazy) {
        const std::size_t k = allowed.size();
        const double aa = invalid[k], ss = invalid[k + 1], as = invalid[k + 2];
        dense_staleness = ss > 0 ? std::sqrt(std::max(0.0, aa + ss - 2 * as) / ss) : 1.0;
        invert = !(dense_staleness <= dense_tolerance);
      }
      if (invert) {
        dev.launch(KH_DENSE_INVERT, c.n_rows, {c.row_ptr, c.col, c.val, dense_inverse, status});  // no scratch used
        if (dense_tolerance > 0) {
          if (dense_basis.size() != std::size_t(c.nnz)) dense_basis = DeviceArray<float>(dev, c.nnz);
          dev.copy(dense_basis.data(), c.val, sizeof(float) * std::size_t(c.nnz));
        }
        dense_staleness = 0.0;
        ++dense_inversions;
      } else {
        ++dense_skips;
      }
      direct_ready = true;
    }
    if (coarse_bf16)
      for (std::size_t i = 1; i < levels.size(); ++i) {
        Level& l = levels[i];
        if (l.val16.size() != std::size_t(std::max<Index>(l.nnz, 1))) {
          drop_graphs();
          l.val16 = DeviceArray<std::uint16_t>(dev, std::max<Index>(l.nnz, 1));
        }
        if (l.nnz > 0) dev.launch(KH_TO_BF16, l.nnz, {l.matrix.val, l.val16});
      }
    bf16_ready = coarse_bf16;
    if (learned) learned->set_graph(levels[learned_level].matrix.view());
  }

  // Constant-nullspace projection (linalg/detail.hpp:13-19).
  void project(float* x, std::size_t count, float* sum) {
    if (count == 0) return;
    dev.reduce_into(KH_INTO_SUM, x, x, x, x, count, sum, 0);
    project_with(x, count, sum);
  }
  void project_with(float* x, std::size_t count, float* sum) {
    const float c = static_cast<float>(count);
    dev.launch(KH_SOLVER_PROJECT, count,
               {x, sum, c, static_cast<float>(double(count) - double(c))});
  }

  // One l1-Jacobi sweep (linalg/amg.cpp:272-282). `first` marks the sweep that
  // starts from the zero iterate the cycle's fill would have stored.
  void sweep(Level& l, const DeviceCsr& a, const float* b, const float* in, float* out, bool first,
             float* zero_x, const int* st) {
    if (bf16_level(l)) {
      if (first)
        dev.launch(KH_BF16_SMOOTH_FROM_ZERO, a.n_rows, {a.row_ptr, a.col, l.val16, b, l.l1, out, st});
      else
        dev.launch(KH_BF16_AMG_SMOOTH, a.n_rows, {a.row_ptr, a.col, l.val16, in, b, l.l1, out, st});
      return;
    }
    if (first) {
      if (fused) {
        dev.launch(KH_FUSED_SMOOTH_FROM_ZERO, a.n_rows, {a.row_ptr, a.col, a.val, b, l.l1, out, st});
      } else {
        dev.launch(KH_AMG_SMOOTH_ZERO, a.n_rows, {a.row_ptr, a.col, a.val, zero_x, b, l.l1, out, st});
      }
    } else {
      dev.launch(smooth_kernel(l), a.n_rows, {a.row_ptr, a.col, a.val, in, b, l.l1, out, st});
    }
  }
  // The plain sweep's kernel: the wide-chunk instantiation on the fused path
  // for levels with rows longer than KH_WIDE_ROW (same bits).
  kh_kernel smooth_kernel(const Level& l) const {
    if (!fused || l.max_row <= KH_WIDE_ROW) return KH_AMG_SMOOTH;
    return l.sweep_mode == 1 ? KH_AMG_SMOOTH_ROWWAVE : KH_AMG_SMOOTH_WIDE;
  }

  // What a V-cycle completed beyond z = M^-1 b.
  struct CycleResult {
    bool dot_beta = false;   // dot_into(r,z,4) and solver_pcg_beta already done
    bool sum_ready = false;  // the fine-level projection sum is already in `projection`
  };

  // The fused path's restriction of level l's residual into coarse_b, in one
  // of the restrict_mode forms; `spare` is an iterate buffer free to hold the
  // fine residual (mode 2).
  void restrict_level(Level& l, const DeviceCsr& a, const DeviceCsr& ca, const float* current, const float* b,
                      float* spare, float* coarse_b, int mode, const int* st) {
    if (mode >= 2) {
      dev.launch(mode == 3 ? KH_CSR_RESIDUAL_ROWWAVE : KH_CSR_RESIDUAL_GUARDED, a.n_rows,
                 {a.row_ptr, a.col, a.val, current, b, spare, st});
      dev.launch(KH_AMG_RESTRICT_GUARDED, ca.n_rows, {l.member_offsets, l.members, spare, coarse_b, st});
      return;
    }
    dev.launch(mode == 1 ? KH_FUSED_RESIDUAL_RESTRICT_WIDE : KH_FUSED_RESIDUAL_RESTRICT, ca.n_rows,
               {a.row_ptr, a.col, a.val, current, b, l.member_offsets, l.members, coarse_b, st});
  }
  // The coarsest level's sweeps (bitwise equal, picked by the autotuner): 0 a
  // launch per sweep, 1 all in one workgroup reading the operator from
  // global memory, 2 all in one workgroup with the operator in registers
  // (when the level has a resident partition).
  int coarse_sweeps_mode = 0;
  bool coarse_sweeps_fit(std::size_t index) const {
    const Level& l = levels[index];
    return index > 0 && index + 1 == levels.size() && fused && !nullspace && !bf16_level(l) && l.rows > 24 &&
           l.rows <= KH_COARSE_SWEEPS_MAX_ROWS && !(direct_level > 0 && int(index) == direct_level);
  }

  // linalg/amg.cpp:283-310. Sweep outputs alternate between x and the level's
  // scratch so that the last sweep writes x. `st` guards every launch: the
  // solver's status, or that of the K-cycle correction the cycle belongs to.
  CycleResult cycle(std::size_t index, const DeviceCsr& a, const float* b, float* x, Tail tail,
                    const int* st) {
    Level& l = levels[index];
    float* w = l.r.data();
    CycleResult result;
    const bool grid = grid_on();
    if (fused && grid && int(index) == grid_first) {
      grid_cycle(b, x, st);
      return result;
    }
    if (fused && !grid && tail_first > 0 && int(index) == tail_first) {
      dev.launch(KH_FUSED_COARSE_TAIL, 1,
                 {tail_table, int(levels.size() - index), options.pre_sweeps, options.post_sweeps,
                  options.coarse_sweeps, nullspace ? 1 : 0, b, x, st});
      return result;
    }
    KA_REQUIRE(!coarse_bf16 || bf16_ready, "AMG: refresh before solving with bfloat16 coarse levels");
    if (direct_level > 0 && int(index) == direct_level) {
      KA_REQUIRE(direct_ready, "AMG: refresh before solving with the dense coarse solve");
      dev.launch(KH_DENSE_APPLY, a.n_rows, {dense_inverse, b, x, st});
      return result;
    }
    // The reference clears x first; only the unfused sequence reads that zero.
    if (!fused) dev.fill(x, 0.0f, a.n_rows);
    const bool coarsest = index + 1 == levels.size();
    float* sum = index == 0 ? projection.data() : (nullspace ? l.projection.data() : nullptr);
    if (coarsest && a.n_rows <= 24) {
      dev.launch(KH_AMG_COARSE_SOLVE, 1,
                 {a.row_ptr, a.col, a.val, x, b, l.l1, st, int(a.n_rows), options.coarse_sweeps});
      if (nullspace && index != 0) project(x, a.n_rows, sum);
      return result;
    }
    // A coarsest level too large for the coarse tail (aggregation stalls on
    // anisotropic meshes) may run all its sweeps in one workgroup, bitwise the
    // sweep-by-sweep sequence below, when the autotuner finds that faster.
    if (coarse_sweeps_mode == 2 && l.resident_cap > 0 && coarse_sweeps_fit(index)) {
      dev.launch(KH_COARSE_SWEEPS_RESIDENT, a.n_rows,
                 {a.row_ptr, a.col, a.val, b, l.l1, x, st, options.coarse_sweeps, l.resident, l.resident_cap});
      return result;
    }
    if (coarse_sweeps_mode != 0 && coarse_sweeps_fit(index)) {
      dev.launch(KH_FUSED_COARSE_SWEEPS, a.n_rows,
                 {a.row_ptr, a.col, a.val, b, l.l1, x, st, options.coarse_sweeps});
      return result;
    }
    const int pre = coarsest ? options.coarse_sweeps : options.pre_sweeps;
    const int post = coarsest ? 0 : options.post_sweeps;
    const int total = pre + post;
    // The final sweep is a plain smoothing sweep (not the first sweep, not the
    // prolongation sweep), so a reduction can ride along with it.
    const bool last_plain = total >= 2 && (coarsest || post >= 2);
    const bool fuse_dot = fused && index == 0 && tail == Tail::DotBeta && !nullspace && last_plain;
    const bool fuse_sum = fused && nullspace && last_plain;
    auto target = [&](int t) { return (total - t) % 2 == 0 ? x : w; };
    const float* current = nullptr;
    auto run_sweep = [&](int t, float* out) {
      if (t == total && fuse_dot) {
        dev.launch(KH_FUSED_SMOOTH_DOT_BETA, a.n_rows,
                   {a.row_ptr, a.col, a.val, current, b, l.l1, out, st, scalars.data()});
        result.dot_beta = true;
      } else if (t == total && fuse_sum) {
        dev.launch(KH_FUSED_SMOOTH_SUM, a.n_rows, {a.row_ptr, a.col, a.val, current, b, l.l1, out, st, sum});
      } else {
        sweep(l, a, b, current, out, t == 1, x, st);
      }
      current = out;
    };
    for (int t = 1; t <= pre; ++t) run_sweep(t, target(t));
    if (!coarsest) {
      Level& c = levels[index + 1];
      const DeviceCsr ca = c.matrix.view();
      if (bf16_level(l)) {
        dev.launch(KH_BF16_RESIDUAL_RESTRICT, ca.n_rows,
                   {a.row_ptr, a.col, l.val16, current, b, l.member_offsets, l.members, c.b, st});
      } else if (fused) {
        restrict_level(l, a, ca, current, b, current == x ? w : x, c.b.data(), l.restrict_mode, st);
      } else {
        float* rbuf = current == x ? w : x;
        dev.launch(KH_CSR_RESIDUAL_GUARDED, a.n_rows, {a.row_ptr, a.col, a.val, current, b, rbuf, st});
        dev.launch(KH_AMG_RESTRICT_GUARDED, ca.n_rows, {l.member_offsets, l.members, rbuf, c.b, st});
      }
      if (nullspace) project(c.b.data(), ca.n_rows, c.projection.data());
      if (k_inner(index + 1)) inner(index + 1, st);
      else cycle(index + 1, ca, c.b.data(), c.x.data(), Tail::None, st);
      for (int t = pre + 1; t <= total; ++t) {
        float* out = target(t);
        if (t == pre + 1) {
          if (bf16_level(l)) {
            dev.launch(KH_BF16_PROLONG_SMOOTH, a.n_rows,
                       {a.row_ptr, a.col, l.val16, current, b, l.l1, out, l.aggregate, c.x, st});
          } else if (fused && (l.prolong_mode == 0 || l.prolong_mode == 2)) {
            dev.launch(l.prolong_mode == 2 ? KH_PROLONG_SMOOTH_ROWWAVE : KH_FUSED_PROLONG_SMOOTH, a.n_rows,
                       {a.row_ptr, a.col, a.val, current, b, l.l1, out, l.aggregate, c.x, st});
          } else {
            float* xin = const_cast<float*>(current);
            dev.launch(KH_AMG_PROLONG_GUARDED, a.n_rows, {l.aggregate, c.x, xin, st});
            dev.launch(smooth_kernel(l), a.n_rows, {a.row_ptr, a.col, a.val, xin, b, l.l1, out, st});
          }
          current = out;
        } else {
          run_sweep(t, out);
        }
      }
    }
    if (nullspace) {
      if (index != 0) {
        if (fuse_sum) project_with(x, a.n_rows, sum);
        else project(x, a.n_rows, sum);
      } else {
        result.sum_ready = fuse_sum;
      }
    }
    return result;
  }

  // Preconditioner application (linalg/solver.cpp:197-200). With tail ==
  // DotBeta it also performs dot_into(r,z,4) + solver_pcg_beta(0), as the PCG
  // loop does right after apply (linalg/solver.cpp:295-298).
  void apply(const DeviceCsr& a, const float* rin, float* zout, Tail tail) {
    CycleResult done;
    if (amg) {
      done = cycle(0, a, rin, zout, variable() ? Tail::None : tail, status.data());
    } else {
      dev.launch(KH_KRYLOV_MULTIPLY_GUARDED, n, {rin, jacobi_inverse, zout, status});
    }
    if (done.dot_beta) return;
    if (nullspace) {
      if (!done.sum_ready) dev.reduce_into(KH_INTO_SUM, zout, zout, zout, zout, n, projection.data(), 0);
      if (tail == Tail::DotBeta && fused && !variable()) {
        const float c = static_cast<float>(n);
        dev.launch(KH_FUSED_PROJECT_DOT_BETA, n,
                   {zout, projection, c, static_cast<float>(double(n) - double(c)), r, scalars, status});
        return;
      }
      project_with(zout, n, projection.data());
    }
    if (tail == Tail::DotBeta) {
      // linalg/solver.cpp:295-297: a variable preconditioner (the K-cycle)
      // takes the flexible beta, -alpha z.Ap / rho.
      if (variable()) dev.reduce_into(KH_INTO_DOT2, r.data(), zout, zout, q.data(), n, scalars.data(), 4);
      else dot_into(r.data(), zout, 4);
      dev.launch(KH_SOLVER_PCG_BETA, 1, {scalars, status, variable() ? 1 : 0});
    }
  }

  // linalg/amg.cpp:262: the K-cycle is a variable preconditioner.
  bool variable() const { return amg && options.cycle == AmgCycle::K; }
  // Whether coarse level `c` is reached through the K-cycle's inner
  // corrections (linalg/amg.cpp:301-302): every level with two below it,
  // down to k_depth and of at least k_min_rows rows when set, and never at or
  // below a dense-solved level.
  bool k_inner(std::size_t c) const {
    return variable() && c + 1 < levels.size() && (options.k_depth == 0 || c <= std::size_t(options.k_depth)) &&
           levels[c].rows >= options.k_min_rows && !(direct_level > 0 && c >= std::size_t(direct_level));
  }
  // The first level the one-workgroup tail (a V-cycle) may start at.
  std::size_t tail_floor() const {
    std::size_t c = 1;
    while (c < levels.size() && k_inner(c)) ++c;
    return c;
  }

  // linalg/amg.cpp:315-336: two preconditioned Krylov corrections of the
  // coarse equation A x = b at `index` (A-conjugate directions for SPD, GCR
  // otherwise), each cycle guarded by `parent` then by the level's own status,
  // which also skips the second correction once |t| <= |b| / 4.
  void inner(std::size_t index, const int* parent) {
    Level& l = levels[index];
    const DeviceCsr a = l.matrix.view();
    const std::size_t m = std::size_t(a.n_rows);
    const bool spd = kind == SolverKind::AmgPcg;
    float* s = l.kscalars.data();
    Index* st = l.kstatus.data();
    float *b = l.b.data(), *x = l.x.data(), *p = l.kp.data(), *q = l.kq.data(), *z = l.kz.data(),
          *t = l.kt.data(), *w = l.r.data();
    auto spmv = [&](const float* in, float* out, const int* guard) {
      dev.launch(KH_CSR_SPMV_GUARDED, a.n_rows, {a.row_ptr, a.col, a.val, in, out, guard});
    };
    if (fused) {
      // The same steps, each dot product in the kernel producing its operand
      // and each scalar update in the reduction's finisher.
      const int sp = spd ? 1 : 0;
      cycle(index, a, b, z, Tail::None, parent);
      dev.launch(KH_INNER_FIRST_STEP, a.n_rows, {a.row_ptr, a.col, a.val, z, p, q, b, s, st, parent, sp});
      dev.launch(KH_INNER_FIRST_UPDATE, a.n_rows, {b, p, q, x, t, s, st});
      cycle(index, a, t, z, Tail::None, st);
      dev.launch(KH_INNER_BETA_STEP, a.n_rows, {a.row_ptr, a.col, a.val, z, w, q, s, st, sp});
      dev.launch(KH_SOLVER_DIRECTION, a.n_rows, {z, p, s, st});
      dev.launch(KH_INNER_SECOND_STEP, a.n_rows, {a.row_ptr, a.col, a.val, p, q, t, s, st, parent, sp});
      dev.launch(KH_AMG_INNER_STEP, a.n_rows, {x, p, s, st});
      return;
    }
    cycle(index, a, b, z, Tail::None, parent);
    dev.copy(p, z, sizeof(float) * m);
    spmv(p, q, parent);
    dev.reduce_into(KH_INTO_DOT2, spd ? p : q, q, b, spd ? p : q, m, s, 0);
    dev.launch(KH_AMG_INNER_ALPHA, 1, {s, st, parent, 1});
    dev.launch(KH_AMG_INNER_FIRST, a.n_rows, {b, p, q, x, t, s, st});
    dev.reduce_into(KH_INTO_DOT2, t, t, b, b, m, s, 4);
    dev.launch(KH_AMG_INNER_CHECK, 1, {s, st});
    cycle(index, a, t, z, Tail::None, st);
    if (!spd) spmv(z, w, st);
    dev.reduce_into(KH_INTO_DOT, spd ? z : w, q, spd ? z : w, q, m, s, 4);
    dev.launch(KH_AMG_INNER_BETA, 1, {s, st});
    dev.launch(KH_SOLVER_DIRECTION, a.n_rows, {z, p, s, st});
    spmv(p, q, st);
    dev.reduce_into(KH_INTO_DOT2, spd ? p : q, q, t, spd ? p : q, m, s, 0);
    dev.launch(KH_AMG_INNER_ALPHA, 1, {s, st, parent, 0});
    dev.launch(KH_AMG_INNER_STEP, a.n_rows, {x, p, s, st});
  }

  void residual(const DeviceCsr& a, const float* x, const float* b, float* out) {
    dev.launch(KH_CSR_RESIDUAL, a.n_rows, {a.row_ptr, a.col, a.val, x, b, out});
  }
  double norm(const float* v) {
    ++waits;
    return std::sqrt(dev.reduce_many({HipDevice::dot(v, v, n)})[0]);
  }
  // linalg/solver.cpp:201-222
  bool verified(const DeviceCsr& a, float* x, const float* b, double target, SolveStats& st) {
    if (nullspace) project(x, n, projection.data());
    residual(a, x, b, r.data());
    st.final_residual = norm(r.data());
    verified_current = true;
    st.converged = std::isfinite(st.final_residual) && st.final_residual <= target;
    if (st.final_residual < best_residual) {
      best_residual = st.final_residual;
      dev.copy(best.data(), x, sizeof(float) * n);
    }
    if (nullspace) project(r.data(), n, projection.data());
    return st.converged;
  }
  static bool diverged(const SolveStats& st) {
    return !std::isfinite(st.final_residual) || st.final_residual > 1e3 * st.initial_residual;
  }
  void reset(int iterations) { dev.launch(KH_SOLVER_RESET, 1, {scalars, status, iterations}); }
  bool replacement(const DeviceCsr& a, float* x, const float* b, double target, SolveStats& st,
                   int& restarts, double& last) {
    if (verified(a, x, b, target, st) || diverged(st)) return false;
    restarts = st.final_residual >= 0.9 * last ? restarts + 1 : 0;
    last = st.final_residual;
    return restarts < 12;
  }
  int batch_interval(const SolveControl& c) const {
    return previous_iterations > 0 && previous_iterations < c.residual_check_interval
               ? previous_iterations + 1 : c.residual_check_interval;
  }
  std::array<Index, 3> poll() {
    ++waits;
    const auto host = status.download();
    look_at_grid(host.data() + 3);
    return {host[0], host[1], host[2]};
  }
  void dot_into(const float* x, const float* y, int offset) {
    dev.reduce_into(KH_INTO_DOT, x, y, x, y, n, scalars.data(), offset);
  }

  // HIP graph of one fused PCG iteration (no reference counterpart): the
  // iteration's launches (spmv + p.q + alpha, step + r.r + check, the V-cycle
  // with the fused r.z and beta, direction) read only buffers that stay put
  // from one solve to the next, so the sequence is captured once per operator
  // and x and replayed. Every kernel in it is status-guarded, so a replay
  // past convergence is a no-op, as the launches are. Configuration changes
  // that alter the sequence (tail, dense level, fusion, bfloat16 copies)
  // drop the graph.
  bool graphs = !profiler_attached();
  Graph pcg_graph;
  const Index* graph_rows = nullptr;
  const Index* graph_cols = nullptr;
  const float* graph_vals = nullptr;
  const float* graph_x = nullptr;
  void drop_graphs() {
    pcg_graph.reset();
    graph_rows = graph_cols = nullptr;
    graph_vals = graph_x = nullptr;
  }
  void pcg_iteration(const DeviceCsr& a, float* x) {
    dev.launch(KH_FUSED_SPMV_DOT_ALPHA, n, {a.row_ptr, a.col, a.val, p, q, scalars, status});
    dev.launch(KH_FUSED_STEP_DOT_CHECK, n, {x, r, p, q, scalars, status});
    apply(a, r.data(), z.data(), Tail::DotBeta);
    dev.launch(KH_SOLVER_DIRECTION, n, {z, p, scalars, status});
  }
  void pcg_iteration_replay(const DeviceCsr& a, float* x) {
    if (!pcg_graph || graph_rows != a.row_ptr || graph_cols != a.col || graph_vals != a.val || graph_x != x) {
      drop_graphs();
      pcg_graph = Graph(dev.capture([&] { pcg_iteration(a, x); }));
      graph_rows = a.row_ptr;
      graph_cols = a.col;
      graph_vals = a.val;
      graph_x = x;
    }
    dev.replay(pcg_graph.get());
  }

  // linalg/solver.cpp:271-313
  void pcg(const DeviceCsr& a, float* x, const float* b, const SolveControl& c, double target,
           SolveStats& st) {
    auto restart = [&] {
      reset(st.iterations);
      apply(a, r.data(), z.data(), Tail::None);
      dev.copy(p.data(), z.data(), sizeof(float) * n);
      dot_into(r.data(), z.data(), 0);
    };
    restart();
    int restarts = 0;
    double last = st.initial_residual;
    int interval = batch_interval(c);
    while (st.iterations < c.max_iter) {
      const int batch = std::min(interval, c.max_iter - st.iterations);
      verified_current = false;
      for (int j = 0; j < batch; ++j) {
        if (fused && graphs && st.iterations + j + 1 != c.max_iter) {
          pcg_iteration_replay(a, x);
          continue;
        }
        if (fused) {
          dev.launch(KH_FUSED_SPMV_DOT_ALPHA, n, {a.row_ptr, a.col, a.val, p, q, scalars, status});
          dev.launch(KH_FUSED_STEP_DOT_CHECK, n, {x, r, p, q, scalars, status});
        } else {
          dev.launch(KH_CSR_SPMV_GUARDED, n, {a.row_ptr, a.col, a.val, p, q, status});
          dot_into(p.data(), q.data(), 2);
          dev.launch(KH_SOLVER_PCG_ALPHA, 1, {scalars, status});
          dev.launch(KH_SOLVER_STEP, n, {x, r, p, q, scalars, status});
          dot_into(r.data(), r.data(), 18);
          dev.launch(KH_SOLVER_CHECK, 1, {scalars, status, 1});
        }
        if (st.iterations + j + 1 == c.max_iter) continue;
        apply(a, r.data(), z.data(), Tail::DotBeta);
        dev.launch(KH_SOLVER_DIRECTION, n, {z, p, scalars, status});
      }
      const auto state = poll();
      st.iterations = state[1];
      if (state[0] == 2) break;
      if (state[0] == 1) {
        if (!replacement(a, x, b, target, st, restarts, last) || st.iterations == c.max_iter) break;
        if (st.final_residual <= 10 * target) interval = 1;
        restart();
      }
    }
  }

  // linalg/solver.cpp:314-361, as a resumable loop: the host logic between
  // polls is shared by bicgstab() and the batched driver, which interleaves
  // several systems' batches (KrylovSolver::solve_batched). With the Jacobi
  // preconditioner and fused kernels an iteration is five launches (each with
  // its reduction and scalar update); the first rho and beta after a restart
  // are one more.
  struct BicgRun {
    const DeviceCsr* a = nullptr;
    float* x = nullptr;
    const float* b = nullptr;
    SolveControl c;
    double target = 0;
    SolveStats* st = nullptr;
    int interval = 1, restarts = 0;
    double last = 0;
    bool done = false;
  };
  bool jacobi_fused() const { return fused && !amg; }
  void bicg_restart(const SolveStats& st) {
    reset(st.iterations);
    dev.copy(shadow.data(), r.data(), sizeof(float) * n);
    dev.fill(p.data(), 0.0f, n);
    dev.fill(q.data(), 0.0f, n);
    if (jacobi_fused()) dev.launch(KH_FUSED_DOT_BICG_BETA, n, {shadow, r, scalars, status});
  }
  void bicg_begin(BicgRun& run) {
    bicg_restart(*run.st);
    run.restarts = 0;
    run.last = run.st->initial_residual;
    run.interval = batch_interval(run.c);
    run.done = !(run.st->iterations < run.c.max_iter);
  }
  int bicg_next_batch(const BicgRun& run) {
    verified_current = false;
    return std::min(run.interval, run.c.max_iter - run.st->iterations);
  }
  void bicg_after_poll(BicgRun& run, const std::array<Index, 3>& state) {
    SolveStats& st = *run.st;
    st.iterations = state[1];
    if (state[0] == 2) {
      run.done = true;
      return;
    }
    if (state[0] == 1) {
      if (!replacement(*run.a, run.x, run.b, run.target, st, run.restarts, run.last) ||
          st.iterations == run.c.max_iter) {
        run.done = true;
        return;
      }
      if (st.final_residual <= 10 * run.target) run.interval = 1;
      bicg_restart(st);
    }
    if (!(st.iterations < run.c.max_iter)) run.done = true;
  }
  void bicg_fused_step(const DeviceCsr& a, float* x) {
    dev.launch(KH_FUSED_BICG_DIRECTION, n, {r, q, p, jacobi_inverse, z, scalars, status});
    dev.launch(KH_FUSED_SPMV_SHADOW_ALPHA, n, {a.row_ptr, a.col, a.val, z, q, shadow, scalars, status});
    dev.launch(KH_FUSED_BICG_DIFFERENCE_S, n, {r, q, s, jacobi_inverse, zs, scalars, status});
    dev.launch(KH_FUSED_SPMV_DOT2_OMEGA, n, {a.row_ptr, a.col, a.val, zs, t, s, scalars, status});
    dev.launch(KH_FUSED_BICG_STEP_CHECK_BETA, n, {x, r, z, zs, s, t, shadow, scalars, status});
  }
  void bicg_reference_step(const DeviceCsr& a, float* x) {
    dot_into(shadow.data(), r.data(), 0);
    dev.launch(KH_SOLVER_BICG_BETA, 1, {scalars, status});
    dev.launch(KH_SOLVER_BICG_DIRECTION, n, {r, q, p, scalars, status});
    apply(a, p.data(), z.data(), Tail::None);
    dev.launch(KH_CSR_SPMV_GUARDED, n, {a.row_ptr, a.col, a.val, z, q, status});
    dot_into(shadow.data(), q.data(), 2);
    dev.launch(KH_SOLVER_BICG_ALPHA, 1, {scalars, status});
    dev.launch(KH_SOLVER_BICG_DIFFERENCE, n, {r, q, s, scalars, status});
    dot_into(s.data(), s.data(), 16);
    dev.launch(KH_SOLVER_BICG_S, 1, {scalars, status});
    apply(a, s.data(), zs.data(), Tail::None);
    dev.launch(KH_CSR_SPMV_GUARDED, n, {a.row_ptr, a.col, a.val, zs, t, status});
    dev.reduce_into(KH_INTO_DOT2, t.data(), t.data(), t.data(), s.data(), n, scalars.data(), 2);
    dev.launch(KH_SOLVER_BICG_OMEGA, 1, {scalars, status});
    dev.launch(KH_SOLVER_BICG_STEP, n, {x, r, z, zs, s, t, scalars, status});
    dot_into(r.data(), r.data(), 18);
    dev.launch(KH_SOLVER_CHECK, 1, {scalars, status, 0});
  }
  void bicgstab(const DeviceCsr& a, float* x, const float* b, const SolveControl& c, double target,
                SolveStats& st) {
    BicgRun run;
    run.a = &a;
    run.x = x;
    run.b = b;
    run.c = c;
    run.target = target;
    run.st = &st;
    bicg_begin(run);
    while (!run.done) {
      const int batch = bicg_next_batch(run);
      for (int j = 0; j < batch; ++j) {
        if (jacobi_fused()) bicg_fused_step(a, x);
        else bicg_reference_step(a, x);
      }
      bicg_after_poll(run, poll());
    }
  }
  // The lane of this solver in a batched launch.
  kh_bicg_lane lane(const DeviceCsr& a, float* x) const {
    kh_bicg_lane l{};
    l.row_ptr = a.row_ptr;
    l.col = a.col;
    l.val = a.val;
    l.x = x;
    l.r = r.data();
    l.q = q.data();
    l.p = p.data();
    l.z = z.data();
    l.s = s.data();
    l.t = t.data();
    l.zs = zs.data();
    l.shadow = shadow.data();
    l.inverse = jacobi_inverse.data();
    l.scalars = scalars.data();
    l.status = status.data();
    return l;
  }
  DeviceArray<kh_bicg_lane> batch_table;
  std::vector<kh_bicg_lane> batch_table_host;
  DeviceArray<Index> batch_status;

  // linalg/solver.cpp:97-176, in three parts: the entry (norms, the early
  // exits, limits), the method's loop, and the exit (best-x recovery).
  // solve_begin returns false when no iteration is needed.
  bool solve_begin(const DeviceCsr& a, float* x, const float* b, const SolveControl& c, SolveStats& st,
                   double& target) {
    KA_REQUIRE(a.n_rows == n && a.nnz == nnz, "solver: device or matrix mismatch");
    KA_REQUIRE(x != nullptr && b != nullptr && x != b, "solve: vector size or alias mismatch");
    KA_REQUIRE(c.max_iter >= 0 && std::isfinite(c.rel_tol) && c.rel_tol >= 0 &&
                   std::isfinite(c.abs_tol) && c.abs_tol >= 0 && c.residual_check_interval > 0,
               "solve: invalid control");
    if (!nullspace) residual(a, x, b, r.data());
    ++waits;
    const auto entry = dev.reduce_many({HipDevice::dot(b, b, n), HipDevice::dot(x, x, n),
                                        nullspace ? HipDevice::sum(b, n) : HipDevice::dot(r.data(), r.data(), n)});
    const double bnorm = std::sqrt(entry[0]);
    if (!(std::isfinite(bnorm) && std::isfinite(std::sqrt(entry[1]))))
      throw NonfiniteError("solve: nonfinite input vector");
    st = SolveStats();
    if (nullspace) {
      if (n != 0) {
        KA_REQUIRE(std::abs(entry[2]) <= 1e-6 * std::sqrt(double(n)) * bnorm,
                   "solve: incompatible RHS for constant Neumann nullspace");
        project(x, n, projection.data());
      }
      residual(a, x, b, r.data());
      st.initial_residual = norm(r.data());
    } else st.initial_residual = std::sqrt(entry[2]);
    st.final_residual = st.initial_residual;
    verified_current = true;
    target = std::max(c.abs_tol, c.rel_tol * st.initial_residual);
    if (!std::isfinite(st.initial_residual)) return false;
    if (st.final_residual <= target) {
      st.converged = true;
      return false;
    }
    if (nullspace) project(r.data(), n, projection.data());
    best_residual = st.initial_residual;
    dev.copy(best.data(), x, sizeof(float) * n);
    if (kind != SolverKind::Jacobi) {
      const auto tol = pair_of(target * target);
      const auto div = pair_of(1e6 * st.initial_residual * st.initial_residual);
      dev.launch(KH_SOLVER_LIMITS, 24, {scalars, tol[0], tol[1], div[0], div[1]});
    }
    reset(0);
    return true;
  }
  void solve_end(const DeviceCsr& a, float* x, const float* b, double target, SolveStats& st) {
    if (!verified_current || nullspace) verified(a, x, b, target, st);
    if (!std::isfinite(st.final_residual) || st.final_residual > best_residual) {
      dev.copy(x, best.data(), sizeof(float) * n);
      verified(a, x, b, target, st);
    }
    previous_iterations = st.converged ? st.iterations : 0;
  }
  SolveStats solve(const DeviceCsr& a, float* x, const float* b, const SolveControl& c) {
    SolveStats st;
    double target = 0;
    if (!solve_begin(a, x, b, c, st, target)) return st;
    grid_missed = 0;
    if (grid_rest > 0 && --grid_rest == 0) drop_graphs();
    if (kind == SolverKind::PcgJacobi || kind == SolverKind::AmgPcg) pcg(a, x, b, c, target, st);
    else if (bicg()) bicgstab(a, x, b, c, target, st);
    else if (gmres()) fgmres(a, x, b, c, target, st);
    else jacobi(a, x, b, c, target, st);
    solve_end(a, x, b, target, st);
    return st;
  }

  // linalg/solver.cpp:151-160: damped Jacobi sweeps.
  void jacobi(const DeviceCsr& a, float* x, const float* b, const SolveControl& c, double target,
              SolveStats& st) {
    for (int i = 0; i < c.max_iter; ++i) {
      apply(a, r.data(), z.data(), Tail::None);
      dev.launch(KH_AXPY, n, {x, z, 2.0f / 3.0f});
      verified_current = false;
      ++st.iterations;
      if (st.iterations % c.residual_check_interval == 0 || st.iterations == c.max_iter) {
        if (verified(a, x, b, target, st) || diverged(st)) break;
      } else {
        residual(a, x, b, r.data());
      }
    }
  }

  void refresh(const DeviceCsr& a) {
    KA_REQUIRE(a.n_rows == n && a.nnz == nnz, "solver: device or matrix mismatch");
    if (amg) {
      refresh_amg(a);
    } else {
      dev.launch(KH_KRYLOV_DIAGONAL, n, {a.row_ptr, a.diag, a.val, jacobi_inverse, jacobi_invalid, 0});
      ++waits;
      KA_REQUIRE(dev.reduce_many({HipDevice::max_abs(jacobi_invalid.data(), n)})[0] == 0,
                 "Jacobi: invalid values or zero diagonal");
    }
  }
};

KrylovSolver::KrylovSolver(HipDevice& dev, SolverKind kind, const CsrHost& a, const AmgOptions& options)
    : impl_(std::make_unique<Impl>(dev, kind, a, options)) {}
KrylovSolver::~KrylovSolver() = default;
void KrylovSolver::refresh(const DeviceCsr& a) { impl_->refresh(a); }
SolveStats KrylovSolver::solve(const DeviceCsr& a, float* x, const float* b, const SolveControl& c) {
  return impl_->solve(a, x, b, c);
}
void KrylovSolver::set_fused(bool fused) {
  impl_->drop_graphs();
  impl_->fused = fused;
}
void KrylovSolver::set_graphs(bool on) {
  impl_->drop_graphs();
  impl_->graphs = on && !profiler_attached();
}
bool KrylovSolver::graphs_enabled() const { return impl_->graphs; }

// Several BiCGStab-Jacobi solves in lockstep: each lane keeps its own entry,
// batches, polls, replacements and exit, and its iterations run as lanes of
// the KH_BATCH_* launches, so its iterates are bitwise those of its own
// solve(). A round launches the common part of the active lanes' batches;
// the lanes whose batch ends are polled with one wait.
std::vector<SolveStats> KrylovSolver::solve_batched(const std::vector<KrylovSolver*>& solvers,
                                                    const std::vector<DeviceCsr>& a, const std::vector<float*>& x,
                                                    const std::vector<const float*>& b, const SolveControl& c) {
  const std::size_t lanes = solvers.size();
  KA_REQUIRE(lanes >= 1 && lanes <= KH_BATCH_MAX_LANES && a.size() == lanes && x.size() == lanes &&
                 b.size() == lanes,
             "batched solve: 1 to " + std::to_string(KH_BATCH_MAX_LANES) + " systems with one operator, x and b each");
  Impl& first = *solvers[0]->impl_;
  for (std::size_t k = 0; k < lanes; ++k) {
    const Impl& I = *solvers[k]->impl_;
    KA_REQUIRE(I.kind == SolverKind::BicgstabJacobi && I.jacobi_fused(),
               "batched solve: needs fused BiCGStab-Jacobi solvers");
    KA_REQUIRE(&I.dev == &first.dev && I.n == first.n, "batched solve: solvers of one device and size");
    for (std::size_t j = 0; j < k; ++j) KA_REQUIRE(solvers[j] != solvers[k], "batched solve: a solver twice");
  }
  HipDevice& dev = first.dev;
  const Index n = first.n;
  std::vector<SolveStats> stats(lanes);
  std::vector<double> targets(lanes, 0.0);
  std::vector<Impl::BicgRun> runs(lanes);
  std::vector<bool> iterate(lanes, false);
  for (std::size_t k = 0; k < lanes; ++k) {
    Impl& I = *solvers[k]->impl_;
    iterate[k] = I.solve_begin(a[k], x[k], b[k], c, stats[k], targets[k]);
    if (!iterate[k]) continue;
    auto& run = runs[k];
    run.a = &a[k];
    run.x = x[k];
    run.b = b[k];
    run.c = c;
    run.target = targets[k];
    run.st = &stats[k];
    I.bicg_begin(run);
  }
  std::vector<kh_bicg_lane> table(lanes);
  for (std::size_t k = 0; k < lanes; ++k) table[k] = solvers[k]->impl_->lane(a[k], x[k]);
  const bool same = first.batch_table_host.size() == lanes &&
                    std::memcmp(first.batch_table_host.data(), table.data(), lanes * sizeof(kh_bicg_lane)) == 0;
  if (!same) {
    first.batch_table = to_device(dev, table);
    first.batch_table_host = table;
  }
  if (first.batch_status.size() != 3 * lanes) first.batch_status = DeviceArray<Index>(dev, 3 * lanes);
  std::vector<int> remaining(lanes, 0);
  while (true) {
    int mask = 0, steps = 0;
    for (std::size_t k = 0; k < lanes; ++k) {
      if (!iterate[k] || runs[k].done) continue;
      if (remaining[k] == 0) remaining[k] = solvers[k]->impl_->bicg_next_batch(runs[k]);
      if (remaining[k] <= 0) continue;
      mask |= 1 << k;
      steps = steps == 0 ? remaining[k] : std::min(steps, remaining[k]);
    }
    if (mask == 0) break;
    const int count = int(lanes);
    for (int j = 0; j < steps; ++j) {
      dev.launch(KH_BATCH_BICG_DIRECTION, n, {first.batch_table, count, mask});
      dev.launch(KH_BATCH_SPMV_SHADOW_ALPHA, n, {first.batch_table, count, mask});
      dev.launch(KH_BATCH_BICG_DIFFERENCE_S, n, {first.batch_table, count, mask});
      dev.launch(KH_BATCH_SPMV_DOT2_OMEGA, n, {first.batch_table, count, mask});
      dev.launch(KH_BATCH_BICG_STEP_CHECK_BETA, n, {first.batch_table, count, mask});
    }
    std::vector<std::size_t> polled;
    for (std::size_t k = 0; k < lanes; ++k) {
      if (((mask >> k) & 1) == 0) continue;
      remaining[k] -= steps;
      if (remaining[k] == 0) polled.push_back(k);
    }
    for (std::size_t k : polled)
      dev.copy(first.batch_status.data() + 3 * k, solvers[k]->impl_->status.data(), 3 * sizeof(Index));
    ++first.waits;
    const auto host = first.batch_status.download();
    for (std::size_t k : polled)
      solvers[k]->impl_->bicg_after_poll(runs[k], {host[3 * k], host[3 * k + 1], host[3 * k + 2]});
  }
  for (std::size_t k = 0; k < lanes; ++k)
    if (iterate[k]) solvers[k]->impl_->solve_end(a[k], x[k], b[k], targets[k], stats[k]);
  return stats;
}
int KrylovSolver::set_tail(int first) {
  const int previous = impl_->tail_request;
  impl_->tail_request = first;
  if (first < 0) {
    impl_->grid_request = -1;
    impl_->grid_asked = false;
  }
  try {
    impl_->plan_tail();
  } catch (...) {
    impl_->tail_request = previous;
    impl_->plan_tail();
    throw;
  }
  return impl_->tail_first;
}
int KrylovSolver::tail_level() const { return impl_->tail_first; }
int KrylovSolver::grid_level() const { return impl_->grid_level(); }
int KrylovSolver::set_grid(int first, int limit_us) {
  Impl& I = *impl_;
  KA_REQUIRE(limit_us >= 0, "AMG: the multi-workgroup cycle's wait must not be negative");
  if (first > 0) {
    GridPlan plan;
    KA_REQUIRE(I.plan_grid_at(std::size_t(first), plan),
               "AMG: levels from " + std::to_string(first) + " do not fit the multi-workgroup cycle");
  }
  I.grid_request = first;
  I.grid_asked = first > 0;
  I.grid_off = first == 0;
  I.grid_limit_us = limit_us;
  if (first != 0) I.tail_request = -1;
  I.plan_tail();
  return I.grid_level();
}
std::array<Index, 3> KrylovSolver::grid_report() const {
  const auto host = impl_->status.download();
  const Index* report = host.data() + 3;
  return {report[KH_GRID_REPORT_TOGETHER], report[KH_GRID_REPORT_ALONE], report[KH_GRID_REPORT_GIVEN_UP]};
}
void KrylovSolver::set_grid_polls(int polls) {
  KA_REQUIRE(polls >= 0, "AMG: the polls of the multi-workgroup cycle's barriers must not be negative");
  impl_->set_grid_polls(polls);
}

// The coarse-tail autotuner (no reference counterpart): times `repeats`
// V-cycles for each admissible first level of the tail, and for none, keeps
// the fastest and returns it (-1: the multi-workgroup cycle, timed beside it
// unless the caller turned it off). Every choice gives bitwise the same iterates
// (the tail computes each row as the per-level launches do), so it picks
// only the launch structure: per-level launches are latency-bound below a
// few thousand rows, the one-workgroup tail is compute-bound on one CU, and
// where they cross depends on the hierarchy.
int KrylovSolver::autotune_tail(const DeviceCsr& a, int repeats) {
  Impl& I = *impl_;
  KA_REQUIRE(I.amg && I.fused, "autotune: needs a fused AMG solver");
  KA_REQUIRE(repeats >= 1, "autotune: repeats must be positive");
  KA_REQUIRE(a.n_rows == I.n && a.nnz == I.nnz, "solver: device or matrix mismatch");
  if (I.direct_level > 0) return 0;  // the dense level replaces the tail
  std::vector<int> candidates{0};
  for (std::size_t i = 1; i < I.levels.size(); ++i)
    if (I.tail_fits(i)) candidates.push_back(int(i));
  DeviceArray<float> v(I.dev, I.n), out(I.dev, I.n);
  I.dev.fill(v.data(), 1.0f, I.n);
  // Where PCG iterations are replayed from graphs, each candidate is timed
  // the same way (captured once, replayed), so launch-bound forms are priced
  // as the solve will run them.
  const bool replayed = I.graphs && I.kind == SolverKind::AmgPcg;
  // Where a form is timed alone (restriction, sweep) or decides a large part
  // of the cycle (coarsest level, tail), a later form replaces an earlier
  // one (the first being the default) only when at least 3% faster: forms
  // within timing noise of each other would otherwise flip from run to run.
  constexpr double kKeep = 0.97;
  // The fastest of three timed batches of `repeats` runs, so that one
  // disturbed batch does not decide a form.
  // Under replay the `repeats` runs are captured into one graph, so each run
  // is priced by its launches inside a graph (one replay's own overhead is
  // shared by all of them).
  const auto seconds = [&](const std::function<void()>& body) {
    body();
    I.dev.synchronize();
    Graph graph;
    if (replayed)
      graph = Graph(I.dev.capture([&] {
        for (int k = 0; k < repeats; ++k) body();
      }));
    double best = 0;
    for (int trial = 0; trial < 3; ++trial) {
      const auto t0 = std::chrono::steady_clock::now();
      if (replayed) {
        I.dev.replay(graph.get());
      } else {
        for (int k = 0; k < repeats; ++k) body();
      }
      I.dev.synchronize();
      const double t = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      best = trial == 0 ? t : std::min(best, t);
    }
    return best;
  };
  const int requested = I.tail_request;
  // Restriction form per level: time each form on the level's current data
  // (left by one V-cycle) and keep the fastest. Every form gives the same bits.
  I.tail_request = 0;
  I.plan_tail();
  I.reset(0);
  I.apply(a, v.data(), out.data(), Tail::None);
  for (std::size_t i = 0; i + 1 < I.levels.size(); ++i) {
    Level& l = I.levels[i];
    if (I.bf16_level(l)) continue;
    const DeviceCsr li = i == 0 ? a : l.matrix.view();
    const DeviceCsr ci = I.levels[i + 1].matrix.view();
    const float* xin = i == 0 ? out.data() : l.x.data();
    const float* bin = i == 0 ? v.data() : l.b.data();
    float* spare = l.r.data();
    DeviceArray<float> coarse(I.dev, ci.n_rows);
    double best_form = 0;
    const int forms = l.max_row > KH_WIDE_ROW ? 4 : 3;
    for (int mode = 0; mode < forms; ++mode) {
      const double t =
          seconds([&] { I.restrict_level(l, li, ci, xin, bin, spare, coarse.data(), mode, I.status.data()); });
      if (mode == 0 || t < kKeep * best_form) {
        best_form = t;
        l.restrict_mode = mode;
      }
    }
  }
  // Sweep form per level with long rows: time plain sweeps of each form on
  // the level's current data. Every form gives the same bits.
  for (std::size_t i = 0; i < I.levels.size(); ++i) {
    Level& l = I.levels[i];
    if (I.bf16_level(l) || l.max_row <= KH_WIDE_ROW) continue;
    const DeviceCsr li = i == 0 ? a : l.matrix.view();
    const float* xin = i == 0 ? out.data() : l.x.data();
    const float* bin = i == 0 ? v.data() : l.b.data();
    double thread_form = 0;
    for (int mode = 0; mode < 2; ++mode) {
      l.sweep_mode = mode;
      const kh_kernel k = I.smooth_kernel(l);
      const double t = seconds([&] {
        I.dev.launch(k, li.n_rows, {li.row_ptr, li.col, li.val, xin, bin, l.l1, l.r, I.status.data()});
      });
      if (mode == 0) thread_form = t;
      else l.sweep_mode = t < kKeep * thread_form ? 1 : 0;
    }
  }
  // Prolongation form per level: time whole V-cycles with each of the
  // level's forms in turn (alone, a form runs on cache-warm data and the
  // in-place form changes the level's iterate; inside the cycle the
  // comparison is the one the solve sees) and keep the fastest. One level's
  // difference is a percent or two of a cycle, so no margin applies here.
  // Every form gives the same bits.
  for (std::size_t i = 0; i + 1 < I.levels.size(); ++i) {
    Level& l = I.levels[i];
    if (I.bf16_level(l)) continue;
    double fastest = 0;
    int pick = 0;
    const int forms = l.max_row > KH_WIDE_ROW ? 3 : 2;
    for (int mode = 0; mode < forms; ++mode) {
      l.prolong_mode = mode;
      I.reset(0);
      const double t = seconds([&] { I.apply(a, v.data(), out.data(), Tail::None); });
      if (mode == 0 || t < fastest) {
        fastest = t;
        pick = mode;
      }
    }
    l.prolong_mode = pick;
  }
  // The coarsest level's sweeps: launch by launch, in one workgroup or, where
  // the level has a resident partition, in one that reads the operator once.
  if (I.coarse_sweeps_fit(I.levels.size() - 1)) {
    double fastest = 0;
    int pick = 0;
    const int forms = I.levels.back().resident_cap > 0 ? 3 : 2;
    for (int mode = 0; mode < forms; ++mode) {
      I.coarse_sweeps_mode = mode;
      I.reset(0);
      const double t = seconds([&] { I.apply(a, v.data(), out.data(), Tail::None); });
      if (mode == 0 || t < kKeep * fastest) {
        fastest = t;
        pick = mode;
      }
    }
    I.coarse_sweeps_mode = pick;
  }
  const int previous = requested;
  int best = previous;
  double best_s = 0;
  for (int first : candidates) {
    I.tail_request = first;
    I.plan_tail();
    I.reset(0);
    const double secs = seconds([&] { I.apply(a, v.data(), out.data(), Tail::None); });
    if (best_s == 0 || secs < kKeep * best_s) {
      best_s = secs;
      best = first;
    }
  }
  // The multi-workgroup cycle from each level whose plan fits, in the tail's place.
  int best_grid = 0;
  for (std::size_t i = 1; i < I.levels.size(); ++i) {
    if (I.grid_off || !I.grid_allowed(i)) continue;
    I.tail_request = -1;
    I.grid_request = int(i);
    I.plan_tail();
    if (I.grid_first == 0 || !I.grid_spread) continue;
    I.reset(0);
    const double secs = seconds([&] { I.apply(a, v.data(), out.data(), Tail::None); });
    if (secs < kKeep * best_s) {
      best_s = secs;
      best = -1;
      best_grid = int(i);
    }
  }
  I.poll();
  I.grid_asked = false;
  I.grid_request = best_grid;
  I.tail_request = best;
  I.plan_tail();
  return I.grid_level() > 0 ? -1 : I.tail_first;
}
int KrylovSolver::host_waits() const { return impl_->waits; }
int KrylovSolver::set_direct(Index rows) { return impl_->set_direct(rows); }
void KrylovSolver::set_dense_tolerance(double tolerance) {
  KA_REQUIRE(std::isfinite(tolerance) && tolerance >= 0, "AMG: the dense refresh tolerance must be finite and >= 0");
  impl_->dense_tolerance = tolerance;
  if (tolerance == 0) impl_->dense_basis = DeviceArray<float>();
}
void KrylovSolver::dense_refreshes(long* inversions, long* skips, double* staleness) const {
  *inversions = impl_->dense_inversions;
  *skips = impl_->dense_skips;
  *staleness = impl_->dense_staleness;
}
void KrylovSolver::set_coarse_bf16(bool on) { impl_->set_coarse_bf16(on); }
void KrylovSolver::set_learned(int level, int layers, std::uint64_t seed, int capacity) {
  impl_->set_learned(level, layers, seed, capacity);
}
void KrylovSolver::set_learned_mode(int mode, double reduction, double max_relative) {
  KA_REQUIRE(mode >= 0 && mode <= 2, "learned stage: mode must be 0 (off), 1 (harvest) or 2 (apply)");
  KA_REQUIRE(mode == 0 || impl_->learned != nullptr, "learned stage: not configured");
  KA_REQUIRE(std::isfinite(reduction) && reduction >= 0 && reduction < 1,
             "learned stage: reduction per step must be in [0, 1)");
  KA_REQUIRE(!std::isnan(max_relative) && max_relative > 0,
             "learned stage: the largest unexplained fraction must be positive");
  impl_->learned_mode = mode;
  impl_->learned_reduction = reduction;
  impl_->learned_max_relative = max_relative;
}
int KrylovSolver::learned_targets(double rel_tol) { return impl_->learned_targets(rel_tol); }
TrainResult KrylovSolver::learned_train(int steps, float lr, int pairs) {
  return impl_->learned_train(steps, lr, pairs);
}
double KrylovSolver::learned_evaluate(int first, int count) { return impl_->learned_evaluate(first, count); }
LearnedReport KrylovSolver::learned_report() const {
  const auto& i = *impl_;
  LearnedReport r;
  r.level = i.learned_level;
  r.rows = i.learned ? i.levels[i.learned_level].rows : 0;
  r.mode = i.learned_mode;
  r.harvested = i.harvested;
  r.targets = i.targeted;
  r.applications = i.learned_applications;
  r.fallbacks = i.learned_fallbacks;
  r.solves = i.learned_solves;
  r.gated = i.learned_gated;
  r.last_loss = i.learned_loss;
  r.relative = i.learned_relative;
  return r;
}
std::vector<float> KrylovSolver::learned_parameters() const {
  KA_REQUIRE(impl_->learned != nullptr, "learned stage: not configured");
  return impl_->learned->parameters();
}
void KrylovSolver::set_learned_parameters(const std::vector<float>& theta) {
  KA_REQUIRE(impl_->learned != nullptr, "learned stage: not configured");
  impl_->learned->set_parameters(theta);
}
void KrylovSolver::set_restart(int m) {
  KA_REQUIRE(m >= 1 && m <= 63, "FGMRES: restart length must be in [1, 63]");
  impl_->restart_length = m;
}

// linalg/amg.cpp:263-269, linalg/solver.cpp:178-184
std::string KrylovSolver::describe() const {
  std::ostringstream out;
  const bool pcg = impl_->kind == SolverKind::PcgJacobi || impl_->kind == SolverKind::AmgPcg;
  out << (impl_->kind == SolverKind::Jacobi ? "damped Jacobi"
          : pcg                             ? "PCG"
          : impl_->gmres()                  ? "FGMRES(" + std::to_string(impl_->restart_length) + ")"
                                            : "BiCGStab")
      << ", ";
  if (impl_->amg)
    out << "aggregation AMG " << (impl_->options.cycle == AmgCycle::K ? 'K' : 'V') << "-cycle, "
        << impl_->levels.size() << " levels, op complexity "
        << std::fixed << std::setprecision(3) << impl_->complexity;
  else out << "Jacobi";
  if (impl_->nullspace) out << ", constant-nullspace projection";
  if (impl_->direct_level > 0)
    out << ", FP64 dense solve of level " << impl_->direct_level << " ("
        << impl_->levels[impl_->direct_level].rows << " rows)";
  if (impl_->coarse_bf16) out << ", bfloat16 coarse-level values";
  if (impl_->learned && impl_->learned_mode == 2)
    out << ", learned correction on level " << impl_->learned_level << " ("
        << impl_->levels[impl_->learned_level].rows << " rows)";
  return out.str();
}
void KrylovSolver::set_plan(int restrict_mode, int coarse_sweeps, int prolong_mode, int sweep_mode) {
  KA_REQUIRE(restrict_mode >= -1 && restrict_mode <= 3 && coarse_sweeps >= -1 && coarse_sweeps <= 2 &&
                 prolong_mode >= -1 && prolong_mode <= 2 && sweep_mode >= -1 && sweep_mode <= 1,
             "solver plan: restriction form -1..3, coarsest sweeps -1..2, prolongation form -1..2, sweep form "
             "-1..1");
  impl_->drop_graphs();
  if (restrict_mode >= 0)
    for (auto& l : impl_->levels) l.restrict_mode = restrict_mode;
  if (prolong_mode >= 0)
    for (auto& l : impl_->levels) l.prolong_mode = prolong_mode;
  if (sweep_mode >= 0)
    for (auto& l : impl_->levels) l.sweep_mode = sweep_mode;
  // Form 2 needs the level's resident partition; without one the level
  // runs form 1, the same bits.
  if (coarse_sweeps >= 0) impl_->coarse_sweeps_mode = coarse_sweeps;
}
std::string KrylovSolver::plan() const {
  std::ostringstream out;
  const auto& L = impl_->levels;
  out << "restriction per level";
  for (std::size_t i = 0; i + 1 < L.size(); ++i)
    out << (i ? "," : " ")
        << (L[i].restrict_mode == 3   ? "split-wave"
            : L[i].restrict_mode == 2 ? "split"
            : L[i].restrict_mode == 1 ? "wide"
                                      : "fused");
  out << "; prolongation per level";
  for (std::size_t i = 0; i + 1 < L.size(); ++i)
    out << (i ? "," : " ")
        << (L[i].prolong_mode == 2 ? "fused-wave" : L[i].prolong_mode == 1 ? "split" : "fused");
  if (!L.empty() && impl_->coarse_sweeps_fit(L.size() - 1))
    out << "; coarsest level "
        << (impl_->coarse_sweeps_mode == 0                                      ? "sweep launches"
            : impl_->coarse_sweeps_mode == 2 && L.back().resident_cap > 0 ? "register-resident sweeps"
                                                                            : "one-workgroup sweeps");
  if (!impl_->grid_on()) out << "; tail from level " << impl_->tail_first;
  if (impl_->grid_level() > 0) {
    const GridPlan& g = impl_->grid_plan;
    out << (impl_->grid_on() ? "; " : ", ") << "multi-workgroup cycle from level " << impl_->grid_first << " (" << g.parts << " workgroups, " << g.grid
        << " of " << g.count << " levels shared, row sums";
    for (int k = 0; k < g.count; ++k) out << (k ? "," : " ") << (g.table[std::size_t(k)].mode ? "split" : "whole");
    out << ")";
    if (impl_->grid_rest > 0) out << " resting for " << impl_->grid_rest - 1 << " more solves";
  }
  out << "; longest row per level";
  for (std::size_t i = 0; i < L.size(); ++i) out << (i ? "," : " ") << L[i].max_row;
  out << "; sweeps per level";
  for (std::size_t i = 0; i < L.size(); ++i)
    out << (i ? "," : " ")
        << (impl_->smooth_kernel(L[i]) == KH_AMG_SMOOTH_ROWWAVE ? "wave"
            : impl_->smooth_kernel(L[i]) == KH_AMG_SMOOTH_WIDE  ? "wide"
                                                                 : "thread");
  return out.str();
}
std::vector<std::pair<Index, Index>> KrylovSolver::levels() const {
  std::vector<std::pair<Index, Index>> out;
  for (const auto& l : impl_->levels) out.emplace_back(l.rows, l.nnz);
  return out;
}
std::vector<Index> KrylovSolver::transfer(std::size_t level, int which) const {
  if (level >= impl_->levels.size() || !impl_->levels[level].has_transfer) return {};
  const auto& l = impl_->levels[level];
  const DeviceArray<Index>& a = which == 0 ? l.aggregate : which == 1 ? l.member_offsets
      : which == 2 ? l.members : which == 3 ? l.entry_offsets : l.entries;
  return a.download();
}
std::vector<float> KrylovSolver::level_values(std::size_t level) const {
  if (level == 0 || level >= impl_->levels.size()) return {};
  return impl_->levels[level].matrix.val.download();
}

}  // namespace kutta_amd
