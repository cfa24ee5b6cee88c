"""The multi-workgroup V-cycle (KH_GRID_CYCLE) against the per-level launches
it replaces: bitwise-identical iterates, iteration counts and residuals from
every admissible first level, through graph replays and direct launches, with
its workgroups together and with one working alone (a wait of zero), on
hierarchies that end in the few-row coarse solve, in coarse sweeps, and in
levels too large for the one-workgroup part. Both ways give the same bits, so
which of them ran is read from the cycle's own counts, and which forms a plan
has from plan(): each case states those it is there for."""
import ctypes as C
import re

import numpy as np
import pytest

import kutta_amd
import oracle
from kutta_amd import AmgCycle, AmgOptions, OperatorStructure, SolveControl, SolverKind

pytestmark = pytest.mark.gpu
M = OperatorStructure.SymmetricMMatrix

# Last, the forms of a case's plans: workgroups, "bottom" (levels the first workgroup
# does alone) or "shared" (no such level), and how rows are summed ("split":
# products first; "whole": entry by entry, above 512 rows a workgroup).
CASES = [
    ("poisson V(5,5)", lambda: oracle.poisson(30, 28, 26), SolverKind.AmgPcg, AmgOptions(), "16 bottom split"),
    ("ragged rows V(2,2)", lambda: oracle.poisson(33, 31, 29, 1.0, random=True), SolverKind.AmgPcg,
     AmgOptions(pre_sweeps=2, post_sweeps=2, aggregation_passes=2), "16 shared split"),
    ("V(1,1)", lambda: oracle.poisson(23, 21, 19), SolverKind.AmgPcg, AmgOptions(pre_sweeps=1, post_sweeps=1),
     "16 bottom split"),
    ("pressure, coarse sweeps", lambda: oracle.pressure_problem(18, 17, 16).csr(), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=2, coarse_rows=400, structure=M), "16 bottom split"),
    ("pressure, stalled coarse levels", lambda: oracle.pressure_problem(24, 23, 22).csr(), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=2, structure=M), "16 32 bottom split whole"),
    ("anisotropic, pair aggregates", lambda: oracle.poisson(32, 32, 32, 100), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=1, max_levels=4), "16 shared split whole"),
    ("bicgstab V(2,3)", lambda: oracle.poisson(52, 47, 1, 1.0, wind=2.0), SolverKind.AmgBicgstab,
     AmgOptions(pre_sweeps=2, post_sweeps=3, aggregation_passes=2), "16 bottom split"),
    ("K-cycle", lambda: oracle.pressure_problem(20, 19, 18).csr(), SolverKind.AmgPcg,
     AmgOptions(pre_sweeps=1, post_sweeps=1, coarse_sweeps=4, aggregation_passes=2, structure=M, cycle=AmgCycle.K,
                k_min_rows=5000), "16 bottom split"),
]


@pytest.mark.parametrize("name,make,kind,opts,forms", CASES, ids=[c[0] for c in CASES])
def test_grid_cycle_matches_level_launches(device, name, make, kind, opts, forms):
    a = make()
    host = kutta_amd.CsrMatrixHost(a.row_ptr, a.col, a.diag, a.val)
    matrix = kutta_amd.upload(device, host)
    solver = kutta_amd.make_amg_solver(kind, device, host, opts)
    solver.refresh(matrix)
    b = np.random.default_rng(31).standard_normal(a.n_rows).astype(np.float32)
    rhs = device.upload(b)
    print(f"[grid] {name}: levels {[r for r, _ in solver.levels()]}", flush=True)

    def run():
        x = device.alloc(a.n_rows)
        x.fill(np.float32(0))
        st = solver.solve(matrix, x, rhs, SolveControl(1e-6, 0.0, 300))
        return st, x.download()

    solver.set_tail(0)
    st0, x0 = run()
    assert "multi-workgroup" not in solver.plan()
    seen = set()
    for first in range(1, len(solver.levels())):
        try:
            assert solver.set_grid(first) == first
        except kutta_amd.KuttaError:
            continue
        for graphs, limit in ((True, 2000), (False, 2000), (True, 0)):
            print(f"[grid] {name}: from level {first}, graphs {graphs}, wait {limit} us", flush=True)
            solver.set_graphs(graphs)
            solver.set_grid(first, limit)
            assert f"multi-workgroup cycle from level {first}" in solver.plan()
            before = solver.grid_report()
            for _ in range(2):
                st, x = run()
                assert (st.iterations, st.final_residual) == (st0.iterations, st0.final_residual)
                assert np.array_equal(x.view(np.uint32), x0.view(np.uint32))
            ran = {k: v - before[k] for k, v in solver.grid_report().items()}
            assert ran["given_up"] == 0
            if limit > 0:
                assert ran["together"] >= st0.iterations and ran["alone"] == 0
            else:
                assert ran["alone"] > 0
        plan = re.search(r"\((\d+) workgroups, (\d+) of (\d+) levels shared, row sums ([a-z,]+)\)", solver.plan())
        seen |= {plan.group(1), "shared" if plan.group(2) == plan.group(3) else "bottom", *plan.group(4).split(",")}
    assert seen == set(forms.split())


def test_grid_cycle_follows_new_values_and_limits(device):
    """The plan holds patterns only: after the values change and a refresh the
    cycle is the new operator's. Levels that do not fit are refused, and a
    fixed tail turns the cycle off."""
    p = oracle.pressure_problem(18, 17, 16).csr()
    host = kutta_amd.CsrMatrixHost(p.row_ptr, p.col, p.diag, p.val)
    matrix = kutta_amd.upload(device, host)
    opts = AmgOptions(aggregation_passes=2, structure=M)
    solver = kutta_amd.make_amg_solver(SolverKind.AmgPcg, device, host, opts)
    auto = solver.set_grid(-1)
    assert auto >= 1
    with pytest.raises(kutta_amd.KuttaError):
        solver.set_grid(len(solver.levels()) + 2)
    assert solver.set_grid(-1) == auto
    scaled = (p.val * 1.7).astype(np.float32)
    matrix.val.upload(scaled)
    solver.refresh(matrix)
    b = device.upload(np.random.default_rng(2).standard_normal(p.n_rows).astype(np.float32))
    out = []
    for tail in (-1, 0):
        solver.set_tail(tail)
        assert ("multi-workgroup" in solver.plan()) == (tail < 0)
        x = device.alloc(p.n_rows)
        x.fill(np.float32(0))
        solver.solve(matrix, x, b, SolveControl(1e-6, 0.0, 300))
        out.append(x.download())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_a_barrier_that_gives_up_is_an_error(device):
    """With no polls at all the first workgroup at a barrier gives up: every
    launch still ends, the solve raises, and the cycle is off. Asked for again,
    with its polls back, it gives the bits it gave before."""
    p = oracle.pressure_problem(18, 17, 16).csr()
    host = kutta_amd.CsrMatrixHost(p.row_ptr, p.col, p.diag, p.val)
    matrix = kutta_amd.upload(device, host)
    solver = kutta_amd.make_amg_solver(SolverKind.AmgPcg, device, host, AmgOptions(aggregation_passes=2, structure=M))
    solver.refresh(matrix)
    b = device.upload(np.random.default_rng(5).standard_normal(p.n_rows).astype(np.float32))

    def run():
        x = device.alloc(p.n_rows)
        x.fill(np.float32(0))
        solver.solve(matrix, x, b, SolveControl(1e-6, 0.0, 300))
        return x.download().view(np.uint32)

    want = run()
    assert "multi-workgroup" in solver.plan()
    for graphs in (True, False):
        solver.set_graphs(graphs)
        solver.set_grid_polls(0)
        with pytest.raises(kutta_amd.KuttaError, match="gave up"):
            run()
        assert "multi-workgroup" not in solver.plan()
        assert np.array_equal(run(), want)
        solver.set_grid_polls()
        assert solver.set_grid(-1) >= 1
        assert np.array_equal(run(), want)


def test_a_cycle_that_does_not_meet_rests(device):
    """Picked automatically and given no time to meet, the cycle is worked
    alone until the solve's next poll and then left off, for that solve and the
    next 256; then it is tried again. Asked for by level it stays. Always the
    same bits."""
    a = oracle.poisson(17, 16, 15)
    host = kutta_amd.CsrMatrixHost(a.row_ptr, a.col, a.diag, a.val)
    matrix = kutta_amd.upload(device, host)
    solver = kutta_amd.make_amg_solver(SolverKind.AmgPcg, device, host, AmgOptions(pre_sweeps=1, post_sweeps=1))
    solver.refresh(matrix)
    b = device.upload(np.random.default_rng(8).standard_normal(a.n_rows).astype(np.float32))

    def run():
        x = device.alloc(a.n_rows)
        x.fill(np.float32(0))
        assert solver.solve(matrix, x, b, SolveControl(1e-6, 0.0, 300)).iterations > 8  # more than one poll
        return x.download().view(np.uint32), solver.grid_report()

    first = solver.set_grid(-1)
    want, report = run()
    assert first >= 1 and report["together"] > 8 and report["alone"] == 0
    solver.set_grid(-1, 0)
    for k in range(3):
        got, before = run()
        assert np.array_equal(got, want)
        assert f"resting for {256 - k} more solves" in solver.plan()
        assert before["alone"] >= 3 and before["together"] == report["together"]
    for _ in range(254):
        got, after = run()
        assert after == before
    assert "resting for 0 more solves" in solver.plan() and np.array_equal(got, want)
    got, after = run()
    assert after["alone"] > before["alone"] and np.array_equal(got, want)
    assert "resting for 256 more solves" in solver.plan()
    solver.set_grid(first, 0)
    for _ in range(2):
        before = after
        got, after = run()
        assert after["alone"] > before["alone"] + 8 and np.array_equal(got, want)
    assert "resting" not in solver.plan()


def test_the_tuner_says_what_it_chose(device):
    """autotune_tail returns -1 exactly where it chose the cycle, and that given
    to set_tail chooses it again; a cycle turned off by the caller is neither
    tuned in nor brought back by the automatic tail."""
    a = oracle.poisson(30, 28, 26)
    host = kutta_amd.CsrMatrixHost(a.row_ptr, a.col, a.diag, a.val)
    matrix = kutta_amd.upload(device, host)
    solver = kutta_amd.make_amg_solver(SolverKind.AmgPcg, device, host, AmgOptions())
    solver.refresh(matrix)
    tail = solver.set_tail(-1)
    assert tail >= 1 and solver.grid_level >= 1 and f"tail from level {tail}" not in solver.plan()
    for _ in range(2):
        chosen = solver.autotune_tail(matrix, 2)
        assert (chosen == -1) == (solver.grid_level > 0) == ("multi-workgroup" in solver.plan())
        kept = solver.grid_level
        if kept:
            assert solver.set_grid(kept) == kept
        assert solver.set_tail(chosen) == (tail if chosen < 0 else chosen)
        assert (solver.grid_level > 0) == (kept > 0)
        solver.set_tail(0)  # the tuner times the cycle again after a tail was set
    assert solver.set_grid(0) == 0
    assert solver.autotune_tail(matrix, 2) >= 0
    assert solver.grid_level == 0 and "multi-workgroup" not in solver.plan()
    assert solver.set_tail(-1) == tail and solver.grid_level == 0
    assert f"tail from level {tail}" in solver.plan()
    first = solver.set_grid(-1)
    assert first >= 1
    solver.set_coarse_bf16(True)  # the cycle has no such form: the tail runs
    assert solver.grid_level == 0 and "multi-workgroup" not in solver.plan()
    assert f"tail from level {tail}" in solver.plan()
    solver.set_coarse_bf16(False)
    assert solver.grid_level == first


class Level(C.Structure):
    _fields_ = [(k, C.c_void_p) for k in ("row_ptr", "col", "val", "inverse", "member_offsets", "members", "aggregate",
                                          "place", "slot", "local_col", "x", "w", "b")] + [
                (k, C.c_int32) for k in ("rows", "pad")]


class Part(C.Structure):
    _fields_ = [(k, C.c_int32) for k in ("first", "rows", "window", "window_rows", "slot0", "slots", "mode", "lds",
                                         "terms", "iterates")]


def one_level_plan(row_ptr, col, parts):
    """KH_GRID_CYCLE's tables for one shared level, as kutta_hip.h states them."""
    n = len(row_ptr) - 1
    place, slot, local, table = np.zeros(n, np.uint16), [], [], []
    for p in range(parts):
        first, last = n * p // parts, n * (p + 1) // parts
        cols = col[row_ptr[first]:row_ptr[last]]
        low, high = min(first, cols.min()), max(last, cols.max() + 1)
        slot0 = len(slot)
        for i in range(first, last):
            entries = list(range(row_ptr[i], row_ptr[i + 1]))
            chunks = (len(entries) + 3) // 4
            pad = 4 * (chunks | 1 if chunks > 3 else chunks) - len(entries)
            place[i] = len(slot) - slot0
            slot += entries + [-1] * pad
            local += [col[j] - low for j in entries] + [0xffff] * pad
        table.append(Part(first, last - first, low, high - low, slot0, len(slot) - slot0, 1))
    window = (max(t.window_rows for t in table) + 3) // 4 * 4
    base = window + 2 * max(t.slots for t in table)
    for t in table:
        t.terms, t.lds = window, base
    words = base + max(t.slots + t.slots // 2 + 3 * t.rows for t in table)
    assert words <= 39936 and all(t.slots % 4 == 0 and t.window_rows < 0xffff for t in table)
    return place, np.array(slot, np.int32), np.array(local, np.uint16), table, (words + 3) // 4 * 4


@pytest.mark.parametrize("parts", [1, 2, 5, 16, 32])
def test_launch_with_and_without_workgroups_on_the_home_xcd(device, parts):
    """The launch by itself on one level, five sweeps: its workgroups together,
    and, with a home that no XCD has, one of them alone from the first launch
    on, without a wait and without counters. Both as the sweeps' own launches."""
    a = oracle.poisson(11, 10, 9, 1.0, random=True)
    n, K = a.n_rows, kutta_amd.Kernel
    row_ptr, col = np.asarray(a.row_ptr, np.int32), np.asarray(a.col, np.int32)
    rng = np.random.default_rng(parts)
    rows, cols = device.upload(row_ptr), device.upload(col)
    vals, b = device.upload(np.asarray(a.val, np.float32)), device.upload(rng.standard_normal(n).astype(np.float32))
    inverse, status = device.upload((0.1 + 0.1 * rng.random(n)).astype(np.float32)), device.upload(np.zeros(3, np.int32))
    x, w = device.alloc(n), device.alloc(n)
    device.launch(K.fused_smooth_from_zero, n, rows, cols, vals, b, inverse, x, status)
    for _ in range(2):
        device.launch(K.amg_smooth, n, rows, cols, vals, x, b, inverse, w, status)
        device.launch(K.amg_smooth, n, rows, cols, vals, w, b, inverse, x, status)
    want = x.download().view(np.uint32)

    place, slot, local, table, words = one_level_plan(row_ptr, col, parts)
    arrays = [device.upload(v) for v in (place, slot, local)]
    level = Level(rows.ptr, cols.ptr, vals.ptr, inverse.ptr, 0, 0, 0, *(v.ptr for v in arrays), x.ptr, w.ptr, b.ptr, n, 0)
    levels = device.upload(np.frombuffer(bytes(level), np.uint8))
    parts_table = device.upload(np.frombuffer(b"".join(bytes(t) for t in table), np.uint8))
    ctl, report = device.alloc(160, np.uint32), device.upload(np.zeros(3, np.int32))
    device.launch(K.grid_init, 1, ctl)
    block = ctl.download()
    home = int(block[96])
    assert not block[:96].any() and not block[98:100].any() and not block[101:].any()
    assert block[100] == 32  # of 256 workgroups: round-robin over 8 XCDs
    given_up, together, alone = 0, 0, 0
    for on, counted in ((home, True), (15, True), (home, True), (15, False), (home, False)):
        print(f"[grid] {parts} parts, home {on}", flush=True)
        block[96] = on
        block[98:100] = np.array([report.ptr if counted else 0], np.uint64).view(np.uint32)
        ctl.upload(block)
        for _ in range(3):
            out = device.upload(np.full(n, np.nan, np.float32))
            device.launch(K.grid_cycle, 1, levels, parts_table, ctl, 1, 1, 1, 1, 5, parts, words, 2000, b, out, status)
            assert np.array_equal(out.download().view(np.uint32), want)
            assert np.array_equal(ctl.download(), block)  # clear for the next launch
        together += 3 * (counted and on == home)
        alone += 3 * (counted and on != home)
        assert list(report.download()) == [given_up, together, alone]
