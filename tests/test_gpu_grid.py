"""The multi-workgroup V-cycle (KH_GRID_CYCLE) against the per-level launches
it replaces: bitwise-identical iterates, iteration counts and residuals from
every admissible first level, through graph replays and direct launches, with
its workgroups together and with one working alone (a wait of zero), on
hierarchies that end in the few-row coarse solve, in coarse sweeps, and in
levels too large for the one-workgroup part."""
import numpy as np
import pytest

import kutta_amd
import oracle
from kutta_amd import AmgCycle, AmgOptions, OperatorStructure, SolveControl, SolverKind

pytestmark = pytest.mark.gpu
M = OperatorStructure.SymmetricMMatrix

CASES = [
    ("poisson V(5,5)", lambda: oracle.poisson(30, 28, 26), SolverKind.AmgPcg, AmgOptions()),
    ("ragged rows V(2,2)", lambda: oracle.poisson(33, 31, 29, 1.0, random=True), SolverKind.AmgPcg,
     AmgOptions(pre_sweeps=2, post_sweeps=2, aggregation_passes=2)),
    ("V(1,1)", lambda: oracle.poisson(23, 21, 19), SolverKind.AmgPcg, AmgOptions(pre_sweeps=1, post_sweeps=1)),
    ("pressure, coarse sweeps", lambda: oracle.pressure_problem(18, 17, 16).csr(), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=2, coarse_rows=400, structure=M)),
    ("pressure, stalled coarse levels", lambda: oracle.pressure_problem(24, 23, 22).csr(), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=2, structure=M)),
    ("anisotropic, pair aggregates", lambda: oracle.poisson(32, 32, 32, 100), SolverKind.AmgPcg,
     AmgOptions(aggregation_passes=1, max_levels=4)),
    ("bicgstab V(2,3)", lambda: oracle.poisson(52, 47, 1, 1.0, wind=2.0), SolverKind.AmgBicgstab,
     AmgOptions(pre_sweeps=2, post_sweeps=3, aggregation_passes=2)),
    ("K-cycle", lambda: oracle.pressure_problem(20, 19, 18).csr(), SolverKind.AmgPcg,
     AmgOptions(pre_sweeps=1, post_sweeps=1, coarse_sweeps=4, aggregation_passes=2, structure=M, cycle=AmgCycle.K,
                k_min_rows=5000)),
]


@pytest.mark.parametrize("name,make,kind,opts", CASES, ids=[c[0] for c in CASES])
def test_grid_cycle_matches_level_launches(device, name, make, kind, opts):
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
    tried = 0
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
            for _ in range(2):
                st, x = run()
                assert (st.iterations, st.final_residual) == (st0.iterations, st0.final_residual)
                assert np.array_equal(x.view(np.uint32), x0.view(np.uint32))
        tried += 1
    assert tried >= 1


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
