"""NewtonOptions.use_cuda_graph: the device-run Newton loop against the eager
loop on the same inputs.

A captured solve holds the residual at the initial V with its stop test (and,
with a warm-start network, the network's inference before it) and a
predicted number of Newton steps (Jacobian, factor, solve with refinement,
voltage update, next residual, batch max, stop test), each gated on the
device by a control word; steps beyond the prediction run one captured step
at a time.  The loop follows the reference's graph semantics (at most
max_iter - 1 steps; reference
cuPF/cpp/src/newton_solver/core/graph_iteration.hpp:85-146), so on converging
batches it takes the same steps as the eager loop and the results are
bit-identical.  Covered: several solves in a row (a new batch size
recaptures), a prediction above the steps a batch needs (the gated steps do
nothing), below it (continuation steps), the refinement decided on the device
(Mixed), a warm-started solve in one launch, and batch 1; each on a grid that
runs the one-workgroup kernels (118 buses) and on one that runs the level
sweeps (400 buses).
"""

from __future__ import annotations

import numpy as np
import pytest

import capi

pytestmark = pytest.mark.gpu


def _solver(cupf, g, compute, graph, refine=1):
    o = cupf.NewtonOptions()
    o.compute = getattr(cupf.ComputePolicy, compute)
    o.custom.precision = cupf.CustomPrecision.FP64 if compute == "FP64" else cupf.CustomPrecision.FP32
    o.custom.max_panel_width = 64
    o.custom.refine_steps = refine
    o.use_cuda_graph = graph
    s = cupf.NewtonSolver(o)
    s.initialize(g.indptr, g.indices, g.data, g.n_bus, g.n_bus, g.pv, g.pq)
    return s


@pytest.fixture(params=[118, 400])
def grid(request, syn):
    if request.param == 118:
        return syn.workload_grid("case118")
    return syn.make_grid(400, 620, 60, seed=400, load_scale=0.25)


def test_the_grids_run_either_kind_of_loop(gpu, cupf, grid):
    for compute in ("Mixed", "FP64"):
        s = _solver(cupf, grid, compute, False)      # the handle is the solver's
        assert (capi.debug_plan(s.handle)["sys_fronts"] > 0) == (grid.n_bus == 118)


@pytest.mark.parametrize("compute", ["Mixed", "FP64"])
def test_graph_step_matches_eager(gpu, cupf, syn, grid, compute):
    g = grid
    eager = _solver(cupf, g, compute, False)
    graph = _solver(cupf, g, compute, True)
    for call, (B, seed) in enumerate([(70, 3), (70, 4), (70, 3), (33, 5), (70, 6)]):
        S = g.sbus_scaled(syn.load_factors(B, g.n_bus, 0.7, 1.3, seed))
        V0 = g.flat_start(B)
        re = eager.solve_batch(g.indptr, g.indices, g.data, g.n_bus, g.n_bus, S, V0, g.pv, g.pq)
        rg = graph.solve_batch(g.indptr, g.indices, g.data, g.n_bus, g.n_bus, S, V0, g.pv, g.pq)
        print(f"call {call}: B={B} seed={seed} iterations {rg.iterations_numpy[0]}", flush=True)
        assert rg.converged_numpy.all()
        np.testing.assert_array_equal(rg.iterations_numpy, re.iterations_numpy)
        np.testing.assert_array_equal(rg.V_numpy, re.V_numpy)
        np.testing.assert_array_equal(rg.final_mismatch_numpy, re.final_mismatch_numpy)
    assert graph.stats()["factorizations"] == eager.stats()["factorizations"]


def _check_same(re, rg):
    assert rg.converged_numpy.all()
    np.testing.assert_array_equal(rg.iterations_numpy, re.iterations_numpy)
    np.testing.assert_array_equal(rg.V_numpy, re.V_numpy)
    np.testing.assert_array_equal(rg.final_mismatch_numpy, re.final_mismatch_numpy)


@pytest.mark.parametrize("compute", ["Mixed", "FP64"])
def test_gated_steps_over_and_under_the_prediction(gpu, cupf, syn, grid, compute):
    """A flat start (6 or so iterations) teaches the prediction; a start at a
    near-solution then needs fewer steps (the captured solve runs gated
    no-op steps after convergence), and a flat start again needs more than
    that prediction (continuation steps); each equals the eager solver."""
    g = grid
    eager = _solver(cupf, g, compute, False)
    graph = _solver(cupf, g, compute, True)
    B = 70
    S = g.sbus_scaled(syn.load_factors(B, g.n_bus, 0.7, 1.3, 8))
    V0 = g.flat_start(B)
    args = (g.indptr, g.indices, g.data, g.n_bus, g.n_bus)
    ref = eager.solve_batch(*args, S, V0, g.pv, g.pq)
    near = ref.V_numpy * np.exp(1j * 1e-4 * np.random.default_rng(1).standard_normal(ref.V_numpy.shape))
    near[:, 0] = V0[:, 0]                  # the slack voltage is a set point
    eager_before = eager.stats()["factorizations"]
    for call, start in enumerate([V0, V0, near, near, V0, V0]):
        re = eager.solve_batch(*args, S, start, g.pv, g.pq)
        before = graph.stats()["graph_launches"]
        rg = graph.solve_batch(*args, S, start, g.pv, g.pq)
        launches = graph.stats()["graph_launches"] - before
        print(f"call {call}: iterations {rg.iterations_numpy[0]}, graph launches {launches}",
              flush=True)
        _check_same(re, rg)
        if call in (1, 3, 5):              # the prediction is right: one launch
            assert launches == 1
    assert graph.stats()["factorizations"] == eager.stats()["factorizations"] - eager_before


def test_warm_start_inside_the_captured_solve(gpu, cupf, syn, grid):
    """A warm-started solve: inference, the tolerant warm pass and the stop
    tests in one captured launch once the step count is known; V,
    iterations and fallbacks equal the eager solver's with the same
    network."""
    torch = gpu
    g = grid
    eager = _solver(cupf, g, "Mixed", False)
    graph = _solver(cupf, g, "Mixed", True)
    St = torch.from_numpy(g.sbus_scaled(syn.load_factors(2048, g.n_bus, 0.6, 1.4, seed=2))).cuda()
    V0t = torch.from_numpy(g.flat_start(2048)).cuda()
    mlp, _ = cupf.train_warm_start(eager, St, V0t, g.pv, g.pq, hidden=128, depth=2, epochs=20,
                                   batch=256, lr=2e-3, seed=0)
    eager.set_warm_start(mlp, 4)
    graph.set_warm_start(mlp, 4)
    args = (g.indptr, g.indices, g.data, g.n_bus, g.n_bus)
    for call, seed in enumerate([3, 3, 4, 5]):
        S = g.sbus_scaled(syn.load_factors(256, g.n_bus, 0.6, 1.4, seed))
        V0 = g.flat_start(256)
        re = eager.solve_batch(*args, S, V0, g.pv, g.pq)
        se = eager.stats()
        before = graph.stats()["graph_launches"]
        rg = graph.solve_batch(*args, S, V0, g.pv, g.pq)
        sg = graph.stats()
        print(f"call {call}: warm iterations {sg['last_warm_iterations']}, fallbacks "
              f"{sg['last_warm_fallbacks']}, launches {sg['graph_launches'] - before}", flush=True)
        _check_same(re, rg)
        assert sg["last_warm_iterations"] == se["last_warm_iterations"]
        assert sg["last_warm_fallbacks"] == se["last_warm_fallbacks"]
        if call == 1 and sg["last_warm_fallbacks"] == 0:
            assert sg["graph_launches"] - before == 1


@pytest.mark.parametrize("compute", ["Mixed", "FP64"])
def test_batch_one_graph(gpu, cupf, syn, grid, compute):
    """Batch 1: the whole loop in one launch, or the level sweeps of one scenario."""
    g = grid
    eager = _solver(cupf, g, compute, False)
    graph = _solver(cupf, g, compute, True)
    args = (g.indptr, g.indices, g.data, g.n_bus, g.n_bus)
    for seed in (1, 2, 1):
        S = g.sbus_scaled(syn.load_factors(1, g.n_bus, 0.7, 1.3, seed))
        V0 = g.flat_start(1)
        _check_same(eager.solve_batch(*args, S, V0, g.pv, g.pq),
                    graph.solve_batch(*args, S, V0, g.pv, g.pq))


def test_both_kinds_of_loop_run_eagerly_before_their_capture(gpu, cupf, syn):
    """70 scenarios of 30 buses run the one-workgroup kernels, 2,049 the level
    sweeps: the first solve of either kind launches no graph, so no kernel is
    used for the first time inside a capture; every later one is one launch,
    and all equal the eager solver's."""
    g = syn.make_grid(30, 46, 4, seed=30, load_scale=0.25)
    eager = _solver(cupf, g, "FP64", False)
    graph = _solver(cupf, g, "FP64", True)
    S = g.sbus_scaled(syn.load_factors(2049, 30, 0.7, 1.3, 6))
    V0 = g.flat_start(2049)
    args = (g.indptr, g.indices, g.data, 30, 30)
    for B, launches in [(70, 0), (2049, 0), (2049, 1), (70, 1), (2049, 1)]:
        print(f"[graph] B={B}", flush=True)
        re = eager.solve_batch(*args, S[:B], V0[:B], g.pv, g.pq)
        before = graph.stats()["graph_launches"]
        rg = graph.solve_batch(*args, S[:B], V0[:B], g.pv, g.pq)
        assert graph.stats()["graph_launches"] - before == launches
        _check_same(re, rg)


def test_small_grids_keep_their_graphs(gpu, cupf, syn):
    """The one-workgroup launches do not depend on the refinement pattern, nor,
    for one scenario, on the step count: starts that take different steps, and
    torch forwards between warm-started solves, reuse the graphs there are."""
    torch = gpu
    g = syn.workload_grid("case118")
    n = g.n_bus
    args = (g.indptr, g.indices, g.data, n, n)
    eager, graph = (_solver(cupf, g, "Mixed", on) for on in (False, True))
    S, V0 = g.sbus_scaled(syn.load_factors(256, n, 0.7, 1.3, 8)), g.flat_start(256)
    V = eager.solve_batch(*args, S, V0, g.pv, g.pq).V_numpy

    def near(scale):
        v = V * np.exp(1j * scale * np.random.default_rng(1).standard_normal(V.shape))
        v[:, g.slack] = V0[:, g.slack]
        return v

    def solve(B, start):
        _check_same(eager.solve_batch(*args, S[:B], start[:B], g.pv, g.pq),
                    graph.solve_batch(*args, S[:B], start[:B], g.pv, g.pq))
        return capi.debug_captures(graph.handle)

    starts = [V0, near(1e-4), near(1e-2), near(1e-7), V0]
    assert [solve(1, v) for v in starts] == [0, 1, 1, 1, 1]
    assert len({int(eager.solve_batch(*args, S[:1], v[:1], g.pv, g.pq).iterations_numpy[0]) for v in starts}) > 2

    mlp, _ = cupf.train_warm_start(eager, torch.from_numpy(S).cuda(), torch.from_numpy(V0).cuda(), g.pv, g.pq,
                                   hidden=64, depth=2, epochs=3, batch=64, lr=2e-3, seed=0, skip=False)
    graph.set_warm_start(mlp, 10)
    t = [torch.from_numpy(np.ascontiguousarray(v, np.float32)).cuda()
         for v in (g.p_gen, np.zeros(n), np.tile(g.p_load, (256, 1)), np.tile(g.q_load, (256, 1)),
                   np.angle(V0[0]), np.abs(V0[0]))]
    new = []
    for call in range(4):
        print(f"[graph] warm call {call}", flush=True)
        before = capi.debug_captures(graph.handle)
        assert graph.solve_batch(*args, S, V0, g.pv, g.pq).converged_numpy.all()
        assert graph.stats()["last_warm_fallbacks"] == 0
        new.append(capi.debug_captures(graph.handle) - before)
        if call == 1:
            cupf.solve(t[2], t[3], graph, sbus_base_re=t[0], sbus_base_im=t[1], v0_va=t[4], v0_vm=t[5])
    assert new == [0, 1, 0, 0]         # eager, captured, then launched
