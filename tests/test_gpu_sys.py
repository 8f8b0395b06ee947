"""One-workgroup-per-system kernels (sys_kernels.hip) against the oracle, at the
sizes where their parts can go wrong: a grid of two buses, fronts at and
around 16 and 32 rows (a quarter wave, a wave, the whole workgroup), the
largest grids that fit one workgroup's LDS in FP64 and FP32 and the next ones
that do not, and batches of one workgroup, one per CU and on either side of the
hand-over to the level sweeps."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import capi
from test_gpu_lu_capi import LuConfig, _lu_check

pytestmark = pytest.mark.gpu


def _solver(cupf, g, compute, cap=64):
    o = cupf.NewtonOptions()
    o.compute = getattr(cupf.ComputePolicy, compute)
    o.custom.precision = cupf.CustomPrecision.FP64 if compute == "FP64" else cupf.CustomPrecision.FP32
    o.custom.max_panel_width = cap
    s = cupf.NewtonSolver(o)
    s.initialize(g.indptr, g.indices, g.data, g.n_bus, g.n_bus, g.pv, g.pq)
    return s


def _grid(syn, n, ratio=1.55):
    return syn.make_grid(n, max(n - 1, int(n * ratio)) if n > 2 else 1, int(0.15 * n), seed=n,
                         load_scale=min(0.25, 100.0 / n))


# 2..40 buses: quarter-wave and wave fronts; 118: shared root; 150 / 175 FP64
# and 250 / 320 mixed: either side of the LDS limit
@pytest.mark.parametrize("compute,n,B", [
    ("FP64", 2, 1), ("Mixed", 2, 3), ("FP64", 9, 65), ("FP64", 40, 257), ("Mixed", 40, 64),
    ("FP64", 118, 1), ("FP64", 118, 300), ("Mixed", 118, 130), ("FP64", 150, 5), ("FP64", 175, 5),
    ("Mixed", 250, 7), ("Mixed", 320, 7), ("FP64", 30, 2048), ("FP64", 30, 2049)])
def test_solve_matches_oracle(gpu, cupf, syn, oracle, compute, n, B):
    print(f"[sys] {compute} n={n} B={B}", flush=True)
    g = _grid(syn, n)
    S = g.sbus_scaled(syn.load_factors(B, n, 0.7, 1.3, 5))
    V0 = g.flat_start(B)
    r = _solver(cupf, g, compute).solve_batch(g.indptr, g.indices, g.data, n, n, S, V0, g.pv, g.pq)
    k = min(B, 4)
    pick = np.unique(np.r_[np.arange(k), B - 1])
    Vo, io, _, _ = oracle.nr_solve_batch(n, g.indptr, g.indices, g.data, S[pick], V0[pick], g.pv, g.pq,
                                         tol=1e-13)
    assert r.converged_numpy.all()
    # one further Newton step from ||F|| <= 1e-8 is quadratic; the state is
    # within the tolerance times the inverse Jacobian's norm (below 10 here)
    assert np.abs(r.V_numpy[pick] - Vo).max() <= 1e-7
    assert (r.V_numpy[:, g.slack] == V0[:, g.slack]).all()


@pytest.mark.parametrize("compute,tol", [("FP64", 1e-12), ("Mixed", 1e-9)])
@pytest.mark.parametrize("n,B", [(2, 1), (30, 65), (118, 300), (150, 3)])
@pytest.mark.parametrize("transpose", [False, True])
def test_factor_solve(gpu, cupf, syn, oracle, compute, tol, n, B, transpose):
    print(f"[sys] factor+solve {compute} n={n} B={B} transpose={transpose}", flush=True)
    g = _grid(syn, n)
    s = _solver(cupf, g, compute)
    ja = oracle.jacobian_analysis(n, g.indptr, g.indices, g.pv, g.pq)
    rng = np.random.default_rng(n)
    V = rng.uniform(0.97, 1.03, (B, n)) * np.exp(1j * rng.uniform(-0.1, 0.1, (B, n)))
    A = np.stack([oracle.jacobian_values(n, g.indptr, g.indices, g.data, v, g.pv, g.pq, ja["nnz"])
                  for v in V[:5]])[np.arange(B) % 5]
    rhs = rng.standard_normal((B, ja["dim"]))
    x, sing = capi.debug_factor_solve(s.handle, A, rhs, transpose=transpose)
    assert not sing.any()
    for b in np.unique(np.r_[np.arange(min(B, 6)), B - 1]):
        M = sp.csr_matrix((A[b], ja["col_idx"], ja["row_ptr"]), shape=(ja["dim"],) * 2)
        M = M.T if transpose else M
        assert np.linalg.norm(M @ x[b] - rhs[b]) <= tol * np.linalg.norm(rhs[b]), b


def test_iteration_limits_match_the_level_sweeps(gpu, cupf, syn):
    """Out of iterations the loop ends with a step, as the batched loop does
    (2,049 scenarios run the level sweeps, 70 the one-workgroup kernels)."""
    g = _grid(syn, 30)
    S = g.sbus_scaled(syn.load_factors(2049, 30, 0.7, 1.3, 6))
    V0 = g.flat_start(2049)
    args = (g.indptr, g.indices, g.data, 30, 30)
    s = _solver(cupf, g, "FP64")
    for limit in (0, 1, 2, 3):
        c = cupf.NRConfig()
        c.max_iter = limit
        for B in (1, 70):
            a = s.solve_batch(*args, S[:B], V0[:B], g.pv, g.pq, c)
            b = s.solve_batch(*args, S, V0, g.pv, g.pq, c)
            assert (a.iterations_numpy == limit).all() and (b.iterations_numpy == limit).all()
            np.testing.assert_allclose(a.V_numpy, b.V_numpy[:B], rtol=0, atol=1e-12)


def test_small_pivots_are_replaced_and_flagged(gpu, cupf, syn, oracle):
    """A zero diagonal entry of an isolated row: the static pivot rule, per
    scenario."""
    g = _grid(syn, 30)
    s = _solver(cupf, g, "FP64")
    ja = oracle.jacobian_analysis(30, g.indptr, g.indices, g.pv, g.pq)
    A = np.zeros((70, ja["nnz"]))
    rows = np.repeat(np.arange(ja["dim"]), np.diff(ja["row_ptr"]))
    A[:, rows == ja["col_idx"]] = 2.0
    d3 = np.flatnonzero((rows == 3) & (ja["col_idx"] == 3))[0]
    A[7, d3] = 0.0
    A[9, d3] = -1e-12
    x, sing = capi.debug_factor_solve(s.handle, A, np.ones((70, ja["dim"])))
    want = np.full((70, ja["dim"]), 0.5)
    want[7, 3], want[9, 3] = 1e8, -1e8
    np.testing.assert_allclose(x, want, rtol=1e-15)
    assert sing[7] and sing[9] and sing.sum() == 2


def test_panel_cap_shapes_the_level_sweeps_only(gpu, cupf, syn):
    """The level sweeps' plan is the caller's cap's; the one-workgroup plan is
    the same at every cap, and so are its results to the bit."""
    g = syn.workload_grid("case118")
    a = capi.analyze_jacobian(g.n_bus, g.indptr, g.indices, g.pv, g.pq)
    perm = capi.order_jacobian(g.n_bus, g.indptr, g.indices, g.pv, g.pq, a["dim"])
    fronts = {cap: capi.plan_figures(a["row_ptr"], a["col_idx"], perm, cap)["fronts"] for cap in (8, 64, 128)}
    assert fronts[8] > fronts[64]
    S = g.sbus_scaled(syn.load_factors(65, g.n_bus, 0.7, 1.3, 2))
    V0 = g.flat_start(65)
    sys_plan, V = set(), []
    for cap in (8, 64, 128):
        s = _solver(cupf, g, "FP64", cap)
        plan = capi.debug_plan(s.handle)
        assert plan["fronts"] == fronts[cap]
        sys_plan.add((plan["sys_fronts"], plan["sys_levels"]))
        V.append(s.solve_batch(g.indptr, g.indices, g.data, g.n_bus, g.n_bus, S, V0, g.pv, g.pq).V_numpy)
    assert sys_plan == {(fronts[64], 5)}
    assert (V[0] == V[1]).all() and (V[0] == V[2]).all()


def _factor_solve_unshifted(gpu, A, vals, rhs, precision):
    """x, x of the transpose and the flags of the inner solver without static pivots."""
    lib, (B, n) = capi.lib(), rhs.shape
    cfg = LuConfig()
    lib.cupf_lu_default_config(ctypes.byref(cfg))
    cfg.precision, cfg.pivot_strategy, cfg.refine_steps = precision, 0, 0
    h = ctypes.c_void_p()
    _lu_check(lib.cupf_lu_create(ctypes.byref(cfg), ctypes.byref(h)))
    try:
        rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
        _lu_check(lib.cupf_lu_analyze(h, n, A.nnz, ctypes.c_void_p(rp.ctypes.data),
                                      ctypes.c_void_p(ci.ctypes.data), 0))
        _lu_check(lib.cupf_lu_setup(h, B))
        d_vals, d_rhs = gpu.from_numpy(vals).cuda(), gpu.from_numpy(rhs).cuda()
        d_x, d_xt = gpu.empty_like(d_rhs), gpu.empty_like(d_rhs)
        p = [ctypes.c_void_p(t.data_ptr()) for t in (d_vals, d_rhs, d_x, d_xt)]
        _lu_check(lib.cupf_lu_factor(h, p[0], None))
        _lu_check(lib.cupf_lu_solve(h, p[1], p[2], None))
        _lu_check(lib.cupf_lu_solve_transpose(h, p[1], p[3], None))
        flags = np.zeros(B, np.uint8)
        _lu_check(lib.cupf_lu_singular(h, ctypes.c_void_p(flags.ctypes.data)))
        return d_x.cpu().numpy(), d_xt.cpu().numpy(), flags
    finally:
        _lu_check(lib.cupf_lu_destroy(h))


# pivots with a reciprocal that overflows, one that is no normal number, and infinite ones
ENDS = [(0, 2.0 ** -1030, 2.0 ** 1023), (1, 2.0 ** -130, 2.0 ** 127)]


def _ends(tiny, huge, shape):
    pivots = np.array([huge, -huge, 1.75 * huge, np.inf, -np.inf, tiny, -3 * tiny, 2.0])
    return pivots[np.random.default_rng(5).integers(0, len(pivots), shape)]


@pytest.mark.parametrize("precision,tiny,huge", ENDS)
def test_quotients_at_the_ends_of_the_range(gpu, precision, tiny, huge):
    """A diagonal system (fronts of one row), its quotients overflowing and
    underflowing: exactly what the division gives."""
    print(f"[sys] quotients precision={precision}", flush=True)
    T = np.float32 if precision else np.float64
    top = float(np.finfo(T).max)
    d = _ends(tiny, huge, (70, 40))
    b = np.array([1.0, -3.0, tiny, 0.75 * top, top])[np.random.default_rng(6).integers(0, 5, d.shape)]
    with np.errstate(over="ignore"):
        want = (b.astype(T) / d.astype(T)).astype(np.float64)
    assert np.isinf(want).any() and (want == 0).any()
    x, xt, flags = _factor_solve_unshifted(gpu, sp.identity(40, format="csr"), d, b, precision)
    assert not flags.any()
    np.testing.assert_array_equal(x, want)
    np.testing.assert_array_equal(xt, want)


@pytest.mark.parametrize("precision,tiny,huge", ENDS)
@pytest.mark.parametrize("rows", [12, 24, 40, 90])
def test_pivots_at_the_ends_of_the_range(gpu, precision, tiny, huge, rows):
    """The same pivots on the diagonal of a full front of zeros (16 lanes, the
    workgroup in both its forms): the quotients here are 1, -1, 1/2 and 0, for
    a zero of the front times an infinite one would be no number by division
    either."""
    print(f"[sys] pivots rows={rows} precision={precision}", flush=True)
    A = sp.csr_matrix(np.ones((rows, rows)))
    d = _ends(tiny, huge, (70, rows))
    vals = np.zeros((70, rows * rows))
    vals[:, ::rows + 1] = d
    want = np.array([1.0, -1.0, 0.5])[np.random.default_rng(6).integers(0, 3, d.shape)]
    want[np.isinf(d)] = 0.0
    b = np.where(np.isinf(d), 1.0, np.where(np.isinf(d), 1.0, d) * want)
    x, xt, flags = _factor_solve_unshifted(gpu, A, vals, b, precision)
    assert not flags.any()
    np.testing.assert_array_equal(x, want)
    np.testing.assert_array_equal(xt, want)


@pytest.mark.parametrize("graph", [False, True])
def test_one_scenario_that_does_not_converge(gpu, cupf, syn, graph):
    """A tolerance of zero: the loop ends at the limit, 100 evaluations, with the
    same state as the level sweeps' (2,049 scenarios) and, captured, after more
    than one launch, so no launch is as long as the limit."""
    g = _grid(syn, 30)
    S = g.sbus_scaled(syn.load_factors(2049, 30, 0.7, 1.3, 6))
    V0 = g.flat_start(2049)
    args = (g.indptr, g.indices, g.data, 30, 30)
    c = cupf.NRConfig()
    c.tolerance, c.max_iter = 0.0, 100
    o = cupf.NewtonOptions()
    o.compute, o.use_cuda_graph = cupf.ComputePolicy.FP64, graph
    s = cupf.NewtonSolver(o)
    s.initialize(g.indptr, g.indices, g.data, 30, 30, g.pv, g.pq)
    many = s.solve_batch(*args, S, V0, g.pv, g.pq, c)
    for call in range(3):
        before = s.stats()["graph_launches"]
        one = s.solve_batch(*args, S[:1], V0[:1], g.pv, g.pq, c)
        assert one.iterations_numpy[0] == many.iterations_numpy[0] == 100
        np.testing.assert_allclose(one.V_numpy, many.V_numpy[:1], rtol=0, atol=1e-12)
        launches = s.stats()["graph_launches"] - before
        assert launches == (0 if not graph or call == 0 else 4)     # 32 + 32 + 32 + 3 steps


@pytest.mark.parametrize("compute", ["Mixed", "FP64"])
@pytest.mark.parametrize("graph", [False, True])
def test_a_step_whose_pivots_have_no_reciprocal(gpu, cupf, syn, compute, graph):
    """Two buses, S and Y scaled by a power of two that takes the Jacobian's
    pivots out of the range of reciprocals (2^1023 in FP64, 2^127 in FP32), so
    that every step divides: the voltages equal the unscaled grid's, whose steps
    differ by that power throughout (1e-9: the quotients' rounding near the
    range's end, over a Jacobian of condition about one)."""
    g = syn.make_grid(2, 1, 0, seed=2, load_scale=0.25)
    y = float(np.abs(g.data).max())
    scale = 2.0 ** ((1023 if compute == "FP64" else 127) - np.floor(np.log2(y)) - 1)
    V = {}
    for k in (1.0, scale):
        o = cupf.NewtonOptions()
        o.compute = getattr(cupf.ComputePolicy, compute)
        o.custom.precision = cupf.CustomPrecision.FP64 if compute == "FP64" else cupf.CustomPrecision.FP32
        o.use_cuda_graph = graph
        s = cupf.NewtonSolver(o)
        s.initialize(g.indptr, g.indices, k * g.data, 2, 2, g.pv, g.pq)
        c = cupf.NRConfig()
        c.tolerance, c.max_iter = 1e-12 * k, 12
        S = k * g.sbus_scaled(syn.load_factors(3, 2, 0.7, 1.3, 1))
        for call in range(2):
            r = s.solve_batch(g.indptr, g.indices, k * g.data, 2, 2, S, g.flat_start(3), g.pv, g.pq, c)
            assert r.converged_numpy.all()
        V[k] = r.V_numpy
    np.testing.assert_allclose(V[scale], V[1.0], rtol=0, atol=1e-9)
