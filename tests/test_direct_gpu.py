"""The direct linear solve (multifrontal block Cholesky, the default) against
the PCG (an explicit pcg_segment) on the graph shapes its elimination plan can
meet: single poses, chains, reversed and repeated factors, stars, hubs, several
components, cliques, and the graphs it declines (too wide, singular), which run
the PCG either way.  The 20,000-pose laps have levels of every launch shape (fronts
of up to 8 rows with 64 and 256 threads, wider ones with 256 and 1,024, one or
more workgroups a front); the plan's test checks that they do.

Bar: the same iteration counts and poses within 1e-6 m.  Both solve each step
to at most 1e-9 (PCG) and 1e-10 (direct) of its right-hand side; the graphs'
condition numbers stay below about 1e3 per unit of pose, so steps agree to
1e-6 with room.
"""
import os
import subprocess

import numpy as np
import pytest

from rpgo_amd import _capi, problem, synth

pytestmark = pytest.mark.gpu
TOL = 1e-6


@pytest.fixture(scope="module")
def ctx():
    c = _capi.Context(0)
    yield c
    c.close()


def _pose(rng, n, spread=5.0):
    return synth.rot_exp(rng.normal(0, 0.5, (n, 3))), rng.normal(0, spread, (n, 3))


def _graph(n, edges, seed, priors=(0,)):
    """Noisy between factors over `edges`, priors, perturbed initial poses."""
    rng = np.random.default_rng(seed)
    R, t = _pose(rng, n)
    e = np.array(edges, np.int64).reshape(-1, 2)
    Rz, tz = synth.se3_rel(R[e[:, 0]], t[e[:, 0]], R[e[:, 1]], t[e[:, 1]])
    Rz, tz = synth.se3_mul(Rz, tz, synth.rot_exp(rng.normal(0, 0.01, (len(e), 3))), rng.normal(0, 0.02, (len(e), 3)))
    p = np.array(priors, np.int64)
    kind = np.concatenate([np.zeros(len(e), np.int32), np.ones(len(p), np.int32)])
    ki = np.concatenate([e[:, 0], p]).astype(np.int32)
    kj = np.concatenate([e[:, 1], p]).astype(np.int32)
    meas = np.concatenate([synth.se3_pack(Rz, tz), synth.se3_pack(R[p], t[p])])
    info = np.tile(np.diag([1e4] * 3 + [2500.0] * 3).reshape(36), (len(kind), 1))
    info[len(e):] = (np.eye(6) * 100.0).reshape(36)
    Rx, tx = synth.se3_mul(R, t, synth.rot_exp(rng.normal(0, 0.02, (n, 3))), rng.normal(0, 0.05, (n, 3)))
    order = rng.permutation(len(kind))
    return synth.se3_pack(Rx, tx), kind[order], ki[order], kj[order], meas[order], info[order]


def _chain(n):
    return [(k, k + 1) for k in range(n - 1)]


def _flip(edges, seed):
    rng = np.random.default_rng(seed)
    return [(b, a) if rng.uniform() < 0.5 else (a, b) for a, b in edges]


def _shuffled(n, n_lc, seed):
    """A chain over shuffled pose numbers with loop closures and repeats."""
    rng = np.random.default_rng(seed)
    name = rng.permutation(n)
    e = [(int(name[a]), int(name[b])) for a, b in _chain(n)]
    while len(e) < n - 1 + n_lc:
        a, b = (int(v) for v in rng.integers(0, n, 2))
        if a != b:
            e.append((a, b))
    return _flip(e + e[::3], seed)


def _clique(n):
    return [(a, b) for a in range(n) for b in range(a + 1, n)]


def _chain_hub(n, seen):
    """A chain of n poses and pose n, seen from `seen` of them."""
    return n + 1, _chain(n) + [(k * n // seen, n) for k in range(seen)]


def _laps(n, lap, every):
    """Laps of `lap` poses, joined at every `every`th pose."""
    return _chain(n) + [(k + lap, k) for k in range(0, n - lap, every)]


CASES = {
    "one_pose": (1, [], (0,)),
    "two_poses": (2, [(1, 0)], (1,)),
    "chain_63": (63, _chain(63), (0,)),
    "chain_64_reversed": (64, _flip(_chain(64), 1), (63,)),
    "chain_65_repeated": (65, _chain(65) + _flip(_chain(65)[::2], 2), (30,)),
    "shuffled_130": (130, _shuffled(130, 40, 3), (0,)),
    "star_70": (70, _flip([(0, k) for k in range(1, 70)], 4), (0,)),
    "hub_60_of_200": (*_chain_hub(200, 60), (0,)),
    "hub_300_of_300": (*_chain_hub(300, 300), (0,)),
    "two_components": (41, _chain(20) + [(k, k + 1) for k in range(20, 40)] + [(3, 15)], (0, 20)),
    "laps_20000": (20000, _laps(20000, 100, 5), (0,)),
    "clique_6": (6, _clique(6), (0,)),
    "clique_11": (11, _flip(_clique(11), 5), (0,)),
    "clique_40": (40, _flip(_clique(40), 6), (0,)),
    "clique_193": (193, _clique(193), (0,)),      # the widest front the plan takes
    "clique_200": (200, _clique(200), (0,)),      # wider: PCG
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_direct_equals_pcg(ctx, name):
    n, edges, priors = CASES[name]
    g = _graph(n, edges, len(name), priors)
    print(f"[direct] {name} N={n} F={len(g[1])}", flush=True)
    a, wa, ra = ctx.solve(*g)
    b, wb, rb = ctx.solve(*g, pcg_segment=16, pcg_rel_tol=1e-9)
    d = np.abs(a - b).max()
    print(f"[direct] lm {ra.lm_iterations}/{rb.lm_iterations} solves {ra.pcg_iterations} pcg {rb.pcg_iterations} "
          f"cost {ra.final_cost:.9g}/{rb.final_cost:.9g} d {d:.1e}", flush=True)
    assert ra.lm_iterations == rb.lm_iterations and d < TOL
    assert ra.final_cost == pytest.approx(rb.final_cost, rel=1e-9, abs=1e-12)
    if name != "clique_200":  # the direct path ran, and gives the same bits again
        assert ra.pcg_iterations <= 4 * ra.linearizations
        again, _, _ = ctx.solve(*g)
        assert np.array_equal(a, again)


def test_gauss_newton_and_no_prior(ctx):
    """Gauss-Newton with a prior runs the direct path; without one no factor
    holds the poses, the matrix is singular and the step is the PCG's, as with
    an explicit pcg_segment."""
    n, edges, _ = CASES["shuffled_130"]
    g = _graph(n, edges, 9)
    a, _, ra = ctx.solve(*g, solver=_capi.SOLVER_GN)
    b, _, rb = ctx.solve(*g, solver=_capi.SOLVER_GN, pcg_segment=16, pcg_rel_tol=1e-9)
    assert ra.lm_iterations == rb.lm_iterations and np.abs(a - b).max() < TOL
    n, edges, _ = CASES["chain_63"]
    g = _graph(n, edges, 9, priors=())
    a, _, ra = ctx.solve(*g, solver=_capi.SOLVER_GN)
    b, _, rb = ctx.solve(*g, solver=_capi.SOLVER_GN, pcg_segment=16)
    assert ra.pcg_iterations > 4 * ra.linearizations
    assert np.isfinite(a).all() and ra.final_cost == pytest.approx(rb.final_cost, rel=1e-6)


def test_gnc_large_refinement(ctx):
    """Above 8,192 poses the last step is refined once more: the poses stay
    within 1e-6 m of the PCG's at 1e-9 (no soft-mode bias)."""
    gr = synth.se3_helix(n_poses=9001, n_lc=900, outlier_frac=0.0, seed=3)
    arrs = problem.solve_arrays(gr)
    a, wa, ra = ctx.solve(*arrs[:-1])
    b, wb, rb = ctx.solve(*arrs[:-1], pcg_segment=16, pcg_rel_tol=1e-9)
    d = np.abs(a - b).max()
    print(f"[direct] 9001 poses lm {ra.lm_iterations}/{rb.lm_iterations} d {d:.1e}", flush=True)
    assert ra.lm_iterations == rb.lm_iterations and d < TOL


def test_hub_not_slower_than_pcg(ctx):
    """A landmark seen from a tenth of a chain: the plan's levels stay few, so
    a direct solve takes less device time than the PCG (about a tenth)."""
    n, edges = _chain_hub(3000, 300)
    g = _graph(n, edges, 5)
    ctx.solve(*g)
    a, _, ra = ctx.solve(*g)
    ctx.solve(*g, pcg_segment=16, pcg_rel_tol=1e-9)
    b, _, rb = ctx.solve(*g, pcg_segment=16, pcg_rel_tol=1e-9)
    d = np.abs(a - b).max()
    print(f"[direct] hub 300/3000 {ra.ms_total:.2f} ms, pcg {rb.ms_total:.2f} ms, d {d:.1e}", flush=True)
    assert ra.lm_iterations == rb.lm_iterations and d < TOL
    assert ra.ms_total < rb.ms_total


def test_allocation_failure_binary():
    """A device allocation of the direct path that fails (tests/cpp): the solve
    goes on with the PCG, and a later one takes the direct path again."""
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_alloc_failure")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0


def _weakly_held(n, stiff, soft=1e-2, seed=1):
    """A chain of consistent stiff factors held by one weak prior a few metres
    off: the solution moves along the softest mode, where b is stiff / soft
    times smaller than the terms of H dx."""
    rng = np.random.default_rng(seed)
    R, t = _pose(rng, n)
    e = np.array(_chain(n))
    Rz, tz = synth.se3_rel(R[e[:, 0]], t[e[:, 0]], R[e[:, 1]], t[e[:, 1]])
    kind = np.r_[np.zeros(n - 1, np.int32), np.ones(1, np.int32)]
    ki, kj = np.r_[e[:, 0], 0].astype(np.int32), np.r_[e[:, 1], 0].astype(np.int32)
    meas = np.r_[synth.se3_pack(Rz, tz), synth.se3_pack(R[:1], t[:1] + [[1.0, 2.0, 3.0]])]
    info = np.tile((np.eye(6) * stiff).reshape(36), (n, 1))
    info[-1] = (np.eye(6) * soft).reshape(36)
    return synth.se3_pack(R, t), kind, ki, kj, meas, info


@pytest.mark.parametrize("n, stiff, direct", [(20, 1e4, True), (100, 1e4, True), (20, 1e8, False), (100, 1e8, False),
                                              (100, 1e9, False)])
def test_residual_decides(ctx, n, stiff, direct):
    """A Gauss-Newton step's residual cannot be refined below about 1e-16 stiff /
    soft (times a chain factor): 5e-9 and 1e-8 at 1e4, 4e-5 and 1e-4 at 1e8.
    Above pcg_rel_tol (1e-6) and 1e-8 the step is the PCG's, not accepted as it
    is; with a tolerance of 1e-2 all are accepted."""
    g = _weakly_held(n, stiff)
    kw = dict(solver=_capi.SOLVER_GN, lm_max_iterations=1)
    a, _, ra = ctx.solve(*g, **kw)
    b, _, rb = ctx.solve(*g, pcg_rel_tol=1e-2, **kw)
    print(f"[direct] weakly held {n} {stiff:.0e}: {ra.pcg_iterations} at 1e-6, {rb.pcg_iterations} at 1e-2", flush=True)
    assert np.isfinite(a).all() and rb.pcg_iterations <= 4
    assert (ra.pcg_iterations <= 4) == direct


@pytest.mark.parametrize("n, n_lc", [(1000, 0), (1000, 100), (20000, 0), (20000, 2000)])
def test_free_graph_undamped(ctx, n, n_lc):
    """Gauss-Newton without a prior: the matrix is singular and its last pivots
    are noise of either sign, up to 2e-10 of the diagonal at 20,000 poses, so
    the step is the PCG's without a factorization (its iterations come in
    eights; a factorization would count one more).  LM whose lambda is lost in
    the diagonal starts with the PCG too, and never raises the cost."""
    gr = synth.se3_helix(n_poses=n, n_lc=max(n_lc, 2), outlier_frac=0.0, seed=3)
    a = problem.solve_arrays(gr, lc_idx=np.arange(n_lc))
    keep = a[1] == 0
    g = [a[0]] + [v[keep] for v in a[1:6]]
    g[0], _, r0 = ctx.solve(*g)
    assert r0.pcg_iterations <= 4 * (r0.linearizations + 1)  # damped: direct
    x, _, r = ctx.solve(*g, solver=_capi.SOLVER_GN, lm_max_iterations=1)
    print(f"[direct] free {n} {n_lc}: {r.pcg_iterations} cost {r0.final_cost:.10g} {r.final_cost:.10g}", flush=True)
    assert r.pcg_iterations > 0 and r.pcg_iterations % 8 == 0
    assert np.isfinite(x).all()
    x, _, r = ctx.solve(*g, lambda_initial=1e-20, lm_max_iterations=1, lm_relative_error_tol=1e-30)
    assert r.pcg_iterations >= 8 and np.isfinite(x).all() and r.final_cost <= r0.final_cost * (1 + 1e-9)
    # lambda added as it is (not times the diagonal): the PCG; direct with a prior
    for damped in (g, a[:6]):
        x, _, r = ctx.solve(*damped, lm_diagonal_damping=0, lm_max_iterations=1)
        assert (r.pcg_iterations % 8 == 0) == (damped is g) and np.isfinite(x).all()


@pytest.mark.parametrize("use_gnc", [0, 1])
def test_zero_weight_frees_a_part(ctx, use_gnc):
    """Two chains, a prior on the first only, joined by one factor: while its
    weight holds the second chain the Gauss-Newton steps are direct, at weight
    0 (GNC's initial weights here) they are the PCG's."""
    edges = [(k, k + 1) for k in range(59) if k != 29] + [(0, 20), (5, 25), (30, 50), (35, 55), (10, 40)]
    poses, kind, ki, kj, meas, info = _graph(60, edges, 4)
    link = (kind == 0) & (ki == 10) & (kj == 40)
    order = np.argsort(link, kind="stable")  # the link last, all others known
    g = (poses,) + tuple(np.ascontiguousarray(v[order]) for v in (kind, ki, kj, meas, info))
    kw = dict(solver=_capi.SOLVER_GN, use_gnc=use_gnc, known_inliers=len(kind) - 1 if use_gnc else 0,
              gnc_max_iterations=0)
    its = {}
    for w in (1.0, 1e-3, 0.0):
        x, _, r = ctx.solve(*g, init_weights=np.r_[np.ones(len(kind) - 1), w], **kw)
        its[w] = r.pcg_iterations
        assert np.isfinite(x).all()
        assert (r.pcg_iterations <= 4 * r.linearizations) == (w > 0.0)
    print(f"[direct] freed part: {its}", flush=True)


def test_failed_factorization_is_remembered(ctx):
    """A Gauss-Newton matrix that is singular to FP64 (a prior of 1e-2 under a
    chain of 1e10) is factored once, not at every step; the PCG's iterations
    come in eights."""
    g = _weakly_held(20, 1e10)
    _, _, r = ctx.solve(*g, solver=_capi.SOLVER_GN, lm_relative_error_tol=0.0, lm_absolute_error_tol=0.0,
                        lm_max_iterations=3)
    print(f"[direct] singular: {r.linearizations} linearizations, {r.pcg_iterations} iterations", flush=True)
    assert r.linearizations == 3 and r.pcg_iterations > 8 and r.pcg_iterations % 8 == 1
