"""V-cycles whose coarse levels are one dense matrix (the first level of at
most 1024 vertices, 2048 where rows are short, and everything below it),
against the oracle's cycle from every level: the levels above it, the collapsed one, and those below."""
import numpy as np
import pytest

import oracle_ffi as O
import ligmg_amd
from ligmg_amd import _ffi, graphs

pytestmark = pytest.mark.gpu

VARIANTS = {
    "default": {},
    "jacobi": {"smoother_type": _ffi.SMOOTHER_JACOBI},
    "smooth_3_1": {"pre_smooth": 3, "post_smooth": 1},
    "no_pre_smooth": {"pre_smooth": 0, "post_smooth": 2},
    "no_post_smooth": {"pre_smooth": 2, "post_smooth": 0},
    "constant_correction": {"constant_correction": 1},
    "kcycle": {"kcycle": 1},  # nothing is collapsed
}
GRAPHS = {
    "grid64x32": lambda: graphs.grid2d(64, 32),  # the base level has exactly 2048 vertices
    "grid683x3": lambda: graphs.grid2d(683, 3, graphs.W_UNIFORM, 0.1, 10.0, 3),  # 2049: one above
    "dense1024": lambda: graphs.barabasi_albert(1024, 20, seed=2),  # long rows: at the smaller bound
    "dense1025": lambda: graphs.barabasi_albert(1025, 20, seed=2),
    "rmat12": lambda: graphs.rmat_config(12, "lognormal", pendants=True),
    "tiny": lambda: graphs.barabasi_albert(60, 2, seed=1),
}


@pytest.mark.parametrize("variant", list(VARIANTS))
@pytest.mark.parametrize("name", list(GRAPHS))
def test_collapsed_cycles_match_oracle(name, variant):
    """The cycle is the same operator with its sums in another order: 1e-10,
    the bound the per-level cycles are held to (test_cycle_matches_oracle)."""
    g, kw = GRAPHS[name](), VARIANTS[variant]
    d = ligmg_amd.Solver(g, ligmg_amd.Options(precision=_ffi.PREC_MIXED, **kw))
    r = O.OracleSolver(g, O.default_options(**kw))
    base = 1 if d.level_info(0)[0] == _ffi.LEVEL_ELIM else 0
    rng = np.random.default_rng(8)
    for l in range(base, d.num_levels()):
        n = d.level_info(l)[1]
        u = rng.standard_normal(n)
        u -= u.mean()
        ref = r.apply_cycle(l, u)
        tol = 1e-10 * max(np.linalg.norm(ref), 1e-300)
        assert np.linalg.norm(d.apply_cycle(l, u) - ref) <= tol, (l, n)
        z32 = d.apply_cycle(l, u, _ffi.PREC_MIXED)
        assert np.linalg.norm(z32 - ref) <= 1e-4 * np.linalg.norm(ref) + 1e-30, (l, n)


@pytest.mark.parametrize("k", [1, 3, 8, 16, 40])
@pytest.mark.parametrize("prec", [_ffi.PREC_FP64, _ffi.PREC_MIXED])
def test_collapsed_batch_and_blocks(k, prec):
    """A union of graphs (the collapsed matrix is block diagonal) in batches
    of every dense kernel's width, against single solves."""
    gs = [graphs.barabasi_albert(n, 4, seed=s) for s, n in enumerate([900, 120, 2500])]
    u = graphs.union(gs)
    s = ligmg_amd.Solver(u, ligmg_amd.Options(precision=prec, outer_ksp_type=_ffi.KSP_FCG), comp_ptr=u.comp_ptr)
    B = graphs.rhs(u.n, k, 3, comp_ptr=u.comp_ptr).reshape(u.n, k, order="F")
    X, info, its = s.solve_batch(B)
    assert info.status == _ffi.CONVERGED and info.full_rel_residual <= 1e-7
    for c in {0, k - 1}:
        x = s.solve(np.ascontiguousarray(B[:, c])).solution
        assert np.linalg.norm(X[:, c] - x) <= 1e-7 * np.linalg.norm(x)


@pytest.mark.parametrize("kw", [{}, {"precision": _ffi.PREC_MIXED, "outer_ksp_type": _ffi.KSP_FCG},
                                {"outer_ksp_type": _ffi.KSP_FGMRES}, {"kcycle": 1, "outer_ksp_type": _ffi.KSP_FCG}])
def test_empty_coarsest_level(kw):
    """min_size = 0 coarsens on until an elimination takes every vertex: the
    levels below are empty, and nothing is launched for them."""
    g = graphs.barabasi_albert(300, 3, seed=4)
    s = ligmg_amd.Solver(g, ligmg_amd.Options(min_size=0, **kw))
    assert s.level_info(s.num_levels() - 1)[1] == 0
    info = s.solve(graphs.rhs(g.n, 1, 0))
    assert info.status == _ffi.CONVERGED and info.rel_residual() <= 1e-8


@pytest.mark.parametrize("k", [1, 3, 8, 16, 33])
@pytest.mark.parametrize("kw", [{}, {"kcycle": 1, "outer_ksp_type": _ffi.KSP_FCG},
                                {"kcycle": 1, "precision": _ffi.PREC_MIXED, "outer_ksp_type": _ffi.KSP_FCG}])
@pytest.mark.parametrize("name", ["one", "union"])
def test_empty_coarsest_level_batch(name, kw, k):
    """The same in batches, at a width of every dense kernel: one graph
    (collapsed in V-cycles, not in K-cycles), and a union of stars whose
    first level of at most 2048 vertices is the empty one."""
    star = graphs.from_edges(4, np.zeros(3, np.int64), np.arange(1, 4), np.ones(3))
    u = graphs.union([graphs.barabasi_albert(300, 3, seed=4)] if name == "one" else [star] * 2100)
    print(f"{name} {kw} k={k} n={u.n}", flush=True)
    s = ligmg_amd.Solver(u, ligmg_amd.Options(min_size=0, **kw), comp_ptr=u.comp_ptr)
    assert s.level_info(s.num_levels() - 1)[1] == 0
    B = graphs.rhs(u.n, k, 3, comp_ptr=u.comp_ptr).reshape(u.n, k, order="F")
    X, info, its = s.solve_batch(B)
    assert info.status == _ffi.CONVERGED and info.full_rel_residual <= 1e-7
    x = s.solve(np.ascontiguousarray(B[:, k - 1])).solution
    A = u.to_scipy()
    assert np.linalg.norm(A @ (X[:, k - 1] - x)) <= 2e-7 * np.linalg.norm(B[:, k - 1])
