"""The cluster order of the solve layout: levels of even rows (65536 vertices
and more) follow their aggregates; nothing a caller sees changes with it."""
import numpy as np
import pytest

import ligmg_amd
from ligmg_amd import _ffi, graphs

pytestmark = pytest.mark.gpu


def shuffled_grid(nx, ny, extra=0):
    """A grid with randomly numbered vertices; `extra` vertices hang from one
    vertex (a hub among even rows)."""
    n = nx * ny
    p = np.random.default_rng(1).permutation(n)
    i = np.arange(n).reshape(nx, ny)
    u = np.concatenate([i[1:].ravel(), i[:, 1:].ravel()])
    v = np.concatenate([i[:-1].ravel(), i[:, :-1].ravel()])
    w = np.random.default_rng(2).uniform(0.5, 2.0, len(u) + extra)
    return graphs.from_edges(n + extra, np.concatenate([p[u], np.arange(n, n + extra)]),
                             np.concatenate([p[v], np.full(extra, p[0])]), w)


@pytest.mark.parametrize("prec", [_ffi.PREC_FP64, _ffi.PREC_MIXED])
@pytest.mark.parametrize("name,g", [("even", lambda: shuffled_grid(300, 301)), ("hub", lambda: shuffled_grid(300, 301, 90)),
                                    ("grid3d", lambda: graphs.grid3d(50, 41, 47, graphs.W_UNIFORM, 0.1, 10.0, 2))])
def test_cluster_layout_is_invisible(name, g, prec):
    g = g()
    assert g.n >= 1 << 16
    kw = {"precision": prec, "outer_ksp_type": _ffi.KSP_FCG}
    a = ligmg_amd.Solver(g, ligmg_amd.Options(**kw))
    b = ligmg_amd.Solver(g, ligmg_amd.Options(solve_layout=0, **kw))
    assert a.num_levels() == b.num_levels()
    # the order each is there for: degree order where a row is longer than 8
    # mean ones, cluster order where none is
    layouts = [a.level_plan(l)[0] for l in range(a.num_levels())]
    rows = [np.diff(a.level_matrix(l)[0]) for l in range(a.num_levels() - 1)]
    assert layouts == [0 if len(r) < 1 << 16 else 1 if r.max() > 8 * r.mean() else 2 for r in rows] + [0]
    assert layouts[0] == (1 if name == "hub" else 2)
    assert not any(b.level_plan(l)[0] for l in range(b.num_levels()))
    rng = np.random.default_rng(3)
    for l in range(a.num_levels()):
        assert a.level_info(l) == b.level_info(l)
        for x, y in zip(a.level_matrix(l), b.level_matrix(l)):
            assert np.array_equal(x, y)
        if l + 1 < a.num_levels():
            assert np.array_equal(a.level_map(l), b.level_map(l))
    base = 1 if a.level_info(0)[0] == _ffi.LEVEL_ELIM else 0
    u = rng.standard_normal(a.level_info(base)[1])
    u -= u.mean()
    za, zb = a.apply_cycle(base, u), b.apply_cycle(base, u)
    assert np.linalg.norm(za - zb) <= 1e-10 * np.linalg.norm(zb)  # the sums' order alone
    B = graphs.rhs(g.n, 3, 4).reshape(g.n, 3, order="F")
    x, y = a.solve(np.ascontiguousarray(B[:, 0])), b.solve(np.ascontiguousarray(B[:, 0]))
    X = a.solve_batch(B)[0]
    for s in (x.solution, X[:, 0]):
        d = (s - s.mean()) - (y.solution - y.solution.mean())
        assert np.linalg.norm(d) <= 1e-6 * np.linalg.norm(y.solution)
    assert abs(x.iters() - y.iters()) <= 1 and x.full_rel_residual <= 1e-7
