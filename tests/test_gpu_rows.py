"""The row-kernel SpMV (groups of lanes straight from memory) and the rule
that picks it, against scipy: mean row lengths of several lane counts, and
longest rows on both sides of the limit of 32 entries a lane."""
import numpy as np
import pytest
import scipy.sparse as sp

import ligmg_amd
from ligmg_amd import _ffi, graphs

pytestmark = pytest.mark.gpu


def ring(n, reach, hub):
    """Every vertex joined to the `reach` next ones; vertex 0 to `hub` others."""
    i = np.arange(n)
    u = np.concatenate([i] * reach + [np.zeros(hub, np.int64)])
    v = np.concatenate([(i + d + 1) % n for d in range(reach)] + [np.arange(reach + 1, reach + 1 + hub)])
    w = np.random.default_rng(n + reach + hub).uniform(0.5, 2.0, len(u))
    return graphs.from_edges(n, u, v, w)


@pytest.mark.parametrize("n,reach,hub,lanes", [(9, 1, 0, 1), (300, 1, 25, 1), (300, 1, 29, 1), (300, 1, 30, 0), (257, 3, 0, 2),
                                               (500, 4, 60, 4), (500, 4, 119, 4), (500, 4, 120, 0), (500, 4, 200, 0),
                                               (1500, 8, 120, 8), (1500, 8, 200, 8), (1500, 8, 239, 8), (1500, 8, 240, 0),
                                               (2000, 20, 1900, 0), (700, 300, 0, 64)])
def test_level_spmv_rows(n, reach, hub, lanes):
    g = ring(n, reach, hub)
    s = ligmg_amd.Solver(g, ligmg_amd.Options(precision=_ffi.PREC_MIXED, elim_degree=0, always_elim=0))
    rp, ci, v = s.level_matrix(0)
    assert s.level_plan(0)[1] == lanes  # the kernel this case is there for
    A = sp.csr_matrix((v, ci, rp), shape=(n, n))
    x = np.random.default_rng(0).standard_normal(n)
    bound = abs(A) @ abs(x) * np.diff(rp).max()  # one rounding per term
    assert (np.abs(s.level_spmv(0, x) - A @ x) <= 2.0 ** -52 * bound).all()
    assert (np.abs(s.level_spmv(0, x, _ffi.PREC_MIXED) - A @ x) <= 4 * 2.0 ** -24 * (abs(A) @ abs(x))).all()


@pytest.mark.parametrize("nx", [2896, 2900])
def test_reduction_segments_are_capped(nx):
    """8,386,816 and 8,410,000 vertices, on both sides of 2048 segments of
    4096 rows: a block never has more, and the norms are numpy's."""
    g = graphs.grid2d(nx, nx)
    s = ligmg_amd.Solver(g, ligmg_amd.Options(always_elim=0, top_elim=0, iters=2))
    n = s.level_info(0)[1]
    assert n == g.n and s.level_plan(0)[2] == (2048 if nx == 2896 else -(-n // 6144))
    b = graphs.rhs(n, 1, 0)
    info = s.solve(b)
    r = b - g.to_scipy() @ info.solution
    assert info.residuals[0] == pytest.approx(np.linalg.norm(b), rel=1e-12)
    assert info.residuals[-1] == pytest.approx(np.linalg.norm(r), rel=1e-7)  # recurrence and true residual
    assert info.full_rel_residual == pytest.approx(np.linalg.norm(r) / np.linalg.norm(b), rel=1e-9)
