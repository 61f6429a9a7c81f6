"""The smoother's lambda_max estimate on the device (the estimator's CG in
four launches a step) against the same steps in numpy with exactly rounded
inner products: sizes around one reduction segment (4096 rows) and past one
segment a lane (64 segments), several blocks, and no steps at all."""
import numpy as np
import pytest

import lanczos_np
import ligmg_amd
from ligmg_amd import _ffi, graphs

pytestmark = pytest.mark.gpu


def chorded_ring(n):
    i = np.arange(n)
    r = np.random.default_rng(n)
    u, v = np.concatenate([i, i]), np.concatenate([(i + 1) % n, (i + 2) % n])
    return graphs.from_edges(n, u, v, r.uniform(0.5, 2.0, len(u)))


@pytest.mark.parametrize("n,iters", [(9, 0), (9, 1), (9, 2), (4095, 10), (4096, 10), (4097, 3), (4097, 10),
                                     (65 * 4096 + 1, 5)])
def test_lambda_max(n, iters):
    g = chorded_ring(n)
    print(f"n={n} iters={iters}", flush=True)
    o = ligmg_amd.Options(cheby_eig_iters=iters, elim_degree=0, always_elim=0, top_elim=0, min_size=0)
    s = ligmg_amd.Solver(g, o)
    l = next(l for l in range(s.num_levels()) if s.level_info(l)[0] == _ffi.LEVEL_AGG)
    rp, ci, v = s.level_matrix(l)
    want = lanczos_np.lambda_max(rp, ci, v, o.seed, l, iters, lanczos_np.ORDERS["exact"])
    # the sums' rounding, n * 2^-53 relative at most, grows over the steps by
    # less than 1e3 (Lanczos far from convergence)
    assert s.level_cheby(l)[1] == pytest.approx(o.cheby_upper * want, rel=max(n, 1000) * 2.0 ** -53 * 1e3)


def test_lambda_max_blocks():
    """A hierarchy of several blocks has a reduction plan by block; the
    estimate is over the whole level."""
    n = 5000
    i = np.arange(n)
    h = n // 2
    u, v = np.concatenate([i, i]), np.concatenate([(i + 1) % h + h * (i >= h), (i + 2) % h + h * (i >= h)])
    g = graphs.from_edges(n, u, v, np.random.default_rng(1).uniform(0.5, 2.0, len(u)))
    o = ligmg_amd.Options(elim_degree=0, always_elim=0, top_elim=0)
    s = ligmg_amd.Solver(g, o, comp_ptr=np.array([0, h, n]))
    rp, ci, v = s.level_matrix(0)
    want = lanczos_np.lambda_max(rp, ci, v, o.seed, 0, 10, lanczos_np.ORDERS["exact"])
    assert s.level_cheby(0)[1] == pytest.approx(o.cheby_upper * want, rel=n * 2.0 ** -53 * 1e3)
