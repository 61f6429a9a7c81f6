"""Setup's row passes at the row lengths where their kernels change (0 to 9
entries around one round of eight lanes, 63 to 66 around the wavefront rows):
every result of the passes is the oracle's, bit for bit.  (The smoother's
bounds are left to tests of their own: on the 7-vertex levels met here the
order of the estimator's sums alone moves them by 8%.)"""
import numpy as np
import pytest

import ligmg_amd
import oracle_ffi as O
from ligmg_amd import _ffi, graphs
from test_gpu_parity import opts_pair

pytestmark = pytest.mark.gpu


def degrees_graph(degrees, copies, seed):
    """For every degree d and copy, a hub with d neighbours; the hubs' leaves
    come from one shared ring, so rows of many lengths interleave."""
    r = np.random.default_rng(seed)
    hubs = np.repeat(degrees, copies)
    m = 4 * int(max(degrees)) + 40
    u, v = [np.arange(m)], [(np.arange(m) + 1) % m]
    for h, d in enumerate(hubs):
        u.append(np.full(d, m + h))
        v.append(r.choice(m, d, replace=False))
    u, v = np.concatenate(u), np.concatenate(v)
    return graphs.from_edges(m + len(hubs), u, v, r.uniform(0.5, 2.0, len(u)))


@pytest.mark.parametrize("kw", [{}, {"aff_scaling": 1}, {"strength_metric": _ffi.STRENGTH_ALGEBRAIC_DISTANCE},
                                {"neighbor_of_neighbor": 1}])
@pytest.mark.parametrize("degrees", [[1, 2, 6, 7, 8, 9], [14, 15, 16, 17], [61, 62, 63, 64, 65, 66]])
def test_setup_rows(degrees, kw):
    print(f"degrees={degrees} {kw}", flush=True)
    g = degrees_graph(degrees, 37, 5)
    do, oo = opts_pair(min_size=0, **kw)
    d, r = ligmg_amd.Solver(g, do), O.OracleSolver(g, oo)
    assert d.num_levels() == r.num_levels()
    for l in range(d.num_levels()):
        assert d.level_info(l) == r.level_info(l), l
        kind = d.level_info(l)[0]
        pairs = list(zip(d.level_matrix(l), r.level_matrix(l)))
        if kind != _ffi.LEVEL_COARSE:
            pairs.append((d.level_map(l), r.level_map(l)))
        if kind == _ffi.LEVEL_AGG:
            pairs += zip(d.level_states(l), r.level_states(l))
            pairs.append((d.level_strength(l), r.level_strength(l)))
        assert all(np.array_equal(a, b) for a, b in pairs), (l, [np.array_equal(a, b) for a, b in pairs])
