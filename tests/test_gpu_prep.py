"""Device graph preprocessing through the C ABI against the oracle, bit for
bit: component labels, the largest component's renumbering and submatrix,
and the adjacency -> Laplacian conversion (canonical-order row sums)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle_ffi as O
import ligmg_amd
from ligmg_amd import _ffi, graphs, prep
from test_prep import random_components

pytestmark = pytest.mark.gpu


def adjacency_of(g):
    """The weighted adjacency matrix behind a generated Laplacian."""
    A = -g.to_scipy()
    A.setdiag(0)
    A.eliminate_zeros()
    A = A.tocsr()
    A.sort_indices()
    return A


def cases():
    yield "components7", random_components(11)
    yield "components_big", random_components(12, parts=40, isolated=300)
    g = graphs.rmat_config(12, "lognormal", pendants=True)
    yield "rmat12", adjacency_of(g)
    u = graphs.union([graphs.barabasi_albert(n, 3, seed=s) for s, n in enumerate([900, 300, 900])])
    yield "ba_union_tie", adjacency_of(u)


@pytest.mark.parametrize("mem", ["host", "device"])
@pytest.mark.parametrize("name,A", list(cases()))
def test_prep_matches_oracle(name, A, mem):
    import torch
    print(f"case={name} n={A.shape[0]} nnz={A.nnz} mem={mem}", flush=True)
    rp, ci, v = A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(np.float64)
    if mem == "device":
        dev = torch.device("cuda:0")
        args = (torch.from_numpy(rp).to(dev), torch.from_numpy(ci).to(dev), torch.from_numpy(v).to(dev))
        back = lambda t: t.cpu().numpy()  # noqa: E731
    else:
        args = (rp, ci, v)
        back = lambda t: t  # noqa: E731
    lab, k = prep.components(args)
    rlab, rk = O.components(rp, ci)
    assert k == rk and np.array_equal(back(lab), rlab)
    orp, oci, ov, nid = prep.largest_component(args)
    r = O.largest_component(rp, ci, v)
    for a, b in zip((orp, oci, ov, nid), r):
        assert np.array_equal(back(a), b)
    lrp, lci, lv = prep.adjacency_to_laplacian(args)
    r = O.adjacency_to_laplacian(rp, ci, v)
    for a, b in zip((lrp, lci, lv), r):
        assert np.array_equal(back(a), b)


def test_prep_full_size_rmat_pipeline():
    """R-MAT 20 adjacency (as generated, LCC already taken): components,
    largest component and Laplacian on the device against the oracle, and
    the resulting Laplacian solves."""
    g = graphs.rmat_config(20, "uniform")
    A = adjacency_of(g)
    # add isolated vertices and a small separate component at the end
    n0 = A.shape[0]
    extra = sp.coo_matrix((np.ones(2), ([n0 + 1, n0 + 2], [n0 + 2, n0 + 1])), shape=(n0 + 5, n0 + 5))
    A = (sp.block_diag([A, sp.csr_matrix((5, 5))]) + extra).tocsr()
    A.sort_indices()
    rp, ci, v = A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data
    lab, k = prep.components((rp, ci, v))
    rlab, rk = O.components(rp, ci)
    assert k == rk == 5 and np.array_equal(lab, rlab)
    orp, oci, ov, nid = prep.largest_component((rp, ci, v))
    assert len(orp) - 1 == n0 and np.array_equal(nid[:n0], np.arange(n0))
    lrp, lci, lv = prep.adjacency_to_laplacian((orp, oci, ov))
    rl = O.adjacency_to_laplacian(orp, oci, ov)
    assert all(np.array_equal(a, b) for a, b in zip((lrp, lci, lv), rl))
    s = ligmg_amd.Solver((lrp, lci, lv))
    b = graphs.rhs(n0, 1, 1)
    info = s.solve(b)
    assert info.rel_residual() <= 1e-8


def test_invalid_csr_is_rejected_before_use():
    """Malformed input becomes an error code: row pointers are checked
    before any column is read, columns before any gather."""
    lib = _ffi.solver_lib()
    import ctypes as C
    rp = np.array([0, 2, 1, 3], np.int32)  # decreasing
    ci = np.array([0, 1, 2], np.int32)
    lab = np.empty(3, np.int32)
    k = C.c_int64()
    assert lib.ligmg_components(3, rp.ctypes.data, ci.ctypes.data, _ffi.MEM_HOST, lab.ctypes.data,
                                C.byref(k)) == _ffi.ERR_INVALID
    rp = np.array([0, 2, 3, 3], np.int32)
    ci = np.array([0, 7, 1], np.int32)  # column out of range
    assert lib.ligmg_components(3, rp.ctypes.data, ci.ctypes.data, _ffi.MEM_HOST, lab.ctypes.data,
                                C.byref(k)) == _ffi.ERR_INVALID
    assert b"out of range" in lib.ligmg_last_error()
    # the solver checks the same and also wants sorted rows
    g = graphs.grid2d(4, 4)
    ci2 = g.colind.copy()
    ci2[1], ci2[2] = ci2[2], ci2[1]
    with pytest.raises(ligmg_amd.LigmgError):
        ligmg_amd.Solver((g.rowptr, ci2, g.vals))


@pytest.mark.parametrize("n,hub,diagonal", [(1, 0, 0.0), (70, 0, 0.5), (700, 64, 1.0), (3000, 1025, 0.0),
                                            (3000, 2999, 0.3), (5000, 4096, 0.5)])
def test_prep_entry_chunks(n, hub, diagonal):
    """Passes over stored entries in chunks of 1024: rows that cross chunks,
    empty rows, hub rows, stored and missing diagonals, one-sided patterns,
    and a submatrix that drops entries of its rows and reorders them."""
    import torch
    rng = np.random.default_rng(n + hub)
    A = sp.random(n, n, density=min(1.0, 3.0 / n), random_state=rng, format="lil")
    A[rng.integers(0, n, n // 5), :] = 0
    if hub:
        A[n // 2, rng.permutation(n)[:hub]] = 1.5
    A.setdiag(np.where(rng.random(n) < diagonal, 2.0, 0.0))
    A = A.tocsr()
    A.eliminate_zeros()
    A.sort_indices()
    rp, ci, v = A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(np.float64)
    dev = torch.device("cuda:0")
    d = tuple(torch.from_numpy(a).to(dev) for a in (rp, ci if len(ci) else np.zeros(1, np.int32), v if len(v) else np.zeros(1)))
    lab, k = prep.components(d)
    nc, c = sp.csgraph.connected_components(A, directed=False)
    top = np.full(nc, -1)
    np.maximum.at(top, c, np.arange(n))
    assert k == nc and np.array_equal(lab.cpu().numpy(), top[c])
    L = prep.adjacency_to_laplacian(d)
    for a, b in zip(L, O.adjacency_to_laplacian(rp, ci, v)):
        assert np.array_equal(a.cpu().numpy(), b)
    keep = rng.permutation(n)[:max(1, 2 * n // 3)]  # new id of kept vertex keep[i]: i
    nid = np.full(n, -1, np.int32)
    nid[keep] = np.arange(len(keep))
    sub = A[np.sort(keep)][:, np.sort(keep)].tocoo()  # entries in the input's column order
    rows, cols = nid[np.sort(keep)[sub.row]], nid[np.sort(keep)[sub.col]]
    order = np.lexsort((np.arange(len(rows)), rows))
    dn = torch.from_numpy(nid).to(dev)
    orp = torch.empty(len(keep) + 1, dtype=torch.int32, device=dev)
    oci = torch.empty(max(1, sub.nnz), dtype=torch.int32, device=dev)
    ov = torch.empty(max(1, sub.nnz), dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    lib = _ffi.solver_lib()
    args = (n, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), dn.data_ptr(), len(keep), _ffi.MEM_DEVICE)
    assert lib.ligmg_extract(*args, orp.data_ptr(), oci.data_ptr(), ov.data_ptr()) == 0
    assert np.array_equal(np.diff(orp.cpu().numpy()), np.bincount(rows, minlength=len(keep)))
    assert np.array_equal(oci.cpu().numpy()[:sub.nnz], cols[order])
    assert np.array_equal(ov.cpu().numpy()[:sub.nnz], sub.data[order])
    # outputs that overlap the inputs: the same result
    assert lib.ligmg_extract(*args, orp.data_ptr(), d[1].data_ptr(), d[2].data_ptr()) == 0
    assert np.array_equal(d[1].cpu().numpy()[:sub.nnz], cols[order])
    assert np.array_equal(d[2].cpu().numpy()[:sub.nnz], sub.data[order])
    dn[int(keep[0])] = len(keep)
    torch.cuda.synchronize()
    assert lib.ligmg_extract(*args, orp.data_ptr(), oci.data_ptr(), ov.data_ptr()) == _ffi.ERR_INVALID


@pytest.mark.parametrize("scale", [14, 15, 16, 17])
def test_prep_chunk_sizes(scale):
    """Entry counts whose passes take chunks of 128 to 1024 entries (64 is in
    the cases above), with hubs that cross many of them."""
    import torch
    A = adjacency_of(graphs.rmat_config(scale, "lognormal", pendants=True))
    assert (1 << 18) << (scale - 14) < A.nnz and (scale == 17 or A.nnz <= (1 << 19) << (scale - 14))
    print(f"scale={scale} n={A.shape[0]} nnz={A.nnz}", flush=True)
    n, (rp, ci, v) = A.shape[0], (A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    d = tuple(torch.from_numpy(a).cuda() for a in (rp, ci, v))
    lab, k = prep.components(d)
    nc, c = sp.csgraph.connected_components(A, directed=False)
    top = np.full(nc, -1)
    np.maximum.at(top, c, np.arange(n))
    assert k == nc and np.array_equal(lab.cpu().numpy(), top[c])
    for got, want in ((prep.adjacency_to_laplacian(d), O.adjacency_to_laplacian(rp, ci, v)),
                      (prep.largest_component(d), O.largest_component(rp, ci, v))):
        for a, b in zip(got, want):
            assert np.array_equal(a.cpu().numpy(), b)
