"""Gauss-Seidel overwrites a row from its neighbours: what stood in a first-colour row that no other block reads
does not matter, an infinity or NaN included.  On panels, in the coarse tail and in the general kernels, with rows of
fewer entries than the widest."""
import numpy as np
import pytest

from test_gpu_block_sweep import operator

pytestmark = pytest.mark.gpu


# one level below (steps of panels: 3 to 8 slots); the tail; the general kernels (rows of 9 slots)
@pytest.mark.parametrize("n,offsets", [(3001, (1,)), (3777, (1, 57, 58)), (50001, (1, 201)), (700, (1, 23)),
                                       (2600, (1, 51, 52)), (4000, (1, 2, 61, 62))])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_a_row_s_own_value_does_not_enter(cs, n, offsets, value):
    import scipy.sparse as sp
    import torch

    A = operator(n, offsets, seed=n)
    nc = -(-n // (4 if n < 10000 else 200))
    P = sp.csr_matrix((np.ones(n), (np.arange(n), np.minimum(np.arange(n) * nc // n, nc - 1))), shape=(n, nc))
    R = sp.csr_matrix(P.T)
    Ac = sp.csr_matrix(R @ A @ P)
    Ac.sort_indices()
    md = cs.MultigridData.from_matrices([A, Ac], [R], [P], steps=2)
    blk, _ = md.blocks(0)
    color, _ = md.colors(0)
    C = A.tocoo()
    far = np.unique(C.col[blk[C.row] != blk[C.col]])
    rows = np.setdiff1d(np.flatnonzero(color == 0), far)
    short = rows[np.diff(A.indptr)[rows] < np.diff(A.indptr).max()]
    assert len(short)
    rng = np.random.default_rng(n)
    b, u0 = torch.tensor(rng.standard_normal(n), device="cuda"), rng.standard_normal(n)
    results = []
    for v in (0.0, value):
        u0[rows] = v
        u = torch.tensor(u0, device="cuda")
        cs.multigrid_vcycles(u, b, md, 2, cs.block_gauss_seidel, steps=2, coarse_direct=True)
        results.append(u)
    assert torch.isfinite(results[1]).all()
    assert torch.equal(*results)
