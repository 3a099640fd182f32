"""The learned smoother's scale at the sizes where its loads per thread change, and the error loss with rows
of R of at most 8 entries (all loads at once) and of more (slot by slot), against the float64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ring(cs, n, agg):
    import learned as LO
    import scipy.sparse as sp

    i = np.arange(n)
    W = sp.csr_matrix((np.ones(2 * n), (np.r_[i, i], np.r_[(i + 1) % n, (i - 1) % n])), shape=(n, n))
    A = (sp.diags(np.full(n, 2.5)) - W).tocsr()
    m = -(-n // agg)
    R = sp.csr_matrix((np.full(n, 1.0 / agg), (i // agg, i)), shape=(m, n))
    P = sp.csr_matrix((np.ones(n), (i, i // agg)), shape=(n, m))
    Ac = (sp.diags(np.full(m, 2.5)) - sp.diags(np.ones(m - 1), 1) - sp.diags(np.ones(m - 1), -1)).tocsr()
    for M in (A, R, P, Ac):
        M.sort_indices()
    csr = lambda M: (M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data.astype(np.float64))  # noqa: E731
    md = cs.MultigridData.from_matrices([csr(A), csr(Ac)], [csr(R)], [csr(P)], steps=2)
    lv = LO.Level(*csr(A), R=LO.Csr(*csr(R), ncols=n), Pr=LO.Csr(*csr(P), ncols=m))
    nn = cs.LearnedSmoother(md, seed=8)
    p = nn.get_params().astype(np.float64)
    p = (p + 0.1 * np.random.default_rng(4).standard_normal(p.size)).astype(np.float32)
    nn.set_params(p)
    return nn, lv, p.astype(np.float64)


@pytest.mark.parametrize("n", [65536, 65537, 262144, 262145])
def test_scale_at_its_loads_per_thread(O, cs, n):
    import learned as LO
    import torch

    nn, lv, p = ring(cs, n, 60)
    r = O.uniform_form(3, n).astype(np.float32)
    r[-1] = 40.0 * np.sqrt(n)  # the last row carries the scale
    c = nn.forward(0, torch.tensor(r[None], device="cuda"), precise=True).cpu().numpy()[0]
    ref, _ = LO.forward(p, lv, r.astype(np.float64))
    # float32 arithmetic throughout, as for the levels of a sphere
    assert np.linalg.norm(c - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("n,agg", [(65, 2), (640, 4), (1003, 8), (1003, 9), (640, 12)])
def test_error_loss_by_row_width(O, cs, n, agg):
    import learned as LO
    import torch

    nn, lv, p = ring(cs, n, agg)
    R = np.stack([O.uniform_form(20 + i, n) for i in range(3)]).astype(np.float32)
    E = np.stack([O.uniform_form(40 + i, n) for i in range(3)]).astype(np.float32)
    loss, g = nn.loss_grad(0, torch.tensor(R, device="cuda"), torch.tensor(E, device="cuda"))
    lref, gref = LO.loss_err_grad(p, lv, R.astype(np.float64), E.astype(np.float64))
    # activations and weights of 8-bit mantissas in the dense layers, as for a sphere's levels
    assert loss == pytest.approx(lref, rel=3e-2)
    assert np.linalg.norm(g - gref) <= 0.1 * np.linalg.norm(gref)
