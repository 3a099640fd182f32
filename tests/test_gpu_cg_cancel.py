"""A step of the CG smoother that cuts ‖r‖ to little more than the stopping threshold, sqrt(eps) (1 + ‖r0‖): the next
r·r, as the difference of sums a thousand million million times as large, would be its rounding error, and end the
smoothing.  On levels of one workgroup, of several, and small ones whose rows are wider than one workgroup takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cg(A, b, steps):
    u, r = np.zeros_like(b), b
    p, g = r, r @ r
    stop = np.sqrt(np.finfo(float).eps) * (1 + np.sqrt(g))
    for _ in range(steps):
        q = A @ p
        a = g / (p @ q)
        u, r = u + a * p, r - a * q
        g, old = r @ r, g
        if np.sqrt(g) <= stop:
            break
        p = r + g / old * p
    return u


# (rows, bands): one workgroup; rows of 9 slots, or more rows than one workgroup takes: a launch per step
@pytest.mark.parametrize("n,bands", [(300, 1), (300, 4), (8200, 1), (100003, 1)])
@pytest.mark.parametrize("drop", [1.6e-8, 2e-8, 1e-6])
def test_second_step_is_taken(cs, n, bands, drop):
    import scipy.sparse as sp
    import torch

    for seed in range(12):
        rng = np.random.default_rng(seed)
        i = np.arange(n)
        W = sp.coo_matrix((n, n))
        for d in range(1, bands + 1):
            W = W + sp.coo_matrix((rng.random(n - d), (i[:-d], i[d:])), shape=(n, n))
        W = W + W.T
        L = (sp.diags(np.asarray(W.sum(1)).ravel()) - W).tocsr()
        b = 1e3 * rng.standard_normal(n)
        Lb = L @ b
        spread = np.linalg.norm((b @ Lb) / (b @ b) * b - Lb) / np.linalg.norm(b)
        A = sp.csr_matrix(sp.identity(n) + drop / spread * L)  # the first step leaves ‖r‖ = drop ‖b‖
        A.sort_indices()
        md = cs.MultigridData.from_matrices([A], [], [], steps=2)
        u = torch.zeros(n, dtype=torch.float64, device="cuda")
        cs.multigrid_vcycles(u, torch.tensor(b, device="cuda"), md, 1, cs.cg, steps=2)
        want = cg(A, b, 2)
        # two steps leave drop² ‖b‖ (1e-12 at most); one would leave drop ‖b‖
        assert np.linalg.norm(u.cpu().numpy() - want) <= 2e-12 * np.linalg.norm(want), seed
