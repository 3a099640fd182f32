"""The CG smoother's one-workgroup kernels at the edges of their rows per thread (512 threads of 1, 2, 4, 6
and 7 rows), the two-level tail with one and two rows per thread of the coarsest level, and the levels just
above them, against the textbook recurrence in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(n, halve):
    """A five-point operator on n points in rows of 37, aggregates of 4, and their restriction; with `halve`
    every aggregate passes half of its neighbour's value too (rows of P with two entries)."""
    import scipy.sparse as sp

    i = np.arange(n)
    W = sp.coo_matrix((n, n))
    for d in (1, 37):
        W = W + sp.coo_matrix((np.ones(n - d) * (1.0 + 0.3 * (i[:-d] % 3)), (i[:-d], i[d:])), shape=(n, n))
    W = (W + W.T).tocsr()
    A = (sp.diags(np.asarray(W.sum(1)).ravel() + 0.05) - W).tocsr()
    nc = -(-n // 4)
    P = sp.csr_matrix((np.ones(n), (i, i // 4)), shape=(n, nc))
    if halve:
        odd = i[(i % 4 == 3) & (i // 4 + 1 < nc)]
        P = P.tolil()
        for k in odd:
            P[k, k // 4], P[k, k // 4 + 1] = 0.5, 0.5
        P = P.tocsr()
    R = (P.T / 4).tocsr()
    for M in (A, P, R):
        M.sort_indices()
    return A, R, P


def cg(A, b, u, steps):
    r = b - A @ u
    p, g = r, r @ r
    stop = np.sqrt(np.finfo(float).eps) * (1 + np.sqrt(g))
    if np.sqrt(g) <= stop:
        return u
    for _ in range(steps):
        q = A @ p
        a = g / (p @ q)
        u, r = u + a * p, r - a * q
        g, old = r @ r, g
        if np.sqrt(g) <= stop:
            break
        p = r + g / old * p
    return u


def cycle(As, Rs, Ps, k, u, b, mu, steps):
    u = cg(As[k], b, u, steps)
    if k + 1 == len(As):
        return u
    bc = Rs[k] @ (b - As[k] @ u)
    z = cycle(As, Rs, Ps, k + 1, np.zeros(len(bc)), bc, mu, steps)
    if mu > 1:
        z = cycle(As, Rs, Ps, k + 1, z, bc, mu - 1, steps)
    return cg(As[k], b, u + Ps[k] @ z, steps)


@pytest.mark.parametrize("n", [511, 512, 513, 1025, 2048, 2049, 3073, 3584, 3585, 4097])
@pytest.mark.parametrize("mu,steps,halve", [(1, 3, False), (2, 3, True), (3, 2, True), (2, 1, False)])
def test_cycles_match_numpy(cs, n, mu, steps, halve):
    """n: the second coarsest level; a finer one of 4 n rows (several workgroups) above it.  The dot
    products add in another order and β comes from the same sums as α, so u agrees to rounding times the
    condition of a few steps: 1e-11 holds with room."""
    import torch

    if n > 3500:
        As, Rs, Ps = [], [], []
    else:  # with a level above, whose rows are n's aggregates
        A, R, P = chain(4 * n, halve)
        As, Rs, Ps = [A], [R], [P]
    A, R, P = chain(n, halve)
    As, Rs, Ps = As + [A], Rs + [R], Ps + [P]
    As.append(chain(R.shape[0], False)[0])
    md = cs.MultigridData.from_matrices(As, Rs, Ps, steps=steps)
    rng = np.random.default_rng(n)
    b = rng.standard_normal(As[0].shape[0])
    u0 = rng.standard_normal(As[0].shape[0])
    want = u0
    for _ in range(2):
        want = cycle(As, Rs, Ps, 0, want, b, mu, steps)
    u = torch.tensor(u0, device="cuda")
    cs.multigrid_mu_cycles(u, torch.tensor(b, device="cuda"), md, 2, cs.cg, mu, steps=steps)
    got = u.cpu().numpy()
    assert np.linalg.norm(got - want) <= 1e-11 * np.linalg.norm(want)


@pytest.mark.parametrize("scale", [0.0, 1e-10])
def test_small_residuals_stop_at_once(cs, scale):
    """A residual below the threshold leaves u as it is, on every kind of level (its norm, sqrt(2800) scale =
    5.3e-9, lies under sqrt(eps) = 1.5e-8)."""
    import torch

    A, R, P = chain(4 * 700, True)
    A2, R2, P2 = chain(700, True)
    A3 = chain(175, False)[0]
    md = cs.MultigridData.from_matrices([A, A2, A3], [R, R2], [P, P2], steps=3)
    b = torch.full((2800,), scale, dtype=torch.float64, device="cuda")
    u = torch.zeros_like(b)
    cs.multigrid_vcycles(u, b, md, 2)
    assert not u.any()
