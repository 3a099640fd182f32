"""The preconditioned CG variants where CG does not bring the residual down at its first check and plain V-cycles
finish the solve: a plane Laplacian scaled on both sides, whose first CG step moves the residual from rows of
scale 1 to rows of scale 1000."""
import functools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@functools.lru_cache
def scaled_plane(m):
    """The five-point operator on (2 m + 1)² points, scaled, linear interpolation from every second point, the
    coarse operator, and a right-hand side on the rows of scale 1."""
    import scipy.sparse as sp

    n1 = 2 * m + 1
    T = sp.diags([-np.ones(n1 - 1), 2 * np.ones(n1), -np.ones(n1 - 1)], [-1, 0, 1])
    A = sp.kron(sp.identity(n1), T) + sp.kron(T, sp.identity(n1))
    entries = [((i * n1 + j), c[0] * (m + 2) + c[1], 1.0 if i % 2 == 0 and j % 2 == 0 else 0.5)
               for i in range(n1) for j in range(n1) for c in {(i // 2, j // 2), ((i + 1) // 2, (j + 1) // 2)}]
    r, c, v = zip(*entries)
    P = sp.csr_matrix((v, (r, c)), shape=(n1 * n1, (m + 2) ** 2))
    P = P[:, np.flatnonzero(np.asarray(P.sum(0)).ravel())]
    s = np.where(np.arange(n1 * n1) % 7 == 3, 1.0, 1000.0)
    A = sp.csr_matrix(sp.diags(s) @ A @ sp.diags(s))
    P = sp.csr_matrix(sp.diags(1 / s) @ P)
    R = sp.csr_matrix(P.T)
    Ac = sp.csr_matrix(R @ A @ P)
    for M in (A, P, R, Ac):
        M.sort_indices()
    b = np.where(s == 1.0, np.random.default_rng(m).standard_normal(n1 * n1), 0.0)
    return A, Ac, R, P, b


@functools.lru_cache
def first_drop(m):
    """‖r‖ after CG's first step over ‖b‖, with one Gauss-Seidel V(1,1) cycle as preconditioner."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sla

    A, Ac, R, P, b = scaled_plane(m)
    L, U = sp.tril(A, format="csr"), sp.triu(A, format="csr")
    z = sla.spsolve_triangular(L, b)
    z = z + P @ (np.linalg.pinv(Ac.toarray()) @ (R @ (b - A @ z)))
    z = z + sla.spsolve_triangular(U, b - A @ z, lower=False)
    q = A @ z
    return np.linalg.norm(b - (b @ z) / (z @ q) * q) / np.linalg.norm(b)


@pytest.mark.parametrize("m", [15, 27])  # 961 rows: one workgroup a cycle; 3,025: panel sweeps
@pytest.mark.parametrize("variant", ["plain", "mixed", "pcg", "pcg_mixed"])
@pytest.mark.parametrize("graph", [True, False])
def test_every_variant_converges(cs, m, variant, graph, monkeypatch):
    import torch

    if not graph:
        monkeypatch.setenv("DEC_MG_NO_GRAPH", "1")
    A, Ac, R, P, b = scaled_plane(m)
    assert first_drop(m) > 10  # a rate of 0.9 hands over to plain cycles
    md = cs.MultigridData.from_matrices([A, Ac], [R], [P], steps=2)
    x, cycles, rr = cs.solve(md, torch.tensor(b, device="cuda"), tol=1e-9, max_cycles=60, variant=variant, steps=1)
    x = x.cpu().numpy()
    assert cycles > 5
    assert rr <= 1e-9 and np.linalg.norm(b - A @ x) <= 1.01e-9 * np.linalg.norm(b)
