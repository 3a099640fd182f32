"""The hybrid block Gauss-Seidel sweep in its panel form and its general form, against numpy: row widths 3 to
8 on panels, 9 and graphs whose blocks have more neighbours than a panel's threads cover on the general
kernel; one and two rows per thread; odd and even step counts; float64 cycles and float32 ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def operator(n, offsets, random_edges=0, seed=0):
    import scipy.sparse as sp

    rng = np.random.default_rng(seed)
    i = np.arange(n)
    W = sp.coo_matrix((n, n))
    for d in offsets:
        W = W + sp.coo_matrix((0.5 + rng.random(n - d), (i[:-d], i[d:])), shape=(n, n))
    for _ in range(random_edges):
        p = rng.permutation(n)
        h = n // 2
        W = W + sp.coo_matrix((0.5 + rng.random(h), (p[:h], p[h:2 * h])), shape=(n, n))
    W = W + W.T
    A = (sp.diags(np.asarray(W.sum(1)).ravel() * 1.05) - W).tocsr()
    A.sum_duplicates()
    A.sort_indices()
    return A


def sweep(A, blk, col, u, b, reverse):
    """Colours in order, neighbours in other blocks from the start of the sweep."""
    import scipy.sparse as sp

    C = A.tocoo()
    diag = A.diagonal()
    off = C.row != C.col
    same = blk[C.row] == blk[C.col]
    inner = sp.csr_matrix((C.data[off & same], (C.row[off & same], C.col[off & same])), shape=A.shape)
    outer = sp.csr_matrix((C.data[off & ~same], (C.row[off & ~same], C.col[off & ~same])), shape=A.shape)
    far, x = outer @ u, u.copy()
    order = range(col.max(), -1, -1) if reverse else range(col.max() + 1)
    for c in order:
        r = np.flatnonzero(col == c)
        x[r] = (b[r] - far[r] - (inner @ x)[r]) / diag[r]
    return x


CASES = [
    # (rows, offsets of the bands, random matchings): width 3 .. 8 on panels
    (3001, (1,), 0), (3100, (1, 57), 0), (3777, (1, 57, 58), 0), (50001, (1, 201), 0), (100003, (1, 317, 318), 0),
    (400009, (1, 631), 0), (5000, (1, 57, 58), 1),
    # wider rows, and blocks with too many neighbours: the general kernel
    (4000, (1, 2, 61, 62), 0), (6000, (1,), 3), (6000, (1,), 5),
]


@pytest.mark.parametrize("n,offsets,matchings", CASES)
@pytest.mark.parametrize("steps", [1, 2])
def test_two_level_cycles(cs, n, offsets, matchings, steps):
    import scipy.sparse as sp
    import torch

    A = operator(n, offsets, matchings, seed=n)
    nc = -(-n // (4 if n < 10000 else 200))
    agg = np.minimum(np.arange(n) * nc // n, nc - 1)
    P = sp.csr_matrix((np.ones(n), (np.arange(n), agg)), shape=(n, nc))
    half = np.arange(0, n, 3)
    P = P.tolil()
    for k in half[:-1]:
        if agg[k] + 1 < nc:
            P[k, agg[k]], P[k, agg[k] + 1] = 0.75, 0.25
    P = P.tocsr()
    R = sp.csr_matrix(P.T)
    Ac = sp.csr_matrix(R @ A @ P)
    for M in (P, R, Ac):
        M.sort_indices()
    md = cs.MultigridData.from_matrices([A, Ac], [R], [P], steps=steps)
    blk, nb = md.blocks(0)
    col, _ = md.colors(0)
    cblk, ccol = np.zeros(nc, int), md.colors(1)[0]
    rng = np.random.default_rng(n)
    b, u0 = rng.standard_normal(n), rng.standard_normal(n)

    def cycle(u):
        for _ in range(steps):
            u = sweep(A, blk, col, u, b, False)
        bc = R @ (b - A @ u)
        z = np.zeros(nc)
        for _ in range(steps):
            z = sweep(Ac, cblk, ccol, z, bc, False)
        u = u + P @ z
        for _ in range(steps):
            u = sweep(A, blk, col, u, b, True)
        return u

    want = cycle(cycle(u0))
    u = torch.tensor(u0, device="cuda")
    cs.multigrid_vcycles(u, torch.tensor(b, device="cuda"), md, 2, cs.block_gauss_seidel, steps=steps)
    # sums of at most nine products in another order, 2 (2 steps) sweeps of a contraction
    assert np.linalg.norm(u.cpu().numpy() - want) <= 1e-13 * np.linalg.norm(want)
    # every solve variant (zero starts, the float32 sweeps, CG on top) reaches its residual
    for variant in ("plain", "mixed", "pcg", "pcg_mixed"):
        x, _, rr = cs.solve(md, torch.tensor(b, device="cuda"), tol=1e-9, variant=variant, steps=2, coarse_direct=True)
        x = x.cpu().numpy()
        assert rr <= 1e-9 and np.linalg.norm(b - A @ x) <= 1.01e-9 * np.linalg.norm(b), variant
