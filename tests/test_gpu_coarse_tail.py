"""The coarse tail's register/LDS launches against one launch per phase, bit for
bit: one, two and three rows per thread and the sizes around them, row widths 3 to
8 (and 9, which the general kernel takes), coarsest levels of one row, of more
than the 1024 columns that a workgroup's threads start with, restriction rows of
more than eight entries, and several smoothed levels in one tail."""
import numpy as np
import pytest

from test_gpu_block_sweep import operator

pytestmark = pytest.mark.gpu

# (rows of each level, offsets of the finest one's bands)
CASES = [
    ((2, 1), (1,)), ((5, 2), (1, 3)), ((255, 64), (1,)), ((1023, 255), (1, 37)), ((1024, 257), (1, 37, 38)),
    ((1025, 500), (1, 41)), ((2048, 1100), (1, 2)), ((2049, 150), (1, 41, 42)), ((3000, 1500), (1,)),
    ((3000, 642), (1, 61, 62)), ((2500, 625), (1, 2, 61, 62)), ((2600, 650, 160, 40), (1, 51, 52)),
    ((3000, 1900, 400), (1,)), ((4001, 2000, 1000, 500), (1,)), ((9000, 1200, 300, 75), (1, 91)),
]


def hierarchy(sizes, offsets):
    import scipy.sparse as sp

    As, Rs, Ps = [operator(sizes[0], offsets, seed=sizes[0])], [], []
    for n, nc in zip(sizes, sizes[1:]):
        i = np.arange(n)
        agg = i * nc // n
        P = sp.lil_matrix(sp.csr_matrix((np.ones(n), (i, agg)), shape=(n, nc)))
        for k in i[::3]:
            if agg[k] + 1 < nc and len(As) == 1:
                P[k, agg[k]], P[k, agg[k] + 1] = 0.75, 0.25
        P = P.tocsr()
        R = sp.csr_matrix(P.T)
        A = sp.csr_matrix(R @ As[-1] @ P)
        for M in (P, R, A):
            M.sort_indices()
        As, Rs, Ps = As + [A], Rs + [R], Ps + [P]
    return As, Rs, Ps


@pytest.mark.parametrize("sizes,offsets", CASES, ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("steps", [1, 2])
def test_tail_equals_launches_per_phase(cs, sizes, offsets, steps, monkeypatch):
    import torch

    As, Rs, Ps = hierarchy(sizes, offsets)
    rng = np.random.default_rng(sizes[0])
    b = torch.tensor(rng.standard_normal(sizes[0]), device="cuda")

    def run():
        md = cs.MultigridData.from_matrices(As, Rs, Ps, steps=steps)
        return [cs.solve(md, b, tol=1e-9, variant=v, steps=steps, coarse_direct=True) for v in ("plain", "mixed", "pcg")]

    fast = run()
    monkeypatch.setenv("DEC_MG_NO_FUSE", "1")
    monkeypatch.setenv("DEC_MG_NO_GRAPH", "1")
    for (u, c, r), (v, d, q) in zip(fast, run()):
        assert c == d and r == q and torch.equal(u, v)
        x = u.cpu().numpy()
        assert np.linalg.norm(b.cpu().numpy() - As[0] @ x) <= 1.01e-9 * np.linalg.norm(b.cpu().numpy())
