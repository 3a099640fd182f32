"""Batches of many samples on levels of fewer rows than a workgroup takes: one workgroup per sample in the
launches that write partial sums, so that their buffers go by samples and not by rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def wide(cs):
    """A ring of 41 rows with ten neighbours each (the general kernels) above one of 12."""
    import scipy.sparse as sp

    def ring(n, reach):
        i = np.arange(n)
        W = sum(sp.csr_matrix((np.ones(2 * n), (np.r_[i, i], np.r_[(i + d) % n, (i - d) % n])), shape=(n, n))
                for d in range(1, reach + 1))
        A = (sp.diags(np.asarray(W.sum(1)).ravel() + 0.5) - W).tocsr()
        A.sort_indices()
        return A

    i = np.arange(41)
    P = sp.csr_matrix((np.ones(41), (i, i * 12 // 41)), shape=(41, 12))
    R = sp.csr_matrix(P.T / 4)
    return cs.MultigridData.from_matrices([ring(41, 5), ring(12, 5)], [R], [P], steps=2)


@pytest.mark.parametrize("which", ["sphere", "wide"])
@pytest.mark.parametrize("precise", [False, True])
@pytest.mark.parametrize("level,copies", [(0, 32), (1, 2048)])
def test_many_samples_are_the_mean_of_a_few(O, cs, which, precise, level, copies):
    import torch

    md = wide(cs) if which == "wide" else cs.MultigridData(cs.icosphere(0), cs.BinarySubdivision, 1, cs.DiagonalHodge,
                                                           2, project=True)
    assert md.sizes == ([41, 12] if which == "wide" else [42, 12])
    nn = cs.LearnedSmoother(md, seed=3)
    nn.set_params((nn.get_params() + 0.1 * np.random.default_rng(5).standard_normal(nn.nparams)).astype(np.float32))
    n = md.sizes[level]

    def form(seed, rows):
        x = np.stack([O.uniform_form(seed + i, rows) for i in range(8)]).astype(np.float32)
        return torch.tensor(x, device="cuda")

    R, E = form(70, n), form(90, n) if level == 0 else None
    loss, g = nn.loss_grad(level, R, E, precise=precise)
    # a larger call on the finest level first: its rows leave room, its samples do not
    nn.loss_grad(0, form(50, md.sizes[0]).repeat(40, 1), None, precise=precise)
    many = nn.loss_grad(level, R.repeat(copies, 1), None if E is None else E.repeat(copies, 1), precise=precise)
    # (copies: a power of two, so that the scale 1 / B changes no rounding)  The loss adds doubles, the gradient
    # runs of float32 sums and then doubles: rounding to 24 bits, 1e-5 of the norm holds with room
    assert many[0] == pytest.approx(loss, rel=1e-12)
    assert np.linalg.norm(many[1] - g) <= 1e-5 * np.linalg.norm(g)
