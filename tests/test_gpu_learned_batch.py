"""Batches on the learned smoother's tile kernels: tiles of 64 rows, several samples in one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows: 42 and 162 (one and three tiles), 642 (not a multiple of 64), 10242 (more tiles than a launch has
# wavefronts per XCD at 8 samples); the error loss needs a coarser level below
@pytest.mark.parametrize("level,base,levels", [(0, 0, 1), (0, 1, 1), (0, 1, 2), (0, 1, 4)])
@pytest.mark.parametrize("batch", [2, 8])
@pytest.mark.parametrize("kind", ["residual", "error"])
def test_batch_equals_its_samples(O, cs, level, base, levels, batch, kind):
    """A batch's forward is its samples' own, bit for bit, and its loss and gradient are their means: the
    scale 1/B (a power of two) changes no rounding, so only the order of the float32 sums differs.  Each
    sum has at most 8 * 10242 terms added pairwise or in runs of up to some tens: 1e-5 of the norm of the
    samples' gradients holds well."""
    import torch

    md = cs.MultigridData(cs.icosphere(base), cs.BinarySubdivision, levels, cs.DiagonalHodge, 2, project=True)
    nn = cs.LearnedSmoother(md, seed=3)
    rng = np.random.default_rng(5)
    nn.set_params((nn.get_params() + 0.1 * rng.standard_normal(nn.nparams)).astype(np.float32))
    n = md.sizes[level]
    R = torch.tensor(np.stack([O.uniform_form(70 + i, n) for i in range(batch)]), dtype=torch.float32, device="cuda")
    E = torch.tensor(np.stack([O.uniform_form(90 + i, n) for i in range(batch)]), dtype=torch.float32, device="cuda")
    c = nn.forward(level, R)
    loss, g = nn.loss_grad(level, R, E if kind == "error" else None)
    one = [nn.loss_grad(level, R[i].contiguous(), E[i].contiguous() if kind == "error" else None) for i in range(batch)]
    for i in range(batch):
        assert torch.equal(c[i], nn.forward(level, R[i].contiguous()))
    assert loss == pytest.approx(np.mean([x[0] for x in one]), rel=1e-12)
    gs = np.stack([x[1] for x in one]).astype(np.float64)
    assert np.linalg.norm(g - gs.mean(0)) <= 1e-5 * np.linalg.norm(gs, axis=1).mean()
    # the float32 path on the same samples: every parameter's gradient, so that no block of them is missed
    # (BF16 activations: a few percent of each block's norm, as in the oracle's comparison)
    _, gp = nn.loss_grad(level, R, E if kind == "error" else None, precise=True)
    cut = np.cumsum([0, 64, 32, 2048, 32, 2048, 32, 32, 1, 1])
    for a, b in zip(cut[:-1], cut[1:]):
        assert np.linalg.norm(g[a:b] - gp[a:b]) <= 0.1 * np.linalg.norm(gp), (a, b)
