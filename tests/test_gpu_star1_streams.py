"""The geometric ⋆1⁻¹ applied on two streams in turn: a call returns when its solve has let go of the operator's
work vectors, so nothing orders the streams between calls."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("center", ["Circumcenter", "Barycenter"])  # conjugate gradients, BiCGSTAB
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("k", [1, 4])
def test_alternating_streams(cs, center, dtype, k):
    import torch

    td = getattr(torch, dtype)
    m = cs.dualize(cs.icosphere(k), getattr(cs, center))
    op = cs.dec_inv_hodge_star(1, m, cs.GeometricHodge, cast_float=td)
    xs = [cs.fill_uniform(torch.empty(m.ne, dtype=td, device="cuda"), 7 + i) for i in range(60)]
    want = [op.apply(x) for x in xs]
    outs = [torch.full_like(x, 9.0) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for i, (x, out) in enumerate(zip(xs, outs)):
        op.apply(x, out=out, stream=streams[i % 2])
    torch.cuda.synchronize()
    for out, w in zip(outs, want):
        assert torch.equal(out, w)
