"""The dual-dual wedge on a complex of edges alone: its dual 0-form has no entries, no edge has a coface, and the
product is zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edges", [1, 2, 4, 7, 1000])  # incomplete, complete and many groups of two and four
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("degrees", [(0, 1), (1, 0)])
def test_dual_dual_wedge_is_zero(cs, edges, dtype, degrees):
    import torch

    td = getattr(torch, dtype)
    i = np.arange(edges)
    points = np.stack([np.arange(edges + 1.0), np.zeros(edges + 1), np.zeros(edges + 1)], 1)
    none = np.zeros(0, np.int32)
    m = cs.dualize(cs.mesh_from_arrays(points, i + 1, i, none, none, none), cs.Barycenter)
    op = cs.dec_wedge_product_dd(*degrees, m, cast_float=td).operator
    assert (op.rows, min(op.cols, op.cols2)) == (edges, 0)
    forms = [torch.ones(n, dtype=td, device="cuda") for n in (op.cols, op.cols2)]
    out = torch.full((edges,), 5.0, dtype=td, device="cuda")
    cs.apply_many([(op, *forms, out)])
    assert not out.any()
    if op.cols:  # (a single call takes no empty first form)
        out = torch.full((edges,), 5.0, dtype=td, device="cuda")
        op.apply(*forms, out=out)
        assert not out.any()
    else:
        with pytest.raises(Exception, match="NULL form"):
            op.apply(*forms, out=out)
