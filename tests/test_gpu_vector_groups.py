"""The operators' vector loads: groups of two (float64) or four (float32) simplices, the incomplete last group
and forms at every alignment give the same bits as the element by element path."""
import pytest

pytestmark = pytest.mark.gpu


# (2 x 2 .. 5 x 4 points: every remainder of the numbers of vertices, edges and triangles by four)
@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 2), (4, 2), (5, 2), (3, 3), (5, 4), (41, 23)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_alignment_changes_no_bit(cs, nx, ny, dtype):
    import torch

    td = getattr(torch, dtype)
    m = cs.triangulated_grid(nx - 1, (ny - 1) * 0.75 ** 0.5, 1, 0.75 ** 0.5, False)
    cs.dualize(m, cs.Barycenter)
    W = lambda a, b: cs.dec_wedge_product(a, b, m, cast_float=td).operator  # noqa: E731
    ops = [W(0, 1), W(1, 0), W(1, 1), W(0, 2), cs.dec_wedge_product_dd(0, 1, m, cast_float=td).operator,
           cs.dec_wedge_product_dd(1, 0, m, cast_float=td).operator, cs.dec_differential(0, m, cast_float=td),
           cs.dec_differential(1, m, cast_float=td), cs.avg01_mat(m, cast_float=td)]
    ops += [cs.dec_hodge_star(k, m, cs.DiagonalHodge, cast_float=td) for k in range(3)]

    def form(n, off, seed):
        x = torch.empty(n + 4, dtype=td, device="cuda")
        cs.fill_uniform(x, seed)
        x[off:off + n] = cs.fill_uniform(torch.empty(n, dtype=td, device="cuda"), seed)
        return x[off:off + n]

    for i, op in enumerate(ops):
        want = None
        # one element off everything: the element by element path; then each alignment of each form
        for a, b, c in ((1, 1, 1), (0, 0, 0), (2, 2, 2), (0, 2, 0), (2, 0, 0), (0, 0, 2), (3, 0, 0), (0, 0, 1)):
            x, y = form(op.cols, a, 10 + i), form(op.cols2, b, 50 + i) if op.cols2 else None
            out = form(op.rows, c, 99)
            op.apply(x, y, out=out)
            grouped = form(op.rows, c, 98)
            cs.apply_many([(op, x, y, grouped)])
            want = out.clone() if want is None else want
            assert torch.equal(out, want) and torch.equal(grouped, want), (i, a, b, c)
