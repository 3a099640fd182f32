"""The fused launches of the dual-dual composites and of the geometric ⋆1⁻¹
against the separate operators: ℒ_dd's last launch adds the products of d̃0 and
⋆1 that separate applications write; the solve's first iteration forms D⁻¹b at
the columns, accumulates -x, and answers the host through a pinned word."""
import numpy as np
import pytest

from test_gpu_ops import F64_TOL, gpu_mesh_like, rel, to_dev

pytestmark = pytest.mark.gpu


def mesh(O, cs, name):
    """grid: hanging boundary and ragged rows; ico0: fewer edges than a
    workgroup; ico5: edges for several workgroups, not a multiple of one;
    ico7: more edges than the solve's grid has threads."""
    if name.startswith("grid"):
        om = O.triangulated_grid(7.3, 5.1, 0.31, 0.29)
    else:
        om = O.icosphere(int(name[3]))
    gm = gpu_mesh_like(cs, om)
    cs.dualize(gm, cs.Barycenter if name.endswith("bary") else cs.Circumcenter)
    return gm


MESHES = ["grid", "grid_bary", "ico0", "ico5", "ico5_bary", "ico7"]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", MESHES)
def test_lie_equals_its_parts(O, cs, name, dtype):
    import torch

    td = torch.float64 if dtype == "f64" else torch.float32
    gm = mesh(O, cs, name)
    lie = cs.lie_derivative_dd(1, 1, gm, cast_float=td)
    n = cs.dec_dual_derivative(0, gm, cast_float=td).rows
    f, g = (to_dev(torch, O.uniform_form(80 + i, n), td) for i in range(2))
    i11 = cs.interior_product_dd(1, 1, gm, cast_float=td)
    i12 = cs.interior_product_dd(1, 2, gm, cast_float=td)
    d0, d1 = cs.dec_dual_derivative(0, gm, cast_float=td), cs.dec_dual_derivative(1, gm, cast_float=td)
    parts = -(d0(i11(f, g))) - i12(f, d1(g))
    assert torch.equal(lie(f, g), parts)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", MESHES)
def test_dual_laplacian1_equals_its_parts(O, cs, name, dtype):
    """Δᵈ(1) x = ⋆1 d0 (⋆0⁻¹ d̃1 x) + d̃0 ⋆2 d1 ⋆1⁻¹ x with its factors applied one by
    one.  The products' rows hold few terms, so forming them differs from applying
    the factors by a few roundings of the largest entries."""
    import torch

    td = torch.float64 if dtype == "f64" else torch.float32
    gm = mesh(O, cs, name)
    L1 = cs.dual_laplacian(1, gm, cast_float=td)
    x = to_dev(torch, O.uniform_form(83, L1.rows), td)
    y = L1(x)
    z = x.clone()
    L1.apply(z, out=z)                              # in place
    assert torch.equal(z, y)
    H = cs.GeometricHodge
    op = lambda k, f, *a: f(k, gm, *a, cast_float=torch.float64)  # noqa: E731
    w = x.double()
    m = op(1, cs.dec_hodge_star, H)(op(0, cs.dec_differential)(op(0, cs.dec_inv_hodge_star, H)(
        op(1, cs.dec_dual_derivative)(w))))
    nz = op(0, cs.dec_dual_derivative)(op(2, cs.dec_hodge_star, H)(op(1, cs.dec_differential)(
        op(1, cs.dec_inv_hodge_star, H)(w))))
    ref = (m + nz).cpu().numpy()
    assert rel(y.cpu().numpy(), ref) <= (F64_TOL if dtype == "f64" else 1e-4)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", MESHES)
def test_inv_hodge1_edges_and_replay(O, cs, name, dtype):
    """Zero, in-place and captured solves; a replay that is still in flight when
    an eager solve starts does not answer for it."""
    import torch

    td = torch.float64 if dtype == "f64" else torch.float32
    gm = mesh(O, cs, name)
    inv = cs.dec_inv_hodge_star(1, gm, cs.GeometricHodge, cast_float=td)
    H = cs.dec_hodge_star(1, gm, cs.GeometricHodge, cast_float=td)
    n = inv.rows
    xs = [to_dev(torch, O.uniform_form(90 + i, n), td) for i in range(4)]
    ref = [inv(x) for x in xs]
    tol = F64_TOL if dtype == "f64" else 1e-4
    for x, r in zip(xs, ref):
        assert rel(-H(r).cpu().numpy(), x.cpu().numpy()) <= tol
    zero = torch.zeros(n, dtype=td, device="cuda")
    assert torch.count_nonzero(inv(zero)).item() == 0
    assert torch.equal(inv(xs[0]), ref[0])          # a stopped solve leaves nothing behind
    z = xs[1].clone()
    inv.apply(z, out=z)
    assert torch.equal(z, ref[1])
    x, out = xs[0].clone(), torch.empty_like(xs[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        inv.apply(x, out=out)
    for i in (1, 2, 3):
        x.copy_(xs[i])
        g.replay()
        eager = inv(xs[(i + 1) % 4])                # while the replay runs
        torch.cuda.synchronize()
        assert torch.equal(out, ref[i])
        assert torch.equal(eager, ref[(i + 1) % 4])
