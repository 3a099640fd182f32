"""Batched heat steps where the packed columns begin and end: rows of fewer than
7 slots (icosahedron, a fan's rim), of 7, of more (the fan's hub), and meshes of
the last size whose columns are packed and the next one, in one batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fan(cs, n):
    t = 2 * np.pi * np.arange(n) / n
    p = np.vstack([[0.0, 0.0, 0.0], np.c_[np.cos(t), np.sin(t), np.zeros(n)]])
    return cs.mesh_from_triangles(p, np.array([sorted((0, 1 + i, 1 + (i + 1) % n)) for i in range(n)]))


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_packed_columns_match_the_operator(cs, dtype):
    import torch

    td = torch.float32 if dtype == "f32" else torch.float64
    small = [cs.icosphere(0), cs.icosphere(3), fan(cs, 5), fan(cs, 6), fan(cs, 7), fan(cs, 12),
             cs.triangulated_grid(7.3, 5.1, 0.31, 0.29)]
    large = [cs.triangulated_grid(510.0, 512.0, 1.0, 1.0), cs.triangulated_grid(511.0, 511.0, 1.0, 1.0)]
    meshes = [cs.dualize(m, cs.Barycenter) for m in small + large]
    batch = cs.HeatBatch(meshes + meshes[:4], td)
    sizes = np.diff(batch.offsets)
    assert list(sizes[7:9]) == [2 ** 18 - 1, 2 ** 18]
    u = torch.empty(batch.total, dtype=td, device="cuda")
    for i in range(len(sizes)):
        cs.fill_uniform(batch.instance(u, i), 500 + i)
    ref = u.clone()
    batch.steps(u, 3, graph=False)
    g = ref.clone()
    for _ in range(3):                     # one step per replay: odd counts copy back
        batch.steps(g, 1)
    assert torch.equal(g, u)
    for i, m in enumerate(meshes + meshes[:4]):
        x, L = batch.instance(ref, i), cs.fast_laplace_beltrami(m, cs.DiagonalHodge, cast_float=td)
        for _ in range(3):
            x = x - batch.dt[i] * (L @ x)
        assert torch.equal(batch.instance(u, i), x), i
