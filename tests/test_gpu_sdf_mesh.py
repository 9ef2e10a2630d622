"""Mesh SDFs where the build takes another route: node counts that leave a
brick of 4 x 4 x 4 part empty, fewer and more triangles than a workgroup has
lanes, meshes that are not closed or whose triangles share no vertices,
triangles without area, and nodes that lie on the surface.

Distances are FP64 minima rounded to FP32 on both sides (the device's square
root may differ in the last bit).  A sign may differ only at the surface,
where the winding number is 1/2 up to its rounding.
"""
import numpy as np
import pytest

from bubbles_amd import shapes

pytestmark = pytest.mark.gpu


def _turned(v, a=25, b=10):
    return shapes.transform_points(shapes.rotate_y(a) @ shapes.rotate_x(b), v)


def _mesh(kind):
    if kind == "one triangle":
        return np.array([[0.0, 0.0, 0.0], [0.3, 0.1, 0.0], [0.1, 0.25, 0.2]]), np.array([[0, 1, 2]], dtype=np.int32)
    if kind == "open box":
        v, t = shapes.cube_mesh(0.4)
        return _turned(v), t[:-2]
    if kind == "box on the grid":  # 10 spacings of 0.04 plus margins: faces on node planes
        return shapes.cube_mesh(0.4)
    v, t = shapes.icosphere(0.25, subdivisions=3 if kind == "many" else 2)
    v = _turned(v * np.array([1.0, 0.8, 0.9]), 17, 31)
    if kind == "no shared vertices":
        return v[t].reshape(-1, 3), np.arange(3 * len(t), dtype=np.int32).reshape(-1, 3)
    if kind == "no area":
        return v, np.concatenate([t, [[0, 0, 1], [2, 2, 2]]]).astype(np.int32)
    if kind == "two balls":  # overlapping: winding number 2 in the overlap
        return np.concatenate([v, v + [0.2, 0.05, 0.0]]), np.concatenate([t, t + len(v)]).astype(np.int32)
    return v, t


def _segment(grid, a, b):
    """Distance of every node to the segment a -> b, its parameter in [1e-4, 1]."""
    k, j, i = np.meshgrid(*(np.arange(n) for n in grid.nodes[::-1]), indexing="ij")
    p = np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1) * np.array(grid.spacing) + np.array(grid.origin)
    u = np.clip((p - a) @ (b - a) / ((b - a) @ (b - a)), 1e-4, 1.0)
    return np.linalg.norm(p - a - u[:, None] * (b - a), axis=1)


@pytest.mark.parametrize("dx", [0.04, 0.017])
@pytest.mark.parametrize("kind", ["one triangle", "open box", "box on the grid", "few", "many", "no shared vertices",
                                  "no area", "two balls"])
def test_sdf_from_mesh_routes(bbx, oracle, kind, dx):
    v, t = _mesh(kind)
    g = bbx.Sdf.from_mesh(v, t, dx=dx, margin=0.1).download()
    # the oracle has no distance to a triangle without area: the device passes
    # over a point and takes a segment's two edges
    o = oracle.sdf_from_mesh(v, t[:-2] if kind == "no area" else t, dx=dx, margin=0.1, threads=16)
    assert g.nodes == o.nodes
    want = o.values
    if kind == "no area":
        near = np.minimum(_segment(g, v[0], v[1]), _segment(g, v[1], v[0]))
        want = np.where(near < np.abs(want), np.sign(want) * np.maximum(near, 1e-5), want)
    want = want.astype(np.float32).astype(np.float64)
    np.testing.assert_allclose(np.abs(g.values), np.abs(want), rtol=2.5e-7, atol=0)
    flipped = np.sign(g.values) != np.sign(want)
    assert np.all(np.abs(want[flipped]) <= 2e-5)
