"""Mesh SDFs of few triangles, at the edges of the routes: every pair evaluated
(up to 8 triangles, up to 16 on at most 131,072 nodes), one wave a brick (up to
64), four waves; closed and open meshes, whole and partly filled bricks.
Distances are FP64 minima rounded to FP32 on both sides (the device's square
root may differ in the last bit); a sign may differ only at the surface."""
import time

import numpy as np
import pytest

from bubbles_amd import shapes

pytestmark = pytest.mark.gpu


def _turned(v):
    return shapes.transform_points(shapes.rotate_y(25) @ shapes.rotate_x(10), np.asarray(v))


def _part(count):
    """`count` triangles of a ball of 80 (a closed box for 12)."""
    if count == 12:
        v, t = shapes.cube_mesh(0.4)
        return _turned(v), np.asarray(t)
    v, t = shapes.icosphere(0.25, subdivisions=1)
    return _turned(v), np.asarray(t)[:count]


@pytest.mark.parametrize("nodes", [5, 17, 52])
@pytest.mark.parametrize("count", [1, 8, 9, 12, 16, 17, 64, 65, 80])
def test_routes_by_size(bbx, oracle, count, nodes):
    v, t = _part(count)
    dx = 1.2 * np.ptp(v[np.unique(t), 0]) / (nodes - 1)
    g = bbx.Sdf.from_mesh(v, t, dx=dx, margin=0.1).download()
    o = oracle.sdf_from_mesh(v, t, dx=dx, margin=0.1, threads=16)
    assert g.nodes == o.nodes
    want = o.values.astype(np.float32).astype(np.float64)
    np.testing.assert_allclose(np.abs(g.values), np.abs(want), rtol=2.5e-7, atol=0)
    flipped = np.sign(g.values) != np.sign(want)
    assert np.all(np.abs(want[flipped]) <= 2e-5)


def test_box_costs_less_than_a_ball(bbx):
    """A box (12 triangles) on 14k nodes against a ball of 80: a seventh of the
    pairs, and the same allocations and launch otherwise (two fifths of the
    call).  Both at their best of forty."""
    def best(v, t):
        b = np.inf
        for _ in range(40):
            a = time.perf_counter()
            s = bbx.Sdf.from_mesh(v, t, dx=0.05, margin=0.1)
            b = min(b, time.perf_counter() - a)
            s.close()
        return b

    box = shapes.cube_mesh(1.0)
    v, t = shapes.icosphere(0.5, subdivisions=1)
    small, large = best(*box), best(v, t)
    print(f"box {1e6 * small:.0f} us, ball {1e6 * large:.0f} us")
    assert small <= 0.7 * large
