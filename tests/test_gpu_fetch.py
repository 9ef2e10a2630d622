"""Field downloads in id order at the sizes where their route changes: a field
in the pinned ring, one that passes through it in chunks, the helper threads,
and the 16-wide features that take several passes through the scratch buffer;
after a substep has moved particles between slots, and after the set has
grown."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import learned, scenes

pytestmark = pytest.mark.gpu


def _scene(nx, ny, nz):
    rng = np.random.default_rng(nx * ny * nz)
    sc = scenes.dam_break(nx, ny, nz, spacing=0.01, tank=(0.02 * nx + 0.1, 0.02 * ny + 0.1, 0.02 * nz + 0.1), seed=4)
    p = sc.positions[rng.permutation(sc.n)].astype(np.float32).astype(np.float64)  # ids in no storage order
    v = rng.normal(size=p.shape).astype(np.float32).astype(np.float64)
    return dataclasses.replace(sc, positions=p, velocities=v)


# 1, 195 and 43,691 particles in the ring, 360,000 in chunks, 505,000 with helpers
@pytest.mark.parametrize("dims", [(1, 1, 1), (13, 5, 3), (43691, 1, 1), (100, 60, 60), (100, 50, 101)])
def test_fields_come_in_id_order(bbx, dims):
    sc = _scene(*dims) if dims[0] < 1000 else dataclasses.replace(
        _scene(37, 37, 32), positions=_scene(37, 37, 32).positions[:43691], velocities=_scene(37, 37, 32).velocities[:43691])
    s = bbx.Solver(sc)
    assert np.array_equal(s.get("position"), sc.positions)
    assert np.array_equal(s.get("velocity"), sc.velocities)
    s.distribute()
    density = s.get("density")
    x = s.get("position")
    assert np.array_equal(x, sc.positions) and np.all(density > 0)
    # the same particles in another id order give the same values by particle
    other = np.argsort(sc.positions[:, 0] * 7 + sc.positions[:, 1] * 3 + sc.positions[:, 2], kind="stable")
    s2 = bbx.Solver(dataclasses.replace(sc, positions=sc.positions[other], velocities=sc.velocities[other]))
    s2.distribute()
    np.testing.assert_allclose(s2.get("density"), density[other], rtol=1e-5)  # another order of the sum


def test_features_and_growth(bbx):
    sc = _scene(30, 20, 25)
    s = bbx.Solver(sc)
    s.attach_mlp(learned.load())
    s.keep_features(True)
    s.pcisph_substep(sc.dt, 5, 0.01, bbx.MODE_TEXTBOOK, bbx.WARM_MLP)
    f = s.get("features")
    assert np.array_equal(f[:, 2], s.bucket_counts())
    np.testing.assert_allclose(f[:, 0], s.get("density") / 1000.0 - 1.0, atol=2e-7)
    h = bbx.Solver(sc)
    features, targets, _ = h.harvest(sc.dt, 5, 0.01)
    assert np.array_equal(features.astype(np.float64)[:, 2], f[:, 2])
    p = h.get("pressure") / (h.delta(sc.dt) * 1000.0)
    assert np.array_equal(targets, p.astype(np.float32))
    s.append(np.array([[0.0, 0.2, 0.0], [0.01, 0.2, 0.0]]))
    s.reserve(200000)
    x = s.get("position")
    assert x.shape == (sc.n + 2, 3) and np.allclose(x[-2:, 1], 0.2)
