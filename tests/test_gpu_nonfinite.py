"""Values that have left the range of FP32 stay with the particles they belong
to: a predicted position so far away that its distances overflow is no
neighbour of anyone's (the container clamps predicted positions, a collider
list without one does not), and an infinite pressure takes no part in the
pairs that the gradient leaves out (the particle itself, coincident ones) nor
in a bucket's unused entries."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes, shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env", [{}, {"BBX_TILE_CAP": "0"}])
@pytest.mark.parametrize("speed", [1e27, 1e38])
def test_predicted_position_out_of_range(bbx, oracle, monkeypatch, speed, env):
    """One particle of a block leaves at a speed that takes its x* beyond the
    square root of FP32's range.  Without viscosity its neighbours' motion is
    that of the block, and their predicted densities lack it alone: x* is
    rounded to 2^-24 of at most 0.5, 1e-5 of a neighbour's distance and 1e-4 of
    its kernel value at most."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    base = scenes.dam_break(8, 8, 8, spacing=0.01, tank=(0.5, 0.25, 0.5), seed=2)
    v = np.zeros_like(base.positions)
    fast = 300
    v[fast] = [speed, 0.0, 0.0]
    sc = dataclasses.replace(base, positions=base.positions.astype(np.float32).astype(np.float64), velocities=v)
    wall = [shapes.sphere(shapes.translate(0.2, 0.1, 0.2), 0.01)]  # no container
    over = dict(viscosity=0.0, drag_coefficient=0.0)
    g, o = bbx.Solver(sc, **over), oracle.Sim(sc, **over)
    g.set_colliders(wall)
    o.set_colliders(wall)
    g.pcisph_substep(sc.dt, 1, 0.01, bbx.MODE_TEXTBOOK)
    o.pcisph_substep(sc.dt, 1, 0.01, oracle.MODE_TEXTBOOK)
    near = np.linalg.norm(sc.positions - sc.positions[fast], axis=1) < 2 * base.kernel_radius
    assert near.sum() > 30
    np.testing.assert_allclose(g.get("density_predicted"), o.get("density_predicted"), rtol=1e-4)
    others = np.arange(sc.n) != fast
    assert np.isfinite(g.get("velocity")[others]).all()
    np.testing.assert_allclose(g.get("position")[others], o.get("position")[others], atol=5e-7)


@pytest.mark.parametrize("kind", ["pcisph", "sph"])
@pytest.mark.parametrize("env", [{}, {"BBX_TILE_CAP": "0"}, {"BBX_TILE_CAP2": "0"}])
def test_infinite_pressure_of_lone_particles(bbx, oracle, monkeypatch, kind, env):
    """Particles further apart than the radius, and two at one place, with a
    negative-pressure scale that takes their pressures out of FP32: no pair of
    theirs counts, so they fall freely."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    g = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * 0.05 - 0.1
    p = np.concatenate([g, g[62:63]]).astype(np.float32).astype(np.float64)
    sc = dataclasses.replace(scenes.dam_break(2, 2, 2, tank=(0.5, 0.5, 0.5)), positions=p, velocities=np.zeros_like(p))
    over = dict(negative_pressure_scale=1e38)
    s = bbx.Solver(sc, kind=bbx.PCISPH if kind == "pcisph" else bbx.SPH, **over)
    o = oracle.Sim(sc, **over)
    if kind == "pcisph":
        s.pcisph_substep(sc.dt, 2, 1e-9, bbx.MODE_TEXTBOOK)
        o.pcisph_substep(sc.dt, 2, 1e-9, oracle.MODE_TEXTBOOK)
    else:
        s.sph_substep(sc.dt)
        o.sph_substep(sc.dt, oracle.SPH_TWO_PHASE)
    assert np.isneginf(s.get("pressure")).all()
    fall = o.get("velocity")
    assert np.all(fall[:, 1] < 0) and np.abs(fall[:, [0, 2]]).max() == 0
    np.testing.assert_allclose(s.get("velocity"), fall, rtol=1e-6)
    np.testing.assert_allclose(s.get("position"), o.get("position"), rtol=0, atol=2.0 ** -24)
