"""The SPH step (forces, integration and the published statistics in one
launch) at the edges of its tiles and of its statistics slots: one particle,
a tile of 128 less one, full and more by one, and more workgroups than the 32
slots.  The forces against the FP64 oracle; the statistics and the largest
force, published by the last workgroup, against those read back by a copy."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(n, spacing=0.016, seed=0):
    rng = np.random.default_rng(seed + n)
    base = scenes.sph_dam_break()
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    mid = (np.asarray(base.positions).max(0) + np.asarray(base.positions).min(0)) / 2 + 0.25
    p = mid + (g - m / 2) * spacing + rng.uniform(-0.2, 0.2, (n, 3)) * spacing
    v = rng.uniform(-0.2, 0.2, (n, 3))
    return dataclasses.replace(base, positions=p.astype(np.float32).astype(np.float64),
                               velocities=v.astype(np.float32).astype(np.float64))


# A density is good to 2e-6; the Tait pressure's seventh power takes that to
# 1.4e-5 of a compressed particle's pressure, and the largest net force is
# above a tenth of the sum of its terms at the surface of a block.
@pytest.mark.parametrize("n", [1, 2, 127, 128, 129, 33 * 128 + 1])
def test_forces_and_moves_match_oracle(bbx, oracle, n):
    sc = _scene(n)
    g, o = bbx.Solver(sc, kind=bbx.SPH), oracle.Sim(sc)
    dt = 1e-6
    g.sph_substep(dt)
    o.sph_substep(dt, oracle.SPH_TWO_PHASE)
    f = o.get("force")
    tol = 1.4e-4 * np.abs(f).max()
    assert np.abs(g.get("force") - f).max() <= tol
    v = o.get("velocity")
    dv = dt / o.info()["mass"] * tol + 1e-6 * np.abs(v).max()
    assert np.abs(g.get("velocity") - v).max() <= dv
    assert np.abs(g.get("position") - o.get("position")).max() <= dt * dv + 2.0 ** -23 * np.abs(sc.positions).max()


@pytest.mark.parametrize("env", [{}, {"BBX_TILE_CAP": "0"}])
@pytest.mark.parametrize("n", [1, 129, 32 * 128, 33 * 128 + 1, 66000])
def test_published_statistics_equal_the_copied_ones(bbx, monkeypatch, n, env):
    sc = _scene(n, spacing=0.011)  # buckets over the cap
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    res = []
    for signal in ("1", "0"):
        monkeypatch.setenv("BBX_LOOP_SIGNAL", signal)
        s = bbx.Solver(sc, kind=bbx.SPH)
        out = []
        for _ in range(3):
            st = s.sph_substep(2e-5)
            out.append((st.bucket_overflows, st.lost_particles, st.full_redistribution,
                        s.number_of_time_steps(1.0, 1.0)))
            f = s.get("force")
            out.append(np.linalg.norm(f, axis=1).max())
        res.append((out, [s.get(k) for k in ("force", "position", "velocity", "density")]))
        s.close()
    assert res[0][0] == res[1][0]
    for a, b in zip(res[0][1], res[1][1]):
        np.testing.assert_array_equal(a, b)
    # the rule 0.25 sqrt(r m / max |f|) with this step's force, or sound speed
    s = bbx.Solver(sc, kind=bbx.SPH)
    _, fmax = res[0][0][-2:]
    steps = res[0][0][-2][-1]
    inf = s.info()
    limit = min(0.4 * inf["kernel_radius"] / s.params.sound_speed,
                0.25 * np.sqrt(inf["kernel_radius"] * inf["mass"] / fmax))
    assert abs(steps - 1.0 / limit) <= 1 + 1e-6 / limit


@pytest.mark.parametrize("signal,xsph", [("1", 0.0), ("0", 0.0), ("1", 2000.0)])
@pytest.mark.parametrize("n", [1, 300, 66000])
def test_advance_equals_its_substeps(bbx, monkeypatch, signal, xsph, n):
    """sph_advance queues the next substep's grid pass before this one's force
    is known; the state is that of the same substeps one by one."""
    monkeypatch.setenv("BBX_LOOP_SIGNAL", signal)
    sc = _scene(n)
    a, b = (bbx.Solver(sc, kind=bbx.SPH, pseudo_viscosity=xsph) for _ in range(2))
    for interval in (2.5e-4, 1.2e-3):
        steps, left = a.sph_advance(interval), interval
        for _ in range(steps):
            dt = left / b.number_of_time_steps(left, 1.0)
            b.sph_substep(dt)
            left -= dt
        assert left <= float(np.float32(1e-4)) < left + dt  # the rule's constant is an FP32 one
        for k in ("position", "velocity", "force", "density"):
            np.testing.assert_array_equal(a.get(k), b.get(k))
        for x, y in zip(a.chains(), b.chains()):
            np.testing.assert_array_equal(x, y)
