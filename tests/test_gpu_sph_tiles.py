"""The SPH step at the edges of its tiles of 256 particles (two lanes each) and
of its 32 statistics slots: a full tile less one, full and more by one; 31, 32
and 33 workgroups, with a full and a nearly empty last one.  Forces and moves
against the FP64 oracle; the statistics and the largest force that the last
workgroup to arrive publishes against those read back by a copy."""
import numpy as np
import pytest

from tests.test_gpu_sph_step import _scene

pytestmark = pytest.mark.gpu

TILE, SLOTS = 256, 32


# tolerances as in test_gpu_sph_step.py
@pytest.mark.parametrize("n", [TILE - 1, TILE, TILE + 1, SLOTS * TILE + 1, (SLOTS + 1) * TILE + 1])
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


@pytest.mark.parametrize("n", [TILE, TILE + 1, (SLOTS - 1) * TILE + 1, SLOTS * TILE, SLOTS * TILE + 1,
                               (SLOTS + 1) * TILE, (SLOTS + 1) * TILE + 1, 2 * SLOTS * TILE + 1])
def test_published_statistics_equal_the_copied_ones(bbx, monkeypatch, n):
    sc = _scene(n, spacing=0.011)  # buckets over the cap
    res = []
    for signal in ("1", "0"):
        monkeypatch.setenv("BBX_LOOP_SIGNAL", signal)
        s = bbx.Solver(sc, kind=bbx.SPH)
        out = []
        for _ in range(4):
            st = s.sph_substep(2e-5)
            out.append((st.bucket_overflows, st.lost_particles, st.full_redistribution,
                        s.number_of_time_steps(1.0, 1.0)))
            # the rule 0.25 sqrt(r m / max |f|) with this step's force, or sound speed
            inf = s.info()
            fmax = np.linalg.norm(s.get("force"), axis=1).max()
            limit = min(0.4 * inf["kernel_radius"] / s.params.sound_speed,
                        0.25 * np.sqrt(inf["kernel_radius"] * inf["mass"] / fmax))
            assert abs(out[-1][-1] - 1.0 / limit) <= 1 + 1e-6 / limit
        res.append(out)
        s.close()
    assert res[0] == res[1] and res[0][0][0] > 0
