"""A small set grows in less time than a new one takes to make (both allocate
every field; growing copies instead of uploading), many particles appended to
one particle take about as long as a solver of that many, and what is uploaded
and cleared on the way is right."""
import dataclasses
import time

import numpy as np
import pytest

from bubbles_amd import scenes

pytestmark = pytest.mark.gpu


def test_reserve_costs_less_than_a_new_solver(bbx):
    sc = scenes.dam_break(8, 8, 8, spacing=0.01, tank=(0.5, 0.25, 0.5), seed=2)
    new, grow = np.inf, np.inf
    for _ in range(30):
        t = time.perf_counter()
        s = bbx.Solver(sc)
        u = time.perf_counter()
        s.reserve(2 * sc.n + 500)
        grow = min(grow, time.perf_counter() - u)
        new = min(new, u - t)
        s.close()
    print(f"new {1e6 * new:.0f} us, grown {1e6 * grow:.0f} us")
    assert grow <= 0.8 * new


@pytest.mark.parametrize("count", [1, 31, 32, 33, 256, 257, 5000])
def test_appended_state(bbx, count):
    sc = scenes.dam_break(4, 4, 4, spacing=0.01, tank=(0.5, 0.25, 0.5), seed=2)
    rng = np.random.default_rng(count)
    s = bbx.Solver(sc)
    s.pcisph_substep(sc.dt, 3, 1e-9, bbx.MODE_TEXTBOOK)
    before = {k: s.get(k) for k in ("position", "velocity", "force", "density", "pressure")}
    x = rng.uniform(-0.2, 0.2, (count, 3)).astype(np.float32).astype(np.float64) * [1, 0.5, 1]
    v = rng.normal(size=(count, 3)).astype(np.float32).astype(np.float64)
    x = x.astype(np.float32).astype(np.float64)
    s.append(x, v)
    assert np.array_equal(s.get("position"), np.concatenate([before["position"], x]))
    assert np.array_equal(s.get("velocity"), np.concatenate([before["velocity"], v]))
    start, members = s.chains()
    assert np.array_equal(np.sort(members), np.arange(sc.n + count))
    st = s.pcisph_substep(sc.dt, 3, 1e-9, bbx.MODE_TEXTBOOK)
    assert st.lost_particles == 0 and np.isfinite(s.get("velocity")).all()


def test_large_append_to_a_small_set(bbx):
    """The upload's and the growth's share of a new solver, twice over."""
    sc = scenes.dam_break(64, 32, 64, spacing=0.01, tank=(1.0, 0.5, 1.0), seed=2)
    one = dataclasses.replace(sc, positions=sc.positions[:1], velocities=sc.velocities[:1])
    new, grow = np.inf, np.inf
    for _ in range(6):
        t = time.perf_counter()
        s = bbx.Solver(sc)
        new = min(new, time.perf_counter() - t)
        s.close()
        s = bbx.Solver(one)
        t = time.perf_counter()
        s.append(sc.positions[1:])
        grow = min(grow, time.perf_counter() - t)
        s.close()
    print(f"new {1e6 * new:.0f} us, grown {1e6 * grow:.0f} us")
    assert grow <= 3 * new
