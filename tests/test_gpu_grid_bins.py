"""Ranks counted from the cells' key bins at their edges: cells of exactly as
many particles as a bin holds (32), one more, and several times that; enough
particles in no chain for several LDS chunks; and a grid of more cells than
65,536 and than particles, which has no bins.  Chains, which are integers,
exact against the oracle over full, incremental and append passes."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes
from tests.test_gpu_grid import assert_chains_equal

pytestmark = pytest.mark.gpu


def _scene(cells, counts, lost, seed=0):
    """counts[k] particles inside cell k of the grid's diagonal, 500 anywhere,
    `lost` outside; shuffled."""
    rng = np.random.default_rng(seed + lost)
    tank = np.array(cells) * 0.02
    parts = [rng.uniform(-0.48, 0.48, (500, 3)) * tank, 10 + rng.uniform(0, 1, (lost, 3))]
    for k, m in enumerate(counts):
        lo = -tank / 2 + 0.02 * (k + 1)
        parts.append(lo + rng.uniform(0.002, 0.018, (m, 3)))
    p = np.concatenate(parts)
    p = p[rng.permutation(len(p))].astype(np.float32).astype(np.float64)
    base = scenes.dam_break(2, 2, 2)
    return dataclasses.replace(base, positions=p, velocities=np.zeros_like(p), tank_size=tuple(float(t) for t in tank))


@pytest.mark.parametrize("cells", [(12, 9, 11), (41, 41, 41)])
@pytest.mark.parametrize("lost", [0, 3, 256, 900])
def test_chains_over_passes(bbx, oracle, cells, lost):
    sc = _scene(cells, (31, 32, 33, 64, 150), lost)
    g, o = bbx.Solver(sc), oracle.Sim(sc)
    rng = np.random.default_rng(11)
    for step in range(4):
        st = g.distribute()
        o.distribute()
        assert_chains_equal(g.chains(), o.chains())
        assert st.lost_particles == (np.abs(g.get("position")).max(1) > 5).sum()
        if step == 1:  # forty more beside the first particle, two without a chain
            add = np.concatenate([np.tile(sc.positions[:1], (40, 1)), [[7.0, 7.0, 7.0], [-9.0, 0.0, 0.0]]])
            g.append(add)
            o.append(add)
            assert_chains_equal(g.chains(), o.chains())
            continue
        p = g.get("position")
        inside = np.abs(p).max(1) < 5
        p[inside] += rng.uniform(-0.009, 0.009, (inside.sum(), 3))
        half = np.array(sc.tank_size) / 2 - 1e-3
        p[inside] = np.clip(p[inside], -half, half)
        p = p.astype(np.float32).astype(np.float64)
        g.set("position", p)
        o.set("position", p)
