"""The grid pass at the edges of its scan (one workgroup, several in one
launch, two launches: the cell table has cells + 1 entries, 2,048 per
workgroup, up to sixteen in one launch) and of the cell counts that a pass
leaves at zero for the next: chains exact against the oracle over passes,
with particles that leave the grid and with particles added in between."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes
from tests.test_gpu_grid import assert_buckets_equal, assert_chains_equal

pytestmark = pytest.mark.gpu


def _scene(cells, n, seed=0):
    """n particles anywhere in a tank of `cells` cells of edge 0.02."""
    rng = np.random.default_rng(seed + n)
    tank = np.array(cells) * 0.02
    p = (rng.uniform(-0.5, 0.5, (n, 3)) * tank).astype(np.float32).astype(np.float64)
    v = rng.normal(size=(n, 3)).astype(np.float32).astype(np.float64)
    base = scenes.dam_break(2, 2, 2)
    return dataclasses.replace(base, positions=p, velocities=v, tank_size=tuple(float(t) for t in tank))


# 2,001 (one workgroup), 2,049 (two), 31,745 (sixteen), 32,769 (seventeen: two launches) entries
@pytest.mark.parametrize("cells", [(10, 10, 20), (16, 16, 8), (32, 32, 31), (32, 32, 32)])
def test_chains_over_passes(bbx, oracle, cells):
    sc = _scene(cells, 3000)
    g, o = bbx.Solver(sc), oracle.Sim(sc)
    assert g.info()["grid"].total == cells[0] * cells[1] * cells[2]
    rng = np.random.default_rng(7)
    for step in range(3):
        assert_chains_equal(g.chains(), o.chains())
        st = g.distribute()
        o.distribute()
        assert_chains_equal(g.chains(), o.chains())
        assert_buckets_equal(g.buckets(), o.buckets())
        # within half a cell, so that the incremental pass follows
        p = g.get("position") + rng.uniform(-0.009, 0.009, (g.n, 3))
        p = np.clip(p, -np.array(sc.tank_size) / 2 + 1e-3, np.array(sc.tank_size) / 2 - 1e-3)
        p = p.astype(np.float32).astype(np.float64)
        g.set("position", p)
        o.set("position", p)
        assert st.lost_particles == 0


def test_counts_between_passes(bbx):
    """Setup, substeps, added particles and particles outside the grid, one
    after the other on one solver, give the chains of a new solver that is
    given the same particles."""
    sc = _scene((12, 9, 11), 1500)
    g = bbx.Solver(sc)
    g.pcisph_substep(1e-4, 2, 0.01, bbx.MODE_TEXTBOOK)
    g.append(np.array([[0.01, 0.01, 0.01], [5.0, 5.0, 5.0], [0.0, 0.0, 0.0]]))
    g.flag = 1
    st = g.distribute()
    assert st.full_redistribution == 1 and st.lost_particles == 1 and st.bucket_overflows == 0
    h = bbx.Solver(dataclasses.replace(sc, positions=g.get("position"), velocities=g.get("velocity")))
    h.distribute()
    assert_chains_equal(g.chains(), h.chains())
    assert_buckets_equal(g.buckets(), h.buckets())
    assert np.array_equal(g.get("density"), h.get("density"))
