"""Cells of far more particles than a key bin holds.  Chains exact against the
oracle over full, incremental and append passes, also after the set has grown
(the blocks behind the bins are sized by the capacity), with every cell of a
small grid crowded and with one cell that holds nearly all; and ranking them
from the bins takes no longer than through the index, which is the route of a
grid without bins."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes
from tests.test_gpu_grid import assert_chains_equal

pytestmark = pytest.mark.gpu


def _scene(cells, crowds, per, seed=0):
    """`crowds` cells of the grid with `per` particles in each; shuffled."""
    rng = np.random.default_rng(seed + per)
    tank = np.array(cells) * 0.02
    m = min(cells) - 2
    k = np.arange(crowds)
    lo = -tank / 2 + 0.02 * (1 + np.stack([k % m, k // m % m, k // m // m], axis=-1))
    p = (lo[:, None] + rng.uniform(0.002, 0.018, (crowds, per, 3))).reshape(-1, 3)
    p = p[rng.permutation(len(p))].astype(np.float32).astype(np.float64)
    base = scenes.dam_break(2, 2, 2)
    return dataclasses.replace(base, positions=p, velocities=np.zeros_like(p), tank_size=tuple(float(t) for t in tank))


@pytest.mark.parametrize("crowds,per", [(1, 33), (1, 64), (1, 65), (9, 96), (9, 97), (7, 1000), (1, 5000)])
def test_crowded_chains(bbx, oracle, crowds, per):
    sc = _scene((12, 12, 12), crowds, per)
    g, o = bbx.Solver(sc), oracle.Sim(sc)
    rng = np.random.default_rng(1)
    for step in range(5):
        if step == 2:  # grown, and all of one cell's particles once more at its tail
            add = sc.positions[: 2 * per + 100]
            g.reserve(4 * sc.n + 3000)
            g.append(add)
            o.append(add)
        elif step:
            p = g.get("position")
            p += rng.uniform(-0.006, 0.006, p.shape)
            p = p.astype(np.float32).astype(np.float64)
            g.set("position", p)
            o.set("position", p)
            g.flag = o.flag = int(step == 3)
            g.distribute()
            o.distribute()
        assert_chains_equal(g.chains(), o.chains())


def test_passes_go_round(bbx, oracle):
    """More passes than a block's entry can number."""
    sc = _scene((12, 12, 12), 3, 70)
    g, o = bbx.Solver(sc), oracle.Sim(sc)
    for step in range(8300):
        g.distribute()
        if 8180 < step < 8200 or step == 8299:
            assert_chains_equal(g.chains(), o.chains())


def _rank_us(bbx, sc):
    s = bbx.Solver(sc)
    best = np.inf
    for _ in range(6):
        s.flag = 1
        s.profile(True)
        s.profile_reset()
        s.distribute()
        d = s.profile_get()
        best = min(best, 1e3 * sum(d[k]["total_ms"] for k in ("grid_hash", "grid_scatter", "grid_rank_move") if k in d))
    most = np.diff(s.chains()[0]).max()
    s.close()
    return best, "grid_scatter" not in d, most


@pytest.mark.parametrize("crowds,per", [(100, 100), (10, 1000), (1, 10000)])
def test_crowded_cells_cost_no_more_than_through_the_index(bbx, crowds, per):
    """Hash, scatter and rank of 10,000 particles with bins and without; what
    the two routes read of a cell is the same, so twice as long and 20 us (a
    few launches' latency) is the bound."""
    small = _scene((30, 30, 30), crowds, per)
    large = dataclasses.replace(small, tank_size=(1.0, 1.0, 1.0))  # 125,000 cells and more: no bins
    with_bins, a, m = _rank_us(bbx, small)
    without, b, m2 = _rank_us(bbx, large)
    assert m == m2 == per
    print(f"{crowds} cells of {per}: {with_bins:.1f} us with bins, {without:.1f} us without")
    assert a and not b
    assert with_bins <= 2 * without + 20
