"""Particles inside the grid but in no chain (a jump of more than a cell that
an incremental pass does not follow, a return from outside, members that
set_chains leaves out).  They are stored behind the chained ones in no order
of their cells, look for neighbours from the cell they are in and are nobody's
candidates.  A tile that holds one must not take its range of cells from its
first and last particle.  Chains, buckets, densities and features of all
particles against the FP64 oracle, for the three bucket kernels (four lanes
per particle, own tile tables, a table kernel before it)."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import scenes
from tests.test_gpu_grid import assert_buckets_equal, assert_chains_equal

pytestmark = pytest.mark.gpu


def _scene(n):
    """n jittered points on a lattice around the origin, sorted by nothing."""
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    p = (g - m / 2) * 0.01 + rng.uniform(-0.002, 0.002, (n, 3))
    p = p[rng.permutation(n)].astype(np.float32).astype(np.float64)
    return dataclasses.replace(scenes.dam_break(2, 2, 2, tank=(2.0, 1.0, 2.0)), positions=p,
                               velocities=np.zeros_like(p))


def _fp32(p):
    return p.astype(np.float32).astype(np.float64)


# A density is good to 2e-6 of itself (the tolerance of the other parity
# tests); a feature is a mean of at most 100 FP32 terms of at most 1, each
# rounded a few times and added with one rounding: 100 * 2^-24 * 2 = 1.2e-5.
FEATURE_TOL = 2e-5


@pytest.mark.parametrize("case", ["one_lower", "five_anywhere", "back_from_outside", "left_out"])
@pytest.mark.parametrize("n", [700, 57600, 262400])
def test_particles_in_no_chain(bbx, oracle, n, case):
    sc = _scene(n)
    order = np.argsort(sc.positions.sum(1))  # lowest corner first
    rng = np.random.default_rng(3)
    moved = sc.positions.copy()
    if case == "one_lower":  # from the highest corner to the lowest
        moved[order[-1]] = moved[order[0]] + 0.004
    elif case == "five_anywhere":
        moved[order[-5:]] = moved[order[[0, n // 2, n // 3, 5, n // 4]]] + 0.003
    elif case == "back_from_outside":
        sc.positions[order[-3:]] += 5.0
        moved[order[-3:]] = moved[order[[1, n // 2, n // 5]]] + 0.003
        moved[order[0]] = [7.0, 7.0, 7.0]  # and one that leaves
    moved = _fp32(moved)
    g, o = bbx.Solver(sc), oracle.Sim(sc, threads=8)
    if case == "left_out":
        start, members = g.chains()
        out = np.concatenate([[0, 1], rng.choice(len(members), 5, replace=False)])
        keep = np.ones(len(members), bool)
        keep[out] = False
        cells = np.repeat(np.arange(len(start) - 1), np.diff(start))[keep]
        chains = np.searchsorted(cells, np.arange(len(start))).astype(np.int32), members[keep]
        g.set_chains(*chains)
        o.set_chains(*chains)
    g.set("position", moved)
    o.set("position", moved)
    a, b = g.distribute(), o.distribute()
    assert a.full_redistribution == b.full_redistribution == 0
    assert a.lost_particles == b.lost_particles > 0
    assert a.bucket_overflows == b.bucket_overflows
    assert_chains_equal(g.chains(), o.chains())
    assert_buckets_equal(g.buckets(), o.buckets())
    o.stage("interaction")
    o.stage("density", 0)
    np.testing.assert_allclose(g.get("density"), o.get("density"), rtol=2e-6)
    f = g.harvest(sc.dt, 1, 0.01)[0]
    ref = o.features(sc.dt)
    assert np.array_equal(f[:, 2], ref[:, 2])
    np.testing.assert_allclose(f, ref, rtol=0, atol=FEATURE_TOL)
