"""The bucket build's two kernels: four lanes per particle for small sets (up
to 57,344 particles) and one lane per particle above.

Buckets are exact against the FP64 oracle.  A density is an FP32 sum of at
most 100 non-negative terms with compensation; each term has a few roundings
of 2^-24, so 2e-6 relative bounds it (the tolerance of the other parity
tests).  Both kernels add the same terms in the same order."""
import dataclasses

import numpy as np
import pytest

from bubbles_amd import learned, scenes
from tests.test_gpu_grid import assert_buckets_equal

pytestmark = pytest.mark.gpu


def _points(n, spacing, seed=0):
    """n jittered lattice points around the origin (FP32 values), shuffled."""
    rng = np.random.default_rng(seed + n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    p = (g - m / 2) * spacing + rng.uniform(-0.2, 0.2, (n, 3)) * spacing
    return p[rng.permutation(n)].astype(np.float32).astype(np.float64)


def _scene(p):
    return dataclasses.replace(scenes.dam_break(2, 2, 2, tank=(2.0, 1.0, 2.0)), positions=p,
                               velocities=np.zeros_like(p))


# spacings: ordinary (~30 neighbours), more than the 64 a lane group keeps in
# LDS (~70), over the cap of 100 (~110), cells of more than 32 particles
@pytest.mark.parametrize("spacing", [0.01, 0.0078, 0.0067, 0.005])
@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 2000])
def test_split_buckets_match_oracle(bbx, oracle, n, spacing):
    sc = _scene(_points(n, spacing))
    g, o = bbx.Solver(sc), oracle.Sim(sc)
    st = g.distribute()
    o.distribute()
    b = o.buckets()
    assert_buckets_equal(g.buckets(), b)
    o.stage("interaction")
    o.stage("density", 1)
    np.testing.assert_allclose(g.get("density"), o.get("density"), rtol=2e-6)
    # the reference's cap: what a bucket of 100 leaves out
    d2 = ((sc.positions[:, None] - sc.positions[None]) ** 2).sum(-1)
    within = (np.sqrt(d2) ** 2 - sc.kernel_radius ** 2 <= -1e-8).sum(1)
    assert st.bucket_overflows == np.maximum(within - 100, 0).sum()


@pytest.mark.parametrize("n", [57344, 262144])
def test_both_kernels_agree_at_the_boundary(bbx, n):
    """57,344 particles take the split kernel, 262,144 the one that makes its
    tiles' tables; the same with one more, far away, the next kernel: the same
    buckets, features and network pressures."""
    p = _points(n, 0.01)
    extra = np.array([[0.9, 0.4, 0.9]], dtype=np.float32).astype(np.float64)
    assert np.abs(p).max() < 0.5
    res = []
    for q in (p, np.concatenate([p, extra])):
        s = bbx.Solver(_scene(q))
        s.attach_mlp(learned.load())
        s.keep_features(True)
        s.distribute()
        counts, ids = s.buckets()
        s.pcisph_substep(5e-4, 1, 0.01, bbx.MODE_TEXTBOOK, bbx.WARM_MLP)
        res.append([x[:n] for x in (counts, ids, s.get("density"), s.get("features"), s.get("warm_pressure"))])
        s.close()
    a, b = res
    assert_buckets_equal((a[0], a[1]), (b[0], b[1]))
    for x, y in zip(a[2:], b[2:]):  # the same sums in the same order
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("env", [{"BBX_TILE_CAP": "0"}, {"BBX_TILE_CAP": "1500", "BBX_TILE_CAP2": "900"},
                                 {"BBX_BUCKET_ROW_MAX": "0"}, {"BBX_BUCKET_ROW_MAX": "20"}])
def test_large_set_routes_bit_identical(bbx, monkeypatch, env):
    """Staged and unstaged tiles, row masks and cell walks above the boundary."""
    sc = _scene(_points(66000, 0.01))
    res = []
    for k in range(2):
        if k:
            for name, v in env.items():
                monkeypatch.setenv(name, v)
        s = bbx.Solver(sc)
        s.pcisph_substep(5e-4, 2, 1e-9, bbx.MODE_TEXTBOOK)
        res.append([s.get("position"), s.get("velocity"), s.get("density")])
        s.close()
    for a, b in zip(*res):
        np.testing.assert_array_equal(a, b)
