"""A set grows wherever its fields have room: the key bins of the grid pass, an
option that many cells make large, give way.  Where the fields have none, the
set goes on as it was, whichever of them the memory ended at.  Runs in a process of its own,
where tests/cpp/hip_faults.c stands before the HIP runtime and refuses device
memory beyond a budget."""
import pytest

from tests.test_gpu_fetch_faults import _run, faults  # noqa: F401  (a fixture)

pytestmark = pytest.mark.gpu

BUDGET = """
import dataclasses
size = lambda name: word(name, C.c_size_t)
sc = dataclasses.replace(scene(13, 5, 3), tank_size=(0.8, 0.8, 0.7))  # 56,000 cells
more = scene(36, 36, 36).positions
cells = 56000
bins = 8 * cells * 32
res, names = [], []
for run in range(2):
    # first the fields alone, whose peak is the second run's budget
    size("faults_refuse").value = bins if run == 0 else 0
    s = abi.Solver(sc)
    assert s.info()["grid"].total == cells and s.capacity() == 256
    live = size("faults_live").value
    size("faults_peak").value = live
    if run == 0:
        base = live
    else:
        assert live - base >= bins  # this one has bins
        size("faults_budget").value = peak
    s.reserve(60000)
    assert s.capacity() == 60032
    if run == 0:
        peak = size("faults_peak").value
    s.append(more)
    s.profile(True)
    s.distribute()
    names.append("grid_scatter" in s.profile_get())
    res.append([s.get("position"), s.get("density"), *s.chains()])
    size("faults_budget").value = 0
    s.close()
for a, b in zip(*res):
    assert np.array_equal(a, b)
assert names[0], names  # the first went through the index
print("done")
"""


def test_growth_within_the_fields_own_memory(faults):  # noqa: F811
    _run(faults, BUDGET)


FAILED = """
size = lambda name: word(name, C.c_size_t)
sc = scene(16, 8, 16)
a, b = abi.Solver(sc), abi.Solver(sc)
for s in (a, b):
    s.pcisph_substep(sc.dt, 3, 1e-9, abi.MODE_TEXTBOOK)
fields = ("position", "velocity", "force", "density", "pressure")
full = 950 * 60000
for part in range(1, 20):  # the memory ends after more and more of the fields
    size("faults_budget").value = size("faults_live").value + full * part // 20
    try:
        a.reserve(60000)
    except abi.BbxError:
        pass
    else:
        break
    finally:
        size("faults_budget").value = 0
    assert a.capacity() == b.capacity()
    for f in fields:
        assert np.array_equal(a.get(f), b.get(f)), (part, f)
    a.stage_density()  # buckets are as they were or empty
    for s in (a, b):
        s.pcisph_substep(sc.dt, 3, 1e-9, abi.MODE_TEXTBOOK)
    for f in fields:
        assert np.array_equal(a.get(f), b.get(f)), (part, f)
assert part > 5
print("done")
"""


def test_failed_growth_leaves_a_sound_solver(faults):  # noqa: F811
    _run(faults, FAILED)
