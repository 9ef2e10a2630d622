"""Downloads where something failed: a corrupt id table gives an error before
anything is written, whatever the field's route, and a set that has grown
without a larger pinned ring comes through the smaller one.  Each case runs in
a process of its own, where tests/cpp/hip_faults.c stands before the HIP
runtime."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

pytestmark = pytest.mark.gpu

PRELUDE = """
import ctypes as C, sys
import numpy as np
faults = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from bubbles_amd import abi, scenes
L = abi.load()
runtime = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
faults.faults_init(runtime.encode())
word = lambda name, t=C.c_int: t.in_dll(faults, name)
def scene(nx, ny, nz):
    return scenes.dam_break(nx, ny, nz, spacing=0.01, tank=(0.02 * nx + 0.1, 0.02 * ny + 0.1, 0.02 * nz + 0.1), seed=4)
"""

# 3,000 vectors come straight into the ring, 360,000 in chunks on one thread,
# 505,000 with helpers; the 16-wide features in several passes
CORRUPT = """
dims = tuple(int(a) for a in sys.argv[2:5])
sc = scene(*dims)
if sc.n > 32768:  # the ring's eighth: 32,768 rows a chunk
    word("faults_copy_bytes", C.c_size_t).value = 16 * 32768
else:
    ring = min(4 << 20, (-(-sc.n // 64) * 64 * 64 + 4095) // 4096 * 4096)
    word("faults_copy_bytes", C.c_size_t).value = ring // 8 // 16 * 16
word("faults_copy_offset", C.c_size_t).value = 16 * 7 + 12
word("faults_copy_word").value = sc.n
s = abi.Solver(sc)
assert word("faults_copy_bytes", C.c_size_t).value == 0
for field in ("position", "velocity", "density", "features"):
    out = np.full((sc.n, {"position": 3, "velocity": 3, "density": 1, "features": 16}[field]), 7.25)
    rc = L.bbx_solver_download(s.h, abi.FIELD[field], out.ctypes.data_as(C.POINTER(C.c_double)))
    assert rc != 0 and b"corrupt particle id" in L.bbx_last_error(), (field, rc)
    assert (out == 7.25).all(), field
print("done")
"""

GROWN = """
sc = scene(13, 5, 3)
more = scene(36, 36, 36).positions
parts = [sc.positions, more, more]
fields = []
for fail in (1, 0):
    s = abi.Solver(sc)
    word("faults_host_malloc").value = fail
    s.reserve(60000)
    assert s.capacity() >= 60000
    s.append(more)
    both = np.concatenate(parts[:2]).astype(np.float32).astype(np.float64)
    assert np.array_equal(s.get("position"), both)
    assert word("faults_host_malloc").value == 0
    word("faults_host_malloc").value = fail
    s.append(more)  # grows by itself
    both = np.concatenate(parts).astype(np.float32).astype(np.float64)
    assert np.array_equal(s.get("position"), both)
    s.distribute()
    fields.append([s.get(f) for f in ("position", "density", "features")])
    word("faults_host_malloc").value = 0
for a, b in zip(*fields):
    assert np.array_equal(a, b)
print("done")
"""


@pytest.fixture(scope="module")
def faults(bbx, tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("faults") / "hip_faults.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", lib, os.path.join(ROOT, "tests", "cpp", "hip_faults.c"), "-ldl"],
                   check=True)
    return lib


def _run(faults, code, *args):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, faults, *map(str, args)], cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr


@pytest.mark.parametrize("dims", [(20, 15, 10), (100, 60, 60), (100, 50, 101)])
def test_corrupt_ids_write_nothing(faults, dims):
    _run(faults, CORRUPT, *dims)


def test_growth_without_a_larger_ring(faults):
    _run(faults, GROWN)
