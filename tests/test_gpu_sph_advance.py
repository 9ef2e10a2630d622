"""An SPH Advance that ends in an error (forces beyond FP32, for which the
time-step rule has no step) leaves what the substeps before it left: the grid
pass that is queued ahead for the next substep is taken back."""
import dataclasses

import numpy as np
import pytest

from tests.test_gpu_sph_step import _scene

pytestmark = pytest.mark.gpu

FIELDS = ("position", "velocity", "force", "density", "pressure")


def _same(a, b):
    assert a.flag == b.flag
    for k in FIELDS:
        np.testing.assert_array_equal(a.get(k), b.get(k))
    for x, y in zip(a.chains() + a.buckets(), b.chains() + b.buckets()):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("signal", ["1", "0"])
@pytest.mark.parametrize("n", [300, 66000])
def test_error_leaves_the_last_substep(bbx, monkeypatch, n, signal):
    monkeypatch.setenv("BBX_LOOP_SIGNAL", signal)
    sc = _scene(n)
    v = sc.velocities.copy()
    v[n // 2] = [1e25, 0.0, 0.0]  # its drag force squared is infinite
    sc = dataclasses.replace(sc, velocities=v)
    a, b = bbx.Solver(sc, kind=bbx.SPH), bbx.Solver(sc, kind=bbx.SPH)
    interval = 1e-3
    dt = interval / b.number_of_time_steps(interval, 1.0)
    with pytest.raises(bbx.BbxError, match="time-step rule"):
        a.sph_advance(interval)
    b.sph_substep(dt)
    assert b.flag == 1  # it jumped
    _same(a, b)
    for s in (a, b):  # and both go on alike
        s.set("velocity", sc.velocities * (np.abs(sc.velocities) < 1e3))
        st = s.sph_substep(1e-6)
        assert st.full_redistribution == 1
    _same(a, b)
