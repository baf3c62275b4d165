"""fsg_checkpoint_save / load: another call's error, which the runtime still reports to
hipGetLastError, is not theirs; the saved state comes back whole."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from fluid_simulation_amd import fsg, scenes

pytestmark = pytest.mark.gpu


def test_checkpoint_after_an_error_of_another_call():
    sc = scenes.dam_break(64)
    d = fsg.Domain.from_scene(sc, cg_tol=1e-6, cg_max_iter=200, solver=fsg.SOLVER_MG)
    d.step(fsg.PICFLIP, sc.dt)
    d.synchronize()
    want = (d.particles(), *d.velocity(fsg.VEL_FRONT), *d.velocity(fsg.VEL_BACK))
    hip = ctypes.CDLL("libamdhip64.so.7", mode=ctypes.RTLD_GLOBAL)
    assert hip.hipGetLastError() == 0
    try:
        assert hip.hipSetDevice(4096) != 0   # no such device: refused on the host
        d.checkpoint_save(0)
        assert hip.hipSetDevice(4096) != 0
        d.checkpoint_load(0)
    finally:
        hip.hipGetLastError()
    d.step(fsg.PICFLIP, sc.dt)
    d.checkpoint_load(0)
    got = (d.particles(), *d.velocity(fsg.VEL_FRONT), *d.velocity(fsg.VEL_BACK))
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    d.close()
