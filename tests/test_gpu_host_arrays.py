"""Large host arrays of one call that share memory: the later one's values end there, as when
they are copied one after the other."""
from __future__ import annotations

import numpy as np
import pytest

from fluid_simulation_amd import fsg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1 << 18])
def test_velocity_into_shared_memory(shift):
    nx, ny = 1400, 1300
    rng = np.random.default_rng(3)
    u = rng.standard_normal((ny, nx)).astype(np.float32)
    v = rng.standard_normal((ny, nx)).astype(np.float32)
    d = fsg.Domain(nx, ny, nx, ny, 0.01, 0.05)
    d.set_velocity(u, v)
    want = np.zeros(nx * ny + shift, np.float32)
    want[:nx * ny] = u.ravel()
    want[shift:] = v.ravel()
    for _ in range(20):
        got = np.zeros(nx * ny + shift, np.float32)
        d._chk(d._L.fsg_get_velocity(d._h, fsg.VEL_FRONT, got.ctypes.data,
                                     got.ctypes.data + 4 * shift), "fsg_get_velocity")
        assert np.array_equal(got, want)
    d.close()
