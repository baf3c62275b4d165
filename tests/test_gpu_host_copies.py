"""Arrays between host and device around the sizes at which a copy to the host goes through
pinned chunks (3 MiB) and fills one, all and more than all of them (four of 4 MiB): every
value arrives, whatever memory the caller's array lies in."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from fluid_simulation_amd import fsg

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("n", [1, 3 * MIB // 16 - 1, 3 * MIB // 16, 4 * MIB // 16,
                               4 * MIB // 16 + 1, 16 * MIB // 16 - 1, 16 * MIB // 16 + 1,
                               37 * MIB // 16 + 7])
def test_particles_round_trip(n):
    rng = np.random.default_rng(n)
    d = fsg.Domain(16, 16, 16.0, 16.0, 0.01, 0.05)
    a = rng.standard_normal((n, 4)).astype(np.float32)
    d.set_particles(a)
    assert np.array_equal(d.particles().view(np.uint32), a.view(np.uint32))
    # again, into an array at an odd place and one in pinned memory
    b = a[::-1].copy()
    d.set_particles(b)
    raw = np.zeros(16 * n + 4, np.uint8)
    d._chk(d._L.fsg_get_particles(d._h, raw.ctypes.data + 4, n), "fsg_get_particles")
    assert np.array_equal(raw[4:].view(np.uint32).reshape(n, 4), b.view(np.uint32))
    pin = torch.zeros((n, 4), pin_memory=True)
    d._chk(d._L.fsg_get_particles(d._h, C.c_void_p(pin.data_ptr()), n), "fsg_get_particles")
    assert np.array_equal(pin.numpy().view(np.uint32), b.view(np.uint32))
    d.close()


def test_velocity_round_trip():
    nx, ny = 1500, 1100  # 6.3 MiB each: the ring wraps within and between the two
    rng = np.random.default_rng(3)
    d = fsg.Domain(nx, ny, float(nx), float(ny), 0.01, 0.05)
    u, v = (rng.standard_normal((ny, nx)).astype(np.float32) for _ in range(2))
    d.set_velocity(u, v)
    gu, gv = d.velocity()
    assert np.array_equal(gu, u) and np.array_equal(gv, v)
    d.set_velocity(v, None)  # one component alone
    gu, gv = d.velocity()
    assert np.array_equal(gu, v) and np.array_equal(gv, v)
    d.close()
