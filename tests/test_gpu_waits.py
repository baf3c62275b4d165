"""Waits between the workgroups of a pressure solve: one that runs out (here after a few
polls, set from the host; every kernel still ends by itself) sends the plain form to its many
launches and fails the others, whose next solve is whole again; and solves of several blocks
from several threads at once."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from fluid_simulation_amd import fsg, scenes

from test_gpu_pcg import _cg, _system

pytestmark = pytest.mark.gpu


def _spin_max(d, polls):
    f = d._L.fsg_test_spin_max
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_int32], ctypes.c_int
    assert f(d._h, polls) == 0


def _solve(d, lab, u, v):
    d.set_labels(lab)
    d.set_velocity(u, v)
    d.run_phase("PRESSURE", 0.01)
    st = d.stats()
    return d.pressure(), (st.n_fluid, st.cg_iterations)


@pytest.mark.parametrize("nx,ny,n", [(200, 191, 33000), (700, 600, 400000)])
def test_plain_form_solves_again(nx, ny, n):
    """The many launches' iterate is the FP64 one to 1e-4, as test_gpu_pcg's, with the
    counters of that solve; the launch after it is the one-launch form's own, bit for bit."""
    lab, u, v = _system(nx, ny, n, 7)
    d = fsg.Domain(nx, ny, nx, ny, 0.01, 0.05)
    d.set_params(solver=fsg.SOLVER_PLAIN, cg_tol=1e-6, cg_max_iter=30)
    d.set_timing(True)
    p0, s0 = _solve(d, lab, u, v)
    assert "cg_iteration" not in d.timing()
    assert s0 == (n, 30)
    _spin_max(d, 1)
    p1, s1 = _solve(d, lab, u, v)
    assert "cg_iteration" in d.timing()
    assert s1 == s0
    want = _cg(lab, d.rhs(), 30, 1e-6)
    assert np.abs(p1 - want).max() <= 1e-4 * np.abs(want).max()
    assert np.array_equal(d.fluid_indices()[lab == fsg.LIQUID], np.arange(n))
    d.synchronize()   # no solve is left that gave up
    _spin_max(d, 0)
    p2, s2 = _solve(d, lab, u, v)
    assert s2 == s0 and np.array_equal(p0.view(np.uint32), p2.view(np.uint32))
    st = d.stats()
    assert (st.total_unknown_iterations, st.total_solves) == (3 * 30 * n, 3)
    d.close()


@pytest.mark.parametrize("solver", [fsg.SOLVER_PERSISTENT, fsg.SOLVER_REFINED],
                         ids=["persistent", "refined"])
def test_persistent_forms_report_it(solver):
    lab, u, v = _system(200, 191, 33000, 8)
    d = fsg.Domain(200, 191, 200, 191, 0.01, 0.05)
    d.set_params(solver=solver, cg_tol=1e-6, cg_max_iter=200)
    p0, s0 = _solve(d, lab, u, v)
    _spin_max(d, 1)
    for ask in (d.synchronize, d.stats, d.stats):
        d.set_velocity(u, v)
        d.run_phase("PRESSURE", 0.01)
        with pytest.raises(fsg.FsgError, match="abandoned"):
            ask()
        with pytest.raises(fsg.FsgError, match="abandoned"):
            ask()
    _spin_max(d, 0)
    p1, s1 = _solve(d, lab, u, v)
    assert s1 == s0 and np.array_equal(p0.view(np.uint32), p1.view(np.uint32))
    d.close()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("n", [130, 400])
def test_multigrid_form_reports_it(n, graph):
    sc = scenes.dam_break(n)
    d = fsg.Domain.from_scene(sc, cg_tol=1e-6, cg_max_iter=200, solver=fsg.SOLVER_MG,
                              deterministic=1, graph=graph)
    d.step(fsg.PICFLIP, sc.dt)
    d.checkpoint_save(0)
    d.step(fsg.PICFLIP, sc.dt)
    want = (d.particles(), *d.velocity())
    d.checkpoint_load(0)
    _spin_max(d, 1)
    with pytest.raises(fsg.FsgError, match="ran out"):
        d.step(fsg.PICFLIP, sc.dt)
    _spin_max(d, 0)
    d.checkpoint_load(0)
    d.step(fsg.PICFLIP, sc.dt)
    for a, b in zip(want, (d.particles(), *d.velocity())):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    d.close()


@pytest.mark.parametrize("solver", [fsg.SOLVER_PLAIN, fsg.SOLVER_REFINED],
                         ids=["plain", "refined"])
def test_several_threads(solver):
    """Domains of 2 to 16 blocks of unknowns, stepped by a thread each, end as they do one
    after the other."""
    def run(n, out):
        sc = scenes.dam_break(n)
        d = fsg.Domain.from_scene(sc, cg_tol=1e-6, cg_max_iter=300, solver=solver,
                                  deterministic=1)
        for _ in range(6):
            d.step(fsg.PICFLIP, sc.dt)
        out[n] = (d.pressure().copy(), d.stats().cg_iterations)
        d.close()

    sizes = [200, 257, 384, 512]
    alone, together = {}, {}
    for n in sizes:
        run(n, alone)
    threads = [threading.Thread(target=run, args=(n, together)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n in sizes:
        assert together[n][1] == alone[n][1] > 0
        assert np.array_equal(together[n][0].view(np.uint32), alone[n][0].view(np.uint32))
