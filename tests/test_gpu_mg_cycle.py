"""The multigrid levels that share one launch: around the tile count from which a level has
launches of its own, hierarchies whose one-workgroup levels do and do not fit its registers,
coarsest levels of every width, and several solves under way at once on streams of their
own."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from fluid_simulation_amd import fsg, scenes

from helpers import rel_err
from test_gpu_mg import LIQ, _solve_pair, irregular_labels

pytestmark = pytest.mark.gpu


# level 1 of 64 and of 65 tiles; one column of interior cells (1000 cells in one workgroup,
# more below them than there are threads); coarsest levels 3, 4, 2 and 1 cells wide
@pytest.mark.parametrize("sweeps", [2, 5])
@pytest.mark.parametrize("nx,ny,seed", [(4096, 20, 61), (4098, 20, 62), (3, 4000, 63),
                                        (97, 70, 64), (128, 66, 65), (70, 140, 66),
                                        (20, 300, 67), (257, 255, 68)])
def test_cycle_against_fp64(nx, ny, seed, sweeps):
    lab = irregular_labels(nx, ny, seed, n_obst=3 if nx > 3 else 0)
    d, g = _solve_pair(lab, seed, mg_level_sweeps=sweeps)
    st = g.stats()
    liq = lab == LIQ
    ep = rel_err(g.pressure()[liq], d.pressure[liq])
    print(f"{nx}x{ny}, level sweeps {sweeps}: {st.cg_iterations} iterations, "
          f"|r|/|b| {st.cg_error:.2e}, p vs fp64 {ep:.2e}")
    # the residual bound of the solve, and with it the error at a condition of at most 1e4
    assert st.cg_error <= 1e-10
    assert ep <= 1e-6


def test_cycles_of_several_threads():
    """Six domains stepped by a thread each end as they do one after the other."""
    def run(n, out):
        sc = scenes.dam_break(n)
        d = fsg.Domain.from_scene(sc, cg_tol=1e-6, cg_max_iter=200, solver=fsg.SOLVER_MG,
                                  deterministic=1)
        for _ in range(12):
            d.step(fsg.PICFLIP, sc.dt)
        out[n] = (d.pressure().copy(), d.stats().cg_iterations)
        d.close()

    sizes = [96, 130, 200, 257, 384, 512]
    alone, together = {}, {}
    for n in sizes:
        run(n, alone)
    threads = [threading.Thread(target=run, args=(n, together)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n in sizes:
        assert together[n][1] == alone[n][1]
        assert np.array_equal(together[n][0].view(np.uint32), alone[n][0].view(np.uint32))
