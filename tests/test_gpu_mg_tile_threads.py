"""Multigrid hierarchies whose level 1 has 256, 257 and more tiles: levels with launches of
their own above those that share one, against the FP64 oracle."""
from __future__ import annotations

import pytest

from fluid_simulation_amd import fsg  # noqa: F401  (the library is loaded before the oracle)

from helpers import rel_err
from test_gpu_mg import LIQ, _solve_pair, irregular_labels

pytestmark = pytest.mark.gpu


# level 1 is (nx + 1) // 2 x (ny + 1) // 2 cells in tiles of 32 x 32
@pytest.mark.parametrize("sweeps", [2, 5, 6])
@pytest.mark.parametrize("nx,ny,seed", [(16384, 20, 51), (16386, 20, 52), (1090, 1027, 53)])
def test_tile_threads_against_fp64(nx, ny, seed, sweeps):
    lab = irregular_labels(nx, ny, seed, liquid_frac=0.85 if ny > 20 else 0.7)
    d, g = _solve_pair(lab, seed, mg_level_sweeps=sweeps)
    st = g.stats()
    liq = lab == LIQ
    ep = rel_err(g.pressure()[liq], d.pressure[liq])
    print(f"{nx}x{ny}, level sweeps {sweeps}: {st.cg_iterations} iterations, "
          f"|r|/|b| {st.cg_error:.2e}, p vs fp64 {ep:.2e}")
    # the residual bound of the solve, and with it the error at a condition of at most 1e4
    assert st.cg_error <= 1e-10
    assert ep <= 1e-6
