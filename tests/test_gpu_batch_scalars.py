"""The packed batch's per-scene CG: level-0 tiles that hold cells of one, of up to four, and
of more than four scenes (whose sums then take a kernel of their own): every scene steps like
a domain of its own."""
from __future__ import annotations

import numpy as np
import pytest

from fluid_simulation_amd import fsg, scenes

from helpers import rel_err

pytestmark = pytest.mark.gpu


# scenes of 9 x 12 cells: up to nine per tile; 20 x 17: up to four; 64 to 90: mostly one
@pytest.mark.parametrize("lo,hi,count", [(9, 12, 14), (17, 20, 9), (64, 90, 5)])
def test_scenes_match_single_domains(lo, hi, count):
    scs = scenes.dam_break_batch(count, lo, hi, seed=7)
    b = fsg.Batch.from_scenes(scs, cg_tol=1e-10, cg_max_iter=500)
    singles = [fsg.Domain.from_scene(sc, cg_tol=1e-10, cg_max_iter=500, solver=fsg.SOLVER_MG)
               for sc in scs]
    for _ in range(3):
        b.step(fsg.PICFLIP, 0.01)
        for d in singles:
            d.step(fsg.PICFLIP, 0.01)
    # both solve to 1e-10: within 1e-5 after three steps, as for the larger batches
    for s, d in enumerate(singles):
        assert rel_err(b.scene_particles(s), d.particles()) <= 1e-5
        assert np.array_equal(b.scene_labels(s), d.labels())
