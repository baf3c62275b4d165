"""The particle density's float form (deterministic sums off) against FP64 sums of the same
float32 terms: blocks whose footprint fits the LDS copy (sorted) and does not (mixed), a
particle that is not a number among them, and weights far below one."""
from __future__ import annotations

import numpy as np
import pytest

from fluid_simulation_amd import fsg

pytestmark = pytest.mark.gpu


def _terms(p, nx, ny, dx):
    """(cell, term) of every particle: float32 weights, as Grid::addToValueInterpolated."""
    f = np.float32
    xs, ys = (p[:, 0] / f(dx)).astype(f), (p[:, 1] / f(dx)).astype(f)
    i, j = xs.astype(np.int32), ys.astype(np.int32)
    fi, fj = xs - i.astype(f), ys - j.astype(f)
    cells, terms = [], []
    for b, wy in ((0, f(1) - fj), (1, fj)):
        for a, wx in ((0, f(1) - fi), (1, fi)):
            cells.append(np.clip(i + a, 0, nx - 1) + np.clip(j + b, 0, ny - 1) * nx)
            terms.append((wx * wy).astype(np.float64))
    return np.concatenate(cells), np.concatenate(terms)


def _density(p, nx, ny, dx):
    """FP64 sums, and the bound of any order of float32 additions: every addition is off by
    at most 2^-24 of the terms' absolute sum, n additions in a cell of n terms."""
    c, t = _terms(p, nx, ny, dx)
    sums = np.zeros(nx * ny)
    np.add.at(sums, c, t)
    bound, count = np.zeros(nx * ny), np.zeros(nx * ny)
    np.add.at(bound, c, np.abs(t))
    np.add.at(count, c, 1.0)
    return sums.reshape(ny, nx), (bound * count * 2.0 ** -24).reshape(ny, nx)


@pytest.mark.parametrize("order", ["sorted", "mixed"])
@pytest.mark.parametrize("nx,ny,dx,n", [(40, 30, 1.0, 1), (40, 30, 1.0, 255), (64, 32, 0.5, 4097),
                                        (300, 200, 0.5, 20001), (2048, 3, 1.0, 3001)])
def test_float_sums(nx, ny, dx, n, order):
    rng = np.random.default_rng(n)
    p = np.zeros((n, 4), np.float32)
    p[:, 0] = rng.uniform(-0.4, nx + 0.4, n) * dx
    p[:, 1] = rng.uniform(-0.4, ny + 0.4, n) * dx
    if order == "sorted":
        p = p[np.lexsort((np.floor(p[:, 0] / dx / 8), np.floor(p[:, 1] / dx / 8)))]
    d = fsg.Domain(nx, ny, nx * dx, ny * dx, 0.01, 0.05)
    d.set_params(deterministic=0)
    d.set_particles(p)
    want, bound = _density(p, nx, ny, dx)
    assert (np.abs(d.density() - want) <= bound).all()
    # a particle that is not a number reaches its own cells only
    k = n // 2
    p[k, 0] = np.nan
    d.set_particles(p)
    rest = np.delete(p, k, 0)
    want, bound = _density(rest, nx, ny, dx)
    got = d.density()
    j = min(max(int(np.float32(p[k, 1]) / np.float32(dx)), 0), ny - 1)
    lost = np.isnan(got)
    assert lost.any() and not np.delete(lost, [j, min(j + 1, ny - 1)], 0).any()
    assert (np.abs(got - want)[~lost] <= bound[~lost]).all()
    d.close()


@pytest.mark.parametrize("k", range(1, 21))
def test_small_weights(k):
    """One particle a little past a grid line in both directions: the far corner's weight,
    about 2^-2k, is as exact as float32 multiplies it (a single term in every cell)."""
    nx, ny = 40, 30
    f = np.float32
    # an odd number of units in the last place of a coordinate in [1, 2)
    frac = f(max(int(1.37 * 2.0 ** (23 - k)) | 1, 3)) * f(2.0 ** -23)
    p = np.array([[f(1) + frac, f(1) + frac, 0, 0]], f)
    d = fsg.Domain(nx, ny, nx, ny, 0.01, 0.05)
    d.set_params(deterministic=0)
    d.set_particles(p)
    want, bound = _density(p, nx, ny, 1.0)
    assert want[2, 2] > 0
    assert (np.abs(d.density() - want) <= bound).all()
    d.close()
