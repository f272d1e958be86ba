"""Cells whose element needs no joining are built one per lane, the others one
per wave: both in one call, bit by bit equal to the oracle, at cell counts
around a wave's 64 and with every number of lines per cube, all corner
patterns, corners exactly on the iso-value and values that are no number."""
import numpy as np
import pytest

import cornelius_lib as CL
import gpuvh

pytestmark = pytest.mark.gpu
V0 = 0.5


def smooth(dim, n, rng):
    """Corners of a plane with a little curvature that passes near the middle."""
    bits = np.array([[(c >> (dim - 1 - k)) & 1 for k in range(dim)] for c in range(1 << dim)]) - 0.5
    g = rng.standard_normal((n, dim))
    v = g @ bits.T + 0.05 * rng.standard_normal((n, 1 << dim))
    return V0 + v + 0.8 * rng.standard_normal((n, 1))


def patterns(dim, rng):
    """Every pattern of corners above and below (a sample of them in 4-D)."""
    nc = 1 << dim
    masks = np.arange(1 << nc) if dim == 3 else rng.permutation(1 << nc)[:6000]
    side = np.where((masks[:, None] >> np.arange(nc)) & 1, 1.0, -1.0)
    return V0 + side * rng.uniform(0.01, 1.0, side.shape)


def check(dim, cells, dx):
    counts, cen, nrm = gpuvh.cornelius_cells(dim, cells, dx, V0)
    for i, c in enumerate(cells):
        a, b = CL.find(dim, c, dx, V0)
        assert counts[i] == len(a), i
        assert np.array_equal(cen[i, :len(a)], a) and np.array_equal(nrm[i, :len(a)], b), i


@pytest.mark.parametrize("dim", [3, 4])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
def test_smooth_cells(dim, n):
    rng = np.random.default_rng(100 * dim + n)
    cells = smooth(dim, n, rng)
    # corners exactly on the iso-value, next to it, and far beyond it
    for i in range(0, n, 3):
        k = rng.integers(0, 1 << dim, 2)
        cells[i, k] = [V0, V0 + rng.choice([0.0, 1e-300, -1e-17, 1e300])]
    check(dim, cells, np.array([0.1, 0.15, 0.2, 0.05][:dim]))


@pytest.mark.parametrize("dim", [3, 4])
def test_corner_patterns(dim):
    check(dim, patterns(dim, np.random.default_rng(dim)), np.array([1.0, 0.5, 0.25, 2.0][:dim]))


@pytest.mark.parametrize("dim", [3, 4])
def test_values_that_are_no_number(dim):
    """Such cells take the general search, as all did; the others of their
    waves are not touched by them."""
    rng = np.random.default_rng(7)
    cells = smooth(dim, 256, rng)
    bad = cells.copy()
    bad[5::16, 1] = np.nan
    bad[9::16, 2] = np.inf
    dx = np.ones(dim)
    a, b = gpuvh.cornelius_cells(dim, cells, dx, V0), gpuvh.cornelius_cells(dim, bad, dx, V0)
    same = np.isfinite(bad).all(axis=1)
    for x, y in zip(a, b):
        assert np.array_equal(x[same], y[same])
