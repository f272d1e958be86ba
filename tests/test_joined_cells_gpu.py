"""Cells whose polygons are joined into several polyhedra, every pattern of a
hexagon next to other cubes, polygons of three to six lines, and spacings on
both sides of the range that one lane per cell takes: bit by bit equal to the
oracle."""
import numpy as np
import pytest

import cornelius_lib as CL
import gpuvh

pytestmark = pytest.mark.gpu
V0 = 0.5
CORNERS = np.arange(16)


def cells_of(masks, rng):
    side = np.where((np.asarray(masks)[:, None] >> CORNERS) & 1, 1.0, -1.0)
    return V0 + side * rng.uniform(0.01, 1.0, side.shape)


def check(dim, cells, dx):
    counts, cen, nrm = gpuvh.cornelius_cells(dim, cells, np.full(dim, dx), V0)
    for i, c in enumerate(cells):
        a, b = CL.find(dim, c, np.full(dim, dx), V0)
        assert counts[i] == len(a), i
        assert np.array_equal(cen[i, :len(a)], a, equal_nan=True), i
        assert np.array_equal(nrm[i, :len(a)], b, equal_nan=True), i
    return counts


def test_several_polyhedra():
    """Corners with no neighbour of their own kind: an element around each, or
    around several, as the means of the crossed squares have it."""
    even = [c for c in range(16) if bin(c).count("1") % 2 == 0]
    masks = [sum(1 << c for k, c in enumerate(even) if n >> k & 1) for n in range(256)]
    counts = check(4, cells_of(masks + [m ^ 0xffff for m in masks], np.random.default_rng(1)), 0.1)
    assert counts.max() > 2


def test_hexagons():
    """The six corners next to one corner's opposite, in each of the eight
    cubes, with every state of the opposite cube's corners that are left."""
    rng = np.random.default_rng(2)
    masks = []
    for axis in range(4):
        for j in range(2):
            cube = [c for c in range(16) if (c >> (3 - axis) & 1) == j]
            other = [c for c in range(16) if (c >> (3 - axis) & 1) != j]
            for p in range(8):  # a corner and its three neighbours, less one: six cut squares
                near = [c for c in cube if bin(c ^ cube[p]).count("1") <= 1]
                for n in rng.integers(0, 256, 24):
                    masks.append(sum(1 << c for c in near) | sum(1 << c for k, c in enumerate(other) if n >> k & 1))
    check(4, cells_of(masks, rng), 0.2)


@pytest.mark.parametrize("dim", [3, 4])
@pytest.mark.parametrize("dx", [1e-62, 1e-59, 1e59, 1e62])
def test_spacings(dim, dx):
    rng = np.random.default_rng(3)
    check(dim, V0 + rng.standard_normal((130, 1 << dim)), dx)
