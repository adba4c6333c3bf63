"""The device voxelizer where few triangles (at most 64) meet many blocks (512
tiles of 8^3 cells per triangle, or more): a thread per cell, a wave's lanes
choosing among the triangles.  Block edges around a wave's 64 and 256 cells, one
and 64 triangles, and 65; all blocks byte for byte against calls with too few
blocks for that way (one triangle keeps to it), every 31st against the oracle."""
import numpy as np
import pytest

from octlb_amd import geometry
from oracle import binding

pytestmark = pytest.mark.gpu


def _bounds(k):
    """k^3 blocks that tile the unit cube."""
    at = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3) / k
    return np.concatenate([at, at + 1.0 / k], 1)


def _equal(bounds, n, *args):
    got, exact = geometry.voxelize_part(bounds, n, *args)
    parts = [geometry.voxelize_part(np.ascontiguousarray(b), n, *args) for b in np.array_split(bounds, 16)]
    np.testing.assert_array_equal(got, np.concatenate([m for m, _ in parts]))
    assert exact == sum(e for _, e in parts)
    some = np.ascontiguousarray(bounds[::31])
    np.testing.assert_array_equal(got[::31], binding.voxelize_part(some, n, *args))
    return got, exact


# 12 triangles: 6,144 tiles and more from 6,859 blocks of one tile, or 1,000 of eight
@pytest.mark.parametrize("k, n", [
    (19, 1), (19, 3), (19, 4), (19, 7), (19, 8), (10, 9), (10, 16), (18, 4)])  # 18: too few
def test_box(k, n):
    got, _ = _equal(_bounds(k), n, geometry.box_soup((0.13, 0.12, 0.11), (0.83, 0.71, 0.5)),
                    geometry.PART_EXTERNAL_OBSTACLE)
    assert set(np.unique(got)) >= {geometry.MAT_FLUID, geometry.MAT_BOUNDARY}


@pytest.mark.parametrize("count", [1, 63, 64, 65])
def test_counts(count):
    """A lattice soup: degenerate triangles, vertices and edges on cell faces and
    centres, so that filters stay open.  64 triangles take 32,768 tiles."""
    rng = np.random.default_rng(count)
    soup = (np.round(rng.random((count, 3, 3)) * 64) / 64).reshape(-1, 9)
    soup[::7, 3:6] = soup[::7, :3]
    _, exact = _equal(_bounds(32), 2, soup, geometry.PART_EXTERNAL_OBSTACLE)
    assert exact > 0 or count == 1


@pytest.mark.parametrize("n", [2, 3])
def test_channel(n):
    outer = geometry.box_soup((0.05, 0.05, 0.05), (0.95, 0.95, 0.95))
    inner = geometry.box_soup((0.21, 0.22, 0.23), (0.81, 0.79, 0.77))
    got, _ = _equal(_bounds(27), n, np.concatenate([outer, inner]), geometry.PART_INTERNAL_CHANNEL, inner)
    assert set(np.unique(got)) == {geometry.MAT_FLUID, geometry.MAT_SOLID, geometry.MAT_BOUNDARY}
