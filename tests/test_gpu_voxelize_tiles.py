"""The device voxelizer on blocks that are not one 8^3 tile and on soups
around its triangle groups of 64 and candidate queue, against the oracle
byte for byte."""
import numpy as np
import pytest

from octlb_amd import geometry
from oracle import binding

pytestmark = pytest.mark.gpu

BOUNDS = np.array([[0.0, 0.0, 0.0, 0.5, 0.5, 0.5], [0.5, 0.0, 0.0, 1.0, 0.5, 0.5], [0.0, 0.5, 0.5, 0.5, 1.0, 1.0]])


def _soup(name):
    if name == "box":  # large triangles: every cell of a tile in reach of each; corners on cell faces
        return geometry.box_soup((0.125, 0.125, 0.125), (0.75, 0.4, 0.375))
    if name == "cylinder":  # open along z, slivers
        return geometry.cylinder_soup(0.41, 0.43, 0.21, -0.1, 1.1, 31, 1)
    if name == "sphere":  # 2 * 8^2 triangles: two whole groups
        return geometry.sphere_soup((0.47, 0.31, 0.29), 0.23, 8)
    return geometry.sphere_soup((0.51, 0.48, 0.5), 0.37, 40)  # 3,200 triangles: the queue fills


@pytest.mark.parametrize("n", [4, 7, 8, 9, 16, 18])
@pytest.mark.parametrize("name", ["box", "cylinder", "sphere", "fine sphere"])
def test_obstacle(n, name):
    soup = _soup(name)
    got, _ = geometry.voxelize_part(BOUNDS, n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    want = binding.voxelize_part(BOUNDS, n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    np.testing.assert_array_equal(got, want)
    assert (got != 0).any()


@pytest.mark.parametrize("n", [5, 8, 12])
def test_channel(n):
    outer = geometry.box_soup((0.05, 0.05, 0.05), (0.95, 0.95, 0.95))
    inner = geometry.sphere_soup((0.5, 0.45, 0.5), 0.3, 12)
    args = (BOUNDS, n, np.concatenate([outer, inner]), geometry.PART_INTERNAL_CHANNEL, inner)
    got, _ = geometry.voxelize_part(*args)
    np.testing.assert_array_equal(got, binding.voxelize_part(*args))
