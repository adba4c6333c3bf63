"""The device voxelizer's exact pass (one wave per cell that the filters leave
open, its candidate triangles queued 64 at a time) on soups symmetric about
cell faces and cell centres, where many predicates are exactly zero: fewer
triangles than one wave, queues that fill several times over, every triangle
twice; against the oracle byte for byte."""
import numpy as np
import pytest

from octlb_amd import geometry
from oracle import binding

pytestmark = pytest.mark.gpu

BOUNDS = np.array([[0.0, 0.0, 0.0, 0.5, 0.5, 0.5], [0.5, 0.5, 0.0, 1.0, 1.0, 0.5]])
CENTRE = (0.5, 0.5, 0.5)


def _soup(name):
    if name == "octants":  # 32 triangles, vertices on the axes through cell faces
        return geometry.sphere_soup(CENTRE, 0.375, 4)
    if name == "fan":  # 480 triangles that all meet at two points
        return geometry.sphere_soup(CENTRE, 0.375, 16)[:480]
    if name == "twice":
        s = geometry.sphere_soup(CENTRE, 0.25, 8)
        return np.concatenate([s, s[::-1]])
    return np.concatenate([geometry.box_soup((k / 64.0,) * 3, (1.0 - k / 64.0,) * 3) for k in range(0, 24, 2)])


@pytest.mark.parametrize("n", [4, 8, 9])
@pytest.mark.parametrize("name", ["octants", "fan", "twice", "nested boxes"])
def test_obstacle(n, name):
    soup = _soup(name)
    got, exact = geometry.voxelize_part(BOUNDS, n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    np.testing.assert_array_equal(got, binding.voxelize_part(BOUNDS, n, soup, geometry.PART_EXTERNAL_OBSTACLE))
    if name != "nested boxes" and n != 9:  # its centres and faces miss the soup's vertices
        assert exact > 0


@pytest.mark.parametrize("n", [8, 9])
def test_channel(n):
    inner = geometry.sphere_soup(CENTRE, 0.25, 8)
    args = (BOUNDS, n, np.concatenate([geometry.sphere_soup(CENTRE, 0.4375, 8), inner]),
            geometry.PART_INTERNAL_CHANNEL, inner)
    got, exact = geometry.voxelize_part(*args)
    np.testing.assert_array_equal(got, binding.voxelize_part(*args))
    if n != 9:
        assert exact > 0


def test_more_open_cells_than_the_first_room():
    """More cells than the call's first queue holds (131,072), against the same
    blocks in calls that each stay below."""
    k = 46
    at = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3) / k
    bounds = np.concatenate([at, at + 1.0 / k], 1)
    soup = geometry.sphere_soup(CENTRE, 0.375, 4)
    got, exact = geometry.voxelize_part(bounds, 8, soup, geometry.PART_EXTERNAL_OBSTACLE)
    parts = [geometry.voxelize_part(b, 8, soup, geometry.PART_EXTERNAL_OBSTACLE) for b in np.array_split(bounds, 24)]
    assert exact > 131072 > max(n for _, n in parts)
    assert exact == sum(n for _, n in parts)
    assert np.array_equal(got, np.concatenate([m for m, _ in parts]))
