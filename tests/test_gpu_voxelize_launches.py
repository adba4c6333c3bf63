"""The device voxelizer where its tiles are more workgroups than one launch
holds (2^32 threads): 2.1 million blocks of 9^3 cells, eight tiles each,
against the same blocks in two calls that each fit one launch."""
import numpy as np
import pytest

from octlb_amd import geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("more", [0, 128])  # a thread per cell; a workgroup per tile
def test_more_tiles_than_one_launch_holds(more):
    count, n = 2_100_000, 9
    assert count * 8 * 256 >= 2 ** 32
    at = np.stack(np.unravel_index(np.arange(count), (130, 130, 130)), -1).astype(np.float64)
    bounds = np.concatenate([at, at + 1.0], 1)
    soup = geometry.box_soup((0.3, 0.3, 0.3), (129.6, 129.6, 129.6))
    if more:
        soup = np.concatenate([soup, geometry.sphere_soup((500.0, 600.0, 700.0), 1.0, 8)])
    got, exact = geometry.voxelize_part(bounds, n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    half = count // 2
    lo, lo_exact = geometry.voxelize_part(bounds[:half], n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    assert np.array_equal(got[:half], lo)
    hi, hi_exact = geometry.voxelize_part(bounds[half:], n, soup, geometry.PART_EXTERNAL_OBSTACLE)
    assert np.array_equal(got[half:], hi)
    assert exact == lo_exact + hi_exact
    assert (hi == geometry.MAT_SOLID).any() and (hi == geometry.MAT_FLUID).any()
