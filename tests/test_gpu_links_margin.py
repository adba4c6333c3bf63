"""The link build's pruning by group boxes keeps the first minimum of the full
scan where computed edge points fall beyond their box: a wall of triangles
whose long edges, from coordinates of +200 to +500, end 1e-4 in front of cell
centres near -100, so that b - a is rounded by up to 4 ulps of the end point.
Ends differ by a few ulps between the groups of 64, so a point beyond its box
is the nearest one for nearly every cell.  Bit for bit against the oracle."""
import numpy as np
import pytest

from octlb_amd import geometry
from oracle import binding

pytestmark = pytest.mark.gpu

ORIGIN, DX = -100.0, 1.0 / 64.0


def _wall(seed, groups):
    """A group per layer of 64 triangles, one for each cell of the layer next
    to the wall; the first group's edges are short and exact."""
    rng = np.random.default_rng(seed)
    at = ORIGIN + (np.arange(8) + 0.5) * DX
    y, z = (v.reshape(-1) for v in np.meshgrid(at, at, indexing="ij"))
    x = ORIGIN + 3.5 * DX + 1e-4
    out = []
    for g in range(groups):
        ulps, near, far = (rng.integers(1, 4), 300.0, 600.0) if g else (0, 1.0, 40.0)
        end = np.stack([np.full(64, x + ulps * abs(np.spacing(x))), y, z], 1)
        start = np.stack([x + rng.uniform(near, far, (64, 2)), ORIGIN + rng.uniform(0.0, 8 * DX, (64, 2)),
                          ORIGIN + rng.uniform(0.0, 8 * DX, (64, 2))], -1)
        out.append(np.concatenate([start[:, 0], end, start[:, 1]], 1))
    return np.concatenate(out)


@pytest.mark.parametrize("seed,groups", [(0, 2), (1, 24), (2, 90)])
def test_first_minimum_beyond_its_box(seed, groups):
    material = np.zeros((1, 8, 8, 8), np.uint8)  # [block][k][j][i]
    material[..., 4:] = geometry.MAT_SOLID
    bounds = np.array([[ORIGIN] * 3 + [ORIGIN + 8 * DX] * 3])
    soup = _wall(seed, groups)
    link, q = geometry.build_links(bounds, 8, material, soup)
    want_link, want_q = binding.build_links(bounds, 8, material, soup)
    assert len(want_q) >= 64
    np.testing.assert_array_equal(link, want_link)
    np.testing.assert_array_equal(q, want_q)
