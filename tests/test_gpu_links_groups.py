"""The link build's nearest-point search by groups of 64 triangles: soups
just below, at and above whole groups, triangles in an order without
locality, duplicated triangles (the first of equal minima counts) and
degenerate ones, against the oracle bit for bit."""
import numpy as np
import pytest

from octlb_amd import cases, geometry
from oracle import binding

pytestmark = pytest.mark.gpu

CENTRE, R = (0.53, 0.47, 0.51), 0.31


def _soup(count, order, seed):
    s = geometry.sphere_soup(CENTRE, R, 24)
    rng = np.random.default_rng(seed)
    s = s[rng.permutation(len(s))[:count]]
    if order == "twice":
        s = np.concatenate([s, s[::-1]])
    if order == "degenerate":
        s[::3, 3:6] = s[::3, 0:3]
        s[1::7, 3:] = np.tile(s[1::7, :3], 2)
    return s


@pytest.mark.parametrize("count", [1, 63, 64, 65, 128, 1000])
@pytest.mark.parametrize("order", ["shuffled", "twice", "degenerate"])
def test_links_bitwise(count, order):
    topo = cases.synthetic_forest(2, 1, (0.5,)).topology(8, 1)
    x, y, z = CENTRE
    mat = geometry.material_field(topo, lambda a, b, c: (a - x) ** 2 + (b - y) ** 2 + (c - z) ** 2 < R * R)
    soup = _soup(count, order, count)
    link, q = geometry.build_links(topo.bounds, 8, mat, soup)
    want_link, want_q = binding.build_links(topo.bounds, 8, mat, soup)
    assert len(want_q) > 0
    np.testing.assert_array_equal(link, want_link)
    np.testing.assert_array_equal(q, want_q)
