"""The link build's two ways to go over the triangles -- each wave over the
groups near its cell, or a workgroup's waves over the whole soup 256 triangles at
a time -- around the line between them: soups of up to 256 triangles, groups that
hold every cell or none, one kept group in two, groups of more than 64 triangles,
candidate cells that are no multiple of four; bit for bit against the oracle."""
import numpy as np
import pytest

from octlb_amd import geometry
from oracle import binding

pytestmark = pytest.mark.gpu


def _slivers(count, seed):
    """Across the whole domain: every group's box holds every cell."""
    a, b = np.random.default_rng(seed).random((2, count, 3))
    return np.concatenate([a, b, b + 1e-3], 1)


def _plate(count, seed, sort):
    """Small triangles in the plane z = 0.5; no box holds a cell centre.  The
    first `sort` of them are in the order of their place."""
    rng = np.random.default_rng(seed)
    a = np.concatenate([rng.random((count, 2)), np.full((count, 1), 0.5)], 1)
    at = np.lexsort((a[:, 1], np.floor(a[:, 0] * 8.0)))
    a[:sort] = a[at][:sort]
    step = np.concatenate([rng.normal(0.0, 0.02, (count, 2)), np.zeros((count, 1))], 1)
    return np.concatenate([a, a + step, a + step[:, [1, 0, 2]]], 1)


def _check(soup, solid, seed, rest=geometry.MAT_FLUID, those=geometry.MAT_SOLID):
    """`solid` cells of one material among the rest of the other."""
    at = np.stack(np.meshgrid(*[np.arange(2)] * 3, indexing="ij"), -1).reshape(-1, 3) / 2.0
    bounds = np.concatenate([at, at + 0.5], 1)
    rng = np.random.default_rng(seed)
    material = np.full((8, 8, 8, 8), rest, np.uint8)
    material.reshape(-1)[rng.permutation(8 * 512)[:solid]] = those
    link, q = geometry.build_links(bounds, 8, material, soup)
    want_link, want_q = binding.build_links(bounds, 8, material, soup)
    assert len(want_q) > 0 or solid < 40 or len(soup) == 1
    np.testing.assert_array_equal(link, want_link)
    np.testing.assert_array_equal(q, want_q)


@pytest.mark.parametrize("count", [1, 255, 256, 257, 576, 577, 3000])
@pytest.mark.parametrize("name", ["slivers", "plate", "sorted plate", "half sorted plate"])
def test_links_bitwise(count, name):
    soup = _slivers(count, count) if name == "slivers" else _plate(
        count, count, {"plate": 0, "sorted plate": count, "half sorted plate": count // 2}[name])
    for solid in (1, 40):
        _check(soup, solid, count + solid)


@pytest.mark.parametrize("sort", [0, 1])
def test_groups_of_more_than_64(sort):
    count = 64 * 16384 + 100  # two times 64 triangles a group
    _check(_plate(count, 7, sort * count), 5, 7, rest=geometry.MAT_SOLID, those=geometry.MAT_FLUID)
