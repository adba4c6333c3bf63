"""Padded blocks in FP32: the FD boundary pass, the output fields and the
average in the reference's order, at edges that are no multiple of the 8^3
tile, against the FP64 oracle or 64-bit arithmetic.

Tolerances: a population is at most about 0.1 and leaves a step after some
hundred roundings of 2^-24, so a step adds at most 1e-6; it passes on what it
got at most doubled, which makes (2^k - 1) 1e-6 after k steps.  Density and
momentum are sums of 19 populations: 20 2^-24 times the sum of their sizes,
the division included."""
import numpy as np
import pytest

from octlb_amd import cases
from tests.test_gpu_ordered_average import _case as average_case
from tests.test_gpu_padded_boundary import _case
from tests.util import make_gpu, make_oracle, random_pops

pytestmark = pytest.mark.gpu

STEP = 1e-6


@pytest.mark.parametrize("n,halo", [(4, 1), (5, 2), (8, 3), (9, 1), (17, 3)])
@pytest.mark.parametrize("scatter", [False, True])
def test_fd_pass(n, halo, scatter):
    case = _case(n, halo, scatter)
    pops = random_pops(case, n, 0.002).astype(np.float32).astype(np.float64)
    o, g = make_oracle(case, pops), make_gpu(case, 32, pops)
    for k in (1, 2, 3):
        o.advance(1)
        g.advance(1)
        assert np.abs(g.download_core() - o.download_core()).max() <= (2 ** k - 1) * STEP


@pytest.mark.parametrize("n,halo", [(4, 1), (8, 2), (9, 1), (17, 2), (20, 3)])
def test_fields(n, halo):
    case = _case(n, halo, False)
    g = make_gpu(case, 32, random_pops(case, n, 0.002))
    rho, u = g.macro_fields()
    f = g.download_core()  # [block, x, y, z, 19]
    r = 1.0 + f.sum(-1)
    m = f @ np.asarray(cases.C, np.float64)
    tol = 20 * 2.0 ** -24 * np.abs(f).sum(-1)
    assert (np.abs(rho.transpose(0, 3, 2, 1) - r) <= tol).all()
    assert (np.abs(u.transpose(0, 3, 2, 1, 4) - m / r[..., None]) <= 2 * tol[..., None]).all()


@pytest.mark.parametrize("n,halo", [(4, 1), (9, 3), (10, 2), (21, 1), (34, 3)])
@pytest.mark.parametrize("seed,spread", [(2, 0.05), (3, 0.2)])
def test_average(n, halo, seed, spread):
    case = average_case(n, halo, seed, spread)
    o, g = make_oracle(case), make_gpu(case, 32)
    for k in (1, 2, 3):
        o.advance(1)
        g.advance(1)
        assert abs(g.average_rho() - o.average_rho()) <= (2 ** k - 1) * STEP
