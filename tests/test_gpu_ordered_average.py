"""The ConstRho average summed in the reference's cell order: the parallel
sum rounds exactly as the one-by-one loop of the oracle, so average and
populations are equal bit for bit, whatever the values are -- sums that cross
many binades, ties, negative densities (which the parallel form leaves to the
loop) and cells that do not count."""
import numpy as np
import pytest

from octlb_amd import cases
from tests.util import make_gpu, make_oracle

pytestmark = pytest.mark.gpu


def _case(n, halo, seed, spread):
    case = cases.cavity(n, tau=0.7, halo=halo)
    rng = np.random.default_rng(seed)
    rho = np.exp(rng.uniform(-spread, spread, case.kinds.shape))
    if seed % 2:  # values that are multiples of 2^-20: every add of a long run may tie
        rho = np.round(rho * 2.0 ** 20) / 2.0 ** 20
    if spread > 2.0:
        rho[0, 1, 1, : n // 2] = -0.25
    case.init_field = (rho, rng.uniform(-0.01, 0.01, case.kinds.shape + (3,)))
    return case


# cells per side: below one chunk of 1,024 cells (9^3), just beside whole
# chunks (10^3, 16^3), several chunks with a remainder
@pytest.mark.parametrize("n,halo", [(4, 1), (9, 3), (10, 2), (16, 3), (21, 1), (34, 3)])
@pytest.mark.parametrize("seed,spread", [(2, 0.05), (3, 0.4), (4, 3.0)])
def test_padded_average_bitwise(n, halo, seed, spread):
    case = _case(n, halo, seed, spread)
    o, g = make_oracle(case), make_gpu(case)
    for _ in range(3):
        o.advance(1)
        g.advance(1)
        assert g.average_rho() == o.average_rho()
    np.testing.assert_array_equal(g.download_core(), o.download_core())
