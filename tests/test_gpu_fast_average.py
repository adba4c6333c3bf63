"""The ConstRho average summed by chunks of 4,096 partials (fast_stats), a
partial per x plane of a block: members of less than a chunk, exactly one, several; step by step and from a captured graph, against the average
in the reference's order.  N positive values summed in any order are within
(N - 1) 2^-53 of the exact sum, so the two differ by at most twice that, once per
step taken."""
import numpy as np
import pytest

from octlb_amd import cases
from octlb_amd.solver import GpuSolver

pytestmark = pytest.mark.gpu


def _solver(sizes, precision, fast):
    members = [cases.cavity_blocked(n, 0.6 + 0.05 * m, 0.03 + 0.01 * m, 1, x0=2.0 * m) for m, n in enumerate(sizes)]
    ens = cases.ensemble(members, fast_stats=fast)
    s = GpuSolver.ensemble(ens, precision)
    s.set_bc_kinds(ens.kinds)
    s.init_equilibrium(1.0, (0.0, 0.0, 0.0), 0xFF)
    return s


# 8 partials, 1,000, 4,096 (a whole chunk), 5,832 (two chunks), 13,824; members of both kinds
@pytest.mark.parametrize("sizes", [(8,), (40,), (64,), (72,), (96,), (48, 8, 72, 40)])
@pytest.mark.parametrize("precision", [64, 32])
def test_matches_the_ordered_average(sizes, precision):
    fast, ordered = _solver(sizes, precision, 1), _solver(sizes, precision, 0)
    for k, steps in enumerate((1, 1, 1, 4)):
        for s in (fast, ordered):
            if steps == 1:
                s.advance(1)
            else:
                s.advance_graph(steps)
        taken = 1 + k if steps == 1 else 3 + steps
        for m, n in enumerate(sizes):
            want = ordered.member_average_rho(m)
            tol = 2 * taken * n ** 3 * 2.0 ** -53 if precision == 64 else 2 * taken * n ** 3 * 2.0 ** -53 + 2.0 ** -24
            assert abs(fast.member_average_rho(m) - want) <= tol * want
    again = _solver(sizes, precision, 1)
    again.advance(3)
    again.advance_graph(4)
    assert [again.member_average_rho(m) for m in range(len(sizes))] == [fast.member_average_rho(m)
                                                                       for m in range(len(sizes))]
    for s in (fast, ordered, again):
        s.close()


@pytest.mark.parametrize("n", [8, 40])
def test_a_member_beside_longer_ones(n):
    """Members of up to 1,024 partials go to a smaller kernel when all are: the
    same sum, bit for bit, as among longer ones."""
    alone, beside = _solver((n,), 64, 1), _solver((n, 72), 64, 1)
    for s in (alone, beside):
        s.advance(2)
        s.advance_graph(4)
    assert alone.member_average_rho(0) == beside.member_average_rho(0)
    for s in (alone, beside):
        s.close()
