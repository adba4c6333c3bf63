"""Push tiles made of wave tasks: same state and averages as the pull scheme.

A push tile holds 16 tasks of 64 cells, filled over block and member borders,
so the sizes give one push block (half a tile), odd counts and one member
without any; both statistics orders, populations and averages bit for bit.
The pull scheme itself is held against the oracle elsewhere.
"""
import numpy as np
import pytest

from octlb_amd import cases
from octlb_amd.solver import GpuSolver

pytestmark = pytest.mark.gpu


def _run(ens, precision, variant, count):
    s = GpuSolver.ensemble(ens, precision)
    s.set_bc_kinds(ens.kinds)
    s.init_equilibrium(1.0, (0.0, 0.0, 0.0), 0xFF)
    s.set_kernel_variant(variant)
    s.advance(2)
    s.advance_graph(9)
    out = s.download_core(), [s.member_average_rho(m) for m in range(count)], s.kernel_variant()[1]
    s.close()
    return out


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("fast_stats", [0, 1])
@pytest.mark.parametrize("sizes,npush", [((24,), 1), ((16, 24, 40), 28), ((40, 48), 91)])
def test_push_tasks_match_pull(sizes, npush, fast_stats, precision):
    members = [cases.cavity_blocked(n, 0.6 + 0.05 * m, 0.03 + 0.01 * m, 1, x0=2.0 * m) for m, n in enumerate(sizes)]
    ens = cases.ensemble(members, fast_stats=fast_stats)
    pull = _run(ens, precision, 0, len(sizes))
    push = _run(ens, precision, 1, len(sizes))
    assert pull[2] == 0 and push[2] == npush
    np.testing.assert_array_equal(push[0], pull[0])
    assert push[1] == pull[1]
