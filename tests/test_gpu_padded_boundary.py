"""Padded blocks: the FD boundary pass and the output fields at block edges
that are no multiple of the 8^3 tile, against the oracle bit for bit."""
import numpy as np
import pytest

from octlb_amd import abi, cases
from octlb_amd.forest import single_block_topology
from tests.util import make_gpu, make_oracle, random_pops

pytestmark = pytest.mark.gpu


def _case(n, halo, scatter):
    """Velocity and pressure faces; with `scatter`, cells of both kinds in
    the interior and next to the faces as well."""
    topo = single_block_topology(n, halo)
    kinds = np.zeros((1, n, n, n), np.uint8)
    specs = [abi.make_spec(abi.XMIN, abi.BC_INTERP_VELOCITY, inlet=abi.INLET_UNIFORM, inlet_u=(0.03, 0.004, -0.002)),
             abi.make_spec(abi.XMAX, abi.BC_INTERP_PRESSURE, rho_target=1.01),
             abi.make_spec(abi.ZMIN, abi.BC_INTERP_VELOCITY),
             abi.make_spec(abi.ZMAX, abi.BC_INTERP_PRESSURE, rho_target=0.99),
             abi.make_spec(abi.YMAX, abi.BC_INTERP_VELOCITY, u_wall=(0.02, 0.0, 0.0))]
    cases.stamp_tree_boundary(kinds, topo.tree_boundary, specs)
    if scatter:
        rng = np.random.default_rng(n)
        at = rng.random(kinds.shape) < 0.08
        kinds[at] = rng.choice([abi.KIND_VELOCITY_DIRICHLET, abi.KIND_PRESSURE_DIRICHLET], at.sum())
    return cases.Case(name="padded", topo=topo, omega=1 / 0.7, handler=abi.HANDLER_CONCRETE, const_rho=0, bouzidi=0,
                      snapshot=0, specs=specs, kinds=kinds)


# the halo decides where a stencil beyond the block reads padding or a mirrored cell
@pytest.mark.parametrize("n,halo", [(4, 1), (5, 2), (8, 3), (9, 1), (17, 3)])
@pytest.mark.parametrize("scatter", [False, True])
def test_fd_pass_bitwise(n, halo, scatter):
    case = _case(n, halo, scatter)
    pops = random_pops(case, n, 0.002)
    o, g = make_oracle(case, pops), make_gpu(case, pops=pops)
    o.advance(1)
    g.advance(1)
    np.testing.assert_array_equal(g.download_core(), o.download_core())


@pytest.mark.parametrize("n,halo", [(4, 1), (8, 2), (9, 1), (20, 3)])
def test_fields_bitwise(n, halo):
    case = _case(n, halo, False)
    g = make_gpu(case, pops=random_pops(case, n, 0.002))
    rho, u = g.macro_fields()
    f = g.download_core()  # [block, x, y, z, 19], summed in population order as CellProxy does
    r, m = np.ones(f.shape[:-1]), np.zeros(f.shape[:-1] + (3,))
    for i in range(19):
        r = r + f[..., i]
        for d in range(3):
            if cases.C[i, d]:
                m[..., d] += f[..., i] * float(cases.C[i, d])
    np.testing.assert_array_equal(rho, r.transpose(0, 3, 2, 1))
    np.testing.assert_array_equal(u, (m / r[..., None]).transpose(0, 3, 2, 1, 4))
