"""The electrostatic potential at points (a wave per point) against a FP64 sum on the host.

Fewer and more sites than a wave's lanes and remainders of them, one point, remainders of a block.
The same FP64 terms in another order: n terms of size v / cancellation, so 1e-11 of the largest
potential is a thousand times the rounding of 1000 terms.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


@pytest.mark.parametrize('waters, points', [(3, 1), (14, 5), (16, 64), (17, 257), (60, 1003)])
def test_potential(mb, waters, points):
    w = mb.systems.cluster(waters, seed=2)
    sysm = mb.forcefield.create_system(waters, nonbonded_method='CutoffNonPeriodic', nonbonded_cutoff=1e3,
                                       dipole_epsilon=1e-6, components=16)
    ctx = mb.Context(sysm, precision='double')
    pos = mb.forcefield.water_positions_with_m(w)
    ctx.setPositions(pos)
    pts = np.random.default_rng(4).uniform(2.5, 4.0, (points, 3))
    got = ctx.getElectrostaticPotential(pts)
    q, mu = ctx.getCharges(), ctx.getInducedDipoles()
    d = pos[None] - pts[:, None]
    r = np.sqrt((d * d).sum(-1))
    ref = (q / r - (mu[None] * d).sum(-1) / r ** 3).sum(1)
    scale = (np.abs(q) / r).sum(1).max()
    factor = (got @ ref) / (ref @ ref)  # the unit conversion (kJ nm / mol e^2)
    print(waters, points, factor, np.abs(got - factor * ref).max() / (factor * scale), flush=True)
    assert abs(factor - 138.935) < 0.01
    assert np.abs(got - factor * ref).max() <= 1e-11 * factor * scale
