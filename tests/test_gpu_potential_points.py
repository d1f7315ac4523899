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


def potential(mb, ctx, pts):
    import ctypes
    dp = ctypes.POINTER(ctypes.c_double)
    out = np.full(len(pts), np.nan)
    rc = mb.api.library().mbpol_context_get_electrostatic_potential(ctx._h, len(pts), pts.ctypes.data_as(dp),
                                                                    out.ctypes.data_as(dp))
    assert rc == 0, mb.api.library().mbpol_last_error()
    return out


@pytest.mark.parametrize('waters', [1, 3, 16, 17, 60, 'box'])
def test_same_bits_for_any_number_of_points(mb, waters):
    """A point's potential is the same however many lanes take it."""
    if waters == 'box':
        w, box = mb.systems.config1()
        sysm = mb.forcefield.create_system(256, nonbonded_method='PME', box=box, ewald_error_tolerance=1e-5,
                                           dipole_epsilon=1e-6, components=16)
    else:
        w = mb.systems.cluster(waters, seed=2)
        sysm = mb.forcefield.create_system(waters, nonbonded_method='CutoffNonPeriodic', nonbonded_cutoff=1e3,
                                           dipole_epsilon=1e-6, components=16)
    ctx = mb.Context(sysm, precision='double')
    ctx.setPositions(mb.forcefield.water_positions_with_m(w))
    ctx.getState(components=16)
    pts = np.random.default_rng(6).uniform(2.5, 4.0, (200001, 3))
    most = potential(mb, ctx, pts)
    for n in (1, 63, 4096, 4097, 65537, 100000):
        assert np.array_equal(potential(mb, ctx, pts[:n].copy()), most[:n])


def test_more_points_than_a_launch_has_waves(mb):
    """2^26 points and more: 64 threads a point would be 2^32 threads."""
    sysm = mb.forcefield.create_system(1, nonbonded_method='CutoffNonPeriodic', nonbonded_cutoff=1e3,
                                       dipole_epsilon=1e-6, components=16)
    ctx = mb.Context(sysm, precision='double')
    ctx.setPositions(mb.forcefield.water_positions_with_m(mb.systems.cluster(1, seed=2)))
    ctx.getState(components=16)
    few = np.random.default_rng(8).uniform(2.5, 4.0, (4099, 3))
    want = potential(mb, ctx, few)
    total = 2 ** 26 + 4099
    got = potential(mb, ctx, np.resize(few, (total, 3)))
    whole = total // len(few) * len(few)
    assert (got[:whole].reshape(-1, len(few)) == want).all()
    assert np.array_equal(got[whole:], want[:total - whole])
