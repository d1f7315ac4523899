"""3-body lists of more lower pairs than the trimer pass has groups of lanes.

A droplet without cutoffs, whose lower lists hold every pair: the pass strides over them, and the energies
and forces are those of the same droplet with a cutoff just beyond where the term ends (the same contributing
trimers, summed in fixed point), bit for bit.
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


def droplet(n):
    k = int(np.ceil(n ** (1 / 3)))
    rng = np.random.default_rng(n)
    site = np.stack(np.meshgrid(*(np.arange(k),) * 3, indexing='ij'), axis=-1).reshape(-1, 3)[:n]
    oxygen = site * 0.31 + rng.uniform(-0.015, 0.015, (n, 3))
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    turn = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
    return oxygen[:, None] + h @ turn


def energy(mb, waters, cutoff):
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='CutoffNonPeriodic', threebody_cutoff=cutoff,
                                       components=4)
    ctx = mb.Context(sysm, precision='double')
    ctx.uploadPositions(mb.forcefield.water_positions_with_m(waters))
    e = ctx.evaluateResident(components=4)
    return e, ctx.downloadForces(), ctx.getStats()


def test_more_lower_pairs_than_groups(mb):
    """4.5 M pairs of lower molecules on 2^22 groups of lanes."""
    waters = droplet(3000)
    e0, f0, s0 = energy(mb, waters, 0.95)  # chains: two O-O distances below 0.45 nm, the third below 0.9
    e1, f1, s1 = energy(mb, waters, 1e10)
    print(s0['num_trimers'], s1['num_trimers'], e0[2], e1[2], flush=True)
    assert s1['num_trimers'] == s0['num_trimers']
    assert np.array_equal(e0, e1) and np.array_equal(f0, f1)
