"""What a short 2- or 3-body list, whose units are spread over several blocks, is rounded to.

Energies and force components are summed in fixed point, 2^-32 kJ/mol (and /nm) a quantum.  A unit is
summed in FP64 and rounded once, however many blocks share it: one trimer then differs from the
term-by-term kernel (one block per unit, the same FP64 value to about 1e-12) by one quantum at most,
where the two values lie on either side of a rounding boundary; rounded in each of 6 blocks it is off by
up to 3.  (One dimer's force components, sums of much larger terms, differ by up to 3 quanta between the
kernels in FP64 already.)
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUANTUM = 2.0 ** -32


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


def context(mb, n, components, kernel, monkeypatch):
    monkeypatch.setenv('MBPOL_HIP_2B_KERNEL', kernel)
    monkeypatch.setenv('MBPOL_HIP_3B_KERNEL', kernel)
    sysm = mb.forcefield.create_system(n, nonbonded_method='CutoffNonPeriodic', components=components)
    return mb.Context(sysm, precision='double')


def evaluate(mb, ctx, waters, components):
    ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
    st = ctx.getState(components=components)
    return st.getPotentialEnergy(), st.getForces(), st.stats


def test_one_trimer_is_rounded_once(mb, monkeypatch):
    components, size = 4, 3
    box = mb.systems.config1()[0]
    orbit = context(mb, size, components, 'orbit', monkeypatch)
    terms = context(mb, size, components, 'terms', monkeypatch)
    worst, used = 0.0, 0
    for first in range(0, 200):
        # a water and its nearest neighbours
        near = np.argsort(((box[:, 0] - box[first, 0]) ** 2).sum(-1), kind='stable')[:size]
        e0, f0, st = evaluate(mb, terms, box[near], components)
        e1, f1, _ = evaluate(mb, orbit, box[near], components)
        if st['num_dimers'] + st['num_trimers'] != 1:
            continue
        used += 1
        off = max(abs(e1 - e0), np.abs(f1 - f0).max())
        worst = max(worst, off / QUANTUM)
        assert off <= QUANTUM, (first, off / QUANTUM)
    print(used, 'units, worst', worst, 'quanta', flush=True)
    assert used > 100
