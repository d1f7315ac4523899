"""The 2- and 3-body kernels over list lengths that change their launch: lists of
one unit of 64 and less, remainders of a unit, and lists whose passes are spread
over 6, 3 and 2 blocks and over one.  Slabs of the 256-water lattice without a box
(6, 3, 2) and of the 4096-water one (1), against the term-by-term kernels (pinned to
the oracle by the kernel tests).

Tolerance: both kernels evaluate in FP64 and differ in summation order (1e-15 of
the polynomial's terms, which cancel by about 1e3: 1e-12 of the sums; 1e-10 is
allowed), and every unit's energy and force component is rounded to 2^-32 before it
is summed, so that each unit may add a quantum of difference; 8 are allowed.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


def evaluate(mb, waters, kernel):
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='CutoffNonPeriodic', components=6)
    old = {k: os.environ.get(k) for k in ('MBPOL_HIP_2B_KERNEL', 'MBPOL_HIP_3B_KERNEL')}
    os.environ.update({k: kernel for k in old})
    try:
        ctx = mb.Context(sysm, precision='double')
    finally:
        for k, v in old.items():
            os.environ.pop(k)
            if v is not None:
                os.environ[k] = v
    ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
    st = ctx.getState(components=6)
    return st.getComponentEnergies(), st.getForces(), st.stats


@pytest.mark.parametrize('n', [2, 3, 6, 12, 13, 30, 60, 90, 120, 160, 256])
def test_list_lengths(mb, n):
    waters = mb.systems.config1()[0][:n]
    e0, f0, _ = evaluate(mb, waters, 'terms')
    e1, f1, st = evaluate(mb, waters, 'orbit')
    units = ((st['num_dimers'] + 63) // 64, (st['num_trimers'] + 63) // 64)
    off, norm = np.linalg.norm(f1 - f0), np.linalg.norm(f0)
    print(n, 'waters, units', units, 'forces off %.2g of %.2g' % (off, norm), e1, flush=True)
    quanta = 8 * 2.0 ** -32
    for term, m in (('twobody', st['num_dimers']), ('threebody', st['num_trimers'])):
        assert abs(e1[term] - e0[term]) <= 1e-10 * abs(e0[term]) + quanta * m
    # a unit moves 18 or 27 force components
    assert off <= 1e-10 * norm + quanta * np.sqrt(18 * st['num_dimers'] + 27 * st['num_trimers'])


@pytest.mark.parametrize('n', [700, 1500])
def test_long_lists(mb, n):
    waters = mb.systems.config2()[0][:n]
    e0, f0, _ = evaluate(mb, waters, 'terms')
    e1, f1, st = evaluate(mb, waters, 'orbit')
    assert 2 * ((st['num_dimers'] + 63) // 64) > 256 or n < 1500  # one block a unit on 256 CUs
    assert 2 * ((st['num_trimers'] + 63) // 64) > 256
    off, norm = np.linalg.norm(f1 - f0), np.linalg.norm(f0)
    print(n, 'waters', st['num_dimers'], st['num_trimers'], 'forces off %.2g of %.2g' % (off, norm), e1, flush=True)
    quanta = 8 * 2.0 ** -32
    for term, m in (('twobody', st['num_dimers']), ('threebody', st['num_trimers'])):
        assert abs(e1[term] - e0[term]) <= 1e-10 * abs(e0[term]) + quanta * m
    assert off <= 1e-10 * norm + quanta * np.sqrt(18 * st['num_dimers'] + 27 * st['num_trimers'])
