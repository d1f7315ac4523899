"""Dispersion over its cell grids (half-cutoff cells, and none) against the oracle.

Boxes with the fewest cells per axis, unequal axes, and a dense slab beside empty cells, whose ranges
exceed 64 atoms.  FP64 mode; the tolerances are the parity tests' (1e-9 of the energy, 1e-8 of the RMS
force): both sum the same pairs in FP64 in another order.
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


@pytest.mark.parametrize('box, lattice, slab', [
    ((1.9, 2.0, 1.85), (6, 6, 6), None),
    ((2.25, 2.25, 2.25), (7, 7, 7), None),
    ((2.3, 2.75, 3.2), (7, 8, 10), None),
    ((2.3, 2.3, 6.0), (9, 9, 7), (0.3, 1.9)),
])
def test_dispersion_matches_oracle(mb, oracle, box, lattice, slab):
    rng = np.random.default_rng(5)
    low, high = np.zeros(3), np.array(box)
    if slab:
        low[2], high[2] = slab
    site = np.stack(np.meshgrid(*(np.arange(c) for c in lattice), indexing='ij'), axis=-1).reshape(-1, 3)
    oxygen = low + (site + 0.5) * (high - low) / np.array(lattice) + rng.uniform(-0.01, 0.01, (len(site), 3))
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    waters = oxygen[:, None, :] + h + rng.integers(-1, 2, (len(site), 1, 3)) * np.array(box)
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='PME', box=box, components=8)
    pos = mb.forcefield.water_positions_with_m(waters)
    ctx = mb.Context(sysm, precision='double')
    ctx.setPositions(pos)
    st = ctx.getState(components=8)
    E, F = oracle.evaluate_system(sysm, pos, components=8)
    err = np.sqrt(np.mean((st.getForces() - F) ** 2) / np.mean(F ** 2))
    print(len(waters), st.getPotentialEnergy(), E['dispersion'], 'force rel rms %.2g' % err, flush=True)
    assert abs(st.getPotentialEnergy() - E['dispersion']) <= 1e-9 * abs(E['dispersion'])
    assert err <= 1e-8


@pytest.mark.parametrize('edge', [
    2.8,    # 6^3 cells of half the cutoff, three atoms each: taken
    3.2,    # 7^3: cells of the cutoff
    46.5,
    650.0,  # half cells would be more than an int holds
])
def test_few_waters_in_a_large_box(mb, oracle, edge):
    rng = np.random.default_rng(9)
    # a droplet across a corner of the box
    site = np.stack(np.meshgrid(*(np.arange(6),) * 3, indexing='ij'), axis=-1).reshape(-1, 3)
    oxygen = (site - 2.5) * 0.31 + rng.uniform(-0.01, 0.01, (len(site), 3))
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    waters = oxygen[:, None, :] + h
    waters += np.where(waters[:, :1] < 0, edge, 0.0)
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='PME', box=edge, components=8)
    pos = mb.forcefield.water_positions_with_m(waters)
    ctx = mb.Context(sysm, precision='double')
    ctx.setPositions(pos)
    st = ctx.getState(components=8)
    E, F = oracle.evaluate_system(sysm, pos, components=8)
    err = np.sqrt(np.mean((st.getForces() - F) ** 2) / np.mean(F ** 2))
    print(edge, st.getPotentialEnergy(), E['dispersion'], 'force rel rms %.2g' % err, flush=True)
    assert abs(st.getPotentialEnergy() - E['dispersion']) <= 1e-9 * abs(E['dispersion'])
    assert err <= 1e-8
